// Row-gathered GEMMs for the translation operators.
//
//   C[crow[i] + n] (=|+=) alpha * sum_k A[arow[i] + k] * B[k][n]
//
// Used for the pseudo-inverse applications of P2M / L2P (reference
// fmm_scale_invariant.h:189-193, 215-219: two gemv per leaf, here one launch
// over the leaves of all levels), for M2M (fmm_scale_invariant.h:243-251: the
// 8 child vectors of a parent are contiguous, so a level is one GEMM with
// K = 8*nsurf against the stacked transposed M2M matrices) and for L2L
// (fmm_scale_invariant.h:260-268: N = 8*nsurf against the concatenated
// transposed L2L matrices, accumulating into the contiguous child vectors).
//
// All of them run on the matrix cores.  Complex operands (Helmholtz) come as
// real GEMMs: interleaved (re, im) rows times the operator expanded into real
// 2 x 2 blocks [[Re, Im], [-Im, Re]] (K and N doubled, built once by the
// engine when the operators are set).
#include <algorithm>

#include "kernels.h"

namespace xfmm {

// Compute types: FP64 (v_mfma_f64_16x16x4_f64, result register q of lane
// group g = row g + 4q) or FP32 (v_mfma_f32_16x16x4_f32, row 4g + q) for
// operators that tolerate it; A (the vectors) is FP64 in memory and rounded
// as it is used, B (the operator) is read in the compute type, results are
// stored as FP64.  KL = consecutive K entries of a lane per fragment (16
// bytes of B), KB = 4 KL = K entries of a fragment.
template <typename CT>
struct GemmMfma;
template <>
struct GemmMfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  typedef double frag __attribute__((ext_vector_type(2)));
  static constexpr int KL = 2, KB = 8;
  static __device__ __forceinline__ v4 mma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int q) { return g + 4 * q; }
};
template <>
struct GemmMfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  typedef float frag __attribute__((ext_vector_type(4)));
  static constexpr int KL = 4, KB = 16;
  static __device__ __forceinline__ v4 mma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int q) { return 4 * g + q; }
};

// Packed operators.  Lane (g, j) of a wave (g = lane / 16, j = lane % 16)
// feeds step s < KL of K block kb with k = kb KB + KL g + s, for A and B
// alike (the order of the K sum is free), so that its entries are
// consecutive: one 16-byte load of B, one or two of A.  B is stored as
// [column group of 64][kb][column tile of 16][lane][KL], zero beyond (K, N).
static size_t packed_off(int nkb, int KL, int col, int kb, int lane) {
  return ((size_t(col / 64) * nkb + kb) * 256 + size_t(col / 16 % 4) * 64 + lane) * KL;
}

size_t gemm_packed_size(bool f32, int k, int n) {
  const int KB = f32 ? GemmMfma<float>::KB : GemmMfma<double>::KB;
  const int KL = f32 ? GemmMfma<float>::KL : GemmMfma<double>::KL;
  return packed_off((k + KB - 1) / KB, KL, (n + 63) / 64 * 64, 0, 0);
}

// k, n: sizes of the real form; CPLX: the matrix has k / 2 x n / 2 complex
// entries, each the real block [[Re, Im], [-Im, Re]].  Entry (r, c) of the
// matrix is src[r / ns ns + c][r % ns], rows of ns entries: the transpose of
// one ns x ns matrix, or of 8 of them stacked by rows (M2M) or columns (L2L).
template <typename CT, bool CPLX>
__global__ void k_gemm_pack(int ns, int k, int n, const double* __restrict__ src, CT* __restrict__ out, size_t total) {
  constexpr int KB = GemmMfma<CT>::KB, KL = GemmMfma<CT>::KL, V = CPLX ? 2 : 1;
  const int nkb = (k + KB - 1) / KB;
  const size_t stride = size_t(gridDim.x) * blockDim.x;
  for (size_t e = size_t(blockIdx.x) * blockDim.x + threadIdx.x; e < total; e += stride) {
    const int s = int(e % KL), lane = int(e / KL % 64), ct = int(e / (KL * 64) % 4);
    const size_t gk = e / (KL * 256);  // column group * nkb + kb
    const int kk = int(gk % nkb) * KB + KL * (lane >> 4) + s;
    const int cc = int(gk / nkb) * 64 + ct * 16 + (lane & 15);
    double v = 0;
    if (kk < k && cc < n) {
      const int r = kk / V;
      const double* z = src + ((size_t(r / ns) * ns + cc / V) * ns + r % ns) * V;
      if constexpr (CPLX) v = ((kk ^ cc) & 1) == 0 ? z[0] : (kk & 1) ? -z[1] : z[1];
      else v = z[0];
    }
    out[e] = CT(v);
  }
}

void launch_gemm_pack(bool f32, bool cplx, int ns, int k, int n, const double* src, void* out, hipStream_t s) {
  if (cplx) k *= 2, n *= 2;
  const size_t total = gemm_packed_size(f32, k, n);
  if (total == 0) return;
  const dim3 g(unsigned(std::min<size_t>((total + 255) / 256, 65536))), b(256);
  auto go = [&](auto kern, auto* o) { hipLaunchKernelGGL(kern, g, b, 0, s, ns, k, n, src, o, total); };
  if (f32) cplx ? go(k_gemm_pack<float, true>, static_cast<float*>(out)) : go(k_gemm_pack<float, false>, static_cast<float*>(out));
  else cplx ? go(k_gemm_pack<double, true>, static_cast<double*>(out)) : go(k_gemm_pack<double, false>, static_cast<double*>(out));
}

// A wave computes a (16 TA) x (16 TB) tile of C; a workgroup is RW x CW such
// tiles, each with KW waves that share its K range and add their sums through
// LDS in a fixed order (in FP64).  Operands go straight from global memory
// (L1 / L2) to registers, two K blocks ahead, with no LDS and no barrier in
// the K loop: an FP64 MFMA takes 64 cycles for 8 flop per lane and byte of
// operand, so a wave needs only ~6 bytes a cycle, and small tiles cost
// little.  What bounds it: the FP64 matrix cores (52-60 of 78.6 TFLOP/s on the
// large shapes) and, in FP32, the loads of A in FP64.  Against the previous
// kernel (128 x 128 or 64 x 64 workgroup tiles staged through LDS, one launch per
// level, split-K partial sums in memory): FP64 32768 x 488 x 224 172 -> 129 us, 4096 x 160 x
// 296 64 -> 12, 4096 x 481 x 488 99 -> 39, 4096 x 488 x 3904 333 -> 256;
// FP32 4096 x 488 x 3904 213 -> 157, 4096 x 3904 x 488 249 -> 217, 1 x 488 x 3904
// 19 -> 9 us.
// Tiles are numbered segment by segment, row band by row band; XCD x
// (workgroup id % 8) takes a contiguous eighth of them, so that a band of A
// is read into one L2.
template <typename CT, int TA, int TB, int KW, int RW, int CW, bool BETA>
__global__ __launch_bounds__(64 * KW * RW * CW, 2) void k_gemm_rows(GemmGroup G, const double* __restrict__ A,
                                                                  const long* __restrict__ arow,
                                                                  const CT* __restrict__ B, double* __restrict__ C,
                                                                  const long* __restrict__ crow) {
  typedef GemmMfma<CT> M;
  typedef typename M::v4 v4;
  typedef typename M::frag frag;
  constexpr int KL = M::KL, KB = M::KB, PF = 2;
  static_assert(TB == 1 || TB == 2 || TB == 4, "column tiles of a wave lie in one packed group");
  static_assert(KW == 1 || RW * CW == 1, "waves that share a K range are one tile");
  typedef double dv __attribute__((ext_vector_type(KL)));
  const int per = (G.ntile + 7) / 8;
  const int tile = int(blockIdx.x & 7) * per + int(blockIdx.x >> 3);
  if (int(blockIdx.x >> 3) >= per || tile >= G.ntile) return;  // uniform per workgroup
  int si = 0;
  while (si + 1 < G.nseg && tile >= G.seg[si + 1].tile0) si++;
  const GemmSeg sg = G.seg[si];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int j = lane & 15, g = lane >> 4;
  const int ks = wv % KW, cw = wv / KW % CW, rw = wv / (KW * CW);
  const int nct = (sg.n + 15) / 16, ncg = (nct + TB * CW - 1) / (TB * CW);
  const int row0 = ((tile - sg.tile0) / ncg * RW + rw) * 16 * TA;
  const int ct0 = ((tile - sg.tile0) % ncg * CW + cw) * TB;
  const int nkb = (sg.k + KB - 1) / KB, kfull = sg.k / KB;  // kfull: blocks without a K remainder
  const double* pa[TA];
#pragma unroll
  for (int a = 0; a < TA; a++) pa[a] = A + arow[sg.row0 + min(row0 + a * 16 + j, sg.m - 1)] + KL * g;
  // (a wave past the last column tile or row has no work: its K range is empty)
  const bool live = ct0 < nct && row0 < sg.m;
  const int ctc = live ? ct0 : 0;
  const CT* pb = B + sg.boff + (size_t(ctc / 4) * nkb * 256 + size_t(ctc % 4) * 64 + lane) * KL;
  v4 acc[TA][TB];
#pragma unroll
  for (int a = 0; a < TA; a++)
#pragma unroll
    for (int b = 0; b < TB; b++) acc[a][b] = v4{0, 0, 0, 0};
  const int kper = (nkb + KW - 1) / KW;
  const int kb0 = ks * kper, kb1 = live ? min(nkb, kb0 + kper) : kb0, kbf = min(kfull, kb1);
  // FP32: sums of at most FOLD K blocks (128 products), added to their total
  // one by one, so that rounding does not grow with K (a single chain of 488 or
  // 976 gave 1.2 times the error of the evaluation)
  constexpr int FOLD = 8;
  constexpr bool FOLDS = sizeof(CT) == 4;
  v4 tot[TA][TB];
  auto fold = [&]() {
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
      for (int b = 0; b < TB; b++) {
        tot[a][b] += acc[a][b];
        acc[a][b] = v4{0, 0, 0, 0};
      }
  };
  if constexpr (FOLDS) {
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
      for (int b = 0; b < TB; b++) tot[a][b] = v4{0, 0, 0, 0};
  }
  dv fa[PF][TA];
  frag fb[PF][TB];
  // row offsets are even numbers of doubles: 16-byte aligned loads
  auto load = [&](int kb, dv* xa, frag* xb) {
#pragma unroll
    for (int a = 0; a < TA; a++) {
      const double2* p = reinterpret_cast<const double2*>(pa[a] + kb * KB);
#pragma unroll
      for (int s = 0; s < KL; s += 2) {
        const double2 v = p[s / 2];
        xa[a][s] = v.x;
        xa[a][s + 1] = v.y;
      }
    }
#pragma unroll
    for (int b = 0; b < TB; b++) xb[b] = *reinterpret_cast<const frag*>(pb + (kb * 256 + b * 64) * KL);
  };
  auto mul = [&](const dv* xa, const frag* xb) {
#pragma unroll
    for (int s = 0; s < KL; s++)
#pragma unroll
      for (int a = 0; a < TA; a++) {
        const CT av = CT(xa[a][s]);
#pragma unroll
        for (int b = 0; b < TB; b++) acc[a][b] = M::mma(av, xb[b][s], acc[a][b]);
      }
  };
  if (kb0 < kbf) {
#pragma unroll
    for (int u = 0; u < PF; u++) load(min(kb0 + u, kbf - 1), fa[u], fb[u]);
    int kb = kb0;
    for (; kb + PF <= kbf; kb += PF) {
#pragma unroll
      for (int u = 0; u < PF; u++) {
        mul(fa[u], fb[u]);
        load(min(kb + u + PF, kbf - 1), fa[u], fb[u]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (FOLDS) {
        if ((kb - kb0) % FOLD == FOLD - PF) fold();
      }
    }
#pragma unroll
    for (int u = 0; u < PF; u++)
      if (kb + u < kbf) mul(fa[u], fb[u]);
  }
  if (kfull < kb1 && kfull >= kb0) {  // K remainder: A past the row's end is not read
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
      for (int s = 0; s < KL; s++) fa[0][a][s] = (kfull * KB + KL * g + s < sg.k) ? pa[a][kfull * KB + s] : 0.0;
#pragma unroll
    for (int b = 0; b < TB; b++) fb[0][b] = *reinterpret_cast<const frag*>(pb + (kfull * 256 + b * 64) * KL);
    mul(fa[0], fb[0]);
  }
  if constexpr (FOLDS) {
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
      for (int b = 0; b < TB; b++) acc[a][b] += tot[a][b];
  }
  // result register q of lane (g, j): row M::row(g, q), column j of the tile
  auto put = [&](int r, int cc, double v) {
    double* c = C + crow[sg.row0 + r] + cc;
    v *= sg.alpha;
    *c = BETA ? *c + v : v;
  };
  if constexpr (KW == 1) {
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int r = row0 + a * 16 + M::row(g, q);
        if (r >= sg.m) continue;
#pragma unroll
        for (int b = 0; b < TB; b++) {
          const int cc = (ct0 + b) * 16 + j;
          if (cc < sg.n) put(r, cc, double(acc[a][b][q]));
        }
      }
  } else {
    constexpr int NV = TA * TB * 4;
    __shared__ CT red[KW][NV][64];
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
      for (int b = 0; b < TB; b++)
#pragma unroll
        for (int q = 0; q < 4; q++) red[ks][(a * TB + b) * 4 + q][lane] = acc[a][b][q];
    __syncthreads();
    for (int e = ks; e < NV; e += KW) {
      double v = 0;
#pragma unroll
      for (int z = 0; z < KW; z++) v += double(red[z][e][lane]);
      const int r = row0 + e / 4 / TB * 16 + M::row(g, e & 3), cc = (ct0 + e / 4 % TB) * 16 + j;
      if (r < sg.m && cc < sg.n) put(r, cc, v);
    }
  }
}

template <typename CT, int TA, int TB, int KW, int RW, int CW>
static void launch_tiles(GemmGroup G, const double* A, const long* arow, const CT* B, double* C, const long* crow,
                         bool beta, hipStream_t s) {
  G.ntile = 0;
  for (int i = 0; i < G.nseg; i++) {
    GemmSeg& sg = G.seg[i];
    const int nct = (sg.n + 15) / 16;
    sg.tile0 = G.ntile;
    G.ntile += ((nct + TB * CW - 1) / (TB * CW)) * ((sg.m + 16 * TA * RW - 1) / (16 * TA * RW));
  }
  const dim3 grid(unsigned((G.ntile + 7) / 8 * 8)), block(64 * KW * RW * CW);
  if (beta) hipLaunchKernelGGL((k_gemm_rows<CT, TA, TB, KW, RW, CW, true>), grid, block, 0, s, G, A, arow, B, C, crow);
  else hipLaunchKernelGGL((k_gemm_rows<CT, TA, TB, KW, RW, CW, false>), grid, block, 0, s, G, A, arow, B, C, crow);
}

// Tile and K split by the number of 32 x 64 (w4) and 32 x 32 (w2) wave tiles
// against the chip's 1024 SIMDs, and by the length of K (measured, us):
//  w4 >= 2560: 64 x 128 workgroups of four 32 x 64 tiles (2.5 waves a SIMD hide
//    their own loads; 16 Plummer problems, L2L of some 870 x 2368 x 296, w4 = 1036:
//    the evaluation 3365 with them, 3260 with 32 x 32 tiles);
//  w4 >= 768 and K long: 32 x 64 tiles with K over 4 waves (FP32 4096 x 488 x 3904,
//    w4 = 1024: 157, four waves without a split 203);
//  w2 >= 128: 32 x 32 tiles with K over 4 waves (FP64 4096 x 160 x 296, w2 =
//    640: 12, four waves without a split 14, 32 x 64 23), over 8 or 16
//    when K is long (FP64 512 x 296 x 2368, w2 = 160: 28 with 4, 26 with 8; FP32
//    512 x 488 x 3904 38, 37, 39 with 4, 8, 16: 16, whose FP32 sums are the shortest);
//  else 16 x 16 tiles with K over 8 or 16 waves (FP32 64 x 488 x 3904: 19 and 20,
//    32 x 32 over 8 34; FP64 512 x 160 x 296 5, 32 x 32 over 8 6).
template <typename CT>
static void launch_group(const GemmGroup& G, const double* A, const long* arow, const CT* B, double* C,
                         const long* crow, bool beta, hipStream_t s) {
  constexpr int KLONG = sizeof(CT) == 4 ? 16 : 8;  // waves of a long K
  long w4 = 0, w2 = 0;
  int k = 0;
  for (int i = 0; i < G.nseg; i++) {
    const GemmSeg& sg = G.seg[i];
    w4 += long((sg.m + 31) / 32) * ((sg.n + 63) / 64);
    w2 += long((sg.m + 31) / 32) * ((sg.n + 31) / 32);
    k = std::max(k, sg.k);
  }
  const bool klong = k >= 1024;
  if (w4 >= (klong ? 768 : 2560)) {
    if (klong) launch_tiles<CT, 2, 4, 4, 1, 1>(G, A, arow, B, C, crow, beta, s);
    else launch_tiles<CT, 2, 4, 1, 2, 2>(G, A, arow, B, C, crow, beta, s);
  } else if (w2 >= 128) {
    if (klong) launch_tiles<CT, 2, 2, KLONG, 1, 1>(G, A, arow, B, C, crow, beta, s);
    else launch_tiles<CT, 2, 2, 4, 1, 1>(G, A, arow, B, C, crow, beta, s);
  } else {
    if (klong) launch_tiles<CT, 1, 1, 16, 1, 1>(G, A, arow, B, C, crow, beta, s);
    else launch_tiles<CT, 1, 1, 8, 1, 1>(G, A, arow, B, C, crow, beta, s);
  }
}

void launch_gemm_rows(bool f32, const GemmGroup& G, const double* A, const long* arow, const void* B, double* C,
                      const long* crow, int beta, hipStream_t s) {
  GemmGroup H;
  for (int i = 0; i < G.nseg; i++)
    if (G.seg[i].m > 0 && G.seg[i].n > 0) H.seg[H.nseg++] = G.seg[i];
  if (H.nseg == 0) return;
  if (f32) launch_group<float>(H, A, arow, static_cast<const float*>(B), C, crow, beta != 0, s);
  else launch_group<double>(H, A, arow, static_cast<const double*>(B), C, crow, beta != 0, s);
}

__global__ void k_zero(double* __restrict__ p, size_t n) {
  size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const size_t stride = size_t(gridDim.x) * blockDim.x;
  for (; i < n; i += stride) p[i] = 0.0;
}

void launch_zero(double* p, size_t n, hipStream_t s) {
  if (n == 0) return;
  size_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(k_zero, dim3(unsigned(blocks)), dim3(256), 0, s, p, n);
}

__global__ __launch_bounds__(256) void k_zero_rows(double* __restrict__ p, const long* __restrict__ rows, int len) {
  double* r = p + rows[blockIdx.x];
  for (int i = threadIdx.x; i < len; i += 256) r[i] = 0.0;
}

void launch_zero_rows(double* p, const long* rows, int n, int len, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_zero_rows, dim3(n), dim3(256), 0, s, p, rows, len);
}

__global__ __launch_bounds__(256) void k_charge_sums(const double* __restrict__ q, int n, bool cplx,
                                                     double* __restrict__ out) {
  __shared__ double red[3][256];
  double a = 0, b = 0, c = 0;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += CHARGE_SUM_BLOCKS * 256) {
    const double re = cplx ? q[2 * size_t(i)] : q[i], im = cplx ? q[2 * size_t(i) + 1] : 0.0;
    a += re;
    b += im;
    c += sqrt(re * re + im * im);
  }
  red[0][threadIdx.x] = a;
  red[1][threadIdx.x] = b;
  red[2][threadIdx.x] = c;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w)
      for (int k = 0; k < 3; k++) red[k][threadIdx.x] += red[k][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 3) out[3 * blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}

// One wave per sum: the block sums of a lane, then the lanes, in a fixed order
// (a thread per sum over all 256 blocks: 7 us of load latency, this 3).
__global__ __launch_bounds__(192) void k_charge_sums_total(double* __restrict__ out) {
  const int k = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double t = 0;
#pragma unroll
  for (int b = 0; b < CHARGE_SUM_BLOCKS / 64; b++) t += out[3 * (lane + 64 * b) + k];
  for (int o = 32; o > 0; o >>= 1) t += __shfl_down(t, o, 64);
  if (lane == 0) out[3 * CHARGE_SUM_BLOCKS + k] = t;
}

void launch_charge_sums(const double* q, int n, bool cplx, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_charge_sums, dim3(CHARGE_SUM_BLOCKS), dim3(256), 0, s, q, n, cplx, out);
  hipLaunchKernelGGL(k_charge_sums_total, dim3(1), dim3(192), 0, s, out);
}

__global__ void k_scale_values(double* __restrict__ val, const double* __restrict__ scale, int n, int vw) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const size_t w = size_t(4) * vw;
  if (i >= size_t(n) * w) return;
  const size_t t = i / w, a = (i % w) / vw;
  val[i] *= scale[2 * t + (a == 0 ? 0 : 1)];
}

void launch_scale_values(double* val, const double* scale, int n, int vw, hipStream_t s) {
  const size_t m = size_t(n) * 4 * vw;
  if (m == 0) return;
  hipLaunchKernelGGL(k_scale_values, dim3(unsigned((m + 255) / 256)), dim3(256), 0, s, val, scale, n, vw);
}

__global__ void k_scatter_values(const double* __restrict__ v, const int* __restrict__ perm, int n, int w,
                                 double* __restrict__ out) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= size_t(n) * w) return;
  const size_t t = i / w, e = i % w;
  out[size_t(perm[t]) * w + e] = v[i];
}

void launch_scatter_values(const double* sorted_val, const int* perm, int n, int vw, double* out, hipStream_t s) {
  const int w = 4 * vw;
  const size_t tot = size_t(n) * w;
  if (tot == 0) return;
  hipLaunchKernelGGL(k_scatter_values, dim3(unsigned((tot + 255) / 256)), dim3(256), 0, s, sorted_val, perm, n, w, out);
}

}  // namespace xfmm
