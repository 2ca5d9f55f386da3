// Particle/surface evaluation kernels for gfx950: P2P, M2P, L2P (particle
// targets), P2M check potentials and P2L (surface targets), and the direct
// summation used by verify().
//
// Kernel formulas follow exafmm-t's scalar loops (targets t, sources s,
// d = x_s - x_t, results scaled by 1/(4 pi) at the end):
//   Laplace   laplace.h:139-162:            phi += q/r,            grad += q d / r^3
//   Yukawa    modified_helmholtz.h:149-170: phi += q e^{-kr}/r,    grad += q e^{-kr}(kr+1) d / r^3
//   Helmholtz helmholtz.h:186-207:          phi += q e^{ikr}/r,    grad += (1/r^2 - ik/r) phi_ij d
// Pairs with r = 0 contribute nothing (laplace.h:57, `invr &= r2 > zero`).
//
// Layout: particle targets in tiles of 64 per leaf (P2P and M2P: sources in LDS;
// L2P: a target per lane, sources read as wave-uniform vectors); surface targets with a wave per node, sources
// staged through LDS in tiles of 64.  Coordinates are made relative to a leaf
// centre in FP64 before any FP32 conversion, so the mixed path keeps
// |d| accuracy at the scale of the leaf.  In the FP32 path each tile of 64
// sources is summed in plain FP32 and tiles are combined with compensated
// (Kahan) summation.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "kernels.h"

namespace xfmm {

// Helmholtz with a real wave number (Im k = 0) and phases k r < 2^30 in the
// tree's box (real_phases): the evaluation kernels are instantiated without
// the damping factor e^{-Im(k) r}, which is then exactly 1, and in FP64 with
// sincos_near.  Internal to the launchers of this file.
constexpr int HELMHOLTZ_REAL = 3;

template <int KIND>
constexpr bool kcplx() { return KIND == HELMHOLTZ || KIND == HELMHOLTZ_REAL; }

template <int KIND, typename R>
__device__ __forceinline__ void phase(R x, R* s, R* c) {
  if constexpr (KIND == HELMHOLTZ_REAL && sizeof(R) == 8) sincos_near(x, s, c);
  else dsincos(x, s, c);
}

// 1/r of a pair.  RSQ_LIB: library rsqrt, r = 0 gives 0 (the direct sum used as
// accuracy check).  RSQ_MASK: hardware estimate refined to full precision
// (rsqrt_sep), r^2 <= rmin2 gives 0 (a leaf with itself, where a target may
// coincide with a source; the FP32 near field also leaves out the
// near-coincident pairs that k_close_fix adds in FP64).  RSQ_SEP: rsqrt_sep
// without the test (surfaces never touch particles).  RSQ_SOFT: rsqrt_sep(r^2 +
// rmin2) for two leaves, whose points are distinct but can be rounded to the same
// numbers in the target leaf's frame (soft_r2; the sum starts from rmin2, so
// it costs no instruction).
enum RsqMode { RSQ_LIB = 0, RSQ_MASK = 1, RSQ_SEP = 2, RSQ_SOFT = 3 };
template <int RM, typename R>
__device__ __forceinline__ R dist2(R dx, R dy, R dz, R rmin2) {
  if constexpr (RM == RSQ_SOFT) return fma(dz, dz, fma(dx, dx, fma(dy, dy, rmin2)));
  else return dx * dx + dy * dy + dz * dz;
}
template <int RM, typename R>
__device__ __forceinline__ R inv_r(R r2, R rmin2) {
  if constexpr (RM == RSQ_LIB) return rsqrt_pos(r2);
  else if constexpr (RM == RSQ_MASK) return r2 > rmin2 ? rsqrt_sep(r2) : R(0);
  else return rsqrt_sep(r2);
}

// potential + gradient of one pair, accumulated into a[] (4 or 8 values)
template <int KIND, typename R, int RM>
__device__ __forceinline__ void pair_grad(R dx, R dy, R dz, R qr, R qi, R kr, R ki, R* a, R rmin2 = R(0)) {
  const R r2 = dist2<RM>(dx, dy, dz, rmin2);
  const R invr = inv_r<RM>(r2, rmin2);
  if constexpr (KIND == LAPLACE) {
    const R qinv = qr * invr;
    a[0] += qinv;
    const R s = qinv * invr * invr;
    a[1] += s * dx;
    a[2] += s * dy;
    a[3] += s * dz;
  } else if constexpr (KIND == YUKAWA) {
    const R r = r2 * invr;
    const R qinv = qr * dexp(-kr * r) * invr;
    a[0] += qinv;
    const R s = qinv * (R(1) + kr * r) * invr * invr;
    a[1] += s * dx;
    a[2] += s * dy;
    a[3] += s * dz;
  } else {
    const R r = r2 * invr;
    const R e = KIND == HELMHOLTZ_REAL ? invr : dexp(-ki * r) * invr;
    R sn, cs;
    phase<KIND>(kr * r, &sn, &cs);
    const R gr = e * cs, gi = e * sn;
    const R pr = qr * gr - qi * gi;
    const R pim = qr * gi + qi * gr;
    a[0] += pr;
    a[1] += pim;
    const R cgr = (KIND == HELMHOLTZ_REAL ? invr : (R(1) + ki * r) * invr) * invr;
    const R cgi = -kr * invr;
    const R fr = cgr * pr - cgi * pim;
    const R fi = cgr * pim + cgi * pr;
    a[2] += dx * fr;
    a[3] += dx * fi;
    a[4] += dy * fr;
    a[5] += dy * fi;
    a[6] += dz * fr;
    a[7] += dz * fi;
  }
}

// potential of one pair into a[0] (and a[1] for Helmholtz)
template <int KIND, typename R, int RM>
__device__ __forceinline__ void pair_pot(R dx, R dy, R dz, R qr, R qi, R kr, R ki, R* a) {
  const R r2 = dx * dx + dy * dy + dz * dz;
  const R invr = inv_r<RM>(r2, R(0));
  if constexpr (KIND == LAPLACE) {
    a[0] += qr * invr;
  } else if constexpr (KIND == YUKAWA) {
    a[0] += qr * dexp(-kr * (r2 * invr)) * invr;
  } else {
    const R r = r2 * invr;
    const R e = KIND == HELMHOLTZ_REAL ? invr : dexp(-ki * r) * invr;
    R sn, cs;
    phase<KIND>(kr * r, &sn, &cs);
    const R gr = e * cs, gi = e * sn;
    a[0] += qr * gr - qi * gi;
    a[1] += qr * gi + qi * gr;
  }
}

template <typename R, int NA>
__device__ __forceinline__ void fold_tile(R* acc, R* comp, const R* part) {
  if constexpr (sizeof(R) == 4) {
#pragma unroll
    for (int a = 0; a < NA; a++) kahan_add(acc[a], comp[a], part[a]);
  } else {
#pragma unroll
    for (int a = 0; a < NA; a++) acc[a] += part[a];
  }
}

constexpr int TILE = 64;

// Sum the potentials of the m (<= TILE) staged sources of a tile into part[], in
// source order, four pairs per loop trip so that the LDS reads of a trip are
// issued together.
template <int KIND, typename R, int RM>
__device__ __forceinline__ void tile_sum(int m, const R* sx, const R* sy, const R* sz, const R* sq, const R* sqi, R tx,
                                         R ty, R tz, R kr, R ki, R* part) {
  constexpr bool C = kcplx<KIND>();
  int j = 0;
  for (; j + 4 <= m; j += 4) {
#pragma unroll
    for (int u = 0; u < 4; u++)
      pair_pot<KIND, R, RM>(sx[j + u] - tx, sy[j + u] - ty, sz[j + u] - tz, sq[j + u], C ? sqi[j + u] : R(0), kr, ki,
                            part);
  }
  for (; j < m; j++)
    pair_pot<KIND, R, RM>(sx[j] - tx, sy[j] - ty, sz[j] - tz, sq[j], C ? sqi[j] : R(0), kr, ki, part);
}

// Squared distance below which the FP32 near field of a leaf with itself
// leaves a pair to k_close_fix: (side / 16)^2 of the target leaf when the
// near-coincident pairs are listed (t.close), else 0 (only r = 0 masked).
template <typename R>
__device__ __forceinline__ R close_rmin2(const DevTree& t, int leaf) {
  if constexpr (sizeof(R) == 4) {
    if (t.close) {
      const double side = 2.0 * t.r0 * ldexp(1.0, -t.level[leaf]);
      return R(side * side * (1.0 / 256.0));
    }
  }
  return R(0);
}

// RSQ_SOFT's term for a target leaf.  Two points of different leaves closer than
// a rounding of the leaf's size can get the same position in its frame: r^2 = 0,
// 1/r infinite and a gradient of infinity times zero.  FP32: (2^-18 side)^2 keeps
// their FP32 value finite, below their true value and, since such pairs are listed
// (k_close_find), corrected to it in FP64; it changes 1/r of an unlisted pair (r >=
// side / 16) by less than 2^-29.  FP64: (2^-54 side)^2, of the size of the
// distances that the frame resolves.
template <typename R>
__device__ __forceinline__ R soft_r2(const DevTree& t, int leaf) {
  const double e = 2.0 * t.r0 * ldexp(1.0, -t.level[leaf] - (sizeof(R) == 4 ? 18 : 54)), e2 = e * e;
  if constexpr (sizeof(R) == 4) return R(e2);
  // one value for all lanes: FP64 keeps it in scalar registers (W = 16 would take
  // 122 vector registers, with them 120)
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(e2)),
                          __builtin_amdgcn_readfirstlane(__double2loint(e2)));
}

// ---------------------------------------------- particle targets: P2P, M2P, L2P
//
// One workgroup of W waves per (leaf, tile of TILE targets), work[2 b] = leaf,
// work[2 b + 1] = tile.  In L2P and M2P a full tile has a target per lane; a tail
// tile of nt <= t.p2p_split (<= TILE / 2) targets gives each target TILE / nt lanes
// (target lane % nt, phase lane / nt) that take every (TILE / nt)-th source.  L2P
// reads its sources as wave-uniform vectors (scalar loads from constant address
// space, no LDS and no barriers), M2P and P2P stage theirs in LDS.  The W waves
// share the sources; the partial sums of a target are added in FP64 through LDS in
// a fixed order.  Pairs are summed in chunks of 64 sources (plain sums, FP32 chunks
// combined with Kahan summation).
// W (particle_waves): a wave per tile leaves a small tree's chip idle and its
// longest tile is the time.
template <int KIND>
constexpr int nval() { return kcplx<KIND>() ? 8 : 4; }  // values per target

// The tile of this workgroup and the target of this lane.
template <typename R>
struct Tile {
  int leaf, tb, nt, k, ti, ph, wave;
  bool split, act;
  double cx, cy, cz;
  R tx, ty, tz;  // target relative to its leaf centre
  __device__ __forceinline__ Tile(const DevTree& t, const int* work) {
    leaf = work[2 * blockIdx.x];
    const int t0 = TILE * work[2 * blockIdx.x + 1];
    const int lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    cx = t.center[3 * leaf];
    cy = t.center[3 * leaf + 1];
    cz = t.center[3 * leaf + 2];
    tb = t.trg_begin[leaf] + t0;
    nt = min(TILE, t.trg_count[leaf] - t0);
    split = nt <= t.p2p_split;
    k = split ? TILE / nt : 1;
    ti = split ? lane % nt : lane;
    ph = split ? lane / nt : 0;
    act = split ? ph < k : ti < nt;
    tx = ty = tz = 0;
    if (ti < nt) {
      const double* x = t.trg + 3 * size_t(tb + ti);
      tx = R(x[0] - cx);
      ty = R(x[1] - cy);
      tz = R(x[2] - cz);
    }
  }
};

// trg_value of the tile's targets = (with t.set_values) or += the sums of its
// lanes and waves / 4 pi (+ near_add).
template <int NA, int W, typename R>
__device__ __forceinline__ void put_tile(const DevTree& t, const Tile<R>& T, const R* acc, const R* comp,
                                         const double* near_add) {
  auto add = [&](int i, const double* v) {
    double* o = t.trg_value + size_t(T.tb + i) * NA;
    const double* n = near_add ? near_add + size_t(T.tb + i) * NA : nullptr;
#pragma unroll
    for (int a = 0; a < NA; a++) {
      const double r = (t.set_values ? 0.0 : o[a]) + v[a] * FOUR_PI_INV;
      o[a] = n ? r + n[a] : r;
    }
  };
  if (W == 1 && !T.split) {
    if (T.act) {
      double v[NA];
#pragma unroll
      for (int a = 0; a < NA; a++) v[a] = double(acc[a]) - double(comp[a]);
      add(T.ti, v);
    }
    return;
  }
  __shared__ double red[W][NA][TILE];
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int a = 0; a < NA; a++) red[T.wave][a][lane] = double(acc[a]) - double(comp[a]);
  __syncthreads();
  if (int(threadIdx.x) < T.nt) {
    double v[NA];
#pragma unroll
    for (int a = 0; a < NA; a++) {
      v[a] = 0;
      for (int w = 0; w < W; w++)
        for (int ph = 0; ph < T.k; ph++) v[a] += red[w][a][threadIdx.x + ph * T.nt];
    }
    add(threadIdx.x, v);
  }
}

// Readers of a list of sources: get(u, v) puts x, y, z, q (and Im q, else 0) of
// source u from the current one on into v, skip(n) moves on by n sources.
// P, E: pointers to positions (stride PS) and densities (stride ES); with ES = 0
// the densities follow the position.
template <typename R, int NQ, int PS, int ES, typename P, typename E>
struct Sources {
  P p;
  E e;
  __device__ __forceinline__ Sources(P p_, E e_) : p(p_), e(e_) {}
  __device__ __forceinline__ void skip(int n) {
    p += size_t(PS) * n;
    if constexpr (ES > 0) e += size_t(ES) * n;
  }
  __device__ __forceinline__ void get(int u, R* v) const {
#pragma unroll
    for (int d = 0; d < 3; d++) v[d] = p[PS * u + d];
#pragma unroll
    for (int d = 0; d < 2; d++) {
      if constexpr (ES > 0) v[3 + d] = d < NQ ? R(e[ES * u + (d < NQ ? d : 0)]) : R(0);
      else v[3 + d] = d < NQ ? p[PS * u + (d < NQ ? 3 + d : 0)] : R(0);
    }
  }
};

// Sum of n sources of a full tile in chunks of TILE, four pairs per loop trip.
template <int KIND, typename R, int RM, typename SRC>
__device__ __forceinline__ void sum_uniform(int n, SRC src, R ux, R uy, R uz, R kr, R ki, R* acc, R* comp, R rmin2) {
  constexpr int NA = nval<KIND>();
  for (int s0 = 0; s0 < n; s0 += TILE) {
    const int m = min(TILE, n - s0);
    R part[NA] = {0};
    int j = 0;
    for (; j + 4 <= m; j += 4) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        R v[5];
        src.get(u, v);
        pair_grad<KIND, R, RM>(v[0] - ux, v[1] - uy, v[2] - uz, v[3], v[4], kr, ki, part, rmin2);
      }
      src.skip(4);
    }
    for (; j < m; j++) {
      R v[5];
      src.get(0, v);
      pair_grad<KIND, R, RM>(v[0] - ux, v[1] - uy, v[2] - uz, v[3], v[4], kr, ki, part, rmin2);
      src.skip(1);
    }
    fold_tile<R, NA>(acc, comp, part);
  }
}
// The same for a split tile: this lane's sources ph, ph + k, ..., in chunks of
// TILE per lane; the loads of four pairs are issued together (one at a time
// their latency is the time).
template <int KIND, typename R, int RM, typename SRC>
__device__ __forceinline__ void sum_split(int n, const Tile<R>& T, SRC src, R ux, R uy, R uz, R kr, R ki, R* acc,
                                          R* comp, R rmin2) {
  constexpr int NA = nval<KIND>();
  src.skip(T.ph);
  for (int s0 = 0; s0 < n; s0 += TILE * T.k) {
    const int e = min(n, s0 + TILE * T.k);
    R part[NA] = {0};
    if (T.act) {
      int j = s0 + T.ph;
      for (; j + 3 * T.k < e; j += 4 * T.k) {
        R v[4][5];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          src.get(0, v[u]);
          src.skip(T.k);
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
          pair_grad<KIND, R, RM>(v[u][0] - ux, v[u][1] - uy, v[u][2] - uz, v[u][3], v[u][4], kr, ki, part, rmin2);
      }
      for (; j < e; j += T.k) {
        R v[5];
        src.get(0, v);
        src.skip(T.k);
        pair_grad<KIND, R, RM>(v[0] - ux, v[1] - uy, v[2] - uz, v[3], v[4], kr, ki, part, rmin2);
      }
    }
    fold_tile<R, NA>(acc, comp, part);
  }
}

// Values of a source in LDS: position, charge.
template <int KIND>
constexpr int npack() { return kcplx<KIND>() ? 5 : 4; }

// A workgroup of W waves per (leaf, tile of TILE targets).  A lane holds M targets
// (target l + u L of the tile in lane l, L = ceil(nt / M)), so that k = 64 / L
// lanes share a target's sources and few lanes are left over: leaves of 24
// targets use 60 of 64 lanes (48 with one target in a lane).  The sources of
// all leaves of the list are one sequence, moved into the target leaf's frame
// on their way to LDS (subtracted in FP64, rounded once), padded with zero
// charges to whole trips of the loop; the W waves take a part of every block
// each, the k lane groups every k-th source of it, two of them per trip, and the
// sums are added in FP64 in a fixed order.  A tile of more than t.p2p_split
// targets uses two lane groups at most; with t.p2p_split = 0 a single wave sums a
// target's sources in one lane (W = M = 1).
// Sources packed beforehand relative to their own leaf (half the bytes in FP32)
// and shifted here cost FP32 two more roundings per coordinate, 5 to 7 times the
// error of a pair across a leaf plane, and were no faster (2M points 1.18 ms
// either way; Helmholtz FP32, 4096 leaves of 49, 312 and 305 us).
// Bound by the vector units: 14 instructions a pair (Laplace FP32).  Per source
// leaf and tile instead (full tiles with a target per lane and scalar loads,
// others with the lane groups reading each leaf from the vector cache) the small
// leaves paid for remainders and for 16 lanes' worth of cache reads a pair.  That
// and this, us: FP32, 32768 leaves of 30 targets 519 and 475, of 61 1214 and 1200; 38841
// Plummer leaves of 15 478 and 377; Yukawa FP32, 15074 leaves of 20 220 and 180; FP64,
// 12069 leaves of 41 1228 and 1105; Helmholtz FP64, 512 leaves of 59 268 and 191.
// 128 sources a wave: 256 cost up to 7 %, 512 up to 40 % (fewer workgroups on a
// CU); the next block loaded ahead gives nothing.
// M = 1 for Helmholtz where M = 2 costs waves by its registers (FP32, 4096 leaves
// of 49: 284 and 303 us; FP64 with sincos_near, 512 leaves of 59: 186 and 195), but
// not in FP64 with the library's sincos, whose branch wants pairs to overlap (460
// and 268).
template <int KIND, typename R>
constexpr int points_per_lane() { return kcplx<KIND>() && (sizeof(R) == 4 || KIND == HELMHOLTZ_REAL) ? 1 : 2; }

template <int KIND, typename R, int W, int M = points_per_lane<KIND, R>()>
__global__ __launch_bounds__(64 * W) void k_p2p(DevTree t, Wavek wk, const int* __restrict__ work) {
  constexpr int NA = nval<KIND>(), NP = npack<KIND>();
  constexpr int CAP = 128 * W;  // sources in LDS
  constexpr int NE = 64;        // source leaves listed at a time
  // (with ROOM, which nothing uses, a CU holds fewer of these workgroups beside the
  // transforms on the other stream, which finish sooner: the evaluation in FP64,
  // 60k -> 100k Laplace 881 and 871 us, 30k Helmholtz 507 and 499; this kernel alone the same)
  constexpr int ROOM = 3 * NE * sizeof(R);
  constexpr int SZ = std::max(int(CAP * NP * sizeof(R)), int(W * NA * 64 * sizeof(double))) + ROOM;
  __shared__ __attribute__((aligned(16))) char smem[SZ];
  __shared__ int pre[NE + 1], first[NE], self;
  R* sp = reinterpret_cast<R*>(smem);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int leaf = work[2 * blockIdx.x], t0 = TILE * work[2 * blockIdx.x + 1];
  const int tb = t.trg_begin[leaf] + t0, nt = min(TILE, t.trg_count[leaf] - t0);
  const int L = (nt + M - 1) / M, kmax = 64 / L, k = nt <= t.p2p_split ? kmax : t.p2p_split > 0 ? min(kmax, 2) : 1;
  const int l = lane % L, ph = lane / L < k ? lane / L : 0;
  const double cx = t.center[3 * leaf], cy = t.center[3 * leaf + 1], cz = t.center[3 * leaf + 2];
  const R far = R(4.0 * t.r0 * ldexp(1.0, -t.level[leaf]));
  const R kr = R(wk.re), ki = R(wk.im), rmin2 = close_rmin2<R>(t, leaf), soft = soft_r2<R>(t, leaf);
  R x[M][3], acc[M][NA], comp[M][NA];
#pragma unroll
  for (int u = 0; u < M; u++) {
    const double* p = t.trg + 3 * size_t(tb + min(l + u * L, nt - 1));
    x[u][0] = R(p[0] - cx);
    x[u][1] = R(p[1] - cy);
    x[u][2] = R(p[2] - cz);
#pragma unroll
    for (int a = 0; a < NA; a++) { acc[u][a] = 0; comp[u][a] = 0; }
  }
  const int unit = 2 * W * k, most = min(CAP / unit * unit, TILE * W * k);  // at most TILE sources a lane and block
  // source i of the tree in the target leaf's frame
  auto get = [&](int i, R* v) {
    const double* p = t.src + 3 * size_t(i);
    const double* q = t.q + size_t(i) * (NP - 3);
    v[0] = R(p[0] - cx);
    v[1] = R(p[1] - cy);
    v[2] = R(p[2] - cz);
#pragma unroll
    for (int d = 3; d < NP; d++) v[d] = R(q[d - 3]);
  };
  // all pairs of total sources, source i read by load(i, v)
  auto sums = [&](auto RM, int total, auto load) {
    for (int s0 = 0; s0 < total; s0 += most) {
      const int m = min(most, total - s0), n = (m + unit - 1) / unit * unit, steps = n / (W * k);
      __syncthreads();
      for (int i = tid; i < n; i += 64 * W) {
        R v[NP] = {far};
        if (i < m) load(s0 + i, v);
#pragma unroll
        for (int d = 0; d < NP; d++) sp[NP * i + d] = v[d];
      }
      __syncthreads();
      const R* S = sp + NP * (wave * steps * k + ph);
      R part[M][NA] = {};
      for (int j = 0; j < steps; j += 2) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const R w[5] = {S[0], S[1], S[2], S[3], NP > 4 ? S[NP - 1] : R(0)};
          S += NP * k;
#pragma unroll
          for (int u = 0; u < M; u++)
            pair_grad<KIND, R, decltype(RM)::value>(w[0] - x[u][0], w[1] - x[u][1], w[2] - x[u][2], w[3], w[4], kr, ki,
                                                    part[u], RM == RSQ_MASK ? rmin2 : soft);
        }
      }
#pragma unroll
      for (int u = 0; u < M; u++) fold_tile<R, NA>(acc[u], comp[u], part[u]);
    }
  };
  if (tid == 0) self = 0;
  const int g1 = t.p2p_off[leaf + 1];
  for (int g0 = t.p2p_off[leaf]; g0 < g1; g0 += NE) {
    __syncthreads();
    if (tid < NE) {
      int n = 0;
      if (g0 + tid < g1) {
        const int s = t.p2p_src[g0 + tid];
        if (s == leaf) self = 1;
        else n = t.src_count[s];
        first[tid] = t.src_begin[s];
      }
#pragma unroll
      for (int d = 1; d < 64; d *= 2) {
        const int o = __shfl_up(n, d);
        if (tid >= d) n += o;
      }
      pre[tid + 1] = n;
      if (tid == 0) pre[0] = 0;
    }
    __syncthreads();
    sums(std::integral_constant<int, RSQ_SOFT>(), pre[NE], [&](int i, R* v) {
      int e = 0;  // the last leaf with pre[e] <= i
#pragma unroll
      for (int d = NE / 2; d > 0; d /= 2)
        if (pre[e + d] <= i) e += d;
      get(first[e] + i - pre[e], v);
    });
  }
  __syncthreads();
  // only a leaf with itself can pair coinciding points
  if (self)
    sums(std::integral_constant<int, RSQ_MASK>(), t.src_count[leaf],
         [&](int i, R* v) { get(t.src_begin[leaf] + i, v); });
  double* red = reinterpret_cast<double*>(smem);
#pragma unroll
  for (int u = 0; u < M; u++) {
    __syncthreads();
#pragma unroll
    for (int a = 0; a < NA; a++) red[(wave * NA + a) * 64 + lane] = double(acc[u][a]) - double(comp[u][a]);
    __syncthreads();
    const int n = min(L, nt - u * L);
    for (int i = tid; i < n * NA; i += 64 * W) {
      const int ti = i / NA, a = i % NA;
      double v = 0;
      for (int w = 0; w < W; w++)
        for (int h = 0; h < k; h++) v += red[(w * NA + a) * 64 + ti + h * L];
      double* o = t.trg_value + size_t(tb + u * L) * NA + i;
      *o = (t.set_values ? 0.0 : *o) + v * FOUR_PI_INV;
    }
  }
}

// L2P (fmm_scale_invariant.h:198-230, fmm.h:188-218).  The sources are the points
// of the leaf's own downward equivalent surface (alpha 2.95), from a per-level
// table relative to the box centre, with the leaf's densities: the same for
// every lane of a full tile.  The W waves share the points.
template <int KIND, typename R, int W>
__global__ __launch_bounds__(64 * W) void k_l2p_smem(DevTree t, Wavek wk, const int* __restrict__ work) {
  constexpr int NA = nval<KIND>();
  constexpr bool C = kcplx<KIND>();
  typedef const double __attribute__((address_space(4))) * CD;
  // surface points in the arithmetic type (no per-source conversions)
  typedef const R __attribute__((address_space(4))) * CR;
  const Tile<R> T(t, work);
  const R kr = R(wk.re), ki = R(wk.im);
  const int ns = t.nsurf;
  const R* tab;
  if constexpr (sizeof(R) == 4) tab = t.surf_tab32;
  else tab = t.surf_tab;
  tab += size_t(t.level[T.leaf]) * ns * 4;
  const double* eq = t.dn + size_t(T.leaf) * ns * (C ? 2 : 1);
  R acc[NA], comp[NA];
#pragma unroll
  for (int a = 0; a < NA; a++) { acc[a] = 0; comp[a] = 0; }
  const int per = ((ns + W - 1) / W + 3) / 4 * 4, j0 = min(ns, T.wave * per), n = min(ns, j0 + per) - j0;
  constexpr int NQ = C ? 2 : 1;
  const R* p0 = tab + 4 * size_t(j0);
  const double* e0 = eq + NQ * size_t(j0);
  const Sources<R, NQ, 4, NQ, const R*, const double*> vec(p0, e0);
  const Sources<R, NQ, 4, NQ, CR, CD> uni((CR)(p0), (CD)(e0));
  // the surface never touches the targets
  if (T.split) sum_split<KIND, R, RSQ_SEP>(n, T, vec, T.tx, T.ty, T.tz, kr, ki, acc, comp, R(0));
  else sum_uniform<KIND, R, RSQ_SEP>(n, uni, T.tx, T.ty, T.tz, kr, ki, acc, comp, R(0));
  put_tile<NA, W>(t, T, acc, comp, t.near_add);
}

// M2P (fmm_base.h:97-124): the sources are the upward equivalent surfaces (alpha
// 1.05) of the nodes of the M2P list.  Few leaves have such lists and their
// nodes lie all over memory, so what counts is latency: the W waves stage a
// node's points (relative to the target leaf's centre, formed in FP64) and
// densities in LDS at once and share them.  16 Plummer problems (2007 leaves
// with 1..16 nodes, 74 M pairs): a wave per leaf, 64 points staged at a time
// 225 us; four waves 88.
template <int KIND, typename R, int W>
__global__ __launch_bounds__(64 * W) void k_m2p(DevTree t, Wavek wk, const int* __restrict__ work) {
  constexpr int NA = nval<KIND>();
  constexpr bool C = kcplx<KIND>();
  constexpr int NP = npack<KIND>(), NB = 256;  // points per LDS block
  __shared__ R sp[NB * NP];
  const Tile<R> T(t, work);
  const R kr = R(wk.re), ki = R(wk.im);
  const int ns = t.nsurf;
  R acc[NA], comp[NA];
#pragma unroll
  for (int a = 0; a < NA; a++) { acc[a] = 0; comp[a] = 0; }
  for (int g = t.m2p_off[T.leaf]; g < t.m2p_off[T.leaf + 1]; g++) {
    const int snode = t.m2p_src[g];
    const double b = 1.05 * t.r0 * ldexp(1.0, -t.level[snode]);
    const double ox = t.center[3 * snode] - T.cx, oy = t.center[3 * snode + 1] - T.cy,
                 oz = t.center[3 * snode + 2] - T.cz;
    const double* eq = t.up + size_t(snode) * ns * (C ? 2 : 1);
    for (int s0 = 0; s0 < ns; s0 += NB) {
      const int m = min(NB, ns - s0);
      __syncthreads();
      for (int i = threadIdx.x; i < m; i += 64 * W) {
        const int si = s0 + i;
        R* p = sp + NP * i;
        p[0] = R(ox + t.unit_surf[3 * si] * b);
        p[1] = R(oy + t.unit_surf[3 * si + 1] * b);
        p[2] = R(oz + t.unit_surf[3 * si + 2] * b);
        p[3] = R(eq[C ? 2 * si : si]);
        if (C) p[NP - 1] = R(eq[2 * si + 1]);
      }
      __syncthreads();
      const int per = ((m + W - 1) / W + 3) / 4 * 4, j0 = min(m, T.wave * per), n = min(m, j0 + per) - j0;
      const Sources<R, NP - 3, NP, 0, const R*, int> src(sp + NP * j0, 0);
      if (T.split) sum_split<KIND, R, RSQ_SEP>(n, T, src, T.tx, T.ty, T.tz, kr, ki, acc, comp, R(0));
      else sum_uniform<KIND, R, RSQ_SEP>(n, src, T.tx, T.ty, T.tz, kr, ki, acc, comp, R(0));
    }
  }
  put_tile<NA, W>(t, T, acc, comp, nullptr);
}

template <int KIND, typename R, int MODE>
__global__ __launch_bounds__(64) void k_eval_surface(DevTree t, Wavek wk, const int* __restrict__ work,
                                                     double* __restrict__ check) {
  constexpr bool C = kcplx<KIND>();
  constexpr int NA = C ? 2 : 1;
  __shared__ R sx[TILE], sy[TILE], sz[TILE], sq[TILE], sqi[TILE];
  const int node = work[blockIdx.x];
  const int lane = threadIdx.x;
  const double cx = t.center[3 * node], cy = t.center[3 * node + 1], cz = t.center[3 * node + 2];
  const double b = ((MODE == MODE_P2M) ? 2.95 : 1.05) * t.r0 * ldexp(1.0, -t.level[node]);
  const R kr = R(wk.re), ki = R(wk.im);
  const int vw = t.vw;
  int g0 = 0, g1 = 1;
  if (MODE == MODE_P2L) { g0 = t.p2l_off[node]; g1 = t.p2l_off[node + 1]; }
  for (int i0 = TILE * blockIdx.y; i0 < t.nsurf; i0 += TILE * gridDim.y) {
    const int i = i0 + lane;
    const bool act = i < t.nsurf;
    R px = 0, py = 0, pz = 0;
    if (act) {
      px = R(t.unit_surf[3 * i] * b);
      py = R(t.unit_surf[3 * i + 1] * b);
      pz = R(t.unit_surf[3 * i + 2] * b);
    }
    R acc[NA], comp[NA];
#pragma unroll
    for (int a = 0; a < NA; a++) { acc[a] = 0; comp[a] = 0; }
    for (int g = g0; g < g1; g++) {
      const int snode = (MODE == MODE_P2L) ? t.p2l_src[g] : node;
      const int sb = t.src_begin[snode], ns = t.src_count[snode];
      for (int s0 = 0; s0 < ns; s0 += TILE) {
        const int m = min(TILE, ns - s0);
        __syncthreads();
        if (lane < m) {
          const double* x = t.src + 3 * size_t(sb + s0 + lane);
          sx[lane] = R(x[0] - cx);
          sy[lane] = R(x[1] - cy);
          sz[lane] = R(x[2] - cz);
          const double* qq = t.q + size_t(sb + s0 + lane) * vw;
          sq[lane] = R(qq[0]);
          if (C) sqi[lane] = R(qq[1]);
        }
        __syncthreads();
        R part[NA];
#pragma unroll
        for (int a = 0; a < NA; a++) part[a] = 0;
        // check surfaces are well separated from the source particles
        tile_sum<KIND, R, RSQ_SEP>(m, sx, sy, sz, sq, sqi, px, py, pz, kr, ki, part);
        fold_tile<R, NA>(acc, comp, part);
      }
    }
    if (act) {
      if (MODE == MODE_P2M) {
        double* o = check + (size_t(blockIdx.x) * t.nsurf + i) * vw;
#pragma unroll
        for (int a = 0; a < NA; a++) o[a] = (double(acc[a]) - double(comp[a])) * FOUR_PI_INV;
      } else {
        double* o = t.dn + (size_t(node) * t.nsurf + i) * vw;
#pragma unroll
        for (int a = 0; a < NA; a++) o[a] += (double(acc[a]) - double(comp[a])) * FOUR_PI_INV;
      }
    }
  }
}

// Direct sum: block (x = 64 targets, y = source split).  Differences are
// formed in FP64; tiles are combined with compensated summation in both
// precisions (this kernel is the repository's accuracy check).
template <int KIND, typename R, bool GRAD>
__global__ __launch_bounds__(64) void k_direct(const double* __restrict__ src, const double* __restrict__ q, int ns,
                                               const double* __restrict__ trg, int nt, double* __restrict__ partial,
                                               int chunk, Wavek wk) {
  constexpr bool C = kcplx<KIND>();
  constexpr int NA = GRAD ? (C ? 8 : 4) : (C ? 2 : 1);
  constexpr int vw = C ? 2 : 1;
  __shared__ double sx[TILE], sy[TILE], sz[TILE];
  __shared__ R sq[TILE], sqi[TILE];
  const int lane = threadIdx.x;
  const int ti = blockIdx.x * TILE + lane;
  const bool act = ti < nt;
  double tx = 0, ty = 0, tz = 0;
  if (act) { tx = trg[3 * size_t(ti)]; ty = trg[3 * size_t(ti) + 1]; tz = trg[3 * size_t(ti) + 2]; }
  const int sbeg = blockIdx.y * chunk;
  const int send = min(ns, sbeg + chunk);
  const R kr = R(wk.re), ki = R(wk.im);
  R acc[NA], comp[NA];
#pragma unroll
  for (int a = 0; a < NA; a++) { acc[a] = 0; comp[a] = 0; }
  for (int s0 = sbeg; s0 < send; s0 += TILE) {
    const int m = min(TILE, send - s0);
    __syncthreads();
    if (lane < m) {
      const size_t si = size_t(s0 + lane);
      sx[lane] = src[3 * si];
      sy[lane] = src[3 * si + 1];
      sz[lane] = src[3 * si + 2];
      sq[lane] = R(q[si * vw]);
      if (C) sqi[lane] = R(q[si * vw + 1]);
    }
    __syncthreads();
    R part[NA];
#pragma unroll
    for (int a = 0; a < NA; a++) part[a] = 0;
    for (int j = 0; j < m; j++) {
      const R dx = R(sx[j] - tx), dy = R(sy[j] - ty), dz = R(sz[j] - tz);
      if (GRAD) pair_grad<KIND, R, RSQ_LIB>(dx, dy, dz, sq[j], C ? sqi[j] : R(0), kr, ki, part);
      else pair_pot<KIND, R, RSQ_LIB>(dx, dy, dz, sq[j], C ? sqi[j] : R(0), kr, ki, part);
    }
#pragma unroll
    for (int a = 0; a < NA; a++) kahan_add(acc[a], comp[a], part[a]);
  }
  if (act) {
    double* o = partial + (size_t(blockIdx.y) * nt + ti) * NA;
#pragma unroll
    for (int a = 0; a < NA; a++) o[a] = double(acc[a]) - double(comp[a]);
  }
}

__global__ void k_direct_reduce(const double* __restrict__ partial, int nsplit, int nt, int na,
                                double* __restrict__ out) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= size_t(nt) * na) return;
  double s = 0, c = 0;
  for (int k = 0; k < nsplit; k++) kahan_add(s, c, partial[size_t(k) * nt * na + i]);
  out[i] += (s - c) * FOUR_PI_INV;
}

// ------------------------------------------------- near-coincident pairs
//
// The FP32 near field forms a pair's difference vector from coordinates
// relative to leaf centres, each rounded to FP32: an absolute error of about
// 2^-24 of the leaf size per coordinate, so a relative error of about
// 2^-24 L / r in 1/r (and twice that in the gradient) for a pair at
// distance r.  Only pairs much closer than the leaf size are hurt, and they
// are rare: they are listed once per tree (k_close_find, FP64 distances) and
// after every FP32 near field k_close_fix replaces each one's FP32
// contribution, recomputed from the very operands the near-field kernel used,
// by its FP64 value.
__global__ __launch_bounds__(64) void k_close_find(DevTree t, const int* __restrict__ work, int* __restrict__ out,
                                                   int cap, int* __restrict__ count) {
  const int leaf = work[blockIdx.x];
  const int tb = t.trg_begin[leaf], nt = t.trg_count[leaf];
  const double side = 2.0 * t.r0 * ldexp(1.0, -t.level[leaf]);
  // (side / 16)^2 with a margin, so that every pair the FP32 near field
  // leaves out (FP32 r^2 <= (side / 16)^2, close_rmin2) is listed
  const double d2 = side * side * (1.002 / 256.0);
  const int g0 = t.p2p_off[leaf], g1 = t.p2p_off[leaf + 1];
  for (int i = threadIdx.x; i < nt; i += blockDim.x) {
    const double* x = t.trg + 3 * size_t(tb + i);
    const double x0 = x[0], x1 = x[1], x2 = x[2];
    for (int g = g0; g < g1; g++) {
      const int sn = t.p2p_src[g], sb = t.src_begin[sn], ns = t.src_count[sn];
      for (int j = 0; j < ns; j++) {
        const double* y = t.src + 3 * size_t(sb + j);
        const double dx = y[0] - x0, dy = y[1] - x1, dz = y[2] - x2;
        const double r2 = dx * dx + dy * dy + dz * dz;
        if (r2 < d2 && r2 > 0.0) {
          const int k = atomicAdd(count, 1);
          if (k < cap) {
            int* o = out + 4 * size_t(k);
            o[0] = tb + i;
            o[1] = sb + j;
            o[2] = leaf;
            o[3] = sn;
          }
        }
      }
    }
  }
}

void launch_close_find(const DevTree& t, const int* work, int nwork, int* out, int cap, int* count, hipStream_t s) {
  if (nwork <= 0) return;
  hipLaunchKernelGGL(k_close_find, dim3(nwork), dim3(64), 0, s, t, work, out, cap, count);
}

// The correction of each listed pair per unit charge, once per tree: one
// thread per pair, coef[k][a] = FP64 minus FP32 value of the pair with q = 1
// (real kernels: a = potential, gradient; Helmholtz: their (re, im) parts).
// The FP32 operands are formed as the near-field kernel forms them: source and
// target relative to the target leaf's centre, each rounded once.  A pair is
// linear in its charge, so per evaluation its correction is q coef (complex
// product for Helmholtz); the FP32 value of a charged pair differs from q
// times that of a unit charge by the rounding of the products, ~1e-7 of the
// pair's value.
template <int KIND>
__global__ __launch_bounds__(256) void k_close_coef(DevTree t, Wavek wk, int npairs, double* __restrict__ coef) {
  constexpr bool C = kcplx<KIND>();
  constexpr int NA = C ? 8 : 4;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= npairs) return;
  const int* cp = t.close + 4 * size_t(k);
  const int it = cp[0], is = cp[1], tl = cp[2], sl = cp[3];
  const double cx = t.center[3 * tl], cy = t.center[3 * tl + 1], cz = t.center[3 * tl + 2];
  const double* x = t.trg + 3 * size_t(it);
  const double* y = t.src + 3 * size_t(is);
  const float tx = float(x[0] - cx), ty = float(x[1] - cy), tz = float(x[2] - cz);
  const float kr = float(wk.re), ki = float(wk.im);
  float a32[NA];
  double a64[NA];
#pragma unroll
  for (int a = 0; a < NA; a++) {
    a32[a] = 0.f;
    a64[a] = 0.0;
  }
  const float dx = float(y[0] - cx) - tx, dy = float(y[1] - cy) - ty, dz = float(y[2] - cz) - tz;
  // a leaf with itself: the near-field kernel left out the pairs with FP32
  // r^2 <= rmin2 (their FP32 value is 0 here too)
  if (tl == sl) pair_grad<KIND, float, RSQ_MASK>(dx, dy, dz, 1.f, 0.f, kr, ki, a32, close_rmin2<float>(t, tl));
  else pair_grad<KIND, float, RSQ_SOFT>(dx, dy, dz, 1.f, 0.f, kr, ki, a32, soft_r2<float>(t, tl));
  pair_grad<KIND, double, RSQ_MASK>(y[0] - x[0], y[1] - x[1], y[2] - x[2], 1.0, 0.0, wk.re, wk.im, a64);
#pragma unroll
  for (int a = 0; a < NA; a++) coef[size_t(k) * NA + a] = a64[a] - double(a32[a]);
}

void launch_close_coef(int kind, const DevTree& t, Wavek k, int npairs, double* coef, hipStream_t s) {
  if (npairs <= 0) return;
  const dim3 g((npairs + 255) / 256), b(256);
  if (kind == LAPLACE) hipLaunchKernelGGL(k_close_coef<LAPLACE>, g, b, 0, s, t, k, npairs, coef);
  else if (kind == YUKAWA) hipLaunchKernelGGL(k_close_coef<YUKAWA>, g, b, 0, s, t, k, npairs, coef);
  else hipLaunchKernelGGL(k_close_coef<HELMHOLTZ>, g, b, 0, s, t, k, npairs, coef);
}

// One thread per target with listed pairs, its pairs in list order (so the
// result does not depend on scheduling): trg_value += sum of q_s coef / 4 pi.
template <int KIND>
__global__ __launch_bounds__(256) void k_close_fix(DevTree t) {
  constexpr bool C = kcplx<KIND>();
  constexpr int NA = C ? 8 : 4;
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= t.nclose) return;
  double fix[NA];
#pragma unroll
  for (int a = 0; a < NA; a++) fix[a] = 0.0;
  const int k0 = t.close_off[u], k1 = t.close_off[u + 1];
  for (int k = k0; k < k1; k++) {
    const int is = t.close[4 * size_t(k) + 1];
    const double* cf = t.close_coef + size_t(k) * NA;
    const double qr = t.q[size_t(is) * t.vw];
    if constexpr (C) {
      const double qi = t.q[size_t(is) * t.vw + 1];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        fix[2 * c] += qr * cf[2 * c] - qi * cf[2 * c + 1];
        fix[2 * c + 1] += qr * cf[2 * c + 1] + qi * cf[2 * c];
      }
    } else {
#pragma unroll
      for (int a = 0; a < NA; a++) fix[a] += qr * cf[a];
    }
  }
  double* o = t.trg_value + size_t(t.close[4 * size_t(k0)]) * 4 * t.vw;
#pragma unroll
  for (int a = 0; a < NA; a++) o[a] += fix[a] * FOUR_PI_INV;
}

// ---------------------------------------------------------------- launchers

// Points and surfaces of a tree are within 6 r0 of each other in a coordinate.
static bool real_phases(Wavek k, const DevTree& t) {
  return k.im == 0.0 && std::fabs(k.re) * 16.0 * t.r0 < 1073741824.0;
}

// Waves per tile: doubled up to 4 while the tiles times waves are fewer than 4096
// (Helmholtz, whose pairs cost more: 16384).  Near field with 1, 2, 4 waves, us:
//   Laplace FP64, 64 tiles of 47 targets 80, 45, 28 (8 and 16 waves: 26, 27, the same
//     evaluation); 519 tiles of 46 85, 71, 43 (42, 59); FP32 75, 47, 32 (31, 49);
//     64 tiles of 16: 4, 8, 16 waves 12, 14, 20;
//   Yukawa FP64, 1015 tiles of 20 157, 83, 56; 3570 of 17 143, 101, 86;
//   Helmholtz FP64, 64 tiles of 47 251, 134, 70; 623 of 59 324, 284, 205; 4161 of 49
//     960, 857, 779; FP32, 4161 of 49 390, 314, 277.
// Above the line more waves only take slots from the transforms beside the near
// field.  The evaluation with 1, 2, 4 waves: Laplace, 4551 tiles, FP64 709, 713, 746
// (FP32 478, 476, 453), 32768 tiles, FP32 1027, 1050, 1110; Yukawa, 15074 tiles, FP32
// 1226, 1239, 1248; Helmholtz, 4161 tiles, FP64 1473, 1416, 1375, FP32 720, 680, 663,
// 32891 tiles, FP32 2668, 2636, 2716.
template <int KIND>
static int particle_waves(int ntiles) {
  int w = 1;
  while (w < 4 && ntiles * w < (kcplx<KIND>() ? 16384 : 4096)) w *= 2;
  return w;
}

template <int KIND, typename R>
static void eval_targets_t(int mode, const DevTree& t, Wavek k, const int* tiles, int ntiles, hipStream_t s) {
  if (ntiles <= 0) return;
  auto go = [&](auto W) {
    constexpr int w = decltype(W)::value;
    const dim3 g(ntiles), b(64 * w);
    if (mode == MODE_P2P) hipLaunchKernelGGL((k_p2p<KIND, R, w>), g, b, 0, s, t, k, tiles);
    else if (mode == MODE_M2P) hipLaunchKernelGGL((k_m2p<KIND, R, 4>), g, dim3(256), 0, s, t, k, tiles);
    else hipLaunchKernelGGL((k_l2p_smem<KIND, R, w>), g, b, 0, s, t, k, tiles);
  };
  // the near field of few tiles: 8 waves in FP64 Helmholtz without the library's
  // sincos (4 and 8 waves: 64 tiles 70 and 63 us, 623 tiles 205 and 178, 1869 tiles 207 and
  // 201, 4161 tiles 779 and 793), else the 4 that particle_waves gives below 1024
  constexpr int FEW = KIND == HELMHOLTZ_REAL && sizeof(R) == 8 ? 8 : 4;
  // t.p2p_split = 0: nothing is split over lanes, of one wave or of several
  const bool whole = t.p2p_split == 0 && mode != MODE_M2P;
  const int w = whole ? 1 : particle_waves<KIND>(ntiles);
  if (whole && mode == MODE_P2P) {
    hipLaunchKernelGGL((k_p2p<KIND, R, 1, 1>), dim3(ntiles), dim3(64), 0, s, t, k, tiles);
  } else if (mode == MODE_P2P && ntiles < 1024) {
    hipLaunchKernelGGL((k_p2p<KIND, R, FEW>), dim3(ntiles), dim3(64 * FEW), 0, s, t, k, tiles);
  } else if (w == 1) go(std::integral_constant<int, 1>());
  else if (w == 2) go(std::integral_constant<int, 2>());
  else go(std::integral_constant<int, 4>());
  // FP32 near field: the near-coincident pairs in FP64 (same stream, after it)
  if constexpr (sizeof(R) == 4) {
    if (mode == MODE_P2P && t.nclose > 0 && t.close && t.close_off && t.close_coef)
      hipLaunchKernelGGL(k_close_fix<KIND == HELMHOLTZ_REAL ? int(HELMHOLTZ) : KIND>, dim3((t.nclose + 255) / 256),
                         dim3(256), 0, s, t);
  }
}

void launch_eval_targets(int kind, bool f32, int mode, const DevTree& t, Wavek k, const int* tiles, int ntiles,
                         hipStream_t s) {
  switch (kind) {
    case LAPLACE: f32 ? eval_targets_t<LAPLACE, float>(mode, t, k, tiles, ntiles, s)
                      : eval_targets_t<LAPLACE, double>(mode, t, k, tiles, ntiles, s); break;
    case YUKAWA: f32 ? eval_targets_t<YUKAWA, float>(mode, t, k, tiles, ntiles, s)
                     : eval_targets_t<YUKAWA, double>(mode, t, k, tiles, ntiles, s); break;
    default:
      if (real_phases(k, t)) f32 ? eval_targets_t<HELMHOLTZ_REAL, float>(mode, t, k, tiles, ntiles, s)
                           : eval_targets_t<HELMHOLTZ_REAL, double>(mode, t, k, tiles, ntiles, s);
      else f32 ? eval_targets_t<HELMHOLTZ, float>(mode, t, k, tiles, ntiles, s)
               : eval_targets_t<HELMHOLTZ, double>(mode, t, k, tiles, ntiles, s);
      break;
  }
}

template <int KIND, typename R>
static void eval_surface_t(int mode, const DevTree& t, Wavek k, const int* work, int nwork, double* check,
                           hipStream_t s) {
  if (nwork <= 0) return;
  // the surface's chunks of 64 points over several waves while the nodes do not
  // fill the chip (Helmholtz FP64 P2M of 512 leaves 67 -> 37 us, Laplace P2L of
  // 2106 nodes 92 -> 40)
  const int nchunk = (t.nsurf + TILE - 1) / TILE;
  const dim3 g(nwork, std::max(1, std::min(nchunk, 16384 / nwork)));
  if (mode == MODE_P2M) hipLaunchKernelGGL((k_eval_surface<KIND, R, MODE_P2M>), g, dim3(64), 0, s, t, k, work, check);
  else hipLaunchKernelGGL((k_eval_surface<KIND, R, MODE_P2L>), g, dim3(64), 0, s, t, k, work, check);
}

void launch_eval_surface(int kind, bool f32, int mode, const DevTree& t, Wavek k, const int* work, int nwork,
                         double* check, hipStream_t s) {
  switch (kind) {
    case LAPLACE: f32 ? eval_surface_t<LAPLACE, float>(mode, t, k, work, nwork, check, s)
                      : eval_surface_t<LAPLACE, double>(mode, t, k, work, nwork, check, s); break;
    case YUKAWA: f32 ? eval_surface_t<YUKAWA, float>(mode, t, k, work, nwork, check, s)
                     : eval_surface_t<YUKAWA, double>(mode, t, k, work, nwork, check, s); break;
    default:
      if (real_phases(k, t)) f32 ? eval_surface_t<HELMHOLTZ_REAL, float>(mode, t, k, work, nwork, check, s)
                           : eval_surface_t<HELMHOLTZ_REAL, double>(mode, t, k, work, nwork, check, s);
      else f32 ? eval_surface_t<HELMHOLTZ, float>(mode, t, k, work, nwork, check, s)
               : eval_surface_t<HELMHOLTZ, double>(mode, t, k, work, nwork, check, s);
      break;
  }
}

template <int KIND, typename R>
static void direct_t(Wavek k, const double* src, const double* q, int ns, const double* trg, int nt, double* out,
                     int gradient, double* scratch, int nsplit, hipStream_t s) {
  const int na = (gradient ? 4 : 1) * (KIND == HELMHOLTZ ? 2 : 1);
  int chunk = (ns + nsplit - 1) / nsplit;
  chunk = ((chunk + TILE - 1) / TILE) * TILE;
  if (chunk == 0) chunk = TILE;
  dim3 grid((nt + TILE - 1) / TILE, nsplit);
  if (gradient) hipLaunchKernelGGL((k_direct<KIND, R, true>), grid, dim3(64), 0, s, src, q, ns, trg, nt, scratch, chunk, k);
  else hipLaunchKernelGGL((k_direct<KIND, R, false>), grid, dim3(64), 0, s, src, q, ns, trg, nt, scratch, chunk, k);
  const size_t n = size_t(nt) * na;
  hipLaunchKernelGGL(k_direct_reduce, dim3((n + 255) / 256), dim3(256), 0, s, scratch, nsplit, nt, na, out);
}

void launch_direct(int kind, bool mixed, bool cplx, Wavek k, const double* src, const double* q, int ns,
                   const double* trg, int nt, double* out, int gradient, double* scratch, int nsplit,
                   hipStream_t s) {
  (void)cplx;
  if (nt <= 0) return;
  switch (kind) {
    case LAPLACE: mixed ? direct_t<LAPLACE, float>(k, src, q, ns, trg, nt, out, gradient, scratch, nsplit, s)
                        : direct_t<LAPLACE, double>(k, src, q, ns, trg, nt, out, gradient, scratch, nsplit, s); break;
    case YUKAWA: mixed ? direct_t<YUKAWA, float>(k, src, q, ns, trg, nt, out, gradient, scratch, nsplit, s)
                       : direct_t<YUKAWA, double>(k, src, q, ns, trg, nt, out, gradient, scratch, nsplit, s); break;
    default: mixed ? direct_t<HELMHOLTZ, float>(k, src, q, ns, trg, nt, out, gradient, scratch, nsplit, s)
                   : direct_t<HELMHOLTZ, double>(k, src, q, ns, trg, nt, out, gradient, scratch, nsplit, s); break;
  }
}

}  // namespace xfmm
