"""The work that users of this framework have it do, as cases that can be timed and compared.

A case is a dict of plain values; `prepare` makes what the user's program has in hand before the call (points,
charges, the tree and operators on the device), `run` is one pass through the public entry points, `exact` the
same answer by direct summation in 64 bits with plain torch, `work` what a pass cannot do without.

Three kinds of program are covered:
  "engine"   an iterative solver or time stepper that keeps its tree: every pass brings new charges, in the user's
             own order, in device memory, and takes potential and gradient back in the user's order (exafmm.abi on
             device pointers; "nprob" > 1: exafmm.batch.LaplaceBatch, many problems as one forest).  Programs that
             choose the mixed or FLOAT path are single-precision programs: they keep the answer as 32-bit values;
             FP64 programs take the values as the engine holds them.
  "adjoint"  a gradient computation on host arrays: forward evaluation and adjoint pass on one tree
             (exafmm.adjoint.AdjointFmm), which returns phi, dL/dq and dL/dy.
  "direct"   the direct sum on device pointers (xfmm_direct_noalloc): checks of sampled targets, small problems.

All points lie in a box that every seed shares (two of its corners, or the poles of the sphere, are among the
points), so that a program that builds many trees, as this file does, computes an operator set once.
"""
import ctypes
import math
import os
import sys
import tempfile

import numpy as np
import torch  # before exafmm: the engine then shares torch's HIP runtime

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "exafmm-t_amd"))

import exafmm  # noqa: E402
from exafmm import abi  # noqa: E402
from exafmm.adjoint import AdjointFmm  # noqa: E402
from exafmm.batch import LaplaceBatch  # noqa: E402

KERNEL = {"laplace": abi.LAPLACE, "helmholtz": abi.HELMHOLTZ, "modified_helmholtz": abi.MODIFIED_HELMHOLTZ}
PRECISION = {"fp64": abi.FP64, "mixed": abi.MIXED, "float": abi.FLOAT}

_dir = tempfile.mkdtemp(prefix="fmm_cases_")
_operators = {}  # operator sets by kernel, order, wave number, precision, box and depth


def _case(kind, kernel, n, p=8, ncrit=64, precision="fp64", wavek=0.0, dist="cube", charges="uniform", ntrg=0,
          graph=False, nprob=1, name=None):
    c = {"kind": kind, "kernel": kernel, "n": n, "ntrg": ntrg, "p": p, "ncrit": ncrit, "precision": precision,
         "wavek": wavek, "dist": dist, "charges": charges, "graph": graph, "nprob": nprob}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the check of a solution at sampled targets: 1,000 targets against all sources (potential and gradient)
        _case("direct", "laplace", 10_000, ntrg=1_000, name="direct_laplace_1k_x_10k"),
        # a small molecule or a test problem inside an iteration: two levels, every launch is short
        _case("engine", "laplace", 3_001, p=6, ncrit=64, name="laplace_3k_p6_fp64"),
        # the middle size at the benchmark's small configuration: masses (charges of one sign), mixed precision
        _case("engine", "laplace", 100_000, p=8, ncrit=64, precision="mixed", charges="u01",
              name="laplace_100k_p8_mixed"),
        # probes that are not the sources, ragged numbers of both, double precision
        _case("engine", "laplace", 60_001, ntrg=100_003, p=8, ncrit=100, name="laplace_60k_to_100k_p8_fp64"),
        # low order at a million points, as the published timings at P = 4, in the FLOAT mode
        _case("engine", "laplace", 1_000_000, p=4, ncrit=64, precision="float", name="laplace_1m_p4_float"),
        # the headline configuration: replays of the captured evaluation
        _case("engine", "laplace", 2_000_000, p=10, ncrit=128, precision="mixed", graph=True,
              name="laplace_2m_p10_mixed"),
        # high accuracy in double precision
        _case("engine", "laplace", 500_000, p=10, ncrit=128, graph=True, name="laplace_500k_p10_fp64"),
        # boundary integrals on a surface: an adaptive tree with M2P and P2L lists, screened kernel
        _case("engine", "modified_helmholtz", 300_000, p=8, ncrit=64, precision="mixed", wavek=5.0, dist="sphere",
              charges="normal", name="yukawa_sphere_300k_p8_mixed"),
        # scattering: complex charges, mixed precision
        _case("engine", "helmholtz", 200_000, p=8, ncrit=128, precision="mixed", wavek=20.0,
              name="helmholtz_200k_p8_mixed"),
        # scattering in double precision, small
        _case("engine", "helmholtz", 30_011, p=6, ncrit=100, wavek=10.0, name="helmholtz_30k_p6_fp64"),
        # many independent star clusters (strongly adaptive trees) as one forest
        _case("engine", "laplace", 30_000, p=8, ncrit=64, precision="mixed", dist="plummer", charges="mass", nprob=16,
              graph=True, name="batch_16_plummer_p8_mixed"),
        # derivatives of a screened potential with respect to charges and positions, on host arrays
        _case("adjoint", "modified_helmholtz", 20_000, p=6, ncrit=64, wavek=5.0, dist="sphere", charges="normal",
              name="adjoint_yukawa_sphere_20k_p6_fp64"),
    ]


def _spread(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    most = max(work(c)["flops"] for c in listed())
    while True:
        x = rng.random()
        if x < 0.1:
            kernel = rng.choice(["laplace", "laplace", "modified_helmholtz", "helmholtz"])
            c = _case("direct", kernel, _spread(rng, 1_000, 40_000), ntrg=_spread(rng, 100, 10_000),
                      precision=rng.choice(["fp64", "fp64", "mixed"]),
                      wavek=0.0 if kernel == "laplace" else rng.choice([1.0, 5.0, 10.0]))
        elif x < 0.2:
            kernel = rng.choice(["laplace", "modified_helmholtz"])
            c = _case("adjoint", kernel, _spread(rng, 1_000, 40_000), p=rng.randint(4, 7), ncrit=_spread(rng, 40, 200),
                      wavek=0.0 if kernel == "laplace" else 5.0, dist=rng.choice(["cube", "sphere"]), charges="normal")
        elif x < 0.3:
            c = _case("engine", "laplace", _spread(rng, 3_000, 60_000), p=rng.randint(4, 9), ncrit=_spread(rng, 40, 150),
                      precision=rng.choice(["fp64", "mixed", "float"]), dist=rng.choice(["cube", "plummer"]),
                      charges=rng.choice(["uniform", "mass"]), nprob=rng.randint(2, 12), graph=rng.random() < 0.7)
        else:
            kernel = rng.choice(["laplace", "laplace", "laplace", "modified_helmholtz", "helmholtz"])
            small = kernel == "helmholtz"
            n = _spread(rng, 1_000, 100_000 if small else 800_000)
            dist = rng.choice(["cube", "cube", "sphere"] + ([] if small else ["plummer"]))
            c = _case("engine", kernel, n, p=rng.randint(5 if small else 4, 7 if small else 8 if kernel != "laplace" else 10),
                      ncrit=_spread(rng, 40, 250), precision=rng.choice(["fp64", "mixed", "mixed", "float"]),
                      wavek=0.0 if kernel == "laplace" else 1.0 if dist == "plummer" else rng.choice([1.0, 5.0, 10.0]),
                      dist=dist,
                      charges=rng.choice(["uniform", "uniform", "normal", "u01"]),
                      ntrg=_spread(rng, n / 4, n) if rng.random() < 0.25 else 0, graph=rng.random() < 0.4)
        if work(c)["flops"] <= 0.9 * most:
            return c


def _points(dist, n, rng):
    if dist == "cube":
        x = rng.random((n, 3))
        x[0], x[-1] = 0.0, 1.0
    elif dist == "sphere":
        x = rng.normal(size=(n, 3))
        x /= np.linalg.norm(x, axis=1)[:, None]
        x[0], x[-1] = (1.0, 0.0, 0.0), (-1.0, 0.0, 0.0)
    else:  # a Plummer sphere of scale radius 1, cut at radius 10
        r = np.minimum(1.0 / np.sqrt((rng.random(n) * 0.999) ** (-2.0 / 3.0) - 1.0), 10.0)
        v = rng.normal(size=(n, 3))
        x = v / np.linalg.norm(v, axis=1)[:, None] * r[:, None]
        x[0], x[-1] = (10.0, 0.0, 0.0), (-10.0, 0.0, 0.0)
    return x


def _inputs(case, seed):
    """[(sources, charges, targets), ...] in the user's order; targets is sources for the N-body cases."""
    rng = np.random.default_rng([seed, case["n"]])
    out = []
    for i in range(case["nprob"]):
        # the problems of a batch: sizes spread around n
        n = case["n"] if case["nprob"] == 1 else max(16, int(case["n"] * 4.0 ** (((37 * i) % 16) / 8.0 - 1.0)))
        x = _points(case["dist"], n, rng)
        kind = case["charges"]
        draw_q = {"uniform": lambda: rng.uniform(-1.0, 1.0, n), "normal": lambda: rng.normal(size=n),
                  "u01": lambda: rng.random(n), "mass": lambda: rng.uniform(0.5, 1.5, n) / n}[kind]
        q = draw_q() + 1j * draw_q() if case["kernel"] == "helmholtz" else draw_q()
        out.append((x, q, _points(case["dist"], case["ntrg"], rng) if case["ntrg"] else x))
    return out


def _fmm(case):
    mod, name = getattr(exafmm, case["kernel"]), os.path.join(_dir, "operators.dat")
    if case["kernel"] == "laplace":
        fmm = mod.LaplaceFmm(case["p"], case["ncrit"], name)
    elif case["kernel"] == "helmholtz":
        fmm = mod.HelmholtzFmm(case["p"], case["ncrit"], complex(case["wavek"]), name)
    else:
        fmm = mod.ModifiedHelmholtzFmm(case["p"], case["ncrit"], case["wavek"], name)
    fmm.precision = PRECISION[case["precision"]]
    return mod, fmm


class _Device:
    """Device memory of the engine, for torch.as_tensor."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f8", "version": 2}


def _prepare_engine(case, seed):
    probs = _inputs(case, seed)
    if case["nprob"] > 1:
        batch = LaplaceBatch(probs, case["p"], case["ncrit"], PRECISION[case["precision"]],
                             os.path.join(_dir, "batch.dat"), graph=case["graph"])
        eng, forest = batch.engine, batch.forest
        passes = [batch.run]
        src = np.concatenate([np.asarray(b) + forest.soff[i] for i, b in enumerate(forest.src_ibody)])
        trg = np.concatenate([np.asarray(b) + forest.toff[i] for i, b in enumerate(forest.trg_ibody)])
        keep = batch
    else:
        x, q, t = probs[0]
        mod, fmm = _fmm(case)
        tree = mod.setup(mod.init_sources(x, q), mod.init_targets(t), fmm, precompute=False)
        flat = fmm.flat_tree(tree)
        key = (case["kernel"], case["p"], case["wavek"], case["precision"], fmm.r0, 0 if case["kernel"] == "laplace" else fmm.depth)
        if key not in _operators:
            fmm.precompute()
            _operators[key] = fmm.operators()
            if os.path.exists(fmm.filename):  # operators of another box or wave number may follow
                os.remove(fmm.filename)
        eng = abi.Engine(KERNEL[case["kernel"]], case["p"], case["wavek"], PRECISION[case["precision"]])
        eng.set_operators(_operators[key])
        eng.set_tree(flat)
        src, trg = np.asarray(flat["src_ibody"]), np.asarray(flat["trg_ibody"])
        if case["graph"]:
            eng.set_charges(q[src])
            eng.graph_capture()
            passes = [eng.graph_launch]
        else:
            passes = [eng.upward_pass, eng.downward_pass]
        keep = (fmm, tree)
    q = torch.from_numpy(np.concatenate([p[1] for p in probs])).cuda()
    width = 8 if case["kernel"] == "helmholtz" else 4
    values = torch.as_tensor(_Device(eng.values_device_ptr(), (len(trg), width)), device="cuda")
    return {"engine": eng, "passes": passes, "q": q, "src": torch.from_numpy(src.astype(np.int64)).cuda(),
            "trg": torch.from_numpy(trg.astype(np.int64)).cuda(), "values": values, "keep": keep, "single": case["precision"] != "fp64",
            "complex": width == 8}


def _run_engine(s):
    q = s["q"].index_select(0, s["src"])  # the user's order -> the tree's
    torch.cuda.current_stream().synchronize()  # the engine has streams of its own
    s["engine"].set_charges_device(q.data_ptr())
    for step in s["passes"]:
        step()
    s["engine"].synchronize()
    v = s["values"].float() if s["single"] else s["values"]
    v = torch.empty_like(v).index_copy_(0, s["trg"], v)  # the tree's order -> the user's
    return torch.view_as_complex(v.view(-1, 4, 2)) if s["complex"] else v


def _prepare_adjoint(case, seed):
    (x, q, t), = _inputs(case, seed)
    w = np.random.default_rng([seed, 5]).normal(size=len(t))
    a = AdjointFmm(case["kernel"], x, t, case["p"], case["ncrit"], case["wavek"], PRECISION[case["precision"]])
    return {"fmm": a, "q": q, "w": w}


def _run_adjoint(s):
    phi = s["fmm"](s["q"])
    dq, dy = s["fmm"].backward(s["w"])
    return phi, dq, dy


def _prepare_direct(case, seed):
    (x, q, _), = _inputs(dict(case, ntrg=0), seed)
    cplx = case["kernel"] == "helmholtz"
    t = np.random.default_rng([seed, 7]).choice(len(x), min(case["ntrg"], len(x)), replace=False)
    x, q = torch.from_numpy(x).cuda(), torch.from_numpy(q).cuda()
    f = abi.load().xfmm_direct_noalloc
    p, i, d = ctypes.c_void_p, ctypes.c_int, ctypes.c_double
    f.argtypes, f.restype = [i, i, d, d, p, p, i, p, i, p, i, p], i
    return {"call": f, "x": x, "q": q, "t": x[torch.from_numpy(t).cuda()].contiguous(), "wavek": case["wavek"],
            "kernel": KERNEL[case["kernel"]], "precision": PRECISION[case["precision"]],
            "dtype": torch.complex128 if cplx else torch.float64, "single": case["precision"] != "fp64"}


def _run_direct(s):
    out = torch.zeros((len(s["t"]), 4), dtype=s["dtype"], device="cuda")
    rc = s["call"](s["kernel"], s["precision"], s["wavek"], 0.0, s["x"].data_ptr(), s["q"].data_ptr(), len(s["x"]),
                   s["t"].data_ptr(), len(s["t"]), out.data_ptr(), 1, torch.cuda.current_stream().cuda_stream)
    if rc != 0:
        raise RuntimeError("xfmm_direct_noalloc: status %d" % rc)
    if s["single"]:
        out = out.to(torch.complex64 if out.is_complex() else torch.float32)
    return out


def prepare(case, seed):
    make = {"engine": _prepare_engine, "adjoint": _prepare_adjoint, "direct": _prepare_direct}[case["kind"]]
    return dict(make(case, seed), kind=case["kind"])


def run(state):
    return {"engine": _run_engine, "adjoint": _run_adjoint, "direct": _run_direct}[state["kind"]](state)


def _sum(kernel, k, y, q, x):
    """Potential and gradient (len(x), 4) at x of the charges q at y, in 64 bits; coinciding points leave each other out."""
    q = q.to(torch.complex128 if kernel == "helmholtz" else torch.float64)
    out = torch.empty((len(x), 4), dtype=q.dtype, device=x.device)
    step = max(1, 60_000_000 // len(y))
    for i in range(0, len(x), step):
        t = x[i:i + step]
        d = [y[None, :, a] - t[:, None, a] for a in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        inv = torch.where(r2 > 0, r2.rsqrt(), torch.zeros_like(r2))
        if kernel == "laplace":
            g = inv
            s = inv * inv * inv
        elif kernel == "modified_helmholtz":
            kr = k * (r2 * inv)
            g = torch.exp(-kr) * inv
            s = g * (1.0 + kr) * inv * inv
        else:
            g = torch.polar(inv, k * (r2 * inv))
            s = g * torch.complex(inv * inv, -k * inv)
        out[i:i + step, 0] = g @ q
        for a in range(3):
            out[i:i + step, 1 + a] = (d[a] * s) @ q
        del d, r2, inv, g, s
    return out / (4.0 * math.pi)


def exact(case, seed):
    if work(case)["pairs"] > 1.0e11:
        return None
    cuda = [tuple(torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in p) for p in _inputs(dict(case, ntrg=0) if case["kind"] == "direct" else case, seed)]
    k = case["wavek"]
    if case["kind"] == "direct":
        (y, q, x), = cuda
        t = np.random.default_rng([seed, 7]).choice(len(x), min(case["ntrg"], len(x)), replace=False)
        return _sum(case["kernel"], k, y, q, x[torch.from_numpy(t).cuda()])
    if case["kind"] == "adjoint":
        (y, q, x), = cuda
        w = torch.from_numpy(np.random.default_rng([seed, 5]).normal(size=len(x))).cuda()
        back = _sum(case["kernel"], k, x, w, y)
        return [_sum(case["kernel"], k, y, q, x).cpu().numpy(), back[:, 0].cpu().numpy(), (q[:, None] * back[:, 1:]).cpu().numpy()]
    return torch.cat([_sum(case["kernel"], k, y, q, x) for y, q, x in cuda])


def work(case):
    """Bytes: positions and charges in, values out, once.  Flops: a direct sum's pairs, or an estimate of what the
    fast multipole method sums at this order and leaf size: near pairs, the Hadamard products of the M2L (512 a pair
    of parents and frequency), the translations and the surface evaluations."""
    n = case["n"] * case["nprob"]
    nt = case["ntrg"] or n
    v = 2 if case["kernel"] == "helmholtz" else 1
    size = n * (24 + 8 * v) + nt * (24 + 32 * v)
    per_pair = 20 if case["kernel"] == "laplace" else 30 if v == 1 else 50
    pairs = float(n) * nt / case["nprob"]
    if case["kind"] == "direct":
        return {"bytes": size, "flops": pairs * per_pair, "pairs": pairs}
    p, total = case["p"], max(n, nt)
    surf, freq = 6 * (p - 1) ** 2 + 2, (2 * p) ** 2 * (2 * p if v == 2 else p + 1)
    if case["dist"] == "cube":
        depth = max(1, math.ceil(math.log(max(8.0, total / case["nprob"] / case["ncrit"]), 8) - 0.05))
        leaves = min(float(total), case["nprob"] * 8.0 ** depth)
        near = 27.0
    else:
        leaves, near = max(8.0, 2.5 * total / case["ncrit"]), 16.0
    parents = leaves / 7.0
    near_pairs = min(pairs, n / leaves * nt * near)
    far = 24.0 * parents * freq * 512 + 2 * 16.0 * parents * (surf * v) ** 2 + 8.0 * leaves * (surf * v) ** 2 * 0.7
    flops = near_pairs * per_pair + far + (12.0 * n + 20.0 * nt) * surf * v
    times = 2 if case["kind"] == "adjoint" else 1
    return {"bytes": times * size, "flops": times * flops, "pairs": pairs * times}
