"""The translation GEMMs against plain FP64 products with the same operators: M2M, L2L and the pseudo-inverse solve of
L2P, on levels of 1 to 32768 rows (every tile shape and K split), K and N off the multiples of the tiles, several
levels in one launch, real and complex operators, FP64 and the FP32 stages of the FLOAT mode.

Every entry is held within (K + 8) u of the sum of the products' absolute values, u = 2^-53 or 2^-24: the bound of a
sum of K products in any order, with operands rounded once."""
import numpy as np
import pytest

from exafmm import abi
from fmm_cases import make_problem

pytestmark = pytest.mark.gpu

CASES = [  # kernel, p, n, ncrit, dist, depth (None: adaptive), precision
    ("laplace", 5, 33000, 64, "cube", 5, abi.FP64),
    ("laplace", 10, 33000, 64, "cube", 5, abi.FLOAT),
    ("laplace", 6, 6000, 64, "cube", 4, abi.FLOAT),
    ("laplace", 2, 3000, 30, "clusters", None, abi.FP64),
    ("modified_helmholtz", 3, 9000, 20, "clusters", None, abi.FP64),
    ("helmholtz", 4, 2000, 64, "cube", 3, abi.FP64),
    ("helmholtz", 5, 4000, 64, "sphere", None, abi.FLOAT),
]


@pytest.fixture(scope="module", params=CASES, ids=lambda c: "%s-p%d-%s-%d" % (c[0], c[1], c[4], c[6]))
def problem(request, require_gpu):
    kernel, p, n, ncrit, dist, depth, precision = request.param
    pr = make_problem(kernel, n, p, ncrit, dist, seed=3, depth=depth)
    eng = abi.Engine(pr["kid"], p, pr["wavek"], precision)
    eng.set_operators(pr["ops"])
    eng.set_tree(pr["flat"])
    f, ops, ns, nl = pr["flat"], pr["ops"], eng.nsurf, int(pr["ops"]["nlevels"])
    shape = dict(m2m=(nl, 8, ns, ns), l2l=(nl, 8, ns, ns), dc2e_u=(nl, ns, ns), dc2e_v=(nl, ns, ns))
    mats = {k: np.asarray(ops[k]).reshape(s) for k, s in shape.items()}
    lo, child0 = np.asarray(f["level_offset"]), np.asarray(f["child0"])
    yield dict(eng=eng, mats=mats, lo=lo, child0=child0, depth=int(f["depth"]), kid=pr["kid"], nl=nl,
               bodies=np.asarray(f["src_count"]) + np.asarray(f["trg_count"]),
               u=2.0 ** -53 if precision == abi.FP64 else 2.0 ** -24,
               rng=np.random.default_rng(p), vw=2 if pr["kid"] == abi.HELMHOLTZ else 1)
    eng.close()


def vectors(t):
    shape = (t["eng"].nnodes, t["eng"].nsurf)
    v = t["rng"].normal(size=shape)
    return v + 1j * t["rng"].normal(size=shape) if t["vw"] == 2 else v


def mags(a):
    """|Re| + |Im| (the real GEMM form of a complex product sums the four real products)."""
    return np.abs(a.real) + np.abs(a.imag) if np.iscomplexobj(a) else np.abs(a)


def check(got, want, mag, k, t):
    assert np.all(np.abs(got - want) <= (t["vw"] * k + 8) * t["u"] * mag + 1e-300)


def test_m2m(problem):
    t = problem
    up = vectors(t)
    t["eng"].set_equiv(up=up)
    t["eng"].op("M2M")
    got = t["eng"].equiv()[0]
    ns = up.shape[1]
    for lv in range(t["depth"]):
        nodes = np.arange(t["lo"][lv], t["lo"][lv + 1])
        rows = nodes[t["child0"][nodes] >= 0]
        if len(rows) == 0:
            continue
        kids = got[t["child0"][rows][:, None] + np.arange(8)].reshape(len(rows), 8 * ns)
        op = t["mats"]["m2m"][0 if t["nl"] == 1 else lv].transpose(0, 2, 1).reshape(8 * ns, ns)
        check(got[rows], up[rows] + kids @ op, mags(up[rows]) + mags(kids) @ mags(op), 8 * ns, t)
    leaf = t["child0"] < 0
    assert np.array_equal(got[leaf], up[leaf])


def test_l2l(problem):
    t = problem
    dn = vectors(t)
    t["eng"].set_equiv(dn=dn)
    t["eng"].op("L2L")
    got = t["eng"].equiv()[1]
    ns = dn.shape[1]
    assert np.array_equal(got[:t["lo"][1]], dn[:t["lo"][1]])
    for lv in range(t["depth"]):
        nodes = np.arange(t["lo"][lv], t["lo"][lv + 1])
        rows = nodes[t["child0"][nodes] >= 0]
        if len(rows) == 0:
            continue
        op = t["mats"]["l2l"][0 if t["nl"] == 1 else lv].transpose(2, 0, 1).reshape(ns, 8 * ns)
        kids = (t["child0"][rows][:, None] + np.arange(8))
        want = dn[kids].reshape(len(rows), 8 * ns) + got[rows] @ op
        mag = mags(dn[kids]).reshape(len(rows), 8 * ns) + mags(got[rows]) @ mags(op)
        check(got[kids].reshape(len(rows), 8 * ns), want, mag, ns, t)


def test_l2p_solve(problem):
    t = problem
    dn = vectors(t)
    t["eng"].set_equiv(dn=dn)
    t["eng"].op("L2P")
    got = t["eng"].equiv()[1]
    ns = dn.shape[1]
    for lv in range(t["depth"] + 1):
        nodes = np.arange(t["lo"][lv], t["lo"][lv + 1])
        rows = nodes[(t["child0"][nodes] < 0) & (t["bodies"][nodes] > 0)]
        if len(rows) == 0:
            continue
        L, scale = (0 if t["nl"] == 1 else lv), (0.5 ** lv if t["kid"] == abi.LAPLACE else 1.0)
        u, v = t["mats"]["dc2e_u"][L].T, t["mats"]["dc2e_v"][L].T
        want = scale * ((dn[rows] @ u) @ v)
        check(got[rows], want, scale * ((mags(dn[rows]) @ mags(u)) @ mags(v)), 2 * ns, t)
