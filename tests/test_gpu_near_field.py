"""P2P and M2P against the oracle where the number of waves that share a tile of targets changes: trees of one
to thousands of tiles, full tiles, tails just below and above the source split, more than one tile per leaf, the
three kernels.  FP64 within 1e-12 of the values' norm (the operators are applied to the same inputs; sums of at most
some 1e4 terms in another order), FP32 within 1e-5."""
import os

import numpy as np
import pytest

import oracle as O
from exafmm import abi
from fmm_cases import CACHE, KERNELS, charges, make_problem, rel_err

pytestmark = pytest.mark.gpu

CASES = [  # kernel, n, ncrit, dist: tiles and their sizes
    ("laplace", 40, 64, "cube"),              # one leaf, one tail tile
    ("laplace", 500, 200, "cube"),            # leaves of about 62: one tile, above and below 64
    ("laplace", 1600, 300, "cube"),           # leaves of about 200: several tiles with tails
    ("laplace", 9000, 30, "clusters"),        # thousands of tiles, M2P lists
    ("modified_helmholtz", 1100, 150, "cube"),
    ("modified_helmholtz", 7000, 12, "clusters"),
    ("helmholtz", 70, 100, "cube"),
    ("helmholtz", 2000, 260, "cube"),
    ("helmholtz", 9000, 20, "clusters"),
]


@pytest.mark.parametrize("kernel,n,ncrit,dist", CASES)
@pytest.mark.parametrize("precision,split", [(abi.FP64, 32), (abi.FP64, 0), (abi.FLOAT, 32)])
def test_particle_targets(require_gpu, kernel, n, ncrit, dist, precision, split):
    pr = make_problem(kernel, n, 4, ncrit, dist, seed=5)
    eng = abi.Engine(pr["kid"], 4, pr["wavek"], precision)
    eng.set_operators(pr["ops"])
    eng.set_tree(pr["flat"])
    eng.set_charges(pr["qs"])
    eng.set_tuning(abi.TUNE_P2P_SPLIT, split)
    orc = O.Oracle(pr["kid"], 4, pr["flat"], pr["ops"], pr["wavek"])
    orc.set_charges(pr["qs"])
    rng = np.random.default_rng(1)
    up = rng.normal(size=(eng.nnodes, eng.nsurf))
    if eng.cplx:
        up = up + 1j * rng.normal(size=up.shape)
    tol = 1e-12 if precision == abi.FP64 else 1e-5

    def check(v, r):
        if np.linalg.norm(r) == 0:
            assert np.linalg.norm(v) == 0
            return
        assert rel_err(v[:, 0], r[:, 0]) < tol
        assert rel_err(v[:, 1:], r[:, 1:]) < tol

    for op in ("P2P", "M2P"):
        eng.clear()
        orc.clear()
        eng.set_equiv(up=up)
        orc.up[:] = up
        eng.op(op)
        orc.run(O.STAGES[op])
        check(eng.values(), orc.val)
    eng.close()


@pytest.mark.parametrize("kernel,n,ncrit,dist", [("laplace", 9000, 30, "clusters"), ("helmholtz", 2000, 260, "cube")])
def test_passes_read_as_zeroed(require_gpu, kernel, n, ncrit, dist):
    """After an upward pass the target values and dn read as zero, single operators add to zeros, and a pass after
    foreign values, in another order or repeated gives the values of a fresh one bit for bit."""
    pr = make_problem(kernel, n, 4, ncrit, dist, seed=6)

    def engine():
        eng = abi.Engine(pr["kid"], 4, pr["wavek"], abi.FP64)
        eng.set_operators(pr["ops"])
        eng.set_tree(pr["flat"])
        eng.set_charges(pr["qs"])
        return eng

    a = engine()
    a.upward_pass()
    a.downward_pass()
    want, (up, dn) = a.values(), a.equiv()
    a.upward_pass()
    assert not np.any(a.values()) and not np.any(a.equiv()[1])
    assert np.array_equal(a.equiv()[0], up)
    a.op("P2P")
    p2p = a.values()
    a.op("P2P")
    assert np.array_equal(a.values(), 2 * p2p)
    a.downward_pass()
    assert np.array_equal(a.values(), want) and np.array_equal(a.equiv()[1], dn)
    b = engine()
    b.values_device_ptr()
    b.set_equiv(up=np.full(up.shape, 7.0), dn=np.full(dn.shape, 7.0))
    b.op("P2P")
    b.upward_pass()
    assert not np.any(b.values())
    b.upward_pass()
    b.downward_pass()
    assert np.array_equal(b.values(), want)
    assert np.array_equal(b.equiv()[0], up) and np.array_equal(b.equiv()[1], dn)
    b.graph_capture()
    b.upward_pass()
    assert not np.any(b.equiv()[1])
    for _ in range(3):
        b.graph_launch()
        assert np.array_equal(b.values(), want) and np.array_equal(b.equiv()[1], dn)
    a.close()
    b.close()


@pytest.mark.parametrize("kernel,ncrit", [("laplace", 70), ("modified_helmholtz", 40), ("helmholtz", 64)])
@pytest.mark.parametrize("precision", [abi.FP64, abi.FLOAT])
def test_long_source_lists(require_gpu, kernel, ncrit, precision):
    """P2P lists of more than 64 leaves (a large leaf beside a dense layer), leaves of 1 to 58 targets.  Tolerances as
    above."""
    mod, cls, kid, wavek = KERNELS[kernel]
    rng = np.random.default_rng(3)
    x = np.concatenate([rng.random((9000, 3)) * [0.04, 1, 1] + [0.46, 0, 0],
                        rng.random((ncrit - 3, 3)) * 0.5 + [0.5, 0, 0], [[0, 0, 0], [1, 1, 1]]])
    q = charges("centered", len(x), rng, kid == 1)
    name = os.path.join(CACHE, "%s_long_%d.dat" % (kernel, ncrit))
    fmm = getattr(mod, cls)(4, ncrit, **({} if wavek is None else {"wavek": wavek}), filename=name)
    tree = mod.setup(mod.init_sources(x, q), mod.init_targets(x), fmm)
    flat = fmm.flat_tree(tree)
    count = np.diff(flat["p2p_offset"])
    assert np.any((count > 64) & (flat["trg_count"] > 0))
    wk = 0.0 if wavek is None else wavek
    eng = abi.Engine(kid, 4, wk, precision)
    eng.set_operators(fmm.operators())
    eng.set_tree(flat)
    eng.set_charges(fmm.sorted_charges(tree))
    orc = O.Oracle(kid, 4, flat, fmm.operators(), wk)
    orc.set_charges(fmm.sorted_charges(tree))
    eng.clear()
    orc.clear()
    eng.op("P2P")
    orc.run(O.STAGES["P2P"])
    v, r = eng.values(), orc.val
    tol = 1e-12 if precision == abi.FP64 else 1e-5
    assert rel_err(v[:, 0], r[:, 0]) < tol
    assert rel_err(v[:, 1:], r[:, 1:]) < tol
    eng.close()


@pytest.mark.parametrize("wavek", [0.5, 50.0, 3.0e4, 1.0e7, 1.0e10])
def test_helmholtz_phases(require_gpu, wavek):
    """Near field with phases k r from below 1 to beyond 2^30 (the library's reduction).  k r is rounded to 53 bits and
    r to about 3 ulp on both sides: 8 k r 2^-53 rad a pair, times 8 for the cancellation of sums of 400 charges of
    both signs."""
    pr = make_problem("helmholtz", 400, 3, 64, "cube", seed=8, wavek=wavek)
    eng = abi.Engine(pr["kid"], 3, wavek, abi.FP64)
    eng.set_operators(pr["ops"])
    eng.set_tree(pr["flat"])
    eng.set_charges(pr["qs"])
    orc = O.Oracle(pr["kid"], 3, pr["flat"], pr["ops"], wavek)
    orc.set_charges(pr["qs"])
    eng.clear()
    orc.clear()
    eng.op("P2P")
    orc.run(O.STAGES["P2P"])
    v, r = eng.values(), orc.val
    tol = 1e-13 + 64 * wavek * np.sqrt(3.0) * 2.0 ** -53
    assert rel_err(v[:, 0], r[:, 0]) < tol
    assert rel_err(v[:, 1:], r[:, 1:]) < tol
    eng.close()
