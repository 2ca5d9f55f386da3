"""What a small tree does not launch: Hadamard blocks of more than 1024 M2L targets (the default then is 256 targets a
block and two tiles a wave), and the kernels of a damped wave number."""
import numpy as np
import pytest

import oracle as O
from exafmm import abi
from fmm_cases import make_problem, rel_err

pytestmark = pytest.mark.gpu

FP64_TOL, FP32_TOL = 1e-10, 1e-5  # the parity bars against the oracle on the same operators


def engine(pr, precision):
    eng = abi.Engine(pr["kid"], pr["p"], pr["wavek"], precision)
    eng.set_operators(pr["ops"])
    eng.set_tree(pr["flat"])
    eng.set_charges(pr["qs"])
    return eng


def evaluate(eng):
    eng.upward_pass()
    eng.downward_pass()
    return eng.values()


def reference(pr):
    orc = O.Oracle(pr["kid"], pr["p"], pr["flat"], pr["ops"], pr["wavek"])
    orc.set_charges(pr["qs"])
    return orc.evaluate()


# 256-target blocks: 7 of 13 full, 5 closed by a full colour (640 union slots); 5 of 20 and 14; 20 of 26 and none, one
# operator set a level; 8 of 14 and 3
@pytest.mark.parametrize("kernel,n,p,ncrit,dist,depth", [
    ("laplace", 30000, 4, 6, "cube", None), ("laplace", 40000, 4, 64, "cube", 5),
    ("modified_helmholtz", 20000, 4, 4, "sphere", None), ("helmholtz", 20000, 3, 4, "cube", None)])
@pytest.mark.parametrize("precision", [abi.FP64, abi.MIXED])
def test_many_targets(require_gpu, kernel, n, p, ncrit, dist, depth, precision):
    pr = make_problem(kernel, n, p, ncrit, dist, seed=31, depth=depth, precision=precision)
    m2l = np.asarray(pr["flat"]["m2l_source"]).reshape(-1, 26)
    assert np.sum(np.any(m2l >= 0, axis=1)) > 2048
    eng = engine(pr, precision)
    assert eng.get_tuning(abi.TUNE_HAD_TILES) == 2
    assert precision == abi.FP64 or eng.get_tuning(abi.TUNE_HAD_GROUPS) == 4
    v, r = evaluate(eng), reference(pr)
    tol = FP64_TOL if precision == abi.FP64 else FP32_TOL
    print(kernel, precision, rel_err(v[:, 0], r[:, 0]), rel_err(v[:, 1:], r[:, 1:]), flush=True)
    assert rel_err(v[:, 0], r[:, 0]) < tol and rel_err(v[:, 1:], r[:, 1:]) < tol
    # the launch shape changes no value
    for groups in (1, 2, 4) if precision != abi.FP64 else (1,):
        for tiles in (1, 2):
            for kch in (1, 6, 16):
                eng.set_tuning(abi.TUNE_HAD_GROUPS, groups)
                eng.set_tuning(abi.TUNE_HAD_TILES, tiles)
                eng.set_tuning(abi.TUNE_HAD_KCH, kch)
                assert np.array_equal(evaluate(eng), v), (groups, tiles, kch)
    eng.close()


@pytest.mark.parametrize("n,ncrit,dist", [(1500, 150, "cube"), (6000, 40, "cube"), (7000, 12, "clusters")])
@pytest.mark.parametrize("precision", [abi.FP64, abi.MIXED, abi.FLOAT])
def test_damped_helmholtz(require_gpu, n, ncrit, dist, precision):
    pr = make_problem("helmholtz", n, 5, ncrit, dist, seed=32, wavek=5.0 + 2.0j, precision=precision)
    f = pr["flat"]
    if dist == "clusters":
        assert f["m2p_offset"][-1] > 0 and f["p2l_offset"][-1] > 0
    eng = engine(pr, precision)
    v, r = evaluate(eng), reference(pr)
    eng.close()
    tol = FP64_TOL if precision == abi.FP64 else FP32_TOL
    print(n, dist, precision, rel_err(v[:, 0], r[:, 0]), rel_err(v[:, 1:], r[:, 1:]), flush=True)
    assert rel_err(v[:, 0], r[:, 0]) < tol and rel_err(v[:, 1:], r[:, 1:]) < tol
