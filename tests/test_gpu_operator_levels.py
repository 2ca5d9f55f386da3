"""Operators of a level-dependent kernel handed over as one set: it serves every level, in the M2L and in the
translations, as in the oracle.  Other counts below the tree's depth are refused before any kernel is launched."""
import numpy as np
import pytest

import oracle as O
from exafmm import abi
from fmm_cases import make_problem, rel_err

pytestmark = pytest.mark.gpu


def one_level(ops, keep):
    """The operators with the first of the levels only, for the M2L alone (keep) or for all of them."""
    o = dict(ops, m2l=np.asarray(ops["m2l"]).reshape(ops["nm2l"], -1)[0].copy(), nm2l=1)
    if not keep:
        for k in ("uc2e_u", "uc2e_v", "dc2e_u", "dc2e_v", "m2m", "l2l"):
            o[k] = np.asarray(ops[k]).reshape(ops["nlevels"], -1)[1].copy()
        o["nlevels"] = 1
    return o


@pytest.mark.parametrize("kernel", ["modified_helmholtz", "helmholtz"])
@pytest.mark.parametrize("precision,tol", [(abi.FP64, 1e-10), (abi.MIXED, 1e-5)])
def test_one_operator_set(require_gpu, kernel, precision, tol):
    pr = make_problem(kernel, 6000, 4, 40, "cube", seed=15, precision=precision)
    assert pr["flat"]["depth"] >= 3 and pr["ops"]["nm2l"] >= 3
    eng = abi.Engine(pr["kid"], 4, pr["wavek"], precision)
    eng.set_operators(pr["ops"])
    eng.set_tree(pr["flat"])
    eng.set_charges(pr["qs"])
    # all levels, then one set, with the tree already there, and back
    for ops in (pr["ops"], one_level(pr["ops"], True), one_level(pr["ops"], False), pr["ops"]):
        eng.set_operators(ops)
        eng.upward_pass()
        eng.downward_pass()
        v = eng.values()
        orc = O.Oracle(pr["kid"], 4, pr["flat"], ops, pr["wavek"])
        orc.set_charges(pr["qs"])
        r = orc.evaluate()
        print(kernel, precision, ops["nlevels"], ops["nm2l"], rel_err(v[:, 0], r[:, 0]), rel_err(v[:, 1:], r[:, 1:]), flush=True)
        assert rel_err(v[:, 0], r[:, 0]) < tol
        assert rel_err(v[:, 1:], r[:, 1:]) < tol
    eng.close()


@pytest.mark.parametrize("kernel", ["modified_helmholtz", "helmholtz"])
def test_too_few_levels_refused(require_gpu, kernel):
    pr = make_problem(kernel, 6000, 4, 40, "cube", seed=15)
    ops = pr["ops"]
    eng = abi.Engine(pr["kid"], 4, pr["wavek"], abi.FP64)
    eng.set_tree(pr["flat"])
    n = ops["nm2l"] - 1
    for bad in (dict(ops, m2l=np.asarray(ops["m2l"]).reshape(ops["nm2l"], -1)[:n].copy(), nm2l=n),
                dict(ops, nlevels=ops["nlevels"] - 1)):
        eng.set_operators(bad)
        with pytest.raises(abi.XfmmError, match="fewer levels"):
            eng.upward_pass()
        with pytest.raises(abi.XfmmError, match="fewer levels"):
            eng.op("M2L")
    eng.close()


@pytest.mark.parametrize("precision", [abi.FP64, abi.MIXED])
def test_failed_upload_leaves_no_operators(require_gpu, precision):
    """A set of operators whose upload fails part of the way (an M2L of more bytes than there is memory) replaces
    some of the earlier ones: the passes refuse to run on the mixture until a whole set is there."""
    pr = make_problem("modified_helmholtz", 6000, 4, 40, "cube", seed=15)
    eng = abi.Engine(pr["kid"], 4, pr["wavek"], precision)
    eng.set_operators(pr["ops"])
    eng.set_tree(pr["flat"])
    eng.set_charges(pr["qs"])
    eng.upward_pass()
    eng.downward_pass()
    want = eng.values()
    with pytest.raises(abi.XfmmError):
        eng.set_operators(dict(pr["ops"], nm2l=2 ** 30))
    with pytest.raises(abi.XfmmError, match="operators not set"):
        eng.upward_pass()
    eng.set_operators(pr["ops"])
    eng.upward_pass()
    eng.downward_pass()
    assert np.array_equal(eng.values(), want)
    eng.close()
