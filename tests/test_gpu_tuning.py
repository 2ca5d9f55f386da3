"""The launch-shape parameters: what is set is what is read, every setting runs, and none changes a Hadamard value."""
import numpy as np
import pytest

import oracle as O
from exafmm import abi
from fmm_cases import make_problem, rel_err

pytestmark = pytest.mark.gpu


def engine(pr, precision):
    eng = abi.Engine(pr["kid"], pr["p"], pr["wavek"], precision)
    eng.set_operators(pr["ops"])
    eng.set_tree(pr["flat"])
    eng.set_charges(pr["qs"])
    return eng


@pytest.mark.parametrize("precision", [abi.FP64, abi.MIXED])
def test_parameters_read_as_set(require_gpu, precision):
    pr = make_problem("laplace", 6000, 4, 40, "cube", seed=15, precision=precision)
    new = abi.Engine(pr["kid"], pr["p"], pr["wavek"], precision)
    eng = engine(pr, precision)
    for e in (new, eng):  # without and with a tree
        for param, values in ((abi.TUNE_HAD_KCH, range(1, 257)), (abi.TUNE_P2P_SPLIT, range(33)),
                              (abi.TUNE_HAD_GROUPS, (1, 2, 4)), (abi.TUNE_HAD_TILES, (1, 2))):
            default = e.get_tuning(param)
            assert default in values
            for v in values:
                e.set_tuning(param, v)
                assert e.get_tuning(param) == v
            for v in (min(values) - 1, max(values) + 1):
                with pytest.raises(abi.XfmmError):
                    e.set_tuning(param, v)
            assert e.get_tuning(param) == max(values)
    new.close()
    eng.close()


def test_automatic_frequencies_read_back(require_gpu):
    """The chunk that is read while none was set is the one that runs: setting it changes no value, and small grids
    have fewer frequencies than the largest default."""
    pr = make_problem("laplace", 6000, 4, 40, "cube", seed=15, precision=abi.MIXED)
    eng = engine(pr, abi.MIXED)
    k = eng.get_tuning(abi.TUNE_HAD_KCH)
    assert k < 16 and k % 2 == 0
    eng.close()


@pytest.mark.parametrize("kernel", ["laplace", "helmholtz"])
@pytest.mark.parametrize("precision", [abi.FP64, abi.FLOAT])
def test_no_split_sums_in_one_lane(require_gpu, kernel, precision):
    """With a split of 0 the sources of a target are summed by one lane in their order: the first two of the only
    leaf lie at one place with charges of +-2^60, whose terms cancel exactly when they are added one after the
    other and swallow 60 bits of the sum when anything is added between them or they are added apart.  (The Yukawa kernel rounds
its term within the addition, so that there the two do not cancel exactly.)"""
    pr = make_problem(kernel, 60, 3, 64, "cube", seed=4)
    f, q = dict(pr["flat"]), np.array(pr["qs"])
    assert f["nnodes"] == 1
    x = np.array(f["src_coord"]).reshape(-1, 3)
    x[1] = x[0]
    q[0], q[1] = 2.0 ** 60, -(2.0 ** 60)
    f["src_coord"] = x.reshape(-1)
    eng = engine(dict(pr, flat=f, qs=q), precision)
    eng.set_tuning(abi.TUNE_P2P_SPLIT, 0)
    eng.clear()
    eng.op("P2P")
    v = eng.values()[:, 0]
    eng.close()
    q[:2] = 0
    r = O.direct(pr["kid"], x, q, np.array(f["trg_coord"]).reshape(-1, 3), pr["wavek"])[:, 0]
    # targets near the pair have its FP64 correction in FLOAT, added apart
    far = np.linalg.norm(np.array(f["trg_coord"]).reshape(-1, 3) - x[0], axis=1) > 0.2
    assert np.sum(far) > 20
    assert rel_err(v[far], r[far]) < (1e-12 if precision == abi.FP64 else 1e-5)
