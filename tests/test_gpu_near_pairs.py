"""FP32 near field of close pairs across a leaf plane: the rounding of their positions."""
import numpy as np
import pytest

import oracle as O
from exafmm import abi
from fmm_cases import make_problem

pytestmark = pytest.mark.gpu


def face_neighbours(f):
    """(target leaf, source leaf, side) of leaves of one size that share a face normal to x, each leaf once on
    either side, the source leaf in the target leaf's P2P list."""
    c = np.asarray(f["center"]).reshape(-1, 3)
    lev, off, lst = f["level"], f["p2p_offset"], f["p2p_source"]
    used_t, used_s, out = set(), set(), []
    for t in range(f["nnodes"]):
        if f["child0"][t] >= 0 or f["trg_count"][t] == 0:
            continue
        side = 2.0 * f["r0"] * 0.5 ** lev[t]
        for s in lst[off[t]:off[t + 1]]:
            d = (c[s] - c[t]) / side
            if lev[s] == lev[t] and f["src_count"][s] > 0 and np.allclose(d, [1, 0, 0], atol=1e-6) \
                    and t not in used_t and s not in used_s:
                used_t.add(t)
                used_s.add(int(s))
                out.append((t, int(s), side))
    return out


def planted(kernel, place, rng):
    """A problem whose first target of a leaf and first source of its neighbour in x are put at place(side) =
    (target, source), relative to the target leaf's centre; the other sources have no charge."""
    pr = make_problem(kernel, 12000, 4, 60, "cube", seed=23)
    f = dict(pr["flat"])
    src = np.array(f["src_coord"]).reshape(-1, 3)
    trg = np.array(f["trg_coord"]).reshape(-1, 3)
    q = np.zeros(len(src), dtype=np.asarray(pr["qs"]).dtype)
    c = np.asarray(f["center"]).reshape(-1, 3)
    rows = []
    for t, s, side in face_neighbours(f):
        a, b = place(side)
        it, js = f["trg_begin"][t], f["src_begin"][s]
        trg[it], src[js] = c[t] + a, c[t] + b
        q[js] = rng.choice([-1.0, 1.0])
        rows.append(it)
    f["src_coord"], f["trg_coord"] = src.reshape(-1), trg.reshape(-1)
    return pr, f, q, np.array(rows)


def near_field(pr, f, q, precision=abi.FLOAT):
    eng = abi.Engine(pr["kid"], 4, pr["wavek"], precision)
    eng.set_operators(pr["ops"])
    eng.set_tree(f)
    eng.set_charges(q)
    orc = O.Oracle(pr["kid"], 4, f, pr["ops"], pr["wavek"])
    orc.set_charges(q)
    eng.clear()
    orc.clear()
    eng.op("P2P")
    orc.run(O.STAGES["P2P"])
    v, r = eng.values(), orc.val.copy()
    eng.close()
    return v, r


def row_err(v, r):
    return np.linalg.norm(v - r, axis=1) / np.linalg.norm(r, axis=1)


@pytest.mark.parametrize("kernel", ["laplace", "modified_helmholtz", "helmholtz"])
def test_positions_rounded_once(require_gpu, kernel):
    """Pairs at 1/14 to 1/10 of a leaf's side, just beyond those that are corrected in FP64, at positions relative to
    the target leaf's centre that FP32 holds exactly: rounded once there, they lose nothing, and what is left is the
    FP32 arithmetic of a pair (r^2, 1/r within one ulp, three products: at most 12 2^-24 = 7.3e-7 of a gradient, a
    third of it in the root of the mean square).  Positions relative to the source leaf, shifted in FP32, lose
    another two roundings of about 2^-25 of the side, 14 times that of the distance."""
    rng = np.random.default_rng(2)

    def place(side):
        d = rng.normal(size=3)
        d *= side * rng.uniform(1 / 14.0, 1 / 10.0) / np.linalg.norm(d)
        d[0] = abs(d[0])
        a = np.array([0.5, *rng.uniform(-0.4, 0.4, 2)]) * side
        a[0] -= 0.5 * d[0]
        a = a.astype(np.float32)
        return a.astype(np.float64), (a + d.astype(np.float32)).astype(np.float64)

    pr, f, q, rows = planted(kernel, place, rng)
    assert len(rows) > 50
    v, r = near_field(pr, f, q)
    e = [np.sqrt(np.mean(row_err(v[rows][:, c], r[rows][:, c]) ** 2)) for c in (slice(0, 1), slice(1, 4))]
    print(kernel, len(rows), "potential %.2e gradient %.2e" % tuple(e), flush=True)
    assert e[1] < 2.5e-7


@pytest.mark.parametrize("kernel", ["laplace", "modified_helmholtz", "helmholtz"])
@pytest.mark.parametrize("gap", [1e-3, 1e-6, 1e-9, 1e-13])
def test_points_rounded_together(require_gpu, kernel, gap):
    """Two points on either side of a leaf plane, `gap` leaf sides apart with equal other coordinates, the smaller
    ones rounded to one position in FP32: finite, and within the near field's 1e-6 (potential) and 5e-6 (gradient)
    of the oracle for each of the targets."""
    rng = np.random.default_rng(3)

    def place(side):
        yz = rng.uniform(-0.4, 0.4, 2) * side
        return np.array([0.5 * side - 0.5 * gap * side, *yz]), np.array([0.5 * side + 0.5 * gap * side, *yz])

    pr, f, q, rows = planted(kernel, place, rng)
    src, trg = np.asarray(f["src_coord"]).reshape(-1, 3), np.asarray(f["trg_coord"]).reshape(-1, 3)
    assert len(rows) > 50 and np.all(np.min(np.linalg.norm(src[q != 0][:, None] - trg[rows], axis=2), axis=0) > 0)
    v, r = near_field(pr, f, q)
    assert np.all(np.isfinite(v))
    e = [np.max(row_err(v[rows][:, c], r[rows][:, c])) for c in (slice(0, 1), slice(1, 4))]
    print(kernel, gap, "potential %.2e gradient %.2e" % tuple(e), flush=True)
    assert e[0] < 1e-6 and e[1] < 5e-6


@pytest.mark.parametrize("kernel", ["laplace", "modified_helmholtz", "helmholtz"])
def test_points_rounded_together_fp64(require_gpu, kernel):
    """The same at a leaf plane through zero, where FP64 numbers lie closer together than the rounding of a leaf's
    size: two points 2e-30 apart give a finite value at their target, of the sign of the charge and at least that
    of the distance a leaf resolves, and leave all other targets within 1e-12."""
    pr = make_problem(kernel, 12000, 4, 60, "cube", seed=23)
    f = dict(pr["flat"])
    src, trg, c = (np.array(f[k]).reshape(-1, 3) for k in ("src_coord", "trg_coord", "center"))
    near = face_neighbours(f)
    planes = np.array([c[t, 0] + 0.5 * side for t, _, side in near])
    zero = planes[len(planes) // 2]
    near = [p for p, x in zip(near, planes) if abs(x - zero) < 1e-9]
    assert len(near) > 10
    for a in (src, trg, c):
        a[:, 0] -= zero
    f["x0"] = np.array(f["x0"]) - [zero, 0, 0]
    q = np.zeros(len(src), dtype=np.asarray(pr["qs"]).dtype)
    rows, sides = [], []
    for t, s, side in near:
        c[[t, s], 0] = [-0.5 * side, 0.5 * side]
        it, js = f["trg_begin"][t], f["src_begin"][s]
        trg[it], src[js] = c[t], c[t]
        trg[it, 0], src[js, 0], q[js] = -1e-30, 1e-30, 1.0
        rows.append(it)
        sides.append(side)
    f["src_coord"], f["trg_coord"], f["center"] = src.reshape(-1), trg.reshape(-1), c.reshape(-1)
    v, r = near_field(pr, f, q, abi.FP64)
    assert np.all(np.isfinite(v))
    assert np.all(v[rows, 0].real > 2.0 ** 52 / np.array(sides) / (4 * np.pi))
    rest = np.setdiff1d(np.arange(len(v)), rows)
    assert np.linalg.norm(v[rest] - r[rest]) < 1e-12 * np.linalg.norm(r[rest])
