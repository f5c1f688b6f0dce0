"""The direct sums at the edges of their split (groups of 8 targets, chunks of
whole runs of 1024 sources) and at the distances that leave the fast path
(coincident, denormal and overflowing r^2), against sums in long double.

Bound per term, in units of 2^-53: differences and r^2 give 1 / r at most 2,
the inverse square root 1.5, the weight and the run of four sources 4; the
compensated sums add about one of the result.  8 x 2^-53 = 8.9e-16 of the sum of
absolute terms, and one rounding of the result: 1.1e-15 in all."""
import numpy as np
import pytest

import kifmm_amd as K

pytestmark = pytest.mark.gpu


def exact(t, s, w):
    """(sums, sums of absolute terms) over 4 pi, r = 0 excluded."""
    t, s, w = (a.astype(np.longdouble) for a in (t, s, w))
    out = []
    for k in range(t.shape[1]):
        r = np.sqrt(((s - t[:, k : k + 1]) ** 2).sum(0))
        v = np.divide(w, r, out=np.zeros_like(r), where=r != 0)
        out.append((v.sum(), np.abs(v).sum()))
    return np.array(out).T / (4 * np.arccos(np.longdouble(-1)))


@pytest.mark.parametrize("n,nt", [(1000, 1), (1023, 7), (1024, 8), (1025, 9), (4099, 65), (9000, 3000), (70000, 33)])
def test_direct_split_edges(n, nt):
    print(f"case n={n} nt={nt}", flush=True)
    prob = K.Problem.create(n, "ellipsoid", 64, np_=4, seed=n)
    tree = prob.tree()
    s = np.array([tree[k] for k in ("sx", "sy", "sz")])
    t = np.random.default_rng(nt).uniform(-1.0, 1.0, (3, nt))
    pick = np.random.default_rng(n).choice(n, (nt + 1) // 2, replace=False)
    t[:, : pick.size] = s[:, pick]  # r = 0 pairs
    if nt > 8:
        near = pick[:4]
        t[:, 4:8] = s[:, near] * (1.0 + np.array([2.0**-52, 1e-13, 1e-9, 1e-4]))  # close pairs
    got = K.GpuEvaluator(prob).direct(*t)
    want, scale = exact(t, s, tree["sden"])
    assert np.all(np.abs(got - want) <= 1.1e-15 * scale)


def test_direct_at_extreme_distances():
    rng = np.random.default_rng(5)
    s, w = rng.uniform(-1.0, 1.0, (3, 1000)), rng.uniform(0.5, 1.0, 1000)
    s[:, 300] = 0.0
    ev = K.GpuEvaluator(K.Problem.from_points(*s, w, pts_max=64, np_=4))
    # from the source at the origin: r^2 normal, denormal (exact powers of two) and underflowing to 0
    for x in (2.0**-300, 2.0**-520, 2.0**-530):
        got = ev.direct(np.array([x]), np.zeros(1), np.zeros(1))
        assert got[0] == pytest.approx(w[300] / x / (4 * np.pi), rel=1e-14)
    got = ev.direct(np.array([2.0**-560]), np.zeros(1), np.zeros(1))
    want, _ = exact(np.zeros((3, 1)), s, w)
    assert got[0] == pytest.approx(float(want[0]), rel=1e-14)
    # 1e153: r^2 = 1e306 is still a normal number; beyond, it overflows and w / sqrt(inf) = 0
    far = np.array([1e153, 1e170, 1e300, np.inf])
    got = ev.direct(far, np.zeros(4), np.zeros(4))
    assert got[0] == pytest.approx(w.sum() / (4 * np.pi) / 1e153, rel=1e-13)
    assert np.all(got[1:] == 0.0)
    assert np.isnan(ev.direct(*np.full((3, 1), np.nan))[0])
