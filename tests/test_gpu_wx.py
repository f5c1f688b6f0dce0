"""W and X lists in one launch (k_wx): items of at most 32 points, source
chunks laid out over the lanes, list entries near their node on coordinate
differences instead of the Gram form, and the mixed path's own X sums onto
check surfaces (k_x_surf), against the CPU oracle on the same points."""
import numpy as np
import pytest

import kifmm_amd as K
import oracle_lib as O
from test_gpu_parity import raw_ops, rel

pytestmark = pytest.mark.gpu


def clustered(n, side, seed):
    """A sparse uniform set and a dense cube of width `side` whose corner lies
    1.5 side beyond the face x = 0: leaves at x < 0 get W boxes far below
    their own level, one box width away."""
    rng = np.random.default_rng(seed)
    p = rng.uniform(-1.0, 1.0, (3, n))
    k = n // 2
    p[:, :k] = np.array([[1.5 * side], [0.3], [0.3]]) + side * rng.random((3, k))
    return p, rng.random(n)


def near_entries(t):
    """W entries closer than 1/8 of the target leaf's half-width."""
    h = 2.0 ** -t["depth"].astype(float)
    c = (2.0 * t["path"] + 1.0) * h[:, None]
    count = 0
    for i in range(t["n_nodes"]):
        s = t["w_idx"][t["w_ptr"][i]:t["w_ptr"][i + 1]]
        gap = np.maximum(np.abs(c[i] - c[s]) - (h[i] + h[s])[:, None], 0.0)
        count += int(np.sum(np.sum(gap * gap, axis=1) < (h[i] / 8) ** 2))
    return count


@pytest.mark.parametrize("n,side,q,np_", [(700, 2.0 ** -7, 8, 3), (3000, 2.0 ** -9, 33, 4), (1500, 2.0 ** -8, 31, 6),
                                          (4000, 2.0 ** -6, 700, 4)])
@pytest.mark.parametrize("same", [True, False], ids=["coincident", "separate"])
def test_near_and_far_entries_match_oracle(n, side, q, np_, same):
    print(f"case n={n} side={side} q={q} NP={np_} coincident={same}", flush=True)
    s, den = clustered(n, side, 5)
    t = s if same else clustered(n, side, 6)[0]
    prob = K.Problem.from_points(*s, den, *([None] * 3 if same else t), pts_max=q, np_=np_)
    tree = prob.tree()
    near = near_entries(tree)
    print(f"  W {tree['w_idx'].size} ({near} near), X {tree['x_idx'].size}", flush=True)
    if q < 100:
        assert near > 0
    orc = O.Oracle(n, q=q, np_=np_, points=dict(zip(("sx", "sy", "sz", "den", "tx", "ty", "tz"), (*s, den, *t))))
    orc.set_operators(*raw_ops(prob))
    ref, _ = orc.evaluate(O.KERNEL_EXACT)
    pot = prob.scatter(K.GpuEvaluator(prob).evaluate()[0])
    r = rel(pot, ref)
    print(f"  rel L2 {r:.3e}", flush=True)
    assert r <= O.PARITY_RTOL[np_]
    if np_ <= 4:
        mixed = prob.scatter(K.GpuEvaluator(prob, precision=K.PREC_MIXED).evaluate()[0])
        assert rel(mixed, ref) <= 5e-7  # the mixed path's bound against the oracle


@pytest.mark.parametrize("n,dist,q,np_,c,prec", [(300, "gaussmix", 1, 3, 1, K.PREC_FP64),
                                                 (300, "gaussmix", 1, 3, 1, K.PREC_MIXED),
                                                 (9000, "ellipsoid", 40, 6, 0, K.PREC_FP64),
                                                 (60000, "gaussmix", 400, 4, 0, K.PREC_FP64),
                                                 (60000, "gaussmix", 400, 4, 0, K.PREC_MIXED)])
def test_lists_together_and_apart(n, dist, q, np_, c, prec):
    """W and X selected one at a time sum to W and X in one call, on the
    potentials and on the check values (two terms: one rounding apart)."""
    prob = K.Problem.create(n, dist, q, np_=np_, seed=8, coincide=c)
    ev = K.GpuEvaluator(prob, precision=prec)
    got = {}
    for name, mask in (("w", K.PHASE_UP | K.PHASE_W), ("x", K.PHASE_UP | K.PHASE_X),
                       ("wx", K.PHASE_UP | K.PHASE_W | K.PHASE_X)):
        got[name] = (ev.evaluate_phases(mask)[0], ev.intermediate("dchk"))
    assert np.abs(got["x"][1]).max() > 0 or np.abs(got["x"][0]).max() > 0
    for k in range(2):
        both = got["w"][k] + got["x"][k]
        assert np.all(np.abs(got["wx"][k] - both) <= 4e-16 * (np.abs(got["w"][k]) + np.abs(got["x"][k])))


@pytest.mark.parametrize("n,seed", [(500, 0), (700, 2), (900, 1), (900, 3)])
def test_near_pairs_are_as_exact_as_by_differences(n, seed):
    """One source in a W-list leaf closer than h/2 to targets in a corner of
    their leaf: each pair within 6e-15 of long double, the bound of the difference
    form ((3/2) e^2 = 5.3e-15 for an estimate e of 2^-24, and the roundings of
    r^2 and the scale, 4 x 1.1e-16).  In Gram form the roundings of |t|^2 + |s|^2 -
    2 t.s alone are 3e-14 at h/8."""
    rng = np.random.default_rng(seed)
    s = rng.uniform(-1.0, 1.0, (3, n))
    s[:, :200] = rng.uniform([[0.001], [0.47], [0.47]], [[0.03], [0.499], [0.499]], (3, 200))
    s[:, 200:206] = rng.uniform([[0.0313], [0.47], [0.47]], [[0.036], [0.499], [0.499]], (3, 6))
    t = rng.uniform([[-0.005], [0.46], [0.46]], [[0.0], [0.4999], [0.4999]], (3, n))
    prob = K.Problem.from_points(*s, rng.uniform(0.5, 1.0, n), *t, pts_max=8, np_=3)
    tree = prob.tree()
    ev = K.GpuEvaluator(prob)
    h = 2.0 ** -tree["depth"].astype(float)
    c = (2.0 * tree["path"] + 1.0) * h[:, None]
    pairs, worst = 0, 0.0
    for i in np.flatnonzero((tree["child"] == -1) & (tree["trg_num"] > 0)):
        for b in tree["w_idx"][tree["w_ptr"][i] : tree["w_ptr"][i + 1]]:
            gap = np.maximum(np.abs(c[i] - c[b]) - (h[i] + h[b]), 0.0)
            if tree["child"][b] != -1 or not 0 < tree["src_num"][b] < K.n_e(3) or np.sqrt(np.sum(gap * gap)) >= 0.5 * h[i]:
                continue
            j, k = tree["src_beg"][b], slice(tree["trg_beg"][i], tree["trg_beg"][i] + tree["trg_num"][i])
            den = np.zeros(n)
            den[j] = 1.0
            ev.set_densities(den)
            got = ev.evaluate_phases(K.PHASE_UP | K.PHASE_W)[0][k]
            x = [tree[a][k].astype(np.longdouble) - np.longdouble(tree[b_][j]) for a, b_ in (("tx", "sx"), ("ty", "sy"), ("tz", "sz"))]
            want = 1 / np.sqrt(x[0] ** 2 + x[1] ** 2 + x[2] ** 2) / (4 * np.arccos(np.longdouble(-1)))
            pairs += got.size
            worst = max(worst, float(np.max(np.abs(got / want - 1))))
    print(f"  {pairs} pairs, worst {worst:.2e}", flush=True)
    assert pairs > 0 and worst <= 6e-15
