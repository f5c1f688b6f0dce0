"""The U-list's wave kernel (small inputs) at the edges of its items and rows,
against long double sums over the U-list: leaves of 1 to 17 and 40 targets, fewer
sources than a row, more than 64 ranges per item, targets with none, a few and
more than 16 close pairs, coincident points; and the same bits as the block
kernels.

Bound per unit of sum |w| / r: the Gram form 2e-13 at the edge of the close
pairs, the Newton step 2e-14, the sums 2000 x 1.1e-16: below 5e-13."""
import numpy as np
import pytest

import kifmm_amd as K

pytestmark = pytest.mark.gpu


def u_sums(t):
    """U-list potentials and sums of absolute terms, in long double."""
    s = np.array([t[k] for k in ("sx", "sy", "sz")]).astype(np.longdouble)
    x = np.array([t[k] for k in ("tx", "ty", "tz")]).astype(np.longdouble)
    w = t["sden"].astype(np.longdouble)
    out = np.zeros((2, x.shape[1]), dtype=np.longdouble)
    for i in np.flatnonzero((t["child"] == -1) & (t["trg_num"] > 0)):
        boxes = t["u_idx"][t["u_ptr"][i] : t["u_ptr"][i + 1]]
        j = np.concatenate([np.arange(t["src_beg"][b], t["src_beg"][b] + t["src_num"][b]) for b in boxes] or [[]])
        k = np.arange(t["trg_beg"][i], t["trg_beg"][i] + t["trg_num"][i])
        j = j.astype(int)
        r = np.sqrt(((x[:, k][:, :, None] - s[:, j][:, None, :]) ** 2).sum(0))
        v = np.divide(w[j], r, out=np.zeros_like(r), where=r != 0)
        out[:, k] = v.sum(1), np.abs(v).sum(1)
    return out / (4 * np.arccos(np.longdouble(-1)))


def points(n, kind, rng):
    if kind == "uniform":
        return rng.uniform(-1.0, 1.0, (3, n))
    x = rng.normal(0.0, 0.15, (3, n)) + rng.choice([-0.4, 0.3], (3, 1))
    x[:, : n // 8] = x[:, :1] + rng.normal(0.0, 1e-4, (3, n // 8))  # many close pairs for some targets
    return np.clip(x, -0.99, 0.99)


# groups of 8 targets below 8192: one group per item; above: two
@pytest.mark.parametrize("n,q,kind,same", [(1, 8, "uniform", True), (7, 8, "uniform", False), (300, 1, "uniform", True),
                                           (700, 17, "cluster", True), (2000, 40, "cluster", False),
                                           (4000, 3, "cluster", True), (70000, 9, "uniform", True),
                                           (45000, 40, "cluster", False)])
def test_wave_items(n, q, kind, same):
    print(f"case n={n} q={q} {kind} same={same}", flush=True)
    rng = np.random.default_rng(n + q)
    src = points(n, kind, rng)
    trg = src if same else points(n, kind, rng)
    den = rng.uniform(-1.0, 1.0, n)
    prob = K.Problem.from_points(*src, den, *trg, pts_max=q, np_=3)
    ev = K.GpuEvaluator(prob)
    got, _ = ev.evaluate_phases(K.PHASE_U)
    got = np.array(got)
    if n <= 5000:
        want, scale = u_sums(prob.tree())
        assert np.all(np.abs(got - want) <= 5e-13 * scale)
    for form in (K.P2P_STATIC64, K.P2P_PERSISTENT):
        ev.set_tuning(form, 8, K.HAD_MFMA)
        assert np.array_equal(ev.evaluate_phases(K.PHASE_U)[0], got), form
