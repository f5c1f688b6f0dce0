"""Level applies spread over blocks by row (k_level_op): M2M, the leaf UC2UE
and DC2DE on levels of one column to a few thousand, whole and ragged 16-column
tiles, the NP = 6 stack in parts along K and whole, L2L + DC2DE in two launches
and in the fused kernel, against the column GEMMs."""
import numpy as np
import pytest

import kifmm_amd as K
import oracle_lib as O
from test_gpu_parity import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,dist,q,np_,prec", [
    (40, "uniform", 2, 3, K.PREC_FP64),          # a handful of columns per level
    (300, "gaussmix", 1, 6, K.PREC_FP64),        # one or two parents on deep levels
    (9000, "ellipsoid", 20, 4, K.PREC_FP64),     # ragged column tiles
    (60000, "uniform", 3, 6, K.PREC_FP64),       # 4096 parents on a level: UE2UC stack and L2L + DC2DE unsplit
    (90000, "uniform", 8, 4, K.PREC_FP64),       # leaf UC2UE above the k_level_op size
    (9000, "ellipsoid", 20, 4, K.PREC_MIXED),
    (60000, "uniform", 8, 3, K.PREC_MIXED),
])
def test_level_op_matches_column_gemms(n, dist, q, np_, prec):
    print(f"case {dist} n={n} q={q} NP={np_} prec={prec}", flush=True)
    prob = K.Problem.create(n, dist, q, np_=np_, seed=31)
    t = prob.tree()
    src, trg = (t["tag"] & K.KIFMM_SRCNODE) != 0, (t["tag"] & K.KIFMM_TRGNODE) != 0
    ev = K.GpuEvaluator(prob, precision=prec)
    assert ev.tuning()["up_form"] == K.LEVEL_AUTO
    got = {}
    for form in (K.LEVEL_AUTO, K.LEVEL_FUSED, K.LEVEL_GEMM):
        ev.set_tuning(up_form=form, down_form=form)
        pot, _ = ev.evaluate()
        got[form] = pot, ev.intermediate("uden"), ev.intermediate("dchk"), ev.intermediate("dden")
    tol = O.PARITY_RTOL[np_] if prec == K.PREC_FP64 else 1e-7  # mixed: FP32 roundings flip with the order
    for k, mask in ((0, slice(None)), (1, src & (t["depth"] >= 2)), (2, trg & (t["depth"] >= 2)),
                    (3, trg & (t["depth"] >= 2))):
        a, f, g = (got[form][k][mask] for form in (K.LEVEL_AUTO, K.LEVEL_FUSED, K.LEVEL_GEMM))
        assert np.array_equal(a, f)
        if a.size and np.any(g):
            r = rel(a, g)
            print(f"  {('pot', 'uden', 'dchk', 'dden')[k]}: {r:.2e}", flush=True)
            assert r <= (tol if k == 0 else 1e3 * tol)
