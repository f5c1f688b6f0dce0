"""Handles and trees from pooled streams and memory: a problem built, evaluated
and destroyed again and again, between others of other sizes and on several
threads at once, gives the same tree and the same bits every time."""
import threading

import numpy as np
import pytest

import kifmm_amd as K

pytestmark = pytest.mark.gpu

SIZES = [(3000, "uniform", 4, K.PREC_FP64), (20000, "ellipsoid", 6, K.PREC_FP64), (60000, "gaussmix", 4, K.PREC_MIXED)]


def once(n, dist, np_, prec, new_densities=False):
    p = K.Problem.create(n, dist, 64, np_=np_, seed=n, coincide=0, device=0)
    ev = K.GpuEvaluator(p, precision=prec)
    if new_densities:  # set twice with no evaluation between: the second replaces the first
        den = p.tree()["sden"]
        ev.set_densities(2.0 * den)
        ev.set_densities(den)
    pot = np.array(ev.evaluate()[0])
    tree = p.tree()
    ev.close()
    return pot, tree


def same(a, b):
    assert np.array_equal(a[0], b[0])
    assert all(np.array_equal(a[1][k], b[1][k]) for k in a[1])


def test_rebuilt_between_others():
    first = [once(*s) for s in SIZES]
    for r in range(3):
        for k in (2, 0, 1):
            print(f"case {SIZES[k]} again {r}", flush=True)
            same(once(*SIZES[k], new_densities=r == 1), first[k])


def test_on_several_threads():
    first = [once(*s) for s in SIZES]
    errors = []

    def work(k):
        try:
            for _ in range(4):
                same(once(*SIZES[k]), first[k])
        except BaseException as e:  # noqa: BLE001
            errors.append((k, e))

    threads = [threading.Thread(target=work, args=(k % len(SIZES),)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_release_between_and_beside_others():
    """Idle memory and streams given back between handles, and while handles on
    other threads are built and evaluate: the same bits."""
    first = [once(*s) for s in SIZES]
    K.release_idle()
    errors = []

    def work(k):
        try:
            for _ in range(3):
                same(once(*SIZES[k]), first[k])
                K.release_idle()
        except BaseException as e:  # noqa: BLE001
            errors.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(SIZES))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    K.release_idle()
    same(once(*SIZES[0]), first[0])
