"""What the library's host code takes from the HIP runtime and gives back, and
what it makes of the runtime's errors, on the fake runtime (fake_device.py)."""
import pytest

import fake_device


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = fake_device.build(tmp_path_factory.mktemp("fake"))
    return lambda code: fake_device.run(so, code)


def test_tree_build_that_did_not_end_keeps_nothing(fake):
    """A tree build whose stream cannot be waited for, from any of its waits
    on: its memory and stream are freed, not handed to the next owner."""
    fake("""
    for skip in range(100):
        n0 = fake.fake_calls(b"hipStreamSynchronize")
        fail("hipStreamSynchronize", skip, 1 << 30)
        try:
            K.Problem.create(500, "uniform", 40, np_=3, seed=1, device=0)
        except K.KifmmError:
            pass
        fail("hipStreamSynchronize", 0, 0)
        fake.hipGetLastError()
        failed = fake.fake_calls(b"hipStreamSynchronize") - n0 - skip
        if failed <= 0:
            break  # it has no more waits
        assert fake.fake_streams() == 0, skip
        # (the last wait of all is the stream's own, after one that ended the work on the memory)
        assert fake.fake_used() == 0 or (failed == 1 and skip > 3), (skip, failed, fake.fake_used())
    assert 3 < skip < 99
    """)


def test_idle_memory_and_streams_are_given_back(fake):
    """What handles and tree builds leave for the next ones goes back to the
    runtime on request, whatever handles live; they work on afterwards."""
    fake("""
    prob = K.Problem.create(5000, "ellipsoid", 40, np_=4, seed=1, device=None)
    ops = prob.operators()
    live = K.GpuEvaluator(prob, operators=ops)
    K.release_idle()  # its set-up leaves idle memory too
    used, streams = fake.fake_used(), fake.fake_streams()
    K.Problem.create(5000, "ellipsoid", 40, np_=4, seed=1, device=0)
    K.GpuEvaluator(prob, operators=ops).close()
    assert fake.fake_used() > used and fake.fake_streams() > streams, (fake.fake_used(), used, fake.fake_streams(), streams)
    K.release_idle()
    assert fake.fake_used() == used and fake.fake_streams() == streams, (fake.fake_used(), used, fake.fake_streams(), streams)
    K.release_idle()
    live.evaluate()
    K.GpuEvaluator(prob, operators=ops).close()
    live.close()
    K.release_idle()
    assert fake.fake_used() == 0 and fake.fake_streams() == 0 and fake.fake_events() == 0
    """)


@pytest.mark.parametrize("then", ["K.GpuEvaluator(prob, operators=ops).close()", "build()", "K.release_idle()",
                                  "fake.fake_limit(1 << 14); out_of_memory()"])
def test_device_reset_between_owners(fake, then):
    """hipDeviceReset with no handle alive destroys what is idle: a handle or a
    tree build after it takes nothing of that, and nothing of it is freed
    (runs on the fake runtime only, which lists each use of what is gone)."""
    fake(f"""
    prob = K.Problem.create(5000, "ellipsoid", 40, np_=4, seed=1)
    ops = prob.operators()
    def build():
        K.Problem.create(5000, "ellipsoid", 40, np_=4, seed=1, device=0)
    def out_of_memory():
        try:
            build()
            assert False
        except K.KifmmError:
            pass
    build()
    K.GpuEvaluator(prob, operators=ops).close()
    assert fake.fake_used() > 0 and fake.fake_streams() > 0
    fake.fake_reset()
    {then}
    fake.fake_limit(1 << 40)
    fake.hipGetLastError()
    ev = K.GpuEvaluator(prob, operators=ops)
    ev.evaluate()
    ev.close()
    K.release_idle()
    assert fake.fake_used() == 0 and fake.fake_streams() == 0
    """)


def test_allocation_that_needs_the_idle_memory_leaves_no_error(fake):
    """An allocation that fails until the idle blocks are given back succeeds
    as if it had at once: the runtime's error does not stay for a later launch
    to find."""
    fake("""
    prob = K.Problem.create(60000, "uniform", 64, np_=4, seed=1)
    ops = prob.operators()
    ev = K.GpuEvaluator(prob, operators=ops)
    room = fake.fake_used() + (1 << 20)
    second = K.GpuEvaluator(prob, operators=ops)
    ev.close()
    second.close()
    idle = fake.fake_used()  # of two handles: more than one takes
    fake.fake_limit(room)
    n0 = fake.fake_calls(b"hipFree")
    ev = K.GpuEvaluator(prob, operators=ops)
    assert fake.fake_calls(b"hipFree") > n0, (room, idle, fake.fake_used())  # idle blocks were given back
    ev.evaluate()
    """)


def test_every_allocation_can_have_the_idle_memory(fake):
    """Direct sums and the cost model's network need device memory that only
    the idle blocks hold: they get it."""
    fake("""
    prob = K.Problem.create(60000, "uniform", 64, np_=4, seed=1)
    ops = prob.operators()
    ev = K.GpuEvaluator(prob, operators=ops)
    others = [K.GpuEvaluator(prob, operators=ops) for _ in range(2)]
    t = np.zeros((3, 100000))
    def leave_idle():
        for e in others:
            e.close()
        fake.fake_limit(fake.fake_used())
    leave_idle()
    n0 = fake.fake_calls(b"hipFree")
    ev.direct(*t)
    assert fake.fake_calls(b"hipFree") > n0 + 1
    ev.evaluate()
    fake.fake_limit(1 << 40)
    others = [K.GpuEvaluator(prob, operators=ops) for _ in range(2)]
    leave_idle()
    h, w = C.c_void_p(), (C.c_float * 8192)()
    assert K.lib.kifmm_mlp_create(0, w, C.byref(h)) == 0, K.last_error()
    fake.fake_limit(1 << 40)
    others = [K.GpuEvaluator(prob, operators=ops) for _ in range(2)]
    leave_idle()
    n = 10000
    assert K.lib.kifmm_mlp_predict(h, (C.c_float * (16 * n))(), n, (C.c_float * (4 * n))()) == 0, K.last_error()
    assert K.lib.kifmm_mlp_destroy(h) == 0
    """)


@pytest.mark.parametrize("what", ["hipHostMalloc", "hipHostGetDevicePointer"])
@pytest.mark.parametrize("prec", ["K.PREC_FP64", "K.PREC_MIXED"])
def test_no_pinned_memory_leaves_no_error(fake, what, prec):
    """Without pinned memory, or its device address, a handle is created and
    evaluates, takes densities and sums directly all the same: the runtime's
    error is not left for the next launch check to find."""
    fake(f"""
    prob = K.Problem.create(3000, "ellipsoid", 20, np_=4, seed=1)
    fail({what!r}, 0, 1 << 30, OUT_OF_MEMORY)
    ev = K.GpuEvaluator(prob, precision={prec})
    ev.evaluate()
    assert (ev.output() is None) == ({what!r} == "hipHostMalloc")
    ev.set_densities(prob.tree()["sden"])
    ev.evaluate()
    ev.direct(*np.zeros((3, 5)))
    ev.close()
    K.Problem.create(3000, "ellipsoid", 20, np_=4, seed=1, device=0)
    """)


def test_capture_that_does_not_begin(fake):
    """A graph handle whose capture cannot begin reports it, and is an eager
    handle as before until a later capture succeeds: phase times included."""
    fake("""
    prob = K.Problem.create(3000, "ellipsoid", 20, np_=4, seed=1)
    ev = K.GpuEvaluator(prob, graph=True)
    fail("hipStreamBeginCapture")
    try:
        ev.evaluate()
        assert False
    except K.KifmmError as e:
        assert e.code == -3, e
    fake.hipGetLastError()
    _, t = ev.evaluate_phases(K.PHASE_UP | K.PHASE_V)
    assert t["up"] > 0 and t["v_hadamard"] > 0 and t["total"] >= t["up"] + t["vlist"]
    log()
    _, t = ev.evaluate()
    assert any(ln.startswith("graph") for ln in log()) and t["ulist"] > 0
    """)


@pytest.mark.parametrize("np_,prec", [(3, "K.PREC_FP64"), (4, "K.PREC_FP64"), (6, "K.PREC_FP64"),
                                      (3, "K.PREC_MIXED"), (4, "K.PREC_MIXED")])
def test_hadamard_block_size_that_was_set_is_launched(fake, np_, prec):
    """A block size given to set_tuning is the launched kernel's, on an input
    too small to fill the chip with it; without one the handle picks (2
    here), and a C caller's round trip through get_tuning keeps that."""
    fake(f"""
    ev = K.GpuEvaluator(K.Problem.create(3000, "uniform", 20, np_={np_}, seed=1), precision={prec})
    def launched():
        log()
        ev.evaluate()
        names = [k[4] for k in kernels() if "k_hadamard" in k[4]]
        assert len(names) == 1
        return int(names[0].split(">(")[0].split(",")[-1])
    def auto():
        t = K.GpuTuning()
        K._check(K.lib.kifmm_gpu_get_tuning(ev._h, C.byref(t)))
        return t, (t.hadamard_fb, t.hadamard_auto)
    assert launched() == ev.work_counts()["hadamard_block"] == 2 and auto()[1] == (8, 1)
    for form in (K.HAD_VALU, K.HAD_MFMA):
        for fb in (2, 4, 8, 16):
            ev.set_tuning(K.P2P_STATIC, fb, form)
            assert launched() == ev.work_counts()["hadamard_block"] == fb == ev.tuning()["hadamard_fb"], (form, fb)
            assert auto()[1] == (fb, 0)
    ev.set_tuning(overlap=4)
    t, a = auto()
    assert launched() == 2 and a == (8, 1)
    t.overlap = 0
    K._check(K.lib.kifmm_gpu_set_tuning(ev._h, C.byref(t)))
    assert launched() == 2 and auto()[1] == (8, 1)
    for bad in (K.GpuTuning(0, 8, 1, 0, 0, 0, 2), K.GpuTuning(0, 8, 1, 0, 0, 0, -1), K.GpuTuning(0, 3, 1), K.GpuTuning(0, 1, 1)):
        assert K.lib.kifmm_gpu_set_tuning(ev._h, C.byref(bad)) == -1
    # the autotuner times 2 where the handle would pick it by itself
    fake.fake_kernel_ms(b"k_hadamard", 5.0)
    fake.fake_kernel_ms(b"k_hadamard_{"mfma" if "MIXED" in prec else "fact"}<{np_}, 2>", 0.5)
    best, ms = ev.autotune(reps=1)
    assert (best["hadamard_fb"], best["hadamard_form"]) == (2, K.HAD_MFMA) and launched() == 2 and np.all(ms[3:9] == 5.0)
    """)


def test_hadamard_block_size_on_inputs_that_fill_the_chip(fake):
    """... where the handle picks 8, and the autotuner chooses from 4, 8, 16."""
    fake("""
    ev = K.GpuEvaluator(K.Problem.create(300000, "uniform", 8, np_=4, seed=1))
    assert ev.work_counts()["hadamard_block"] == 8
    fake.fake_kernel_ms(b"k_hadamard", 5.0)
    fake.fake_kernel_ms(b"k_hadamard_fact<4, 2>", 0.5)
    fake.fake_kernel_ms(b"k_hadamard_fact<4, 16>", 4.0)
    best, ms = ev.autotune(reps=1)
    assert best["hadamard_fb"] == 16 == ev.work_counts()["hadamard_block"]
    """)


def test_x_sums_of_their_own_launch_are_xlist_time(fake):
    """Mixed path: the time of the X sums onto check surfaces, launches of
    their own, is X's, not shared out to W; one list alone has all of its time."""
    fake("""
    for n, d in (b"k_wx(", 4.0), (b"k_wx_reduce(", 2.0), (b"k_x_surf(", 1000.0), (b"k_x_surf_reduce(", 500.0):
        fake.fake_kernel_ms(n, d)
    prob = K.Problem.create(20000, "gaussmix", 100, np_=4, seed=1)
    ev = K.GpuEvaluator(prob, precision=K.PREC_MIXED)
    log()
    _, t = ev.evaluate()
    names = " ".join(k[4] for k in kernels())
    surf = 1000.0 + (500.0 if "k_x_surf_reduce" in names else 0.0)
    assert "k_x_surf(" in names and "k_wx(" in names
    assert surf <= t["xlist"] <= surf + 6.0 and 0.0 < t["wlist"] < 6.0, t
    assert t["wlist"] + t["xlist"] == surf + 6.0
    _, t = ev.evaluate_phases(K.PHASE_UP | K.PHASE_W)
    assert (t["wlist"], t["xlist"]) == (6.0, 0.0)
    _, t = ev.evaluate_phases(K.PHASE_UP | K.PHASE_X)
    assert (t["wlist"], t["xlist"]) == (0.0, surf + 6.0)
    """)


@pytest.mark.parametrize("prec", ["K.PREC_FP64", "K.PREC_MIXED"])
def test_large_early_chunks_are_copied_beside_the_later_ones(fake, prec):
    """Stream layouts with some U-list chunks early, a million targets or more
    of them: their potentials go to the host on a stream that runs no U-list,
    so that the later chunks do not wait for PCIe; whole and once, whatever
    buffer the caller gave.  Fewer: the join writes them, and no copy is made."""
    fake(f"""
    for n, large in ((3600000, (2, 3, 5, 6)), (2200000, (3, 6)), (280000, ())):
        prob = K.Problem.create(n, "uniform", 512, np_=3, seed=1)
        ev = K.GpuEvaluator(prob, precision={prec})
        own = np.zeros(ev.n_trg)
        for layout in range(7):
            ev.set_tuning(overlap=layout)
            for into in (False, True):
                log()
                ev.evaluate_into(own) if into else ev.evaluate(copy="view")
                lines = log()
                copies = [ln.split() for ln in lines if ln.startswith("copy")]
                if layout not in large:
                    assert not copies, (layout, copies)
                    continue
                early = sum(int(c[3]) for c in copies)
                assert len(copies) == (1 if layout in (2, 5) else 2) and all(c[2] == "d2h" for c in copies), copies
                assert 8 << 20 <= early < 8 * ev.n_trg
                u = [ln.split()[1] for ln in lines if "k_p2p" in ln or "k_join_pot" in ln]
                assert len(u) >= 3 and all(c[1] not in u for c in copies), (u, copies)
                at = [ln for ln in lines if "k_join_pot" in ln or " d2h " in ln or "k_p2p" in ln]
                assert "k_join_pot" in at[1] and all(" d2h " in ln for ln in at[2 : 2 + len(copies)])  # before the later chunks
        ev.close()
    K.release_idle()
    assert fake.fake_streams() == 0 and fake.fake_events() == 0
    """)


@pytest.mark.parametrize("n,pinned", [(1000, True), (1 << 20, True), ((1 << 20) + 1, False), (2000000, False)])
def test_route_of_new_densities(fake, n, pinned):
    """Up to a million sources the packing kernel reads pinned memory; beyond,
    the runtime's copy, waited for: there the pinned route is the slower one."""
    fake(f"""
    prob = K.Problem.create({n}, "uniform", 512, np_=3, seed=1, coincide=1)
    ev = K.GpuEvaluator(prob)
    den = np.zeros({n})
    ev.set_densities(den)
    log()
    ev.set_densities(den)
    lines = log()
    assert sum("k_set_w" in ln for ln in lines) == 1
    assert [ln.split()[2:] for ln in lines if ln.startswith("copy")] == ([] if {pinned} else [["h2d", "{8 * n}"]]), lines
    """)
