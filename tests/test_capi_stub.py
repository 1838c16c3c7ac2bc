"""Host logic of the C-ABI runtime (oa_capi.cpp) on the CPU: compiled with g++ against stand-ins
for the HIP runtime and the kernel launchers (tests/cpp/capi_stub.cpp), which fail allocations on
request and check every launch's buffers."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from opticks_amd import _lib as L
from opticks_amd import configs
from opticks_amd.qsim import QSim, SEventConfig

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "opticks_amd", "csrc")


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("no g++ or no HIP headers")
    out = tmp_path_factory.mktemp("stub") / "libcapi_stub.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", CSRC,
                    "-I/opt/rocm/include", os.path.join(CSRC, "oa_capi.cpp"),
                    os.path.join(ROOT, "tests", "cpp", "capi_stub.cpp"), "-Wl,-Bsymbolic", "-o", str(out)], check=True)
    return str(out)


@pytest.fixture
def stub(built, monkeypatch):
    monkeypatch.setattr(L, "LIBPATH", built)
    monkeypatch.setattr(L, "_lib", None)
    lib = L.lib()
    lib.stub_limit.argtypes = [L.C.c_size_t]
    lib.stub_largest.restype = L.C.c_size_t
    lib.stub_reset()
    yield lib
    assert lib.stub_bad() == 0


def event(n):
    return configs.config0(num_photon=n).gensteps


def sim_of(**kw):
    w = configs.config0(num_photon=1)
    return QSim(w.geometry, w.physics, SEventConfig(seed=1, **kw))


def test_outputs_follow_the_handles_mask(stub):
    """simulate() gives the arrays that the handle was configured for, also where the caller's
    config object changed since, or the handle was configured by set_config_c."""
    sim = sim_of()
    sim.config.output_mask = L.MI_OUT_HIT                      # changed, not applied
    assert len(sim.simulate(event(100))) == 50
    assert sim.photon.shape == (100, 4, 4) and sim.seq.shape == (100, 2, 2)
    assert np.array_equal(sim.photon[:, 0, 0], np.arange(100)) and np.array_equal(sim.seq[:, 0, 0], np.arange(100))
    sim.config.output_mask = L.MI_OUT_PHOTON | L.MI_OUT_SEQ | L.MI_OUT_HIT
    c = sim.get_config_c()
    c.output_mask = L.MI_OUT_HIT
    sim.set_config_c(c)
    assert np.array_equal(sim.simulate(event(100))[:, 0, 0], np.arange(1, 100, 2))
    assert sim.photon is None and sim.seq is None
    sim.config.output_mask = L.MI_OUT_PHOTON
    assert sim.simulate(event(100)) is None
    sim.close()


def run_device(lib, sim, gs, n_photon=-1, n_alloc=None):
    """mi_sim_simulate_device over host arrays: (return code, hits)"""
    n = int(gs[:, 0, 3].view(np.int32).sum()) if n_alloc is None else n_alloc
    photon = np.zeros((n, 4, 4), np.float32)
    hit = np.zeros((n, 4, 4), np.float32)
    m = L.C.c_int64(-1)
    rc = lib.mi_sim_simulate_device(sim.handle, 0, gs.ctypes.data, len(gs), n_photon, 0, photon.ctypes.data, None,
                                    hit.ctypes.data, n, L.C.byref(m), None)
    return rc, m.value


@pytest.mark.parametrize("grow", ["event", "batch"])
@pytest.mark.parametrize("known", [True, False])
def test_event_after_a_failed_allocation(stub, grow, known):
    """An event or a batch too large for the memory fails with an error; the events after it get
    buffers that hold them."""
    sim = sim_of()
    small, large = event(1000), event(1_000_000)
    assert run_device(stub, sim, small) == (0, 500)
    for limit in (100_000, 1_000_000, 3_900_000):
        stub.stub_limit(limit)                         # the first, second, ... buffer cannot grow
        if grow == "event":
            rc, _ = run_device(stub, sim, large, n_photon=1_000_000)
        else:
            ev, off, po, ho = (np.array(a, t) for a, t in (([0], np.int32), ([0, 1], np.int64), ([0, 0], np.int64),
                                                           ([0, 0], np.int64)))
            rc = stub.mi_sim_simulate_batch_device(sim.handle, 1, ev.ctypes.data, off.ctypes.data, large.ctypes.data,
                                                   po.ctypes.data, None, None, None, 0, ho.ctypes.data, None)
        assert rc < 0 and "stub" in L.last_error()
        assert run_device(stub, sim, small, n_photon=1000 if known else -1) == (0, 500)
        assert stub.stub_bad() == 0
    stub.stub_reset()
    assert run_device(stub, sim, large) == (0, 500_000)
    sim.close()


@pytest.mark.parametrize("n_photon", [1001, 10 ** 6, 10 ** 12])
@pytest.mark.parametrize("tape", [0, 32])
def test_too_many_photons_are_refused_without_buffers_for_them(stub, n_photon, tape):
    sim = sim_of(adjoint_tape=tape)
    for first in (False, True):
        stub.stub_reset()
        rc, m = run_device(stub, sim, event(1000), n_photon=n_photon, n_alloc=1000)
        assert rc == -1 and m == 0 and f"n_photon {n_photon} exceeds the gensteps' 1000 photons" in L.last_error()
        assert stub.stub_largest() < 1001 * 12 * max(tape, 1) + 4096
        assert run_device(stub, sim, event(1000)) == (0, 500)
    sim.close()


def test_tape_of_an_event_of_unknown_size_is_its_own(stub):
    """The adjoint tape of a small event after a large one without a tape is as large as the
    small event needs."""
    sim = sim_of()
    assert run_device(stub, sim, event(1_000_000)) == (0, 500_000)
    sim.config.adjoint_tape = 32
    sim.set_config(sim.config)
    stub.stub_reset()
    for n in (1000, 3000, 500, 3000):
        assert run_device(stub, sim, event(n)) == (0, n // 2)
        assert stub.stub_bad() == 0 and stub.stub_largest() <= 3000 * 32 * 12
        assert stub.stub_tape_stride() in (0, n)           # 0: the launch's own photon count
    sim.config.adjoint_tape = 64                           # records of the same tape, more of them
    sim.set_config(sim.config)
    assert run_device(stub, sim, event(3000)) == (0, 1500)
    assert run_device(stub, sim, event(1_300_000)) == (0, 650_000)    # buffers, and what the host reads, move
    sim.config.max_slot = 2000                             # slices of one event: the event's count
    sim.set_config(sim.config)
    gs = np.concatenate([event(1500), event(1000), event(700)])
    assert run_device(stub, sim, gs) == (0, 750 + 500 + 350)
    assert stub.stub_tape_stride() == 3200
    sim.close()


@pytest.mark.parametrize("waves_per_cu", [0, 3, 8, 64])
def test_first_photons_are_dealt_to_resident_waves(stub, waves_per_cu):
    """Photons dealt out by position go to waves that start at once: the grid has no more waves
    than fit the GPU (2 CUs of stub_resident() one-wave blocks, one fewer with lite output)."""
    sim = sim_of(waves_per_cu=waves_per_cu)
    gs = event(1000)
    lite = np.zeros((1000, 4), np.uint32)
    m = L.C.c_int64(0)
    for is_lite, fit in ((False, stub.stub_resident()), (True, stub.stub_resident_lite())):
        if is_lite:
            assert stub.mi_sim_simulate_lite_device(sim.handle, 0, gs.ctypes.data, 1, -1, 0, lite.ctypes.data, None, None,
                                                    None, 0, L.C.byref(m), None) == 0
        else:
            assert run_device(stub, sim, gs) == (0, 500)
        assert stub.stub_grid() == stub.stub_waves_dealt() == 2 * min(waves_per_cu or fit, fit)
    queries = stub.stub_queries()
    for _ in range(3):                                         # asked once for each kernel
        assert run_device(stub, sim, gs) == (0, 500)
        assert stub.mi_sim_simulate_lite_device(sim.handle, 0, gs.ctypes.data, 1, -1, 0, lite.ctypes.data, None, None, None, 0,
                                                L.C.byref(m), None) == 0
    assert stub.stub_queries() == queries
    sim.close()


@pytest.mark.parametrize("n", [1, 4096, 30_011, 120_000])
def test_results_are_ordinary_memory(stub, n):
    """Results that outlive a call are not in memory of the HIP runtime, whose mappings a forked
    child does not have and which cannot be freed during a graph capture; copied in pieces of all
    sizes, also where the pieces' pinned memory cannot be had."""
    stub.stub_known.argtypes = [L.C.c_void_p]
    sim = sim_of()
    gs = event(n)
    for limited in (False, True):
        hit = sim.simulate(gs)
        for a in (sim.photon, sim.seq) + ((hit,) if len(hit) else ()):
            assert not stub.stub_known(a.ctypes.data)
        assert np.array_equal(sim.photon[:, 0, 0], np.arange(n)) and np.array_equal(sim.seq[:, 0, 0], np.arange(n))
        assert np.array_equal(hit[:, 0, 0], 2 * np.arange(n // 2) + 1)
        out = L.MiEventOut()
        assert stub.mi_sim_simulate(sim.handle, 0, gs.ctypes.data, len(gs), L.C.byref(out)) == 0
        assert not any(stub.stub_known(p) for p in (out.photon, out.seq, out.hit))
        got = np.ctypeslib.as_array((L.C.c_float * (16 * n)).from_address(out.photon)).reshape(n, 4, 4)
        assert np.array_equal(got, sim.photon)
        sim.close()
        sim = sim_of()
        stub.stub_limit(max(64 * n, 3 << 20))                  # too little for the ring, but for the last n
    sim.close()


def test_fetch_into_pinned_and_ordinary_memory(stub):
    n = 50_000
    sim = sim_of()
    gs = event(n)
    out = L.MiEventOut()
    assert stub.mi_sim_run(sim.handle, 0, gs.ctypes.data, len(gs), L.C.byref(out)) == 0
    p = L.C.c_void_p()
    assert stub.mi_host_alloc(64 * n, L.C.byref(p)) == 0 and stub.stub_known(p)
    seq = np.zeros((n, 2, 2), np.uint64)
    assert stub.mi_sim_fetch(sim.handle, p, seq.ctypes.data, None) == 0
    got = np.ctypeslib.as_array((L.C.c_float * (16 * n)).from_address(p.value)).reshape(n, 4, 4)
    assert np.array_equal(got[:, 0, 0], np.arange(n)) and np.array_equal(seq[:, 0, 0], np.arange(n))
    stub.mi_host_free(p)
    sim.close()


def test_spare_memory_follows_the_events(stub, monkeypatch):
    """Memory kept for later events is bounded in buffers and bytes, and after large events many
    small ones find theirs in it; where memory is short it is given up for the arrays asked for."""
    sim = sim_of()
    pool = sim._host
    kept = []
    for _ in range(4):
        sim.simulate(event(100_000))
        kept.append((sim.photon, sim.seq, sim.hit))
    kept.clear()
    sim.simulate(event(100_000))
    assert 0 < len(pool._spare) <= pool.most
    for _ in range(20):
        sim.simulate(event(1000))
    sizes = lambda: [m.nbytes for _, m in pool._spare]
    assert 0 < len(pool._spare) <= pool.most and max(sizes()) <= 64 * 1000
    before = {m.ctypes.data for _, m in pool._spare}
    sim.simulate(event(1000))
    assert {a.ctypes.data for a in (sim.photon, sim.seq, sim.hit)} <= before
    sim.simulate(event(100_000))
    monkeypatch.setattr(type(pool), "most_bytes", 64 * 100_000 - 1)
    sim.simulate(event(1000))
    assert sum(sizes()) < 64 * 100_000
    empty, failures = np.empty, []

    def short_of_memory(size, dtype):
        if pool._spare:
            failures.append(size)
            raise MemoryError
        return empty(size, dtype)

    monkeypatch.setattr("opticks_amd.qsim.np.empty", short_of_memory)
    assert len(sim.simulate(event(400_000))) == 200_000 and failures
    monkeypatch.undo()
    sim.photon = sim.seq = sim.hit = None
    stub.mi_sim_destroy(sim.handle)
    sim.handle = None


def test_fetch_after_a_failed_simtrace(stub):
    """A simtrace that fails has used the photon buffer of the run before it: that run's outputs
    cannot be fetched any more, as after one that succeeds."""
    sim = sim_of()
    gs = event(1000)
    out = L.MiEventOut()
    photon = np.zeros((1000, 4, 4), np.float32)
    frame = configs.frame_gensteps((0, 0, 0, 100.0), (0, 0, 0, 0, 0, 0, 1000, 1))
    for fails in (True, False):
        assert stub.mi_sim_run(sim.handle, 0, gs.ctypes.data, 1, L.C.byref(out)) == 0
        assert stub.mi_sim_fetch(sim.handle, photon.ctypes.data, None, None) == 0
        stub.stub_fail_trace(int(fails))
        if fails:
            with pytest.raises(RuntimeError):
                sim.simtrace(frame)
        else:
            assert len(sim.simtrace(frame)) == 1000
        assert stub.mi_sim_fetch(sim.handle, photon.ctypes.data, None, None) == -1
        assert "no such output" in L.last_error()
    sim.close()


def test_calls_sharing_the_noalloc_scratch_take_turns(stub):
    """All no-allocation calls on a GPU share its scratch, in which the compaction of one waits for
    counts that the clearing of another would take away: they run one after the other."""
    import threading
    gs = event(1000)
    rcs = []

    def calls():
        sim = sim_of()
        m = L.C.c_int64(0)
        for _ in range(3):
            rcs.append(stub.mi_sim_simulate_device_noalloc(sim.handle, 0, gs.ctypes.data, 1, -1, 0, None, None, None, 0,
                                                           L.C.byref(m), None))
            assert m.value == 500
        sim.close()

    threads = [threading.Thread(target=calls) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert rcs == [0] * 12 and stub.stub_overlap() == 0


def test_a_refused_call_keeps_the_tape(stub):
    """A call refused for its photon count has propagated nothing: the adjoint of the event before
    it still finds that event's tape."""
    from opticks_amd.adjoint import LengthParams
    w = configs.config0(num_photon=1)
    params = LengthParams(w.physics, ("Water",), n_bin=4)
    adj = params.c_struct(1)
    grad = np.zeros((1, params.n_param), np.float32)
    sim = sim_of(adjoint_tape=4)
    gs, other = event(2000), event(1500)

    def adjoint_has_tape():
        assert stub.mi_sim_adjoint_device(sim.handle, 0, gs.ctypes.data, 1, 2000, 0, None, 0, L.C.byref(adj), grad.ctypes.data,
                                          None) == 0
        return stub.stub_adjoint_tape()

    assert run_device(stub, sim, gs) == (0, 1000) and adjoint_has_tape()
    for n_photon, g in ((2001, gs), (1600, other), (10 ** 9, other)):
        rc, _ = run_device(stub, sim, g, n_photon=n_photon, n_alloc=2000)
        assert rc == -1 and adjoint_has_tape()
    assert run_device(stub, sim, event(0), n_alloc=1) == (1, 0) and adjoint_has_tape()
    assert run_device(stub, sim, other) == (0, 750) and not adjoint_has_tape()
    assert run_device(stub, sim, gs) == (0, 1000) and adjoint_has_tape()
    sim.close()
