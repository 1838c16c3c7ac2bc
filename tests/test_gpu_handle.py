"""One handle that sees events of very different sizes and kinds: each event's results and what it
costs are those of a handle of its own (MI355X only)."""
import gc

import numpy as np
import pytest

import pyoracle as po
from opticks_amd import configs
from opticks_amd import _lib as L
from opticks_amd.adjoint import yield_jacobian
from opticks_amd.qsim import QSim, SEventConfig

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

DEV = torch.device("cuda:0")


class Device:
    """An event's gensteps and output buffers on the GPU."""

    def __init__(self, gensteps):
        self.gs = torch.from_numpy(np.ascontiguousarray(gensteps, np.float32)).to(DEV)
        self.n = int(np.ascontiguousarray(gensteps, np.float32).view(np.int32)[:, 0, 3].sum())
        self.photon = torch.zeros((self.n, 4, 4), dtype=torch.float32, device=DEV)
        self.seq = torch.zeros((self.n, 2, 2), dtype=torch.int64, device=DEV)
        self.hit = torch.zeros((self.n, 4, 4), dtype=torch.float32, device=DEV)

    def run(self, sim, n_photon=-1, eventID=0):
        for t in (self.photon, self.seq, self.hit):
            t.zero_()
        m = sim.simulate_device(self.gs, self.photon, self.seq, self.hit, eventID=eventID, n_photon=n_photon)
        return [t.cpu().numpy().view(np.uint32).copy() for t in (self.photon, self.seq, self.hit[:m])]


def test_tape_after_a_larger_event():
    """Taped events of unknown size after a larger one without a tape, after a larger taped one and
    in slices: photons and adjoint of a handle that saw nothing else."""
    w = configs.config3(num_gs=6, per_gs=500)
    params = w.meta["params"]
    cfg = dict(seed=w.seed, adjoint_tape=16)
    small, mid = Device(w.gensteps[:2]), Device(w.gensteps)

    def taped(sim, ev, n_photon):
        out = ev.run(sim, n_photon)
        G = yield_jacobian(sim, params, ev.gs, ev.hit, len(out[2]), 2000, n_photon=ev.n)
        return out + [G.cpu().numpy().view(np.uint32)]

    want = {}
    for ev in (small, mid):
        fresh = QSim(w.geometry, w.physics, SEventConfig(**cfg))
        want[ev.n] = taped(fresh, ev, ev.n)
        fresh.close()
    assert want[mid.n][3].any()
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=w.seed))
    Device(configs.config3(num_gs=4, per_gs=100_000).gensteps).run(sim)
    free = torch.cuda.mem_get_info()[0]
    sim.set_config(SEventConfig(**cfg))
    for ev, n_photon in ((small, -1), (mid, -1), (small, -1), (small, small.n), (mid, mid.n)):
        for got, ref in zip(taped(sim, ev, n_photon), want[ev.n]):
            assert np.array_equal(got, ref)
    assert free - torch.cuda.mem_get_info()[0] < 400_000 * 12 * 16 // 2
    sim.set_config(SEventConfig(max_slot=1000, **cfg))
    for got, ref in zip(taped(sim, mid, -1), want[mid.n]):
        assert np.array_equal(got, ref)
    sim.close()


def best_time(f, n=40):
    import time
    best = 1e9
    for _ in range(n):
        t = time.perf_counter()
        f()
        best = min(best, time.perf_counter() - t)
    return best


def test_small_events_after_a_large_one():
    """After an event of 400M photons, events of a few photons have the oracle's results, and do
    not pay for what that one needed."""
    w = configs.config0(num_photon=1000)
    ref = {}
    for n in (1, 64, 1000, 16385, 40001):
        gs = w.gensteps.copy()
        gs.view(np.uint32)[:, 0, 3] = n
        ref[n] = (Device(gs), po.World(w.geometry, w.physics).simulate(gs, event_idx=3, seed=5))
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=5))
    ev = ref[1000][0]
    one = lambda: sim.simulate_device(ev.gs, ev.photon, ev.seq, ev.hit, eventID=3)
    alone = best_time(one)
    big = w.gensteps.copy()
    big.view(np.uint32)[:, 0, 3] = 400_000_000
    photon_t = torch.empty((400_000_000, 4, 4), dtype=torch.float32, device=DEV)
    assert sim.simulate_device(torch.from_numpy(big).to(DEV), photon_t, None, None) > 0
    del photon_t
    torch.cuda.empty_cache()
    after = best_time(one)
    assert after < 2.0 * alone + 50e-6, (alone, after)     # 57 us alone; 350 us when it cleared for 400M
    for n in (40001, 1, 1000, 16385, 64, 40001):
        ev, (photon, seq) = ref[n]
        want = photon[(photon[:, 3, 3].view(np.uint32) & 0x40) != 0]
        got = ev.run(sim, eventID=3)
        assert np.array_equal(got[0], photon.view(np.uint32)) and np.array_equal(got[2], want.view(np.uint32))
        assert np.array_equal(got[1].view(np.uint64).reshape(seq.shape), seq)
    sim.close()


# events smaller and larger than the resident waves hold, on grids of fewer and of more waves
@pytest.mark.parametrize("n", [1, 65, 9001, 200_003, 600_001])
@pytest.mark.parametrize("waves_per_cu", [1, 13, 48])
def test_grids_beyond_residency_keep_results(n, waves_per_cu):
    w = configs.config1(num_gs=1, per_gs=n)
    photon, seq = po.World(w.geometry, w.physics).simulate(w.gensteps, event_idx=2, seed=7)
    ev = Device(w.gensteps)
    for kw in (dict(), dict(block_size=256), dict(adjoint_tape=8)):
        sim = QSim(w.geometry, w.physics, SEventConfig(seed=7, waves_per_cu=waves_per_cu, **kw))
        got = ev.run(sim, eventID=2)
        assert np.array_equal(got[0], photon.view(np.uint32))
        assert np.array_equal(got[1].view(np.uint64).reshape(seq.shape), seq)
        sim.close()


@pytest.mark.parametrize("num_det, n", [(2000, 30_000), (20_000, 30_000), (20_000, 900_000)])
def test_lite_output_of_deep_detectors(num_det, n):
    """Lite records of detectors whose traversal stack leaves a CU fewer blocks with lite output
    than without: time and flags of the photon records, the oracle's among them."""
    w = configs.detector_shell(num_det=num_det, num_gs=6, per_gs=n // 6)
    ev = Device(w.gensteps)
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=w.seed))
    photon = ev.run(sim)[0]
    lite = torch.zeros((ev.n, 4), dtype=torch.int32, device=DEV)
    seq = torch.zeros_like(ev.seq)
    sim.simulate_lite_device(ev.gs, lite, None, seq, None)
    got = lite.cpu().numpy().view(np.uint32)
    assert np.array_equal(got[:, 1], photon[:, 0, 3]) and np.array_equal(got[:, 3], photon[:, 3, 3])
    assert np.array_equal(got[:, 0] & 0xffff, photon[:, 3, 1] & 0xffff)
    assert torch.equal(seq, ev.seq)
    few = w.gensteps[:1].copy()
    few.view(np.uint32)[:, 0, 3] = min(5000, n // 6)
    ref, _ = po.World(w.geometry, w.physics).simulate(few, seed=w.seed)
    assert np.array_equal(photon[:len(ref)], ref.view(np.uint32))
    sim.close()


def mapping_flags(address):
    """VmFlags of the mapping that holds the address"""
    inside = False
    for line in open("/proc/self/smaps"):
        head = line.split()[0]
        if "-" in head and not head.endswith(":"):
            lo, hi = (int(x, 16) for x in head.split("-"))
            inside = lo <= address < hi
        elif inside and line.startswith("VmFlags:"):
            return line.split()[1:]
    raise AssertionError("no such mapping")


@pytest.mark.parametrize("n", [1000, 300_000])
def test_results_are_ordinary_memory(n):
    """Result arrays can be used like any other: a forked child has them (its mappings are not
    those of the GPU's driver), and dropping them during a graph capture leaves it valid."""
    w = configs.config0(num_photon=n)
    photon, seq = po.World(w.geometry, w.physics).simulate(w.gensteps, seed=w.seed)
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=w.seed))
    kept = []
    for _ in range(3):
        sim.simulate(w.gensteps)
        kept.append((sim.photon, sim.seq, sim.hit))
    for arrays in kept:
        assert np.array_equal(arrays[0].view(np.uint32), photon.view(np.uint32)) and np.array_equal(arrays[1], seq)
        for a in arrays:
            assert a.flags.writeable and not {"dc", "io", "pf"} & set(mapping_flags(a.ctypes.data))
    frame = configs.frame_gensteps((0, 0, 0, 500.0), (0, 0, 0, 0, 0, 0, n, 1), gridscale=0.1)
    rays = po.World(w.geometry, w.physics).simtrace(frame, seed=w.seed)
    assert np.array_equal(sim.simtrace(frame).view(np.uint32), rays.view(np.uint32))
    x = torch.zeros(1024, device=DEV)
    sim.photon = sim.seq = sim.hit = None
    del arrays, a
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        y = x + 1
        kept.clear()                                           # nine arrays, more than a handle keeps
        gc.collect()
        z = y + 1
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert z[0].item() == 2.0
    sim.close()


def test_device_times_cover_the_work():
    """The parts of last_timing reach from the first genstep read to the last hit written: the
    compaction takes no less than its records' bytes at the card's nominal 8 TB/s (15 us here; 6.4
    where the tile that ended first but one gave the time), and the total is what events around
    the call see, but for launching and waiting."""
    w = configs.config0(num_photon=1, sensor=True)
    gs = np.repeat(w.gensteps, 40_000, 0)
    gs.view(np.uint32)[:, 0, 3] = 25
    ev = Device(gs)
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=w.seed))
    stream = torch.cuda.Stream()
    parts, rest = [], []
    for i in range(12):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        torch.cuda.synchronize()
        a.record(stream)
        m = sim.simulate_device(ev.gs, ev.photon, ev.seq, ev.hit, eventID=i, stream=stream)
        b.record(stream)
        b.synchronize()
        t = sim.last_timing()
        assert m > 900_000 and 128 * m / 8e9 < t["compact_ms"] < t["total_ms"] < a.elapsed_time(b)
        assert abs(t["seed_ms"] + t["propagate_ms"] + t["compact_ms"] - t["total_ms"]) < 1e-6
        rest.append(a.elapsed_time(b) - t["total_ms"])
    assert sorted(rest)[6] < 0.1
    sim.close()


def same_detector(n, ids):
    hit = torch.zeros((n, 4, 4), dtype=torch.float32, device=DEV)
    hit.view(torch.int32)[:, 3, 1] = ids
    return hit


# detectors on both sides of the bins of one block, chunks of a few hits, and of 65,535 of one
# detector (16,776,960 hits), which fill its half of a word
@pytest.mark.parametrize("n", [1, 1025, 8193, 2_100_001, 16_776_960])
def test_hit_counts_of_busy_detectors(n):
    """However the hits are shared among the detectors, the counts are right, and those of one
    detector take no longer than those of 2,000 (22.7 ms against 0.27 where each hit added to the
    totals)."""
    from opticks_amd.adjoint import hits_per_detector
    g = torch.Generator(device=DEV).manual_seed(n)
    even = torch.randint(0, 2002, (n,), generator=g, dtype=torch.int32, device=DEV)
    shares = {"even": even, "skewed": torch.minimum(even, even // 37 + 1), "one": torch.full_like(even, 2),
              "last": torch.full_like(even, 65535), "all": torch.randint(0, 65536, (n,), generator=g, dtype=torch.int32, device=DEV)}
    times = {}
    for name, ids in shares.items():
        hit = same_detector(n, ids)
        for n_det in (1, 2, 2000, 32767, 32768, 32769, 65534, 65535, 70_000):
            want = torch.zeros(max(n_det, 65535) + 1, dtype=torch.int64, device=DEV)
            want[:65536] = torch.bincount(ids.long(), minlength=65536)
            got = hits_per_detector(hit, n, n_det)
            assert got.shape == (n_det,) and torch.equal(got, want[1:n_det + 1].to(torch.float32)), (name, n_det)
        times[name] = best_time(lambda: (hits_per_detector(hit, n, 2000), torch.cuda.synchronize()), 10)
    assert times["one"] < 2.0 * times["even"] + 100e-6, times


@pytest.mark.parametrize("half, walk", [(2000.0, False), (9000.0, True)])
def test_simtrace_around_the_persistent_kernel(half, walk):
    """Grids of 4M rays that the front instances settle, and that walk: the oracle's records, and
    no step in the time where the choice of a kernel begins (the settled: 1.6 times where it went
    by the number alone)."""
    w = configs.config1(num_gs=1, per_gs=10)
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=9))
    gs = configs.frame_gensteps((0, 0, 0, half), (-50, 49, 0, 0, -20, 19, 1000, 1), gridscale=0.02)
    times = []
    for last in (999, 1000, 1037):                             # 3,999,999, 4,000,000 and 4,000,037 rays
        gs.view(np.uint32)[-1, 0, 3] = last
        gs_t = torch.from_numpy(gs).to(DEV)
        n = 3_999_000 + last
        out_t = torch.empty((n, 4, 4), dtype=torch.float32, device=DEV)
        times.append(best_time(lambda: sim.simtrace_device(gs_t, out_t, n_photon=n), 10))
    ref = po.World(w.geometry, w.physics).simtrace(gs, seed=9)
    out = out_t.cpu().numpy().view(np.uint32)
    assert np.array_equal(out, ref.view(np.uint32))
    instances = out[:, 3, 3] >> 16
    assert (np.count_nonzero(instances[instances != 0xffff]) > 100_000) == walk
    assert max(times[1:]) < 1.3 * times[0] + 30e-6, times
    sim.close()


def test_persistent_simtrace_of_extended_leaves():
    """Rays that walk among hyperboloids and cones around a free ball, enough of them for the
    persistent kernel's instantiation with those leaves."""
    from opticks_amd.foundry import Foundry, Node
    from opticks_amd.physics import BoundaryLib, Material, Surface, gaussian_icdf
    lib = BoundaryLib()
    lib.add_material(Material("Water", 1.33, 20000.0, 30000.0))
    lib.add_material(Material("Acrylic", 1.5, 1e6, 1e6))
    lib.add_surface(Surface("wallSurf", detect=0.5, absorb=0.5))
    b_world = lib.boundary("Water/wallSurf/wallSurf/Water")
    b_obj = lib.boundary("Water///Acrylic")
    fd = Foundry()
    s0 = fd.addSolid("world", [fd.addPrim(Node.box3(13000.0, 13000.0, 13000.0), b_world), fd.addPrim(Node.sphere(5000.0), b_obj)])
    kinds = [fd.addSolid("hyperboloid", [fd.addPrim(Node.hyperboloid(120.0, 160.0, -200.0, 240.0), b_obj)]),
             fd.addSolid("cone", [fd.addPrim(Node.cone(200.0, -100.0, 60.0, 160.0), b_obj)])]
    fd.addInstance(np.eye(4), s0)
    for i, d in enumerate(configs.fibonacci_sphere(400)):
        t = configs.rotation_z_to(-d)
        t[3, :3] = 5500.0 * d
        fd.addInstance(t, kinds[i % 2])
    phys = lib.arrays()
    phys["icdf"], phys["icdf_hd_factor"] = gaussian_icdf()
    gs = configs.frame_gensteps((0, 0, 0, 6000.0), (-50, 49, 0, 0, -20, 20, 1000, 1), gridscale=0.02)
    gs[:, 5, 1] = 3000.0                                       # off the middle: more of them leave the ball
    sim = QSim(fd.arrays(), phys, SEventConfig(seed=3))
    out = sim.simtrace_device(torch.from_numpy(gs).to(DEV)).cpu().numpy().view(np.uint32)
    ref = po.World(fd.arrays(), phys).simtrace(gs, seed=3).view(np.uint32)
    assert np.array_equal(out, ref)
    instances = out[:, 3, 3] >> 16
    assert np.count_nonzero((instances > 0) & (instances != 0xffff)) > 50_000
    sim.close()
