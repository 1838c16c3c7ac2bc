"""The propagation kernels' launch shapes against the CPU checker (MI355X only): geometries
whose traversal stack is far deeper than a detector's, which changes the LDS of a block."""
import numpy as np
import pytest

import pyoracle as po
from opticks_amd import configs
from opticks_amd import _lib as L
from opticks_amd.foundry import Foundry, Node
from opticks_amd.physics import BoundaryLib, Material, Surface, gaussian_icdf
from opticks_amd.qsim import QSim, SEventConfig

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)


def onions(shells, num_photon=20_000, seed=42):
    """Two instances of a solid of concentric spheres, radii growing by 11%, in a water box:
    each SAH split of such a solid takes the largest sphere off, so its BLAS is a chain and
    the traversal stack holds about one entry a shell."""
    lib = BoundaryLib()
    lib.add_material(Material("Water", 1.33, 20000.0, 30000.0))
    lib.add_material(Material("Acrylic", 1.36, 1e6, 1e6))
    lib.add_surface(Surface("wallSurf", detect=0.5, absorb=0.5))
    b_world = lib.boundary("Water/wallSurf/wallSurf/Water")
    b_obj = lib.boundary("Water///Acrylic")
    fd = Foundry()
    s0 = fd.addSolid("world", [fd.addPrim(Node.box3(6000.0, 6000.0, 6000.0), b_world)])
    s1 = fd.addSolid("onion", [fd.addPrim(Node.sphere(10.0 * 1.11 ** k), b_obj) for k in range(shells)])
    fd.addInstance(np.eye(4), s0)
    for x in (-1100.0, 1100.0):
        t = np.eye(4)
        t[3, 0] = x
        fd.addInstance(t, s1)
    phys = lib.arrays()
    phys["icdf"], phys["icdf_hd_factor"] = gaussian_icdf()
    gs = np.stack([configs.torch_genstep(num_photon // 2, configs.T_POINT_ISO, pos=p, wavelength=300.0, weight=300.0)
                   for p in ((0.0, 0.0, 0.0), (-1100.0, 3.0, 2.0))]).astype(np.float32)
    return configs.Workload("onions", fd.arrays(), phys, gs, seed=seed)


# 3 shells: a shallow stack; 40: 27 + 41 words a lane, past 64 KB for a 256-thread block
@pytest.mark.parametrize("shells", [3, 40])
@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("kernel", [L.MI_KERNEL_PLAIN, L.MI_KERNEL_WAVEFRONT])
def test_stack_depths_match_checker(shells, block, kernel):
    w = onions(shells)
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=w.seed, block_size=block, kernel=kernel))
    hits = sim.simulate(w.gensteps, 0)
    photon, seq = po.World(w.geometry, w.physics).simulate(w.gensteps, seed=w.seed)
    assert np.array_equal(sim.seq, seq)
    assert np.array_equal(sim.photon.view(np.uint32), photon.view(np.uint32))
    assert len(hits) == np.count_nonzero(photon[:, 3, 3].view(np.uint32) & 0x40)
    sim.close()


def front_world(kind, num_photon=40_000, seed=42):
    """A world solid of several large prims tested ahead of the TLAS, with eight small spheres
    inside it. `plain`: leaves of every type the scalar front test takes, one of them under a
    node transform; `tree`: also a Boolean tree, which sends the front solid down the general
    path."""
    from opticks_amd.foundry import CSG_DIFFERENCE
    lib = BoundaryLib()
    lib.add_material(Material("Water", 1.33, 20000.0, 30000.0))
    lib.add_material(Material("Acrylic", 1.50, 1e6, 1e6))
    lib.add_surface(Surface("wallSurf", detect=0.5, absorb=0.5))
    b_world = lib.boundary("Water/wallSurf/wallSurf/Water")
    b_obj = lib.boundary("Water///Acrylic")
    fd = Foundry()
    tilted = Node.cylinder(2500.0, -2500.0, 2500.0)
    tilted.transform = configs.rotation_z_to([0.3, -0.5, 0.81])
    tilted.transform[3, :3] = (40.0, -60.0, 20.0)
    prims = [fd.addPrim(Node.box3(9000.0, 9000.0, 9000.0), b_world), fd.addPrim(tilted, b_obj),
             fd.addPrim(Node.zsphere(2300.0, -1900.0, 2100.0), b_obj), fd.addPrim(Node.sphere(1500.0), b_obj)]
    if kind == "tree":
        prims.append(fd.addPrim(Node.op(CSG_DIFFERENCE, Node.sphere(1300.0), Node.sphere(1200.0)), b_obj))
    s0 = fd.addSolid("world", prims)
    s1 = fd.addSolid("ball", [fd.addPrim(Node.sphere(150.0), b_world)])
    fd.addInstance(np.eye(4), s0)
    for k in range(8):
        t = np.eye(4)
        t[3, :3] = [(800.0 if k >> a & 1 else -700.0) for a in range(3)]
        fd.addInstance(t, s1, sensor_identifier=k, sensor_index=k)
    phys = lib.arrays()
    phys["icdf"], phys["icdf_hd_factor"] = gaussian_icdf()
    gs = np.stack([configs.torch_genstep(num_photon // 2, configs.T_POINT_ISO, pos=p, wavelength=300.0, weight=300.0)
                   for p in ((0.0, 0.0, 0.0), (30.0, -2900.0, 100.0))]).astype(np.float32)
    return configs.Workload("front_world", fd.arrays(), phys, gs, seed=seed)


@pytest.mark.parametrize("kind", ["plain", "tree"])
def test_front_solids_match_checker(kind):
    w = front_world(kind)
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=w.seed))
    sim.simulate(w.gensteps, 0)
    photon, seq = po.World(w.geometry, w.physics).simulate(w.gensteps, seed=w.seed)
    assert np.array_equal(sim.seq, seq)
    assert np.array_equal(sim.photon.view(np.uint32), photon.view(np.uint32))
    sim.close()


# the smallest events (one wave, partly filled), a wave and a lane, and enough photons for
# refills to mix lanes that wait for the instance walk with fresh ones
@pytest.mark.parametrize("n", [1, 63, 65, 4097, 600_001])
@pytest.mark.parametrize("batch", [1, 16, 64])
def test_waiting_lanes_keep_results(n, batch):
    w = configs.config1(num_gs=1, per_gs=n)
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=7, refill_batch=batch))
    sim.simulate(w.gensteps, 3)
    photon, seq = po.World(w.geometry, w.physics).simulate(w.gensteps, event_idx=3, seed=7)
    assert np.array_equal(sim.seq, seq)
    assert np.array_equal(sim.photon.view(np.uint32), photon.view(np.uint32))
    sim.close()


# gensteps on either side of what one block prefixes by itself, some without photons; photon
# counts around a compaction tile (16,384 photons)
@pytest.mark.parametrize("n_gs, total", [(1, 16384), (2047, 16385), (2048, 32767), (2049, 32768), (5000, 40001)])
def test_event_setup_and_compaction_match_checker(n_gs, total):
    g = np.random.default_rng(n_gs)
    counts = np.zeros(n_gs, np.int64)
    some = g.choice(n_gs, max(1, n_gs // 2), replace=False)
    counts[some] = g.multinomial(total, np.full(len(some), 1.0 / len(some)))
    w = configs.config0(num_photon=100)
    one = configs.torch_genstep(1, configs.T_POINT_ISO, wavelength=300.0, weight=200.0)
    gs = np.repeat(one[None], n_gs, 0).astype(np.float32)
    gs[:, 1, :3] = g.uniform(-300, 300, (n_gs, 3))
    gs.view(np.uint32)[:, 0, 3] = counts
    photon, seq = po.World(w.geometry, w.physics).simulate(gs, event_idx=2, seed=5)
    want = photon[(photon[:, 3, 3].view(np.uint32) & 0x40) != 0]
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=5))
    dev = torch.device("cuda:0")
    small = torch.from_numpy(w.gensteps).to(dev)
    gs_t = torch.from_numpy(gs).to(dev)
    photon_t = torch.zeros((total, 4, 4), dtype=torch.float32, device=dev)
    seq_t = torch.zeros((total, 2, 2), dtype=torch.int64, device=dev)
    hit_t = torch.zeros((total, 4, 4), dtype=torch.float32, device=dev)
    # a first event smaller than the one that follows: its buffers have to grow
    assert sim.simulate_device(small, photon_t, seq_t, hit_t) <= 100
    for n_photon in (-1, total):
        photon_t.zero_()
        hit_t.zero_()
        m = sim.simulate_device(gs_t, photon_t, seq_t, hit_t, eventID=2, n_photon=n_photon)
        assert m == len(want)
        assert np.array_equal(photon_t.cpu().numpy().view(np.uint32), photon.view(np.uint32))
        assert np.array_equal(seq_t.cpu().numpy().view(np.uint64), seq)
        assert np.array_equal(hit_t.cpu().numpy()[:m].view(np.uint32), want.view(np.uint32))
    # refused on the device: nothing is written, and the next event is not disturbed
    photon_t.zero_()
    with pytest.raises(RuntimeError):
        sim.simulate_device(gs_t, photon_t, seq_t, hit_t, eventID=2, n_photon=total + 1)
    assert not photon_t.any()
    assert sim.simulate_device(gs_t, photon_t, seq_t, hit_t, eventID=2) == len(want)
    # a short hit buffer: the count is still reported, the hits that fit are in it
    with pytest.raises(RuntimeError):
        sim.simulate_device(gs_t, photon_t, seq_t, hit_t[:7], eventID=2)
    assert np.array_equal(hit_t.cpu().numpy()[:7].view(np.uint32), want[:7].view(np.uint32))
    sim.close()


def test_event_arrays_are_their_own():
    """Result arrays keep their values over later events, a reset and the handle's end, and
    memory of dropped ones is used again, a bounded number of buffers of it."""
    w = configs.config0(num_photon=1000)
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=1))
    kept = []
    for e in range(5):
        hit = sim.simulate(w.gensteps, e)
        kept.append((hit, sim.photon, sim.seq, hit.copy(), sim.photon.copy(), sim.seq.copy()))
    sim.photon[0] = 0.0                                    # writable, and nobody else's
    kept[-1][4][0] = 0.0
    sim.reset()
    for e in range(20):
        sim.simulate(w.gensteps, 100 + e)                  # the arrays of the event before are dropped
    assert len(sim._host._spare) <= sim._host.most
    sim.close()
    assert not sim._host._spare
    for hit, photon, seq, hit0, photon0, seq0 in kept:
        assert np.array_equal(hit.view(np.uint32), hit0.view(np.uint32))
        assert np.array_equal(photon.view(np.uint32), photon0.view(np.uint32))
        assert np.array_equal(seq, seq0)


# fewer rays than lanes, around a wave, and enough for the persistent kernel, with and without a
# whole number of its claims of 256
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 4099, 700_001, 3_999_999, 4_000_000, 4_000_037])
@pytest.mark.parametrize("world", ["shell", "plain", "tree", "onions", "zoo"])
def test_simtrace_queue_matches_checker(world, n):
    """Rays that the front instances settle, that wait for the walk and for the leaf phase, and
    that miss everything, with gensteps of uneven size, some without rays."""
    w = {"shell": lambda: configs.config1(num_gs=1, per_gs=10), "plain": lambda: front_world("plain", 10),
         "tree": lambda: front_world("tree", 10), "onions": lambda: onions(12, 10),
         "zoo": lambda: configs.leaf_zoo(num_photon=10)}[world]()
    g = np.random.default_rng(n)
    n_gs = 5 if n < 1000 else 301
    counts = np.zeros(n_gs, np.int64)
    some = g.choice(n_gs, n_gs // 2, replace=False)
    counts[some] = g.multinomial(n, np.full(len(some), 1.0 / len(some)))
    extent = 20000.0 if world == "shell" else 1000.0
    gs = np.repeat(configs.frame_gensteps((0, 0, 0, extent), (0, 0, 0, 0, 0, 0, 1, 1), gridscale=1.0), n_gs, 0)
    gs[:, 5, :3] = g.uniform(-extent, extent, (n_gs, 3))
    gs.view(np.uint32)[:, 0, 1] = g.integers(0, 4, n_gs)
    gs.view(np.uint32)[:, 0, 3] = counts
    ref = po.World(w.geometry, w.physics).simtrace(gs, seed=9)
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=9))
    gs_t = torch.from_numpy(gs).to("cuda:0")
    for _ in range(2):
        out = sim.simtrace_device(gs_t).cpu().numpy()
        assert out.shape == ref.shape == (n, 4, 4)
        assert np.array_equal(out.view(np.uint32), ref.view(np.uint32))
    sim.close()
