"""
Timed workloads of the propagation path, through the public entry points of `opticks_amd`.

A case is a dict of plain values; `kind` names the call a program makes:

  event           QSim.simulate_device: one event, gensteps and outputs resident on the GPU
  host_event      QSim.simulate: one event, host gensteps in, host photons / histories / hits out
  lite_merge      QSim.simulate_lite_device, then QSim.merge_hits_device of the lite records
  batch           Batch.launch / wait: many events replayed from one captured graph
  gradient        expected_hits(theta) and its backward: one step of a fit of optical lengths
  batch_gradient  the captured graph with the yield adjoint of all its hits
  simtrace        QSim.simtrace_device: rays of a planar grid through the geometry
  merge           QSim.merge_hits_device of full photon records

`world` names the geometry: a water sphere in a detecting box, a liquid-scintillator sphere
with `n_det` CSG detectors around it (`shell`), or one of the shape and surface collections.
`source` names the gensteps: isotropic torch points, scintillation steps, Cerenkov steps, or
a charged track's alternating Cerenkov and scintillation steps.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from opticks_amd import configs
from opticks_amd import _lib as L
from opticks_amd.adjoint import LengthParams, expected_hits, perturbed_theta
from opticks_amd.qsim import FLAG, QSim, SEventConfig

DEV = "cuda:0"
ZOOS = {"leaf_zoo": configs.leaf_zoo, "boolean_zoo": configs.boolean_zoo, "list_zoo": configs.list_zoo}
TAPE = 32            # segment records per photon: at least max_bounce, so no photon is replayed


def listed():
    return [
        # a single calibration point: launches and waits are what counts
        dict(name="torch_1k", kind="event", world="water_sphere", source="torch", n_gs=1, n_photon=1000),
        # one low-energy particle in a detector: some ten thousand photons over a few dozen steps
        dict(name="track_12k", kind="event", world="shell", n_det=2000, source="track", n_gs=48, n_photon=12347),
        # one event of a large detector
        dict(name="scint_1M", kind="event", world="shell", n_det=20000, source="scint", n_gs=200, n_photon=1_000_003),
        # the calibration workload: 1,000 torch points in the scintillator ball
        dict(name="torch_10M", kind="event", world="shell", n_det=2000, source="torch", n_gs=1000, n_photon=10_000_000),
        # cones, hyperboloids, polyhedra and phi cuts; the xorwow generator
        dict(name="zoo_200k", kind="event", world="leaf_zoo", source="torch", n_gs=4, n_photon=200_000, rng="xorwow"),
        # the service call: host arrays in and out, as a Geant4 program makes it
        dict(name="host_300k", kind="host_event", world="shell", n_det=2000, source="track", n_gs=400, n_photon=300_007),
        # compact output and hit merging of a bright event
        dict(name="lite_merge_3M", kind="lite_merge", world="shell", n_det=2000, source="track", n_gs=700,
             n_photon=3_000_017, window=1.0),
        # production: a batch of events in one replay
        dict(name="batch_64", kind="batch", world="shell", n_det=20000, n_event=64, mean_gs=200, mean_photons=5000),
        # one step of a fit of 256 optical lengths to one event's yields
        dict(name="gradient_1M", kind="gradient", world="shell", n_det=2000, source="torch", n_gs=100,
             n_photon=1_000_000, n_bin=64),
        # the same over a batch of events, in one replay
        dict(name="batch_gradient_16", kind="batch_gradient", world="shell", n_det=20000, n_event=16, mean_gs=200,
             mean_photons=5000, n_bin=64),
        # a cross-section picture of the geometry
        dict(name="simtrace_10M", kind="simtrace", world="shell", n_det=2000, nx=201, nz=201, rays=250),
        # merging the hits of a very bright event by sensor and time
        dict(name="merge_10M", kind="merge", n_record=10_000_000, n_det=2000, share=0.2, window=1.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["event", "event", "event", "host_event", "lite_merge", "batch", "gradient", "batch_gradient",
                       "simtrace", "merge"])
    world = rng.choice(["shell", "shell", "water_sphere"] + (sorted(ZOOS) if kind == "event" else []))
    if kind in ("batch", "gradient", "batch_gradient", "lite_merge"):
        world = "shell"
    c = dict(kind=kind, world=world)
    if world == "shell":
        c["n_det"] = _log_int(rng, 1500, 20000)
    if kind in ("batch", "batch_gradient"):
        c.update(n_event=_log_int(rng, 2, 40 if kind == "batch" else 12), mean_gs=_log_int(rng, 20, 200),
                 mean_photons=_log_int(rng, 500, 5000))
    elif kind == "simtrace":
        c.update(nx=2 * _log_int(rng, 8, 100) + 1, nz=2 * _log_int(rng, 8, 100) + 1, rays=_log_int(rng, 10, 250))
    elif kind == "merge":
        c = dict(kind=kind, n_record=_log_int(rng, 1000, 10_000_000), n_det=_log_int(rng, 100, 20000),
                 share=round(rng.uniform(0.05, 0.6), 3), window=round(rng.uniform(0.2, 10.0), 2))
    else:
        most = dict(event=10_000_000, host_event=1_000_000, lite_merge=4_000_000, gradient=2_000_000)[kind]
        c["n_photon"] = _log_int(rng, 1000, most)
        c["n_gs"] = min(_log_int(rng, 1, 1000), max(1, c["n_photon"] // 20))
        c["source"] = "torch" if world in ZOOS else rng.choice(
            ["torch", "cerenkov"] if world == "water_sphere" else ["torch", "scint", "track"])
        if kind == "event":
            c["rng"] = rng.choice(["philox", "philox", "philox", "xorwow"])
        if kind == "lite_merge":
            c["window"] = round(rng.uniform(0.2, 10.0), 2)
    if kind in ("gradient", "batch_gradient"):
        c["n_bin"] = rng.randrange(8, 65)
    return c


# ---------------------------------------------------------------- geometries


@functools.lru_cache(maxsize=16)
def _world(world, n_det):
    """(geometry, physics, meta) arrays, built once: a program has its geometry before it simulates"""
    if world == "shell":
        w = (configs.config1(1, 1) if n_det == 2000 else configs.config2(1, 1, 1) if n_det == 20000
             else configs.detector_shell(n_det, 1, 1))
        line = w.physics["boundary_names"].index("Acrylic///LS") * 4 + 3
        meta = dict(radius=w.meta["ls_r"], index=1.49, line=line, **w.meta)
    elif world == "water_sphere":
        w = configs.config0(1)
        line = w.physics["boundary_names"].index("Vacuum///Water") * 4 + 3
        meta = dict(radius=900.0, index=1.333, line=line, **w.meta)
    else:
        w = ZOOS[world](4)
        meta = dict(radius=0.0, index=1.33, line=0)
    return w.geometry, w.physics, meta


def _case_world(case):
    return _world(case["world"], case.get("n_det", 0))


# ------------------------------------------------------------------ gensteps


def _directions(g, n):
    d = g.normal(size=(n, 3))
    return d / np.linalg.norm(d, axis=1, keepdims=True)


def _torch_gensteps(counts, pos):
    gs = np.repeat(configs.torch_genstep(1, configs.T_POINT_ISO, wavelength=200.0, weight=600.0)[None], len(counts), 0)
    gs[:, 1, :3] = pos
    gs.view(np.uint32)[:, 0, 3] = counts
    return gs


def _scint_gensteps(counts, pos, time, step):
    gs = np.repeat(configs.scint_genstep(1, (0, 0, 0), step_length=1.0, charge=1.0, scint_time=1.5,
                                         mean_velocity=0.9 * 299.792458)[None], len(counts), 0)
    gs[:, 1, :3], gs[:, 1, 3], gs[:, 2, :3] = pos, time, step
    gs[:, 2, 3] = np.linalg.norm(step, axis=1)
    gs.view(np.uint32)[:, 0, 3] = counts
    return gs


def _cerenkov_gensteps(counts, pos, time, step, meta):
    one = configs.cerenkov_genstep(1, meta["line"], (0, 0, 0), 0.0, (0, 0, 10.0), 0.99, n_max=meta["index"], n1=100.0,
                                   n2=80.0, post_beta=0.985)
    gs = np.repeat(one[None], len(counts), 0)
    gs[:, 1, :3], gs[:, 1, 3], gs[:, 2, :3] = pos, time, step
    gs[:, 2, 3] = np.linalg.norm(step, axis=1)
    gs.view(np.uint32)[:, 0, 3] = counts
    return gs


def _event_gensteps(case, g, meta, n_gs, n_photon):
    counts = 1 + g.multinomial(n_photon - n_gs, np.full(n_gs, 1.0 / n_gs))
    source = case.get("source", "scint")
    if case["world"] in ZOOS:
        spots = np.array([(200, 200, 0), (-200, 200, 50), (200, -200, -50), (-200, -200, 0)], float)
        gs = _torch_gensteps(counts, spots[np.arange(n_gs) % 4] + g.uniform(-20, 20, (n_gs, 3)))
    elif source == "torch":
        gs = _torch_gensteps(counts, configs.uniform_ball(g, n_gs, meta["radius"]))
    elif source == "scint":
        gs = _scint_gensteps(counts, configs.uniform_ball(g, n_gs, meta["radius"]), g.uniform(0, 10, n_gs),
                             _directions(g, n_gs))
    else:
        # 10 mm steps along a straight track through the medium, or scattered ones (cerenkov)
        step = 10.0 * _directions(g, n_gs)
        pos, time = configs.uniform_ball(g, n_gs, 0.9 * meta["radius"]), g.uniform(0, 1, n_gs)
        if source == "track":
            d, k = _directions(g, 1)[0], np.arange(n_gs) // 2
            pitch = min(10.0, 1.8 * meta["radius"] / max(1, n_gs // 2))
            along = (k - k.mean()) * pitch
            pos, step, time = along[:, None] * d, np.repeat(pitch * d[None], n_gs, 0), k * pitch / 299.792458
        gs = _cerenkov_gensteps(counts, pos, time, step, meta)
        if source == "track":
            gs[1::2] = _scint_gensteps(counts[1::2], pos[1::2], time[1::2], step[1::2])
    return np.ascontiguousarray(gs, np.float32)


def _batch_gensteps(case, g, meta):
    """(gensteps of all events, first genstep of each event); the events' sizes are the case's"""
    size = np.random.default_rng([case["n_event"], case["mean_gs"], case["mean_photons"]])
    events = []
    for _ in range(case["n_event"]):
        n_gs = max(1, int(size.poisson(case["mean_gs"])))
        events.append(_event_gensteps(case, g, meta, n_gs, n_gs + int(size.poisson(n_gs * case["mean_photons"]))))
    return np.concatenate(events), np.concatenate([[0], np.cumsum([len(e) for e in events])])


# ------------------------------------------------------------------- prepare


class _State:
    def __init__(self, **kw):
        self.__dict__.update(kw)


def _photons(n):
    return torch.zeros((n, 4, 4), dtype=torch.float32, device=DEV)


def prepare(case, seed):
    g = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "merge":
        geometry, physics, meta = _world("water_sphere", 0)
    else:
        geometry, physics, meta = _case_world(case)
    cfg = SEventConfig(seed=seed, rng=case.get("rng", "philox"))
    s = _State(kind=kind, case=dict(case), meta=meta)
    if kind in ("gradient", "batch_gradient"):
        cfg.adjoint_tape = TAPE
        s.params = LengthParams(physics, ("LS", "Water"), n_bin=case["n_bin"])
        theta = perturbed_theta(s.params, configs.CONFIG3_BASE_LENGTHS, seed=seed)
        physics = dict(physics, bnd=s.params.apply(physics["bnd"], theta))
    s.sim = QSim(geometry, physics, cfg)
    s.event = int(seed) % 1000
    if kind in ("event", "host_event", "lite_merge", "gradient"):
        s.n = case["n_photon"]
        s.gs_host = _event_gensteps(case, g, meta, case["n_gs"], s.n)
        s.gs = torch.from_numpy(s.gs_host).to(DEV)
    if kind == "host_event":
        s.hit = np.zeros((s.n, 4, 4), np.float32)
    elif kind == "event":
        s.photon, s.hit = _photons(s.n), _photons(s.n)
        s.seq = torch.empty((s.n, 2, 2), dtype=torch.int64, device=DEV)
    elif kind == "lite_merge":
        s.lite = torch.empty((s.n, 4), dtype=torch.int32, device=DEV)
        s.merged = torch.zeros_like(s.lite)
    elif kind == "gradient":
        s.theta = torch.from_numpy(theta).to(DEV).requires_grad_(True)
        s.observed = torch.from_numpy(g.poisson(0.1 * s.n / case["n_det"], case["n_det"]).astype(np.float32)).to(DEV)
    elif kind in ("batch", "batch_gradient"):
        gs, offsets = _batch_gensteps(case, g, meta)
        n = int(gs.view(np.uint32)[:, 0, 3].sum(dtype=np.int64))
        s.gs = torch.from_numpy(gs).to(DEV)
        s.photon, s.hit = _photons(n), _photons(n // 2)
        s.seq = torch.empty((n, 2, 2), dtype=torch.int64, device=DEV)
        s.grad = adjoint = None
        if kind == "batch_gradient":
            s.grad = torch.empty((case["n_det"], s.params.n_param), dtype=torch.float32, device=DEV)
            adjoint = s.params.c_struct(case["n_det"])
        s.batch = s.sim.batch(s.gs, offsets, np.arange(case["n_event"]), s.photon, s.seq, s.hit, adjoint, s.grad)
    elif kind == "simtrace":
        s.gs_host = _simtrace_gensteps(case, seed)
        s.gs = torch.from_numpy(s.gs_host).to(DEV)
        s.n = case["nx"] * case["nz"] * case["rays"]
        s.out = _photons(s.n)
    elif kind == "merge":
        s.records = _merge_records(case, seed)
        s.out = torch.zeros_like(s.records)
    return s


@functools.lru_cache(maxsize=8)
def _grid(half, nx, nz, rays):
    ix, iz = nx // 2, nz // 2
    pitch = half / max(ix, iz)
    return configs.frame_gensteps((0.0, 0.0, 0.0, 1.0), (-ix, ix, 0, 0, -iz, iz, rays, 1), gridscale=pitch)


def _simtrace_gensteps(case, seed):
    """an XZ grid over the world, its plane shifted in y by the seed"""
    meta = _case_world(case)[2]
    gs = _grid(0.97 * meta["world_half"], case["nx"], case["nz"], case["rays"]).copy()
    gs[:, 5, 1] += np.float32(np.random.default_rng(seed).uniform(-0.2, 0.2) * meta["radius"])
    return gs


def _merge_records(case, seed):
    """sphoton records: the share that was detected carries a sensor and an arrival time"""
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    n = case["n_record"]
    r = torch.randn((n, 4, 4), generator=g, device=DEV)
    word = r.view(torch.int32)
    r[:, 0, 3] = 25.0 - 20.0 * torch.log(1.0 - torch.rand(n, generator=g, device=DEV))
    hit = torch.rand(n, generator=g, device=DEV) < case["share"]
    sensor = torch.randint(1, case["n_det"] + 1, (n,), generator=g, device=DEV, dtype=torch.int32)
    word[:, 1, 3] = 0x00010000 + sensor
    word[:, 3, 0] = torch.where(hit, FLAG["SD"], FLAG["SA"]).to(torch.int32)
    word[:, 3, 1] = torch.where(hit, sensor, 0)
    word[:, 3, 2] = torch.arange(n, dtype=torch.int32, device=DEV)
    word[:, 3, 3] = FLAG["SI"] | FLAG["BT"] | word[:, 3, 0]
    return r


# ----------------------------------------------------------------------- run


def run(s):
    """Hits and merged records come in buffers of a fixed size, with their number"""
    if s.kind == "event":
        m = s.sim.simulate_device(s.gs, s.photon, s.seq, s.hit, eventID=s.event)
        return dict(photon=s.photon, seq=s.seq, hit=s.hit, n_hit=m)
    if s.kind == "host_event":
        hit = s.sim.simulate(s.gs_host, eventID=s.event)
        s.hit[:len(hit)] = hit
        return dict(photon=s.sim.photon, seq=s.sim.seq.view(np.int64), hit=s.hit, n_hit=len(hit))
    if s.kind == "lite_merge":
        s.sim.simulate_lite_device(s.gs, s.lite, eventID=s.event)
        m = len(s.sim.merge_hits_device(s.lite, time_window=s.case["window"], out_t=s.merged))
        return dict(lite=s.lite, merged=s.merged, n_merged=m)
    if s.kind in ("batch", "batch_gradient"):
        s.batch.launch()
        offsets, _ = s.batch.wait()
        out = dict(photon=s.photon, seq=s.seq, hit=s.hit, offsets=offsets)
        if s.grad is not None:
            out["grad"] = s.grad
        return out
    if s.kind == "gradient":
        s.theta.grad = None
        counts = expected_hits(s.theta, s.sim, s.params, s.gs, s.case["n_det"], event_id=s.event, n_photon=s.n)
        loss = ((counts - s.observed) ** 2).mean()
        loss.backward()
        return dict(counts=counts.detach(), loss=loss.detach(), grad=s.theta.grad)
    if s.kind == "simtrace":
        return dict(simtrace=s.sim.simtrace_device(s.gs, s.out, n_photon=s.n))
    m = len(s.sim.merge_hits_device(s.records, time_window=s.case["window"], out_t=s.out))
    return dict(merged=s.out, n_merged=m)


# ---------------------------------------------------------------------- work


def work(case):
    """Inputs read once and outputs written once; arithmetic of the needed steps alone: about
    three propagation steps a photon (nearest surface and physics, some 600 operations each),
    one nearest surface a simtrace ray, one key a merged record."""
    kind = case["kind"]
    if kind == "merge":
        return dict(bytes=case["n_record"] * 64.0 * (1.0 + case["share"] * 0.1), flops=2.0 * case["n_record"])
    if kind == "simtrace":
        points = case["nx"] * case["nz"]
        return dict(bytes=96.0 * points + 64.0 * points * case["rays"], flops=300.0 * points * case["rays"])
    if kind in ("batch", "batch_gradient"):
        n_gs = case["n_event"] * case["mean_gs"]
        n = float(n_gs * case["mean_photons"])
    else:
        n_gs, n = case["n_gs"], float(case["n_photon"])
    out = dict(event=64 + 32 + 12, host_event=64 + 32 + 12, lite_merge=16 + 2, batch=64 + 32 + 8, gradient=0,
               batch_gradient=64 + 32 + 8)[kind]
    grad = 0.0
    if kind == "gradient":
        grad = 4.0 * (2 * case["n_det"] + 8 * case["n_bin"])
    elif kind == "batch_gradient":
        grad = 4.0 * 4 * case["n_det"] * case["n_bin"]
    return dict(bytes=96.0 * n_gs + out * n + grad, flops=1800.0 * n)


# --------------------------------------------------------------------- exact


def exact(case, seed):
    """Merged records and simtrace records in 64 bits (None for the most rays among the most
    detectors, where the search over all of them takes too long). A photon's history has no 64-bit value:
    each step's outcome is a comparison with a random number, and another rounding takes
    another branch, so the propagating kinds give None."""
    if case["kind"] == "merge":
        return dict(merged=_exact_merge(case, seed), n_merged=None)
    if case["kind"] == "simtrace" and case["nx"] * case["nz"] * case["rays"] * case.get("n_det", 1) < 4e10:
        return dict(simtrace=_exact_simtrace(case, seed))
    return None


def _exact_merge(case, seed):
    """The record of each (sensor, time bucket)'s earliest hit, first in input order on ties. The
    bucket is the integer part of the single-precision quotient, as the operation defines it."""
    r = _merge_records(case, seed).cpu().numpy()
    r = r[(r.view(np.int32)[:, 3, 3] & FLAG["SD"]) != 0]
    time = r[:, 0, 3]
    key = (r.view(np.int64)[:, 3, 0] >> 32) << 32 | (time / np.float32(case["window"])).astype(np.int64)
    order = np.lexsort((time, key))
    _, first, count = np.unique(key[order], return_index=True, return_counts=True)
    out = np.zeros((case["n_record"], 4, 4), np.float32)
    out[:len(first)] = r[order[first]]
    word = out.view(np.uint32)[:len(first)]
    word[:, 1, 3] = (word[:, 1, 3] & 0xFFFF) | (count.astype(np.uint32) & 0xFFFF) << 16
    return out


def _philox(seed, n):
    """the first two uniforms of streams 0..n-1 (Philox4x32-10, counter (0, 0, stream, 0))"""
    lo32 = np.uint64(0xFFFFFFFF)
    c = [np.zeros(n, np.uint64), np.zeros(n, np.uint64), np.arange(n, dtype=np.uint64), np.zeros(n, np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    for _ in range(10):
        p0, p1 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & lo32, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & lo32]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return [((w >> np.uint64(8)) + np.uint64(1)) * 2.0 ** -24 for w in c[:2]]


def _exact_simtrace(case, seed):
    gs = _simtrace_gensteps(case, seed).astype(np.float64)
    n = case["nx"] * case["nz"] * case["rays"]
    phi = 2.0 * np.pi * _philox(int(seed), n)[0]
    rows = np.repeat(np.arange(len(gs)), case["rays"])
    place = gs[:, 1, :3] @ gs[:, 2:5, :3].reshape(len(gs), 3, 3)[0] + gs[:, 5, :3]
    dev = DEV if torch.cuda.is_available() else "cpu"
    pos = torch.from_numpy(place[rows]).to(dev)
    dir_ = torch.from_numpy(np.stack([np.cos(phi), np.zeros(n), np.sin(phi)], 1)).to(dev)
    out = torch.zeros((n, 4, 4), dtype=torch.float64, device=dev)
    geometry, _, meta = _case_world(case)
    spheres = [meta["sphere_r"]] if case["world"] == "water_sphere" else [meta["ls_r"], meta["ls_r"] + 120.0]
    frames = geometry["inst"].reshape(-1, 4, 4)[1:].astype(np.float64)
    chunk = max(1, 200_000_000 // max(1, len(frames)))
    for a in range(0, n, chunk):
        p, d = pos[a:a + chunk], dir_[a:a + chunk]
        t, normal = _nearest(p, d, meta["world_half"], spheres, frames, 0.05)
        o = out[a:a + chunk]
        o[:, 0, :3], o[:, 0, 3] = normal, t
        o[:, 1, :3], o[:, 1, 3] = p + t[:, None] * d, 0.05
        o[:, 2, :3], o[:, 3, :3] = p, d
    return out.cpu().numpy()


def _slab(p, d, lo, hi):
    a, b = (lo - p) / d, (hi - p) / d
    return torch.minimum(a, b), torch.maximum(a, b)


def _quadric(a, b, c):
    """[near, far] of a t^2 + 2 b t + c <= 0, empty (inf, -inf) where there is none"""
    disc = b * b - a * c
    root = torch.sqrt(disc.clamp(min=0))
    none = disc <= 0
    return torch.where(none, math.inf, (-b - root) / a), torch.where(none, -math.inf, (-b + root) / a)


def _nearest(p, d, half, spheres, frames, tmin):
    """distance to and unnormalised normal of the nearest surface beyond tmin: a box about the
    origin, spheres about it, and the CSG detectors (ellipsoid cap joined with a neck, less a
    bore) in the frames given"""
    n0, f0 = (torch.stack(v) for v in zip(*[_slab(p[:, k], d[:, k], -half, half) for k in range(3)]))
    t = f0.min(0).values
    axis = f0.argmin(0)
    normal = torch.nn.functional.one_hot(axis, 3).to(p) * torch.sign(torch.gather(d, 1, axis[:, None]))
    for r in spheres:
        near, far = _quadric((d * d).sum(1), (p * d).sum(1), (p * p).sum(1) - r * r)
        ts = torch.where(near > tmin, near, far)
        hit = (ts > tmin) & (ts < t)
        t = torch.where(hit, ts, t)
        normal = torch.where(hit[:, None], (p + ts[:, None] * d) / r, normal)
    if not len(frames):
        return t, normal
    M = torch.from_numpy(frames[:, :3, :3].copy()).to(p)
    C = torch.from_numpy(frames[:, 3, :3].copy()).to(p)
    # detectors whose bounding sphere the segment to the nearest hit so far meets
    centre = C + torch.tensor([0.0, 0.0, -25.0], dtype=p.dtype, device=p.device) @ M
    along = ((d @ centre.T) - (p * d).sum(1, keepdim=True)).clamp(min=0)
    along = torch.minimum(along, t[:, None])
    off2 = (p * p).sum(1, keepdim=True) + (centre * centre).sum(1) - 2 * (p @ centre.T)
    off2 += along * along - 2 * along * ((d @ centre.T) - (p * d).sum(1, keepdim=True))
    ray, det = torch.nonzero(off2 < 300.0 ** 2, as_tuple=True)
    o = torch.einsum("nj,nij->ni", p[ray] - C[det], M[det])
    v = torch.einsum("nj,nij->ni", d[ray], M[det])
    s = 190.0 / 254.0
    oe, ve = o * torch.tensor([s, s, 1.0]).to(o), v * torch.tensor([s, s, 1.0]).to(o)
    ends, kinds = [], []
    e0, e1 = _quadric((ve * ve).sum(1), (oe * ve).sum(1), (oe * oe).sum(1) - 190.0 ** 2)
    for parts in (((e0, e1), (-50.0, 190.0)),
                  (_radial(o, v, 127.0), (-240.0, -40.0)), (_radial(o, v, 120.0), (-260.0, -60.0))):
        (q0, q1), (lo, hi) = parts
        z0, z1 = _slab(o[:, 2], v[:, 2], lo, hi)
        ends += [torch.maximum(q0, z0), torch.minimum(q1, z1)]
        kinds += [q0 >= z0, q1 <= z1]                     # on the curved part
    a0, a1, b0, b1, c0, c1 = ends
    for x0, x1 in ((a0, a1), (b0, b1), (c0, c1)):
        empty = x0 >= x1
        x0[empty], x1[empty] = math.inf, math.inf
    every = torch.stack([torch.where(x > tmin, x, math.inf) for x in ends], 1)
    order = torch.cat([torch.full_like(every[:, :1], tmin), every.sort(1).values], 1)
    mid = 0.5 * (order[:, 1:] + order[:, :-1])
    mid = torch.cat([mid, torch.full_like(mid[:, :1], math.inf)], 1)

    def within(m):
        return (((m > a0[:, None]) & (m < a1[:, None])) | ((m > b0[:, None]) & (m < b1[:, None]))) & \
            ~((m > c0[:, None]) & (m < c1[:, None]))

    cross = torch.isfinite(order[:, 1:]) & (within(mid[:, :-1]) != within(mid[:, 1:]))
    td = torch.where(cross, order[:, 1:], math.inf).min(1).values
    best = t.clone().scatter_reduce(0, ray, td, "amin")
    win = torch.isfinite(td) & (td <= best[ray]) & (td < t[ray])
    ray, det, td, o, v = ray[win], det[win], td[win], o[win], v[win]
    which = torch.stack([(e[win] - td).abs() for e in ends], 1).argmin(1)
    curved = torch.stack([k[win] for k in kinds], 1).gather(1, which[:, None])[:, 0]
    x = o + td[:, None] * v
    r = torch.tensor([0.0, 0.0, 127.0, 127.0, 120.0, 120.0]).to(x)[which]
    side = torch.where((which < 2)[:, None], x * torch.tensor([s * s, s * s, 1.0]).to(x) / 190.0,
                       torch.cat([x[:, :2] / r[:, None].clamp(min=1), torch.zeros_like(x[:, :1])], 1))
    flat = torch.zeros_like(x)
    flat[:, 2] = torch.where(which % 2 == 0, -1.0, 1.0) * torch.sign(v[:, 2])
    nl = torch.where(curved[:, None], side, flat)
    nl = torch.where((which >= 4)[:, None], -nl, nl)     # the bore's surface faces into it
    t[ray] = td
    normal[ray] = torch.einsum("nj,nji->ni", nl, M[det])
    return t, normal


def _radial(o, v, r):
    a = (v[:, :2] ** 2).sum(1)
    return _quadric(a, (o[:, :2] * v[:, :2]).sum(1), (o[:, :2] ** 2).sum(1) - r * r)
