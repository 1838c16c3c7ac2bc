"""GPU hit merge (mi_sim_merge_hits_device) against the CPU restatement
(oracle/spm.py), bit for bit: real hits of the CSG workload, synthetic records
with many (identity, bucket) collisions and time ties, both record types,
selection-only and already-selected modes, and the edge cases."""
import numpy as np
import pytest

import spm
from opticks_amd import configs
from opticks_amd import _lib as L
from opticks_amd.qsim import QSim, SEventConfig

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

DEV = torch.device("cuda:0")
SD, SA = 0x40, 0x80


@pytest.fixture(scope="module")
def sim_and_photons():
    w = configs.config1(num_gs=20, per_gs=5000)
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=w.seed))
    N = w.num_photon
    gs = torch.from_numpy(w.gensteps).to(DEV)
    photon = torch.empty((N, 4, 4), dtype=torch.float32, device=DEV)
    sim.simulate_device(gs, photon, None, None, n_photon=N)
    yield sim, photon
    sim.close()


def synthetic(n, seed):
    rng = np.random.default_rng(seed)
    p = np.zeros((n, 4, 4), np.float32)
    u = p.view(np.uint32)
    p[:, 0, 0] = np.arange(n)
    p[:, 0, 3] = rng.integers(0, 40, n) * 0.25          # many exact time ties
    u[:, 1, 3] = (rng.integers(1, 4, n).astype(np.uint32) << 16) | 3
    u[:, 3, 1] = rng.integers(1, 30, n).astype(np.uint32) | (rng.integers(0, 2, n).astype(np.uint32) << 16)
    u[:, 3, 3] = np.where(rng.random(n) < 0.6, SD, SA).astype(np.uint32) | (rng.integers(0, 4, n).astype(np.uint32) << 2)
    return p


@pytest.mark.parametrize("tw", [1.0, 0.5, 7.0, 0.0])
def test_photon_merge_real_hits(sim_and_photons, tw):
    sim, photon = sim_and_photons
    out = sim.merge_hits_device(photon, SD, tw)
    ref = spm.merge_photons(photon.cpu().numpy(), SD, tw)
    assert out.shape[0] == len(ref) > 0
    assert np.array_equal(out.cpu().numpy().view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("seed", [1, 2])
def test_photon_merge_synthetic_collisions(sim_and_photons, seed):
    sim, _ = sim_and_photons
    P = synthetic(50_000, seed)
    t = torch.from_numpy(P).to(DEV)
    for mask, tw in [(SD, 1.0), (SD | SA, 2.5), (L.MI_MERGE_ALREADY_SELECTED, 1.0), (SD, 0.0)]:
        out = sim.merge_hits_device(t, mask, tw).cpu().numpy()
        ref = spm.merge_photons(P, mask, tw)
        assert np.array_equal(out.view(np.uint32), ref.view(np.uint32)), (mask, tw)


def test_lite_merge_synthetic(sim_and_photons):
    sim, _ = sim_and_photons
    P = synthetic(40_000, 9)
    u = P.view(np.uint32)
    lt = np.stack([(u[:, 1, 3] & 0xFFFF0000) | (u[:, 3, 1] & 0xFFFF), u[:, 0, 3], np.arange(len(P), dtype=np.uint32),
                   u[:, 3, 3]], axis=1).astype(np.uint32)
    t = torch.from_numpy(lt.view(np.int32)).to(DEV)
    for mask, tw in [(SD, 1.0), (L.MI_MERGE_ALREADY_SELECTED, 0.75), (SD, 0.0)]:
        out = sim.merge_hits_device(t, mask, tw).cpu().numpy().view(np.uint32)
        ref = spm.merge_lites(lt, mask, tw)
        assert np.array_equal(out, ref), (mask, tw)


def test_merge_edge_cases(sim_and_photons):
    sim, _ = sim_and_photons
    empty = torch.empty((0, 4, 4), dtype=torch.float32, device=DEV)
    assert sim.merge_hits_device(empty, SD, 1.0).shape[0] == 0
    P = synthetic(1000, 4)
    P.view(np.uint32)[:, 3, 3] = SA
    t = torch.from_numpy(P).to(DEV)
    assert sim.merge_hits_device(t, SD, 1.0).shape[0] == 0          # nothing selected
    small = torch.empty((3, 4, 4), dtype=torch.float32, device=DEV)
    with pytest.raises(RuntimeError, match="out_capacity"):
        sim.merge_hits_device(t, SA, 1.0, out_t=small)
    with pytest.raises(RuntimeError):
        sim.merge_hits_device(t, SA, -1.0)


def test_photonlite_output_matches_checker_and_merges():
    import pyoracle as po
    w = configs.config1(num_gs=20, per_gs=2000)
    sim = QSim(w.geometry, w.physics, SEventConfig(seed=w.seed))
    N = w.num_photon
    gs = torch.from_numpy(w.gensteps).to(DEV)
    photon = torch.empty((N, 4, 4), dtype=torch.float32, device=DEV)
    seq = torch.empty((N, 2, 2), dtype=torch.int64, device=DEV)
    lite = torch.empty((N, 4), dtype=torch.int32, device=DEV)
    sim.simulate_lite_device(gs, lite, photon, seq, n_photon=N)
    G = lite.cpu().numpy().view(np.uint32)
    P = photon.cpu().numpy()
    rp, rs, rl = po.World(w.geometry, w.physics).simulate_lite(w.gensteps, seed=w.seed)
    same = np.all(seq.cpu().numpy().view(np.uint64) == rs, axis=(1, 2))
    assert same.mean() >= 0.999
    assert np.array_equal(G[same], rl[same])
    # lite fields are the photon's identity, time and flagmask, hitcount 1
    u = P.view(np.uint32)
    assert np.array_equal(G[:, 0] & 0xFFFF, u[:, 3, 1] & 0xFFFF)
    assert np.all(G[:, 0] >> 16 == 1)
    assert np.array_equal(G[:, 1], u[:, 0, 3])
    assert np.array_equal(G[:, 3], u[:, 3, 3])
    # most detected photons arrive from the centre onto the detector front (local z > 0),
    # some on the side or neck (lposcost <= 0, clamped to 0 by the 16-bit packing)
    sd = (u[:, 3, 3] & SD) != 0
    assert sd.sum() > 100 and ((G[sd, 2] >> 16) > 0).mean() > 0.5
    assert np.ptp((G[sd, 2] & 0xFFFF).astype(np.int64)) > 30000      # azimuths spread round the axis
    # same results with and without the lite instantiation
    p2 = torch.empty_like(photon)
    sim.simulate_device(gs, p2, None, None, n_photon=N)
    assert np.array_equal(p2.cpu().numpy().view(np.uint32), u)
    # lite hits selected and merged on the GPU equal the restatement on the checker's lites
    out = sim.merge_hits_device(lite, SD, 1.0).cpu().numpy().view(np.uint32)
    ref = spm.merge_lites(rl[same], SD, 1.0) if same.all() else None
    if ref is not None:
        assert np.array_equal(out, ref)
    assert np.array_equal(out, spm.merge_lites(G, SD, 1.0))
    sim.close()


@pytest.mark.parametrize("n", [1, 255, 256, 257, 4095, 4096, 4097, 3 * 4096 + 17, 300_001])
def test_merge_tiles_and_key_widths(sim_and_photons, n):
    """Sizes around the 4096-record tiles; keys of few bits, of more than 32, of one value, of
    buckets up to 32 bits; long and single-record runs."""
    sim, _ = sim_and_photons
    rng = np.random.default_rng(n)
    late = np.array([0.0, 1.0, 2.1e9], np.float32)
    for kind in ("narrow", "wide", "one", "late"):
        P = synthetic(n, n + 1)
        u = P.view(np.uint32)
        if kind == "wide":
            P[:, 0, 3] = rng.random(n).astype(np.float32) * 4.0e6
            u[:, 3, 1] = rng.integers(0, 65536, n).astype(np.uint32)
        if kind == "one":
            P[:, 0, 3], u[:, 3, 1] = 0.0, 0
        if kind == "late":
            P[:, 0, 3] = rng.choice(late, n)
        lt = np.stack([(u[:, 1, 3] & 0xFFFF0000) | (u[:, 3, 1] & 0xFFFF), u[:, 0, 3], np.arange(n, dtype=np.uint32),
                       u[:, 3, 3]], axis=1).astype(np.uint32)
        t, tl = torch.from_numpy(P).to(DEV), torch.from_numpy(lt.view(np.int32)).to(DEV)
        for tw in (0.5, 0.0):
            ref, refl = spm.merge_photons(P, SD, tw), spm.merge_lites(lt, SD, tw)
            for rows, merged, ref_bits in ((t, sim.merge_hits_device(t, SD, tw), ref.view(np.uint32)),
                                           (tl, sim.merge_hits_device(tl, SD, tw), refl)):
                got = merged.cpu().numpy().view(np.uint32)
                assert got.shape == ref_bits.shape and np.array_equal(got, ref_bits), (kind, tw)
                tight = torch.full((len(ref_bits),) + tuple(rows.shape[1:]), 0, dtype=rows.dtype, device=DEV)
                if len(ref_bits):                  # a buffer of just the merged size, then one short of it
                    sim.merge_hits_device(rows, SD, tw, out_t=tight)
                    assert np.array_equal(tight.cpu().numpy().view(np.uint32), ref_bits), (kind, tw)
                if len(ref_bits) > 1:
                    short = torch.zeros_like(tight)[:-1].contiguous()
                    with pytest.raises(RuntimeError, match="out_capacity"):
                        sim.merge_hits_device(rows, SD, tw, out_t=short)
                    assert not short.cpu().numpy().any()


def bucket(time, tw):
    """(unsigned)(time / window) as the GPU converts: towards zero, clamped to 32 bits, not-a-number 0"""
    q = np.float32(time) / np.float32(tw)
    return 0 if not q > 0 else min(int(min(float(q), 2.0 ** 33)), 0xffffffff)


def smaller(a, b):
    """fminf: a number rather than not-a-number"""
    return b if np.isnan(a) else a if np.isnan(b) else min(a, b)


@pytest.mark.parametrize("kind", ["mixed", "one run", "nan runs"])
def test_merge_times_that_are_no_ordinary_numbers(sim_and_photons, kind):
    """NaN, infinite, negative and zero times of both signs in short runs and in runs that a wave
    folds in pieces: the record types' reduce_op applied left to right in the sorted order."""
    sim, _ = sim_and_photons
    rng = np.random.default_rng(len(kind))
    n, tw = 9001, 1.0
    P = synthetic(n, 5)
    u = P.view(np.uint32)
    special = np.array([np.nan, np.inf, -np.inf, -3.5, -0.25, 0.0, -0.0, 0.25, 0.75, 1.5, 5.0e9, 1e-40], np.float32)
    P[:, 0, 3] = rng.choice(special, n)
    u[:, 3, 1] = rng.integers(1, 4, n).astype(np.uint32)
    u[:, 3, 3] = SD | (rng.integers(0, 8, n).astype(np.uint32) << 8)
    if kind == "one run":
        P[:, 0, 3] = rng.choice(np.array([np.nan, -3.5, -0.0, 0.0, 0.25, 0.75], np.float32), n)
        u[:, 3, 1] = 7
    if kind == "nan runs":
        P[:, 0, 3] = np.nan
        u[:, 3, 1] = rng.integers(0, 400, n).astype(np.uint32)
    t = P[:, 0, 3]
    lt = np.stack([(u[:, 1, 3] & 0xFFFF0000) | (u[:, 3, 1] & 0xFFFF), u[:, 0, 3], np.arange(n, dtype=np.uint32), u[:, 3, 3]],
                  axis=1).astype(np.uint32)
    runs = {}
    for i in range(n):
        runs.setdefault((int(u[i, 3, 1]) & 0xffff, bucket(t[i], tw)), []).append(i)
    want, wantl = [], []
    for key in sorted(runs):
        best = first = runs[key][0]
        hc, fm, tt = int(u[best, 1, 3]) >> 16, int(u[best, 3, 3]), t[best]
        for b in runs[key][1:]:
            if not smaller(t[best], t[b]) == t[best]:
                best = b
            tt = smaller(tt, t[b])
            hc, fm = (hc + (int(u[b, 1, 3]) >> 16)) & 0xffff, fm | int(u[b, 3, 3])
        r = u[best].copy()
        r[1, 3] = (int(r[1, 3]) & 0xffff) | (hc << 16)
        r[3, 3] = fm
        want.append(r)
        wantl.append((hc << 16 | int(lt[first, 0]) & 0xffff, tt, int(lt[first, 2]), fm))
    got = sim.merge_hits_device(torch.from_numpy(P).to(DEV), SD, tw).cpu().numpy().view(np.uint32)
    assert np.array_equal(got, np.array(want))
    gl = sim.merge_hits_device(torch.from_numpy(lt.view(np.int32)).to(DEV), SD, tw).cpu().numpy().view(np.uint32)
    assert len(gl) == len(wantl)
    for col in (0, 2, 3):
        assert np.array_equal(gl[:, col], np.array([w[col] for w in wantl], np.uint32))
    # the smaller of two zeros, or of two that are no numbers, is either
    assert np.array_equal(gl[:, 1].copy().view(np.float32), np.array([w[1] for w in wantl], np.float32), equal_nan=True)


def merged_lites(lt, tw):
    """spm.merge_lites of selected records with ordinary times >= 0, by whole arrays"""
    t = lt[:, 1].view(np.float32)
    keys = ((lt[:, 0] & 0xffff).astype(np.uint64) << 32) | (t / np.float32(tw)).astype(np.float32).astype(np.uint64)
    order = np.argsort(keys, kind="stable")
    ks = keys[order]
    start = np.flatnonzero(np.r_[True, ks[1:] != ks[:-1]])
    hc = np.add.reduceat((lt[order, 0] >> 16).astype(np.uint64), start) & 0xffff
    out = np.empty((len(start), 4), np.uint32)
    first = order[start]
    out[:, 0] = (hc.astype(np.uint32) << 16) | (lt[first, 0] & 0xffff)
    out[:, 1] = np.minimum.reduceat(t[order], start).view(np.uint32)
    out[:, 2] = lt[first, 2]
    out[:, 3] = np.bitwise_or.reduceat(lt[order, 3], start)
    # the photon record kept: the earliest in input order among the run's smallest times
    run = np.repeat(np.arange(len(start)), np.diff(np.r_[start, len(ks)]))
    pos = np.flatnonzero(t[order] == out[run, 1].view(np.float32))
    keep = np.full(len(start), -1)
    keep[run[pos][::-1]] = order[pos][::-1]
    return out, keep


# selected counts on both sides of the tiles of 2,048 (selection and sort) and 1,024 (runs), past the
# 256 sort tiles of one step of a digit's sums, and past the 8,192 selection tiles of one step of theirs
@pytest.mark.parametrize("n, lite_only", [(1023, False), (1024, False), (1025, False), (2047, False), (2048, False),
                                          (2049, False), (600_001, False), (16_900_123, True)])
def test_merge_of_all_records(sim_and_photons, n, lite_only):
    sim, _ = sim_and_photons
    rng = np.random.default_rng(n)
    lt = np.empty((n, 4), np.uint32)
    lt[:, 0] = (rng.integers(1, 5, n) << 16) | rng.integers(1, 3000, n)
    lt[:, 1] = (rng.integers(0, 4000, n) * np.float32(0.125)).astype(np.float32).view(np.uint32)
    lt[:, 2] = np.arange(n)
    lt[:, 3] = 1 << rng.integers(0, 16, n)
    want, keep = merged_lites(lt, 4.0)
    if n < 3000:
        assert np.array_equal(want, spm.merge_lites(lt, L.MI_MERGE_ALREADY_SELECTED, 4.0))
    got = sim.merge_hits_device(torch.from_numpy(lt.view(np.int32)).to(DEV), L.MI_MERGE_ALREADY_SELECTED, 4.0)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), want)
    if lite_only:
        return
    P = np.zeros((n, 4, 4), np.uint32)
    P[:, 0, 0], P[:, 0, 3], P[:, 3, 1], P[:, 3, 3] = lt[:, 2], lt[:, 1], lt[:, 0] & 0xffff, lt[:, 3]
    P[:, 1, 3] = lt[:, 0] & 0xffff0000
    ref = P[keep].copy()
    ref[:, 1, 3], ref[:, 3, 3] = want[:, 0] & 0xffff0000, want[:, 3]
    got = sim.merge_hits_device(torch.from_numpy(P.view(np.float32)).to(DEV), L.MI_MERGE_ALREADY_SELECTED, 4.0)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), ref)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 511, 513, 1793, 2047, 2048, 2049])
def test_merge_of_few_records_keeps_their_order(sim_and_photons, n):
    """Numbers of pairs around a wave, a round of four waves and a tile of the sort; keys of one to
    six bytes. The index of a run's first record and its flags show the order of equal keys."""
    sim, _ = sim_and_photons
    rng = np.random.default_rng(n)
    for n_id, n_bucket in ((1, 1), (3, 2), (300, 1), (3000, 40), (3, 3_000_000), (65535, 60_000_000)):
        lt = np.empty((n, 4), np.uint32)
        lt[:, 0] = (rng.integers(1, 5, n) << 16) | rng.integers(max(1, n_id - 7), n_id + 1, n)
        lt[:, 1] = (rng.integers(max(0, n_bucket - 5), n_bucket, n) * np.float32(1.0)).astype(np.float32).view(np.uint32)
        lt[:, 2] = np.arange(n)
        lt[:, 3] = 1 << rng.integers(0, 16, n)
        ref = spm.merge_lites(lt, L.MI_MERGE_ALREADY_SELECTED, 1.0)
        out = sim.merge_hits_device(torch.from_numpy(lt.view(np.int32)).to(DEV), L.MI_MERGE_ALREADY_SELECTED, 1.0)
        assert np.array_equal(out.cpu().numpy().view(np.uint32), ref), (n_id, n_bucket)
