/*
 * oa_kernels.hip : gfx950 kernels of the propagation path other than the
 * propagation kernels themselves (oa_sim.h, launched through oa_sim.hip).
 *
 *   k_gs_prefix       exclusive prefix of genstep numphoton (QEvt.cu:181-226 seeding
 *                     reduce)
 *   k_setup           start of a single-event launch: prefix, seeds and cleared counters
 *   k_seed_fill       the expand: genstep index of every photon, one block per
 *                     genstep writing its photon range (QEvt.cu:181-226 seed
 *                     buffer, sysrap/iexpand.h); k_gs_event the event of every
 *                     genstep for batched launches
 *   k_simtrace, k_simtrace_few   frame-genstep rays, nearest hit
 *   k_hit_counts      hits per detector
 *   k_compact         stable stream compaction of flagmask&hit_mask photons via
 *                     a per-64-photon bitmask (QEvt::gatherHit_, SU.cu:145-160)
 *   k_trace           nearest-hit query (simtrace-style)
 *   k_refit_level     GPU refit of the TLAS levels after instance moves
 */
#include <hip/hip_runtime.h>
#include <mutex>
#include "oa_sim.h"
#include "oa_sim_launch.h"
#include "oa_kernels.h"

using namespace oa;

/* ------------------------------------------------------------ seeding */

/* seed[i] = genstep of photon i for i < n_photon: blocks stride over gensteps,
   threads over each genstep's photon range [prefix[g], prefix[g+1]) (coalesced
   writes). Photons past the gensteps' total (a caller's n_photon larger than
   the gensteps hold) get the last genstep, as the binary search gave them. */
__global__ void __launch_bounds__(256) k_seed_fill(const int64_t* prefix, int64_t n_gs, int64_t n_photon,
                                                   uint32_t* seed)
{
    for (int64_t g = blockIdx.x; g < n_gs; g += gridDim.x) {
        const int64_t b = prefix[g], e = prefix[g + 1] < n_photon ? prefix[g + 1] : n_photon;
        for (int64_t i = b + threadIdx.x; i < e; i += blockDim.x) seed[i] = (uint32_t)g;
    }
    if (blockIdx.x == 0)
        for (int64_t i = prefix[n_gs] + threadIdx.x; i < n_photon; i += blockDim.x) seed[i] = (uint32_t)(n_gs - 1);
}

/* gs_event[g] = event owning genstep g, from the events' genstep boundaries */
__global__ void __launch_bounds__(256) k_gs_event(const int64_t* ev_gs_begin, int32_t n_event, int32_t* gs_event)
{
    for (int32_t e = blockIdx.x; e < n_event; e += gridDim.x)
        for (int64_t g = ev_gs_begin[e] + threadIdx.x; g < ev_gs_begin[e + 1]; g += blockDim.x) gs_event[g] = e;
}

/* exclusive prefix of the gensteps' photon counts, 1,024 a block: `sums` has each block's
   total (k_gs_sums) where there is more than one */
__global__ void __launch_bounds__(1024) k_gs_sums(const float* gs, int64_t n_gs, int64_t* sums, LaunchResult* out)
{
    __shared__ int64_t part[16];
    if (out && blockIdx.x == 0 && threadIdx.x == 0) out->setup_begins = wall_clock64();
    const int64_t g = (int64_t)blockIdx.x * 1024 + threadIdx.x;
    int64_t v = g < n_gs ? (int64_t)__float_as_uint(gs[24 * g + 3]) : 0;
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t t = 0;
        for (int k = 0; k < 16; ++k) t += part[k];
        sums[blockIdx.x] = t;
    }
}

/* inclusive scan of one value a thread over the block (at most 16 waves); part: 16 words of LDS */
OA_D int64_t block_scan(int64_t v, int64_t* part)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int o = 1; o < 64; o <<= 1) {
        const int64_t u = __shfl_up(v, o);
        if (lane >= o) v += u;
    }
    if (lane == 63) part[wave] = v;
    __syncthreads();
    for (int q = 0; q < wave; ++q) v += part[q];
    return v;
}

__global__ void __launch_bounds__(1024) k_gs_prefix(const float* gs, int64_t n_gs, const int64_t* sums, int64_t* prefix)
{
    __shared__ int64_t part[16], s_before[16];
    const int t = threadIdx.x;
    const int64_t g = (int64_t)blockIdx.x * 1024 + t;
    /* gensteps of the blocks before this one */
    int64_t b = 0;
    for (int64_t k = t; k < (int64_t)blockIdx.x; k += 1024) b += sums[k];
    for (int o = 32; o > 0; o >>= 1) b += __shfl_xor(b, o);
    if ((t & 63) == 0) s_before[t >> 6] = b;
    const int64_t v = g < n_gs ? (int64_t)__float_as_uint(gs[24 * g + 3]) : 0;
    const int64_t incl = block_scan(v, part);
    int64_t before = 0;
    for (int k = 0; k < 16; ++k) before += s_before[k];
    if (g < n_gs) prefix[g] = before + incl - v;
    if (g == n_gs - 1) prefix[n_gs] = before + incl;
}

/*
 * Start of a single-event launch: genstep of every photon (QEvt.cu:181-226), cleared hit
 * words and counters, event bounds, and the launch's photon count on the device, where the
 * propagation and the compaction read it: the host need not wait for the gensteps' total
 * before it launches them. The count is n_arg, or the gensteps' total for n_arg < 0; it is 0,
 * and nothing is propagated, when that is more than the gensteps have or than the launch's
 * buffers hold (cap): the host sees the total and reports it or tries again.
 * SMALL: up to OA_SETUP_GS gensteps; every block forms their prefix in LDS by itself (a few
 * loads a thread), so one kernel does all of it. Else the prefix is there already (k_gs_sums has
 * stamped the begin).
 */
template <bool SMALL>
__global__ void __launch_bounds__(256) k_setup(const float* gs, int64_t n_gs, int64_t n_arg, int64_t cap, int64_t* prefix,
                                               uint32_t* seed, unsigned long long* words, int64_t bitmask, int64_t* ev,
                                               int32_t* ev_id, int32_t event_id, int64_t* n_dev, LaunchResult* out,
                                               int64_t n_wave)
{
    constexpr int PER = SMALL ? OA_SETUP_GS / 256 : 1;
    __shared__ int64_t s_prefix[SMALL ? OA_SETUP_GS + 1 : 1];
    __shared__ int64_t part[16];
    const int t = threadIdx.x;
    const bool first = blockIdx.x == 0;
    if (SMALL && first && t == 0) out->setup_begins = wall_clock64();
    if (SMALL) {
        int64_t c[PER], sum = 0;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int64_t g = (int64_t)t * PER + k;
            c[k] = g < n_gs ? (int64_t)__float_as_uint(gs[24 * g + 3]) : 0;
        }
#pragma unroll
        for (int k = 0; k < PER; ++k) sum += c[k];
        int64_t run = block_scan(sum, part) - sum;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int64_t g = (int64_t)t * PER + k;
            if (g <= n_gs) {
                s_prefix[g] = run;
                if (first) prefix[g] = run;
            }
            run += c[k];
        }
        if (t == 255 && n_gs == OA_SETUP_GS) {
            s_prefix[n_gs] = run;
            if (first) prefix[n_gs] = run;
        }
        __syncthreads();
    }
    const int64_t* pre = SMALL ? s_prefix : prefix;
    const int64_t total = pre[n_gs];
    int64_t n = n_arg < 0 ? total : n_arg;
    if (n > total || n > cap) n = 0;
    const int64_t stride = (int64_t)gridDim.x * 256, id = (int64_t)blockIdx.x * 256 + t;
    /* the photon counter starts behind the photons dealt first; of the bitmask and the tiles, what
       n photons use */
    const int64_t width = wave_width(n, n_wave), n_words = (n + 63) / 64, n_tiles = (n_words + 255) / 256;
    for (int64_t i = id; i < OA_WORDS_STATE + n_tiles; i += stride) words[i] = i == 0 ? (unsigned long long)(n_wave * width) : 0ull;
    for (int64_t i = id; i < n_words; i += stride) words[bitmask + i] = 0ull;
    for (int64_t i = 4 * id; i < n; i += 4 * stride) {
        int64_t g = upper_index(pre, 0, n_gs, i);
        uint32_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            while (g + 1 < n_gs && pre[g + 1] <= i + u) ++g;
            v[u] = (uint32_t)g;
        }
        if (i + 4 <= n) *reinterpret_cast<uint4*>(seed + i) = make_uint4(v[0], v[1], v[2], v[3]);
        else for (int u = 0; i + u < n; ++u) seed[i + u] = v[u];
    }
    if (first && t == 0) {
        ev[0] = 0; ev[1] = n_gs; ev[2] = 0; ev[3] = n;
        ev_id[0] = event_id;
        n_dev[0] = n;
        n_dev[1] = width;
        out->total = total;
        out->n_photon = n;
        out->n_hit = 0;
    }
    __syncthreads();
    if (t == 0) result_ends(out)[blockIdx.x] = wall_clock64();
}

/* ------------------------------------------------------------ simtrace */

/* largest k in [0, n) with a[k] <= v, the same v on every lane of a wave: 64 ways a step,
   three dependent loads for 40,000 gensteps where halving takes sixteen */
__device__ int64_t wave_upper_index(const int64_t* a, int64_t n, int64_t v, int lane)
{
    int64_t lo = 0;
    for (int64_t len = n; len > 1;) {
        const int64_t step = (len + 63) / 64, probe = lane * step;
        const unsigned long long m = __ballot(probe < len && a[lo + probe] <= v);
        const int64_t k = m ? 63 - __clzll((long long)m) : 0;
        lo += k * step;
        len = len - k * step < step ? len - k * step : step;
    }
    return lo;
}

/* the ray of photon idx of genstep gq: qsim::generate_photon_simtrace_frame
   (qudarap/qsim.h:2460-2522) on RNG stream (event 0, photon index) */
__device__ void simtrace_ray(const SimParams& P, const float4* gq, int64_t idx, v3& pos, v3& dir)
{
    PhiloxRng rng;
    rng.key = P.seed;
    rng.photon = (uint64_t)idx;
    rng.pos = P.rng_offset;
    float u[2];
    draw<2>(rng, u);
    const uint32_t gridaxes = __float_as_uint(gq[0].y);
    const float u0 = u[0];
    float sinPhi, cosPhi;
    oa_sincosf(2.f * OA_PI_F * u0, &sinPhi, &cosPhi);
    const float u1 = u[1];
    const float cosTheta = 2.f * u1 - 1.f;
    const float sinTheta = sqrtf(1.f - cosTheta * cosTheta);
    dir = gridaxes == 1u ? mk(0.f, cosPhi, sinPhi)
        : gridaxes == 2u ? mk(cosPhi, 0.f, sinPhi)
        : gridaxes == 3u ? mk(cosPhi, sinPhi, 0.f)
        : mk(sinTheta * cosPhi, sinTheta * sinPhi, cosTheta);
    const float4 q1 = gq[1];
    pos = q_right(gq + 2, mk(q1.x, q1.y, q1.z), 1.f);
    dir = q_right(gq + 2, dir, 0.f);
}

/* sevent::add_simtrace (sysrap/sevent.h:670-696); a miss writes q0 = (0.6,0.6,0.6,1), the
   miss program's midgrey background (CSGOptiX7.cu:683-700, CSGOptiX/SBT.cc:185-191) */
__device__ void simtrace_record(const SimParams& P, float4* o, v3 pos, v3 dir, const Prd& prd)
{
    const bool miss = prd.boundary == 0xffffu;
    const float t = miss ? 1.f : prd.t;
    const uint32_t gpb = miss ? 0xffffffffu : (((prd.gprim & 0xffffu) << 16) | (prd.boundary & 0xffffu));
    const uint32_t ii = miss ? 0xffffffffu : prd.iindex_identity;
    o[0] = miss ? make_float4(0.6f, 0.6f, 0.6f, t) : make_float4(prd.normal.x, prd.normal.y, prd.normal.z, t);
    o[1] = make_float4(pos.x + t * dir.x, pos.y + t * dir.y, pos.z + t * dir.z, P.tmin);
    o[2] = make_float4(pos.x, pos.y, pos.z, __uint_as_float(gpb));
    o[3] = make_float4(dir.x, dir.y, dir.z, __uint_as_float(ii));
}

/* CSGOptiX7.cu:563-604 simtrace, a ray to a lane from start to end (see simtrace below) */
template <bool EXT>
__global__ void __launch_bounds__(64) OA_OCC k_simtrace_few(SimParams P, float4* out)
{
    extern __shared__ uint32_t s_lane[];             /* each lane's stack */
    const int lane = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * 64, i = first + lane;
    const int64_t last = first + 63 < P.n_photon ? first + 63 : P.n_photon - 1;
    const int64_t g0 = wave_upper_index(P.gs_prefix, P.n_gs, first, lane);
    const int64_t g1 = g0 + wave_upper_index(P.gs_prefix + g0, P.n_gs - g0, last, lane);
    if (i > last) return;
    const int64_t gsi = upper_index(P.gs_prefix, g0, g1 + 1, i);
    v3 o, d;
    simtrace_ray(P, reinterpret_cast<const float4*>(P.gensteps + 24 * gsi), i, o, d);
    Prd prd;
    trace<64, EXT>(P, s_lane + lane, o, d, P.tmin, P.tmax, prd);
    simtrace_record(P, out + 4 * i, o, d, prd);
}

/*
 * What the host has to know before a simtrace: the number of rays, and from `least` rays on, of
 * OA_RAY_SAMPLES of them, evenly spread, how many leave the free ball and go on to the instance walk
 * (a count a block, at result_ends of out; none where there is no such ball). It takes the place of a
 * copy of the number, and a few microseconds where it samples.
 */
#define OA_RAY_SAMPLES 4096
__global__ void __launch_bounds__(64) k_ray_sample(SimParams P, LaunchResult* out, int64_t least)
{
    const int64_t n = P.gs_prefix[P.n_gs];
    if (blockIdx.x == 0 && threadIdx.x == 0) out->total = n;
    unsigned long long walkers = 0ull;
    if (n >= least && P.front_plain && !P.tlas_empty) {
        const int64_t k = (int64_t)blockIdx.x * 64 + threadIdx.x, i = n / OA_RAY_SAMPLES * k + n % OA_RAY_SAMPLES * k / OA_RAY_SAMPLES;
        const int64_t gsi = upper_index(P.gs_prefix, 0, P.n_gs, i);
        v3 o, d;
        simtrace_ray(P, reinterpret_cast<const float4*>(P.gensteps + 24 * gsi), i, o, d);
        Nearest best;
        nearest_none(best, P.tmax);
        trace_front(P, o, d, P.tmin, best);
        float tlo = P.tmin;
        const float4 fb = const_load(const_ptr(P.free_ball));
        walkers = __ballot(fb.w > 0.f && beyond_free_ball(fb, o, d, P.tmin, best.t, tlo));
    }
    if (threadIdx.x == 0) result_ends(out)[blockIdx.x] = (uint64_t)__popcll(walkers);
}

/* words of a ray in a wave's queue */
#define OA_RAY_WORDS 16

/*
 * CSGOptiX7.cu:563-604 simtrace: one ray per photon of OpticksGenstep_FRAME gensteps, the
 * nearest hit that oa::trace finds. A ray is all that a lane carries, so a wave need not
 * follow 64 of them from start to end. Rays are made and tested against the front instances
 * 64 at a time, and those not settled by them go to a queue in LDS. Lanes are persistent, each
 * at its own point of its own walk (trace's two phases), and the wave does next what enough
 * of them want: lanes that hold an instance leaf wait until OA_RAY_LEAVES do, lanes whose ray
 * is settled until OA_RAY_REFILL are, and record and refill together; the others walk nodes
 * meanwhile. Bound by instruction issue, most of it the CSG trees of the leaf phase: with 64
 * rays from start to end a tree ran on 15 lanes, since a third of a grid's rays meet an
 * instance at all. 10.1M rays among 2,000 detectors: 1.72 ms before, 1.45 ms. OA_RAY_LEAVES 32 /
 * 40 / 48 / 56: 1.55 / 1.47 / 1.45 / 1.47 ms; OA_RAY_REFILL 8 / 12 / 16 / 24: 1.48 / 1.45 / 1.47 / 1.47.
 * Waves claim rays from a counter (P.next, zero at the start), since those among the detectors
 * take longest: dealt out in advance, 2.40 ms. A claim is 256 rays, the counter being one word
 * (64: 2.18 ms, 128: 1.52, 256: 1.45).
 */
#define OA_RAY_LEAVES 48
#define OA_RAY_REFILL 12
#define OA_RAY_CLAIM 256
#define OA_RAY_QUEUE (OA_RAY_REFILL + 64)
template <bool EXT>
__global__ void __launch_bounds__(64) OA_OCC k_simtrace(SimParams P, float4* out)
{
    extern __shared__ uint32_t s_lane[];             /* the queue, then each lane's stack */
    uint32_t* stk = s_lane + OA_RAY_WORDS * OA_RAY_QUEUE + threadIdx.x;
    const int lane = threadIdx.x;
    const float4 fb = const_load(const_ptr(P.free_ball));
    int64_t next = 0, end = 0;                       /* what is left of the claimed rays */
    bool more = true;
    int queued = 0;
    int64_t idx = -1;                                /* this lane's ray; it is settled when `done` */
    bool done = true;
    v3 o = mk(0.f, 0.f, 0.f), d = o;
    float tlo = 0.f;
    Nearest best;
    nearest_none(best, P.tmax);
    int sp = 0;
    uint32_t cur = OA_BVH_EMPTY, leaf = OA_BVH_EMPTY;
    for (;;) {
        const unsigned long long free_lanes = __ballot(done);
        const int n_free = __popcll(free_lanes);
        if (n_free == 64 || (n_free >= OA_RAY_REFILL && more)) {
            if (done && idx >= 0) {
                Prd prd;
                hit_record(P, best, o, d, prd);
                simtrace_record(P, out + 4 * idx, o, d, prd);
                idx = -1;
            }
            while (queued < OA_RAY_REFILL) {
                if (next == end) {
                    unsigned long long c = 0ull;
                    if (lane == 0) c = atomicAdd(P.next, (unsigned long long)OA_RAY_CLAIM);
                    next = (int64_t)__shfl(c, 0);
                    end = next + OA_RAY_CLAIM < P.n_photon ? next + OA_RAY_CLAIM : P.n_photon;
                    if (next >= P.n_photon) { next = end; break; }
                }
                const int64_t last = (next + 64 < end ? next + 64 : end) - 1, i = next + lane;
                const int64_t g0 = wave_upper_index(P.gs_prefix, P.n_gs, next, lane);
                const int64_t g1 = g0 + wave_upper_index(P.gs_prefix + g0, P.n_gs - g0, last, lane);
                bool walks = i <= last;
                v3 ro = mk(0.f, 0.f, 0.f), rd = ro;
                Nearest rb;
                nearest_none(rb, P.tmax);
                float rlo = P.tmin;
                if (walks) {
                    const int64_t gsi = upper_index(P.gs_prefix, g0, g1 + 1, i);
                    simtrace_ray(P, reinterpret_cast<const float4*>(P.gensteps + 24 * gsi), i, ro, rd);
                    if (P.front_plain) {
                        trace_front(P, ro, rd, P.tmin, rb);
                        walks = !P.tlas_empty && beyond_free_ball(fb, ro, rd, P.tmin, rb.t, rlo);
                    }
                    if (!walks) {
                        Prd prd;
                        hit_record(P, rb, ro, rd, prd);
                        simtrace_record(P, out + 4 * i, ro, rd, prd);
                    }
                }
                const unsigned long long m = __ballot(walks);
                if (walks) {
                    uint32_t* w = s_lane + queued + __popcll(m & ((1ull << lane) - 1ull));
                    const uint32_t v[OA_RAY_WORDS] = {
                        (uint32_t)i, (uint32_t)((uint64_t)i >> 32), fbits(ro.x), fbits(ro.y), fbits(ro.z), fbits(rd.x),
                        fbits(rd.y), fbits(rd.z), fbits(rb.t), rb.inst, rb.prim, fbits(rb.is.x), fbits(rb.is.y),
                        fbits(rb.is.z), fbits(rb.is.w), fbits(rlo) };
#pragma unroll
                    for (int q = 0; q < OA_RAY_WORDS; ++q) w[q * OA_RAY_QUEUE] = v[q];
                }
                queued += __popcll(m);
                next = last + 1;
            }
            more = queued > 0;
            /* one wave to a block: the queue's stores are in before it is read */
            __syncthreads();
            const int take = n_free < queued ? n_free : queued;
            if (take == 0 && n_free == 64) break;
            queued -= take;
            const int rank = __popcll(free_lanes & ((1ull << lane) - 1ull));
            if (done && rank < take) {
                uint32_t v[OA_RAY_WORDS];
#pragma unroll
                for (int q = 0; q < OA_RAY_WORDS; ++q) v[q] = s_lane[queued + rank + q * OA_RAY_QUEUE];
                idx = (int64_t)((uint64_t)v[0] | ((uint64_t)v[1] << 32));
                o = mk(__uint_as_float(v[2]), __uint_as_float(v[3]), __uint_as_float(v[4]));
                d = mk(__uint_as_float(v[5]), __uint_as_float(v[6]), __uint_as_float(v[7]));
                best.t = __uint_as_float(v[8]);
                best.inst = v[9];
                best.prim = v[10];
                best.key = best.inst == 0xffffffffu ? ~0ull : ((uint64_t)best.inst << 32) | best.prim;
                best.is.x = __uint_as_float(v[11]); best.is.y = __uint_as_float(v[12]);
                best.is.z = __uint_as_float(v[13]); best.is.w = __uint_as_float(v[14]);
                tlo = __uint_as_float(v[15]);
                sp = 0;
                cur = P.tlas_empty ? OA_BVH_EMPTY : 0u;
                leaf = P.front_plain ? OA_BVH_EMPTY : P.front_leaf;
                done = false;
            }
            __syncthreads();
        }
        v3 inv, oi;
        slab_ray(o, d, inv, oi);
        unsigned long long walking, holding;
        for (;;) {
            holding = __ballot(!done && leaf != OA_BVH_EMPTY);
            walking = __ballot(!done && leaf == OA_BVH_EMPTY);
            if (walking == 0ull || __popcll(holding) >= OA_RAY_LEAVES) break;
            if (more && __popcll(~(holding | walking)) >= OA_RAY_REFILL) break;
            if (!done && leaf == OA_BVH_EMPTY) done = walk_nodes<64>(P, inv, oi, tlo, best, stk, sp, cur, leaf);
        }
        if (__popcll(holding) < OA_RAY_LEAVES && more && __popcll(~(holding | walking)) >= OA_RAY_REFILL) continue;
        if (!done && leaf != OA_BVH_EMPTY) {
            const uint32_t at = leaf;
            leaf = OA_BVH_EMPTY;
            test_leaf<64, EXT>(P, at, o, d, P.tmin, tlo, best, stk, sp);
            /* after a front leaf (the TLAS walk not begun: cur is still the root) */
            if (cur == 0u && !beyond_free_ball(fb, o, d, P.tmin, best.t, tlo)) cur = OA_BVH_EMPTY;
        }
    }
}

/* ---------------------------------------------------- hit compaction */

/*
 * Stable compaction of the hits, one pass: a block takes a tile of 256 bitmask words (16,384
 * photons), counts them, gets the hits before it by a decoupled look-back over the tiles'
 * published counts (D. Merrill, M. Garland, "Single-pass parallel prefix scan with decoupled
 * look-back", NVR-2016-002) and copies its hit records. state[tile] is 0, then count | 1 << 62,
 * then (hits up to the tile's end) | 2 << 62, one word each, so no ordering with other memory
 * is needed; the ticket hands out the tiles, so a tile's predecessors are always running or
 * done. Both start at zero. Where the count is the device's (n_dev), the blocks beyond its tiles
 * leave without a ticket: they are as many as the largest event's tiles.
 * A tile lists its hit photons in LDS first, so that four neighbouring lanes copy one 64 B
 * record: with a lane per photon and a hit fraction of a tenth, most lanes of a wave only
 * watched the others copy. It replaces a count, a scan and a scatter kernel (17 us together on
 * small events). Large launches are bound by the tickets, one atomic on one word for 2 MB of photon
 * records, at the 40-70 ns that such an atomic takes over eight L2s, and close to it by the bytes of
 * the hits: 10M photons with 9.5M hits 291 us (1.2 GB, 611 tiles), 255M with 28.6M 1,054 us (3.7 GB,
 * 15,600 tiles: 68 ns each). (The merge, with a tile of 2,048 records, does without tickets.) Few
 * photons with many hits are bound by what one block copies: 95,000 hits in seven tiles 29 us.
 * word_prefix (hits of the tile before each word) and tile_base (hits before each tile, then
 * the total) serve k_hit_event_offsets. out: null, or host-visible words for the total and
 * the wall clock at the start and end.
 */
__global__ void __launch_bounds__(256) k_compact(const unsigned long long* __restrict__ words, int64_t n_photon,
                                                 const int64_t* n_dev, int32_t* word_prefix, int64_t* tile_base,
                                                 unsigned long long* ticket, unsigned long long* state,
                                                 const float4* __restrict__ photon, float4* __restrict__ hit,
                                                 int64_t hit_cap, LaunchResult* out)
{
    __shared__ int32_t s_wave[4];
    __shared__ int64_t s_tile, s_base;
    __shared__ uint16_t s_list[256 * 64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t n = n_dev ? *n_dev : n_photon;
    const int64_t n_words = (n + 63) / 64, n_tiles = (n_words + 255) / 256;
    if ((int64_t)blockIdx.x >= n_tiles) return;
    if (t == 0) s_tile = (int64_t)atomicAdd(ticket, 1ull);
    __syncthreads();
    const int64_t tile = s_tile;
    if (out && tile == 0 && t == 0) out->compaction_begins = wall_clock64();
    const int64_t w = tile * 256 + t;
    unsigned long long m = w < n_words ? words[w] : 0ull;
    const int32_t c = __popcll(m);
    int32_t incl = c;
    for (int o = 1; o < 64; o <<= 1) {
        const int32_t v = __shfl_up(incl, o);
        if (lane >= o) incl += v;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    int32_t before = incl - c;
    for (int q = 0; q < wave; ++q) before += s_wave[q];
    const int32_t total = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
    const unsigned long long kCount = 1ull << 62, kDone = 2ull << 62, kValue = kCount - 1ull;
    if (wave == 0) {
        int64_t base = 0;
        if (tile > 0) {
            if (lane == 0)
                __hip_atomic_store(&state[tile], kCount | (unsigned long long)total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            /* 64 tiles at a time, the nearest in lane 0 */
            for (int64_t k = tile - 1;; k -= 64) {
                const int64_t mine = k - lane;
                unsigned long long v = kDone;               /* before the first tile: nothing, and the end */
                do {
                    if (mine >= 0) v = __hip_atomic_load(&state[mine], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } while (__ballot(v < kCount) != 0ull);
                const unsigned long long ends = __ballot(v >= kDone);
                const int last = ends ? __ffsll((long long)ends) - 1 : 63;
                int64_t sum = lane <= last ? (int64_t)(v & kValue) : 0;
                for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
                base += sum;
                if (ends) break;
            }
        }
        if (lane == 0) {
            __hip_atomic_store(&state[tile], kDone | (unsigned long long)(base + total), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            s_base = base;
            tile_base[tile] = base;
            if (tile == n_tiles - 1) tile_base[n_tiles] = base + total;
        }
    }
    if (w < n_words) word_prefix[w] = before;
    if (hit && photon) {
        for (int32_t k = before; m; m &= m - 1ull) s_list[k++] = (uint16_t)(t * 64 + __ffsll((long long)m) - 1);
    }
    __syncthreads();
    const int64_t base = s_base;
    if (hit && photon) {
        const int64_t room = hit_cap - base;
        const int32_t n4 = 4 * (int32_t)(room < total ? (room > 0 ? room : 0) : total);
        const float4* src = photon + 4 * tile * 16384;
        float4* dst = hit + 4 * base;
        int32_t i = t;
        /* four records' quarters in flight a lane */
        for (; i + 768 < n4; i += 1024) {
            float4 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = src[4 * (int)s_list[(i + 256 * u) >> 2] + (i & 3)];
#pragma unroll
            for (int u = 0; u < 4; ++u) dst[i + 256 * u] = v[u];
        }
        for (; i < n4; i += 256) dst[i] = src[4 * (int)s_list[i >> 2] + (i & 3)];
    }
    if (!out) return;
    if (tile == n_tiles - 1 && t == 0) out->n_hit = base + total;
    __syncthreads();
    if (t == 0) result_ends(out)[OA_SETUP_BLOCKS + tile] = wall_clock64();
}

/* hits among photons [0, ph) for each event boundary ph = ev_ph_begin[e] */
__global__ void k_hit_event_offsets(const unsigned long long* words, const int32_t* word_prefix,
                                    const int64_t* tile_base, const int64_t* ev_ph_begin, int32_t n_event,
                                    int64_t n_words, int64_t* hit_offsets)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e > n_event) return;
    const int64_t ph = ev_ph_begin[e];
    const int64_t w = ph >> 6;
    int64_t r;
    if (w >= n_words) r = tile_base[(n_words + 255) / 256];
    else r = tile_base[w >> 8] + word_prefix[w] + __popcll(words[w] & ((1ull << (ph & 63)) - 1ull));
    hit_offsets[e] = r;
}

/* --------------------------------------------------------- trace query */

template <int BLOCK, bool EXT>
__global__ void __launch_bounds__(BLOCK) k_trace(SimParams P, const float4* rays, int64_t n, float4* out)
{
    __shared__ uint32_t s_stack[OA_STACK_DEPTH * BLOCK];
    const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    const float4 a = rays[2 * i], b = rays[2 * i + 1];
    Prd prd;
    trace<BLOCK, EXT>(P, s_stack + threadIdx.x, mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), a.w, b.w, prd);
    const bool miss = prd.boundary == 0xffffu;
    const v3 nn = miss ? prd.normal : normalize(prd.normal);
    out[2 * i] = make_float4(nn.x, nn.y, nn.z, prd.t);
    const uint32_t inst = miss ? 0xffffffffu : (prd.iindex_identity >> 16);
    out[2 * i + 1] = make_float4(__uint_as_float(prd.iindex_identity), __uint_as_float(prd.boundary),
                                 prd.lposcost, __uint_as_float(inst));
}

/* --------------------------------------------------------------- refit */

/* union of a node's non-empty child boxes */
__device__ static void node_box(const BvhNode& n, float* lo, float* hi)
{
    for (int k = 0; k < 3; ++k) { lo[k] = 1e30f; hi[k] = -1e30f; }
    for (int c = 0; c < OA_BVH_WIDTH; ++c) {
        if (n.child[c] == OA_BVH_EMPTY) continue;
        lo[0] = fminf(lo[0], n.lox[c]); lo[1] = fminf(lo[1], n.loy[c]); lo[2] = fminf(lo[2], n.loz[c]);
        hi[0] = fmaxf(hi[0], n.hix[c]); hi[1] = fmaxf(hi[1], n.hiy[c]); hi[2] = fmaxf(hi[2], n.hiz[c]);
    }
}

/* box of one child link: a node's children, or the world boxes of a leaf's instances */
__device__ static void link_box(const BvhNode* nodes, const uint32_t* items, const float* inst_box, uint32_t c,
                                float* lo, float* hi)
{
    for (int k = 0; k < 3; ++k) { lo[k] = 1e30f; hi[k] = -1e30f; }
    if (c == OA_BVH_EMPTY) return;
    if (c & OA_BVH_LEAF_BIT) {
        const uint32_t f = c & 0x00ffffffu, n = (c >> 24) & 0x7fu;
        for (uint32_t j = 0; j < n; ++j) {
            const float* b = inst_box + 6 * items[f + j];
            for (int k = 0; k < 3; ++k) { lo[k] = fminf(lo[k], b[k]); hi[k] = fmaxf(hi[k], b[3 + k]); }
        }
    } else {
        node_box(nodes[c], lo, hi);
    }
}

/* refit all TLAS nodes of one depth (deepest level first) */
__global__ void k_refit_level(BvhNode* nodes, int64_t n_nodes, uint32_t depth, const uint32_t* items,
                              const float* inst_box)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_nodes) return;
    BvhNode& n = nodes[i];
    if (n.depth != depth) return;
    for (int c = 0; c < OA_BVH_WIDTH; ++c) {
        if (n.child[c] == OA_BVH_EMPTY) continue;
        float lo[3], hi[3];
        link_box(nodes, items, inst_box, n.child[c], lo, hi);
        n.lox[c] = lo[0]; n.loy[c] = lo[1]; n.loz[c] = lo[2];
        n.hix[c] = hi[0]; n.hiy[c] = hi[1]; n.hiz[c] = hi[2];
    }
}

/* ------------------------------------------------------ host launchers */

namespace oa_launch {

/* histograms (2 x 32) and slow-trace records (up to OA_SLOW_MAX x 3 float4)
   of an OA_STATS build; returns the number of slow traces seen, or -1 */
extern "C" long long oa_stats_dump(unsigned long long* hist64, float* slow, int reset)
{
#ifdef OA_STATS
    unsigned long long n = 0;
    if (hipMemcpyFromSymbol(hist64, HIP_SYMBOL(oa_hist), sizeof(unsigned long long) * 64) != hipSuccess) return -1;
    if (hipMemcpyFromSymbol(&n, HIP_SYMBOL(oa_slow_n), sizeof(n)) != hipSuccess) return -1;
    if (slow && hipMemcpyFromSymbol(slow, HIP_SYMBOL(oa_slow), sizeof(float4) * OA_SLOW_MAX * 3) != hipSuccess) return -1;
    if (reset) {
        static const unsigned long long zh[64] = {};
        const unsigned long long z = 0;
        if (hipMemcpyToSymbol(HIP_SYMBOL(oa_hist), zh, sizeof(zh)) != hipSuccess) return -1;
        if (hipMemcpyToSymbol(HIP_SYMBOL(oa_slow_n), &z, sizeof(z)) != hipSuccess) return -1;
    }
    return (long long)n;
#else
    (void)hist64; (void)slow; (void)reset;
    return -1;
#endif
}

/* counters of an OA_STATS build (zeros otherwise) */
extern "C" int oa_stats_read(unsigned long long* out, int reset)
{
#ifdef OA_STATS
    if (hipMemcpyFromSymbol(out, HIP_SYMBOL(oa_stats), sizeof(unsigned long long) * OA_ST_N) != hipSuccess) return -1;
    if (reset) {
        unsigned long long z[OA_ST_N] = {};
        if (hipMemcpyToSymbol(HIP_SYMBOL(oa_stats), z, sizeof(z)) != hipSuccess) return -1;
    }
#else
    for (int i = 0; i < OA_ST_N; ++i) out[i] = 0ull;
    (void)reset;
#endif
    return 0;
}

hipError_t seed_map(const int64_t* d_prefix, int64_t n_gs, int64_t n_photon, uint32_t* d_seed,
                    const int64_t* d_ev_gs_begin, int32_t n_event, int32_t* d_gs_event, hipStream_t s)
{
    const unsigned gb = (unsigned)std::min<int64_t>(std::max<int64_t>(n_gs, 1), 65535);
    hipLaunchKernelGGL(k_seed_fill, dim3(gb), dim3(256), 0, s, d_prefix, n_gs, n_photon, d_seed);
    if (n_event > 1) {
        const unsigned eb = (unsigned)std::min<int32_t>(n_event, 65535);
        hipLaunchKernelGGL(k_gs_event, dim3(eb), dim3(256), 0, s, d_ev_gs_begin, n_event, d_gs_event);
    }
    return hipGetLastError();
}

int64_t gs_prefix_words(int64_t n_gs) { return n_gs + 1 + (n_gs + 1023) / 1024; }

hipError_t gs_prefix(const float* d_gs, int64_t n_gs, int64_t* d_prefix, hipStream_t s, LaunchResult* out)
{
    const unsigned nb = (unsigned)((n_gs + 1023) / 1024);
    int64_t* sums = d_prefix + n_gs + 1;
    if (nb > 1) hipLaunchKernelGGL(k_gs_sums, dim3(nb), dim3(1024), 0, s, d_gs, n_gs, sums, out);
    hipLaunchKernelGGL(k_gs_prefix, dim3(nb), dim3(1024), 0, s, d_gs, n_gs, sums, d_prefix);
    return hipGetLastError();
}

int setup_blocks(int64_t cap)
{
    const int64_t work = std::max<int64_t>(cap / 8, clear_words(cap));
    return (int)std::min<int64_t>(OA_SETUP_BLOCKS, (work + 255) / 256 + 1);
}

hipError_t setup(const SetupArgs& a, hipStream_t s)
{
    const unsigned nb = (unsigned)setup_blocks(a.cap);
    if (a.n_gs <= OA_SETUP_GS) {
        hipLaunchKernelGGL(k_setup<true>, dim3(nb), dim3(256), 0, s, a.gs, a.n_gs, a.n_arg, a.cap, a.prefix, a.seed, a.words,
                           bitmask_offset(a.cap), a.ev, a.ev_id, a.event_id, a.n_dev, a.out, a.n_wave);
    } else {
        const hipError_t e = gs_prefix(a.gs, a.n_gs, a.prefix, s, a.out);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_setup<false>, dim3(nb), dim3(256), 0, s, a.gs, a.n_gs, a.n_arg, a.cap, a.prefix, a.seed, a.words,
                           bitmask_offset(a.cap), a.ev, a.ev_id, a.event_id, a.n_dev, a.out, a.n_wave);
    }
    return hipGetLastError();
}

/* P.rng_kind selects the instantiation: 0 Philox, 1 precooked, 2 xorwow */
#define OA_SIM_BY_RNG(fn, B, ...)                                                         \
    (P.rng_kind == 1 ? fn##_##B##_1(__VA_ARGS__) : P.rng_kind == 2 ? fn##_##B##_2(__VA_ARGS__) \
                                                 : fn##_##B##_0(__VA_ARGS__))

int wave_blocks_per_cu(int block, int rng_kind, int stack_depth, bool lite, bool ext, bool tape)
{
#define OA_OCCUPANCY(B)                                                                   \
    (rng_kind == 1 ? sim_occupancy_##B##_1(stack_depth, f, tape)                          \
     : rng_kind == 2 ? sim_occupancy_##B##_2(stack_depth, f, tape) : sim_occupancy_##B##_0(stack_depth, f, tape))
    const int f = (lite ? 1 : 0) | (ext ? 2 : 0);
    switch (block) {
        case 64: return OA_OCCUPANCY(64);
        case 128: return OA_OCCUPANCY(128);
        case 256: return OA_OCCUPANCY(256);
        default: return 0;
    }
#undef OA_OCCUPANCY
}

unsigned sim_lds(int block, int rng_kind, int stack_depth)
{
    const unsigned b64 = rng_kind == 1 ? sim_lds_64_1(stack_depth) : rng_kind == 2 ? sim_lds_64_2(stack_depth)
                                                                                   : sim_lds_64_0(stack_depth);
    return b64 * (unsigned)(block / 64);
}

hipError_t simulate(const SimParams& P, int kernel, int block, int grid, hipStream_t s)
{
    switch (block) {
        case 64: return OA_SIM_BY_RNG(sim_launch, 64, P, kernel, grid, s);
        case 128: return OA_SIM_BY_RNG(sim_launch, 128, P, kernel, grid, s);
        case 256: return OA_SIM_BY_RNG(sim_launch, 256, P, kernel, grid, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t compact_hits(unsigned long long* d_words, int64_t n_photon, const int64_t* n_dev, int32_t* d_word_prefix,
                        int64_t* d_tile_base, const float4* d_photon, float4* d_hit, int64_t hit_cap, LaunchResult* out,
                        hipStream_t s)
{
    const int64_t nt = compact_tiles(n_photon);
    if (nt > 0)
        hipLaunchKernelGGL(k_compact, dim3((unsigned)nt), dim3(256), 0, s, d_words + bitmask_offset(n_photon), n_photon,
                           n_dev, d_word_prefix, d_tile_base, d_words + OA_WORDS_TICKET, d_words + OA_WORDS_STATE, d_photon,
                           d_hit, hit_cap, out);
    return hipGetLastError();
}

hipError_t event_hit_offsets(const unsigned long long* d_words, const int32_t* d_word_prefix,
                             const int64_t* d_block_total, const int64_t* d_ev_ph_begin, int32_t n_event,
                             int64_t n_words, int64_t* d_hit_offsets, hipStream_t s)
{
    hipLaunchKernelGGL(k_hit_event_offsets, dim3((n_event + 1 + 255) / 256), dim3(256), 0, s,
                       d_words, d_word_prefix, d_block_total, d_ev_ph_begin, n_event, n_words, d_hit_offsets);
    return hipGetLastError();
}

__global__ void k_zero_u64(unsigned long long* p, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

__global__ void k_zero_u32(uint32_t* p, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

__global__ void k_prefix_check(const int64_t* a, const int64_t* b, int64_t n, unsigned long long* flag)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && a[i] != b[i]) flag[0] = 1ull;
}

hipError_t prefix_check(const int64_t* a, const int64_t* b, int64_t n, unsigned long long* flag, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_prefix_check, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, b, n, flag);
    return hipGetLastError();
}

__global__ void k_clear_launch(unsigned long long* p, int64_t n, unsigned long long next)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i == 0 ? next : 0ull;
}

hipError_t clear_launch(unsigned long long* words, int64_t n_photon, int64_t n_wave, hipStream_t s)
{
    const int64_t n = clear_words(n_photon);
    hipLaunchKernelGGL(k_clear_launch, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, words, n,
                       (unsigned long long)(n_wave * wave_width(n_photon, n_wave)));
    return hipGetLastError();
}

hipError_t zero_u64(unsigned long long* p, int64_t n, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_zero_u64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

/*
 * Persistent waves pay where many rays walk: every claim of rays is an atomic on one word, about 14 ns
 * apiece, which rays that the front instances settle do not repay, and the last rays of a wave run
 * alone. A ray to a lane / persistent, in us, on grids of a 2,000-detector shell by the share of
 * walkers: 4M rays, 0.16 459 / 615, 0.30 696 / 750, 0.36 780 / 792, 0.47 951 / 832; 10M, 0: 427 / 614,
 * 0.16 1,043 / 1,081, 0.22 1,287 / 1,227, 0.42 1,968 / 1,568; 24M, 0.13 2,108 / 2,073, 0.19 2,638 / 2,407.
 * With 20,000 and 60,000 detectors the persistent waves are ahead a little sooner (4M rays, 0.28;
 * 10M, 0.15), on a line of gensteps later. So the line is a number of walkers, 1.6M, and a share of one in eight for
 * the claims of the others; fewer than 4M rays (2M, all walking: 420 / 591) are not sampled. Without a
 * free ball all rays walk, most of them a step or two and in step with their neighbours: a ray to a
 * lane there (6M rays among clusters of prims 552 / 748, among Boolean solids 675 / 1,006 from one point
 * and 1,298 / 985 from a hundred, among the extended leaves 1,040 / 1,170 and 1,127 / 1,011).
 */
#define OA_RAY_MANY 4000000
#define OA_RAY_WALKERS 1600000
hipError_t ray_sample(const SimParams& P, LaunchResult* out, hipStream_t s)
{
    hipLaunchKernelGGL(k_ray_sample, dim3(OA_RAY_SAMPLES / 64), dim3(64), 0, s, P, out, (int64_t)OA_RAY_MANY);
    return hipGetLastError();
}

hipError_t simtrace(const SimParams& P, float4* out, const LaunchResult* sample, hipStream_t s)
{
    int64_t of = 0;
    if (P.n_photon >= OA_RAY_MANY)
        for (int k = 0; k < OA_RAY_SAMPLES / 64; ++k) of += (int64_t)result_ends(sample)[k];
    const int64_t walkers = P.n_photon / OA_RAY_SAMPLES * of;
    if (walkers < OA_RAY_WALKERS || 8 * of < OA_RAY_SAMPLES) {
        const dim3 grid((unsigned)((P.n_photon + 63) / 64));
        const unsigned stacks = 64u * (unsigned)P.stack_depth * 4u;
        if (P.ext_leaves) hipLaunchKernelGGL(k_simtrace_few<true>, grid, dim3(64), stacks, s, P, out);
        else hipLaunchKernelGGL(k_simtrace_few<false>, grid, dim3(64), stacks, s, P, out);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, s, P.next, (int64_t)1);
    const unsigned lds = (unsigned)(OA_RAY_WORDS * OA_RAY_QUEUE + 64 * P.stack_depth) * 4u;
    int dev = 0, n_cu = 0, per_cu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess)
        e = P.ext_leaves ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_simtrace<true>, 64, lds)
                         : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_simtrace<false>, 64, lds);
    if (e != hipSuccess) return e;
    const int64_t need = (P.n_photon + 63) / 64, slots = (int64_t)n_cu * (per_cu > 0 ? per_cu : 8);
    const unsigned nb = (unsigned)(need < slots ? need : slots);
    if (P.ext_leaves) hipLaunchKernelGGL(k_simtrace<true>, dim3(nb), dim3(64), lds, s, P, out);
    else hipLaunchKernelGGL(k_simtrace<false>, dim3(nb), dim3(64), lds, s, P, out);
    return hipGetLastError();
}

hipError_t trace(const SimParams& P, const float4* rays, int64_t n, float4* out, hipStream_t s)
{
    if (P.ext_leaves) hipLaunchKernelGGL((k_trace<128, true>), dim3((unsigned)((n + 127) / 128)), dim3(128), 0, s, P, rays, n, out);
    else hipLaunchKernelGGL((k_trace<128, false>), dim3((unsigned)((n + 127) / 128)), dim3(128), 0, s, P, rays, n, out);
    return hipGetLastError();
}

hipError_t refit(BvhNode* d_tlas, int64_t n_tlas, uint32_t max_depth, const uint32_t* d_tlas_items,
                 const float* d_inst_box, hipStream_t s)
{
    for (int d = (int)max_depth; d >= 0; --d)
        hipLaunchKernelGGL(k_refit_level, dim3((unsigned)((n_tlas + 255) / 256)), dim3(256), 0, s,
                           d_tlas, n_tlas, (uint32_t)d, d_tlas_items, d_inst_box);
    return hipGetLastError();
}

} // namespace oa_launch

/* ======================================== adjoint (replay kernel in oa_sim.h) */

/* zero the score rows of the chunk's hits (grid-stride) */
__global__ void k_zero_rows(float* S, int32_t n_param, int64_t begin, int64_t n_max, const int64_t* hit_off,
                            int32_t n_ev, int64_t hit_cap)
{
    const int64_t n = chunk_hits(begin, n_max, hit_off, n_ev, hit_cap) * (int64_t)n_param;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        S[i] = 0.f;
}

/* detector key (sensor_identifier - 1) of each of the chunk's n_max slots;
   non-sensors and slots past the chunk's hits get n_det. With the segment tape
   it also raises the overflow flag for a hit whose photon had more segments
   than the tape holds (that hit is replayed). */
__global__ void k_hit_det(SimParams P, const float4* hits, int64_t begin, int64_t n_max, const int64_t* hit_off,
                          int32_t n_ev, int64_t hit_cap, uint32_t n_det, uint32_t* key, uint32_t* val)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_max) return;
    const int64_t n = chunk_hits(begin, n_max, hit_off, n_ev, hit_cap);
    uint32_t k = n_det;
    if (i < n) {
        const uint32_t id = __float_as_uint(hits[4 * (begin + i) + 3].y) & 0x00ffffffu;
        k = (id >= 1u && id <= n_det) ? id - 1u : n_det;
        if (P.tape) {
            const int64_t g = hit_photon(P, hits, begin + i, hit_off, n_ev);
            if (g >= 0 && (int32_t)P.tape_n[g] > P.tape_k) atomicOr(P.tape_overflow, 1u);
        }
    }
    key[i] = k;
    val[i] = (uint32_t)i;
}

/*
 * Hits per detector (sensor identifier 1..n_det in an sphoton's low 16 identity bits): whole numbers,
 * turned to float in place at the end. A block counts a chunk of at most 65,535 hits in LDS, two
 * detectors to a word (no count of a chunk carries), OA_COUNT_BINS of them (blockIdx.y picks the range),
 * and adds what it has to the totals. Atomics on the totals alone take as long as the busiest
 * detector's hits one after the other, 11 ns each: 2M hits of one detector 22.7 ms, of eight 7.5, of
 * 2,000 evenly 0.27; so 44, 43 and 45 us with three launches, bound by the 64 B line fetched for each hit
 * (9M: 0.12 ms). 64 / 128 / 256 / 512 blocks: 47 / 44 / 45 / 45 us, of 20,000 detectors 50 / 51 / 57 / 57.
 */
#define OA_COUNT_BINS 32768
#define OA_COUNT_BLOCKS 256
__global__ void __launch_bounds__(1024) k_hit_counts(const uint32_t* __restrict__ hits, int64_t n, uint32_t chunk,
                                                     uint32_t n_det, uint32_t* count)
{
    extern __shared__ uint32_t s_pairs[];
    const uint32_t lo = blockIdx.y * OA_COUNT_BINS, bins = n_det - lo < OA_COUNT_BINS ? n_det - lo : OA_COUNT_BINS;
    for (uint32_t b = threadIdx.x; b < (bins + 1) / 2; b += 1024) s_pairs[b] = 0u;
    __syncthreads();
    const int64_t first = (int64_t)blockIdx.x * chunk, end = first + chunk < n ? first + chunk : n;
    for (int64_t i = first + threadIdx.x; i < end; i += 1024) {
        const uint32_t b = (hits[16 * i + 13] & 0xffffu) - 1u - lo;      /* identifier 0 and others: past the bins */
        if (b < bins) atomicAdd(&s_pairs[b >> 1], 1u << (16u * (b & 1u)));
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < bins; b += 1024) {
        const uint32_t c = s_pairs[b >> 1] >> (16u * (b & 1u)) & 0xffffu;
        if (c) atomicAdd(count + lo + b, c);
    }
}

__global__ void k_count_floats(uint32_t* count, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) count[i] = __float_as_uint((float)count[i]);
}

/* start of each detector's run in the sorted keys */
__global__ void k_det_segments(const uint32_t* key, int64_t n, uint32_t n_det, int64_t* seg)
{
    const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (d > (int64_t)n_det) return;
    int64_t lo = 0, hi = n;
    while (lo < hi) { int64_t mid = (lo + hi) >> 1; if (key[mid] < (uint32_t)d) lo = mid + 1; else hi = mid; }
    seg[d] = lo;
}

#ifndef OA_REDUCE_ROWS
#define OA_REDUCE_ROWS 4
#endif

/* G[d,k] = Kahan sum over the detector's hits (in photon order) of S[h,k];
   with first == 0 the sum and its compensation C continue from an earlier
   chunk of hits (chunks are consecutive in photon order) */
__global__ void __launch_bounds__(256) k_det_reduce(const float* S, const uint32_t* order, const int64_t* seg,
                                                    int32_t n_param, float* G, float* C, int first)
{
    const int d = blockIdx.x;
    const int64_t b = seg[d], e = seg[d + 1];
    for (int k = threadIdx.x; k < n_param; k += blockDim.x) {
        const int64_t o = (int64_t)d * n_param + k;
        float sum = first ? 0.f : G[o], c = first ? 0.f : C[o];
        int64_t i = b;
        /* OA_REDUCE_ROWS rows in flight per step (4, 8 and 16 measure alike), summed in the
           same order as one at a time */
        for (; i + OA_REDUCE_ROWS <= e; i += OA_REDUCE_ROWS) {
            float s[OA_REDUCE_ROWS];
#pragma unroll
            for (int u = 0; u < OA_REDUCE_ROWS; ++u) s[u] = S[(int64_t)order[i + u] * n_param + k];
#pragma unroll
            for (int u = 0; u < OA_REDUCE_ROWS; ++u) {
                const float y = s[u] - c;
                const float t = sum + y;
                c = (t - sum) - y;
                sum = t;
            }
        }
        for (; i < e; ++i) {
            const float y = S[(int64_t)order[i] * n_param + k] - c;
            const float t = sum + y;
            c = (t - sum) - y;
            sum = t;
        }
        G[o] = sum;
        C[o] = c;
    }
}

/* Segment-tape scoring fused with the per-detector reduction, one block per
   detector, over its hits in photon order, 256 at a time: each thread fetches
   one hit's photon, segment count and first OA_TAPE_PRE tape records and forms
   their score terms (the ScoreTape terms the replay forms for that photon), all
   threads at once; the round's later segments (hits with more than OA_TAPE_PRE,
   a few percent) are spread over all threads by a prefix sum, their terms kept
   in LDS (up to OA_TAPE_TAIL of them; beyond that the owner forms them itself).
   Then in sub-rounds of `w` hits, the sub-round's threads apply their terms to
   zeroed LDS rows in segment order (a hit the tape could not hold copies the row
   the replay wrote to S), and each thread adds the entries of its parameters
   over those rows to its Kahan sums in hit order and clears them. The rows and
   the summation are those of k_det_reduce over the dense rows, bit for bit,
   without the dense row array. LDS: w rows of n_param + 1 floats (the pad puts
   row t, entry k in bank (t + k) mod 64), then the later segments' terms, their
   offsets per thread and the threads' photons. */
/* records per hit fetched by their owner (4: 120 VGPRs, four waves per SIMD; 8 holds
   the terms in 165 and measures 0.48 against 0.38 ms on 1.98 M hits x 256 parameters),
   and the LDS slots for the round's later segments (4.5% of hit photons on the 10M
   workload have more than 4 segments, about 90 slots per round of 256 hits) */
#ifndef OA_TAPE_PRE
#define OA_TAPE_PRE 4
#endif
#ifndef OA_TAPE_TAIL
#define OA_TAPE_TAIL 256
#endif

/* a later segment's term in LDS: i0 | i1 << 16 (i2, i3 = i0, i1 + n_bin; all ones: no
   term), sa, ss, a */
OA_D float4 pack_term(const ScoreTerm& t)
{
    const uint32_t w = t.on ? ((uint32_t)t.i0 | ((uint32_t)t.i1 << 16)) : 0xffffffffu;
    return make_float4(__uint_as_float(w), t.sa, t.ss, t.a);
}

OA_D ScoreTerm unpack_term(float4 v, int32_t n_bin)
{
    ScoreTerm t;
    const uint32_t w = __float_as_uint(v.x);
    t.on = w != 0xffffffffu;
    t.i0 = (int32_t)(w & 0xffffu);
    t.i1 = (int32_t)(w >> 16);
    t.i2 = t.i0 + n_bin;
    t.i3 = t.i1 + n_bin;
    t.sa = v.y; t.ss = v.z; t.a = v.w;
    return t;
}

OA_D ScoreTerm record_term(const SimParams& P, const ScoreTape& tape, int64_t g, int j)
{
    const uint32_t* rec = tape_record(P, g, j);
    const uint32_t w0 = rec[0];
    const int line = (int)(w0 & 0x3fffffffu), ev = (int)(w0 >> 30);
    const float wl = __uint_as_float(rec[1]), ell = __uint_as_float(rec[2]);
    const float4 mt = bnd_lookup(P, wl, line, 0);
    return tape.term(line, wl, mt.y, mt.z, ell, ev);
}

template <int NJ>
__global__ void __launch_bounds__(256) k_tape_det_reduce(SimParams P, AdjParams A, const float4* hits, int64_t begin,
                                                         const int64_t* hit_off, int32_t n_ev, const float* S,
                                                         const uint32_t* order, const int64_t* seg, int w, float* G,
                                                         float* C, int first)
{
    using namespace oa;
    extern __shared__ float4 lds4[];
    __shared__ int s_wsum[4];
    const int np = A.n_param, stride = np + 1;
    float* rows = reinterpret_cast<float*>(lds4);
    float4* s_term = lds4 + (w * stride + 3) / 4;                        /* OA_TAPE_TAIL */
    int* s_toff = reinterpret_cast<int*>(s_term + OA_TAPE_TAIL);        /* 257 */
    int64_t* s_tg = reinterpret_cast<int64_t*>(s_toff + 258);           /* 256 */
    const int d = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t b = seg[d], e = seg[d + 1];
    for (int i = tid; i < w * stride; i += 256) rows[i] = 0.f;
    float sum[NJ], c[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int k = tid + 256 * j;
        const int64_t o = (int64_t)d * np + k;
        sum[j] = (first || k >= np) ? 0.f : G[o];
        c[j] = (first || k >= np) ? 0.f : C[o];
    }
    ScoreTape tape;
    tape.optical = P.optical; tape.n_wl = P.n_wl; tape.wl_low = P.wl_low; tape.wl_step = P.wl_step;
    tape.A = A;
    tape.row = nullptr;
    __syncthreads();
    for (int64_t r0 = b; r0 < e; r0 += 256) {
        const int m = (int)(e - r0 < 256 ? e - r0 : 256);
        /* every thread: its hit's photon, count and first records' terms */
        int64_t g = -1;
        uint32_t h = 0;
        int32_t cnt = 0;
        bool dense = false;
        ScoreTerm tm[OA_TAPE_PRE];
        if (tid < m) {
            h = order[r0 + tid];
            g = hit_photon(P, hits, begin + h, hit_off, n_ev);
            if (g >= 0) {
                cnt = P.tape_n[g];
                dense = cnt > P.tape_k;
            }
        }
        uint32_t rw[OA_TAPE_PRE][3];
#pragma unroll
        for (int u = 0; u < OA_TAPE_PRE; ++u) {
            if (!dense && u < cnt) {
                const uint32_t* rec = tape_record(P, g, u);
                rw[u][0] = rec[0]; rw[u][1] = rec[1]; rw[u][2] = rec[2];
            }
        }
#pragma unroll
        for (int u = 0; u < OA_TAPE_PRE; ++u) {
            tm[u].on = false;
            if (!dense && u < cnt) {
                const int line = (int)(rw[u][0] & 0x3fffffffu), ev = (int)(rw[u][0] >> 30);
                const float wl = __uint_as_float(rw[u][1]), ell = __uint_as_float(rw[u][2]);
                const float4 mt = bnd_lookup(P, wl, line, 0);
                tm[u] = tape.term(line, wl, mt.y, mt.z, ell, ev);
            }
        }
        /* later segments: exclusive prefix of their counts over the block, then one
           slot per thread at a time, owner found by binary search of the offsets */
        const int my_tail = (!dense && cnt > OA_TAPE_PRE) ? cnt - OA_TAPE_PRE : 0;
        int incl = my_tail;
        for (int o = 1; o < 64; o <<= 1) {
            const int n = __shfl_up(incl, o);
            if (lane >= o) incl += n;
        }
        if (lane == 63) s_wsum[wave] = incl;
        s_tg[tid] = g;
        __syncthreads();
        int base = 0;
        for (int q = 0; q < wave; ++q) base += s_wsum[q];
        const int my_off = base + incl - my_tail;
        s_toff[tid] = my_off;
        if (tid == 255) s_toff[256] = base + incl;
        __syncthreads();
        const int n_tail = s_toff[256] < OA_TAPE_TAIL ? s_toff[256] : OA_TAPE_TAIL;
        for (int sl = tid; sl < n_tail; sl += 256) {
            int lo = 0, hi = 256;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (s_toff[mid] <= sl) lo = mid; else hi = mid;
            }
            s_term[sl] = pack_term(record_term(P, tape, s_tg[lo], OA_TAPE_PRE + (sl - s_toff[lo])));
        }
        __syncthreads();
        for (int q0 = 0; q0 < m; q0 += w) {
            const int mq = m - q0 < w ? m - q0 : w;
            if (tid >= q0 && tid < q0 + mq && g >= 0) {
                float* row = rows + (tid - q0) * stride;
                if (dense) {
                    const float* src = S + (int64_t)h * np;
                    for (int k = 0; k < np; ++k) row[k] = src[k];
                } else {
#pragma unroll
                    for (int u = 0; u < OA_TAPE_PRE; ++u) ScoreTape::apply(row, tm[u]);
                    for (int32_t j = OA_TAPE_PRE; j < cnt; ++j) {
                        const int sl = my_off + (j - OA_TAPE_PRE);
                        ScoreTape::apply(row, sl < OA_TAPE_TAIL ? unpack_term(s_term[sl], A.n_bin)
                                                                : record_term(P, tape, g, j));
                    }
                }
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int k = tid + 256 * j;
                if (k < np) {
                    float sj = sum[j], cj = c[j];
                    float* q = rows + k;
                    int t = 0;
                    /* eight rows read ahead per step (LDS latency), summed in the same order */
                    for (; t + 8 <= mq; t += 8, q += 8 * stride) {
                        float v[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u) v[u] = q[u * stride];
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            const float y = v[u] - cj;
                            const float tt = sj + y;
                            cj = (tt - sj) - y;
                            sj = tt;
                            q[u * stride] = 0.f;
                        }
                    }
                    for (; t < mq; ++t, q += stride) {
                        const float y = *q - cj;
                        const float tt = sj + y;
                        cj = (tt - sj) - y;
                        sj = tt;
                        *q = 0.f;
                    }
                    sum[j] = sj;
                    c[j] = cj;
                }
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int k = tid + 256 * j;
        if (k < np) {
            const int64_t o = (int64_t)d * np + k;
            G[o] = sum[j];
            C[o] = c[j];
        }
    }
}

#include "oa_radix.h"

namespace oa_launch {

int adjoint_blocks_per_cu(int rng_kind, int stack_depth)
{
    return rng_kind == 1 ? adjoint_occupancy_128_1(stack_depth)
         : rng_kind == 2 ? adjoint_occupancy_128_2(stack_depth) : adjoint_occupancy_128_0(stack_depth);
}

static int det_key_bits(uint32_t n_det)
{
    int end_bit = 1;
    while (end_bit < 32 && (1u << end_bit) <= n_det) ++end_bit;
    return end_bit;
}

/* hits per sub-round of the fused tape reduction (LDS rows; 32 keeps four blocks per
   CU: 16 and 64 measured 10% and 40% slower) */
#ifndef OA_TAPE_ROWS
#define OA_TAPE_ROWS 32
#endif

/* dynamic LDS of the fused tape reduction: w rows of n_param + 1 floats (rounded up to
   16 bytes), OA_TAPE_TAIL terms of 16 bytes, 258 offsets, 256 photon indices */
static size_t tape_reduce_lds(int w, int32_t n_param)
{
    return (size_t)((w * (n_param + 1) + 3) / 4) * 16 + (size_t)OA_TAPE_TAIL * 16 + 258 * 4 + 256 * 8;
}

int tape_reduce_rows(int32_t n_param)
{
    if (n_param > 256 * OA_TAPE_NJ_MAX || n_param > 0xffff) return 0;
    int w = OA_TAPE_ROWS;
    while (w > 0 && tape_reduce_lds(w, n_param) > 65536 - 256) --w;     /* with the kernel's static LDS */
    return w;
}

hipError_t adjoint_chunk(const SimParams& P, const AdjBufs& a, int64_t begin, int64_t n_max, int first, int grid,
                         hipEvent_t mid, hipStream_t s)
{
    AdjParams A;
    A.mat_block = a.mat_block; A.n_mat = a.n_mat; A.sample_bin = a.sample_bin; A.n_bin = a.n_bin; A.n_param = a.n_param;
    const int g = std::max(1, grid);
    const int w = P.tape ? tape_reduce_rows(a.n_param) : 0;
    if (P.tape && w < 1) return hipErrorInvalidValue;
    /* order: detector keys of the chunk's slots (with the tape, the overflow flag too), a
       stable radix sort by detector, and each detector's run */
    auto order = [&]() -> hipError_t {
        if (P.tape) hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, s, P.tape_overflow, (int64_t)1);
        if (n_max > 0) {
            /* the keys are made where an odd or even number of passes ends them in key2, val2 */
            const int bits = det_key_bits(a.n_det);
            const bool even = oa_radix::passes(bits) % 2 == 0;
            uint32_t* k0 = even ? a.key2 : a.key;
            uint32_t* v0 = even ? a.val2 : a.val;
            hipLaunchKernelGGL(k_hit_det, dim3((unsigned)((n_max + 255) / 256)), dim3(256), 0, s, P, a.hit, begin,
                               n_max, a.hit_off, a.n_ev, a.hit_cap, a.n_det, k0, v0);
            hipError_t e = oa_radix::sort(k0, even ? a.key : a.key2, v0, even ? a.val : a.val2, n_max, bits, a.tmp, s);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(k_det_segments, dim3((a.n_det + 1 + 255) / 256), dim3(256), 0, s, a.key2, n_max, a.n_det,
                           a.seg);
        return hipGetLastError();
    };
    /* score rows: the replay of every hit (rows cleared first) or, with the tape, of the
       hits it could not hold (the replay clears their rows; it exits at once when the
       ordering raised no overflow flag) */
    auto replay = [&]() -> hipError_t {
        if (n_max <= 0) return hipGetLastError();
        if (!P.tape)
            hipLaunchKernelGGL(k_zero_rows, dim3((unsigned)(g * 4)), dim3(256), 0, s, a.S, a.n_param, begin, n_max,
                               a.hit_off, a.n_ev, a.hit_cap);
        hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, s, P.next, (int64_t)1);
        return OA_SIM_BY_RNG(adjoint_launch, 128, P, A, a.hit, begin, n_max, a.hit_off, a.n_ev, a.hit_cap, a.S, g, s);
    };
    hipError_t e;
    if (P.tape) {
        if ((e = order()) != hipSuccess || (e = replay()) != hipSuccess) return e;
    } else {
        if ((e = replay()) != hipSuccess || (e = order()) != hipSuccess) return e;
    }
    if (mid && (e = hipEventRecord(mid, s)) != hipSuccess) return e;
    if (!P.tape) {
        hipLaunchKernelGGL(k_det_reduce, dim3(a.n_det), dim3(256), 0, s, a.S, a.val2, a.seg, a.n_param, a.G, a.C, first);
        return hipGetLastError();
    }
    const size_t lds = tape_reduce_lds(w, a.n_param);
    const int nj = (a.n_param + 255) / 256;
#define OA_TAPE_REDUCE(NJ)                                                                                     \
    hipLaunchKernelGGL(k_tape_det_reduce<NJ>, dim3(a.n_det), dim3(256), lds, s, P, A, a.hit, begin, a.hit_off, \
                       a.n_ev, a.S, a.val2, a.seg, w, a.G, a.C, first)
    if (nj <= 1) OA_TAPE_REDUCE(1);
    else if (nj <= 2) OA_TAPE_REDUCE(2);
    else OA_TAPE_REDUCE(4);
#undef OA_TAPE_REDUCE
    return hipGetLastError();
}

hipError_t hit_counts(const void* d_hit, int64_t n, uint32_t n_det, float* d_count, hipStream_t s)
{
    uint32_t* c = reinterpret_cast<uint32_t*>(d_count);
    const dim3 det((n_det + 255u) / 256u);
    hipLaunchKernelGGL(k_zero_u32, det, dim3(256), 0, s, c, (int64_t)n_det);
    if (n > 0) {
        /* identifiers have 16 bits */
        const uint32_t used = n_det < 65535u ? n_det : 65535u, ranges = (used + OA_COUNT_BINS - 1) / OA_COUNT_BINS;
        const int64_t most = OA_COUNT_BLOCKS / ranges, blocks = std::max<int64_t>(std::min<int64_t>(most, (n + 8191) / 8192), (n + 65534) / 65535);
        const uint32_t chunk = (uint32_t)((n + blocks - 1) / blocks);
        const unsigned lds = 4u * ((std::min<uint32_t>(used, OA_COUNT_BINS) + 1u) / 2u);
        hipLaunchKernelGGL(k_hit_counts, dim3((unsigned)blocks, ranges), dim3(1024), lds, s, (const uint32_t*)d_hit, n, chunk,
                           used, c);
    }
    hipLaunchKernelGGL(k_count_floats, det, dim3(256), 0, s, c, (int64_t)n_det);
    return hipGetLastError();
}

size_t adjoint_sort_words(int64_t n_hit, uint32_t n_det) { return oa_radix::words(n_hit, det_key_bits(n_det)); }

} // namespace oa_launch

/* ------------------------------------------- no-allocation scratch */

/* Device memory of the no-allocation simulate entry point: genstep prefix, event
   bounds, refill counter, xorwow jump matrix, hit bitmask and compaction
   prefixes (layout in oa_layout.h). Each GPU holds its own copy for the life of
   the process; every handle on a GPU shares it. */
static __device__ __align__(256) unsigned char scratch[OA_NOALLOC_SCRATCH_BYTES];

/* event bounds {0, n_gs, 0, n_photon} and event id of one no-allocation launch, written by a kernel (no host staging) */
__global__ void k_noalloc_setup(int64_t* ev, int32_t* ev_id, int64_t n_gs, int64_t n_photon, int32_t event_id)
{
    if (threadIdx.x == 0) {
        ev[0] = 0; ev[1] = n_gs; ev[2] = 0; ev[3] = n_photon;
        ev_id[0] = event_id;
    }
}

namespace oa_launch {

#define OA_MAX_DEVICES 64

/* device address of `scratch` on `device`, which must be the current device:
   looked up once per device with hipGetSymbolAddress and kept */
hipError_t noalloc_scratch(int device, void** ptr)
{
    static std::mutex m;
    static void* addr[OA_MAX_DEVICES] = {};
    *ptr = nullptr;
    if (device < 0 || device >= OA_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(m);
    if (!addr[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        addr[device] = p;
    }
    *ptr = addr[device];
    return hipSuccess;
}

hipError_t noalloc_setup(int64_t* ev, int32_t* ev_id, int64_t n_gs, int64_t n_photon, int32_t event_id, hipStream_t s)
{
    hipLaunchKernelGGL(k_noalloc_setup, dim3(1), dim3(64), 0, s, ev, ev_id, n_gs, n_photon, event_id);
    return hipGetLastError();
}

} // namespace oa_launch

/* one translation unit for everything (the OA_STATS counters live in one code object) */
#ifdef OA_SIM_ALL
#define OA_SIM_BLOCK 64
#define OA_SIM_RNG 0
#include "oa_sim.hip"
#undef OA_SIM_RNG
#define OA_SIM_RNG 1
#include "oa_sim.hip"
#undef OA_SIM_RNG
#define OA_SIM_RNG 2
#include "oa_sim.hip"
#undef OA_SIM_RNG
#undef OA_SIM_BLOCK
#define OA_SIM_BLOCK 128
#define OA_SIM_RNG 0
#include "oa_sim.hip"
#undef OA_SIM_RNG
#define OA_SIM_RNG 1
#include "oa_sim.hip"
#undef OA_SIM_RNG
#define OA_SIM_RNG 2
#include "oa_sim.hip"
#undef OA_SIM_RNG
#undef OA_SIM_BLOCK
#define OA_SIM_BLOCK 256
#define OA_SIM_RNG 0
#include "oa_sim.hip"
#undef OA_SIM_RNG
#define OA_SIM_RNG 1
#include "oa_sim.hip"
#undef OA_SIM_RNG
#define OA_SIM_RNG 2
#include "oa_sim.hip"
#undef OA_SIM_RNG
#undef OA_SIM_BLOCK
#endif
