/*
 * oa_merge.hip : hit selection and merging by (sensor identity, time bucket).
 *
 * Restates SPM::merge_partial_select (sysrap/SPM.cu:135-240) for MI355X:
 *   0. select records with flagmask & mask != 0 (skipped for the "already
 *      selected" mask), stable;
 *   1. time window 0: return the selection in input order;
 *   2-4. key = (identity << 48) | (unsigned)(time / window) as a 64-bit
 *      integer, then a stable sort of the selected records by key (oa_radix.h); here the
 *      same order is sorted as identity << b | bucket, with b the bits of the
 *      largest bucket selected and identity its low 16 bits (the shift by 48
 *      keeps the same ones);
 *   6. reduce each run of equal keys with the record type's reduce_op.
 * Record types and their functors:
 *   sphoton     64 B  key/reduce/select  sysrap/sphoton.h:292-320
 *   sphotonlite 16 B  key/reduce/select  sysrap/sphotonlite.h:68-97
 *
 * One pass reads the records (k_select) and keeps of each selected one the 16 bytes that the
 * merge needs, tile by tile, with a count per tile; one block sums the counts (k_tile_offsets)
 * and the keys go to their places by them. Bound by the lines k_select has to fetch, 64 B a
 * photon record for any word of it. The keys are as wide as the selection's largest identity
 * and bucket need, 20 bits for 2,000 sensors and 400 buckets instead of 48: three radix passes
 * over 8-byte pairs instead of six over 12. k_reduce finds the runs again tile by tile and
 * folds each from the kept words, left to right in sorted order, so ties in time keep the
 * earliest record in input order; only the record that a run keeps is fetched.
 * The tiles' offsets come from a small kernel between two passes: a look-back across the tiles
 * needs a ticket each, and tickets, one atomic on one word, come at 40-60 ns apiece over eight
 * L2s (k_select 180 us with 2,441 tiles, 665 with 4,883 and two atomics a tile).
 * 10M records, 2M selected, 0.7M merged: 662 -> 347 us (select 139, keys 11, sort 110, reduce 50;
 * the rest launches and gaps). Before, a flag pass, flagged select, key pass, 48-bit sort,
 * run-length encode and scan, and a reduce over the records themselves.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <utility>
#include "oa_merge.h"
#include "oa_radix.h"

namespace {

struct PhotonAcc {
    /* sphoton: q0 (pos, time), q1 (mom, hitcount_iindex), q2 (pol, wavelength),
       q3 (orient_boundary_flag, identity, index, flagmask) */
    static constexpr int WORDS = 16;
    __device__ static uint32_t identity(const uint32_t* r) { return r[13] & 0x0000ffffu; }   /* 16 bits in the key */
    __device__ static uint32_t time(const uint32_t* r) { return r[3]; }
    __device__ static uint32_t hitcount(const uint32_t* r) { return r[7] >> 16; }
    __device__ static uint32_t flagmask(const uint32_t* r) { return r[15]; }
};

struct LiteAcc {
    /* sphotonlite: hitcount_identity (hi16 hitcount, lo16 identity), time, lpos, flagmask */
    static constexpr int WORDS = 4;
    __device__ static uint32_t identity(const uint32_t* r) { return r[0] & 0x0000ffffu; }
    __device__ static uint32_t time(const uint32_t* r) { return r[1]; }
    __device__ static uint32_t hitcount(const uint32_t* r) { return r[0] >> 16; }
    __device__ static uint32_t flagmask(const uint32_t* r) { return r[3]; }
};

/* a quarter of a record; the arrays that a caller hands in need only their words aligned */
typedef uint32_t quad __attribute__((ext_vector_type(4), aligned(4)));

__device__ inline uint32_t bucket_of(uint32_t time, float tw) { return (uint32_t)(__uint_as_float(time) / tw); }

/* rounds of 256 items that make a tile: records of the selection (their loads are all in
   flight at once), and sorted keys */
#define OA_SELECT_ROUNDS 8
#define OA_REDUCE_ROUNDS 4

/*
 * Ranks of a tile's items, of which thread t marks item 256 k + t by bit k of `marked`: s_pre
 * gets the items before each of the 4 x ROUNDS ballots, rank_in_tile the item's own.
 */
template <int ROUNDS>
__device__ int32_t tile_ranks(uint32_t marked, unsigned long long* s_mask, int32_t* s_pre)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < ROUNDS; ++k) {
        const unsigned long long m = __ballot(marked >> k & 1u);
        if (lane == 0) s_mask[4 * k + wave] = m;
    }
    __syncthreads();
    if (wave == 0) {
        const int32_t c = lane < 4 * ROUNDS ? __popcll(s_mask[lane]) : 0;
        int32_t incl = c;
        for (int o = 1; o < 64; o <<= 1) {
            const int32_t v = __shfl_up(incl, o);
            if (lane >= o) incl += v;
        }
        if (lane < 4 * ROUNDS) s_pre[lane] = incl - c;
        if (lane == 63) s_pre[4 * ROUNDS] = incl;
    }
    __syncthreads();
    return s_pre[4 * ROUNDS];
}

__device__ inline int32_t rank_in_tile(int k, const unsigned long long* s_mask, const int32_t* s_pre)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    return s_pre[4 * k + wave] + __popcll(s_mask[4 * k + wave] & ((1ull << lane) - 1ull));
}

/* a tile's selected, in input order, at the tile's own place in sel; count[tile] of them, and
   the largest identity and bucket */
template <class Acc>
__global__ void __launch_bounds__(256) k_select(const uint32_t* __restrict__ in, int64_t n, uint32_t mask, float tw,
                                                int32_t* count, uint2* most, uint4* __restrict__ sel)
{
    constexpr int ROUNDS = OA_SELECT_ROUNDS;
    __shared__ unsigned long long s_mask[4 * ROUNDS];
    __shared__ int32_t s_pre[4 * ROUNDS + 1];
    __shared__ uint32_t s_max[2];
    if (threadIdx.x < 2) s_max[threadIdx.x] = 0u;
    const int64_t tile = (int64_t)blockIdx.x * (256 * ROUNDS), first = tile + threadIdx.x;
    uint4 v[ROUNDS];
    uint32_t taken = 0, max_id = 0, max_bucket = 0;
#pragma unroll
    for (int k = 0; k < ROUNDS; ++k) {
        const int64_t i = first + k * 256;
        const uint32_t* r = in + (i < n ? i : n - 1) * Acc::WORDS;
        v[k] = make_uint4((uint32_t)i, Acc::time(r), Acc::identity(r) | (Acc::hitcount(r) << 16), Acc::flagmask(r));
    }
#pragma unroll
    for (int k = 0; k < ROUNDS; ++k) {
        const bool take = first + k * 256 < n && (mask == OA_MERGE_ALREADY_SELECTED || (v[k].w & mask) != 0u);
        taken |= (uint32_t)take << k;
        max_id = max(max_id, take ? v[k].z & 0xffffu : 0u);
        max_bucket = max(max_bucket, take ? bucket_of(v[k].y, tw) : 0u);
    }
    const int32_t total = tile_ranks<ROUNDS>(taken, s_mask, s_pre);
#pragma unroll
    for (int k = 0; k < ROUNDS; ++k)
        if (taken >> k & 1u) sel[tile + rank_in_tile(k, s_mask, s_pre)] = v[k];
    for (int o = 32; o > 0; o >>= 1) {
        max_id = max(max_id, (uint32_t)__shfl_xor((int)max_id, o));
        max_bucket = max(max_bucket, (uint32_t)__shfl_xor((int)max_bucket, o));
    }
    if ((threadIdx.x & 63) == 0) { atomicMax(&s_max[0], max_id); atomicMax(&s_max[1], max_bucket); }
    __syncthreads();
    if (threadIdx.x == 0) { count[blockIdx.x] = total; most[blockIdx.x] = make_uint2(s_max[0], s_max[1]); }
}

/* count[0..n) to the items before each tile, in place, and their total into count[n]; that and
   the largest of `most` (null: none) into the host-visible out. One block: 8,192 tiles a step. */
__global__ void __launch_bounds__(1024) k_tile_offsets(int32_t* count, const uint2* most, int64_t n, int64_t* total_out,
                                                       oa_merge::Result* out)
{
    constexpr int EACH = 8;
    __shared__ int32_t s_wave[16];
    __shared__ uint32_t s_max[2];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t < 2) s_max[t] = 0u;
    int32_t base = 0;
    uint32_t max_id = 0, max_bucket = 0;
    for (int64_t i0 = 0; i0 < n; i0 += 1024 * EACH) {
        const int64_t i = i0 + (int64_t)t * EACH;
        int32_t c[EACH], sum = 0;
#pragma unroll
        for (int u = 0; u < EACH; ++u) c[u] = i + u < n ? count[i + u] : 0;
        if (most) {
#pragma unroll
            for (int u = 0; u < EACH; ++u) {
                const uint2 m = most[i + u < n ? i + u : n - 1];
                max_id = max(max_id, m.x);
                max_bucket = max(max_bucket, m.y);
            }
        }
#pragma unroll
        for (int u = 0; u < EACH; ++u) sum += c[u];
        int32_t incl = sum;
        for (int o = 1; o < 64; o <<= 1) {
            const int32_t v = __shfl_up(incl, o);
            if (lane >= o) incl += v;
        }
        __syncthreads();
        if (lane == 63) s_wave[wave] = incl;
        __syncthreads();
        int32_t before = base + incl - sum;
        for (int w = 0; w < 16; ++w) {
            if (w < wave) before += s_wave[w];
            base += s_wave[w];
        }
#pragma unroll
        for (int u = 0; u < EACH; ++u) {
            if (i + u < n) count[i + u] = before;
            before += c[u];
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        max_id = max(max_id, (uint32_t)__shfl_xor((int)max_id, o));
        max_bucket = max(max_bucket, (uint32_t)__shfl_xor((int)max_bucket, o));
    }
    __syncthreads();
    if (lane == 0) { atomicMax(&s_max[0], max_id); atomicMax(&s_max[1], max_bucket); }
    __syncthreads();
    if (t > 0) return;
    count[n] = base;
    *total_out = base;
    if (most) { out->max_id = s_max[0]; out->max_bucket = s_max[1]; }
}

/* a tile's selected records to their places, QUADS lanes copying each */
template <int QUADS>
__global__ void __launch_bounds__(256) k_gather(const quad* __restrict__ in, const uint4* __restrict__ sel,
                                                const int32_t* __restrict__ offset, quad* __restrict__ out)
{
    const int64_t tile = (int64_t)blockIdx.x * (256 * OA_SELECT_ROUNDS), o = offset[blockIdx.x];
    const int32_t c = (int32_t)(offset[blockIdx.x + 1] - o);
    for (int32_t i = threadIdx.x; i < c * QUADS; i += 256)
        out[o * QUADS + i] = in[(int64_t)sel[tile + i / QUADS].x * QUADS + i % QUADS];
}

/* a tile's keys, and the places in sel that they belong to, to their places */
template <class Key>
__global__ void __launch_bounds__(256) k_keys(const uint4* __restrict__ sel, const int32_t* __restrict__ offset, float tw,
                                              int bucket_bits, Key* __restrict__ keys, uint32_t* __restrict__ order)
{
    const int64_t tile = (int64_t)blockIdx.x * (256 * OA_SELECT_ROUNDS), o = offset[blockIdx.x];
    const int32_t c = (int32_t)(offset[blockIdx.x + 1] - o);
    for (int32_t i = threadIdx.x; i < c; i += 256) {
        const uint4 v = sel[tile + i];
        keys[o + i] = (Key)(v.z & 0xffffu) << bucket_bits | (Key)bucket_of(v.y, tw);
        order[o + i] = (uint32_t)(tile + i);
    }
}

/* the sorted keys of a tile at which a run starts, one bit a round */
template <class Key>
__device__ uint32_t run_heads(const Key* keys, int64_t n, int64_t first)
{
    uint32_t heads = 0;
#pragma unroll
    for (int k = 0; k < OA_REDUCE_ROUNDS; ++k) {
        const int64_t i = first + k * 256;
        const bool head = i < n && (i == 0 || keys[i] != keys[i - 1]);
        heads |= (uint32_t)head << k;
    }
    return heads;
}

template <class Key>
__global__ void __launch_bounds__(256) k_count_runs(const Key* __restrict__ keys, int64_t n, int32_t* count)
{
    __shared__ int32_t s_n[4];
    int32_t c = __popc(run_heads(keys, n, (int64_t)blockIdx.x * (256 * OA_REDUCE_ROUNDS) + threadIdx.x));
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
    if ((threadIdx.x & 63) == 0) s_n[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) count[blockIdx.x] = s_n[0] + s_n[1] + s_n[2] + s_n[3];
}

/* the merged record of a run so far. index: input index of the kept record (photon) or the
   first (lite) */
struct Folded {
    uint32_t index;
    float time;
    uint32_t hitcount, flagmask;
};

/*
 * The record types' reduce_op, a before b in sorted order:
 *   sphoton      r = (fminf(a.time, b.time) == a.time) ? a : b; flagmasks OR-ed, 16-bit
 *                hitcounts added
 *   sphotonlite  r = a; r.time = fminf(a.time, b.time); likewise
 * Associative, times that are not numbers included (such an a gives way to any b, such a b to
 * any other a), so a run may be folded in pieces kept in order.
 */
template <bool LITE>
__device__ inline Folded fold(const Folded& a, const Folded& b)
{
    const float m = fminf(a.time, b.time);
    const bool first = LITE || m == a.time;
    return Folded{ first ? a.index : b.index, LITE ? m : first ? a.time : b.time, (a.hitcount + b.hitcount) & 0xffffu,
                   a.flagmask | b.flagmask };
}

/* sorted positions [o, o + len), len > 0, left to right, four records' words in flight a step */
template <bool LITE>
__device__ Folded fold_range(const uint4* sel, const uint32_t* order, int64_t o, int64_t len)
{
    const auto one = [](const uint4& v) { return Folded{ v.x, __uint_as_float(v.y), v.z >> 16, v.w }; };
    Folded r = one(sel[order[o]]);
    for (int64_t j = 1; j < len; j += 4) {
        uint32_t w[4];
        uint4 b[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) w[u] = order[j + u < len ? o + j + u : o];
#pragma unroll
        for (int u = 0; u < 4; ++u) b[u] = sel[w[u]];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (j + u < len) r = fold<LITE>(r, one(b[u]));
    }
    return r;
}

/* the same by a wave: a piece to a lane, then the pieces pairwise */
template <bool LITE>
__device__ Folded fold_range_wave(const uint4* sel, const uint32_t* order, int64_t o, int64_t len, int lane)
{
    const int64_t each = (len + 63) / 64, b = lane * each < len ? lane * each : len;
    const int64_t mine = len - b < each ? len - b : each;
    Folded r{ 0u, 0.f, 0u, 0u };
    if (mine > 0) r = fold_range<LITE>(sel, order, o + b, mine);
    const int pieces = (int)((len + each - 1) / each);
    for (int step = 1; step < 64; step <<= 1) {
        const Folded q{ (uint32_t)__shfl_down((int)r.index, step), __shfl_down(r.time, step),
                        (uint32_t)__shfl_down((int)r.hitcount, step), (uint32_t)__shfl_down((int)r.flagmask, step) };
        if ((lane & (2 * step - 1)) == 0 && lane + step < pieces) r = fold<LITE>(r, q);
    }
    return r;                                        /* lane 0's */
}

/* end of the run of keys[o], which reaches `from` at least */
template <class Key>
__device__ int64_t run_end(const Key* keys, int64_t n, int64_t o, int64_t from)
{
    const Key key = keys[o];
    int64_t lo = from, hi = n;                       /* first position in [lo, hi] with another key */
    for (int64_t step = 1; lo < hi; step *= 2) {     /* most runs end close by */
        const int64_t p = lo + step - 1;
        if (p >= hi) break;
        if (keys[p] != key) { hi = p; break; }
        lo = p + 1;
    }
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (keys[mid] == key) lo = mid + 1; else hi = mid;
    }
    return lo;
}

/* runs of more records than this are folded by a wave: the slowest of 64 lanes sets a wave's
   pace (3M photons' lite records have runs of several hundred: k_reduce 213 us, and 25 so) */
#define OA_LONG_RUN 32

template <bool LITE, class Key>
__global__ void __launch_bounds__(256) k_reduce(const uint32_t* __restrict__ in, const uint4* __restrict__ sel,
                                                const Key* __restrict__ keys, const uint32_t* __restrict__ order, int64_t n,
                                                const int32_t* __restrict__ offset, uint32_t* __restrict__ out,
                                                int64_t out_cap)
{
    constexpr int ROUNDS = OA_REDUCE_ROUNDS;
    __shared__ unsigned long long s_mask[4 * ROUNDS];
    __shared__ int32_t s_pre[4 * ROUNDS + 1];
    __shared__ uint16_t s_head[256 * ROUNDS + 1];
    __shared__ uint16_t s_long[256 * ROUNDS / OA_LONG_RUN + 1];
    __shared__ int32_t s_n_long;
    __shared__ int64_t s_end;                        /* of the last run, which may go on past the tile */
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t first = (int64_t)blockIdx.x * (256 * ROUNDS), base = offset[blockIdx.x];
    const int32_t here = (int32_t)(n - first < 256 * ROUNDS ? n - first : 256 * ROUNDS);
    const uint32_t heads = run_heads(keys, n, first + t);
    const int32_t total = tile_ranks<ROUNDS>(heads, s_mask, s_pre);
#pragma unroll
    for (int k = 0; k < ROUNDS; ++k)
        if (heads >> k & 1u) s_head[rank_in_tile(k, s_mask, s_pre)] = (uint16_t)(k * 256 + t);
    if (t == 0) { s_head[total] = (uint16_t)here; s_n_long = 0; }
    __syncthreads();
    if (t == 0 && total > 0) s_end = run_end(keys, n, first + s_head[total - 1], first + here);
    __syncthreads();
    const int64_t room = out_cap - base;
    const int32_t fit = (int32_t)(room < total ? (room > 0 ? room : 0) : total);
    const auto run_len = [&](int32_t h) { return (h == total - 1 ? s_end - first : (int64_t)s_head[h + 1]) - s_head[h]; };
    /* the record that h0 + 64 wave + lane's run is merged into; photon records are copied by
       four lanes each */
    const auto write = [&](int32_t h, bool have, const Folded& r) {
        if (LITE) {
            if (have) {
                const quad a = reinterpret_cast<const quad*>(in)[r.index];
                reinterpret_cast<quad*>(out)[base + h] = quad{ r.hitcount << 16 | (a.x & 0xffffu), __float_as_uint(r.time),
                                                               a.z, r.flagmask };
            }
            return;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int src = 16 * q + (lane >> 2), part = lane & 3;
            const bool on = __shfl((int)have, src) != 0;
            const uint32_t best = (uint32_t)__shfl((int)r.index, src), hc = (uint32_t)__shfl((int)r.hitcount, src),
                           fm = (uint32_t)__shfl((int)r.flagmask, src);
            const int32_t hq = __shfl(h, src);
            if (!on) continue;
            quad w = reinterpret_cast<const quad*>(in)[(int64_t)best * 4 + part];
            if (part == 1) w.w = (w.w & 0x0000ffffu) | (hc << 16);
            if (part == 3) w.w = fm;
            reinterpret_cast<quad*>(out)[(base + hq) * 4 + part] = w;
        }
    };
    for (int32_t h0 = 0; h0 < fit; h0 += 256) {
        const int32_t h = h0 + t;
        const int64_t len = h < fit ? run_len(h) : 0;
        const bool own = len > 0 && len <= OA_LONG_RUN;
        Folded r{ 0u, 0.f, 0u, 0u };
        if (own) r = fold_range<LITE>(sel, order, first + s_head[h], len);
        if (len > OA_LONG_RUN) s_long[atomicAdd(&s_n_long, 1)] = (uint16_t)h;
        write(h, own, r);
    }
    __syncthreads();
    for (int32_t k = wave; k < s_n_long; k += 4) {
        const int32_t h = s_long[k];
        const Folded r = fold_range_wave<LITE>(sel, order, first + s_head[h], run_len(h), lane);
        write(h, lane == 0, r);
    }
}

inline int bits_of(uint32_t v) { return v ? 32 - __builtin_clz(v) : 0; }

/* the keys are made where an odd or even number of sort passes ends them in keys2, order2 */
template <class Key>
hipError_t sort_t(const uint4* sel, int64_t n_tiles, const int32_t* offset, int64_t n, float tw, int bucket_bits, int bits,
                  Key* keys, Key* keys2, uint32_t* order, uint32_t* order2, uint32_t* tmp, hipStream_t s)
{
    if (oa_radix::passes(bits) % 2 == 0) { std::swap(keys, keys2); std::swap(order, order2); }
    hipLaunchKernelGGL(k_keys<Key>, dim3((unsigned)n_tiles), dim3(256), 0, s, sel, offset, tw, bucket_bits, keys, order);
    return oa_radix::sort(keys, keys2, order, order2, n, bits, tmp, s);
}

template <class Key>
void reduce_t(int record, const void* d_in, const uint4* sel, int64_t n, int64_t n_tiles, const Key* keys,
              const uint32_t* order, int32_t* offset, void* d_out, int64_t out_cap, hipStream_t s)
{
    const dim3 grid((unsigned)n_tiles), block(256);
    if (record == OA_MERGE_PHOTON)
        hipLaunchKernelGGL((k_reduce<false, Key>), grid, block, 0, s, (const uint32_t*)d_in, sel, keys, order, n, offset,
                           (uint32_t*)d_out, out_cap);
    else
        hipLaunchKernelGGL((k_reduce<true, Key>), grid, block, 0, s, (const uint32_t*)d_in, sel, keys, order, n, offset,
                           (uint32_t*)d_out, out_cap);
}

} // namespace

namespace oa_merge {

static int64_t tiles(int64_t n, int rounds) { return (n + 256 * rounds - 1) / (256 * rounds); }
/* counts of the selection's tiles and of the runs', each with a total behind it */
size_t count_words(int64_t n) { return (size_t)(tiles(n, OA_SELECT_ROUNDS) + tiles(n, OA_REDUCE_ROUNDS) + 2); }
size_t most_words(int64_t n) { return (size_t)tiles(n, OA_SELECT_ROUNDS); }

hipError_t select(int record, const void* d_in, int64_t n, uint32_t mask, float tw, int32_t* count, uint2* most, uint4* sel,
                  Result* out, hipStream_t s)
{
    const int64_t nt = tiles(n, OA_SELECT_ROUNDS);
    if (record == OA_MERGE_PHOTON)
        hipLaunchKernelGGL(k_select<PhotonAcc>, dim3((unsigned)nt), dim3(256), 0, s, (const uint32_t*)d_in, n, mask, tw,
                           count, most, sel);
    else
        hipLaunchKernelGGL(k_select<LiteAcc>, dim3((unsigned)nt), dim3(256), 0, s, (const uint32_t*)d_in, n, mask, tw,
                           count, most, sel);
    hipLaunchKernelGGL(k_tile_offsets, dim3(1), dim3(1024), 0, s, count, most, nt, &out->n_sel, out);
    return hipGetLastError();
}

hipError_t gather_selected(int record, const void* d_in, int64_t n, const int32_t* count, const uint4* sel, void* d_out,
                           hipStream_t s)
{
    const dim3 grid((unsigned)tiles(n, OA_SELECT_ROUNDS)), block(256);
    if (record == OA_MERGE_PHOTON)
        hipLaunchKernelGGL(k_gather<4>, grid, block, 0, s, (const quad*)d_in, sel, count, (quad*)d_out);
    else
        hipLaunchKernelGGL(k_gather<1>, grid, block, 0, s, (const quad*)d_in, sel, count, (quad*)d_out);
    return hipGetLastError();
}

int key_bits(uint32_t max_id, uint32_t max_bucket)
{
    const int b = bits_of(max_id) + bits_of(max_bucket);
    return b > 0 ? b : 1;
}

size_t sort_words(int64_t n_sel, int bits) { return oa_radix::words(n_sel, bits); }

hipError_t sort_runs(int64_t n, const int32_t* count, const uint4* sel, int64_t n_sel, float tw, uint32_t max_bucket,
                     int bits, void* keys, void* keys2, uint32_t* order, uint32_t* order2, uint32_t* tmp, hipStream_t s)
{
    const int bb = bits_of(max_bucket);
    const int64_t nt = tiles(n, OA_SELECT_ROUNDS);
    return bits <= 32
        ? sort_t(sel, nt, count, n_sel, tw, bb, bits, (uint32_t*)keys, (uint32_t*)keys2, order, order2, tmp, s)
        : sort_t(sel, nt, count, n_sel, tw, bb, bits, (uint64_t*)keys, (uint64_t*)keys2, order, order2, tmp, s);
}

hipError_t count_runs(int64_t n, int32_t* count, int64_t n_sel, int bits, const void* keys2, Result* out, hipStream_t s)
{
    int32_t* runs = count + tiles(n, OA_SELECT_ROUNDS) + 1;
    const int64_t nt = tiles(n_sel, OA_REDUCE_ROUNDS);
    if (bits <= 32)
        hipLaunchKernelGGL(k_count_runs<uint32_t>, dim3((unsigned)nt), dim3(256), 0, s, (const uint32_t*)keys2, n_sel, runs);
    else
        hipLaunchKernelGGL(k_count_runs<uint64_t>, dim3((unsigned)nt), dim3(256), 0, s, (const uint64_t*)keys2, n_sel, runs);
    hipLaunchKernelGGL(k_tile_offsets, dim3(1), dim3(1024), 0, s, runs, (const uint2*)nullptr, nt, &out->n_runs, out);
    return hipGetLastError();
}

hipError_t reduce_runs(int record, const void* d_in, int64_t n, int32_t* count, const uint4* sel, int64_t n_sel, int bits,
                       const void* keys2, const uint32_t* order2, void* d_out, int64_t out_cap, hipStream_t s)
{
    int32_t* runs = count + tiles(n, OA_SELECT_ROUNDS) + 1;
    const int64_t nt = tiles(n_sel, OA_REDUCE_ROUNDS);
    if (bits <= 32) reduce_t(record, d_in, sel, n_sel, nt, (const uint32_t*)keys2, order2, runs, d_out, out_cap, s);
    else reduce_t(record, d_in, sel, n_sel, nt, (const uint64_t*)keys2, order2, runs, d_out, out_cap, s);
    return hipGetLastError();
}

} // namespace oa_merge
