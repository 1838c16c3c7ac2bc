/*
 * oa_merge.hip : hit selection and merging by (sensor identity, time bucket).
 *
 * Restates SPM::merge_partial_select (sysrap/SPM.cu:135-240) for MI355X:
 *   0. select records with flagmask & mask != 0 (skipped for the "already
 *      selected" mask), stable;
 *   1. time window 0: return the selection in input order;
 *   2-4. key = (identity << 48) | (unsigned)(time / window) as a 64-bit
 *      integer, then a stable sort of the selected records by key; here the
 *      same order is sorted as identity << b | bucket, with b the bits of the
 *      largest bucket selected and identity its low 16 bits (the shift by 48
 *      keeps the same ones);
 *   6. reduce each run of equal keys with the record type's reduce_op.
 * Record types and their functors:
 *   sphoton     64 B  key/reduce/select  sysrap/sphoton.h:292-320
 *   sphotonlite 16 B  key/reduce/select  sysrap/sphotonlite.h:68-97
 *
 * One pass reads the records (k_select) and keeps of each selected one the 16 bytes that the
 * merge needs; bound by the lines it has to fetch, 64 B a photon record for any word of it
 * (640 MB for 10M records, 113 us at 5.7 TB/s). The keys are as wide as the selection's largest
 * identity and bucket need, 20 bits for 2,000 sensors and 400 buckets instead of 48: three
 * radix passes over 8-byte pairs instead of six over 12. k_reduce finds the runs and folds
 * each from the kept words, left to right in sorted order, so ties in time keep the earliest
 * record in input order; only the record that a run keeps is fetched.
 * 10M records, 2M selected, 0.7M merged: 662 us before (flag pass, flagged select, key pass,
 * 48-bit sort, run-length encode, scan, reduce over the records themselves).
 */
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <stdint.h>
#include "oa_merge.h"

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

/* 16 rounds of 256 records or sorted keys make a tile */
#define OA_TILE_ROUNDS 16
#define OA_TILE (256 * OA_TILE_ROUNDS)

/*
 * Items of the tiles before `tile`, by a decoupled look-back over state[tile]: 0, then
 * count | 1 << 62, then (items up to its end) | 2 << 62 (as the hit compaction does it). Run by
 * one wave; the tiles are handed out by ticket, so those before it are running or done.
 */
__device__ int64_t look_back(unsigned long long* state, int64_t tile, int64_t total, int lane)
{
    const unsigned long long kCount = 1ull << 62, kDone = 2ull << 62, kValue = kCount - 1ull;
    int64_t base = 0;
    if (tile > 0) {
        if (lane == 0)
            __hip_atomic_store(&state[tile], kCount | (unsigned long long)total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int64_t k = tile - 1;; k -= 64) {
            const int64_t mine = k - lane;
            unsigned long long v = kDone;
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
    if (lane == 0)
        __hip_atomic_store(&state[tile], kDone | (unsigned long long)(base + total), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    return base;
}

/* The tile's 64 ballot words (4 waves x 16 rounds, in item order) to the items before each word
   (s_pre) and before the tile (returned to every thread); total: the tile's items */
__device__ int64_t tile_prefix(const unsigned long long* s_mask, int32_t* s_pre, int64_t* s_base, unsigned long long* state,
                               int64_t tile, int32_t& total)
{
    __syncthreads();
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        const int32_t c = __popcll(s_mask[lane]);
        int32_t incl = c;
        for (int o = 1; o < 64; o <<= 1) {
            const int32_t v = __shfl_up(incl, o);
            if (lane >= o) incl += v;
        }
        s_pre[lane] = incl - c;
        const int32_t all = __shfl(incl, 63);
        if (lane == 63) s_pre[64] = all;
        const int64_t base = look_back(state, tile, all, lane);
        if (lane == 0) *s_base = base;
    }
    __syncthreads();
    total = s_pre[64];
    return *s_base;
}

template <class Acc>
__global__ void __launch_bounds__(256) k_select(const uint32_t* __restrict__ in, int64_t n, uint32_t mask, float tw,
                                                int64_t n_tiles, unsigned long long* state, uint4* __restrict__ sel,
                                                oa_merge::Result* out)
{
    __shared__ unsigned long long s_mask[64];
    __shared__ int32_t s_pre[65];
    __shared__ int64_t s_tile, s_base;
    __shared__ uint32_t s_max[2];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t == 0) { s_tile = (int64_t)atomicAdd(&state[n_tiles], 1ull); s_max[0] = s_max[1] = 0u; }
    __syncthreads();
    const int64_t tile = s_tile;
    if (tile >= n_tiles) return;
    uint4 v[OA_TILE_ROUNDS];
    uint32_t taken = 0, max_id = 0, max_bucket = 0;
#pragma unroll
    for (int k = 0; k < OA_TILE_ROUNDS; ++k) {
        const int64_t i = tile * OA_TILE + k * 256 + t;
        const uint32_t* r = in + i * Acc::WORDS;
        const uint32_t fm = i < n ? Acc::flagmask(r) : 0u;
        const bool take = i < n && (mask == OA_MERGE_ALREADY_SELECTED || (fm & mask) != 0u);
        if (take) {
            v[k] = make_uint4((uint32_t)i, Acc::time(r), Acc::identity(r) | (Acc::hitcount(r) << 16), fm);
            taken |= 1u << k;
        }
        const unsigned long long m = __ballot(take);
        if (lane == 0) s_mask[4 * k + wave] = m;
    }
#pragma unroll
    for (int k = 0; k < OA_TILE_ROUNDS; ++k) {
        if (!(taken >> k & 1u)) continue;
        max_id = max(max_id, v[k].z & 0xffffu);
        max_bucket = max(max_bucket, bucket_of(v[k].y, tw));
    }
    for (int o = 32; o > 0; o >>= 1) {
        max_id = max(max_id, (uint32_t)__shfl_xor((int)max_id, o));
        max_bucket = max(max_bucket, (uint32_t)__shfl_xor((int)max_bucket, o));
    }
    if (lane == 0) { atomicMax(&s_max[0], max_id); atomicMax(&s_max[1], max_bucket); }
    int32_t total;
    const int64_t base = tile_prefix(s_mask, s_pre, &s_base, state, tile, total);
    /* the running maxima: both in one word each, touched only by tiles that raise them */
    unsigned long long* maxima = state + n_tiles + 1;
    if (t < 2 && (unsigned long long)s_max[t] > __hip_atomic_load(&maxima[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(&maxima[t], (unsigned long long)s_max[t]);
#pragma unroll
    for (int k = 0; k < OA_TILE_ROUNDS; ++k) {
        if (!(taken >> k & 1u)) continue;
        const unsigned long long m = s_mask[4 * k + wave];
        sel[base + s_pre[4 * k + wave] + __popcll(m & ((1ull << lane) - 1ull))] = v[k];
    }
    if (tile == n_tiles - 1 && t == 0) out->n_sel = base + total;
}

/* the maxima are complete when k_select is */
__global__ void k_maxima(const unsigned long long* maxima, oa_merge::Result* out)
{
    out->max_id = (uint32_t)maxima[0];
    out->max_bucket = (uint32_t)maxima[1];
}

__global__ void k_clear(unsigned long long* p, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

/* QUADS lanes copy a record */
template <int QUADS>
__global__ void __launch_bounds__(256) k_gather(const quad* __restrict__ in, const uint4* __restrict__ sel, int64_t n,
                                                quad* __restrict__ out)
{
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n * QUADS) return;
    out[t] = in[(int64_t)sel[t / QUADS].x * QUADS + t % QUADS];
}

template <class Key>
__global__ void __launch_bounds__(256) k_keys(const uint4* __restrict__ sel, int64_t n, float tw, int bucket_bits,
                                              Key* __restrict__ keys, uint32_t* __restrict__ order)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint4 v = sel[i];
    keys[i] = (Key)(v.z & 0xffffu) << bucket_bits | (Key)bucket_of(v.y, tw);
    order[i] = (uint32_t)i;
}

/*
 * The merged record of the run of equal keys that starts at sorted position o, folded left to
 * right with the record type's reduce_op, four records' words in flight a step:
 *   sphoton      r = (fminf(a.time, b.time) == a.time) ? a : b; flagmasks OR-ed, 16-bit
 *                hitcounts added
 *   sphotonlite  r = a; r.time = fminf(a.time, b.time); likewise (first: a's input index)
 * x: input index of the kept record, y: time, z: hitcount, w: flagmask
 */
template <bool LITE, class Key>
__device__ uint4 fold_run(const uint4* sel, const Key* keys, const uint32_t* order, int64_t n, int64_t o)
{
    const Key key = keys[o];
    const uint4 a = sel[order[o]];
    uint32_t best = a.x, fm = a.w, hc = a.z >> 16;
    float bt = __uint_as_float(a.y);
    const auto fold = [&](const uint4& b) {
        const float t = __uint_as_float(b.y);
        if (LITE) bt = fminf(bt, t);
        else if (!(fminf(bt, t) == bt)) { best = b.x; bt = t; }
        fm |= b.w;
        hc = (hc + (b.z >> 16)) & 0xffffu;
    };
    int64_t j = o + 1;
    while (j < n && keys[j] == key) {
        if (j + 4 <= n && keys[j + 3] == key) {
            uint4 b[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) b[u] = sel[order[j + u]];
#pragma unroll
            for (int u = 0; u < 4; ++u) fold(b[u]);
            j += 4;
        } else {
            fold(sel[order[j]]);
            j += 1;
        }
    }
    return make_uint4(best, __float_as_uint(bt), hc, fm);
}

template <bool LITE, class Key>
__global__ void __launch_bounds__(256) k_reduce(const uint32_t* __restrict__ in, const uint4* __restrict__ sel,
                                                const Key* __restrict__ keys, const uint32_t* __restrict__ order, int64_t n,
                                                int64_t n_tiles, unsigned long long* state, uint32_t* __restrict__ out,
                                                int64_t out_cap, oa_merge::Result* res)
{
    __shared__ unsigned long long s_mask[64];
    __shared__ int32_t s_pre[65];
    __shared__ int64_t s_tile, s_base;
    __shared__ uint16_t s_head[OA_TILE];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t == 0) s_tile = (int64_t)atomicAdd(&state[n_tiles], 1ull);
    __syncthreads();
    const int64_t tile = s_tile;
    if (tile >= n_tiles) return;
    const int64_t first = tile * OA_TILE;
    uint32_t heads = 0;
#pragma unroll
    for (int k = 0; k < OA_TILE_ROUNDS; ++k) {
        const int64_t i = first + k * 256 + t;
        const bool head = i < n && (i == 0 || keys[i] != keys[i - 1]);
        if (head) heads |= 1u << k;
        const unsigned long long m = __ballot(head);
        if (lane == 0) s_mask[4 * k + wave] = m;
    }
    int32_t total;
    const int64_t base = tile_prefix(s_mask, s_pre, &s_base, state, tile, total);
#pragma unroll
    for (int k = 0; k < OA_TILE_ROUNDS; ++k) {
        if (!(heads >> k & 1u)) continue;
        const unsigned long long m = s_mask[4 * k + wave];
        s_head[s_pre[4 * k + wave] + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)(k * 256 + t);
    }
    __syncthreads();
    const int64_t room = out_cap - base;
    const int32_t fit = (int32_t)(room < total ? (room > 0 ? room : 0) : total);
    /* a run to a lane, then, of photon records, four lanes to a record */
    for (int32_t h0 = 0; h0 < fit; h0 += 256) {
        const int32_t h = h0 + t;
        uint4 r = make_uint4(0u, 0u, 0u, 0u);
        if (h < fit) r = fold_run<LITE>(sel, keys, order, n, first + s_head[h]);
        if (LITE) {
            if (h < fit) {
                const quad a = reinterpret_cast<const quad*>(in)[r.x];
                reinterpret_cast<quad*>(out)[base + h] = quad{ r.z << 16 | (a.x & 0xffffu), r.y, a.z, r.w };
            }
            continue;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int src = 16 * q + (lane >> 2);              /* the wave's record this lane copies a quarter of */
            const uint32_t best = (uint32_t)__shfl((int)r.x, src), hc = (uint32_t)__shfl((int)r.z, src),
                           fm = (uint32_t)__shfl((int)r.w, src);
            const int32_t hq = h0 + 64 * wave + src;
            if (hq >= fit) continue;
            const int part = lane & 3;
            quad w = reinterpret_cast<const quad*>(in)[(int64_t)best * 4 + part];
            if (part == 1) w.w = (w.w & 0x0000ffffu) | (hc << 16);
            if (part == 3) w.w = fm;
            reinterpret_cast<quad*>(out)[(base + hq) * 4 + part] = w;
        }
    }
    if (tile == n_tiles - 1 && t == 0) res->n_runs = base + total;
}

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }
inline int bits_of(uint32_t v) { return v ? 32 - __builtin_clz(v) : 0; }

template <class Key>
size_t sort_bytes_t(int64_t n, int bits)
{
    size_t b = 0;
    (void)hipcub::DeviceRadixSort::SortPairs(nullptr, b, (Key*)nullptr, (Key*)nullptr, (uint32_t*)nullptr,
                                             (uint32_t*)nullptr, (int)n, 0, bits);
    return b;
}

template <class Key>
hipError_t sort_t(const uint4* sel, int64_t n, float tw, int bucket_bits, int bits, Key* keys, Key* keys2, uint32_t* order,
                  uint32_t* order2, void* tmp, size_t tmp_bytes, hipStream_t s)
{
    hipLaunchKernelGGL(k_keys<Key>, dim3(nblk(n, 256)), dim3(256), 0, s, sel, n, tw, bucket_bits, keys, order);
    return hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, keys, keys2, order, order2, (int)n, 0, bits, s);
}

} // namespace

namespace oa_merge {

static int64_t tiles(int64_t n) { return (n + OA_TILE - 1) / OA_TILE; }
int64_t state_words(int64_t n) { return tiles(n) + 3; }

hipError_t select(int record, const void* d_in, int64_t n, uint32_t mask, float tw, unsigned long long* state, uint4* sel,
                  Result* out, hipStream_t s)
{
    const int64_t nt = tiles(n);
    hipLaunchKernelGGL(k_clear, dim3(nblk(nt + 3, 256)), dim3(256), 0, s, state, nt + 3);
    if (record == OA_MERGE_PHOTON)
        hipLaunchKernelGGL(k_select<PhotonAcc>, dim3((unsigned)nt), dim3(256), 0, s, (const uint32_t*)d_in, n, mask, tw, nt,
                           state, sel, out);
    else
        hipLaunchKernelGGL(k_select<LiteAcc>, dim3((unsigned)nt), dim3(256), 0, s, (const uint32_t*)d_in, n, mask, tw, nt,
                           state, sel, out);
    hipLaunchKernelGGL(k_maxima, dim3(1), dim3(1), 0, s, state + nt + 1, out);
    return hipGetLastError();
}

hipError_t gather_selected(int record, const void* d_in, const uint4* sel, int64_t n, void* d_out, hipStream_t s)
{
    if (record == OA_MERGE_PHOTON)
        hipLaunchKernelGGL(k_gather<4>, dim3(nblk(4 * n, 256)), dim3(256), 0, s, (const quad*)d_in, sel, n, (quad*)d_out);
    else
        hipLaunchKernelGGL(k_gather<1>, dim3(nblk(n, 256)), dim3(256), 0, s, (const quad*)d_in, sel, n, (quad*)d_out);
    return hipGetLastError();
}

int key_bits(uint32_t max_id, uint32_t max_bucket)
{
    const int b = bits_of(max_id) + bits_of(max_bucket);
    return b > 0 ? b : 1;
}

size_t sort_bytes(int64_t n, int bits) { return bits <= 32 ? sort_bytes_t<uint32_t>(n, bits) : sort_bytes_t<uint64_t>(n, bits); }

hipError_t sort_runs(const uint4* sel, int64_t n, float tw, uint32_t max_bucket, int bits, void* keys, void* keys2,
                     uint32_t* order, uint32_t* order2, void* tmp, size_t tmp_bytes, hipStream_t s)
{
    const int bb = bits_of(max_bucket);
    return bits <= 32
        ? sort_t(sel, n, tw, bb, bits, (uint32_t*)keys, (uint32_t*)keys2, order, order2, tmp, tmp_bytes, s)
        : sort_t(sel, n, tw, bb, bits, (uint64_t*)keys, (uint64_t*)keys2, order, order2, tmp, tmp_bytes, s);
}

hipError_t reduce_runs(int record, const void* d_in, const uint4* sel, int64_t n, int bits, const void* keys2,
                       const uint32_t* order2, unsigned long long* state, void* d_out, int64_t out_cap, Result* out,
                       hipStream_t s)
{
    const int64_t nt = tiles(n);
    hipLaunchKernelGGL(k_clear, dim3(nblk(nt + 1, 256)), dim3(256), 0, s, state, nt + 1);
#define OA_REDUCE(LITE, Key)                                                                                            \
    hipLaunchKernelGGL((k_reduce<LITE, Key>), dim3((unsigned)nt), dim3(256), 0, s, (const uint32_t*)d_in, sel,          \
                       (const Key*)keys2, order2, n, nt, state, (uint32_t*)d_out, out_cap, out)
    if (record == OA_MERGE_PHOTON) { if (bits <= 32) OA_REDUCE(false, uint32_t); else OA_REDUCE(false, uint64_t); }
    else { if (bits <= 32) OA_REDUCE(true, uint32_t); else OA_REDUCE(true, uint64_t); }
#undef OA_REDUCE
    return hipGetLastError();
}

} // namespace oa_merge
