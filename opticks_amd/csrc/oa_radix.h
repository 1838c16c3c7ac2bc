/*
 * oa_radix.h : stable least-significant-digit radix sort of (key, 32-bit value) pairs, for the
 * sorts by detector and by (sensor, time): some 1e4 to 1e7 pairs whose keys have 8 to 30
 * significant bits.
 *
 * Digits are as even as the passes allow, 8 bits at most: keys of 2,000 sensors take passes of 6
 * and 5 bits, of 2,000 sensors and 400 time buckets three of 7, 7 and 6. A pass is three kernels:
 * digit counts of each tile of 2,048 pairs (k_radix_count), their running sums over the tiles, a
 * digit to a wave (k_radix_scan), and the scatter (k_radix_scatter). Nothing is waited for inside
 * a kernel and nothing has to be cleared, so a sort can be captured into a graph. Small sorts are
 * bound by the launches, large ones by the scattered stores.
 * Merging 10M photon records (2M pairs of 20 bits) / 3M photons' lite records (0.3M): 385 / 1,830 us
 * with hipCUB's sort, 347 / 1,721 us; tiles of 1,024, 2,048 and 4,096 pairs: 345, 347 and 367 us;
 * digits up to 11 bits (two passes): 377 to 382 us.
 */
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace {
namespace oa_radix {

constexpr int ROUNDS = 8, TILE = 256 * ROUNDS, WAVE_TILE = 64 * ROUNDS, MOST_BITS = 8;

inline int64_t tiles(int64_t n) { return (n + TILE - 1) / TILE; }
inline int passes(int bits) { return bits > 0 ? (bits + MOST_BITS - 1) / MOST_BITS : 1; }
inline int digit_bits(int bits) { return bits > 0 ? (bits + passes(bits) - 1) / passes(bits) : 1; }
/* words of temporary storage for up to n pairs */
inline size_t words(int64_t n, int bits) { return ((size_t)tiles(n) + 1) << digit_bits(bits); }

template <class Key> __device__ inline uint32_t digit_of(Key k, int shift, int d) { return (uint32_t)(k >> shift) & ((1u << d) - 1u); }

/* count[digit * n_tiles + tile] */
template <class Key>
__global__ void __launch_bounds__(256) k_radix_count(const Key* __restrict__ keys, int64_t n, int shift, int d,
                                                     uint32_t n_tiles, uint32_t* __restrict__ count)
{
    extern __shared__ uint32_t s_count[];
    const uint32_t bins = 1u << d;
    for (uint32_t b = threadIdx.x; b < bins; b += 256) s_count[b] = 0u;
    __syncthreads();
    const int64_t first = (int64_t)blockIdx.x * TILE + threadIdx.x;
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const int64_t i = first + r * 256;
        if (i < n) atomicAdd(&s_count[digit_of(keys[i], shift, d)], 1u);
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < bins; b += 256) count[(size_t)b * n_tiles + blockIdx.x] = s_count[b];
}

/* a digit's counts to the pairs of the digit before each tile, in place; their total to total[digit] */
__global__ void __launch_bounds__(64) k_radix_scan(uint32_t* __restrict__ count, uint32_t n_tiles, uint32_t* __restrict__ total)
{
    uint32_t* c = count + (size_t)blockIdx.x * n_tiles;
    const uint32_t lane = threadIdx.x;
    uint32_t base = 0u;
    for (uint32_t t0 = 0; t0 < n_tiles; t0 += 64 * 4) {
        uint32_t v[4], sum = 0u;
#pragma unroll
        for (int u = 0; u < 4; ++u) { v[u] = t0 + 4 * lane + u < n_tiles ? c[t0 + 4 * lane + u] : 0u; sum += v[u]; }
        uint32_t incl = sum;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t x = (uint32_t)__shfl_up((int)incl, o);
            if ((int)lane >= o) incl += x;
        }
        uint32_t before = base + incl - sum;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (t0 + 4 * lane + u < n_tiles) c[t0 + 4 * lane + u] = before;
            before += v[u];
        }
        base += (uint32_t)__shfl((int)incl, 63);
    }
    if (lane == 0) total[blockIdx.x] = base;
}

/*
 * A wave ranks 512 neighbouring pairs in order, 64 a round: the lanes of equal digit are found
 * by a ballot per digit bit, and the wave's count of the digit so far is in LDS. Then a pair goes
 * to (pairs of smaller digits) + (of this digit in earlier tiles, earlier waves, earlier lanes).
 */
template <class Key>
__global__ void __launch_bounds__(256) k_radix_scatter(const Key* __restrict__ keys, const uint32_t* __restrict__ vals,
                                                       int64_t n, int shift, int d, uint32_t n_tiles,
                                                       const uint32_t* __restrict__ count, const uint32_t* __restrict__ total,
                                                       Key* __restrict__ keys_out, uint32_t* __restrict__ vals_out)
{
    extern __shared__ uint32_t s_count[];            /* 4 waves x bins */
    __shared__ uint32_t s_sum[4];
    const uint32_t bins = 1u << d;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (uint32_t b = threadIdx.x; b < 4u * bins; b += 256) s_count[b] = 0u;
    __syncthreads();
    volatile uint32_t* mine = s_count + (size_t)wave * bins;
    const int64_t first = (int64_t)blockIdx.x * TILE + wave * WAVE_TILE + lane;
    Key key[ROUNDS];
    uint32_t val[ROUNDS], rank[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const int64_t i = first + r * 64;
        key[r] = i < n ? keys[i] : (Key)0;
        val[r] = i < n ? vals[i] : 0u;
    }
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const uint32_t g = digit_of(key[r], shift, d);
        const bool valid = first + r * 64 < n;
        unsigned long long same = __ballot(valid);
        for (int b = 0; b < d; ++b) {
            const bool bit = (g >> b & 1u) != 0u;
            const unsigned long long m = __ballot(bit);
            same &= bit ? m : ~m;
        }
        const uint32_t below = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
        const uint32_t so_far = mine[g];
        __builtin_amdgcn_wave_barrier();
        if (valid && below == 0u) mine[g] = so_far + (uint32_t)__popcll(same);
        __builtin_amdgcn_wave_barrier();
        rank[r] = so_far + below;
    }
    /* where each digit starts: the totals' exclusive sums, a digit to a thread */
    const uint32_t b = threadIdx.x, mine_total = b < bins ? total[b] : 0u;
    uint32_t incl = mine_total;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t x = (uint32_t)__shfl_up((int)incl, o);
        if (lane >= o) incl += x;
    }
    if (lane == 63) s_sum[wave] = incl;
    __syncthreads();
    if (b < bins) {
        uint32_t at = incl - mine_total + count[(size_t)b * n_tiles + blockIdx.x];
        for (int w = 0; w < wave; ++w) at += s_sum[w];
        for (int w = 0; w < 4; ++w) {
            const uint32_t c = s_count[(size_t)w * bins + b];
            s_count[(size_t)w * bins + b] = at;
            at += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        if (first + r * 64 >= n) continue;
        const uint32_t p = mine[digit_of(key[r], shift, d)] + rank[r];
        keys_out[p] = key[r];
        vals_out[p] = val[r];
    }
}

/*
 * All passes over at most TILE pairs in one block's LDS, with k_radix_scatter's ranks: from (keys,
 * vals) to (keys_out, vals_out), which may be the same. Bound by its latency (3.8 us for 200 pairs of
 * 11-bit keys, 9.3 where one wave ranks all of them), which the launches of three kernels a pass exceed:
 * with them the taped adjoint of 200 hits took 134 us, so 115; the merge of 1,000 hits in windows of
 * 0.01 ns 107 and 65, of 2,000 128 and 79. One tile is the most that fits the kernel's LDS (52 KB).
 */
template <class Key>
__global__ void __launch_bounds__(256) k_radix_small(const Key* keys, const uint32_t* vals, int32_t n, int np, int d,
                                                     Key* keys_out, uint32_t* vals_out)
{
    __shared__ Key s_key[2][TILE];
    __shared__ uint32_t s_val[2][TILE];
    __shared__ uint32_t s_count[4][1 << MOST_BITS];
    __shared__ uint32_t s_sum[4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int rounds = (n + 255) / 256, first = wave * rounds * 64 + lane;     /* a quarter to each wave */
    for (int i = t; i < n; i += 256) { s_key[0][i] = keys[i]; s_val[0][i] = vals[i]; }
    for (int p = 0; p < np; ++p) {
        const Key* ks = s_key[p & 1];
        const uint32_t* vs = s_val[p & 1];
        for (int b = t; b < 4 << MOST_BITS; b += 256) (&s_count[0][0])[b] = 0u;
        __syncthreads();
        volatile uint32_t* mine = s_count[wave];
        const int shift = p * d;
        uint32_t rank[ROUNDS];
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            if (r >= rounds) break;
            const int i = first + r * 64;
            const bool valid = i < n;
            const uint32_t g = valid ? digit_of(ks[i], shift, d) : 0u;
            unsigned long long same = __ballot(valid);
            for (int b = 0; b < d; ++b) {
                const bool bit = (g >> b & 1u) != 0u;
                const unsigned long long m = __ballot(bit);
                same &= bit ? m : ~m;
            }
            const uint32_t below = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
            const uint32_t so_far = mine[g];
            __builtin_amdgcn_wave_barrier();
            if (valid && below == 0u) mine[g] = so_far + (uint32_t)__popcll(same);
            __builtin_amdgcn_wave_barrier();
            rank[r] = so_far + below;
        }
        __syncthreads();
        /* where each digit of each wave starts, a digit to a thread */
        uint32_t c[4], all = 0u;
#pragma unroll
        for (int w = 0; w < 4; ++w) { c[w] = s_count[w][t]; all += c[w]; }
        uint32_t incl = all;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t x = (uint32_t)__shfl_up((int)incl, o);
            if (lane >= o) incl += x;
        }
        if (lane == 63) s_sum[wave] = incl;
        __syncthreads();
        uint32_t at = incl - all;
        for (int w = 0; w < wave; ++w) at += s_sum[w];
#pragma unroll
        for (int w = 0; w < 4; ++w) { s_count[w][t] = at; at += c[w]; }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            const int i = first + r * 64;
            if (r >= rounds || i >= n) break;
            const uint32_t q = mine[digit_of(ks[i], shift, d)] + rank[r];
            s_key[~p & 1][q] = ks[i];
            s_val[~p & 1][q] = vs[i];
        }
        __syncthreads();
    }
    for (int i = t; i < n; i += 256) { keys_out[i] = s_key[np & 1][i]; vals_out[i] = s_val[np & 1][i]; }
}

/* Sorts by the low `bits` bits of the keys, back and forth between (k0, v0) and (k1, v1): it
   starts in (k0, v0) and ends in (k1, v1) after an odd number of passes, in (k0, v0) after an
   even one. n <= 2^31 - 1, tmp: words(n, bits). */
template <class Key>
hipError_t sort(Key* k0, Key* k1, uint32_t* v0, uint32_t* v1, int64_t n, int bits, uint32_t* tmp, hipStream_t s)
{
    const int np = passes(bits), d = digit_bits(bits);
    if (n <= TILE) {
        hipLaunchKernelGGL(k_radix_small<Key>, dim3(1), dim3(256), 0, s, k0, v0, (int32_t)n, np, d, np % 2 ? k1 : k0,
                           np % 2 ? v1 : v0);
        return hipGetLastError();
    }
    const uint32_t nt = (uint32_t)tiles(n), bins = 1u << d;
    uint32_t* total = tmp + ((size_t)nt << d);
    for (int p = 0; p < np; ++p) {
        const int shift = p * d;
        const Key* ki = p % 2 == 0 ? k0 : k1;
        const uint32_t* vi = p % 2 == 0 ? v0 : v1;
        Key* ko = p % 2 == 0 ? k1 : k0;
        uint32_t* vo = p % 2 == 0 ? v1 : v0;
        hipLaunchKernelGGL(k_radix_count<Key>, dim3(nt), dim3(256), bins * 4u, s, ki, n, shift, d, nt, tmp);
        hipLaunchKernelGGL(k_radix_scan, dim3(bins), dim3(64), 0, s, tmp, nt, total);
        hipLaunchKernelGGL(k_radix_scatter<Key>, dim3(nt), dim3(256), bins * 16u, s, ki, vi, n, shift, d, nt, tmp, total, ko,
                           vo);
    }
    return hipGetLastError();
}

} // namespace oa_radix
} // namespace
