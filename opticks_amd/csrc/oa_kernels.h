/* oa_kernels.h : host-side launchers of the gfx950 kernels (oa_kernels.hip). */
#pragma once
#include <hip/hip_runtime.h>
#include "oa_layout.h"

namespace oa_launch {
/* genstep of each photon (seed) and, for n_event > 1, event of each genstep */
hipError_t seed_map(const int64_t* d_prefix, int64_t n_gs, int64_t n_photon, uint32_t* d_seed,
                    const int64_t* d_ev_gs_begin, int32_t n_event, int32_t* d_gs_event, hipStream_t s);
/* exclusive prefix of the gensteps' photon counts into d_prefix[0..n_gs], which holds
   gs_prefix_words(n_gs) words (block sums behind it) */
int64_t gs_prefix_words(int64_t n_gs);
/* out (may be null): setup_begins is set where the prefix takes several blocks */
hipError_t gs_prefix(const float* d_gs, int64_t n_gs, int64_t* d_prefix, hipStream_t s, LaunchResult* out = nullptr);
/* start of a single-event launch (k_setup): seeds of up to cap photons, its cleared words (words:
   clear_words(cap)), event bounds ev (4) and ev_id (1), the launch's photon count and wave_width
   n_dev (2) */
struct SetupArgs {
    const float* gs; int64_t n_gs, n_arg, cap;
    int64_t* prefix; uint32_t* seed;
    unsigned long long* words;
    int64_t* ev; int32_t* ev_id; int32_t event_id;
    int64_t* n_dev; LaunchResult* out;  /* out: result_bytes(cap) */
    int64_t n_wave;                     /* waves of the propagation grid */
};
hipError_t setup(const SetupArgs& a, hipStream_t s);
int setup_blocks(int64_t cap);
/* Cleared words of a launch of up to n photons: the propagation's photon counter, the compaction's
   ticket and the state of its tiles (256 bitmask words each), then the hit bitmask. The counters
   are in front, so that an event of fewer photons clears and reads what it needs alone. */
#define OA_WORDS_TICKET 1
#define OA_WORDS_STATE 2
inline int64_t compact_tiles(int64_t n_photon) { return ((n_photon + 63) / 64 + 255) / 256; }
inline size_t result_bytes(int64_t n_photon) { return sizeof(LaunchResult) + 8 * (size_t)(OA_SETUP_BLOCKS + compact_tiles(n_photon)); }
inline int64_t bitmask_offset(int64_t n_photon) { return OA_WORDS_STATE + compact_tiles(n_photon); }
inline int64_t clear_words(int64_t n_photon) { return bitmask_offset(n_photon) + (n_photon + 63) / 64; }
hipError_t simulate(const SimParams& P, int kernel, int block, int grid, hipStream_t s);
/* blocks of the persistent kernel that are resident on a CU, of the instantiation that a launch runs */
int wave_blocks_per_cu(int block, int rng_kind, int stack_depth, bool lite, bool ext, bool tape);
unsigned sim_lds(int block, int rng_kind, int stack_depth);   /* LDS bytes of a propagation block */
hipError_t prefix_check(const int64_t* a, const int64_t* b, int64_t n, unsigned long long* flag, hipStream_t s);
hipError_t zero_u64(unsigned long long* p, int64_t n, hipStream_t s);
/* the cleared words of a launch of n photons on n_wave waves, its counter set behind the photons dealt first */
hipError_t clear_launch(unsigned long long* words, int64_t n_photon, int64_t n_wave, hipStream_t s);
/* stable compaction of the hits among n_photon photons, or *n_dev of them where it is given;
   d_words: the launch's cleared words; d_tile_base: compact_tiles + 1 words; out (may be null): the
   hit count and the clock */
hipError_t compact_hits(unsigned long long* d_words, int64_t n_photon, const int64_t* n_dev, int32_t* d_word_prefix,
                        int64_t* d_tile_base, const float4* d_photon, float4* d_hit, int64_t hit_cap, LaunchResult* out,
                        hipStream_t s);
hipError_t event_hit_offsets(const unsigned long long* d_bitmask, const int32_t* d_word_prefix,
                             const int64_t* d_block_total, const int64_t* d_ev_ph_begin, int32_t n_event,
                             int64_t n_words, int64_t* d_hit_offsets, hipStream_t s);
/* before a simtrace: the gensteps' rays, and a sample of where they end, into out */
hipError_t ray_sample(const SimParams& P, LaunchResult* out, hipStream_t s);
/* sample: ray_sample's, complete */
hipError_t simtrace(const SimParams& P, float4* out, const LaunchResult* sample, hipStream_t s);
hipError_t trace(const SimParams& P, const float4* rays, int64_t n, float4* out, hipStream_t s);
hipError_t refit(BvhNode* d_tlas, int64_t n_tlas, uint32_t max_depth, const uint32_t* d_tlas_items,
                 const float* d_inst_box, hipStream_t s);
/* device buffers of the adjoint: parameter map (mat_block, sample_bin), hits with
   optional per-event hit offsets (batched events: the hit count is read on the
   device and clipped to hit_cap), score rows S (n_max rows of n_param), sort
   keys/values and temporary storage, detector runs seg (n_det + 1), and the
   per-detector sums G with their Kahan compensation C (n_det x n_param) */
struct AdjBufs {
    const int32_t* mat_block; int32_t n_mat;
    const int32_t* sample_bin; int32_t n_bin; int32_t n_param;
    const float4* hit; const int64_t* hit_off; int32_t n_ev; int64_t hit_cap;
    uint32_t n_det;
    float* S;
    uint32_t *key, *val, *key2, *val2;
    uint32_t* tmp;
    int64_t* seg;
    float *G, *C;
};
/* adjoint of hits [begin, begin+n) (n = n_max, or the device count): score rows,
   then per-detector Kahan sums in photon order (first: start them, else continue
   from the previous chunk). Without P.tape every hit is replayed into dense rows;
   with it, hits are scored from their tape records inside the per-detector
   reduction and only photons the tape could not hold are replayed. `mid` (may be
   null) is recorded before the reduction. */
hipError_t adjoint_chunk(const SimParams& P, const AdjBufs& a, int64_t begin, int64_t n_max, int first, int grid,
                         hipEvent_t mid, hipStream_t s);
/* hits per round of the fused tape reduction for n_param parameters (0: more
   parameters than it handles, OA_TAPE_NJ_MAX x 256) */
#define OA_TAPE_NJ_MAX 4
int tape_reduce_rows(int32_t n_param);
int adjoint_blocks_per_cu(int rng_kind, int stack_depth);
/* no-allocation entry point: the device address of the per-GPU scratch array
   (call with `device` current), and the per-launch event setup kernel */
hipError_t noalloc_scratch(int device, void** ptr);
hipError_t noalloc_setup(int64_t* ev, int32_t* ev_id, int64_t n_gs, int64_t n_photon, int32_t event_id, hipStream_t s);
/* hits per detector 1..n_det of n sphoton records into n_det floats */
hipError_t hit_counts(const void* d_hit, int64_t n, uint32_t n_det, float* d_count, hipStream_t s);
size_t adjoint_sort_words(int64_t n_hit, uint32_t n_det);
}
