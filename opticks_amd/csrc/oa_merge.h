/*
 * oa_merge.h : launchers of the hit-merge kernels (oa_merge.hip).
 */
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define OA_MERGE_PHOTON 0             /* sphoton records, 64 B */
#define OA_MERGE_PHOTONLITE 1         /* sphotonlite records, 16 B */
#define OA_MERGE_ALREADY_SELECTED 0xffffffffu

namespace oa_merge {

/* what the passes report, in host-visible memory */
struct Result {
    int64_t n_sel;        /* selected records */
    int64_t n_runs;       /* merged records */
    uint32_t max_id, max_bucket;
};

/* state words of a pass over n records: one a tile, the ticket, and the two running maxima */
int64_t state_words(int64_t n);

/* stable flagmask selection into sel (input index, time, identity | hitcount << 16, flagmask),
   its size and the largest identity and time bucket into out */
hipError_t select(int record, const void* d_in, int64_t n, uint32_t mask, float tw, unsigned long long* state, uint4* sel,
                  Result* out, hipStream_t s);
/* the n selected records, input order, into d_out */
hipError_t gather_selected(int record, const void* d_in, const uint4* sel, int64_t n, void* d_out, hipStream_t s);

/* significant key bits: (identity, bucket) as one integer */
int key_bits(uint32_t max_id, uint32_t max_bucket);
/* hipCUB temporary storage for n pairs of such keys */
size_t sort_bytes(int64_t n, int bits);
/* stable sort of the n selected by key: keys, keys2 hold n words of 4 bytes (bits <= 32) or 8,
   order, order2 n words; the sorted keys and positions in sel end in keys2, order2 */
hipError_t sort_runs(const uint4* sel, int64_t n, float tw, uint32_t max_bucket, int bits, void* keys, void* keys2,
                     uint32_t* order, uint32_t* order2, void* tmp, size_t tmp_bytes, hipStream_t s);
/* one merged record per run of equal keys, in key order, as many as fit out_cap; their number into out */
hipError_t reduce_runs(int record, const void* d_in, const uint4* sel, int64_t n, int bits, const void* keys2,
                       const uint32_t* order2, unsigned long long* state, void* d_out, int64_t out_cap, Result* out,
                       hipStream_t s);

} // namespace oa_merge
