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

/* for n records: words of `count` (the tiles' counts, then offsets) and of `most` */
size_t count_words(int64_t n);
size_t most_words(int64_t n);

/* stable flagmask selection of the n records into sel (n words: input index, time, identity |
   hitcount << 16, flagmask), tile by tile, the tiles' offsets into count; the selection's size
   and its largest identity and time bucket into out */
hipError_t select(int record, const void* d_in, int64_t n, uint32_t mask, float tw, int32_t* count, uint2* most, uint4* sel,
                  Result* out, hipStream_t s);
/* the selected records, input order, into d_out */
hipError_t gather_selected(int record, const void* d_in, int64_t n, const int32_t* count, const uint4* sel, void* d_out,
                           hipStream_t s);

/* significant key bits: (identity, bucket) as one integer */
int key_bits(uint32_t max_id, uint32_t max_bucket);
/* words of temporary storage for n_sel pairs of such keys */
size_t sort_words(int64_t n_sel, int bits);
/* stable sort of the n_sel selected by key: keys, keys2 hold n_sel words of 4 bytes (bits <= 32)
   or 8, order, order2 n_sel words; the sorted keys and their places in sel end in keys2, order2 */
hipError_t sort_runs(int64_t n, const int32_t* count, const uint4* sel, int64_t n_sel, float tw, uint32_t max_bucket,
                     int bits, void* keys, void* keys2, uint32_t* order, uint32_t* order2, uint32_t* tmp, hipStream_t s);
/* number of runs of equal keys into out, their tiles' offsets behind the selection's in count */
hipError_t count_runs(int64_t n, int32_t* count, int64_t n_sel, int bits, const void* keys2, Result* out, hipStream_t s);
/* one merged record per run, in key order, as many as fit out_cap */
hipError_t reduce_runs(int record, const void* d_in, int64_t n, int32_t* count, const uint4* sel, int64_t n_sel, int bits,
                       const void* keys2, const uint32_t* order2, void* d_out, int64_t out_cap, hipStream_t s);

} // namespace oa_merge
