/*
 * capi_stub.cpp : host stand-ins for the HIP runtime calls and the kernel launchers that
 * oa_capi.cpp uses, so that its host logic runs on a CPU (tests/test_capi_stub.py). Device
 * memory is host memory, every call completes at once, allocations above a limit fail, and
 * each launch checks that the buffers it is given hold what it would touch instead of
 * touching them.
 */
#include <hip/hip_runtime.h>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include "oa_kernels.h"
#include "oa_merge.h"

namespace {
std::mutex g_m;
std::map<const char*, size_t> g_alloc;         /* live allocations */
size_t g_limit = (size_t)1 << 40, g_largest = 0;
std::atomic<int> g_bad{0}, g_inside{0}, g_overlap{0};
int g_queries = 0, g_adjoint_tape = 0, g_fail_trace = 0, g_resident = 4, g_waves_dealt = 0, g_grid = 0;
int64_t g_n = 0, g_stride = 0;

hipError_t alloc(void** p, size_t n)
{
    std::lock_guard<std::mutex> l(g_m);
    *p = nullptr;
    if (n > g_limit) return hipErrorOutOfMemory;
    if (n > g_largest) g_largest = n;
    *p = std::calloc(1, n + 64);
    g_alloc[(const char*)*p] = n;
    return hipSuccess;
}
hipError_t release(void* p)
{
    std::lock_guard<std::mutex> l(g_m);
    auto it = g_alloc.find((const char*)p);
    if (it != g_alloc.end()) {
        /* what reads it later does not go unnoticed: small blocks are not handed out again */
        const size_t n = it->second;
        std::memset(p, 0xee, n);
        g_alloc.erase(it);
        if (n > 65536) std::free(p);
    } else if (p) {
        g_bad++;
    }
    return hipSuccess;
}
/* whether [p, p + n) lies in one live allocation; otherwise the launch counts as bad */
bool holds(const void* p, size_t n)
{
    std::lock_guard<std::mutex> l(g_m);
    auto it = g_alloc.upper_bound((const char*)p);
    const bool ok = it != g_alloc.begin() && (--it, (const char*)p + n <= it->first + it->second);
    if (!ok) g_bad++;
    return ok;
}
int64_t photons_of(const float* gs, int64_t n)
{
    int64_t t = 0;
    for (int64_t g = 0; g < n; ++g) { uint32_t c; std::memcpy(&c, gs + 24 * g + 3, 4); t += c; }
    return t;
}
}

extern "C" {
void stub_reset() { g_limit = (size_t)1 << 40; g_largest = 0; g_bad = 0; g_overlap = 0; g_fail_trace = 0; }
void stub_limit(size_t n) { g_limit = n; }
void stub_fail_trace(int f) { g_fail_trace = f; }
size_t stub_largest() { return g_largest; }
int stub_bad() { return g_bad; }
int stub_overlap() { return g_overlap; }
/* whether the HIP runtime knows the address: device or pinned memory */
int stub_known(const void* p)
{
    std::lock_guard<std::mutex> l(g_m);
    auto it = g_alloc.upper_bound((const char*)p);
    return it != g_alloc.begin() && (--it, (const char*)p < it->first + it->second);
}
int stub_adjoint_tape() { return g_adjoint_tape; }
int stub_tape_stride() { return (int)g_stride; }
int stub_waves_dealt() { return g_waves_dealt; }
int stub_grid() { return g_grid; }
int stub_queries() { return g_queries; }
int stub_resident() { return g_resident; }
int stub_resident_lite() { return g_resident - 1; }

hipError_t hipMalloc(void** p, size_t n) { return alloc(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return alloc(p, n); }
hipError_t hipFree(void* p) { return release(p); }
hipError_t hipHostFree(void* p) { return release(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) { std::memset(p, 0, sizeof(*p)); p->multiProcessorCount = 2; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    const bool known = stub_known(p);
    std::memset(a, 0, sizeof(*a));
    a->type = known ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return known ? hipSuccess : hipErrorInvalidValue;
}
hipError_t hipStreamCreate(hipStream_t* s) { *s = (hipStream_t)1; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
hipError_t hipGraphCreate(hipGraph_t*, unsigned) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphAddChildGraphNode(hipGraphNode_t*, hipGraph_t, const hipGraphNode_t*, size_t, hipGraph_t) { return hipErrorNotSupported; }
hipError_t hipGraphAddEventRecordNode(hipGraphNode_t*, hipGraph_t, const hipGraphNode_t*, size_t, hipEvent_t) { return hipErrorNotSupported; }
}

namespace oa_launch {
int64_t gs_prefix_words(int64_t n_gs) { return n_gs + 1 + (n_gs + 1023) / 1024; }
hipError_t gs_prefix(const float* gs, int64_t n, int64_t* p, hipStream_t, LaunchResult*)
{
    if (!holds(p, 8 * (size_t)gs_prefix_words(n))) return hipSuccess;
    p[0] = 0;
    for (int64_t g = 0; g < n; ++g) p[g + 1] = p[g] + photons_of(gs + 24 * g, 1);
    return hipSuccess;
}
hipError_t seed_map(const int64_t*, int64_t, int64_t n, uint32_t* seed, const int64_t*, int32_t, int32_t*, hipStream_t)
{
    holds(seed, 4 * (size_t)n);
    return hipSuccess;
}
int setup_blocks(int64_t) { return OA_SETUP_BLOCKS; }
/* the count and the refusals of k_setup */
hipError_t setup(const SetupArgs& a, hipStream_t)
{
    const int64_t total = photons_of(a.gs, a.n_gs);
    int64_t n = a.n_arg < 0 ? total : a.n_arg;
    if (n > total || n > a.cap) n = 0;
    g_n = n;
    g_waves_dealt = (int)a.n_wave;
    holds(a.seed, 4 * (size_t)a.cap);
    holds(a.words, 8 * (size_t)clear_words(a.cap));
    if (holds(a.n_dev, 16)) { a.n_dev[0] = n; a.n_dev[1] = 64; }
    if (!holds(a.out, result_bytes(a.cap))) return hipSuccess;
    a.out->total = total;
    a.out->n_photon = n;
    a.out->n_hit = 0;
    return hipSuccess;
}
hipError_t simulate(const SimParams& P, int, int, int grid, hipStream_t)
{
    g_grid = grid;
    const int64_t n = P.n_dev ? P.n_dev[0] : P.n_photon;
    g_n = n;
    holds(P.hitwords, 8 * (size_t)((n + 63) / 64));
    holds(P.next, 8);
    if (P.tape) {
        g_stride = P.tape_stride;
        holds(P.tape, 12 * (size_t)(P.tape_k - 1) * (size_t)(P.tape_stride ? P.tape_stride : n) + 12 * (size_t)n);
        holds(P.tape_n, (size_t)n);
    }
    if (P.photon)
        for (int64_t i = 0; i < n; ++i) P.photon[4 * i].x = (float)(P.photon_offset + i);
    if (P.seq)
        for (int64_t i = 0; i < n; ++i) P.seq[4 * i] = (uint64_t)i;
    return hipSuccess;
}
/* every second photon is a hit */
hipError_t compact_hits(unsigned long long* words, int64_t cap, const int64_t* n_dev, int32_t* wp, int64_t* tb, const float4* photon, float4* hit, int64_t hit_cap, LaunchResult* out, hipStream_t)
{
    const int64_t n = n_dev ? *n_dev : cap, m = n / 2;
    holds(words, 8 * (size_t)clear_words(cap));
    holds(wp, 4 * (size_t)((cap + 63) / 64));
    if (holds(tb, 8 * (size_t)(compact_tiles(cap) + 1))) tb[compact_tiles(n)] = m;
    for (int64_t i = 0; hit && i < m && i < hit_cap; ++i) std::memcpy(hit + 4 * i, photon + 4 * (2 * i + 1), 64);
    if (out) out->n_hit = m;
    return hipSuccess;
}
int wave_blocks_per_cu(int, int, int, bool lite, bool, bool)
{
    g_queries++;
    return g_resident - (lite ? 1 : 0);
}
unsigned sim_lds(int, int, int) { return 1024; }
hipError_t prefix_check(const int64_t*, const int64_t*, int64_t, unsigned long long*, hipStream_t) { return hipSuccess; }
hipError_t zero_u64(unsigned long long*, int64_t, hipStream_t) { return hipSuccess; }
/* of a batch or no-allocation launch: it takes a while, so that calls sharing the words would overlap */
hipError_t clear_launch(unsigned long long*, int64_t, int64_t n_wave, hipStream_t)
{
    g_waves_dealt = (int)n_wave;
    if (g_inside++) g_overlap++;
    std::this_thread::sleep_for(std::chrono::milliseconds(20));
    g_inside--;
    return hipSuccess;
}
hipError_t event_hit_offsets(const unsigned long long*, const int32_t*, const int64_t*, const int64_t*, int32_t, int64_t, int64_t*, hipStream_t) { return hipSuccess; }
hipError_t ray_sample(const SimParams& P, LaunchResult* out, hipStream_t)
{
    out->total = P.gs_prefix[P.n_gs];
    return hipSuccess;
}
hipError_t simtrace(const SimParams& P, float4* out, const LaunchResult*, hipStream_t)
{
    if (g_fail_trace) return hipErrorLaunchFailure;
    if (holds(out, 64 * (size_t)P.n_photon)) std::memset((void*)out, 0xff, 64 * (size_t)P.n_photon);
    return hipSuccess;
}
hipError_t trace(const SimParams&, const float4*, int64_t, float4*, hipStream_t) { return hipSuccess; }
hipError_t refit(BvhNode*, int64_t, uint32_t, const uint32_t*, const float*, hipStream_t) { return hipSuccess; }
hipError_t adjoint_chunk(const SimParams& P, const AdjBufs&, int64_t, int64_t, int, int, hipEvent_t, hipStream_t)
{
    g_adjoint_tape = P.tape != nullptr;
    return hipSuccess;
}
int tape_reduce_rows(int32_t) { return 32; }
int adjoint_blocks_per_cu(int, int) { return 1; }
hipError_t noalloc_scratch(int, void** p)
{
    static char scratch[OA_NOALLOC_SCRATCH_BYTES];
    *p = scratch;
    std::lock_guard<std::mutex> l(g_m);
    g_alloc[scratch] = sizeof(scratch);
    return hipSuccess;
}
hipError_t noalloc_setup(int64_t*, int32_t*, int64_t, int64_t, int32_t, hipStream_t) { return hipSuccess; }
hipError_t hit_counts(const void*, int64_t, uint32_t, float*, hipStream_t) { return hipSuccess; }
size_t adjoint_sort_words(int64_t, uint32_t) { return 1; }
}

namespace oa_merge {
size_t count_words(int64_t) { return 1; }
size_t most_words(int64_t) { return 1; }
hipError_t select(int, const void*, int64_t, uint32_t, float, int32_t*, uint2*, uint4*, Result*, hipStream_t) { return hipErrorNotSupported; }
hipError_t gather_selected(int, const void*, int64_t, const int32_t*, const uint4*, void*, hipStream_t) { return hipErrorNotSupported; }
int key_bits(uint32_t, uint32_t) { return 1; }
size_t sort_words(int64_t, int) { return 1; }
hipError_t sort_runs(int64_t, const int32_t*, const uint4*, int64_t, float, uint32_t, int, void*, void*, uint32_t*, uint32_t*, uint32_t*, hipStream_t) { return hipErrorNotSupported; }
hipError_t count_runs(int64_t, int32_t*, int64_t, int, const void*, Result*, hipStream_t) { return hipErrorNotSupported; }
hipError_t reduce_runs(int, const void*, int64_t, int32_t*, const uint4*, int64_t, int, const void*, const uint32_t*, void*, int64_t, hipStream_t) { return hipErrorNotSupported; }
}
