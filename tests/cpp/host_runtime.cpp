// The HIP runtime calls of libperegrine_hip on host memory, for tests without a GPU: the library's own objects are linked
// with this file instead of the runtime, kernels are not run but noted (name and grid), and what the library does around
// its launches -- its allocations, its pools, its choice of kernels, what it asks of a capturing stream -- can be
// followed.  `pghost_*` are the test's handles: a limit on device memory, allocations that fail, a stream's capture state, the
// launches, the size of coded streams.
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

namespace {
struct launch_rec { std::string name; unsigned grid[3], block[3]; };
struct state {
    std::recursive_mutex mu;
    std::map<const void *, std::string> kernels;
    std::map<const void *, void *> variables;
    std::map<void *, size_t> device;  // live allocations
    size_t mallocs_left = ~(size_t)0, news_left = ~(size_t)0;  // that succeed: device allocations, host objects
    unsigned long long stream_bytes[2] = {1000, 1000};         // of a coded chunk, by side (chunks take turns)
    size_t used = 0, limit = ~(size_t)0, frees = 0, bad_frees = 0, recorded = 0, copied = 0;
    std::map<hipStream_t, bool> capturing;  // true: capture was broken by a forbidden call
    std::vector<launch_rec> launches;
};
// (never destroyed: the library's objects register their kernels before this file's statics would exist, and unload after)
state &sim() { static state *it = new state; return *it; }
using guard = std::lock_guard<std::recursive_mutex>;

// A call that a capture of this thread forbids (allocation, waiting): it fails and breaks the capture.
bool forbidden() {
    for (auto &c : sim().capturing) c.second = true;
    return !sim().capturing.empty();
}
void note(const void *fn, dim3 grid, dim3 block, void **args) {
    guard g(sim().mu);
    const auto it = sim().kernels.find(fn);
    const std::string name = it == sim().kernels.end() ? "?" : it->second;
    sim().launches.push_back({name, {grid.x, grid.y, grid.z}, {block.x, block.y, block.z}});
    if (!sim().capturing.empty()) { ++sim().recorded; return; }
    // the one kernel whose result the host reads before its next launch: a chunk's bits plus one, in pinned memory
    if (name.find("kv_table_kernel") != std::string::npos)
        for (unsigned i = 0; i < grid.x; ++i) (*static_cast<unsigned long long **>(args[1]))[i] = 8 * sim().stream_bytes[i & 1] + 1;
}
hipError_t take(void **p, size_t bytes) {
    if (forbidden()) return hipErrorStreamCaptureUnsupported;
    if (sim().mallocs_left == 0) return hipErrorOutOfMemory;
    if (sim().mallocs_left != ~(size_t)0) --sim().mallocs_left;
    if (bytes > sim().limit - (sim().used < sim().limit ? sim().used : sim().limit)) return hipErrorOutOfMemory;
    *p = aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
    if (!*p) return hipErrorOutOfMemory;
    sim().device[*p] = bytes;
    sim().used += bytes;
    return hipSuccess;
}
}  // namespace

#define TEST_API extern "C" __attribute__((visibility("default")))
TEST_API void pghost_limit(size_t bytes) { guard g(sim().mu); sim().limit = bytes; }
TEST_API void pghost_fail_after(size_t mallocs, size_t news) { guard g(sim().mu); sim().mallocs_left = mallocs; sim().news_left = news; }
TEST_API void pghost_stream_bytes(size_t k, size_t v) { guard g(sim().mu); sim().stream_bytes[0] = k; sim().stream_bytes[1] = v; }
TEST_API size_t pghost_used() { guard g(sim().mu); return sim().used; }
TEST_API size_t pghost_frees() { guard g(sim().mu); return sim().frees; }
TEST_API size_t pghost_bad_frees() { guard g(sim().mu); return sim().bad_frees; }
TEST_API size_t pghost_recorded() { guard g(sim().mu); return sim().recorded; }
TEST_API size_t pghost_copied() { guard g(sim().mu); return sim().copied; }  // of those, copies and fills by the runtime
TEST_API void pghost_begin_capture(void *stream) { guard g(sim().mu); sim().capturing[(hipStream_t)stream] = false; sim().recorded = sim().copied = 0; }
TEST_API int pghost_end_capture(void *stream) {  // 1: the capture is whole
    guard g(sim().mu);
    const bool broken = sim().capturing[(hipStream_t)stream];
    sim().capturing.erase((hipStream_t)stream);
    return !broken;
}
TEST_API void pghost_clear_launches() { guard g(sim().mu); sim().launches.clear(); }
TEST_API size_t pghost_num_launches() { guard g(sim().mu); return sim().launches.size(); }
TEST_API const char *pghost_launch(size_t i, unsigned *grid) {
    guard g(sim().mu);
    memcpy(grid, sim().launches[i].grid, sizeof sim().launches[i].grid);
    return sim().launches[i].name.c_str();
}

// the library's objects, which it asks for without exceptions
void *operator new(size_t bytes, const std::nothrow_t &) noexcept {
    guard g(sim().mu);
    if (sim().news_left == 0) return nullptr;
    if (sim().news_left != ~(size_t)0) --sim().news_left;
    return malloc(bytes ? bytes : 1);
}

extern "C" {
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *fn, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) { guard g(sim().mu); sim().kernels[fn] = name; }
void __hipRegisterVar(void **, void *var, char *, const char *, int, size_t size, int, int) { guard g(sim().mu); sim().variables[var] = calloc(1, size); }

static thread_local struct { dim3 grid, block; size_t lds; hipStream_t stream; } pushed;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) { pushed = {grid, block, lds, stream}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream) {
    *grid = pushed.grid; *block = pushed.block; *lds = pushed.lds; *stream = pushed.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 grid, dim3 block, void **args, size_t, hipStream_t) { note(fn, grid, block, args); return hipSuccess; }
hipError_t hipExtLaunchKernel(const void *fn, dim3 grid, dim3 block, void **args, size_t, hipStream_t, hipEvent_t, hipEvent_t, int) {
    note(fn, grid, block, args);
    return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t bytes) { guard g(sim().mu); return take(p, bytes); }
hipError_t hipFree(void *p) {
    guard g(sim().mu);
    if (!p) return hipSuccess;
    const auto it = sim().device.find(p);
    if (it == sim().device.end()) { ++sim().bad_frees; return hipErrorInvalidValue; }
    sim().used -= it->second;
    sim().device.erase(it);
    ++sim().frees;
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    guard g(sim().mu);
    if (forbidden()) return hipErrorStreamCaptureUnsupported;
    *p = aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { guard g(sim().mu); if (forbidden()) return hipErrorStreamCaptureUnsupported; memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    guard g(sim().mu);
    if (sim().capturing.empty()) memcpy(d, s, n);
    else { ++sim().recorded; ++sim().copied; }
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
    guard g(sim().mu);
    if (!sim().capturing.empty()) { ++sim().recorded; ++sim().copied; }
    else
        for (size_t i = 0; i < h; ++i) memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    guard g(sim().mu);
    if (sim().capturing.empty()) memset(d, v, n);
    else { ++sim().recorded; ++sim().copied; }
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free((void *)s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { guard g(sim().mu); return forbidden() ? hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
    guard g(sim().mu);
    const auto it = sim().capturing.find(s);
    *st = it == sim().capturing.end() ? hipStreamCaptureStatusNone : it->second ? hipStreamCaptureStatusInvalidated : hipStreamCaptureStatusActive;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free((void *)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }

hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {  // (a macro: the runtime's versioned name)
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *sym) { guard g(sim().mu); *p = sim().variables.at(sym); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : e == hipErrorStreamCaptureUnsupported ? "operation not permitted when stream is capturing" : "error"; }
}
