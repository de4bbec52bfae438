// A HIP runtime in host memory, for CPU tests of what the host code
// (fgl_host.cpp) asks of the runtime: allocations, waits, captures, errors.
// Device memory is host memory with a byte limit; copies are made at once;
// a stream capture refuses and counts what may not be called during one, as
// the real runtime does.  Kernel launches do nothing (the test's build makes
// an empty function of every launch entry point); a draw's counters read back
// as zeros: no overflow.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

#include "fgl_internal.h"

namespace {
std::mutex mu;
std::map<void *, size_t> blocks;  // device blocks
size_t live = 0, peak = 0, limit = ~(size_t)0;
long capture_calls = 0, refuse_sync = 0, mallocs = 0;
int capturing = 0;
hipError_t last = hipSuccess;

hipError_t ret(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
// a call that a capture refuses
bool refused() {
    if (!capturing) return false;
    capture_calls++;
    return true;
}
hipStream_t handle() {
    static size_t next = 0;
    return reinterpret_cast<hipStream_t>(++next);
}
}  // namespace

extern "C" {
void fake_limit(size_t bytes) { limit = bytes; }
size_t fake_live() { return live; }
size_t fake_peak() {
    const size_t p = peak;
    peak = live;
    return p;
}
long fake_mallocs() { return mallocs; }
long fake_capture_calls() { return capture_calls; }
void fake_refuse_sync(long n) { refuse_sync = n; }  // the next n device waits are refused
void fake_capturing(int on) { capturing = on; }
int fake_last_error() { return (int)last; }

hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::mutex> lk(mu);
    if (refused()) return ret(hipErrorStreamCaptureUnsupported);
    if (live + n > limit) return ret(hipErrorOutOfMemory);
    *p = std::calloc(1, n);
    if (!*p) return ret(hipErrorOutOfMemory);
    blocks[*p] = n;
    live += n;
    if (live > peak) peak = live;
    mallocs++;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> lk(mu);
    if (!p) return hipSuccess;
    if (capturing) capture_calls++;
    auto it = blocks.find(p);
    if (it == blocks.end()) std::abort();  // freed twice, or not by its start
    live -= it->second;
    blocks.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    if (refused()) return ret(hipErrorStreamCaptureUnsupported);
    if (refuse_sync > 0) {
        refuse_sync--;
        return ret(hipErrorStreamCaptureUnsupported);
    }
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::calloc(1, n);
    return *p ? hipSuccess : ret(hipErrorOutOfMemory);
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    if (!capturing) std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    if (!capturing) std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return ret(hipErrorInvalidValue); }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "refused"; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = handle();
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return refused() ? ret(hipErrorStreamCaptureUnsupported) : hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(handle());
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    capturing = 1;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    capturing = 0;
    *g = reinterpret_cast<hipGraph_t>(handle());
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    *e = reinterpret_cast<hipGraphExec_t>(handle());
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}

// Every tile shape's launches, doing nothing.
namespace fgl {
namespace {
hipError_t draw(const DrawArgs &, hipStream_t) { return hipSuccess; }
hipError_t pass(const DrawArgs &, int, hipStream_t) { return hipSuccess; }
uint32_t one_block(int, const DrawArgs &, bool) { return 1; }
long multi = 0;  // launches of replayed batches
hipError_t many(int, const MultiArgs &, uint32_t, const DrawArgs &, hipStream_t) {
    multi++;
    return hipSuccess;
}
template <class F>
void set(F &slot) {
    if constexpr (std::is_convertible_v<decltype(&draw), F>) slot = draw;
    else if constexpr (std::is_convertible_v<decltype(&pass), F>) slot = pass;
    else if constexpr (std::is_convertible_v<decltype(&one_block), F>) slot = one_block;
    else slot = many;
}
TileOps ops(int w, int h) {
    TileOps t{};
    t.tw = w;
    t.th = h;
    set(t.zero), set(t.vs), set(t.vs_deferred), set(t.scan_top), set(t.emit), set(t.radix_hist), set(t.radix_scan);
    set(t.radix_scatter), set(t.span_count), set(t.span_scan), set(t.spans), set(t.frag_scan), set(t.shade), set(t.rop);
    set(t.zshade), set(t.stage_blocks), set(t.multi);
    return t;
}
}  // namespace
#define FAKE_OPS(w, h)                      \
    const TileOps &tile_ops_##w##x##h() {   \
        static const TileOps t = ops(w, h); \
        return t;                           \
    }
FGL_TILE_SHAPES(FAKE_OPS)
}  // namespace fgl

extern "C" long fake_count_multi() {
    const long n = fgl::multi;
    fgl::multi = 0;
    return n;
}
