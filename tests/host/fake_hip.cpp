// A HIP runtime and kernel launchers in host memory, for tests of the library's
// host code without a GPU: the C ABI's sources are compiled by the host compiler
// and linked with this file.  Allocations are counted and can be made to fail, a
// failed call stays the thread's last error until it is asked for, as in the
// runtime.  Launchers do nothing but what the host code reads back.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>

#include "../../tdlbcpp_amd/csrc/handle.h"
#include "../../tdlbcpp_amd/csrc/kernels.h"

using namespace tdlb;

namespace {

std::mutex mu;
std::map<void*, size_t> device_memory, pinned_memory;
size_t live = 0, peak = 0, limit = (size_t)288 << 30;
int64_t fail_malloc = -1, fail_pinned = -1;  // allocations until one fails, -1: none does
int64_t mallocs = 0, pinned_mallocs = 0, gathers = 0;
std::atomic<int64_t> fail_new{-1};
thread_local hipError_t last = hipSuccess;
thread_local int within = 0;  // allocations of this file's own do not fail
struct Within {
    Within() { within++; }
    ~Within() { within--; }
};

hipError_t error(hipError_t e) { return last = e; }
hipError_t launched() {  // what a launcher ends with
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}

// one more allocation: true if it is to fail; `once` counts down, below -1 every one fails
bool fails(int64_t& left) {
    if (left == -1) return false;
    if (left < -1) return true;
    return left-- == 0;
}

struct Recorded {
    BatchPlan plan;
    int streaming, steps;
};
Recorded recording{};
bool capturing = false;

void advance(const Recorded& r) {
    for (int m = 0; m < r.plan.n_members; m++) {
        MemberDev& md = r.plan.mem_rw[m];
        md.done += std::min<int64_t>(r.steps, md.n_steps - md.done);
    }
}

}  // namespace

// ---------------------------------------------------------------- what the tests set and read
extern "C" {
void fake_fail_malloc(int64_t n) { fail_malloc = n; }
void fake_fail_pinned(int64_t n) { fail_pinned = n; }
void fake_fail_new(int64_t n) { fail_new = n; }
void fake_limit(uint64_t bytes) { limit = bytes; }
void fake_reset_peak() { peak = live; }
uint64_t fake_live() { return live; }
uint64_t fake_peak() { return peak; }
int64_t fake_mallocs() { return mallocs; }
int64_t fake_pinned() { return (int64_t)pinned_memory.size(); }
int64_t fake_pinned_mallocs() { return pinned_mallocs; }
int64_t fake_gathers() { return gathers; }
}

void* operator new(size_t n) {
    if (!within && fail_new.load() >= 0 && fail_new.fetch_sub(1) == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

// ---------------------------------------------------------------- the runtime
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    Within own;
    std::lock_guard<std::mutex> lk(mu);
    *p = nullptr;
    mallocs++;
    if (fails(fail_malloc) || live + n > limit) return error(hipErrorOutOfMemory);
    *p = std::calloc(n ? n : 1, 1);
    device_memory[*p] = n;
    live += n;
    peak = std::max(peak, live);
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> lk(mu);
    if (!p) return hipSuccess;
    auto it = device_memory.find(p);
    if (it == device_memory.end()) std::abort();  // freed twice, or never allocated
    live -= it->second;
    device_memory.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    Within own;
    std::lock_guard<std::mutex> lk(mu);
    *p = nullptr;
    if (fails(fail_pinned)) return error(hipErrorOutOfMemory);
    pinned_mallocs++;
    *p = std::calloc(n, 1);
    pinned_memory[*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> lk(mu);
    if (pinned_memory.erase(p) != 1) std::abort();
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    std::lock_guard<std::mutex> lk(mu);
    *f = limit - std::min(limit, live);
    *t = limit;
    return hipSuccess;
}
hipError_t hipGetLastError() { return launched(); }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* s) {
    *p = const_cast<void*>(s);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    capturing = false;
    *g = reinterpret_cast<hipGraph_t>(new Recorded(recording));
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
    *x = reinterpret_cast<hipGraphExec_t>(new Recorded(*reinterpret_cast<Recorded*>(g)));
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t) {
    advance(*reinterpret_cast<Recorded*>(x));
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    delete reinterpret_cast<Recorded*>(g);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
    delete reinterpret_cast<Recorded*>(x);
    return hipSuccess;
}
}  // extern "C"

// ---------------------------------------------------------------- the launchers
namespace tdlb {
hipError_t launch_fill_q(int, void*, const Grid&, double, hipStream_t) { return launched(); }
hipError_t launch_zero(void*, size_t, hipStream_t) { return launched(); }
hipError_t launch_probe_planes(int, void*, uint64_t, uint64_t, int, int, hipStream_t) { return launched(); }
hipError_t launch_copy(void* d, const void* s, size_t n, hipStream_t) {
    std::memcpy(d, s, n);
    return launched();
}
hipError_t launch_esotwist(int, int, int, void*, void*, const void*, void*, const uint64_t*, const Grid&,
                           const CollideArgs&, float, hipStream_t) { return launched(); }
hipError_t launch_simple(int, int, const void*, void*, void*, const void*, void*, const uint64_t*, const Grid&,
                         const CollideArgs&, float, hipStream_t) { return launched(); }
hipError_t launch_push_all(int, const void*, void*, const Grid&, hipStream_t) { return launched(); }
hipError_t launch_pull_all(int, const void*, void*, const Grid&, hipStream_t) { return launched(); }
hipError_t launch_bounce_back(int, void*, const Grid&, hipStream_t) { return launched(); }
hipError_t launch_ghost_fill(int, const void*, void*, const Grid&, hipStream_t) { return launched(); }
// the boundary's elements are kept in the first bytes of Q, in their own order
hipError_t launch_q_boundary(int esize, int, int to_boundary, void* Q, void* dense, uint64_t begin, uint64_t end,
                             const Grid&, hipStream_t) {
    char* q = static_cast<char*>(Q) + begin * (uint64_t)esize;
    const size_t n = (size_t)(end - begin) * (size_t)esize;
    if (to_boundary) std::memcpy(dense, q, n);
    else std::memcpy(q, dense, n);
    return launched();
}
hipError_t launch_ghost_fill_decode(int, const void*, void*, const Grid&, float, hipStream_t) { return launched(); }
hipError_t launch_ghost_copy(int, const void*, void*, const Grid&, hipStream_t) { return launched(); }
hipError_t launch_mask_from_f(int, const void*, uint64_t*, uint64_t*, const Grid&, hipStream_t) { return launched(); }
hipError_t launch_masked_f(int prec, const void* F, const uint64_t*, uint64_t begin, uint64_t end, void* out,
                           const Grid&, hipStream_t) {
    const size_t cell = 3 * (prec == 1 ? 8 : 4);
    std::memcpy(out, static_cast<const char*>(F) + begin * cell, (size_t)(end - begin) * cell);
    return launched();
}
hipError_t launch_zero_interior_o(uint8_t*, const Grid&, hipStream_t) { return launched(); }
hipError_t launch_force_prepare(int, const PointsDev&, int64_t, int64_t, void*, const uint64_t*, uint64_t*,
                                const Grid&, hipStream_t) { return launched(); }
hipError_t launch_list_unpack(int, const tdlb_ib_point*, int64_t, int, const PointsDev&, const uint64_t*, uint64_t*,
                              uint64_t, hipStream_t) { return launched(); }
size_t list_marks_bytes(const Grid& g, int* blocks) {
    const size_t plane = (size_t)g.xg1 * g.zg1 * sizeof(uint32_t);
    const bool lds = plane <= kListLdsBytes;
    *blocks = lds ? g.yg1 : std::min(g.yg1, 256);
    return lds ? 0 : plane;
}
hipError_t launch_list_levels(const PointsDev&, int64_t, int64_t*, uint32_t*, int blocks, int32_t*, const Grid&,
                              hipStream_t) {
    return blocks < 1 ? hipErrorInvalidValue : launched();
}
hipError_t launch_list_planes(int, int, int, const PointsDev&, int64_t, int64_t*, uint32_t*, int blocks, const void*,
                              void*, const uint64_t*, uint64_t*, const Grid&, double, double, float, hipStream_t) {
    return blocks < 1 ? hipErrorInvalidValue : launched();
}
hipError_t launch_force_gather(int, int, int, int, const ForceGeom&, const BladeStep&, const GatherBlocks&,
                               const void*, void*, const uint64_t*, uint64_t*, const uint64_t*, const Grid&, float,
                               hipStream_t) {
    gathers++;
    return launched();
}
hipError_t launch_force_levels(int, const ForceGeom&, void*, uint64_t*, const Grid&, double, double, hipStream_t) {
    return launched();
}
hipError_t allow_level_lds(int) { return launched(); }
hipError_t launch_eso_pipe(int, int, int, const PipeArgs&, const Grid&, const CollideArgs&, float, uint32_t, uint32_t,
                           hipStream_t) { return launched(); }
uint32_t row_lanes(const Grid&) { return 256; }
bool line_rows_bytes(const Grid&, size_t) { return false; }
int pipe_xcc_check(hipStream_t) { return 1; }
hipError_t launch_reduce(int, int, int, int, const void*, const void*, const uint64_t*, const Grid&,
                         const ReduceArgs&, float, double*, double*, hipStream_t) { return launched(); }
// {t, t + 1/4, t + 1/2, t + 3/4} of interior cell t
hipError_t launch_macroscopic(int prec, int, int, int, const void*, const void*, const uint64_t*, const Grid&, float,
                              uint64_t begin, uint64_t end, void* out, hipStream_t) {
    for (uint64_t t = begin; t < end; t++)
        for (int a = 0; a < 4; a++) {
            const double v = (double)t + 0.25 * a;
            if (prec == 1) static_cast<double*>(out)[4 * (t - begin) + a] = v;
            else static_cast<float*>(out)[4 * (t - begin) + a] = (float)v;
        }
    return launched();
}
hipError_t launch_regrid(int, const void*, void*, int, const void*, void*, const Grid&, const Grid&, hipStream_t) {
    return launched();
}
hipError_t launch_nu_convert(int, int, const void*, void*, uint64_t, hipStream_t) { return launched(); }
hipError_t launch_plane_xz(int, const void*, const void*, const uint64_t*, const uint8_t*, const Grid&, int, int64_t,
                           int64_t, PlaneRec4*, PlaneRec3*, uint8_t*, hipStream_t) { return launched(); }
hipError_t launch_vorticity(int, int, int, int, const void*, const Grid&, int, int, const uint8_t*, void*, float,
                            hipStream_t) { return launched(); }
hipError_t launch_static_rows(int, const PointsDev&, int64_t, const int32_t*, void*, hipStream_t) {
    return launched();
}
hipError_t launch_solid_mask(double, double, double, uint8_t*, const Grid&, int, hipStream_t) { return launched(); }
hipError_t launch_batch_step(int, int streaming, const BatchPlan& plan, int steps, hipStream_t) {
    recording = Recorded{plan, streaming, steps};
    if (!capturing) advance(recording);
    return launched();
}
int64_t batch_coll_blocks(const Grid&, int, int) { return 1; }
hipError_t launch_batch_fused(int, int, const BatchPlan&, hipStream_t) { return launched(); }
}  // namespace tdlb
