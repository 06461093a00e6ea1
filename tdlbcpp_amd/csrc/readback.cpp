// Device results into pageable host memory.
//
// A copy into pageable memory runs at the pace of one host thread: the runtime's
// own copies out of its staging buffer (17 GB/s on this host, 10 GB/s into fresh
// pages, which the kernel clears on first touch) against 55 GB/s over the link.
// Here the kernel that forms a piece of the result writes it straight into pinned
// memory (as fast as a copy engine: 53 GB/s), and several threads move finished
// pieces on while later ones are formed, so the pages are touched in parallel.
// Measured, rho and velocity of a tank: 512^3 (2.1 GB) 207 -> 45 ms, 96^3 (14 MB)
// 0.88 -> 0.40 ms.
//
// The pinned buffers are kept between calls (fresh ones fault page by page on the
// host's first reads, at 2 GB/s): at most kMaxRings of each of two sizes, shared by
// all handles and threads, given back with the last handle.  A caller that finds
// all of its size in use waits for one.
#include "readback.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace tdlb {
namespace {

constexpr int kMaxRings = 4;
constexpr int kMaxThreads = 8;  // 87 GB/s into fresh pages, above the link's 55
constexpr size_t kMinPiece = (size_t)1 << 20;
// results of one piece, and larger ones: a slot of 4 MiB per thread
constexpr size_t kRingBytes[2] = {kMinPiece, (size_t)kMaxThreads << 22};

std::mutex g_mu;
std::condition_variable g_cv;
std::vector<void*> g_idle[2];
int g_rings[2] = {0, 0}, g_handles = 0;

hipError_t take_ring(int kind, void** ring) {
    std::unique_lock<std::mutex> lk(g_mu);
    g_cv.wait(lk, [&] { return !g_idle[kind].empty() || g_rings[kind] < kMaxRings; });
    if (!g_idle[kind].empty()) {
        *ring = g_idle[kind].back();
        g_idle[kind].pop_back();
        return hipSuccess;
    }
    const hipError_t e = hipHostMalloc(ring, kRingBytes[kind], hipHostMallocPortable);
    if (e == hipSuccess) g_rings[kind]++;
    return e;
}

void give_ring(int kind, void* ring) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_idle[kind].push_back(ring);
    g_cv.notify_all();
}

}  // namespace

void readback_handle(int change) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_handles += change;
    if (g_handles > 0) return;
    for (int kind = 0; kind < 2; kind++) {
        for (void* p : g_idle[kind]) (void)hipHostFree(p);
        g_rings[kind] -= (int)g_idle[kind].size();
        g_idle[kind].clear();
    }
}

hipError_t read_back(int device, hipStream_t s, void* host, size_t bytes, size_t align, const PieceFn& piece) {
    if (bytes == 0) return hipStreamSynchronize(s);
    const int kind = bytes <= kMinPiece ? 0 : 1;
    void* ring = nullptr;
    hipError_t e = take_ring(kind, &ring);
    if (e != hipSuccess) return e;
    // a thread per piece in flight; small results take the calling thread only
    const int cpus = std::max(1, (int)std::thread::hardware_concurrency());
    const int most = (int)std::min<size_t>(std::max(1, std::min(kMaxThreads, cpus / 2)), (bytes + kMinPiece - 1) / kMinPiece);
    const size_t slot = kind == 0 ? kRingBytes[0] : kRingBytes[1] / kMaxThreads;
    const size_t part = std::min(slot, std::max(kMinPiece, (bytes + 2 * most - 1) / (2 * most))) / align * align;
    std::atomic<size_t> next{0};
    std::atomic<int> failed{hipSuccess};
    auto work = [&](int t) {
        hipError_t r = hipSetDevice(device);
        hipEvent_t done = nullptr;
        if (r == hipSuccess) r = hipEventCreateWithFlags(&done, hipEventDisableTiming);
        char* buf = static_cast<char*>(ring) + (size_t)t * slot;
        while (r == hipSuccess && failed.load() == hipSuccess) {
            const size_t begin = next.fetch_add(part);
            if (begin >= bytes) break;
            const size_t end = std::min(bytes, begin + part);
            r = piece(buf, begin, end, s);
            if (r == hipSuccess) r = hipEventRecord(done, s);
            if (r == hipSuccess) r = hipEventSynchronize(done);
            if (r == hipSuccess) std::memcpy(static_cast<char*>(host) + begin, buf, end - begin);
        }
        if (done) (void)hipEventDestroy(done);
        if (r != hipSuccess) failed.store(r);
    };
    std::vector<std::thread> threads;
    try {
        for (int t = 1; t < most; t++) threads.emplace_back(work, t);
    } catch (const std::system_error&) {
        // no more threads to be had: the ones there are do the work
    }
    work(0);
    for (std::thread& t : threads) t.join();
    e = (hipError_t)failed.load();
    if (e != hipSuccess) (void)hipStreamSynchronize(s);  // nothing may write to the ring any more
    give_ring(kind, ring);
    return e;
}

}  // namespace tdlb
