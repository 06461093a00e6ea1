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
// all handles and threads, given back with the last handle or batch.  A caller that finds
// all of its size in use waits for one; where pinned memory is not to be had, pieces
// are formed in device memory and copied from there.  No C++ exception leaves here:
// fewer threads do the work where more are not to be had.
#include "readback.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace tdlb {
namespace {

constexpr int kMaxRings = 4;
constexpr int kMaxThreads = 8;  // 87 GB/s into fresh pages, above the link's 55
constexpr size_t kMinPiece = (size_t)1 << 20;
// results of one piece, and larger ones: a slot of 4 MiB per thread
constexpr size_t kRingBytes[2] = {kMinPiece, (size_t)kMaxThreads << 22};

// Making a buffer and giving it back costs 1 to 4 ms where the buffer is large (the
// next allocations pay for it), so programs that read little between their first
// handle and their last take the plain copy.  A tank created, read and destroyed, by
// plain copies and through buffers made at once: 60^3 with three results (10 MB) 0.92
// and 1.8 ms, 80^3 (23 MB) 1.7 and 2.9, 96^3 one result (14 MB) 2.7 and 2.6, 128^3
// (34 MB) 5.9 and 3.3; of small results 36^3 one (0.7 MB) 0.24 and 0.35.
constexpr int kSmallReads = 4;                      // the small buffer from the fourth small result on
constexpr size_t kLargeRead = (size_t)12 << 20;     // the large one for a result of this size
constexpr size_t kLargeBytes = (size_t)64 << 20;    // or from this many bytes of larger ones on
// Arrays that lie in device memory as they are come by a plain copy up to here: O of
// 30^3 11 us (through a buffer 19), of 60^3 (0.24 MB) 21 (29), of 80^3 (0.55 MB) 35 either way.
constexpr size_t kPlainArray = (size_t)1 << 19;

std::mutex g_mu;
std::condition_variable g_cv;
void* g_idle[2][kMaxRings];
int g_n_idle[2] = {0, 0}, g_rings[2] = {0, 0}, g_handles = 0;
int g_reads[2] = {0, 0};  // reads while there was no buffer, and their bytes
size_t g_bytes[2] = {0, 0};

constexpr int kStageDevices = 64;  // tdlb_cu_create refuses device ids beyond
void* g_stage[kStageDevices] = {};
constexpr int kStageUses = 4;
int g_stage_uses[kStageDevices] = {};  // without a piece that was kept

// null: no buffer of this size is there, and none can be made or is worth it yet
void* take_ring(int kind, size_t bytes) {
    std::unique_lock<std::mutex> lk(g_mu);
    for (;;) {
        if (g_n_idle[kind] > 0) return g_idle[kind][--g_n_idle[kind]];
        if (g_rings[kind] < kMaxRings) {
            if (g_rings[kind] == 0) {
                g_reads[kind]++;
                g_bytes[kind] += bytes;
                if (kind == 0 ? g_reads[kind] < kSmallReads : bytes < kLargeRead && g_bytes[kind] < kLargeBytes)
                    return nullptr;
            }
            void* ring = nullptr;
            if (hipHostMalloc(&ring, kRingBytes[kind], hipHostMallocPortable) == hipSuccess) {
                g_rings[kind]++;
                return ring;
            }
            (void)hipGetLastError();  // not the next launch's
            if (g_rings[kind] == 0) return nullptr;
        }
        g_cv.wait(lk, [&] { return g_n_idle[kind] > 0; });
    }
}

void give_ring(int kind, void* ring) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_idle[kind][g_n_idle[kind]++] = ring;
    g_cv.notify_all();
}

}  // namespace

void readback_handle(int change) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_handles += change;
    if (g_handles > 0) return;
    for (int d = 0; d < kStageDevices; d++) {
        if (g_stage[d]) (void)hipFree(g_stage[d]);
        g_stage[d] = nullptr;
        g_stage_uses[d] = 0;
    }
    for (int kind = 0; kind < 2; kind++) {
        for (int a = 0; a < g_n_idle[kind]; a++) (void)hipHostFree(g_idle[kind][a]);
        g_rings[kind] -= g_n_idle[kind];
        g_n_idle[kind] = 0;
        g_reads[kind] = 0;
        g_bytes[kind] = 0;
    }
}

void* take_stage(int device, size_t want, size_t* bytes) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if (void* p = g_stage[device]) {
            g_stage[device] = nullptr;
            *bytes = kStageBytes;
            return p;
        }
        *bytes = ++g_stage_uses[device] < kStageUses ? std::min(want, kStageBytes) : kStageBytes;
    }
    for (;; *bytes /= 2) {
        void* p = nullptr;
        if (hipMalloc(&p, *bytes) == hipSuccess) return p;
        (void)hipGetLastError();  // not the next launch's
        if (*bytes / 2 < kMinPiece) break;
    }
    return nullptr;
}

void give_stage(int device, void* stage, size_t bytes) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if (bytes == kStageBytes && !g_stage[device]) {
            g_stage[device] = stage;
            return;
        }
    }
    (void)hipFree(stage);
}

// Without pinned memory: pieces in device memory, copied from there one after the other.
static hipError_t by_device_pieces(int device, hipStream_t s, char* host, size_t bytes, size_t align,
                                   const PieceFn& piece) {
    size_t room = 0;
    void* const stage = take_stage(device, bytes, &room);
    if (!stage) return hipErrorOutOfMemory;
    const size_t part = room / align * align;
    hipError_t e = hipSuccess;
    for (size_t begin = 0; begin < bytes && e == hipSuccess; begin += part) {
        const size_t end = std::min(bytes, begin + part);
        e = piece(stage, begin, end, s);
        if (e == hipSuccess) e = hipMemcpyAsync(host + begin, stage, end - begin, hipMemcpyDeviceToHost, s);
    }
    const hipError_t done = hipStreamSynchronize(s);
    give_stage(device, stage, room);
    return e == hipSuccess ? done : e;
}

hipError_t read_back(int device, hipStream_t s, void* host, size_t bytes, size_t align, const PieceFn& piece,
                     const void* array) {
    if (bytes == 0) return hipStreamSynchronize(s);
    const int kind = bytes <= kMinPiece ? 0 : 1;
    void* const ring = array && bytes <= kPlainArray ? nullptr : take_ring(kind, bytes);
    if (!ring && array) {
        const hipError_t e = hipMemcpyAsync(host, array, bytes, hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    if (!ring) return by_device_pieces(device, s, static_cast<char*>(host), bytes, align, piece);
    // a thread per piece in flight; small results take the calling thread only
    const int cpus = std::max(1, (int)std::thread::hardware_concurrency());
    const int most = (int)std::min<size_t>(std::max(1, std::min(kMaxThreads, cpus / 2)), (bytes + kMinPiece - 1) / kMinPiece);
    const size_t slot = kind == 0 ? kRingBytes[0] : kRingBytes[1] / kMaxThreads;
    const size_t part = std::min(slot, std::max(kMinPiece, (bytes + 2 * most - 1) / (2 * most))) / align * align;
    std::atomic<size_t> next{0};
    std::atomic<int> failed{hipSuccess};
    auto work = [&](int t) {
        hipError_t r = hipSetDevice(device);
        hipEvent_t done = nullptr;  // of this thread's pieces among those of several
        if (r == hipSuccess && most > 1) r = hipEventCreateWithFlags(&done, hipEventDisableTiming);
        char* buf = static_cast<char*>(ring) + (size_t)t * slot;
        while (r == hipSuccess && failed.load() == hipSuccess) {
            const size_t begin = next.fetch_add(part);
            if (begin >= bytes) break;
            const size_t end = std::min(bytes, begin + part);
            r = piece(buf, begin, end, s);
            if (r == hipSuccess && done) r = hipEventRecord(done, s);
            if (r == hipSuccess) r = done ? hipEventSynchronize(done) : hipStreamSynchronize(s);
            if (r == hipSuccess) std::memcpy(static_cast<char*>(host) + begin, buf, end - begin);
        }
        if (done) (void)hipEventDestroy(done);
        if (r != hipSuccess) failed.store(r);
    };
    std::thread threads[kMaxThreads];
    int started = 1;
    try {
        for (; started < most; started++) threads[started] = std::thread(work, started);
    } catch (const std::exception&) {
        // no more threads (std::system_error) or memory for one: the ones there are do the work
    }
    work(0);
    for (int t = 1; t < started; t++) threads[t].join();
    const hipError_t e = (hipError_t)failed.load();
    if (e != hipSuccess) (void)hipStreamSynchronize(s);  // nothing may write to the ring any more
    give_ring(kind, ring);
    return e;
}

}  // namespace tdlb
