// Device results into pageable host memory, and the staging of uploads (private to
// the library).
#pragma once

#include <hip/hip_runtime.h>
#include <cstddef>

namespace tdlb {

// A reference to a callable (dst, begin, end, stream) that enqueues whatever writes
// bytes [begin, end) of the result to dst: pinned host memory that the GPU can
// write, or device memory.
class PieceFn {
public:
    template <typename Fn>
    PieceFn(const Fn& fn)
        : fn_(&fn), call_([](const void* f, void* dst, size_t begin, size_t end, hipStream_t s) {
              return (*static_cast<const Fn*>(f))(dst, begin, end, s);
          }) {}
    hipError_t operator()(void* dst, size_t begin, size_t end, hipStream_t s) const {
        return call_(fn_, dst, begin, end, s);
    }

private:
    const void* fn_;
    hipError_t (*call_)(const void*, void*, size_t, size_t, hipStream_t);
};

// `bytes` of a result to host memory, after the work already on `s`; returns when
// they are there.  Pieces are multiples of `align` bytes.  array: the result where it
// lies in device memory as it is, else null.  hipErrorOutOfMemory: neither pinned nor
// device memory for a piece.
hipError_t read_back(int device, hipStream_t s, void* host, size_t bytes, size_t align, const PieceFn& piece,
                     const void* array = nullptr);

// Device memory for `want` bytes of data that are converted on the device on their way,
// piece by piece: kStageBytes, or less where little is wanted or memory is short (bytes says
// how much; null: there is none).  From the fourth call on one piece a device is kept
// between calls: allocating and freeing it costs 50 us, a tenth of the upload of a 60^3
// tank's Q, but more than a small one where a program has a single use for it.  The
// caller's work on it has ended when it is given back.
constexpr size_t kStageBytes = (size_t)16 << 20;
void* take_stage(int device, size_t want, size_t* bytes);
void give_stage(int device, void* stage, size_t bytes);

// A handle or a batch (a server's too) came or went: what is kept between calls is given
// back with the last one.
void readback_handle(int change);

}  // namespace tdlb
