// Device results into pageable host memory (private to the library).
#pragma once

#include <hip/hip_runtime.h>
#include <cstddef>
#include <functional>

namespace tdlb {

// Enqueues on `s` whatever writes bytes [begin, end) of the result to dst, which
// is pinned host memory that the GPU can write.
using PieceFn = std::function<hipError_t(void* dst, size_t begin, size_t end, hipStream_t s)>;

// `bytes` of a result to host memory, after the work already on `s`; returns when
// they are there.  Pieces are multiples of `align` bytes.
hipError_t read_back(int device, hipStream_t s, void* host, size_t bytes, size_t align, const PieceFn& piece);

// A handle came or went: the pinned buffers are given back with the last one.
void readback_handle(int change);

}  // namespace tdlb
