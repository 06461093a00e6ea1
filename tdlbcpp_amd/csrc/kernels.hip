// gfx950 kernels of the 18-velocity Eggels-Somers ComputeUnit.
//
// Mapping: one thread per interior cell, k (the fastest index of both layouts)
// on the lanes, one block per run of k in one (i,j) row.  In LIJK every slot
// load and store of a wavefront is a contiguous 256 B run; every memory
// location is read once and written once per step, so the kernels move the
// algorithmic 2 x 18 x sizeof(T) bytes per cell (+ Nu with LES).
//
// Reference semantics (file:line in the reference tree):
//   collision  CollisionEgglesSomers.hpp:26-181   moments  :185-256
//   Esotwist accessors  StreamingEsoteric.hpp:27-180
//   Simple push/pull    StreamingSimple.hpp:18-126   bounce-back Boundary.hpp:13-250
//   forcing             Forcing.hpp:56-176
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "codec16.h"
#include "device.h"
#include "es_collide.h"
#include "kernels.h"
#include "rushton.h"

namespace tdlb {

namespace {

constexpr int kBlock = 256;
// Stream-collide kernels take one block per interior k-row when the row fits
// (up to kRowBlock lanes).  The population arrays keep interior cells only in
// their rows (see device.h), so a block's run of each slot plane is whole
// lines that no other block touches; at 512^3 one 512-lane block per row
// measured 4 % faster than two 256-lane blocks in FP32 and 3-4 % in 16 bits.
constexpr int kRowBlock = 512;
template <typename S>
constexpr int row_block_max() { return kRowBlock; }

// Blocks take rows in dispatch order (round-robin over the 8 XCDs): every line is
// read by one row only, and all XCDs streaming through one region of HBM together
// are 5 % faster than each XCD on a contiguous range of its own.

// ------------------------------------------------------------------ precisions
// S: stored population type, T: arithmetic and F type, N: stored Nu type, D:
// type the reference's double literals promote to.  kShift: populations are
// stored as scaled deviations from the rest populations (see shift_scale) and
// Nu in the same 16-bit format (enc_nu / dec_nu).
struct PrecF32 {
    using S = float; using T = float; using N = float; using D = double;
    static constexpr bool kShift = false;
};
struct PrecF64 {
    using S = double; using T = double; using N = double; using D = double;
    static constexpr bool kShift = false;
};
// The 16-bit formats: enc rounds the scaled deviation s to the stored type
// (round to nearest even), dec widens it exactly; enc_dev / dec_dev take the
// unscaled deviation s / k of direction d (k = shift_scale(d), a power of two),
// also exactly.  Nu (>= 0, 1e-6 .. 1e-2 in a stirred tank) is stored in 16
// bits, scaled by 2^10 in fp16 so that it stays above fp16's smallest normal
// (6.1e-5) down to 6e-8.
struct PrecF16 {
    using S = _Float16; using T = float; using N = _Float16; using D = float;
    static constexpr bool kShift = true;
    __device__ static S enc(float s) { return (S)s; }
    __device__ static float dec(S x) { return (float)x; }
    __device__ static S enc_dev(float v, int d) { return enc(v * shift_scale(d)); }
    __device__ static float dec_dev(S x, int d) { return dec(x) * (1.0f / shift_scale(d)); }
    __host__ __device__ static N enc_nu(float v) { return (N)(v * 1024.0f); }
    __host__ __device__ static float dec_nu(N x) { return (float)x * (1.0f / 1024.0f); }
};
struct PrecBF16 {
    using S = __bf16; using T = float; using N = __bf16; using D = float;
    static constexpr bool kShift = true;
    __device__ static S enc(float s) { return (S)s; }
    __device__ static float dec(S x) { return (float)x; }
    __device__ static S enc_dev(float v, int d) { return enc(v * shift_scale(d)); }
    __device__ static float dec_dev(S x, int d) { return dec(x) * (1.0f / shift_scale(d)); }
    __host__ __device__ static N enc_nu(float v) { return (N)v; }
    __host__ __device__ static float dec_nu(N x) { return (float)x; }
};
// E3M12 (codec16.h): 12 fraction bits for the deviations, the scale k folded
// into the code's exponent; Nu as in PrecF16.
struct PrecE3M12 {
    using S = int16_t; using T = float; using N = _Float16; using D = float;
    static constexpr bool kShift = true;
    __device__ static S enc(float s) { return e3m12_encode<0>(s); }
    __device__ static float dec(S x) { return e3m12_decode<0>(x); }
    __device__ static S enc_dev(float v, int d) { return d < 6 ? e3m12_encode<1>(v) : e3m12_encode<2>(v); }
    __device__ static float dec_dev(S x, int d) { return d < 6 ? e3m12_decode<1>(x) : e3m12_decode<2>(x); }
    __host__ __device__ static N enc_nu(float v) { return PrecF16::enc_nu(v); }
    __host__ __device__ static float dec_nu(N x) { return PrecF16::dec_nu(x); }
};
// bit patterns moved unchanged
template <typename W>
struct RawBits {
    using S = W; using T = W; using N = W; using D = W;
    static constexpr bool kShift = false;
};

// Cache hints of the stream-collide accesses.  In LIJK a wavefront of the fused
// Esotwist kernel reads and writes most slot planes at its own k positions,
// lines that no other wavefront touches: those accesses carry the
// non-temporal hint (nt).  The planes it reads at k+1 share their edge line
// with the next wavefront, which finds it in the cache only without the hint.
// This holds only when every k-row of a slot plane is a whole number of lines:
// otherwise a row's first and last lines are shared with the neighbouring rows'
// blocks and the hint costs a refetch (line_rows).  Measured (Esotwist, LIJK):
// 512^3 FP32 4.4 % faster with the hint on the unshifted planes (on loads only
// 1.8 % slower, on every access 6 % slower), 320^3 6 % faster in FP32 and FP16;
// rows off the line grid 9-27 % slower (200^3, and 160^3 / 96^3 in 16 bits).
// IJKL (a line holds slots of several cells) is 35 % slower with it; the Simple
// pull shows no difference; batches, whose tiles mix tanks, take no hint.  The
// hint is a template argument: each instantiation holds one kind of access, and
// call sites pick the instantiation per plane (a runtime flag lets the compiler
// merge the two accesses of one address and drop the hint).
template <bool NT, typename S>
__device__ __forceinline__ S load_hint(const S* __restrict__ p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}
template <bool NT, typename S>
__device__ __forceinline__ void store_hint(S* __restrict__ p, S v) {
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}

template <typename PR, bool NT = false>
__device__ __forceinline__ typename PR::T load_pop(const typename PR::S* __restrict__ Q, uint64_t a, int d,
                                                   float rho0) {
    // (dec + c0) / k as one multiply-add: x / k and c0 / k are exact (k a power of two)
    if constexpr (PR::kShift)
        return fmaf(PR::dec(load_hint<NT>(Q + a)), 1.0f / shift_scale(d),
                    shift_offset(rho0) * (1.0f / shift_scale(d)));
    else return load_hint<NT>(Q + a);
}
template <typename PR>
__device__ __forceinline__ typename PR::T load_nu(const typename PR::N* __restrict__ Nu, uint64_t n) {
    if constexpr (PR::kShift) return PR::dec_nu(Nu[n]);
    else return Nu[n];
}
template <typename PR>
__device__ __forceinline__ void store_nu(typename PR::N* __restrict__ Nu, uint64_t n, typename PR::T v) {
    if constexpr (PR::kShift) Nu[n] = PR::enc_nu(v);
    else Nu[n] = v;
}
template <typename PR, bool NT = false>
__device__ __forceinline__ void store_pop(typename PR::S* __restrict__ Q, uint64_t a, int d, typename PR::T v,
                                          float rho0) {
    // k v - c0 as one multiply-add (k v is exact)
    if constexpr (PR::kShift) store_hint<NT>(Q + a, PR::enc(fmaf(v, shift_scale(d), -shift_offset(rho0))));
    else store_hint<NT>(Q + a, v);
}
// k-rows of the population planes start and end on 128-byte lines
template <typename S>
inline bool line_rows(const Grid& g) {
    return ((uint64_t)g.qz * sizeof(S)) % 128 == 0 && ((uint64_t)g.qsize * sizeof(S)) % 128 == 0 &&
           ((uint64_t)g.qyz * sizeof(S)) % 128 == 0;
}

// The fused collision of the 16-bit formats works on deviations from the rest
// populations c0 / k (es_collide_dev): f - c0 / k = dec(s) / k and the stored
// value of a deviation p' is k p', both exact (k a power of two), so the
// 16-bit rounding is the only one between collisions.
template <typename PR, bool NT = false>
__device__ __forceinline__ float load_dev(const typename PR::S* __restrict__ Q, uint64_t a, int d) {
    return PR::dec_dev(load_hint<NT>(Q + a), d);
}
template <typename PR, bool NT = false>
__device__ __forceinline__ void store_dev(typename PR::S* __restrict__ Q, uint64_t a, int d, float v) {
    store_hint<NT>(Q + a, PR::enc_dev(v, d));
}
// density of the rest populations c0 / k summed over the 18 directions
__device__ __forceinline__ float rest_density(float rho0) { return 6.0f * shift_offset(rho0); }
// the hardware's reciprocal and square root (1 ulp) for the float collision of
// the 16-bit formats; the IEEE-exact forms expand to ~9 instructions each
struct HwOps {
    __device__ static float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
    __device__ static float sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
};

// ------------------------------------------------------------------ fills
// every slot of the population array, row padding included
template <typename T>
__global__ void k_fill_q(T* __restrict__ Q, Grid g, T rho) {
    const uint64_t total = g.qsize * (uint64_t)kQ;
    for (uint64_t a = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; a < total;
         a += (uint64_t)gridDim.x * blockDim.x) {
        Q[a] = a < g.qsize ? rho : T(0);
    }
}

// Between the population array of the kernels and the dense array of the boundary
// (layout BL: IJKL n*18 + l, LIJK l*size + n), elements [begin, end) of the
// latter, of which `dense` is element begin; one boundary element per thread.
template <typename W, int BL, bool TO_BOUNDARY>
__global__ void k_q_boundary(W* __restrict__ Q, W* __restrict__ dense, uint64_t begin, uint64_t end, Grid g) {
    for (uint64_t a = begin + blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; a < end;
         a += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t n, l;
        if (BL == LayoutLIJK) {
            l = a / g.size;
            n = a - l * g.size;
        } else {
            n = a / kQ;
            l = a - n * kQ;
        }
        int i, j, k;
        decode_cell(g, n, i, j, k);
        const uint64_t q = qaddr(g, qcell(g, i, j, k), (int)l);
        if (TO_BOUNDARY) dense[a - begin] = Q[q];
        else Q[q] = dense[a - begin];
    }
}

__global__ void k_zero_words(uint32_t* __restrict__ p, uint64_t n) {
    for (uint64_t a = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; a < n; a += (uint64_t)gridDim.x * blockDim.x)
        p[a] = 0u;
}
__global__ void k_zero_bytes(uint8_t* __restrict__ p, uint64_t n) {
    for (uint64_t a = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; a < n; a += (uint64_t)gridDim.x * blockDim.x)
        p[a] = 0;
}
__global__ void k_copy_words(uint32_t* __restrict__ d, const uint32_t* __restrict__ s, uint64_t n) {
    for (uint64_t a = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; a < n; a += (uint64_t)gridDim.x * blockDim.x)
        d[a] = s[a];
}
__global__ void k_copy_bytes(uint8_t* __restrict__ d, const uint8_t* __restrict__ s, uint64_t n) {
    for (uint64_t a = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; a < n; a += (uint64_t)gridDim.x * blockDim.x)
        d[a] = s[a];
}

// A block takes consecutive cells of one interior i plane, rows back to back, so
// only the plane's last block has lanes without a cell.
constexpr int kFlatBlock = 256;
struct FlatTile {
    uint32_t blocks;  // of an i plane
    uint32_t recip;   // ceil(2^32 / zg1): the high word of r * recip is r / zg1 while yg1 * zg1 * zg1 < 2^32
};
__device__ __forceinline__ bool flat_cell(const Grid& g, const FlatTile& tile, int& i, int& j, int& k) {
    const uint32_t ip = blockIdx.x / tile.blocks, r = (blockIdx.x - ip * tile.blocks) * blockDim.x + threadIdx.x;
    if (r >= (uint32_t)g.yg1 * (uint32_t)g.zg1) return false;
    const uint32_t jp = __umulhi(r, tile.recip);
    i = (int)ip + 1;
    j = (int)jp + 1;
    k = (int)(r - jp * (uint32_t)g.zg1) + 1;
    return true;
}

// ------------------------------------------------------------------ Esotwist
// Direction d of cell c is stored at home(c,d) = c + (1 where e_d < 0, periodic
// on the interior), in slot d at even parity and opp(d) at odd parity.  read
// takes the 18 values from there; write puts population d where the read of
// opp(d) looks (StreamingEsoteric.hpp:82-130); writeMoments puts value d back
// where d was read.
// mout receives the moments of MODE_MOM: Q itself (in place) when populations
// are stored as T, a separate T array in the reference layout otherwise.
template <typename PR, int MODE, int EVEN, bool HINT = false>
__device__ __forceinline__ void esotwist_cell(typename PR::S* __restrict__ Q, typename PR::T* mout,
                                              const typename PR::T* __restrict__ F, typename PR::N* __restrict__ Nu,
                                              const uint64_t* __restrict__ fmask, const Grid& g,
                                              const CollideParams<typename PR::T>& P, float rho0, int i, int j,
                                              int k) {
    using T = typename PR::T;
    using D = typename PR::D;
    const uint32_t n = cell_index(g, i, j, k);
    const uint32_t qn = qcell(g, i, j, k);
    const int32_t di = (i == g.xg1) ? -(int32_t)((uint32_t)(g.xg1 - 1) * g.qyz) : (int32_t)g.qyz;
    const int32_t dj = (j == g.yg1) ? -(int32_t)((uint32_t)(g.yg1 - 1) * g.qz) : (int32_t)g.qz;
    const int32_t dk = (k == g.zg1) ? -(g.zg1 - 1) : 1;

    uint32_t home[kQ];
#pragma unroll
    for (int d = 0; d < kQ; d++)
        home[d] = qn + (uint32_t)((twist_dx(d) ? di : 0) + (twist_dy(d) ? dj : 0) + (twist_dz(d) ? dk : 0));

    T v[kQ];
#pragma unroll
    for (int d = 0; d < kQ; d++) {
        const uint64_t a = qaddr(g, home[d], EVEN ? d : opposite(d));
        // reduced-precision storage keeps the moments of MODE_COLL in mout
        // with HINT, the planes read at the cell's own k take the streaming hint
        if constexpr (PR::kShift && MODE == MODE_COLL) v[d] = mout[a];
        else if constexpr (MODE == MODE_FUSED && PR::kShift) {
            if (!HINT || twist_dz(d)) v[d] = load_dev<PR>(Q, a, d);
            else v[d] = load_dev<PR, true>(Q, a, d);
        } else if constexpr (MODE == MODE_FUSED) {
            if (!HINT || twist_dz(d)) v[d] = load_pop<PR>(Q, a, d, rho0);
            else v[d] = load_pop<PR, true>(Q, a, d, rho0);
        }
        else v[d] = load_pop<PR>(Q, a, d, rho0);
    }

    if (MODE == MODE_MOM) {
        T m[kQ];
        es_moments<T, D>(v, m);
#pragma unroll
        for (int d = 0; d < kQ; d++) mout[qaddr(g, home[d], EVEN ? d : opposite(d))] = m[d];
        return;
    }

    T fx = T(0), fy = T(0), fz = T(0);
    if (mask_test(fmask, g, i, j, k)) {
        fx = F[3 * (uint64_t)n + 0];
        fy = F[3 * (uint64_t)n + 1];
        fz = F[3 * (uint64_t)n + 2];
    }
    T nuc = P.use_les ? load_nu<PR>(Nu, n) : T(0);
    T p[kQ];
    if constexpr (MODE == MODE_FUSED && PR::kShift) {
        es_collide_dev<HwOps>(v, rest_density(rho0), fx, fy, fz, nuc, P, p);
    } else if (MODE == MODE_FUSED) {
        T m[kQ];
        es_moments<T, D>(v, m);
        es_collide<T, D>(m, fx, fy, fz, nuc, P, p);
    } else {
        es_collide<T, D>(v, fx, fy, fz, nuc, P, p);
    }
    if (P.use_les) store_nu<PR>(Nu, n, nuc);
    // Recompute the 18 home cells instead of keeping them live through the
    // collision: the opaque copy stops the compiler from reusing the load
    // addresses, which frees ~36 VGPRs and raises occupancy.
    uint32_t n2 = qn;
    int32_t di2 = di, dj2 = dj, dk2 = dk;
    asm volatile("" : "+v"(n2), "+v"(di2), "+v"(dj2), "+v"(dk2));
#pragma unroll
    for (int d = 0; d < kQ; d++) {
        const int e = opposite(d);
        const uint32_t h = n2 + (uint32_t)((twist_dx(e) ? di2 : 0) + (twist_dy(e) ? dj2 : 0) + (twist_dz(e) ? dk2 : 0));
        const uint64_t a = qaddr(g, h, EVEN ? e : opposite(e));
        if constexpr (MODE == MODE_FUSED) {
            if (!HINT || twist_dz(e)) {
                if constexpr (PR::kShift) store_dev<PR>(Q, a, d, p[d]);
                else store_pop<PR>(Q, a, d, p[d], rho0);
            } else {
                if constexpr (PR::kShift) store_dev<PR, true>(Q, a, d, p[d]);
                else store_pop<PR, true>(Q, a, d, p[d], rho0);
            }
        }
        else store_pop<PR>(Q, a, d, p[d], rho0);
    }
}

template <typename PR, int MODE, int EVEN, bool HINT>
__global__ __launch_bounds__(kRowBlock) void k_esotwist(typename PR::S* __restrict__ Q, typename PR::T* mout,
                                                     const typename PR::T* __restrict__ F,
                                                     typename PR::N* __restrict__ Nu,
                                                     const uint64_t* __restrict__ fmask, Grid g,
                                                     CollideParams<typename PR::T> P, uint32_t nkb, float rho0) {
    const RowBlock rb = row_block(g, blockIdx.x, nkb, blockDim.x);
    const int k = rb.k0 + (int)threadIdx.x;
    if (k > g.zg1) return;
    esotwist_cell<PR, MODE, EVEN, HINT>(Q, mout, F, Nu, fmask, g, P, rho0, rb.i, rb.j, k);
}

// Fused step over the cells of an i plane back to back (flat_tile)
template <typename PR, int EVEN>
__global__ __launch_bounds__(kFlatBlock) void k_esotwist_flat(typename PR::S* __restrict__ Q,
                                                              const typename PR::T* __restrict__ F,
                                                              typename PR::N* __restrict__ Nu,
                                                              const uint64_t* __restrict__ fmask, Grid g,
                                                              CollideParams<typename PR::T> P, FlatTile tile, float rho0) {
    int i, j, k;
    if (!flat_cell(g, tile, i, j, k)) return;
    esotwist_cell<PR, MODE_FUSED, EVEN>(Q, nullptr, F, Nu, fmask, g, P, rho0, i, j, k);
}

// ------------------------------------------------------------------ Simple
// In-place collide / moments, or pull from src (the two-lattice form of the
// reference's in-place push: slot d of an interior cell c takes src[c-e_d][d]
// when c-e_d is interior and keeps src[c][d] otherwise).
template <typename PR, int MODE>
__device__ __forceinline__ void simple_cell(const typename PR::S* src,
                                            typename PR::S* dst,   // equal to src for in-place modes
                                            typename PR::T* mout,  // moments output of the MOM modes
                                            const typename PR::T* __restrict__ F, typename PR::N* __restrict__ Nu,
                                            const uint64_t* __restrict__ fmask, const Grid& g,
                                            const CollideParams<typename PR::T>& P, float rho0, int i, int j,
                                            int k) {
    using T = typename PR::T;
    using D = typename PR::D;
    const uint32_t n = cell_index(g, i, j, k);
    const uint32_t qn = qcell(g, i, j, k);

    T v[kQ];
    if (MODE == MODE_FUSED || MODE == MODE_MOM_PULL) {
        const bool im = i >= 2, ip = i <= g.xg1 - 1;  // cell i-1 / i+1 interior
        const bool jm = j >= 2, jp = j <= g.yg1 - 1;
        const bool km = k >= 2, kp = k <= g.zg1 - 1;
#pragma unroll
        for (int d = 0; d < kQ; d++) {
            const int ex = dir_x(d), ey = dir_y(d), ez = dir_z(d);
            const bool ok = (ex > 0 ? im : ex < 0 ? ip : true) && (ey > 0 ? jm : ey < 0 ? jp : true) &&
                            (ez > 0 ? km : ez < 0 ? kp : true);
            const int32_t off = -(ex * (int32_t)g.qyz + ey * (int32_t)g.qz + ez);
            const uint64_t a = qaddr(g, ok ? qn + (uint32_t)off : qn, d);
            if constexpr (PR::kShift && MODE == MODE_FUSED) v[d] = load_dev<PR>(src, a, d);
            else v[d] = load_pop<PR>(src, a, d, rho0);
        }
    } else {
#pragma unroll
        for (int d = 0; d < kQ; d++) {
            if constexpr (PR::kShift && MODE == MODE_COLL) v[d] = mout[qaddr(g, qn, d)];
            else v[d] = load_pop<PR>(src, qaddr(g, qn, d), d, rho0);
        }
    }

    if (MODE == MODE_MOM || MODE == MODE_MOM_PULL) {
        T m[kQ];
        es_moments<T, D>(v, m);
#pragma unroll
        for (int d = 0; d < kQ; d++) mout[qaddr(g, qn, d)] = m[d];
        return;
    }

    T fx = T(0), fy = T(0), fz = T(0);
    if (mask_test(fmask, g, i, j, k)) {
        fx = F[3 * (uint64_t)n + 0];
        fy = F[3 * (uint64_t)n + 1];
        fz = F[3 * (uint64_t)n + 2];
    }
    T nuc = P.use_les ? load_nu<PR>(Nu, n) : T(0);
    T p[kQ];
    if constexpr (MODE == MODE_FUSED && PR::kShift) {
        es_collide_dev<HwOps>(v, rest_density(rho0), fx, fy, fz, nuc, P, p);
    } else if (MODE == MODE_FUSED) {
        T m[kQ];
        es_moments<T, D>(v, m);
        es_collide<T, D>(m, fx, fy, fz, nuc, P, p);
    } else {
        es_collide<T, D>(v, fx, fy, fz, nuc, P, p);
    }
    if (P.use_les) store_nu<PR>(Nu, n, nuc);
#pragma unroll
    for (int d = 0; d < kQ; d++) {
        if constexpr (PR::kShift && MODE == MODE_FUSED) store_dev<PR>(dst, qaddr(g, qn, d), d, p[d]);
        else store_pop<PR>(dst, qaddr(g, qn, d), d, p[d], rho0);
    }
}

template <typename PR, int MODE>
__global__ __launch_bounds__(kRowBlock) void k_simple(const typename PR::S* src, typename PR::S* dst,
                                                   typename PR::T* mout, const typename PR::T* __restrict__ F,
                                                   typename PR::N* __restrict__ Nu,
                                                   const uint64_t* __restrict__ fmask, Grid g,
                                                   CollideParams<typename PR::T> P, uint32_t nkb, float rho0) {
    const RowBlock rb = row_block(g, blockIdx.x, nkb, blockDim.x);
    const int k = rb.k0 + (int)threadIdx.x;
    if (k > g.zg1) return;
    simple_cell<PR, MODE>(src, dst, mout, F, Nu, fmask, g, P, rho0, rb.i, rb.j, k);
}

template <typename PR>
__global__ __launch_bounds__(kFlatBlock) void k_simple_flat(const typename PR::S* src, typename PR::S* dst,
                                                            const typename PR::T* __restrict__ F,
                                                            typename PR::N* __restrict__ Nu,
                                                            const uint64_t* __restrict__ fmask, Grid g,
                                                            CollideParams<typename PR::T> P, FlatTile tile, float rho0) {
    int i, j, k;
    if (!flat_cell(g, tile, i, j, k)) return;
    simple_cell<PR, MODE_FUSED>(src, dst, nullptr, F, Nu, fmask, g, P, rho0, i, j, k);
}

// ------------------------------------------------------------------ data movement on every cell

// push: dst[c][d] = src[c-e_d][d] if c-e_d is interior, else src[c][d] (all cells)
template <typename W>
__global__ void k_push_all(const W* __restrict__ src, W* __restrict__ dst, Grid g) {
    for (uint64_t n = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; n < g.size;
         n += (uint64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        decode_cell(g, n, i, j, k);
        const uint32_t qc = qcell(g, i, j, k);
#pragma unroll
        for (int d = 0; d < kQ; d++) {
            const int si = i - dir_x(d), sj = j - dir_y(d), sk = k - dir_z(d);
            const uint32_t s = is_interior(g, si, sj, sk) ? qcell(g, si, sj, sk) : qc;
            dst[qaddr(g, qc, d)] = src[qaddr(g, s, d)];
        }
    }
}

// pull: interior dst[c][d] = src[c-e_d][d]; ghosts copied
template <typename W>
__global__ void k_pull_all(const W* __restrict__ src, W* __restrict__ dst, Grid g) {
    for (uint64_t n = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; n < g.size;
         n += (uint64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        decode_cell(g, n, i, j, k);
        const bool in = is_interior(g, i, j, k);
        const uint32_t qc = qcell(g, i, j, k);
#pragma unroll
        for (int d = 0; d < kQ; d++) {
            const uint32_t s = in ? qcell(g, i - dir_x(d), j - dir_y(d), k - dir_z(d)) : qc;
            dst[qaddr(g, qc, d)] = src[qaddr(g, s, d)];
        }
    }
}

// The bounce-back, in place, in one launch: ghost slot d (5 inward directions) of a
// face cell takes slot opp(d) of the neighbour g+e_d, and the 12 edge lines theirs
// (Boundary.hpp:41-132: on an edge the one direction pointing inward on both
// boundary axes).  The reference's faces follow one another (i, j, k), and at a rim a
// face reads a ghost cell of another: of a later face its old value, while the later
// face would read back the very value that the earlier one took from it, so it keeps
// its own and nothing that is read is written.  Six faces and the edges as launches
// of their own took 23 us a call at 60^3, this one 5.
template <typename W>
__global__ void k_bounce_back(W* __restrict__ Q, Grid g) {
    const uint64_t fi = (uint64_t)g.yg1 * g.zg1, fj = (uint64_t)g.xg1 * g.zg1, fk = (uint64_t)g.xg1 * g.yg1;
    const uint64_t faces = 2 * (fi + fj + fk);
    const int nmax = max(g.xg1, max(g.yg1, g.zg1));
    const int X0 = g.xg1 + 1, Y0 = g.yg1 + 1, Z0 = g.zg1 + 1;
    for (uint64_t u = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; u < faces + 12ull * nmax;
         u += (uint64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        if (u < faces) {
            const int axis = u < 2 * fi ? 0 : u < 2 * (fi + fj) ? 1 : 2;  // 0 i, 1 j, 2 k
            const uint64_t per = axis == 0 ? fi : axis == 1 ? fj : fk;
            uint64_t t = u - (axis == 0 ? 0 : axis == 1 ? 2 * fi : 2 * (fi + fj));
            const bool far = t >= per;
            if (far) t -= per;
            const int inward = far ? -1 : 1;
            const int nb = axis == 2 ? g.yg1 : g.zg1;  // second free axis extent
            const int a = (int)(t / nb) + 1, b = (int)(t % nb) + 1;
            if (axis == 0) { i = far ? X0 : 0; j = a; k = b; }
            else if (axis == 1) { i = a; j = far ? Y0 : 0; k = b; }
            else { i = a; j = b; k = far ? Z0 : 0; }
            const uint32_t c = qcell(g, i, j, k);
#pragma unroll
            for (int d = 0; d < kQ; d++) {
                const int comp = axis == 0 ? dir_x(d) : axis == 1 ? dir_y(d) : dir_z(d);
                if (comp != inward) continue;
                const int i2 = i + dir_x(d), j2 = j + dir_y(d), k2 = k + dir_z(d);
                if (axis > 0 && (i2 == 0 || i2 == X0)) continue;
                if (axis > 1 && (j2 == 0 || j2 == Y0)) continue;
                Q[qaddr(g, c, d)] = Q[qaddr(g, qcell(g, i2, j2, k2), opposite(d))];
            }
            continue;
        }
        const uint64_t t = u - faces;
        const int line = (int)(t / nmax), s = (int)(t % nmax) + 1;
        int d;
        switch (line) {
            case 0: i = 0; j = 0; k = s; d = Q07; break;
            case 1: i = X0; j = 0; k = s; d = Q14; break;
            case 2: i = 0; j = Y0; k = s; d = Q13; break;
            case 3: i = X0; j = Y0; k = s; d = Q08; break;
            case 4: i = 0; k = 0; j = s; d = Q09; break;
            case 5: i = 0; k = Z0; j = s; d = Q15; break;
            case 6: i = X0; k = Z0; j = s; d = Q10; break;
            case 7: i = X0; k = 0; j = s; d = Q16; break;
            case 8: j = 0; k = 0; i = s; d = Q11; break;
            case 9: j = 0; k = Z0; i = s; d = Q17; break;
            case 10: j = Y0; k = Z0; i = s; d = Q12; break;
            default: j = Y0; k = 0; i = s; d = Q18; break;
        }
        const int lim = line < 4 ? g.zg1 : line < 8 ? g.yg1 : g.xg1;
        if (s > lim) continue;
        const uint32_t c = qcell(g, i, j, k);
        const uint32_t src = qcell(g, i + dir_x(d), j + dir_y(d), k + dir_z(d));
        Q[qaddr(g, c, d)] = Q[qaddr(g, src, opposite(d))];
    }
}

// Ghost cells enumerated face by face without repeats:
// i = 0 and i = xg0 planes, then j = 0 / yg0 with 1 <= i <= xg1, then k = 0 / zg0
// with 1 <= i <= xg1, 1 <= j <= yg1.
__device__ __forceinline__ bool ghost_cell(const Grid& g, uint64_t t, int& i, int& j, int& k) {
    const uint64_t A = (uint64_t)g.yz;                       // one i-plane
    const uint64_t B = (uint64_t)g.xg1 * g.zg;               // one j-plane without i ghosts
    const uint64_t C = (uint64_t)g.xg1 * g.yg1;              // one k-plane without i, j ghosts
    if (t < 2 * A) {
        i = t < A ? 0 : g.xg1 + 1;
        const uint64_t r = t % A;
        j = (int)(r / g.zg);
        k = (int)(r % g.zg);
        return true;
    }
    t -= 2 * A;
    if (t < 2 * B) {
        j = t < B ? 0 : g.yg1 + 1;
        const uint64_t r = t % B;
        i = (int)(r / g.zg) + 1;
        k = (int)(r % g.zg);
        return true;
    }
    t -= 2 * B;
    if (t < 2 * C) {
        k = t < C ? 0 : g.zg1 + 1;
        const uint64_t r = t % C;
        i = (int)(r / g.yg1) + 1;
        j = (int)(r % g.yg1) + 1;
        return true;
    }
    return false;
}
__host__ __device__ inline uint64_t ghost_count(const Grid& g) {
    return 2ull * g.yz + 2ull * (uint64_t)g.xg1 * g.zg + 2ull * (uint64_t)g.xg1 * g.yg1;
}

// Ghost slots the reference rewrites every step from interior values: the push
// into the ghost layer (c-e_d interior) and the bounce-back slots whose source
// g+e_d is interior.  Rim bounce-back slots (ghost source) and never-written
// slots are left as they are in dst.
template <typename PR>
__global__ void k_ghost_fill(const typename PR::S* __restrict__ src, typename PR::T* __restrict__ dst, Grid g,
                             float rho0) {
    const uint64_t total = ghost_count(g);
    for (uint64_t t = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; t < total;
         t += (uint64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        if (!ghost_cell(g, t, i, j, k)) continue;
        const int bi = (i == 0) ? 1 : (i == g.xg1 + 1) ? -1 : 0;  // inward sign per boundary axis
        const int bj = (j == 0) ? 1 : (j == g.yg1 + 1) ? -1 : 0;
        const int bk = (k == 0) ? 1 : (k == g.zg1 + 1) ? -1 : 0;
        const int nb = (bi != 0) + (bj != 0) + (bk != 0);
        const uint32_t c = qcell(g, i, j, k);
#pragma unroll
        for (int d = 0; d < kQ; d++) {
            const int ex = dir_x(d), ey = dir_y(d), ez = dir_z(d);
            const int si = i - ex, sj = j - ey, sk = k - ez;
            if (is_interior(g, si, sj, sk)) {
                dst[qaddr(g, c, d)] = load_pop<PR>(src, qaddr(g, qcell(g, si, sj, sk), d), d, rho0);
                continue;
            }
            bool bb = false;
            if (nb == 1) {
                bb = (bi != 0 && ex == bi) || (bj != 0 && ey == bj) || (bk != 0 && ez == bk);
            } else if (nb == 2) {
                bb = (bi == 0 || ex == bi) && (bj == 0 || ey == bj) && (bk == 0 || ez == bk) &&
                     (bi != 0 || ex == 0) && (bj != 0 || ey == 0) && (bk != 0 || ez == 0);
            }
            if (!bb) continue;
            const int ti = i + ex, tj = j + ey, tk = k + ez;
            if (!is_interior(g, ti, tj, tk)) continue;
            // opp(d) has the rest weight of d
            dst[qaddr(g, c, d)] = load_pop<PR>(src, qaddr(g, qcell(g, ti, tj, tk), opposite(d)), d, rho0);
        }
    }
}

template <typename W>
__global__ void k_ghost_copy(const W* __restrict__ src, W* __restrict__ dst, Grid g) {
    const uint64_t total = ghost_count(g);
    for (uint64_t t = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; t < total;
         t += (uint64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        if (!ghost_cell(g, t, i, j, k)) continue;
        const uint32_t c = qcell(g, i, j, k);
#pragma unroll
        for (int d = 0; d < kQ; d++) dst[qaddr(g, c, d)] = src[qaddr(g, c, d)];
    }
}

// ------------------------------------------------------------------ F occupancy
// Bit per cell: any component of F[c] with a non-zero bit pattern.  gmask gets
// the ghost cells only.
template <typename T>
__global__ void k_mask_from_f(const T* __restrict__ F, uint64_t* __restrict__ mask, uint64_t* __restrict__ gmask,
                              Grid g) {
    const uint64_t words = (uint64_t)g.xg * g.yg * g.mask_w;
    for (uint64_t w = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; w < words;
         w += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t row = w / g.mask_w;
        const int kb = (int)(w % g.mask_w) * 64;
        const int i = (int)(row / g.yg), j = (int)(row % g.yg);
        uint64_t bits = 0, gbits = 0;
        for (int t = 0; t < 64; t++) {
            const int k = kb + t;
            if (k >= g.zg) break;
            const uint64_t n = cell_index(g, i, j, k);
            const T fx = F[3 * n], fy = F[3 * n + 1], fz = F[3 * n + 2];
            const bool nz = fx != T(0) || fy != T(0) || fz != T(0) || signbit(fx) || signbit(fy) || signbit(fz);
            if (nz) {
                bits |= 1ull << t;
                if (!is_interior(g, i, j, k)) gbits |= 1ull << t;
            }
        }
        mask[w] = bits;
        gmask[w] = gbits;
    }
}

// F of cells [begin, end) as the reference holds it: the stored value where the bit is set, else 0.
template <typename T>
__global__ void k_masked_f(const T* __restrict__ F, const uint64_t* __restrict__ mask, uint64_t begin, uint64_t end,
                           T* __restrict__ out, Grid g) {
    for (uint64_t n = begin + blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; n < end;
         n += (uint64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        decode_cell(g, n, i, j, k);
        const bool on = mask_test(mask, g, i, j, k);
        const uint64_t o = 3 * (n - begin);
        out[o + 0] = on ? F[3 * n + 0] : T(0);
        out[o + 1] = on ? F[3 * n + 1] : T(0);
        out[o + 2] = on ? F[3 * n + 2] : T(0);
    }
}

__global__ void k_zero_interior_o(uint8_t* __restrict__ O, Grid g) {
    for (uint64_t n = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; n < g.size;
         n += (uint64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        decode_cell(g, n, i, j, k);
        if (is_interior(g, i, j, k)) O[n] = 0;
    }
}

// ------------------------------------------------------------------ IB forcing
__device__ __forceinline__ int wrap_ik(int a, int a1) {  // Forcing.hpp:85-88
    if (a == 0) return a1;
    if (a == a1 + 1) return 1;
    return a;
}

// Before a forcing pass: F of a stencil cell that was not occupied after the
// previous pass is zero in the reference (F=0 where O==0), so clear it here,
// and mark the cell in the new occupancy mask.
template <typename T>
__device__ __forceinline__ void prepare_point(const PointsDev& p, int64_t q, T* __restrict__ F,
                                              const uint64_t* __restrict__ prev, uint64_t* __restrict__ next,
                                              const Grid& g) {
    const int pi = p.i[q], pj = p.j[q], pk = p.k[q];
    for (int k1 = -1; k1 <= 1; k1++)
        for (int i1 = -1; i1 <= 1; i1++) {
            const int i2 = wrap_ik(pi + i1, g.xg1), k2 = wrap_ik(pk + k1, g.zg1);
            const uint64_t c = cell_index(g, i2, pj, k2);
            if (!mask_test(prev, g, i2, pj, k2)) {
                F[3 * c + 0] = T(0);
                F[3 * c + 1] = T(0);
                F[3 * c + 2] = T(0);
            }
            atomicOr((unsigned long long*)&next[mask_word_index(g, i2, pj, k2)], 1ull << (k2 & 63));
        }
}

template <typename T>
__global__ void k_force_prepare(PointsDev p, int64_t begin, int64_t count, T* __restrict__ F,
                                const uint64_t* __restrict__ prev, uint64_t* __restrict__ next, Grid g) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= count) return;
    prepare_point(p, begin + t, F, prev, next, g);
}

// density and momentum of cell (i,j,k) as the reference's moments() would leave them; 1 <= k <= zg1 for Esotwist,
// whose homes are found by the pitches of the interior rows
template <typename PR, int STREAM, int MOMSRC, int EVEN>
__device__ __forceinline__ void cell_rho_j(const typename PR::S* __restrict__ Q, const Grid& g, int i, int j, int k,
                                           typename PR::T& rho, typename PR::T& jx, typename PR::T& jy,
                                           typename PR::T& jz, float rho0) {
    using T = typename PR::T;
    const uint32_t n = qcell(g, i, j, k);
    if (STREAM == StreamEsotwist) {
        const int32_t di = (i == g.xg1) ? -(int32_t)((uint32_t)(g.xg1 - 1) * g.qyz) : (int32_t)g.qyz;
        const int32_t dj = (j == g.yg1) ? -(int32_t)((uint32_t)(g.yg1 - 1) * g.qz) : (int32_t)g.qz;
        const int32_t dk = (k == g.zg1) ? -(g.zg1 - 1) : 1;
        if (MOMSRC == MOMSRC_STORED) {
            T m[4];
#pragma unroll
            for (int d = 0; d < 4; d++) {
                const uint32_t h = n + (uint32_t)((twist_dx(d) ? di : 0) + (twist_dy(d) ? dj : 0) + (twist_dz(d) ? dk : 0));
                m[d] = (T)Q[qaddr(g, h, EVEN ? d : opposite(d))];
            }
            rho = m[0]; jx = m[1]; jy = m[2]; jz = m[3];
        } else {
            T f[kQ];
#pragma unroll
            for (int d = 0; d < kQ; d++) {
                const uint32_t h = n + (uint32_t)((twist_dx(d) ? di : 0) + (twist_dy(d) ? dj : 0) + (twist_dz(d) ? dk : 0));
                f[d] = load_pop<PR>(Q, qaddr(g, h, EVEN ? d : opposite(d)), d, rho0);
            }
            es_rho_j(f, rho, jx, jy, jz);
        }
    } else {
        if (MOMSRC == MOMSRC_STORED) {
            rho = (T)Q[qaddr(g, n, 0)];
            jx = (T)Q[qaddr(g, n, 1)];
            jy = (T)Q[qaddr(g, n, 2)];
            jz = (T)Q[qaddr(g, n, 3)];
        } else {
            const bool im = i >= 2, ip = i <= g.xg1 - 1;
            const bool jm = j >= 2, jp = j <= g.yg1 - 1;
            const bool km = k >= 2, kp = k <= g.zg1 - 1;
            T f[kQ];
#pragma unroll
            for (int d = 0; d < kQ; d++) {
                const int ex = dir_x(d), ey = dir_y(d), ez = dir_z(d);
                const bool ok = (ex > 0 ? im : ex < 0 ? ip : true) && (ey > 0 ? jm : ey < 0 ? jp : true) &&
                                (ez > 0 ? km : ez < 0 ? kp : true);
                const int32_t off = -(ex * (int32_t)g.qyz + ey * (int32_t)g.qz + ez);
                f[d] = load_pop<PR>(Q, qaddr(g, ok ? n + (uint32_t)off : n, d), d, rho0);
            }
            es_rho_j(f, rho, jx, jy, jz);
        }
    }
}

// Density and momentum of a cell, or the three force components (the fourth unused).
template <typename T>
struct alignas(4 * sizeof(T)) Mom4 {
    T r, x, y, z;
};

// ------------------------------------------------------------------ IB forcing of a list
// The per-call forcing (any list, in its order) in two launches.  k_list_unpack
// spreads the caller's points into arrays and starts the next occupancy mask.
// k_list_planes takes a j plane per workgroup: points of different planes never
// share a cell.  It collects the plane's points in list order, prepares their cells
// and then runs rounds over the first unfinished ones, one a lane: each marks its
// nine cells with the lowest position that wants them (atomicMin), and those that
// hold all their cells run the reference's gather / correct / spread
// (Forcing.hpp:73-135) and make room for the next.  They share no cell, and no
// earlier point is unfinished on theirs, so every cell sees its points in list
// order.  The rounds are bound by the latency of a point's loads.  A call over the
// 13,431 points of a 60^3 tank: 0.12 to 0.28 ms, the kernel 77 us of them (115 with
// the points' moments read when they run); with levels from a hash map on the host
// and a launch per level 8.5 ms.
template <typename T>
__global__ void k_list_unpack(const tdlb_ib_point* __restrict__ in, int64_t n, int ghost, PointsDev p,
                              const uint64_t* __restrict__ base, uint64_t* __restrict__ next, uint64_t words) {
    for (uint64_t t = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; t < max((uint64_t)n, words);
         t += (uint64_t)gridDim.x * blockDim.x) {
        if (t < words) next[t] = base[t];
        if (t >= (uint64_t)n) continue;
        const tdlb_ib_point q = in[t];
        p.i[t] = (int32_t)(q.i + ghost);
        p.j[t] = (int32_t)(q.j + ghost);
        p.k[t] = (int32_t)(q.k + ghost);
        static_cast<T*>(p.ifrac)[t] = (T)q.i_frac;
        static_cast<T*>(p.kfrac)[t] = (T)q.k_frac;
        static_cast<T*>(p.u)[t] = (T)q.u_delta;
        static_cast<T*>(p.v)[t] = (T)q.v_delta;
        static_cast<T*>(p.w)[t] = (T)q.w_delta;
    }
}

// A point in a lane's registers with everything the forcing does not change: the
// moments of its nine cells are asked for when the lane takes it, rounds before use.
template <typename T>
struct ListPoint {
    T wx[3], wz[3], vel[3];
    T rho[9], jx[9], jy[9], jz[9];
    uint32_t at[9];  // cell indices
};

template <typename PR, int STREAM, int EVEN>
__device__ __forceinline__ void list_take(ListPoint<typename PR::T>& a, const PointsDev& p, int64_t q, int pi, int pk,
                                          int pj, const typename PR::S* __restrict__ Q, const Grid& g, float rho0) {
    using T = typename PR::T;
    const T ifr = static_cast<const T*>(p.ifrac)[q], kfr = static_cast<const T*>(p.kfrac)[q];
    a.vel[0] = static_cast<const T*>(p.u)[q];
    a.vel[1] = static_cast<const T*>(p.v)[q];
    a.vel[2] = static_cast<const T*>(p.w)[q];
#pragma unroll
    for (int s = 0; s < 9; s++) {
        const int i2 = wrap_ik(pi + s % 3 - 1, g.xg1), k2 = wrap_ik(pk + s / 3 - 1, g.zg1);
        a.at[s] = cell_index(g, i2, pj, k2);
        cell_rho_j<PR, STREAM, MOMSRC_STORED, EVEN>(Q, g, i2, pj, k2, a.rho[s], a.jx[s], a.jy[s], a.jz[s], rho0);
    }
#pragma unroll
    for (int b = 0; b < 3; b++) {
        a.wx[b] = ib_weight<T>(-ifr + T(b - 1));
        a.wz[b] = ib_weight<T>(-kfr + T(b - 1));
    }
}

// gather, correct and spread of a point, all nine cells by one lane
template <typename PR>
__device__ __forceinline__ void list_point(const ListPoint<typename PR::T>& a, typename PR::T* __restrict__ F,
                                           typename PR::T alfa, typename PR::T beta, bool meets) {
    using T = typename PR::T;
    using D = typename PR::D;
    T f[9][3];
#pragma unroll
    for (int s = 0; s < 9; s++)
#pragma unroll
        for (int d = 0; d < 3; d++) f[s][d] = F[3 * (uint64_t)a.at[s] + d];
    T rhoSum = T(0.0), xSum = T(0.0), ySum = T(0.0), zSum = T(0.0);
#pragma unroll
    for (int s = 0; s < 9; s++) {
        const T ppp = a.wx[s % 3] * a.wz[s / 3];
        const T xx = (T)((D)a.jx[s] + D(0.5) * (D)f[s][0]);
        const T yy = (T)((D)a.jy[s] + D(0.5) * (D)f[s][1]);
        const T zz = (T)((D)a.jz[s] + D(0.5) * (D)f[s][2]);
        rhoSum += ppp * a.rho[s];
        xSum += ppp * xx;
        ySum += ppp * yy;
        zSum += ppp * zz;
    }
    xSum -= rhoSum * a.vel[0];
    ySum -= rhoSum * a.vel[1];
    zSum -= rhoSum * a.vel[2];
    // meets: below 3 interior cells a stencil meets itself, one cell after the other
#pragma unroll
    for (int s = 0; s < 9; s++) {
        T* const c = F + 3 * (uint64_t)a.at[s];
        const T bp = beta * (a.wx[s % 3] * a.wz[s / 3]);
        if (meets)
#pragma unroll
            for (int d = 0; d < 3; d++) f[s][d] = c[d];
        c[0] = alfa * f[s][0] - bp * xSum;
        c[1] = alfa * f[s][1] - bp * ySum;
        c[2] = alfa * f[s][2] - bp * zSum;
    }
}

constexpr int kListBlock = 512, kListRun = 8;  // lanes, and points a lane looks at between two barriers
constexpr uint32_t kNoPoint = 0xffffffffu;
struct ListShared {
    int64_t less[kListBlock / 64];
    int same[kListBlock / 64];
    int wave[2][kListRun][kListBlock / 64];
};
// The points of plane j (pj: the planes of all n) to their part of list, in list order, by the whole workgroup;
// returns their number, mine their part.  A barrier is needed before they are read.
__device__ __forceinline__ uint32_t plane_points(const int32_t* __restrict__ pj, int64_t n, int j,
                                                 int64_t* __restrict__ list, int64_t*& mine, ListShared& sh) {
    constexpr int kWaves = kListBlock / 64;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // the plane's part of the list begins after the points of lower planes
    int64_t less = 0;
    int same = 0;  // of a lane: whether the plane has points
#pragma unroll 8
    for (int64_t q = tid; q < n; q += kListBlock) {
        less += pj[q] < j ? 1 : 0;
        same |= pj[q] == j ? 1 : 0;
    }
    for (int o = 32; o > 0; o >>= 1) less += __shfl_down(less, o, 64);
    const bool any = __ballot(same) != 0;
    if (lane == 0) {
        sh.less[wave] = less;
        sh.same[wave] = any ? 1 : 0;
    }
    __syncthreads();
    int64_t first = 0;
    int points = 0;
    for (int w = 0; w < kWaves; w++) {
        first += sh.less[w];
        points |= sh.same[w];
    }
    mine = list + first;
    if (__builtin_amdgcn_readfirstlane(points) == 0) return 0;  // the same for every lane of every wave
    // its points in list order
    uint32_t count = 0;
    int turn = 0;
    for (int64_t q0 = 0; q0 < n; q0 += kListBlock * kListRun, turn ^= 1) {
        int at_j[kListRun];
        uint64_t vote[kListRun];
#pragma unroll
        for (int u = 0; u < kListRun; u++) {
            const int64_t q = q0 + u * kListBlock + tid;
            at_j[u] = q < n ? pj[q] : 0;
        }
#pragma unroll
        for (int u = 0; u < kListRun; u++) {
            vote[u] = __ballot(at_j[u] == j);
            if (lane == 0) sh.wave[turn][u][wave] = __popcll(vote[u]);
        }
        __syncthreads();  // the last reader of sh.wave[turn] has passed the turn between
#pragma unroll
        for (int u = 0; u < kListRun; u++) {
            uint32_t at = count;
#pragma unroll
            for (int w = 0; w < kWaves; w++) {
                at += w < wave ? sh.wave[turn][u][w] : 0;
                count += sh.wave[turn][u][w];
            }
            if (at_j[u] == j) mine[at + __popcll(vote[u] & ((1ull << lane) - 1ull))] = q0 + u * kListBlock + tid;
        }
    }
    return count;
}

// The marks of a plane's cells, in LDS or, where it does not hold them, in HBM: there a
// mark may sit in this CU's L1 from the round before and is read where the atomics put it.
template <bool LDS>
struct Marks {
    uint32_t* p;
    __device__ __forceinline__ void clear(int c) const { p[c] = kNoPoint; }
    __device__ __forceinline__ void lower(int c, uint32_t t) const { atomicMin(p + c, t); }
    __device__ __forceinline__ uint32_t get(int c) const {
        return LDS ? p[c] : __hip_atomic_load(p + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};
// a stencil's nine cells in a plane's own (i, k) order
__device__ __forceinline__ void plane_cells(int (&cells)[9], int pi, int pk, const Grid& g) {
#pragma unroll
    for (int s = 0; s < 9; s++)
        cells[s] = (wrap_ik(pi + s % 3 - 1, g.xg1) - 1) * g.zg1 + wrap_ik(pk + s / 3 - 1, g.zg1) - 1;
}

// Levels of a list within its planes, one more than the highest level of an earlier
// point that shares a stencil cell: the round in which a point holds all its cells when
// every unfinished point of the plane marks.  list, marks_hbm as in k_list_planes.
template <bool MARKS_LDS>
__global__ __launch_bounds__(kListBlock) void k_list_levels(PointsDev p, int64_t n, int64_t* __restrict__ list,
                                                            uint32_t* __restrict__ marks_hbm, int32_t* __restrict__ lev,
                                                            Grid g) {
    extern __shared__ uint32_t list_lds[];
    __shared__ ListShared s_list;
    __shared__ uint32_t s_done;
    const int tid = (int)threadIdx.x;
    const int plane = g.xg1 * g.zg1;
    const Marks<MARKS_LDS> marks{MARKS_LDS ? list_lds : marks_hbm + (uint64_t)blockIdx.x * plane};
    for (int c = tid; c < plane; c += kListBlock) marks.clear(c);
    for (int j = 1 + (int)blockIdx.x; j <= g.yg1; j += (int)gridDim.x) {
        int64_t* mine;
        const uint32_t count = plane_points(p.j, n, j, list, mine, s_list);
        if (tid == 0) s_done = 0;
        __syncthreads();
        int32_t round = 0;
        for (uint32_t done = 0; done < count; round++) {
            int cells[9];
            for (uint32_t t = tid; t < count; t += kListBlock) {
                const int64_t q = mine[t];
                if (q < 0) continue;
                plane_cells(cells, p.i[q], p.k[q], g);
#pragma unroll
                for (int s = 0; s < 9; s++) marks.lower(cells[s], t);
            }
            __syncthreads();
            uint32_t ended = 0;
            for (uint32_t t = tid; t < count; t += kListBlock) {
                const int64_t q = mine[t];
                if (q < 0) continue;
                plane_cells(cells, p.i[q], p.k[q], g);
                bool ready = true;
#pragma unroll
                for (int s = 0; s < 9; s++) ready = marks.get(cells[s]) == t && ready;
                if (!ready) continue;
                lev[q] = round;
                mine[t] = -1 - q;
                ended++;
            }
            if (ended) atomicAdd(&s_done, ended);
            __syncthreads();
            for (uint32_t t = tid; t < count; t += kListBlock) {
                const int64_t q = mine[t];
                const int64_t a = q < 0 ? -1 - q : q;
                plane_cells(cells, p.i[a], p.k[a], g);
#pragma unroll
                for (int s = 0; s < 9; s++) marks.clear(cells[s]);
            }
            done = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_done);
            __syncthreads();
        }
    }
}

// list: n positions, the planes' points one plane after the other.  marks_hbm: a
// plane of marks per workgroup where the LDS does not hold one.
template <typename PR, int STREAM, int EVEN, bool MARKS_LDS>
__global__ __launch_bounds__(kListBlock) void k_list_planes(PointsDev p, int64_t n, int64_t* __restrict__ list,
                                                            uint32_t* __restrict__ marks_hbm,
                                                            typename PR::T* __restrict__ F,
                                                            const typename PR::S* __restrict__ Q,
                                                            const uint64_t* __restrict__ prev,
                                                            uint64_t* __restrict__ next, Grid g,
                                                            typename PR::T alfa, typename PR::T beta, float rho0) {
    extern __shared__ uint32_t list_lds[];
    __shared__ ListShared s_list;
    __shared__ uint32_t s_next, s_done;
    const int tid = (int)threadIdx.x;
    const int plane = g.xg1 * g.zg1;
    const Marks<MARKS_LDS> marks{MARKS_LDS ? list_lds : marks_hbm + (uint64_t)blockIdx.x * plane};
    for (int c = tid; c < plane; c += kListBlock) marks.clear(c);
    for (int j = 1 + (int)blockIdx.x; j <= g.yg1; j += (int)gridDim.x) {
        int64_t* mine;
        const uint32_t count = plane_points(p.j, n, j, list, mine, s_list);
        if (tid == 0) {
            s_next = kListBlock;
            s_done = 0;
        }
        __syncthreads();
        for (uint32_t t = tid; t < count; t += kListBlock) prepare_point(p, mine[t], F, prev, next, g);
        // the lanes hold a prefix of the plane's list: a lane that finishes its point takes the next
        uint32_t t = tid;
        bool have = t < count;
        ListPoint<typename PR::T> a;
        int cells[9];
        auto take = [&] {
            const int64_t q = mine[t];
            const int pi = p.i[q], pk = p.k[q];
            list_take<PR, STREAM, EVEN>(a, p, q, pi, pk, j, Q, g, rho0);
            plane_cells(cells, pi, pk, g);
        };
        if (have) take();
        __syncthreads();
        // One barrier ends a turn for every lane, so the loop has one way back: with a
        // lane's take() as a second one the compiler made a loop of its own of it, and
        // the barriers of a wavefront's lanes parted.
        for (uint32_t done = 0; done < count;) {
            if (have)
#pragma unroll
                for (int s = 0; s < 9; s++) marks.lower(cells[s], t);
            __syncthreads();
            bool ready = have;
            if (have)
#pragma unroll
                for (int s = 0; s < 9; s++) ready = marks.get(cells[s]) == t && ready;
            __syncthreads();
            if (have)
#pragma unroll
                for (int s = 0; s < 9; s++) marks.clear(cells[s]);
            if (ready) {
                list_point<PR>(a, F, alfa, beta, g.xg1 < 3 || g.zg1 < 3);
                atomicAdd(&s_done, 1u);
                t = atomicAdd(&s_next, 1u);
                have = t < count;
                if (have) take();
            }
            __syncthreads();
            done = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_done);  // changes two barriers from here
        }
    }
}

// ------------------------------------------------------------------ IB forcing by planes
// A bound tank's forcing pass in two launches (ForceGeom in kernels.h).  The
// gather (force_gather) spreads over the whole chip: it generates the step's
// blade points and their stencil rows, starts the next occupancy mask from the
// static bits, clears F of blade cells missing from the previous mask
// (prepare_point), and writes density and momentum of every static and blade
// stencil cell to their caches.  It is bound by the lines of its scattered
// population reads.  The levels (plane_levels) are one workgroup per j plane,
// the sequential list order of Forcing.hpp:73-135 within the plane: static
// levels, then blade levels, passes of a point per quad of lanes with a barrier
// after every level, bound by the latency of that chain.  Gathering inside the
// plane's workgroup instead leaves the gather to one CU per plane (96 of 256 CUs at
// 96^3) and, beyond 256 planes, to rounds of workgroups, and a plane with many points
// then needs several workgroups meeting at barriers in HBM.  Whole pass, that form ->
// this: 24^3 252 -> 27 us, 36^3 69 -> 23, 60^3 Simple 80 -> 25, 96^3 91 -> 30, 131^3 FP16
// 94 -> 40, 192^3 FP64 274 -> 126, 256^3 290 -> 158, 512^3 633 -> 547 (gather 379: 1.63 GB
// read and 0.07 written, 4.5 TB/s; levels 166).

// ---- A point of a plane task on a quad of lanes: lane c = 0..2 of the quad
// takes stencil row k1 = c - 1 (cells s = 3c + m for i1 = m - 1), lane 3 repeats
// row 2 and writes nothing.  Everything of the row that does not depend on the
// flow is in its ForceRow (weights, wall velocity, stencil entries), laid out
// once for the static points and once a step for the blades, so a pass is two
// 16-byte loads, the gather, the sums and the spread.  The nine terms are added
// in the reference's order (s = 0..8) by every lane, each term taken from its
// lane of the quad as a DPP operand of the add: no LDS traffic and no latency
// beyond the add's own.  A level is a chain (gather, sums, spread, barrier) of a
// few hundred lanes, bound by latency: three lanes per point with LDS shuffles
// and the weights' FP64 square roots in every pass took about 9 us a level,
// this form 0.5 us with the plane in LDS.
template <int C>
__device__ __forceinline__ float quad_lane(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), C * 0x55, 0xf, 0xf, true));
}
template <int C>
__device__ __forceinline__ double quad_lane(double x) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(x), C * 0x55, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(x), C * 0x55, 0xf, 0xf, true));
}
template <int C, typename T>
__device__ __forceinline__ void quad_add(T& sum, const T (&t)[3]) {
#pragma unroll
    for (int m = 0; m < 3; m++) sum += quad_lane<C>(t[m]);
}
template <typename T>
__device__ __forceinline__ T quad_sum(const T (&t)[3]) {
    T sum = T(0.0);
    quad_add<0>(sum, t);
    quad_add<1>(sum, t);
    quad_add<2>(sum, t);
    return sum;
}
// j + 0.5 F rounded once, which is what the reference's double sum rounded to T
// gives: exact for T = double, and for T = float a sum of two floats rounded
// first to 53 and then to 24 bits is the correctly rounded sum (53 >= 2 * 24 + 2)
__device__ __forceinline__ float add_half(float j, float f) { return fmaf(0.5f, f, j); }
__device__ __forceinline__ double add_half(double j, double f) { return j + 0.5 * f; }

// the row's nine terms, the point's sums and the row's new force values (f in place)
template <typename T>
__device__ __forceinline__ void force_row(const ForceRow<T>& r, const Mom4<T> (&mo)[3], T (&f)[3][3], T alfa, T beta) {
    T tr[3], tx[3], ty[3], tz[3];
#pragma unroll
    for (int m = 0; m < 3; m++) tr[m] = r.w[m] * mo[m].r;
    const T rho = quad_sum(tr);
#pragma unroll
    for (int m = 0; m < 3; m++) {
        tx[m] = r.w[m] * add_half(mo[m].x, f[m][0]);
        ty[m] = r.w[m] * add_half(mo[m].y, f[m][1]);
        tz[m] = r.w[m] * add_half(mo[m].z, f[m][2]);
    }
    T x = quad_sum(tx), y = quad_sum(ty), z = quad_sum(tz);
    x -= rho * quad_lane<0>(r.vel);
    y -= rho * quad_lane<1>(r.vel);
    z -= rho * quad_lane<2>(r.vel);
#pragma unroll
    for (int m = 0; m < 3; m++) {
        const T bp = beta * r.w[m];
        f[m][0] = alfa * f[m][0] - bp * x;
        f[m][1] = alfa * f[m][1] - bp * y;
        f[m][2] = alfa * f[m][2] - bp * z;
    }
}

// stencil row c of a point: weights as ib_weight gives them in the point's own
// precision, component c of its wall velocity
template <typename T>
__device__ __forceinline__ ForceRow<T> make_row(T ifr, T kfr, int c, T vel) {
    ForceRow<T> r;
    const T wk = ib_weight<T>(-kfr + T(c - 1));
#pragma unroll
    for (int m = 0; m < 3; m++) r.w[m] = ib_weight<T>(-ifr + T(m - 1)) * wk;
    r.vel = vel;
    r.pad = 0;
    return r;
}

// ForceRow of every static point: e[m] = the cell's entry in its plane's list
template <typename T>
__global__ void k_static_rows(PointsDev p, int64_t n, const int32_t* __restrict__ sidx, ForceRow<T>* __restrict__ rows) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= 3 * n) return;
    const int64_t q = t / 3;
    const int c = (int)(t - 3 * q);
    const T* vel = static_cast<const T*>(c == 0 ? p.u : c == 1 ? p.v : p.w);
    ForceRow<T> r = make_row<T>(static_cast<const T*>(p.ifrac)[q], static_cast<const T*>(p.kfrac)[q], c, vel[q]);
#pragma unroll
    for (int m = 0; m < 3; m++) r.e[m] = sidx[9 * q + 3 * c + m];
    rows[t] = r;
}

// Blade levels of a plane.  The generator's list is colour-major (rushton.h
// blade_decode): classes (blade colour, radial index mod 5) of points that never
// share a stencil cell.  Blades at least 3 sqrt(2) cells apart at the inner
// radius never share one either, so one level then takes all blades' points of a
// radial class (5 levels, merged); in smaller tanks a level is one class.
__device__ __forceinline__ BladeEnum blade_enum_of(const BladeLayout& bl) {
    BladeEnum e;
    e.n_blades = bl.n_blades;
    e.n_planes = bl.n_planes;
    e.n_radial = bl.n_radial;
    e.n_bcol = bl.n_bcol;
    return e;
}
// radial classes with points: no level of a plane is empty
__device__ __forceinline__ int radial_classes(const BladeLayout& bl) { return min(bl.n_radial, 5); }
// Blades dealt to `groups` in turn (blade b to group b mod groups): how many a group has and how many the
// groups before it have together.
struct BladeGroup {
    int n, before;
};
__device__ __forceinline__ BladeGroup blade_group(int n_blades, int groups, int g) {
    const int q = n_blades / groups, rem = n_blades - q * groups;
    return BladeGroup{q + (g < rem ? 1 : 0), g * q + min(g, rem)};
}
// radial points of the first m classes of a blade (index mod 5 below m)
__device__ __forceinline__ int radial_before(int n_radial, int m) { return n_radial / 5 * m + min(m, n_radial % 5); }
// points of levels 0..l on one plane
__device__ __forceinline__ int blade_level_end(const BladeLayout& bl, int l) {
    const int per = radial_classes(bl), g = l / per;
    const BladeGroup bg = blade_group(bl.n_blades, bl.merged ? 1 : bl.n_bcol, g);
    return bg.before * bl.n_radial + bg.n * radial_before(bl.n_radial, l - g * per + 1);
}
// list index of radial point r of blade b on blade plane bp
__device__ __forceinline__ int blade_index(const BladeEnum& e, int b, int r, int bp) {
    const int bi = b / e.n_bcol, rmod = r % 5;
    const BladeGroup bg = blade_group(e.n_blades, e.n_bcol, b - bi * e.n_bcol);
    // points per plane of the colours before the blade's, then of its colour's radial classes before rmod
    const int before = bg.before * e.n_radial + bg.n * radial_before(e.n_radial, rmod);
    return before * e.n_planes + (bi * e.n_planes + bp) * ((e.n_radial - rmod + 4) / 5) + r / 5;
}
// position of radial point r of blade b among the plane's points in level order
__device__ __forceinline__ int level_slot(const BladeLayout& bl, int b, int r) {
    const int groups = bl.merged ? 1 : bl.n_bcol, bi = b / groups, rmod = r % 5;
    const BladeGroup bg = blade_group(bl.n_blades, groups, b - bi * groups);
    return bg.before * bl.n_radial + bg.n * radial_before(bl.n_radial, rmod) +
           bi * ((bl.n_radial - rmod + 4) / 5) + r / 5;
}
// blade plane index of plane j and its blade levels (0: no blades)
__device__ __forceinline__ int blade_plane(const ForceGeom& fg, int j, int& nlev) {
    const BladeLayout& bl = fg.blade;
    const int bp = j - bl.ghost - bl.j_lo;
    nlev = (bl.n_blades > 0 && fg.n_rot > 0 && bp >= 0 && bp < bl.n_planes) ? blade_level_count(blade_enum_of(bl), bl.merged != 0) : 0;
    return bp;
}

// Static stencil cells [c0, c1) of fg.cells: density and momentum into the cache,
// thread t of `threads` taking c0 + t, c0 + t + threads, ...
template <typename PR, int STREAM, int MOMSRC, int EVEN>
__device__ __forceinline__ void gather_cells(const ForceGeom& fg, int64_t c0, int64_t c1, int64_t t,
                                             int64_t threads, const typename PR::S* __restrict__ Q, const Grid& g,
                                             float rho0) {
    auto* scache = static_cast<Mom4<typename PR::T>*>(fg.scache);
    for (int64_t e = c0 + t; e < c1; e += threads) {
        const uint32_t n = fg.cells[e];  // below 2^31: 32-bit divisions
        const int i = (int)(n / g.yz);
        const uint32_t r = n - (uint32_t)i * g.yz;
        const int j = (int)(r / (uint32_t)g.zg), k = (int)(r - (uint32_t)j * (uint32_t)g.zg);
        Mom4<typename PR::T> m;
        cell_rho_j<PR, STREAM, MOMSRC, EVEN>(Q, g, i, j, k, m.r, m.x, m.y, m.z, rho0);
        scache[e] = m;
    }
}

// Stencil cell s of blade point t / 9 (s = t % 9; points blade by blade, plane by
// plane): the point from the step's blade orientation (blade_point, the host
// generator's arithmetic), by its first lanes also to the point list and the
// stencil rows; F = 0 where the previous mask lacks the cell; density and
// momentum into the blade cache.
template <typename PR, int STREAM, int MOMSRC, int EVEN>
__device__ __forceinline__ void gather_blade_cell(const ForceGeom& fg, const BladeStep& st, int t,
                                                  const typename PR::S* __restrict__ Q,
                                                  typename PR::T* __restrict__ F, const uint64_t* __restrict__ prev,
                                                  const Grid& g, float rho0) {
    using T = typename PR::T;
    const BladeLayout& bl = fg.blade;
    const BladeEnum be = blade_enum_of(bl);
    const int pt = t / 9, s = t - 9 * pt, c = s / 3;
    const int u = pt / be.n_radial, r = pt - u * be.n_radial, b = u / be.n_planes, pl = u - b * be.n_planes;
    const int e = blade_index(be, b, r, pl);
    tdlb_ib_point p;
    blade_point(bl.cx, bl.cz, bl.r_inner, bl.j_lo + pl, r, st.cosb[b], st.sinb[b], st.omega, &p);
    const int i = (int)p.i + bl.ghost, j = (int)p.j + bl.ghost, k = (int)p.k + bl.ghost;
    const int64_t q = fg.n_static + e;
    if (s == 0) {
        fg.pts.i[q] = i;
        fg.pts.j[q] = j;
        fg.pts.k[q] = k;
        static_cast<T*>(fg.pts.ifrac)[q] = (T)p.i_frac;
        static_cast<T*>(fg.pts.kfrac)[q] = (T)p.k_frac;
        static_cast<T*>(fg.pts.u)[q] = (T)p.u_delta;
        static_cast<T*>(fg.pts.v)[q] = (T)p.v_delta;
        static_cast<T*>(fg.pts.w)[q] = (T)p.w_delta;
    }
    // the plane's points in the order of its levels, for contiguous reads there
    const int64_t at = (int64_t)pl * be.n_blades * be.n_radial + level_slot(bl, b, r);
    if (s == 3 * c) {
        ForceRow<T> row = make_row<T>((T)p.i_frac, (T)p.k_frac, c,
                                      (T)(c == 0 ? p.u_delta : c == 1 ? p.v_delta : p.w_delta));
#pragma unroll
        for (int m = 0; m < 3; m++)
            row.e[m] = (int32_t)cell_index(g, wrap_ik(i + m - 1, g.xg1), j, wrap_ik(k + c - 1, g.zg1));
        static_cast<ForceRow<T>*>(fg.rows)[3 * (fg.n_static + at) + c] = row;
    }
    const int i2 = wrap_ik(i + (s - 3 * c) - 1, g.xg1), k2 = wrap_ik(k + c - 1, g.zg1);
    if (!mask_test(prev, g, i2, j, k2)) {
        const uint64_t cc = cell_index(g, i2, j, k2);
        F[3 * cc + 0] = T(0);
        F[3 * cc + 1] = T(0);
        F[3 * cc + 2] = T(0);
    }
    Mom4<T> m;
    cell_rho_j<PR, STREAM, MOMSRC, EVEN>(Q, g, i2, j, k2, m.r, m.x, m.y, m.z, rho0);
    static_cast<Mom4<T>*>(fg.rcache)[9 * at + s] = m;
}

// Block b of a tank's gather: the blades' blocks first (their points cost the
// most arithmetic), then the static cells', then the mask words'.
template <typename PR, int STREAM, int MOMSRC, int EVEN>
__device__ __forceinline__ void force_gather(const ForceGeom& fg, const BladeStep& st, uint32_t b,
                                             const GatherBlocks& gb, const typename PR::S* __restrict__ Q,
                                             typename PR::T* __restrict__ F, const uint64_t* __restrict__ prev,
                                             uint64_t* __restrict__ next, const uint64_t* __restrict__ static_base,
                                             const Grid& g, float rho0) {
    if (b < gb.blades) {
        const int64_t t = (int64_t)b * kGatherBlock + threadIdx.x;
        if (t < 9 * fg.n_rot)
            gather_blade_cell<PR, STREAM, MOMSRC, EVEN>(fg, st, (int)t, Q, F, prev, g, rho0);
        return;
    }
    b -= gb.blades;
    if (b < gb.cells) {
        const int64_t e = (int64_t)b * kGatherBlock + threadIdx.x;
        gather_cells<PR, STREAM, MOMSRC, EVEN>(fg, e, min(e + 1, fg.n_cells), 0, 1, Q, g, rho0);
        return;
    }
    const uint64_t w = (uint64_t)(b - gb.cells) * kGatherBlock + threadIdx.x;
    if (w < (uint64_t)g.xg * g.yg * g.mask_w) next[w] = static_base[w];
}

template <typename PR, int STREAM, int MOMSRC, int EVEN>
__global__ __launch_bounds__(kGatherBlock) void k_force_gather(ForceGeom fg, BladeStep st, GatherBlocks gb,
                                                               const typename PR::S* __restrict__ Q,
                                                               typename PR::T* __restrict__ F,
                                                               const uint64_t* __restrict__ prev,
                                                               uint64_t* __restrict__ next,
                                                               const uint64_t* __restrict__ static_base, Grid g,
                                                               float rho0) {
    force_gather<PR, STREAM, MOMSRC, EVEN>(fg, st, blockIdx.x, gb, Q, F, prev, next, static_base, g, rho0);
}

// a copy that every lane knows to be the same for the whole wave (scalar registers)
template <typename X>
__device__ __forceinline__ X uniform_copy(const X& x) {
    static_assert(sizeof(X) % 4 == 0, "words");
    struct Words {
        int w[sizeof(X) / 4];
    };
    Words a = __builtin_bit_cast(Words, x);
#pragma unroll
    for (size_t t = 0; t < sizeof(X) / 4; t++) a.w[t] = __builtin_amdgcn_readfirstlane(a.w[t]);
    return __builtin_bit_cast(X, a);
}

// The levels of a plane: passes of a point per quad of lanes, a barrier after every
// level; none is empty.  end_of(l): the end of level l's points, on any lane; row_at(q):
// the lane's stencil row of point q; mom_at(q, row, m): its moments; get and
// put(row, f): its force values.  A turn of the loop is one pass.  Rows are asked
// for three passes ahead and moments one, since neither changes meanwhile.  The
// turn is written out for each place of the ring of rows: with rows moved from one
// variable to the next, every move waited for the row in flight (24^3: 0.72 us a
// level, 0.55 without).  Level ends come from lanes of a register (64 levels at a
// time), the next pass from selects, and what a lane with a point does is the straight
// path: a level is then bound by the latency of its reads, sums, writes and barrier.
// Rows in HBM are asked for by every lane, without a branch (a lane without a point
// takes the level's last): past a branch that may have skipped loads the compiler
// waits for all of them.  Loads return in order, so in HBM a pass asks for its force
// values before the moments and rows of later passes, and within a level for the
// next pass's before it stores its own.
template <typename T, bool ROWS_LDS, bool F_LDS, typename End, typename RowAt, typename MomAt, typename Get, typename Put>
__device__ __forceinline__ void run_levels(int nlev, T alfa, T beta, End&& end_of, RowAt&& row_at, MomAt&& mom_at,
                                           Get&& get, Put&& put) {
    const int slot = (int)(threadIdx.x >> 2), lane = (int)(threadIdx.x & 3), per = (int)(blockDim.x >> 2);
    int begin = 0;
    for (int base = 0; base < nlev; base += 64) {
        const int levels = min(nlev - base, 64);
        // lane i of the wave: the end of level base + i, of the last beyond it
        const int ends = end_of(base + min((int)(threadIdx.x & 63), levels - 1));
        struct Pass {
            int l;       // level from base, `levels` after the last
            int q, end;  // first point, end of the level
        };
        auto next = [&](Pass a) {
            const bool same = a.q + per < a.end;
            const int l = same ? a.l : a.l + 1;
            return Pass{min(l, levels), same ? a.q + per : a.end, __builtin_amdgcn_readlane(ends, min(l, 63))};
        };
        auto on = [&](const Pass& a) { return a.q + slot < a.end; };
        ForceRow<T> r0, r1, r2, r3;
        Mom4<T> m0[3], m1[3];
        T f0[3][3], f1[3][3];
        Pass a0{0, begin, __builtin_amdgcn_readlane(ends, 0)}, a1 = next(a0), a2 = next(a1);
        begin = __builtin_amdgcn_readlane(ends, 63);
        auto load = [&](ForceRow<T>& r, const Pass& a) {
            if (!ROWS_LDS) r = row_at(min(a.q + slot, a.end - 1));
            else if (on(a)) r = row_at(a.q + slot);
        };
        load(r0, a0);
        load(r1, a1);
        load(r2, a2);
        if (on(a0)) mom_at(a0.q + slot, r0, m0);
        bool have = false;  // the pass's force values were asked for in the pass before
        // this pass, the next and the one three ahead
        auto turn = [&](ForceRow<T>& cr, ForceRow<T>& nr, ForceRow<T>& ar, Mom4<T> (&cm)[3], Mom4<T> (&nm)[3],
                        T (&cf)[3][3], T (&nf)[3][3]) {
            const bool on0 = on(a0), on1 = on(a1), same = a1.l == a0.l;
            if ((F_LDS || !have) && __builtin_expect(on0, true)) get(cr, cf);
            if (!F_LDS && same && on1) get(nr, nf);
            if (__builtin_expect(on1, true)) mom_at(a1.q + slot, nr, nm);
            const Pass a3 = next(a2);
            __builtin_amdgcn_sched_barrier(0);  // the row behind them: no wait for moments or forces includes it
            load(ar, a3);
            if (__builtin_expect(on0, true)) {
                force_row(cr, cm, cf, alfa, beta);
                if (lane < 3) put(cr, cf);
            }
            if (!same) __syncthreads();
            a0 = a1;
            a1 = a2;
            a2 = a3;
            have = same;
            return a0.l < levels;
        };
        for (;;) {
            if (!turn(r0, r1, r3, m0, m1, f0, f1)) break;
            if (!turn(r1, r2, r0, m1, m0, f1, f0)) break;
            if (!turn(r2, r3, r1, m0, m1, f0, f1)) break;
            if (!turn(r3, r0, r2, m1, m0, f1, f0)) break;
        }
    }
}

// Static levels.  lm: the moments by entry of the plane, in LDS (MOM_LDS) or the
// cache in HBM; the force values by entry: lf in LDS (F_LDS), else four T an entry
// in the plane's scratch fs.
template <typename T, bool MOM_LDS, bool F_LDS>
__device__ __forceinline__ void static_levels(const ForceGeom& fg, const PlaneDesc& pd, const Mom4<T>* lm, T* lf,
                                              Mom4<T>* fs, T alfa, T beta) {
    const int c = min((int)(threadIdx.x & 3), 2), nlev = pd.n_levels;
    if (nlev == 0) return;
    const int64_t* off = fg.lev_off + pd.lev;
    const int64_t q0 = off[0];
    const ForceRow<T>* rows = static_cast<const ForceRow<T>*>(fg.rows) + 3 * q0 + c;
    run_levels<T, false, F_LDS>(
        nlev, alfa, beta, [&](int l) { return (int)(off[l + 1] - q0); },
        [&](int q) { return rows[3 * (int64_t)q]; },
        [&](int, const ForceRow<T>& r, Mom4<T> (&m)[3]) {
#pragma unroll
            for (int b = 0; b < 3; b++) m[b] = lm[r.e[b]];
        },
        [&](const ForceRow<T>& r, T (&f)[3][3]) {
#pragma unroll
            for (int b = 0; b < 3; b++) {
                if constexpr (F_LDS) {
#pragma unroll
                    for (int a = 0; a < 3; a++) f[b][a] = lf[__umul24(r.e[b], 3) + a];
                } else {
                    const Mom4<T> w = fs[r.e[b]];
                    f[b][0] = w.r;
                    f[b][1] = w.x;
                    f[b][2] = w.y;
                }
            }
        },
        [&](const ForceRow<T>& r, const T (&f)[3][3]) {
#pragma unroll
            for (int b = 0; b < 3; b++) {
                if constexpr (F_LDS) {
#pragma unroll
                    for (int a = 0; a < 3; a++) lf[__umul24(r.e[b], 3) + a] = f[b][a];
                } else {
                    fs[r.e[b]] = Mom4<T>{f[b][0], f[b][1], f[b][2], T(0)};
                }
            }
        });
}

// The blade levels of a plane.  With room in LDS the rows and moments of all its
// points come there first (blade_rows), and if a copy of the whole plane's force
// values fits beside them the stencil cells' too: a level then waits on LDS alone.
// Otherwise the force values stay in F, and without any room the rows and moments
// in the caches.
template <typename T>
struct BladeRow {
    ForceRow<T> r;
    Mom4<T> mo[3];
};
static_assert(3 * sizeof(BladeRow<float>) == blade_row_bytes(4) && 3 * sizeof(BladeRow<double>) == blade_row_bytes(8), "LDS");

// rows and moments of blade plane bp to LDS
template <typename T>
__device__ __forceinline__ void blade_rows(const ForceGeom& fg, int bp, BladeRow<T>* lr) {
    const int n3 = 3 * fg.blade.n_blades * fg.blade.n_radial;
    const ForceRow<T>* __restrict__ rows = static_cast<const ForceRow<T>*>(fg.rows) + 3 * fg.n_static + (int64_t)bp * n3;
    const Mom4<T>* __restrict__ cache = static_cast<const Mom4<T>*>(fg.rcache) + (int64_t)bp * n3 * 3;
    for (int t = (int)threadIdx.x; t < n3; t += (int)blockDim.x) {
        const ForceRow<T> r = rows[t];
        const Mom4<T> a = cache[3 * t], b = cache[3 * t + 1], c = cache[3 * t + 2];
        lr[t].r = r;
        lr[t].mo[0] = a;
        lr[t].mo[1] = b;
        lr[t].mo[2] = c;
    }
}

// lr: the plane's rows, in LDS already (ROWS_LDS); ld: room for its force values (F_LDS)
template <typename T, bool ROWS_LDS, bool F_LDS>
__device__ __forceinline__ void blade_levels(const ForceGeom& fg, const Grid& g, int j, int bp, int nlev,
                                             T* __restrict__ F, uint64_t* __restrict__ next, BladeRow<T>* lr, T* ld,
                                             T alfa, T beta) {
    const int c = min((int)(threadIdx.x & 3), 2), n3 = 3 * fg.blade.n_blades * fg.blade.n_radial;
    const ForceRow<T>* __restrict__ rows = static_cast<const ForceRow<T>*>(fg.rows) + 3 * fg.n_static + (int64_t)bp * n3;
    const Mom4<T>* __restrict__ cache = static_cast<const Mom4<T>*>(fg.rcache) + (int64_t)bp * n3 * 3;
    // the occupancy bits of the rows' cells, and the cells' force values
    for (int t = (int)threadIdx.x; t < n3; t += (int)blockDim.x) {
#pragma unroll
        for (int m = 0; m < 3; m++) {
            const uint32_t n = (uint32_t)(ROWS_LDS ? lr[t].r.e[m] : rows[t].e[m]);
            const int i = (int)(n / g.yz), k = (int)(n - (uint32_t)i * g.yz - (uint32_t)j * (uint32_t)g.zg);
            if constexpr (F_LDS) {
                const int e = (i - 1) * g.zg1 + k - 1;
                lr[t].r.e[m] = e;
#pragma unroll
                for (int a = 0; a < 3; a++) ld[3 * e + a] = F[3 * (uint64_t)n + a];
            }
            atomicOr((unsigned long long*)&next[mask_word_index(g, i, j, k)], 1ull << (k & 63));
        }
    }
    if constexpr (F_LDS) __syncthreads();
    run_levels<T, ROWS_LDS, F_LDS>(
        nlev, alfa, beta,
        [&](int l) { return blade_level_end(fg.blade, l); },
        [&](int q) {
            if constexpr (ROWS_LDS) return lr[3 * q + c].r;
            else return rows[3 * q + c];
        },
        [&](int q, const ForceRow<T>&, Mom4<T> (&m)[3]) {
#pragma unroll
            for (int b = 0; b < 3; b++) {
                if constexpr (ROWS_LDS) m[b] = lr[3 * q + c].mo[b];
                else m[b] = cache[3 * (3 * q + c) + b];
            }
        },
        [&](const ForceRow<T>& r, T (&f)[3][3]) {
#pragma unroll
            for (int b = 0; b < 3; b++)
#pragma unroll
                for (int a = 0; a < 3; a++) f[b][a] = F_LDS ? ld[__umul24(r.e[b], 3) + a] : F[3 * (uint64_t)(uint32_t)r.e[b] + a];
        },
        [&](const ForceRow<T>& r, const T (&f)[3][3]) {
#pragma unroll
            for (int b = 0; b < 3; b++)
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    if constexpr (F_LDS) ld[__umul24(r.e[b], 3) + a] = f[b][a];
                    else F[3 * (uint64_t)(uint32_t)r.e[b] + a] = f[b][a];
                }
        });
    if constexpr (F_LDS) {
        // back to F, once per point and cell: points that share a cell write the same value
        for (int t = (int)threadIdx.x; t < 3 * n3; t += (int)blockDim.x) {
            const int pr = t / 3, p = lr[pr].r.e[t - 3 * pr];
            const int i = p / g.zg1, k = p - i * g.zg1;
            const uint64_t n = cell_index(g, i + 1, j, k + 1);
#pragma unroll
            for (int a = 0; a < 3; a++) F[3 * n + a] = ld[3 * p + a];
        }
    }
}

// The levels of one plane by one workgroup.  Every stencil cell of a plane lies
// in the plane, which no other workgroup touches, so the force values of the
// static cells leave F for the static levels: to LDS, with the moments when both
// fit, else to the plane's scratch in HBM.
template <typename T>
__device__ __forceinline__ void plane_levels(const ForceGeom& fg, const PlaneDesc* plane, T* __restrict__ F,
                                             uint64_t* __restrict__ next, const Grid& g, T alfa, T beta, void* lds,
                                             int64_t lds_bytes) {
    const PlaneDesc pd = uniform_copy(*plane);
    const int tid = (int)threadIdx.x, nt = (int)blockDim.x, nc = (int)(pd.cell_end - pd.cell_begin);
    const int64_t mom_bytes = (int64_t)nc * sizeof(Mom4<T>), f_bytes = (int64_t)nc * 3 * sizeof(T);
    const bool f_lds = f_bytes <= lds_bytes, mom_lds = mom_bytes + f_bytes <= lds_bytes;
    // The blades' rows come at the start if they fit beside what the static levels
    // keep: after them the wait for the rows was 1 to 2 us of a plane's 20.
    int nlev;
    const int bp = blade_plane(fg, pd.j, nlev);
    const bool blades = nlev > 0 && pd.blades;
    const int64_t row_bytes = 3 * (int64_t)fg.blade.n_blades * fg.blade.n_radial * sizeof(BladeRow<T>);
    const bool early = blades && row_bytes + (mom_lds ? mom_bytes + f_bytes : f_lds ? f_bytes : 0) <= lds_bytes;
    auto* const lr = static_cast<BladeRow<T>*>(lds);
    auto* const ld = reinterpret_cast<T*>(static_cast<char*>(lds) + row_bytes);
    if (early) {
        blade_rows(fg, bp, lr);
        lds = ld;
    }
    const auto* gm = static_cast<const Mom4<T>*>(fg.scache) + pd.cell_begin;
    auto* fs = static_cast<Mom4<T>*>(fg.fscr) + pd.cell_begin;
    auto* lm = static_cast<Mom4<T>*>(lds);
    T* lf = mom_lds ? reinterpret_cast<T*>(lm + nc) : static_cast<T*>(lds);
    const uint32_t* __restrict__ cells = fg.cells + pd.cell_begin;
    for (int e = tid; e < nc; e += nt) {
        const uint64_t n = cells[e];
        T f[3];
#pragma unroll
        for (int a = 0; a < 3; a++) f[a] = F[3 * n + a];
        if (mom_lds) lm[e] = gm[e];
        if (f_lds)
#pragma unroll
            for (int a = 0; a < 3; a++) lf[3 * e + a] = f[a];
        else fs[e] = Mom4<T>{f[0], f[1], f[2], T(0)};
    }
    __syncthreads();
    if (mom_lds) static_levels<T, true, true>(fg, pd, lm, lf, nullptr, alfa, beta);
    else if (f_lds) static_levels<T, false, true>(fg, pd, gm, lf, nullptr, alfa, beta);
    else static_levels<T, false, false>(fg, pd, gm, nullptr, fs, alfa, beta);
    // every static level ended with a barrier: the force values back to F before the blade levels read it
    for (int e = tid; e < nc; e += nt) {
        const uint64_t n = cells[e];
        if (f_lds) {
#pragma unroll
            for (int a = 0; a < 3; a++) F[3 * n + a] = lf[3 * e + a];
        } else {
            const Mom4<T> v = fs[e];
            F[3 * n + 0] = v.r;
            F[3 * n + 1] = v.x;
            F[3 * n + 2] = v.y;
        }
    }
    if (!blades) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const bool rows_lds = row_bytes <= lds_bytes;
    if (rows_lds && !early) {
        blade_rows(fg, bp, lr);
        __syncthreads();
    }
    if (row_bytes + plane_force_bytes(g, sizeof(T)) <= lds_bytes)
        blade_levels<T, true, true>(fg, g, pd.j, bp, nlev, F, next, lr, ld, alfa, beta);
    else if (rows_lds)
        blade_levels<T, true, false>(fg, g, pd.j, bp, nlev, F, next, lr, nullptr, alfa, beta);
    else blade_levels<T, false, false>(fg, g, pd.j, bp, nlev, F, next, nullptr, nullptr, alfa, beta);
}

template <typename T>
__global__ __launch_bounds__(level_block<T>()) void k_force_levels(ForceGeom fg, T* __restrict__ F,
                                                                   uint64_t* __restrict__ next, Grid g, T alfa, T beta,
                                                                   int64_t lds_bytes) {
    extern __shared__ float4 levels_lds[];  // lds_bytes, launch-sized
    plane_levels<T>(fg, fg.planes + blockIdx.x, F, next, g, alfa, beta, levels_lds, lds_bytes);
}

// ------------------------------------------------------------------ pipelined Esotwist step
// PipeArgs in kernels.h.  Work items of XCD x, in queue order (nJ planes
// [jlo, jhi], R = nJ * nkb row blocks per i step):
//   A  for i = 1 .. xg1: the R rows (i, j) of the range; after the rows of i
//      the gather of i - 2 (interior planes jlo < j < jhi; a gather of i reads
//      what the rows of i - 1 .. i + 1 wrote, i wrapping periodically), then
//      the gathers of xg1 - 1, xg1 and 1
//   B  the edge planes jlo and jhi (their gathers read rows of the
//      neighbouring XCDs), in chunks, once those XCDs have released their rows
// (The blade cells and the forcing levels follow in launches of their own.)  A row
// item also copies its rows' static occupancy words into next.  Items
// wait only for earlier items, so every wait ends; spins are bounded anyway
// (kBarSpinLimit, flag in the XCD's counters).
//
// Counters (uint32, zero at launch): XCD x at ctr[64 x]: +0 next item, +1 rows
// done, +2 gathers done, +3 rows released to the other XCDs, +4 time-out flag;
// rows done per i step at ctr[64 kXcds + x (xg1 + 2) + i].  The XCD-local
// counters are relaxed agent-scope atomics: the rows a gather reads were
// written through this XCD's L2, and each row's stores are complete
// (s_waitcnt) before its count.  The release of a range for the neighbours is
// an agent-scope fence pair.
// polls of a wait before it gives up and flags a time-out (about a second)
constexpr uint32_t kBarSpinLimit = 1u << 20;
__device__ __forceinline__ uint32_t xcc_id() {
    uint32_t x;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(x));
    return x;
}
__device__ __forceinline__ uint32_t ld_ctr(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// thread 0 polls until every counter reaches its target (or the spin limit)
__device__ __forceinline__ void pipe_wait(const uint32_t* a, uint32_t ta, const uint32_t* b, uint32_t tb,
                                          const uint32_t* c, uint32_t tc, uint32_t* flag) {
    if (threadIdx.x == 0) {
        uint32_t spins = 0;
        while (ld_ctr(a) < ta || (b && ld_ctr(b) < tb) || (c && ld_ctr(c) < tc)) {
            if (++spins >= kBarSpinLimit) {
                atomicOr(flag, 1u);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
    }
    __syncthreads();
}
// rows of one item of the pipe (consecutive j of one i step)
constexpr uint32_t kPipeRows = 8;

// Occupancy of the pipe: 8 waves per SIMD for the 16-bit formats (61
// registers); 5 for FP32, the most without spills (92 registers; the separate
// FP32 kernel runs 6 at 74).
template <typename PR>
constexpr int pipe_waves() { return std::is_same<typename PR::S, float>::value ? 5 : 8; }

template <typename PR, int EVEN, bool HINT>
__global__ __launch_bounds__(kRowBlock) __attribute__((amdgpu_waves_per_eu(pipe_waves<PR>(), 8)))
void k_eso_pipe(PipeArgs a, Grid g, CollideParams<float> P, uint32_t nkb, float rho0) {
    using S = typename PR::S;
    constexpr int STREAM = StreamEsotwist;
    constexpr int MS = MOMSRC_ESO_POPS;
    // the gathers read the populations of the next step's collision
    constexpr int GE = EVEN ? 0 : 1;
    __shared__ uint32_t s_item;
    __shared__ int64_t s_pre[258];
    __shared__ int32_t s_c0[256];
    const uint32_t x = xcc_id() % kXcds;
    uint32_t* cx = a.ctr + 64 * x;
    uint64_t* tx = reinterpret_cast<uint64_t*>(cx + 8);  // phase times (wall clock)
    uint32_t* rows_done = a.ctr + 64 * kXcds + (size_t)x * (g.xg1 + 2);
    int jlo, jhi;
    pipe_range(g.yg1, (int)x, jlo, jhi);
    const int nj = jhi - jlo + 1, ni = g.xg1;
    const uint32_t R = (uint32_t)nj * nkb;                // row blocks per i step
    const uint32_t RG = (R + kPipeRows - 1) / kPipeRows;  // row items per i step
    const uint32_t nA = (uint32_t)ni * (RG + 1) + 3;
    const int rw = g.xg1 + 2;
    const int32_t* rc = a.rowcell;
    const int64_t cl0 = rc[(size_t)jlo * rw + 1], cl1 = rc[(size_t)jlo * rw + ni + 1];
    const int64_t ch0 = rc[(size_t)jhi * rw + 1], ch1 = rc[(size_t)jhi * rw + ni + 1];
    const int64_t chunk = 4 * (int64_t)blockDim.x;
    const uint32_t nBl = (uint32_t)((cl1 - cl0 + chunk - 1) / chunk), nBh = (uint32_t)((ch1 - ch0 + chunk - 1) / chunk);
    const uint32_t nB = nBl + nBh;
    const uint32_t gathers = (uint32_t)ni + nB;
    const uint32_t total = nA + nB;
    S* Q = static_cast<S*>(a.Q);
    float* F = static_cast<float*>(a.F);
    auto* Nu = static_cast<typename PR::N*>(a.Nu);
    const int tid = (int)threadIdx.x;

    // gather of row i over the interior planes of the range
    auto gather_row = [&](int i) {
        const int ninner = nj - 2;
        for (int p = tid; p < ninner; p += blockDim.x) {
            const size_t r = (size_t)(jlo + 1 + p) * rw + i;
            s_c0[p] = rc[r];
            s_pre[p + 1] = rc[r + 1] - rc[r];
        }
        __syncthreads();
        if (tid == 0) {
            s_pre[0] = 0;
            for (int p = 0; p < ninner; p++) s_pre[p + 1] += s_pre[p];
        }
        __syncthreads();
        const int64_t cells = s_pre[ninner];
        for (int64_t t = tid; t < cells; t += blockDim.x) {
            int lo = 0, hi = ninner - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (s_pre[mid] <= t) lo = mid;
                else hi = mid - 1;
            }
            const int64_t e = s_c0[lo] + (t - s_pre[lo]);
            gather_cells<PR, STREAM, MS, GE>(a.fg, e, e + 1, 0, 1, Q, g, rho0);
        }
    };
    auto wait_rows = [&](int i) {
        const int im = i == 1 ? ni : i - 1, ip = i == ni ? 1 : i + 1;
        pipe_wait(rows_done + im, R, rows_done + i, R, rows_done + ip, R, cx + 4);
    };
    auto gather_done = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0 &&
            __hip_atomic_fetch_add(cx + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == gathers)
            tx[2] = tx[3] = (uint64_t)wall_clock64();  // the third phase ends with the second: the levels follow in a launch of their own
    };

    // the next item is taken while the current one runs (each waits only for earlier items)
    uint32_t ticket = 0;
    if (tid == 0) ticket = __hip_atomic_fetch_add(cx, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (;;) {
        __syncthreads();
        if (tid == 0) {
            s_item = ticket;
            if (ticket == 0) tx[0] = (uint64_t)wall_clock64();
            if (ticket < total) ticket = __hip_atomic_fetch_add(cx, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        const uint32_t u = s_item;
        if (u >= total) break;
        if (u < (uint32_t)ni * (RG + 1)) {
            const int i = (int)(u / (RG + 1)) + 1;
            const uint32_t r = u % (RG + 1);
            if (r < RG) {
                // A: row blocks [r G, r G + G) of i step i: row (i, jlo + b / nkb), k chunk b % nkb
                const uint32_t b0 = r * kPipeRows, b1 = min(b0 + kPipeRows, R);
                for (uint32_t b = b0; b < b1; b++) {
                    const int j = jlo + (int)(b / nkb);
                    const int k = (int)((b % nkb) * blockDim.x) + 1 + tid;
                    if (k <= g.zg1)
                        esotwist_cell<PR, MODE_FUSED, EVEN, HINT>(Q, nullptr, F, Nu, a.prev, g, P, rho0, i, j, k);
                    if (b % nkb == 0) {
                        // static occupancy words of the row, and of the ghost rows beside it
                        const int ia = i == 1 ? 0 : i, ib = i == ni ? ni + 1 : i;
                        const int ja = j == 1 ? 0 : j, jb = j == g.yg1 ? g.yg1 + 1 : j;
                        const int nw = (int)g.mask_w;
                        const int cnt = (ib - ia + 1) * (jb - ja + 1) * nw;
                        for (int t = tid; t < cnt; t += blockDim.x) {
                            const int w = t % nw, rr = t / nw;
                            const int jj = ja + rr % (jb - ja + 1), ii = ia + rr / (jb - ja + 1);
                            const uint64_t wi =
                                ((uint64_t)ii * (uint64_t)g.yg + (uint64_t)jj) * g.mask_w + (uint64_t)w;
                            a.next[wi] = a.static_base[wi];
                        }
                    }
                }
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
                if (tid == 0) {
                    __hip_atomic_fetch_add(rows_done + i, b1 - b0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    const uint32_t done =
                        __hip_atomic_fetch_add(cx + 1, b1 - b0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (done + (b1 - b0) == (uint32_t)ni * R) {
                        // every row of the range is in this XCD's L2: write it back for the neighbours
                        tx[1] = (uint64_t)wall_clock64();
                        __threadfence();
                        __hip_atomic_store(cx + 3, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
            } else if (i >= 4) {
                wait_rows(i - 2);
                gather_row(i - 2);
                gather_done();
            }
        } else if (u < nA) {
            const uint32_t tail = u - (uint32_t)ni * (RG + 1);
            const int i = tail == 0 ? ni - 1 : tail == 1 ? ni : 1;
            wait_rows(i);
            gather_row(i);
            gather_done();
        } else if (u < nA + nB) {
            // B: the edge planes, after the neighbouring ranges are released
            const uint32_t b = u - nA;
            const uint32_t xl = (x + kXcds - 1) % kXcds, xh = (x + 1) % kXcds;
            pipe_wait(a.ctr + 64 * xl + 3, 1, cx + 3, 1, a.ctr + 64 * xh + 3, 1, cx + 4);
            __threadfence();
            const int64_t c0 = b < nBl ? cl0 + (int64_t)b * chunk : ch0 + (int64_t)(b - nBl) * chunk;
            const int64_t c1 = b < nBl ? cl1 : ch1;
            gather_cells<PR, STREAM, MS, GE>(a.fg, c0, c0 + chunk < c1 ? c0 + chunk : c1, tid, blockDim.x, Q, g,
                                                 rho0);
            gather_done();
        }
    }
}

__global__ void k_xcc_ids(uint32_t* out) {
    if (threadIdx.x == 0) out[blockIdx.x] = xcc_id();
}

// ------------------------------------------------------------------ FP64 sums and macroscopic fields
// Both read density and momentum through cell_rho_j, so they work on stored
// moments and on the populations of the fused path alike, without changing
// the state.  Interior cells are enumerated t = ((i-1)*y + (j-1))*z + (k-1).
__device__ __forceinline__ void interior_cell(const Grid& g, uint64_t t, int& i, int& j, int& k) {
    k = (int)(t % (uint64_t)g.zg1) + 1;
    const uint64_t r = t / (uint64_t)g.zg1;
    j = (int)(r % (uint64_t)g.yg1) + 1;
    i = (int)(r / (uint64_t)g.yg1) + 1;
}

template <typename T>
__device__ __forceinline__ void cell_force(const T* __restrict__ F, const uint64_t* __restrict__ fmask,
                                           const Grid& g, int i, int j, int k, T& fx, T& fy, T& fz) {
    fx = fy = fz = T(0);
    if (mask_test(fmask, g, i, j, k)) {
        const uint64_t c = cell_index(g, i, j, k);
        fx = F[3 * c + 0];
        fy = F[3 * c + 1];
        fz = F[3 * c + 2];
    }
}

// Per block: {sum rho, sum jx, jy, jz, sum Fx, Fy, Fz, torque} in FP64.  The
// grid is fixed, so the partial sums and their combination are deterministic.
template <typename PR, int STREAM, int MOMSRC, int EVEN>
__global__ __launch_bounds__(kBlock) void k_reduce_cells(const typename PR::S* __restrict__ Q,
                                                         const typename PR::T* __restrict__ F,
                                                         const uint64_t* __restrict__ fmask, Grid g, ReduceArgs ra,
                                                         float rho0, double* __restrict__ partial) {
    using T = typename PR::T;
    double acc[kReduceVals];
#pragma unroll
    for (int v = 0; v < kReduceVals; v++) acc[v] = 0.0;
    const uint64_t n = (uint64_t)g.xg1 * g.yg1 * g.zg1;
    for (uint64_t t = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; t < n; t += (uint64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        interior_cell(g, t, i, j, k);
        T rho, jx, jy, jz, fx, fy, fz;
        cell_rho_j<PR, STREAM, MOMSRC, EVEN>(Q, g, i, j, k, rho, jx, jy, jz, rho0);
        cell_force(F, fmask, g, i, j, k, fx, fy, fz);
        acc[0] += (double)rho;
        acc[1] += (double)jx;
        acc[2] += (double)jy;
        acc[3] += (double)jz;
        acc[4] += (double)fx;
        acc[5] += (double)fy;
        acc[6] += (double)fz;
        const double x = (double)(i - ra.ghost) - ra.cx, z = (double)(k - ra.ghost) - ra.cz;
        if (x * x + z * z <= ra.r2) acc[7] += x * (double)fz - z * (double)fx;
    }
    __shared__ double red[kReduceVals][kBlock / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int v = 0; v < kReduceVals; v++) {
        double a = acc[v];
        for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
        if (lane == 0) red[v][wave] = a;
    }
    __syncthreads();
    if (threadIdx.x < kReduceVals) {
        double a = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) a += red[threadIdx.x][w];
        partial[(uint64_t)blockIdx.x * kReduceVals + threadIdx.x] = a;
    }
}

// The partials added in block order, one lane per value.  The chain of 1024
// dependent adds is the least this order allows (about 5 us); loading each
// partial inside the chain took 150 us, so a workgroup brings them to LDS first.
constexpr int kReduceFinalBlock = 1024;
__global__ __launch_bounds__(kReduceFinalBlock) void k_reduce_final(const double* __restrict__ partial,
                                                                    double* __restrict__ out) {
    __shared__ double p[kReduceBlocks * kReduceVals];
    for (int t = (int)threadIdx.x; t < kReduceBlocks * kReduceVals; t += kReduceFinalBlock) p[t] = partial[t];
    __syncthreads();
    if (threadIdx.x >= kReduceVals) return;
    double a = 0.0;
#pragma unroll 32
    for (int b = 0; b < kReduceBlocks; b++) a += p[b * kReduceVals + (int)threadIdx.x];
    out[threadIdx.x] = a;
}

// {rho, ux, uy, uz} of interior cells [begin, end), u as QVec::velocity(F) forms it
// (QVec.hpp:125-131: (1.0 / rho) * (j + 0.5 * F), double literals).
template <typename PR, int STREAM, int MOMSRC, int EVEN>
__global__ __launch_bounds__(kBlock) void k_macroscopic(const typename PR::S* __restrict__ Q,
                                                        const typename PR::T* __restrict__ F,
                                                        const uint64_t* __restrict__ fmask, Grid g, float rho0,
                                                        uint64_t begin, uint64_t end, Mom4<typename PR::T>* __restrict__ out) {
    using T = typename PR::T;
    using D = typename PR::D;
    for (uint64_t t = begin + blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; t < end;
         t += (uint64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        interior_cell(g, t, i, j, k);
        T rho, jx, jy, jz, fx, fy, fz;
        cell_rho_j<PR, STREAM, MOMSRC, EVEN>(Q, g, i, j, k, rho, jx, jy, jz, rho0);
        cell_force(F, fmask, g, i, j, k, fx, fy, fz);
        const D inv = D(1.0) / (D)rho;
        out[t - begin] = Mom4<T>{rho, (T)(inv * ((D)jx + D(0.5) * (D)fx)), (T)(inv * ((D)jy + D(0.5) * (D)fy)),
                                 (T)(inv * ((D)jz + D(0.5) * (D)fz))};
    }
}

// ------------------------------------------------------------------ regrid and output planes
// doubleResolutionFullCU (ComputeUnit.hpp:229-316, 480-502): every cell of the
// doubled grid, ghosts included, takes old cell (i/2 + i%2, j/2 + j%2, k/2 + k%2).
__device__ __forceinline__ uint32_t regrid_source(const Grid& og, const Grid& ng, uint64_t n) {
    int i, j, k;
    decode_cell(ng, n, i, j, k);
    return cell_index(og, i / 2 + (i & 1), j / 2 + (j & 1), k / 2 + (k & 1));
}

template <typename W>
__global__ void k_regrid_q(const W* __restrict__ old, W* __restrict__ nw, Grid og, Grid ng) {
    for (uint64_t n = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; n < ng.size;
         n += (uint64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        decode_cell(ng, n, i, j, k);
        const uint32_t to = qcell(ng, i, j, k);
        const uint32_t from = qcell(og, i / 2 + (i & 1), j / 2 + (j & 1), k / 2 + (k & 1));
#pragma unroll
        for (int l = 0; l < kQ; l++) nw[qaddr(ng, to, l)] = old[qaddr(og, from, l)];
    }
}

template <typename W>
__global__ void k_regrid_cells(const W* __restrict__ old, W* __restrict__ nw, Grid og, Grid ng) {
    for (uint64_t n = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; n < ng.size;
         n += (uint64_t)gridDim.x * blockDim.x)
        nw[n] = old[regrid_source(og, ng, n)];
}

// savePlaneXZ<float, 4> (ComputeUnitOutput.hpp:354-447) for every plane cell
// (i-major); flags bit 0: a QVec record (cell not excluded), bit 1: an F3 record
// (Force::isNotZero: all three components non-zero, QVec.hpp:54-56).
template <typename T>
__global__ void k_plane_xz(const T* __restrict__ Q, const T* __restrict__ F, const uint64_t* __restrict__ fmask,
                           const uint8_t* __restrict__ exclude, Grid g, int cut, int64_t i0, int64_t k0,
                           PlaneRec4* __restrict__ q, PlaneRec3* __restrict__ f, uint8_t* __restrict__ flags) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= (int64_t)g.xg1 * g.zg1) return;
    const int i = (int)(t / g.zg1) + 1, k = (int)(t % g.zg1) + 1;
    const uint32_t n = cell_index(g, i, cut, k);
    uint8_t fl = 0;
    if (!(exclude && exclude[n])) {
        fl = 1;
        PlaneRec4 r;
        r.i = (uint16_t)(i0 + i - 1);
        r.j = (uint16_t)(cut - 1);
        r.k = (uint16_t)(k0 + k - 1);
        r.pad = 0;
#pragma unroll
        for (int l = 0; l < 4; l++) r.q[l] = (float)Q[qaddr(g, qcell(g, i, cut, k), l)];
        q[t] = r;
        if (mask_test(fmask, g, i, cut, k)) {
            const T fx = F[3 * (uint64_t)n], fy = F[3 * (uint64_t)n + 1], fz = F[3 * (uint64_t)n + 2];
            if (fx != T(0) && fy != T(0) && fz != T(0)) {
                fl |= 2;
                PlaneRec3 s;
                s.i = (uint16_t)(i0 + i - 1);
                s.j = (uint16_t)cut;
                s.k = (uint16_t)(k0 + k - 1);
                s.pad = 0;
                s.q[0] = (float)fx;
                s.q[1] = (float)fy;
                s.q[2] = (float)fz;
                f[t] = s;
            }
        }
    }
    flags[t] = fl;
}

// calcVorticityXZ / XY (ComputeUnitOutput.hpp:113-160, 198-245) before the
// picture: log|curl u|^2 from central differences of QVec::velocity() (j / rho,
// no force term) read through the streaming accessor; excluded cells NaN.  The
// twisted read of a far-side ghost cell leaves the array in the reference, so
// such neighbours give NaN here.  axis 0: plane j = cut, (x, z); 1: k = cut, (x, y).
template <typename PR, int STREAM, int MOMSRC, int EVEN>
__global__ void k_vorticity(const typename PR::S* __restrict__ Q, Grid g, int axis, int cut,
                            const uint8_t* __restrict__ exclude, typename PR::T* __restrict__ out, float rho0) {
    using T = typename PR::T;
    const int nb = axis == 0 ? g.zg1 : g.yg1;
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= (int64_t)g.xg1 * nb) return;
    const int i = (int)(t / nb) + 1, c = (int)(t % nb) + 1;
    const int j = axis == 0 ? cut : c, k = axis == 0 ? c : cut;
    if (exclude && exclude[cell_index(g, i, j, k)]) {
        out[t] = (T)NAN;
        return;
    }
    auto vel = [&](int a, int b, int e, T& ux, T& uy, T& uz) {
        if (STREAM == StreamEsotwist && (a == g.xg1 + 1 || b == g.yg1 + 1 || e == g.zg1 + 1)) {
            ux = uy = uz = (T)NAN;
            return;
        }
        T rho, jx, jy, jz;
        if (STREAM == StreamEsotwist && MOMSRC == MOMSRC_STORED && e == 0) {
            // a ghost cell at k = 0 has its homes in the side region too, whose rows lie closer than the interior's
            T m[4];
#pragma unroll
            for (int d = 0; d < 4; d++) {
                static_assert(!twist_dz(0) && !twist_dz(1) && !twist_dz(2) && !twist_dz(3), "density and momentum stay at k");
                const int a2 = twist_dx(d) ? (a == g.xg1 ? 1 : a + 1) : a, b2 = twist_dy(d) ? (b == g.yg1 ? 1 : b + 1) : b;
                m[d] = (T)Q[qaddr(g, qcell(g, a2, b2, 0), EVEN ? d : opposite(d))];
            }
            rho = m[0]; jx = m[1]; jy = m[2]; jz = m[3];
        } else {
            cell_rho_j<PR, STREAM, MOMSRC, EVEN>(Q, g, a, b, e, rho, jx, jy, jz, rho0);
        }
        ux = jx / rho;
        uy = jy / rho;
        uz = jz / rho;
    };
    T x5, y5, z5, x6, y6, z6, x3, y3, z3, x4, y4, z4, x1, y1, z1, x2, y2, z2;
    vel(i, j, k + 1, x5, y5, z5);
    vel(i, j, k - 1, x6, y6, z6);
    const T uxy = T(0.5) * (x5 - x6);
    vel(i, j + 1, k, x3, y3, z3);
    vel(i, j - 1, k, x4, y4, z4);
    const T uxz = T(0.5) * (x3 - x4);
    vel(i + 1, j, k, x1, y1, z1);
    vel(i - 1, j, k, x2, y2, z2);
    const T uyx = T(0.5) * (y1 - y2);
    const T uyz = T(0.5) * (y3 - y4);
    const T uzx = T(0.5) * (z1 - z2);
    const T uzy = T(0.5) * (z5 - z6);
    const T uxyuyx = uxy - uyx;
    const T uyzuzy = uyz - uzy;
    const T uzxuxz = uzx - uxz;
    out[t] = (T)log((T)(uyzuzy * uyzuzy + uzxuxz * uzxuxz + uxyuyx * uxyuyx));
}

// ------------------------------------------------------------------ geometry on the device
// getExternalPoints as a mask: a cell is outside when its centre lies beyond the
// tank radius from the axis (exact: integer and half-integer coordinates).
__global__ void k_solid_mask(double cx, double cz, double radius, uint8_t* __restrict__ out, Grid g, int ghost) {
    for (uint64_t n = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; n < g.size;
         n += (uint64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        decode_cell(g, n, i, j, k);
        const double dx = (double)(i - ghost) - cx, dz = (double)(k - ghost) - cz;
        out[n] = (dx * dx + dz * dz > radius * radius) ? 1 : 0;
    }
}

template <typename T>
CollideParams<T> to_params(const CollideArgs& c) {
    return make_collide_params<T>(T(c.nu), T(c.cs0), T(c.g3), c.use_les);
}
template <typename T, typename D>
CollideParams<T> to_params(const CollideArgs& c) {
    return make_collide_params<T, D>(T(c.nu), T(c.cs0), T(c.g3), c.use_les);
}

uint32_t grid_blocks(uint64_t n) {
    uint64_t b = (n + kBlock - 1) / kBlock;
    if (b > 65536ull * 16) b = 65536ull * 16;
    return (uint32_t)(b ? b : 1);
}

// rows of interior cells: nkb blocks of bk threads along k, bk a multiple of
// the wavefront (64) covering the row in as few blocks of at most bmax lanes
inline void row_launch(const Grid& g, uint32_t& nkb, uint32_t& nblocks, uint32_t& bk, int bmax) {
    nkb = (uint32_t)((g.zg1 + bmax - 1) / bmax);
    const uint32_t per = ((uint32_t)g.zg1 + nkb - 1) / nkb;
    bk = (per + 63u) / 64u * 64u;
    nblocks = nkb * (uint32_t)g.yg1 * (uint32_t)g.xg1;
}

// Rows of k that are not whole wavefronts leave lanes idle (131: 192 lanes a row);
// over the cells of a plane back to back nearly none are, at the price of a
// division and its own j per lane.  The line, from both mappings at 56 edges from
// 24 to 448 (stream-collide, us, rows -> flat):
//   rows that waste a tenth of their lanes or more gain while the memory does not
//   bound the step: FP32 70^3 22 -> 17, 131^3 79 -> 71, 270^3 636 -> 617, 330^3 1150
//   -> 1113 but Simple 1231 -> 1235; FP16 70^3 18 -> 14, 131^3 49 -> 40, 270^3 343 ->
//   334, 330^3 Simple 686 -> 697: below 2^25 cells.  FP64 131^3 137 -> 128, but 170^3
//   285 -> 290, and rows within a wavefront 36^3 12.0 -> 12.4: 65 to 2^22 cells;
//   16-bit storage is bound by its arithmetic and gains with any idle lane (60^3 15.1
//   -> 13.7, 120^3 35 -> 33) up to 2^22 cells (184^3 122 -> 122);
//   rows of whole lines keep their streaming hints (hints: 224^3 FP32 292 against 337
//   flat, 144^3 FP64 154 against 172), but for small lattices (96^3 FP32 34.6 -> 30.7).
bool flat_tile(const Grid& g, size_t ssize, bool hints, FlatTile& tile, uint32_t& nblocks, uint32_t& bk) {
    const uint64_t row = (uint64_t)g.zg1, lanes = (row + 63) / 64 * 64, plane = row * (uint64_t)g.yg1;
    const uint64_t cells = plane * (uint64_t)g.xg1;
    if (row < 2 || row == lanes || plane * row >= (1ull << 32) || (hints && cells >= (1ull << 20))) return false;
    const bool waste = 10 * row <= 9 * lanes;
    const bool gains = ssize > 4   ? waste && row > 64 && cells < (1ull << 22)
                       : ssize < 4 ? cells < (1ull << 22) || (waste && cells < (1ull << 25))
                                   : waste && cells < (1ull << 25);
    if (!gains) return false;
    bk = kFlatBlock;
    tile.blocks = (uint32_t)((plane + bk - 1) / bk);
    tile.recip = (uint32_t)(((1ull << 32) + row - 1) / row);
    nblocks = tile.blocks * (uint32_t)g.xg1;
    return true;
}

template <typename PR>
hipError_t esotwist_t(int mode, int even, void* Q, void* mout, const void* F, void* Nu, const uint64_t* fm,
                      const Grid& g, const CollideArgs& c, float rho0, hipStream_t s) {
    using S = typename PR::S;
    using T = typename PR::T;
    uint32_t nkb, nb, bk;
    row_launch(g, nkb, nb, bk, row_block_max<S>());
    S* q = static_cast<S*>(Q);
    T* mo = static_cast<T*>(mout);
    const T* f = static_cast<const T*>(F);
    auto* nu = static_cast<typename PR::N*>(Nu);
    const auto P = to_params<T, typename PR::D>(c);
#define TDLB_ESO(M, E, H) \
    hipLaunchKernelGGL((k_esotwist<PR, M, E, H>), dim3(nb), dim3(bk), 0, s, q, mo, f, nu, fm, g, P, nkb, rho0)
    if (mode == MODE_COLL) { if (even) TDLB_ESO(MODE_COLL, 1, false); else TDLB_ESO(MODE_COLL, 0, false); }
    else if (mode == MODE_MOM) { if (even) TDLB_ESO(MODE_MOM, 1, false); else TDLB_ESO(MODE_MOM, 0, false); }
    else if (mode == MODE_FUSED) {
        FlatTile tile;
        if (flat_tile(g, sizeof(S), line_rows<S>(g), tile, nb, bk)) {
            auto* k = even ? &k_esotwist_flat<PR, 1> : &k_esotwist_flat<PR, 0>;
            hipLaunchKernelGGL(k, dim3(nb), dim3(bk), 0, s, q, f, nu, fm, g, P, tile, rho0);
            return hipGetLastError();
        }
        if (line_rows<S>(g)) {
            if (even) TDLB_ESO(MODE_FUSED, 1, true); else TDLB_ESO(MODE_FUSED, 0, true);
            return hipGetLastError();
        }
        if (even) TDLB_ESO(MODE_FUSED, 1, false); else TDLB_ESO(MODE_FUSED, 0, false);
    }
    else return hipErrorInvalidValue;
#undef TDLB_ESO
    return hipGetLastError();
}

template <typename PR>
hipError_t simple_t(int mode, const void* src, void* dst, void* mout, const void* F, void* Nu, const uint64_t* fm,
                    const Grid& g, const CollideArgs& c, float rho0, hipStream_t s) {
    using S = typename PR::S;
    using T = typename PR::T;
    uint32_t nkb, nb, bk;
    row_launch(g, nkb, nb, bk, row_block_max<S>());
    const S* a = static_cast<const S*>(src);
    S* b = static_cast<S*>(dst);
    T* mo = static_cast<T*>(mout);
    const T* f = static_cast<const T*>(F);
    auto* nu = static_cast<typename PR::N*>(Nu);
    const auto P = to_params<T, typename PR::D>(c);
#define TDLB_SIM(M) \
    hipLaunchKernelGGL((k_simple<PR, M>), dim3(nb), dim3(bk), 0, s, a, b, mo, f, nu, fm, g, P, nkb, rho0)
    switch (mode) {
        case MODE_COLL: TDLB_SIM(MODE_COLL); break;
        case MODE_MOM: TDLB_SIM(MODE_MOM); break;
        case MODE_FUSED: {
            FlatTile tile;
            if (flat_tile(g, sizeof(S), false, tile, nb, bk))
                hipLaunchKernelGGL(k_simple_flat<PR>, dim3(nb), dim3(bk), 0, s, a, b, f, nu, fm, g, P, tile, rho0);
            else TDLB_SIM(MODE_FUSED);
            break;
        }
        case MODE_MOM_PULL: TDLB_SIM(MODE_MOM_PULL); break;
        default: return hipErrorInvalidValue;
    }
#undef TDLB_SIM
    return hipGetLastError();
}

}  // namespace

// precision index -> traits: 0 fp32, 1 fp64, 2 fp16 storage, 3 bf16 storage,
// 4 e3m12 storage (the C ABI validates the index at tdlb_cu_create)
#define TDLB_WITH_PREC(prec, ...)                      \
    do {                                               \
        switch (prec) {                                \
            case 0: { using PR = PrecF32; __VA_ARGS__; } break;  \
            case 1: { using PR = PrecF64; __VA_ARGS__; } break;  \
            case 2: { using PR = PrecF16; __VA_ARGS__; } break;  \
            case 3: { using PR = PrecBF16; __VA_ARGS__; } break; \
            default: { using PR = PrecE3M12; __VA_ARGS__; } break; \
        }                                              \
    } while (0)

// ====================================================================== launchers
hipError_t launch_fill_q(int prec, void* Q, const Grid& g, double rho, hipStream_t s) {
    const uint32_t nb = grid_blocks(g.qsize * kQ);
    if (prec == 0) hipLaunchKernelGGL(k_fill_q<float>, dim3(nb), dim3(kBlock), 0, s, (float*)Q, g, (float)rho);
    else hipLaunchKernelGGL(k_fill_q<double>, dim3(nb), dim3(kBlock), 0, s, (double*)Q, g, rho);
    return hipGetLastError();
}

namespace {
template <typename W>
hipError_t q_boundary_t(int blayout, bool to_boundary, void* Q, void* dense, uint64_t begin, uint64_t end,
                        const Grid& g, hipStream_t s) {
    const dim3 nb(grid_blocks(end - begin)), bs(kBlock);
    W* q = static_cast<W*>(Q);
    W* d = static_cast<W*>(dense);
    if (blayout == LayoutIJKL) {
        if (to_boundary) hipLaunchKernelGGL((k_q_boundary<W, LayoutIJKL, true>), nb, bs, 0, s, q, d, begin, end, g);
        else hipLaunchKernelGGL((k_q_boundary<W, LayoutIJKL, false>), nb, bs, 0, s, q, d, begin, end, g);
    } else {
        if (to_boundary) hipLaunchKernelGGL((k_q_boundary<W, LayoutLIJK, true>), nb, bs, 0, s, q, d, begin, end, g);
        else hipLaunchKernelGGL((k_q_boundary<W, LayoutLIJK, false>), nb, bs, 0, s, q, d, begin, end, g);
    }
    return hipGetLastError();
}
}  // namespace

hipError_t launch_q_boundary(int esize, int blayout, int to_boundary, void* Q, void* dense, uint64_t begin,
                             uint64_t end, const Grid& g, hipStream_t s) {
    if (begin >= end) return hipSuccess;
    if (esize == 4) return q_boundary_t<uint32_t>(blayout, to_boundary != 0, Q, dense, begin, end, g, s);
    if (esize == 8) return q_boundary_t<uint64_t>(blayout, to_boundary != 0, Q, dense, begin, end, g, s);
    return hipErrorInvalidValue;
}

// Speed of light of the stream-collide access pattern: one pass reads the
// value of every lane's cell from each of `planes` planes, then writes each
// back with its bits flipped by a run-time mask (so no load or store folds
// away; two passes restore the data).  Blocks of kRowBlock lanes, as the
// stream-collide rows.
constexpr int kProbePlanesMax = 20;
template <typename U, bool NT>
__global__ __launch_bounds__(kRowBlock) void k_probe_planes(U* __restrict__ base, uint64_t stride, uint64_t n,
                                                            int planes, U mask) {
    const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    U v[kProbePlanesMax];
#pragma unroll
    for (int p = 0; p < kProbePlanesMax; p++)
        if (p < planes) v[p] = load_hint<NT>(base + (uint64_t)p * stride + c);
#pragma unroll
    for (int p = 0; p < kProbePlanesMax; p++)
        if (p < planes) store_hint<NT>(base + (uint64_t)p * stride + c, (U)(v[p] ^ mask));
}

template <typename U>
hipError_t probe_t(void* base, uint64_t stride, uint64_t n, int planes, int nt, hipStream_t s) {
    const uint32_t nb = (uint32_t)((n + kRowBlock - 1) / kRowBlock);
    const U mask = (U)0x5555555555555555ull;
    if (nt) hipLaunchKernelGGL((k_probe_planes<U, true>), dim3(nb), dim3(kRowBlock), 0, s, (U*)base, stride, n, planes, mask);
    else hipLaunchKernelGGL((k_probe_planes<U, false>), dim3(nb), dim3(kRowBlock), 0, s, (U*)base, stride, n, planes, mask);
    return hipGetLastError();
}

hipError_t launch_probe_planes(int elem_bytes, void* base, uint64_t stride, uint64_t n, int planes, int nt,
                               hipStream_t s) {
    if (planes < 1 || planes > kProbePlanesMax || n == 0 || (n + kRowBlock - 1) / kRowBlock > 0x7fffffffull)
        return hipErrorInvalidValue;
    if (elem_bytes == 2) return probe_t<uint16_t>(base, stride, n, planes, nt, s);
    if (elem_bytes == 4) return probe_t<uint32_t>(base, stride, n, planes, nt, s);
    if (elem_bytes == 8) return probe_t<uint64_t>(base, stride, n, planes, nt, s);
    return hipErrorInvalidValue;
}

hipError_t launch_zero(void* p, size_t bytes, hipStream_t s) {
    if (bytes == 0) return hipSuccess;
    if (bytes % 4 == 0 && ((uintptr_t)p % 4) == 0)
        hipLaunchKernelGGL(k_zero_words, dim3(grid_blocks(bytes / 4)), dim3(kBlock), 0, s, (uint32_t*)p, (uint64_t)(bytes / 4));
    else
        hipLaunchKernelGGL(k_zero_bytes, dim3(grid_blocks(bytes)), dim3(kBlock), 0, s, (uint8_t*)p, (uint64_t)bytes);
    return hipGetLastError();
}

hipError_t launch_copy(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (bytes == 0) return hipSuccess;
    if (bytes % 4 == 0 && ((uintptr_t)dst % 4) == 0 && ((uintptr_t)src % 4) == 0)
        hipLaunchKernelGGL(k_copy_words, dim3(grid_blocks(bytes / 4)), dim3(kBlock), 0, s, (uint32_t*)dst,
                           (const uint32_t*)src, (uint64_t)(bytes / 4));
    else
        hipLaunchKernelGGL(k_copy_bytes, dim3(grid_blocks(bytes)), dim3(kBlock), 0, s, (uint8_t*)dst,
                           (const uint8_t*)src, (uint64_t)bytes);
    return hipGetLastError();
}

hipError_t launch_esotwist(int prec, int mode, int even, void* Q, void* mout, const void* F, void* Nu,
                           const uint64_t* fmask, const Grid& g, const CollideArgs& c, float rho0, hipStream_t s) {
    hipError_t e = hipErrorInvalidValue;
    TDLB_WITH_PREC(prec, e = esotwist_t<PR>(mode, even, Q, mout, F, Nu, fmask, g, c, rho0, s));
    return e;
}

hipError_t launch_simple(int prec, int mode, const void* src, void* dst, void* mout, const void* F,
                         void* Nu, const uint64_t* fmask, const Grid& g, const CollideArgs& c, float rho0,
                         hipStream_t s) {
    hipError_t e = hipErrorInvalidValue;
    TDLB_WITH_PREC(prec, e = simple_t<PR>(mode, src, dst, mout, F, Nu, fmask, g, c, rho0, s));
    return e;
}

// launch KERNEL<W> over NTHREADS grid-stride threads
#define TDLB_MOVE(KERNEL, W, NTHREADS, ...) \
    hipLaunchKernelGGL(KERNEL<W>, dim3(grid_blocks(NTHREADS)), dim3(kBlock), 0, s, __VA_ARGS__)

hipError_t launch_push_all(int esize, const void* src, void* dst, const Grid& g, hipStream_t s) {
    if (esize == 4) TDLB_MOVE(k_push_all, uint32_t, g.size, (const uint32_t*)src, (uint32_t*)dst, g);
    else TDLB_MOVE(k_push_all, uint64_t, g.size, (const uint64_t*)src, (uint64_t*)dst, g);
    return hipGetLastError();
}

hipError_t launch_pull_all(int esize, const void* src, void* dst, const Grid& g, hipStream_t s) {
    if (esize == 4) TDLB_MOVE(k_pull_all, uint32_t, g.size, (const uint32_t*)src, (uint32_t*)dst, g);
    else TDLB_MOVE(k_pull_all, uint64_t, g.size, (const uint64_t*)src, (uint64_t*)dst, g);
    return hipGetLastError();
}

hipError_t launch_bounce_back(int esize, void* Q, const Grid& g, hipStream_t s) {
    const uint64_t x = (uint64_t)g.xg1, y = (uint64_t)g.yg1, z = (uint64_t)g.zg1;
    const uint64_t n = 2 * (y * z + x * z + x * y) + 12 * std::max(x, std::max(y, z));
    if (esize == 4) TDLB_MOVE(k_bounce_back, uint32_t, n, (uint32_t*)Q, g);
    else TDLB_MOVE(k_bounce_back, uint64_t, n, (uint64_t*)Q, g);
    return hipGetLastError();
}

hipError_t launch_ghost_fill(int esize, const void* src, void* dst, const Grid& g, hipStream_t s) {
    if (esize == 4)
        TDLB_MOVE(k_ghost_fill, RawBits<uint32_t>, ghost_count(g), (const uint32_t*)src, (uint32_t*)dst, g, 0.0f);
    else
        TDLB_MOVE(k_ghost_fill, RawBits<uint64_t>, ghost_count(g), (const uint64_t*)src, (uint64_t*)dst, g, 0.0f);
    return hipGetLastError();
}

hipError_t launch_ghost_fill_decode(int prec, const void* src, void* dst, const Grid& g, float rho0,
                                    hipStream_t s) {
    if (prec == 2)
        TDLB_MOVE(k_ghost_fill, PrecF16, ghost_count(g), (const PrecF16::S*)src, (float*)dst, g, rho0);
    else if (prec == 3)
        TDLB_MOVE(k_ghost_fill, PrecBF16, ghost_count(g), (const PrecBF16::S*)src, (float*)dst, g, rho0);
    else if (prec == 4)
        TDLB_MOVE(k_ghost_fill, PrecE3M12, ghost_count(g), (const PrecE3M12::S*)src, (float*)dst, g, rho0);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_ghost_copy(int esize, const void* src, void* dst, const Grid& g, hipStream_t s) {
    if (esize == 4) TDLB_MOVE(k_ghost_copy, uint32_t, ghost_count(g), (const uint32_t*)src, (uint32_t*)dst, g);
    else TDLB_MOVE(k_ghost_copy, uint64_t, ghost_count(g), (const uint64_t*)src, (uint64_t*)dst, g);
    return hipGetLastError();
}
#undef TDLB_MOVE

hipError_t launch_mask_from_f(int prec, const void* F, uint64_t* mask, uint64_t* gmask, const Grid& g,
                              hipStream_t s) {
    const uint64_t words = (uint64_t)g.xg * g.yg * g.mask_w;
    if (prec != 1) hipLaunchKernelGGL(k_mask_from_f<float>, dim3(grid_blocks(words)), dim3(kBlock), 0, s, (const float*)F, mask, gmask, g);
    else hipLaunchKernelGGL(k_mask_from_f<double>, dim3(grid_blocks(words)), dim3(kBlock), 0, s, (const double*)F, mask, gmask, g);
    return hipGetLastError();
}

hipError_t launch_masked_f(int prec, const void* F, const uint64_t* mask, uint64_t begin, uint64_t end, void* out,
                           const Grid& g, hipStream_t s) {
    if (begin >= end) return hipSuccess;
    const dim3 nb(grid_blocks(end - begin)), bs(kBlock);
    if (prec != 1) hipLaunchKernelGGL(k_masked_f<float>, nb, bs, 0, s, (const float*)F, mask, begin, end, (float*)out, g);
    else hipLaunchKernelGGL(k_masked_f<double>, nb, bs, 0, s, (const double*)F, mask, begin, end, (double*)out, g);
    return hipGetLastError();
}

hipError_t launch_zero_interior_o(uint8_t* O, const Grid& g, hipStream_t s) {
    hipLaunchKernelGGL(k_zero_interior_o, dim3(grid_blocks(g.size)), dim3(kBlock), 0, s, O, g);
    return hipGetLastError();
}

hipError_t launch_force_prepare(int prec, const PointsDev& p, int64_t begin, int64_t count, void* F,
                                const uint64_t* prev, uint64_t* next, const Grid& g, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    const uint32_t nb = (uint32_t)((count + kBlock - 1) / kBlock);
    if (prec != 1) hipLaunchKernelGGL(k_force_prepare<float>, dim3(nb), dim3(kBlock), 0, s, p, begin, count, (float*)F, prev, next, g);
    else hipLaunchKernelGGL(k_force_prepare<double>, dim3(nb), dim3(kBlock), 0, s, p, begin, count, (double*)F, prev, next, g);
    return hipGetLastError();
}

template <int V>
using IC = std::integral_constant<int, V>;

hipError_t launch_list_unpack(int prec, const tdlb_ib_point* in, int64_t n, int ghost, const PointsDev& p,
                              const uint64_t* base, uint64_t* next, uint64_t words, hipStream_t s) {
    const dim3 nb(grid_blocks(std::max<uint64_t>((uint64_t)n, words))), bs(kBlock);
    if (prec != 1) hipLaunchKernelGGL(k_list_unpack<float>, nb, bs, 0, s, in, n, ghost, p, base, next, words);
    else hipLaunchKernelGGL(k_list_unpack<double>, nb, bs, 0, s, in, n, ghost, p, base, next, words);
    return hipGetLastError();
}

// At most this many workgroups where the LDS holds the marks: four times what the chip
// holds at once.  With a workgroup for each of 100,000 planes of 16 x 16 cells and 300
// points a call took 1.0 ms, most of it for planes without any.
constexpr int kListBlocks = 4096;
size_t list_marks_bytes(const Grid& g, int* blocks) {
    const size_t plane = (size_t)g.xg1 * g.zg1 * sizeof(uint32_t);
    const bool lds = plane <= kListLdsBytes;
    // a workgroup per plane at a time; with marks in HBM at most one per CU
    *blocks = std::min(g.yg1, lds ? kListBlocks : 256);
    return lds ? 0 : plane;
}

// A launch of a list kernel may ask for more than 64 KB of LDS: the same most for every
// grid, so that threads with planes of different sizes never lower another's.
static hipError_t allow_list_lds(const void* kernel) {
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kListLdsBytes);
}

hipError_t launch_list_levels(const PointsDev& p, int64_t n, int64_t* list, uint32_t* marks, int blocks, int32_t* lev,
                              const Grid& g, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    int most = 0;
    const size_t hbm = list_marks_bytes(g, &most);
    if ((hbm != 0) != (marks != nullptr) || blocks < 1 || blocks > most) return hipErrorInvalidValue;
    const uint32_t lds = hbm ? 0u : (uint32_t)((size_t)g.xg1 * g.zg1 * sizeof(uint32_t));
    auto* k = hbm ? &k_list_levels<false> : &k_list_levels<true>;
    if (lds > 64 * 1024) {
        const hipError_t e = allow_list_lds(reinterpret_cast<const void*>(k));
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k, dim3((uint32_t)blocks), dim3(kListBlock), lds, s, p, n, list, marks, lev, g);
    return hipGetLastError();
}

hipError_t launch_list_planes(int prec, int streaming, int even, const PointsDev& p, int64_t n, int64_t* list,
                              uint32_t* marks, int blocks, const void* Q, void* F, const uint64_t* prev,
                              uint64_t* next, const Grid& g, double alfa, double beta, float rho0, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    int most = 0;
    const size_t hbm = list_marks_bytes(g, &most);
    if ((hbm != 0) != (marks != nullptr) || blocks < 1 || blocks > most) return hipErrorInvalidValue;
    const uint32_t lds = hbm ? 0u : (uint32_t)((size_t)g.xg1 * g.zg1 * sizeof(uint32_t));
    auto go = [&](auto pr, auto Sc, auto Ec) -> hipError_t {
        using PR = decltype(pr);
        using T = typename PR::T;
        constexpr int S = decltype(Sc)::value, E = decltype(Ec)::value;
        auto* k = hbm ? &k_list_planes<PR, S, E, false> : &k_list_planes<PR, S, E, true>;
        if (lds > 64 * 1024) {
            const hipError_t e = allow_list_lds(reinterpret_cast<const void*>(k));
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(k, dim3((uint32_t)blocks), dim3(kListBlock), lds, s, p, n, list, marks, (T*)F, (const T*)Q, prev,
                           next, g, (T)alfa, (T)beta, rho0);
        return hipGetLastError();
    };
    auto by_stream = [&](auto pr) {
        if (streaming != StreamEsotwist) return go(pr, IC<StreamSimple>{}, IC<1>{});  // plain addressing
        return even ? go(pr, IC<StreamEsotwist>{}, IC<1>{}) : go(pr, IC<StreamEsotwist>{}, IC<0>{});
    };
    if (prec == 0) return by_stream(PrecF32{});
    if (prec == 1) return by_stream(PrecF64{});
    return hipErrorInvalidValue;
}

namespace {
// fn(STREAM, MOMSRC, EVEN) with compile-time values (std::integral_constant)

template <typename PR, int STREAM, typename Fn>
hipError_t with_source(int momsrc, int even, Fn&& fn) {
    if (momsrc == MOMSRC_STORED) {
        if constexpr (PR::kShift) return hipErrorInvalidValue;
        else return even ? fn(IC<STREAM>{}, IC<MOMSRC_STORED>{}, IC<1>{})
                         : fn(IC<STREAM>{}, IC<MOMSRC_STORED>{}, IC<0>{});
    }
    if (momsrc == MOMSRC_ESO_POPS) {
        if constexpr (STREAM != StreamEsotwist) return hipErrorInvalidValue;
        else return even ? fn(IC<STREAM>{}, IC<MOMSRC_ESO_POPS>{}, IC<1>{})
                         : fn(IC<STREAM>{}, IC<MOMSRC_ESO_POPS>{}, IC<0>{});
    }
    if constexpr (STREAM != StreamSimple) return hipErrorInvalidValue;
    else return fn(IC<STREAM>{}, IC<MOMSRC_PULL_POPS>{}, IC<1>{});
}

template <typename PR, typename Fn>
hipError_t with_cell_source(int streaming, int momsrc, int even, Fn&& fn) {
    return streaming == StreamEsotwist ? with_source<PR, StreamEsotwist>(momsrc, even, fn)
                                       : with_source<PR, StreamSimple>(momsrc, even, fn);
}
}  // namespace

hipError_t launch_force_gather(int prec, int streaming, int momsrc, int even, const ForceGeom& fg,
                               const BladeStep& st, const GatherBlocks& gb, const void* Q, void* F,
                               const uint64_t* prev, uint64_t* next, const uint64_t* static_base, const Grid& g,
                               float rho0, hipStream_t s) {
    const uint32_t nb = gb.blades + gb.cells + gb.words;
    if (nb == 0) return hipSuccess;
    hipError_t e = hipErrorInvalidValue;
    TDLB_WITH_PREC(prec, {
        using S = typename PR::S;
        using T = typename PR::T;
        e = with_cell_source<PR>(streaming, momsrc, even, [&](auto Sc, auto Mc, auto Ec) {
            hipLaunchKernelGGL((k_force_gather<PR, decltype(Sc)::value, decltype(Mc)::value,
                                               decltype(Ec)::value>),
                               dim3(nb), dim3(kGatherBlock), 0, s, fg, st, gb, (const S*)Q, (T*)F, prev, next,
                               static_base, g, rho0);
            return hipGetLastError();
        });
    });
    return e;
}

hipError_t launch_force_levels(int prec, const ForceGeom& fg, void* F, uint64_t* next, const Grid& g, double alfa,
                               double beta, hipStream_t s) {
    if (fg.n_planes <= 0) return hipSuccess;
    const dim3 grid((uint32_t)fg.n_planes), block((uint32_t)fg.level_lanes);
    if (prec == 1)
        hipLaunchKernelGGL(k_force_levels<double>, grid, block, fg.level_lds, s, fg, (double*)F, next, g, alfa, beta,
                           (int64_t)fg.level_lds);
    else
        hipLaunchKernelGGL(k_force_levels<float>, grid, block, fg.level_lds, s, fg, (float*)F, next, g, (float)alfa,
                           (float)beta, (int64_t)fg.level_lds);
    return hipGetLastError();
}

// Launches may ask for up to the whole LDS of a CU.
hipError_t allow_level_lds(int prec) {
    const void* k = prec == 1 ? reinterpret_cast<const void*>(&k_force_levels<double>)
                              : reinterpret_cast<const void*>(&k_force_levels<float>);
    return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kCuLdsBytes);
}

bool line_rows_bytes(const Grid& g, size_t ssize) {
    return ssize == 4 ? line_rows<float>(g) : line_rows<_Float16>(g);
}

// the pipe's row blocks take at most 256 lanes: 4 waves, so that several
// workgroups share a CU at the register count of the stream-collide code
constexpr int kPipeLanes = 256;
uint32_t row_lanes(const Grid& g) {
    uint32_t nkb, nb, bk;
    row_launch(g, nkb, nb, bk, kPipeLanes);
    return bk;
}

hipError_t launch_eso_pipe(int prec, int even, int hint, const PipeArgs& a, const Grid& g, const CollideArgs& c,
                           float rho0, uint32_t blocks, uint32_t lanes, hipStream_t s) {
    uint32_t nkb, nb, bk;
    row_launch(g, nkb, nb, bk, kPipeLanes);
    if (lanes != bk) return hipErrorInvalidValue;
    auto go = [&](auto pr) -> hipError_t {
        using PR = decltype(pr);
        const auto P = to_params<float, typename PR::D>(c);
#define TDLB_PIPE(E, H) hipLaunchKernelGGL((k_eso_pipe<PR, E, H>), dim3(blocks), dim3(bk), 0, s, a, g, P, nkb, rho0)
        if (blocks == 0) {
            // persistent grid: every workgroup resident at once
            int per_cu = 0, dev = 0;
            hipDeviceProp_t prop;
            if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess ||
                hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_eso_pipe<PR, 1, true>, (int)bk, 0) !=
                    hipSuccess)
                return hipErrorInvalidValue;
            // at least 8 per CU: workgroups beyond the resident ones find the queues drained
            blocks = (uint32_t)std::max(8, per_cu) * (uint32_t)prop.multiProcessorCount;
        }
        if (even) { if (hint) TDLB_PIPE(1, true); else TDLB_PIPE(1, false); }
        else { if (hint) TDLB_PIPE(0, true); else TDLB_PIPE(0, false); }
#undef TDLB_PIPE
        return hipGetLastError();
    };
    switch (prec) {
        case 0: return go(PrecF32{});
        case 2: return go(PrecF16{});
        case 3: return go(PrecBF16{});
        case 4: return go(PrecE3M12{});
        default: return hipErrorInvalidValue;
    }
}

int pipe_xcc_check(hipStream_t s) {
    constexpr int nb = 64 * kXcds;
    uint32_t* d = nullptr;
    if (hipMalloc((void**)&d, nb * sizeof(uint32_t)) != hipSuccess) return 0;
    hipLaunchKernelGGL(k_xcc_ids, dim3(nb), dim3(64), 0, s, d);
    uint32_t h[nb];
    const bool ok = hipGetLastError() == hipSuccess &&
                    hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, s) == hipSuccess &&
                    hipStreamSynchronize(s) == hipSuccess;
    (void)hipFree(d);
    if (!ok) return 0;
    int seen[kXcds] = {0};
    for (int b = 0; b < nb; b++) {
        if (h[b] >= (uint32_t)kXcds) return 0;
        seen[h[b]]++;
    }
    for (int x = 0; x < kXcds; x++)
        if (seen[x] == 0) return 0;
    return 1;
}

hipError_t launch_reduce(int prec, int streaming, int momsrc, int even, const void* Q, const void* F,
                         const uint64_t* fmask, const Grid& g, const ReduceArgs& ra, float rho0, double* partial,
                         double* out, hipStream_t s) {
    hipError_t e = hipErrorInvalidValue;
    TDLB_WITH_PREC(prec, {
        using S = typename PR::S;
        using T = typename PR::T;
        e = with_cell_source<PR>(streaming, momsrc, even, [&](auto Sc, auto Mc, auto Ec) {
            hipLaunchKernelGGL((k_reduce_cells<PR, decltype(Sc)::value, decltype(Mc)::value,
                                               decltype(Ec)::value>),
                               dim3(kReduceBlocks), dim3(kBlock), 0, s, (const S*)Q, (const T*)F, fmask, g, ra, rho0,
                               partial);
            return hipGetLastError();
        });
    });
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(kReduceFinalBlock), 0, s, partial, out);
    return hipGetLastError();
}

hipError_t launch_macroscopic(int prec, int streaming, int momsrc, int even, const void* Q, const void* F,
                              const uint64_t* fmask, const Grid& g, float rho0, uint64_t begin, uint64_t end, void* out,
                              hipStream_t s) {
    if (begin >= end) return hipSuccess;
    const uint32_t nb = grid_blocks(end - begin);
    hipError_t e = hipErrorInvalidValue;
    TDLB_WITH_PREC(prec, {
        using S = typename PR::S;
        using T = typename PR::T;
        e = with_cell_source<PR>(streaming, momsrc, even, [&](auto Sc, auto Mc, auto Ec) {
            hipLaunchKernelGGL((k_macroscopic<PR, decltype(Sc)::value, decltype(Mc)::value, decltype(Ec)::value>),
                               dim3(nb), dim3(kBlock), 0, s, (const S*)Q, (const T*)F, fmask, g, rho0, begin, end,
                               (Mom4<T>*)out);
            return hipGetLastError();
        });
    });
    return e;
}

hipError_t launch_regrid(int esize, const void* oldQ, void* newQ, int nu_esize, const void* oldNu,
                         void* newNu, const Grid& og, const Grid& ng, hipStream_t s) {
    const uint32_t nb = grid_blocks(ng.size);
    if (esize == 4) {
        hipLaunchKernelGGL((k_regrid_q<uint32_t>), dim3(nb), dim3(kBlock), 0, s, (const uint32_t*)oldQ, (uint32_t*)newQ, og, ng);
    } else if (esize == 8) {
        hipLaunchKernelGGL((k_regrid_q<uint64_t>), dim3(nb), dim3(kBlock), 0, s, (const uint64_t*)oldQ, (uint64_t*)newQ, og, ng);
    } else {
        return hipErrorInvalidValue;
    }
    if (nu_esize == 2)
        hipLaunchKernelGGL(k_regrid_cells<uint16_t>, dim3(nb), dim3(kBlock), 0, s, (const uint16_t*)oldNu, (uint16_t*)newNu, og, ng);
    else if (nu_esize == 4)
        hipLaunchKernelGGL(k_regrid_cells<uint32_t>, dim3(nb), dim3(kBlock), 0, s, (const uint32_t*)oldNu, (uint32_t*)newNu, og, ng);
    else if (nu_esize == 8)
        hipLaunchKernelGGL(k_regrid_cells<uint64_t>, dim3(nb), dim3(kBlock), 0, s, (const uint64_t*)oldNu, (uint64_t*)newNu, og, ng);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

namespace {
// Nu between the 16-bit storage of prec 2/3/4 and the float array of the boundary
template <typename PR, bool TO_FLOAT>
__global__ void k_nu_convert(const void* __restrict__ src, void* __restrict__ dst, uint64_t n) {
    for (uint64_t a = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; a < n; a += (uint64_t)gridDim.x * blockDim.x) {
        if (TO_FLOAT) static_cast<float*>(dst)[a] = PR::dec_nu(static_cast<const typename PR::N*>(src)[a]);
        else static_cast<typename PR::N*>(dst)[a] = PR::enc_nu(static_cast<const float*>(src)[a]);
    }
}
}  // namespace

hipError_t launch_nu_convert(int prec, int to_float, const void* src, void* dst, uint64_t n, hipStream_t s) {
    const uint32_t nb = grid_blocks(n);
    if (prec == 2) {
        if (to_float) hipLaunchKernelGGL((k_nu_convert<PrecF16, true>), dim3(nb), dim3(kBlock), 0, s, src, dst, n);
        else hipLaunchKernelGGL((k_nu_convert<PrecF16, false>), dim3(nb), dim3(kBlock), 0, s, src, dst, n);
    } else if (prec == 3) {
        if (to_float) hipLaunchKernelGGL((k_nu_convert<PrecBF16, true>), dim3(nb), dim3(kBlock), 0, s, src, dst, n);
        else hipLaunchKernelGGL((k_nu_convert<PrecBF16, false>), dim3(nb), dim3(kBlock), 0, s, src, dst, n);
    } else if (prec == 4) {
        if (to_float) hipLaunchKernelGGL((k_nu_convert<PrecE3M12, true>), dim3(nb), dim3(kBlock), 0, s, src, dst, n);
        else hipLaunchKernelGGL((k_nu_convert<PrecE3M12, false>), dim3(nb), dim3(kBlock), 0, s, src, dst, n);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_plane_xz(int prec, const void* Q, const void* F, const uint64_t* fmask,
                           const uint8_t* exclude, const Grid& g, int cut, int64_t i0, int64_t k0, PlaneRec4* q,
                           PlaneRec3* f, uint8_t* flags, hipStream_t s) {
    const uint32_t nb = (uint32_t)(((int64_t)g.xg1 * g.zg1 + kBlock - 1) / kBlock);
#define TDLB_PLANE(T)                                                                                          \
    hipLaunchKernelGGL((k_plane_xz<T>), dim3(nb), dim3(kBlock), 0, s, (const T*)Q, (const T*)F, fmask, exclude, \
                       g, cut, i0, k0, q, f, flags)
    if (prec == 1) {
        TDLB_PLANE(double);
    } else {
        TDLB_PLANE(float);
    }
#undef TDLB_PLANE
    return hipGetLastError();
}

hipError_t launch_vorticity(int prec, int streaming, int momsrc, int even, const void* Q, const Grid& g,
                            int axis, int cut, const uint8_t* exclude, void* out, float rho0, hipStream_t s) {
    const int64_t cells = (int64_t)g.xg1 * (axis == 0 ? g.zg1 : g.yg1);
    const uint32_t nb = (uint32_t)((cells + kBlock - 1) / kBlock);
    hipError_t e = hipErrorInvalidValue;
    TDLB_WITH_PREC(prec, {
        using S = typename PR::S;
        using T = typename PR::T;
        e = with_cell_source<PR>(streaming, momsrc, even, [&](auto Sc, auto Mc, auto Ec) {
            hipLaunchKernelGGL((k_vorticity<PR, decltype(Sc)::value, decltype(Mc)::value,
                                            decltype(Ec)::value>),
                               dim3(nb), dim3(kBlock), 0, s, (const S*)Q, g, axis, cut, exclude, (T*)out, rho0);
            return hipGetLastError();
        });
    });
    return e;
}

hipError_t launch_static_rows(int prec, const PointsDev& p, int64_t n, const int32_t* sidx, void* rows, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const uint32_t nb = (uint32_t)((3 * n + kBlock - 1) / kBlock);
    if (prec != 1) hipLaunchKernelGGL(k_static_rows<float>, dim3(nb), dim3(kBlock), 0, s, p, n, sidx, (ForceRow<float>*)rows);
    else hipLaunchKernelGGL(k_static_rows<double>, dim3(nb), dim3(kBlock), 0, s, p, n, sidx, (ForceRow<double>*)rows);
    return hipGetLastError();
}

hipError_t launch_solid_mask(double cx, double cz, double radius, uint8_t* out, const Grid& g, int ghost,
                             hipStream_t s) {
    hipLaunchKernelGGL(k_solid_mask, dim3(grid_blocks(g.size)), dim3(kBlock), 0, s, cx, cz, radius, out, g, ghost);
    return hipGetLastError();
}

// ====================================================================== batches
// Each kernel below runs the per-member body of the single-handle kernel above
// (same device functions), so a member advances exactly as it would alone.
namespace {

// largest m in [0, n) with off[m] <= x (off non-decreasing, off[0] <= x)
__device__ __forceinline__ int find_slot(const int64_t* __restrict__ off, int n, int64_t x) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= x) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// interior cell of thread threadIdx.x in block b of a member's fused launch
__device__ __forceinline__ bool batch_cell(const Grid& g, int tile, uint32_t b, int& i, int& j, int& k) {
    if (tile == TILE_ROW64) {
        const uint32_t segs = (uint32_t)(g.zg1 + 63) >> 6;
        const uint32_t w = b * (blockDim.x >> 6) + (threadIdx.x >> 6);
        const uint32_t rows = (uint32_t)g.xg1 * (uint32_t)g.yg1;
        if (w >= rows * segs) return false;
        const uint32_t row = w / segs, seg = w - row * segs;
        const uint32_t ii = row / (uint32_t)g.yg1;
        i = (int)ii + 1;
        j = (int)(row - ii * (uint32_t)g.yg1) + 1;
        k = (int)(seg * 64 + (threadIdx.x & 63)) + 1;
        return k <= g.zg1;
    }
    if (tile == TILE_FLAT) {
        const uint32_t plane = (uint32_t)g.yg1 * (uint32_t)g.zg1;
        const uint64_t t = (uint64_t)b * blockDim.x + threadIdx.x;
        if (t >= (uint64_t)g.xg1 * plane) return false;
        const uint32_t ip = (uint32_t)(t / plane), r = (uint32_t)(t - (uint64_t)ip * plane);
        i = (int)ip + 1;
        j = (int)(r / (uint32_t)g.zg1) + 1;
        k = (int)(r - (uint32_t)(j - 1) * (uint32_t)g.zg1) + 1;
        return true;
    }
    const uint32_t plane = (uint32_t)g.yg * (uint32_t)g.zg;
    const uint32_t bpp = (plane + blockDim.x - 1) / blockDim.x;
    const uint32_t ip = b / bpp;
    const uint32_t local = (b - ip * bpp) * blockDim.x + threadIdx.x;
    if (ip >= (uint32_t)g.xg1 || local >= plane) return false;
    i = (int)ip + 1;
    j = (int)(local / (uint32_t)g.zg);
    k = (int)(local - (uint32_t)j * (uint32_t)g.zg);
    return j >= 1 && j <= g.yg1 && k >= 1 && k <= g.zg1;
}

// A member's state `ahead` steps after the one in its descriptor: descriptors
// advance once per recorded sequence of steps, not with a launch in each (a step of
// one 40^3 tank 33.3 -> 32.3 us, of six 64^3 64.7 -> 63.4).
struct MemberStep {
    int64_t done;
    int even, cur, fm;
    bool active;
};
__device__ __forceinline__ MemberStep member_step(const MemberDev& md, int ahead) {
    const int flip = ahead & 1;
    const int64_t done = md.done + ahead;
    return MemberStep{done, md.even ^ flip, md.cur ^ flip, md.fm ^ flip, md.active && done < md.n_steps};
}

template <typename PR, int STREAM>
__global__ __launch_bounds__(kRowBlock) void k_batch_fused(const MemberDev* __restrict__ mem,
                                                        const int64_t* __restrict__ off, int n,
                                                        const int32_t* __restrict__ bm, int ahead) {
    static_assert(std::is_same<typename PR::T, float>::value, "batches compute in float");
    using S = typename PR::S;
    const uint32_t blk = blockIdx.x;
    // one load from the block table instead of a binary search of dependent loads
    const int m = bm ? bm[blk] : find_slot(off, n, blk);
    const MemberDev& md = mem[m];
    const MemberStep ms = member_step(md, ahead);
    if (!ms.active) return;
    int i, j, k;
    if (!batch_cell(md.g, md.tile, (uint32_t)(blk - off[m]), i, j, k)) return;
    const uint64_t* fm = md.fmask[ms.fm];
    if constexpr (STREAM == StreamEsotwist) {
        S* Q = static_cast<S*>(md.Q[0]);
        auto* nu = static_cast<typename PR::N*>(md.Nu);
        if (ms.even) esotwist_cell<PR, MODE_FUSED, 1>(Q, nullptr, md.F, nu, fm, md.g, md.P, md.rho0, i, j, k);
        else esotwist_cell<PR, MODE_FUSED, 0>(Q, nullptr, md.F, nu, fm, md.g, md.P, md.rho0, i, j, k);
    } else {
        simple_cell<PR, MODE_FUSED>(static_cast<const S*>(md.Q[ms.cur]), static_cast<S*>(md.Q[1 - ms.cur]),
                                       nullptr, md.F, static_cast<typename PR::N*>(md.Nu), fm, md.g, md.P,
                                       md.rho0, i, j, k);
    }
}

// the gather of every member (force_gather) from the populations the fused kernel just wrote
template <typename PR, int STREAM>
__global__ __launch_bounds__(kGatherBlock) void k_batch_gather(const MemberDev* __restrict__ mem,
                                                               const int64_t* __restrict__ off,
                                                               const int32_t* __restrict__ bm, int ahead) {
    const int m = bm[blockIdx.x];
    const MemberDev& md = mem[m];
    const MemberStep ms = member_step(md, ahead);
    if (!ms.active) return;
    using S = typename PR::S;
    const uint32_t b = (uint32_t)(blockIdx.x - off[m]);
    const uint64_t* prev = md.fmask[ms.fm];
    uint64_t* next = md.fmask[1 - ms.fm];
    const BladeStep& st = md.steps[ms.done];
    if constexpr (STREAM == StreamEsotwist) {
        const S* Q = static_cast<const S*>(md.Q[0]);
        if (ms.even)
            force_gather<PR, STREAM, MOMSRC_ESO_POPS, 0>(md.fg, st, b, md.gb, Q, md.F, prev, next, md.static_base,
                                                            md.g, md.rho0);
        else
            force_gather<PR, STREAM, MOMSRC_ESO_POPS, 1>(md.fg, st, b, md.gb, Q, md.F, prev, next, md.static_base,
                                                            md.g, md.rho0);
    } else {
        const S* Q = static_cast<const S*>(md.Q[1 - ms.cur]);
        force_gather<PR, STREAM, MOMSRC_PULL_POPS, 1>(md.fg, st, b, md.gb, Q, md.F, prev, next, md.static_base, md.g,
                                                         md.rho0);
    }
}

// the levels of every member's planes: one workgroup per (member, plane) task
__global__ __launch_bounds__(kForcePlaneBlock) void k_batch_levels(const MemberDev* __restrict__ mem,
                                                                   const PlaneTask* __restrict__ tasks,
                                                                   int64_t lds_bytes, int ahead) {
    extern __shared__ float4 batch_lds[];  // lds_bytes, launch-sized
    const PlaneTask tk = tasks[blockIdx.x];
    const MemberDev& md = mem[tk.member];
    const MemberStep ms = member_step(md, ahead);
    if (!ms.active) return;
    const ForceGeom fg = uniform_copy(md.fg);
    const Grid g = uniform_copy(md.g);
    plane_levels<float>(fg, fg.planes + tk.plane, md.F, md.fmask[1 - ms.fm], g, md.alfa, md.beta, batch_lds, lds_bytes);
}

template <int STREAM>
__global__ void k_batch_advance(MemberDev* __restrict__ mem, int n, int steps) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n) return;
    MemberDev& md = mem[m];
    if (!md.active) return;
    const int64_t taken = min((int64_t)steps, md.n_steps - md.done);
    const int flip = (int)(taken & 1);
    md.done += taken;
    if (STREAM == StreamEsotwist) md.even ^= flip;
    else md.cur ^= flip;
    md.fm ^= flip;
    if (md.done >= md.n_steps) md.active = 0;
}

template <typename PR, int STREAM>
hipError_t batch_fused_t(const BatchPlan& p, int ahead, hipStream_t s) {
    if (p.tot_coll <= 0) return hipSuccess;
    hipLaunchKernelGGL((k_batch_fused<PR, STREAM>), dim3((uint32_t)p.tot_coll), dim3(p.bs), 0, s, p.mem,
                       p.off_coll, p.n_members, p.coll_member, ahead);
    return hipGetLastError();
}

template <typename PR, int STREAM>
hipError_t batch_step_t(const BatchPlan& p, int ahead, hipStream_t s) {
    if (p.bs != 256 && p.bs != 512) return hipErrorInvalidValue;
    hipError_t e = batch_fused_t<PR, STREAM>(p, ahead, s);
    if (e != hipSuccess) return e;
    if (p.tot_gather > 0)
        hipLaunchKernelGGL((k_batch_gather<PR, STREAM>), dim3((uint32_t)p.tot_gather), dim3(kGatherBlock), 0, s, p.mem,
                           p.off_gather, p.gather_member, ahead);
    if (p.n_tasks > 0)
        hipLaunchKernelGGL(k_batch_levels, dim3((uint32_t)p.n_tasks), dim3(p.force_bs), (uint32_t)p.force_lds_bytes, s,
                           p.mem, p.tasks, p.force_lds_bytes, ahead);
    return hipGetLastError();
}

template <int STREAM>
hipError_t batch_advance_t(const BatchPlan& p, int steps, hipStream_t s) {
    hipLaunchKernelGGL(k_batch_advance<STREAM>, dim3((uint32_t)(p.n_members + 63) / 64), dim3(64), 0, s, p.mem_rw,
                       p.n_members, steps);
    return hipGetLastError();
}

template <typename Fn>
hipError_t with_batch_prec(int prec, int streaming, Fn&& fn) {
    auto by_stream = [&](auto pr) -> hipError_t {
        using PR = decltype(pr);
        return streaming == StreamEsotwist ? fn(PR{}, IC<StreamEsotwist>{}) : fn(PR{}, IC<StreamSimple>{});
    };
    switch (prec) {
        case 0: return by_stream(PrecF32{});
        case 2: return by_stream(PrecF16{});
        case 3: return by_stream(PrecBF16{});
        case 4: return by_stream(PrecE3M12{});
        default: return hipErrorInvalidValue;
    }
}
}  // namespace

int64_t batch_coll_blocks(const Grid& g, int tile, int bs) {
    if (tile == TILE_ROW64) {
        const int64_t segs = (g.zg1 + 63) / 64;
        const int64_t waves = (int64_t)g.xg1 * g.yg1 * segs;
        return (waves + bs / 64 - 1) / (bs / 64);
    }
    if (tile == TILE_FLAT) return ((int64_t)g.xg1 * g.yg1 * g.zg1 + bs - 1) / bs;
    const int64_t plane = (int64_t)g.yg * g.zg;
    return (int64_t)g.xg1 * ((plane + bs - 1) / bs);
}

hipError_t launch_batch_step(int prec, int streaming, const BatchPlan& plan, int steps, hipStream_t s) {
    return with_batch_prec(prec, streaming, [&](auto pr, auto sc) {
        hipError_t e = hipSuccess;
        for (int k = 0; k < steps && e == hipSuccess; k++)
            e = batch_step_t<decltype(pr), decltype(sc)::value>(plan, k, s);
        if (e != hipSuccess || steps <= 0) return e;
        return batch_advance_t<decltype(sc)::value>(plan, steps, s);
    });
}

hipError_t launch_batch_fused(int prec, int streaming, const BatchPlan& plan, hipStream_t s) {
    return with_batch_prec(prec, streaming, [&](auto pr, auto sc) {
        return batch_fused_t<decltype(pr), decltype(sc)::value>(plan, 0, s);
    });
}

}  // namespace tdlb
