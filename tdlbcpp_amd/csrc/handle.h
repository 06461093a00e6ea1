// State of a ComputeUnit handle (private to the library: capi.cpp, batch.cpp, server.cpp).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/tdlb.h"
#include "kernels.h"

namespace tdlb {
namespace detail {

// records the message for tdlb_last_error() and returns code
int fail(int code, const std::string& msg);

#define HIPCHK(expr)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            return fail(TDLB_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));              \
    } while (0)

#define CHK(expr)                  \
    do {                           \
        int r_ = (expr);           \
        if (r_ != TDLB_OK) return r_; \
    } while (0)

enum Phase { PH_EXPLICIT = 0, PH_LAZY = 1 };

struct DevPoints {
    PointsDev d{};
    int64_t cap = 0;
    size_t tsize = 4;
    void release() {
        void* ptrs[] = {d.i, d.j, d.k, d.ifrac, d.kfrac, d.u, d.v, d.w};
        for (void* p : ptrs)
            if (p) (void)hipFree(p);
        d = PointsDev{};
        cap = 0;
    }
    int reserve(int64_t n, size_t ts) {
        if (n <= cap && ts == tsize) return TDLB_OK;
        release();
        tsize = ts;
        const int64_t c = std::max<int64_t>(n, 256);
        void** ip[] = {(void**)&d.i, (void**)&d.j, (void**)&d.k};
        for (void** p : ip)
            if (hipMalloc(p, sizeof(int32_t) * c) != hipSuccess) return fail(TDLB_ERR_NOMEM, "IB point buffers");
        void** fp[] = {&d.ifrac, &d.kfrac, &d.u, &d.v, &d.w};
        for (void** p : fp)
            if (hipMalloc(p, ts * c) != hipSuccess) return fail(TDLB_ERR_NOMEM, "IB point buffers");
        cap = c;
        return TDLB_OK;
    }
};

// Population arrays: a k-row holds the interior cells k = 1..zg1 only, rows back
// to back (ghost rows in i and j included), and the two k-ghost cells of every row
// sit in a side region after the rows.  The stream-collide kernels never touch a
// k-ghost (Esotwist wraps periodically, the Simple pull reads interior neighbours
// only), so every line they move holds interior cells only, and at zg1 = 512 every
// row starts a 128 B line.  Slot planes of 16 MiB and more start on 1 MiB
// boundaries (planes of 18 concurrent streams whose starts fall at arbitrary
// offsets measured 4 % slower at 512^3), smaller ones on 128 B lines.
inline void set_q_geometry(Grid& g, size_t ssize) {
    g.qz = (uint32_t)g.zg1;
    g.qyz = (uint32_t)((uint64_t)g.yg * g.qz);
    g.qoff = 0xffffffffu;  // (i, j, k) at i*qyz + j*qz + k - 1 (modulo 2^32)
    const uint64_t line = 128 / ssize;  // cells of the stored type in a 128 B line
    g.qside = (uint32_t)(((uint64_t)g.xg * g.qyz + line - 1) / line * line);
    const uint64_t cells = (uint64_t)g.qside + 2ull * g.xg * g.yg;
    const uint64_t align = cells * ssize >= (16ull << 20) ? (1ull << 20) / ssize : line;
    g.qsize = (cells + align - 1) / align * align;
}

// Workgroups of the list kernels and, where the LDS does not hold a plane's, their marks in
// HBM: for fewer workgroups (more planes for each) where memory is short.
inline int reserve_marks(const Grid& g, uint32_t** marks, int* blocks) {
    const size_t each = list_marks_bytes(g, blocks);
    if (each == 0) return TDLB_OK;
    for (;; *blocks /= 2) {
        if (*blocks < 1) return fail(TDLB_ERR_NOMEM, "IB list marks");
        if (hipMalloc((void**)marks, each * (size_t)*blocks) == hipSuccess) return TDLB_OK;
        *marks = nullptr;
        (void)hipGetLastError();  // not the next launch's
    }
}

// Buffers of the per-call forcing, as large as its longest list so far.
struct ListBuffers {
    tdlb_ib_point* raw = nullptr;  // the caller's points
    int64_t* list = nullptr;       // positions, plane by plane
    uint32_t* marks = nullptr;     // reserve_marks
    int blocks = 0;                // workgroups
    int64_t cap = 0;
    void release() {
        for (void* p : {(void*)raw, (void*)list, (void*)marks})
            if (p) (void)hipFree(p);
        raw = nullptr;
        list = nullptr;
        marks = nullptr;
        blocks = 0;
        cap = 0;
    }
    int reserve(int64_t n, const Grid& g) {
        if (n > cap) {
            const int64_t c = std::max<int64_t>(n, 256);
            for (void** p : {(void**)&raw, (void**)&list}) {
                if (*p) (void)hipFree(*p);
                *p = nullptr;
            }
            cap = 0;
            if (hipMalloc((void**)&raw, sizeof(tdlb_ib_point) * (size_t)c) != hipSuccess ||
                hipMalloc((void**)&list, sizeof(int64_t) * (size_t)c) != hipSuccess)
                return fail(TDLB_ERR_NOMEM, "IB list buffers");
            cap = c;
        }
        return n > 0 && blocks == 0 ? reserve_marks(g, &marks, &blocks) : TDLB_OK;
    }
};

// A bound tank's static points and their plane tasks (PlaneDesc): the unique
// stencil cells grouped by plane, points ordered plane by plane and level by level.
struct IndexedSet {
    uint32_t* cells = nullptr;
    int32_t* sidx = nullptr;
    void* rows = nullptr;  // bound tank: ForceRow x 3 per static and blade point
    void* cache = nullptr;
    void* fscr = nullptr;  // bound tank: force scratch of planes beyond the LDS
    PlaneDesc* planes = nullptr;
    int64_t* lev_off = nullptr;
    int64_t n_cells = 0;
    int32_t n_planes = 0, max_levels = 0;
    int32_t level_lanes = 64, level_lds = 0;  // workgroup of the levels launch
    std::vector<float> plane_cost;       // host: duration estimate of each plane (planes order)
    std::vector<PlaneDesc> plane_list;   // host copy of planes
    void release() {
        void* ptrs[] = {cells, sidx, rows, cache, fscr, planes, lev_off};
        for (void* p : ptrs)
            if (p) (void)hipFree(p);
        cells = nullptr;
        sidx = nullptr;
        rows = nullptr;
        cache = nullptr;
        fscr = nullptr;
        planes = nullptr;
        lev_off = nullptr;
        n_cells = 0;
        n_planes = max_levels = 0;
        plane_cost.clear();
        plane_list.clear();
    }
};

// Room for the force values of planes that a levels launch with lds_bytes cannot hold in LDS.
inline int ensure_force_scratch(IndexedSet& set, size_t tsize, int64_t lds_bytes) {
    if (set.fscr) return TDLB_OK;
    for (const PlaneDesc& pd : set.plane_list)
        if ((pd.cell_end - pd.cell_begin) * 3 * (int64_t)tsize > lds_bytes) {
            if (hipMalloc(&set.fscr, (size_t)set.n_cells * 4 * tsize) == hipSuccess) return TDLB_OK;
            set.fscr = nullptr;
            return fail(TDLB_ERR_NOMEM, "IB force scratch");
        }
    return TDLB_OK;
}

// Host-side copy of points in the CU's type, structure of arrays.
struct HostPoints {
    std::vector<int32_t> i, j, k;
    std::vector<uint8_t> ifrac, kfrac, u, v, w;
    void resize(size_t n, size_t ts) {
        i.resize(n); j.resize(n); k.resize(n);
        ifrac.resize(n * ts); kfrac.resize(n * ts); u.resize(n * ts); v.resize(n * ts); w.resize(n * ts);
    }
};

template <typename T>
void put(std::vector<uint8_t>& v, size_t idx, double x) {
    T t = (T)x;
    std::memcpy(v.data() + idx * sizeof(T), &t, sizeof(T));
}

}  // namespace detail
}  // namespace tdlb

using namespace tdlb;
using namespace tdlb::detail;

struct tdlb_cu {
    tdlb_cu_params prm{};
    tdlb_flow flow{};
    Grid g{};
    int64_t xg = 0, yg = 0, zg = 0;
    size_t tsize = 4;  // arithmetic type: F, Nu, points, explicit Q
    size_t ssize = 4;  // stored population type
    hipStream_t stream = nullptr;
    int device = 0;

    void* Q[2] = {nullptr, nullptr};
    int cur = 0;
    void* M = nullptr;   // explicit Q of the reduced-precision storage (float)
    float rho0 = 1.0f;   // rest density of the deviation storage
    double* red = nullptr;  // FP64 partial sums + result of tdlb_cu_reductions
    void* F = nullptr;
    void* Nu = nullptr;
    uint8_t* O = nullptr;
    uint64_t* fmask[2] = {nullptr, nullptr};
    uint64_t* gmask = nullptr;
    uint64_t* static_bits = nullptr;
    uint64_t* static_base = nullptr;
    int fm = 0;
    size_t mask_words = 0;

    bool even = true;
    Phase phase = PH_EXPLICIT;
    bool o_dirty = false;         // O may hold non-zero interior values
    bool static_in_prev = false;  // every static stencil cell is set in fmask[fm]

    // bound Rushton tank
    bool bound = false;
    bool blade_wraps = false;            // a blade stencil may wrap to the other side of the tank
    tdlb_rushton_params rp{};
    DevPoints pts;                       // static points [0, n_static), blades after
    IndexedSet static_set;               // stencil cells of the static points
    void* rot_cache = nullptr;           // 9 moment entries per blade point
    int64_t n_static = 0, n_rot = 0;
    int32_t n_blade_levels = 0;          // blade levels of a plane
    BladeLayout blade{};
    double alfa = 0.97, beta = 1.9;

    // one-launch Esotwist step (launch_eso_pipe), set up at bind when the tank allows it
    bool pipe = false;
    int32_t* rowcell = nullptr;
    uint32_t* pctr = nullptr;

    DevPoints api_pts;  // points of the generic forcing call
    ListBuffers api_lists;

    // event timing of tdlb_cu_run (tdlb_cu_profile)
    bool prof = false;
    std::vector<hipEvent_t> events;        // pool, recorded in pairs
    std::vector<std::pair<int, int>> coll, force;
    size_t ev_used = 0;

    size_t q_cells() const { return (size_t)g.qsize; }  // cells per slot of the kernels' population arrays
    size_t qb_bytes() const { return (size_t)g.size * kQ * tsize; }  // Q as the reference holds it (boundary)
    size_t q_bytes() const { return q_cells() * kQ * tsize; }        // explicit Q on the device
    size_t qs_bytes() const { return q_cells() * kQ * ssize; }       // one population lattice
    size_t f_bytes() const { return (size_t)g.size * 3 * tsize; }
    size_t nu_bytes() const { return (size_t)g.size * (shifted() ? ssize : tsize); }  // Nu on the device
    size_t nub_bytes() const { return (size_t)g.size * tsize; }                       // Nu at the boundary
    size_t mask_bytes() const { return mask_words * sizeof(uint64_t); }
    bool simple() const { return prm.streaming == TDLB_STREAM_SIMPLE; }
    // layout of Q at the boundary (download, upload, checkpoint).  In HBM the
    // lattice is LIJK for every handle: in IJKL a cell's slots are one 72-byte
    // record, of which a wavefront's step reads and writes single slots in the
    // records of four rows (256^3 FP32 Esotwist: 0.86 ms a step even staged through
    // LDS, 0.45 in LIJK).
    int blay() const { return prm.layout == TDLB_LAYOUT_LIJK ? LayoutLIJK : LayoutIJKL; }
    bool shifted() const {
        return prm.precision == TDLB_PREC_F16 || prm.precision == TDLB_PREC_BF16 || prm.precision == TDLB_PREC_E3M12;
    }
    int prec() const { return prm.precision; }            // kernels on the stored populations
    int eprec() const { return prm.precision == TDLB_PREC_F64 ? 1 : 0; }  // kernels on the explicit Q
    void* eq() const { return shifted() ? M : Q[cur]; }   // the explicit Q array

    // the forcing planes of the bound tank
    ForceGeom fgeom() const {
        ForceGeom f{};
        f.pts = pts.d;
        f.n_static = n_static;
        f.n_rot = n_rot;
        f.cells = static_set.cells;
        f.rows = static_set.rows;
        f.scache = static_set.cache;
        f.rcache = rot_cache;
        f.fscr = static_set.fscr;
        f.n_cells = static_set.n_cells;
        f.planes = static_set.planes;
        f.n_planes = static_set.n_planes;
        f.level_lanes = static_set.level_lanes;
        f.level_lds = static_set.level_lds;
        f.lev_off = static_set.lev_off;
        f.blade = blade;
        return f;
    }

    CollideArgs cargs() const {
        CollideArgs c;
        c.nu = flow.nu;
        c.cs0 = flow.cs0;
        c.g3 = flow.g3;
        c.use_les = flow.use_les;
        return c;
    }
};
