/*
 * tdlb.h -- C ABI of the MI355X D3Q19 (18-velocity Eggels-Somers) ComputeUnit.
 *
 * One handle is one ComputeUnit (the reference's ComputeUnitBase<T,18,Layout>,
 * tdlbcpp/src/ComputeUnit.h:39-204) living in the HBM of one GPU.  The entry
 * points mirror that class's virtual surface; each comment names the reference
 * member it replaces.  Conventions:
 *   - every function returns 0 (TDLB_OK) or a negative TDLB_ERR_* code and
 *     sets a thread-local message readable with tdlb_last_error();
 *   - the handle owns its device memory and one HIP stream; calls are
 *     asynchronous on that stream unless they move data to or from the host;
 *   - calls on one handle are not thread-safe; distinct handles may be used
 *     from distinct threads;
 *   - host buffers passed in or out are owned by the caller and are laid out
 *     exactly as the reference lays out its arrays in memory.
 */
#ifndef TDLB_H
#define TDLB_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define TDLB_OK 0
#define TDLB_ERR_INVALID (-1)     /* bad argument or size */
#define TDLB_ERR_HIP (-2)         /* HIP runtime error */
#define TDLB_ERR_NOMEM (-3)       /* device allocation failed */
#define TDLB_ERR_STATE (-4)       /* call not valid in the handle's state */
#define TDLB_ERR_IO (-5)          /* file read or write failed */
#define TDLB_ERR_UNSUPPORTED (-6) /* combination not implemented */

/* MemoryLayoutType (Header.h:38): the order of Q at the boundary (download,
 * upload, checkpoint files).  In HBM the lattice of every handle is LIJK, where
 * the 18 slots of a wavefront's cells are 18 contiguous runs instead of 72-byte
 * strided gathers. */
#define TDLB_LAYOUT_IJKL 0 /* slot l of cell n at q[n*18 + l] */
#define TDLB_LAYOUT_LIJK 1 /* slot l of cell n at q[l*size + n] */
/* no counterpart in the reference: as TDLB_LAYOUT_IJKL */
#define TDLB_LAYOUT_IJKL_SOA 2
/* Streaming (Header.h:37) */
#define TDLB_STREAM_SIMPLE 0
#define TDLB_STREAM_ESOTWIST 1
/* storage / arithmetic type T of the ComputeUnit */
#define TDLB_PREC_F32 0
#define TDLB_PREC_F64 1
/* No counterpart in the reference: populations stored as 16-bit scaled
 * deviations k_d*(f_d - w_d*rho0) (w_d = 1/12 on the 6 faces, 1/24 on the 12
 * edges, k_d = 2 on the faces, 4 on the edges, rho0 = the density of the last
 * tdlb_cu_initialise, initial_rho before it) and Nu in 16 bits, arithmetic in
 * float.  At the boundary T = float for every field (download, upload and
 * checkpoint files convert).  Only tdlb_cu_run advances such a handle; the
 * per-call operations return TDLB_ERR_UNSUPPORTED.  F16: IEEE binary16; BF16:
 * bfloat16; E3M12: sign, 3-bit exponent, 12-bit fraction, offset so that zero
 * is exact and |deviation| < 2^-9 is linear (step 2^-21), range +-0.498,
 * saturating (a quarter of fp16's relative step at the same 2 bytes). */
#define TDLB_PREC_F16 2
#define TDLB_PREC_BF16 3
#define TDLB_PREC_E3M12 4
/* fields of the ComputeUnit */
#define TDLB_FIELD_Q 0  /* size*18 T, in the handle's layout */
#define TDLB_FIELD_F 1  /* size*3 T, {x,y,z} per cell (Force<T>) */
#define TDLB_FIELD_NU 2 /* size T */
#define TDLB_FIELD_O 3  /* size bytes (bool) */

/* ComputeUnitParams (Params/ComputeUnitParams.hpp:26-45) plus the template
 * arguments the reference picks at compile time. */
typedef struct {
    int64_t x, y, z; /* interior cells */
    int64_t ghost;   /* ghost layers; the kernels support ghost == 1 (multiStep default) */
    int64_t i0, j0, k0;
    int64_t resolution;
    int32_t idi, idj, idk, node_id, device_id;
    int32_t layout;    /* TDLB_LAYOUT_* */
    int32_t streaming; /* TDLB_STREAM_* */
    int32_t precision; /* TDLB_PREC_* */
} tdlb_cu_params;

/* FlowParams<T> (Params/FlowParams.hpp:27-61); values are converted to T. */
typedef struct {
    double initial_rho, re_m_nondimensional, uav, cs0, g3, nu;
    double fx0, fy0, fz0, re_m, re_f, uf, alpha, beta;
    int32_t use_les;
    int32_t collision; /* 0 = EgglesSomers (the only implemented collision) */
} tdlb_flow;

/* The fields of PosPolar<tNi,T> that forcing reads (Forcing.hpp:76-78,81,126-128).
 * i, j, k are grid positions without the ghost offset. */
typedef struct {
    int64_t i, j, k;
    double i_frac, k_frac;
    double u_delta, v_delta, w_delta;
} tdlb_ib_point;

/* Geometry of the Rushton-turbine tank generated by this library (the
 * reference's generator library is not part of its source tree). */
typedef struct {
    int64_t tank_diameter;   /* T, the grid x extent (main.cpp:274) */
    int64_t height;          /* planes 0..height-1 hold wall/baffle points */
    double center_x, center_z;
    double tank_radius;
    int32_t n_baffles;
    double baffle_width, baffle_angle0;
    int64_t disk_plane;      /* j of the impeller disk */
    double disk_radius, hub_radius, shaft_radius;
    int32_t n_blades;
    double blade_outer_radius; /* integer valued: impellers[0].blades.outerRadius */
    double blade_inner_radius;
    int64_t blade_plane_lo, blade_planes;
    double tip_speed;          /* uav: blade tip speed in lattice units per step */
    int64_t startup_steps;     /* impellerStartupStepsUntilNormalSpeed */
} tdlb_rushton_params;

#define TDLB_GEOM_FIXED 0
#define TDLB_GEOM_ROTATING_NON_UPDATING 1
#define TDLB_GEOM_ROTATING 2

typedef struct tdlb_cu* tdlb_cu_t;

/* thread-local text of the last error */
const char* tdlb_last_error(void);
int tdlb_version(void);
int tdlb_device_count(int* count);

/* ---- ComputeUnit lifetime: ctor / init / allocateMemory (ComputeUnit.hpp:66-133) */
int tdlb_cu_create(const tdlb_cu_params* params, const tdlb_flow* flow, tdlb_cu_t* out);
int tdlb_cu_destroy(tdlb_cu_t cu);
/* replace the flow parameters (the reference's `flow` member), e.g. after calcNuAndRe_m */
int tdlb_cu_set_flow(tdlb_cu_t cu, const tdlb_flow* flow);

/* FlowParams<T>::calcNuAndRe_m (Params/FlowParams.hpp:65-70) evaluated in T
 * (TDLB_PREC_*): re_m = re_m_nondimensional*pi/2; nu = uav*T(outer_radius)/re_m. */
int tdlb_flow_calc_nu_re_m(tdlb_flow* flow, int32_t impeller_blade_outer_radius, int32_t precision);

/* ---- operator surface (ComputeUnit.h:110-200) */
int tdlb_cu_initialise(tdlb_cu_t cu, double rho);           /* initialise(T), ComputeUnit.hpp:174-190 */
int tdlb_cu_collision(tdlb_cu_t cu);                        /* collision(), CollisionEgglesSomers.hpp:26-181 */
int tdlb_cu_moments(tdlb_cu_t cu);                          /* moments(), CollisionEgglesSomers.hpp:185-256 */
int tdlb_cu_stream_push(tdlb_cu_t cu);                      /* streamingPush(), StreamingSimple.hpp:76-126 /
                                                               StreamingEsoteric.hpp:14-18 */
int tdlb_cu_stream_pull(tdlb_cu_t cu);                      /* streamingPull(), StreamingSimple.hpp:18-66 /
                                                               StreamingEsoteric.hpp:20-24 */
int tdlb_cu_bounce_back(tdlb_cu_t cu);                      /* bounceBackBoundary(), Boundary.hpp:13-250 */
int tdlb_cu_forcing(tdlb_cu_t cu, const tdlb_ib_point* points, int64_t n, double alfa,
                    double beta);                           /* forcing(geom, alfa, beta), Forcing.hpp:56-176 */

/* ---- public members Q, F, Nu, O and evenStep (ComputeUnit.h:71-84) */
int tdlb_cu_field_bytes(tdlb_cu_t cu, int field, size_t* bytes);
int tdlb_cu_download(tdlb_cu_t cu, int field, void* host, size_t bytes);
int tdlb_cu_upload(tdlb_cu_t cu, int field, const void* host, size_t bytes);
int tdlb_cu_get_even_step(tdlb_cu_t cu, int* even);
int tdlb_cu_set_even_step(tdlb_cu_t cu, int even);
/* grid sizes: xg, yg, zg, size (initGridParams, ComputeUnit.hpp:25-40) */
int tdlb_cu_dims(tdlb_cu_t cu, int64_t* xg, int64_t* yg, int64_t* zg, int64_t* size);
int tdlb_cu_synchronize(tdlb_cu_t cu);
/* the handle's HIP stream (hipStream_t), for event timing by the caller */
int tdlb_cu_stream(tdlb_cu_t cu, void** hip_stream);

/* ---- checkpoint files, byte-compatible with the reference (ComputeUnit.hpp:322-439,
 *      names DiskOutputTree.h:560-590):
 *   <dir>/AllParams.<idi>.<idj>.<idk>.<unit>.json    (text given by the caller)
 *   <dir>/checkpoint_grid.<idi>.<idj>.<idk>.<unit>.Q  size*18 T, the handle's layout, moments phase
 *   <dir>/checkpoint_grid.<idi>.<idj>.<idk>.<unit>.F  size*3 T
 *   <dir>/checkpoint_grid.<idi>.<idj>.<idk>.<unit>.Nu size T
 * all_params_json may be NULL (no JSON written).  read: a missing array file leaves
 * that field as it is (the reference logs and continues) and sets its bit in
 * *missing (Q 1, F 2, Nu 4); a file of the wrong size is TDLB_ERR_IO. */
int tdlb_cu_checkpoint_write(tdlb_cu_t cu, const char* dir, const char* unit_name, const char* all_params_json);
int tdlb_cu_checkpoint_read(tdlb_cu_t cu, const char* dir, const char* unit_name, int* missing);

/* ---- Rushton geometry (host generator; replaces the RushtonTurbinePolarCPP calls
 *      of main.cpp:274-303,409-426) */
int tdlb_rushton_defaults(int64_t tank_diameter, int64_t height, double tip_speed, int64_t startup_steps,
                          tdlb_rushton_params* out);
/* group = TDLB_GEOM_*; angle and delta_angle as in generateRotatingGeometry(angle, delta).
 * Writes at most cap points; *n receives the full count. */
int tdlb_rushton_generate(const tdlb_rushton_params* p, int group, double angle, double delta_angle,
                          tdlb_ib_point* out, int64_t cap, int64_t* n);
/* calcThisStepImpellerIncrement(step): angular increment with the start-up ramp */
int tdlb_rushton_step_increment(const tdlb_rushton_params* p, uint64_t step, double* delta);
/* getExternalPoints as a mask: 1 for cells outside the tank, xg*yg*zg bytes, ghosts included */
int tdlb_rushton_solid_mask(const tdlb_rushton_params* p, int64_t xg, int64_t yg, int64_t zg, int64_t ghost,
                            uint8_t* out);

/* ---- fused fast path: the main-loop step of main.cpp:336-455 on the device */
/* Bind the tank: uploads the fixed and rotating-non-updating lists generated for
 * (step, angle) and runs the initial forcing of main.cpp:305.  alfa/beta as forcing.
 * The impeller must lie inside the interior (TDLB_ERR_INVALID otherwise); the
 * blades are forced in colour classes of non-overlapping stencils, a class per
 * blade in tanks too small for shared classes (the generator's rotating list
 * follows the same classes), so every tank size binds.  Arguments that are
 * refused leave an earlier geometry bound; a bind that fails later (memory)
 * leaves the handle without one (TDLB_ERR_STATE from tdlb_cu_run). */
int tdlb_cu_bind_rushton(tdlb_cu_t cu, const tdlb_rushton_params* p, uint64_t step, double angle, double alfa,
                         double beta);
/* Run nsteps iterations of the main loop: step += 1; angle += increment(step);
 * rotate blades on the device; collision; bounceBack; streamingPush; moments;
 * forcing.  *step and *angle are updated (RunningParams). */
int tdlb_cu_run(tdlb_cu_t cu, int64_t nsteps, uint64_t* step, double* angle);
/* the blade list the device generated for the last step, for checks */
int tdlb_cu_rotating_points(tdlb_cu_t cu, tdlb_ib_point* out, int64_t cap, int64_t* n);
/* getExternalPoints mask computed on the device (xg*yg*zg bytes) */
int tdlb_cu_solid_mask(tdlb_cu_t cu, uint8_t* out, size_t bytes);
/* number of IB points of the bound geometry, and the levels that its forcing runs one
 * after the other: the most static levels of a plane, and the blade levels */
int tdlb_cu_forcing_info(tdlb_cu_t cu, int64_t* n_static, int64_t* n_rotating, int64_t* n_levels);
/* 1 when tdlb_cu_run advances this bound tank with the one-launch step (no
 * counterpart in the reference; opt-in: the environment variable TDLB_PIPE=1
 * at bind time): Esotwist in LIJK, float arithmetic, at least 24 interior j
 * planes and 64 k cells, on a GPU whose launches span all 8 XCDs.  The
 * stream-collide and the IB forcing gather then run in one persistent kernel
 * per step, the forcing levels in a second launch, with the same arithmetic in
 * the same order as the separate launches. */
int tdlb_cu_one_launch(tdlb_cu_t cu, int32_t* on);
/* Phase times of the last one-launch step, in microseconds from its first work
 * item (no counterpart in the reference): for each of the 8 XCDs, when its
 * last row was written and its last forcing gather done: us[3 x + 0], us[3 x + 1],
 * and us[3 x + 2] as us[3 x + 1] (the forcing levels run in a launch of their own);
 * n >= 24.  Synchronises the handle's stream. */
int tdlb_cu_one_launch_phases(tdlb_cu_t cu, double* us, int32_t n);
/* Kernel timing of the fused path (no counterpart in the reference, which only
 * has wall-clock phase timers, timer.cpp:127-222): while enabled, tdlb_cu_run
 * brackets each stream-collide launch and each forcing pass with HIP events on
 * the handle's stream.  read returns the summed elapsed times and counts since
 * the last enable and synchronises the stream. */
int tdlb_cu_profile(tdlb_cu_t cu, int enable);
int tdlb_cu_profile_read(tdlb_cu_t cu, double* collide_ms, int64_t* collide_launches, double* forcing_ms,
                         int64_t* forcing_passes);

/* Conservation and torque sums in FP64 on the device (no counterpart in the
 * reference).  Over the interior cells of the reference's current Q and F, in a
 * fixed order (the result does not depend on scheduling): out[0] = sum rho,
 * out[1..3] = sum j (moments M02..M04), out[4..6] = sum F, out[7] = impeller
 * torque sum(x*Fz - z*Fx) over the cells whose centre (x, z), relative to the
 * bound tank's axis, lies within blade_outer_radius + 2 (0 when no geometry is
 * bound).  Power delivered to the fluid = out[7] * angular increment per step.
 * The handle's state is not changed. */
int tdlb_cu_reductions(tdlb_cu_t cu, double out[8]);
/* tdlb_cu_reductions without allocating (no counterpart in the reference; for
 * callers that cannot allocate: code under HIP graph capture, serving loops,
 * harnesses that forbid hipMalloc).  Enqueues the same sums, bit for bit, on
 * the handle's stream, writes the 8 doubles to out_device (device memory, 64
 * bytes) and returns without synchronising.  The partial sums live in a fixed
 * device array of the library (65,600 bytes, one per GPU, held until the
 * process ends); the reduction grid is fixed, so every lattice fits and no
 * handle is rejected for its size.  Calls on one GPU share that array: two
 * calls whose work is not ordered (different streams, no synchronisation in
 * between) race and give wrong sums. */
int tdlb_cu_reductions_noalloc(tdlb_cu_t cu, double* out_device);
/* rho and velocity of every interior cell, {rho, ux, uy, uz} in T, cells in
 * (i, j, k) order with k fastest; u = (1/rho)(j + F/2) as QVec::velocity(F)
 * (QVec.hpp:125-131) forms it, which the output planes of
 * ComputeUnitOutput.hpp:354-447 write.  bytes = x*y*z*4*sizeof(T). */
int tdlb_cu_macroscopic(tdlb_cu_t cu, void* out, size_t bytes);

/* ---- regrid and outputs */
/* doubleResolutionFullCU() (ComputeUnit.hpp:257-316): x, y, z double and
 * resolution += 2; every cell of the new grid, ghosts included, takes Q and Nu
 * of old cell (i/2 + i%2, j/2 + j%2, k/2 + k%2) (indexPreviousResolution,
 * ComputeUnit.hpp:480-502); F and O are zero.  The handle keeps its address but
 * gets new arrays and a new stream, and no geometry is bound: bind the tank of
 * the new size before tdlb_cu_run (main.cpp:349-399 regenerates it). */
int tdlb_cu_double_resolution(tdlb_cu_t cu);
/* ExcludeOutputPoints as main.cpp:309-315,466 sets it before writing output:
 * cells outside the tank and every cell holding a point of the bound geometry
 * (fixed, rotating-non-updating and the current blades); xg*yg*zg bytes. */
int tdlb_cu_output_exclude(tdlb_cu_t cu, uint8_t* out, size_t bytes);
/* savePlaneXZ<float, 4> (ComputeUnitOutput.hpp:354-447) for plane j = cut:
 * tDiskGrid<float,4> records {uint16 i0+i-1, j-1, k0+k-1; float q[4]} (24 bytes,
 * q = the first 4 raw slots of the cell) for every plane cell not excluded,
 * and tDiskGrid<float,3> records {uint16 i0+i-1, j, k0+k-1; float F[3]} (20
 * bytes) where all three F components are non-zero (Force::isNotZero,
 * QVec.hpp:54-56); i-major order.  exclude: xg*yg*zg bytes or NULL.  Both
 * buffers hold x*z records; the counts are returned. */
int tdlb_cu_plane_xz(tdlb_cu_t cu, int64_t cut, const uint8_t* exclude, void* qvec, int64_t* n_qvec, void* f3,
                     int64_t* n_f3);
/* the field calcVorticityXZ / calcVorticityXY (ComputeUnitOutput.hpp:113-160,
 * 198-245) turns into a picture: log|curl u|^2 from central differences of
 * j/rho read through the streaming accessor, NaN where excluded (and where an
 * Esotwist read of a far-side ghost cell would leave the array).  axis 0: plane
 * j = cut, x*z values; axis 1: plane k = cut, x*y values; i-major, T each. */
int tdlb_cu_vorticity(tdlb_cu_t cu, int32_t axis, int64_t cut, const uint8_t* exclude, void* out, size_t bytes);

/* ---- batches of ComputeUnits (no counterpart in the reference, which runs one
 * ComputeUnit per process).  Members are bound handles of one precision
 * (TDLB_PREC_F32, _F16 or _BF16), streaming and layout, on the batch's device,
 * with at least 3 cells in x and z.  tdlb_batch_run advances every member as
 * tdlb_cu_run would (bit for bit), each kernel of the step launched once for
 * the whole batch and the step replayed from a HIP graph.  Between runs the
 * handles may be used as usual (download, reductions, checkpoint); during a
 * run they belong to the batch. */
typedef struct tdlb_batch* tdlb_batch_t;
int tdlb_batch_create(int32_t precision, int32_t layout, int32_t streaming, int32_t device_id, tdlb_batch_t* out);
int tdlb_batch_destroy(tdlb_batch_t b);
/* use_graph: replay captured steps (default 1); autotune: time the candidate
 * tiles and block sizes of the fused kernel per grid shape on scratch lattices
 * (default 1) */
int tdlb_batch_set_options(tdlb_batch_t b, int32_t use_graph, int32_t autotune);
/* time the fused-kernel candidates for cu's grid shape on cu's own arrays,
 * which it overwrites: call between tdlb_cu_create and tdlb_cu_initialise (a
 * server does it while preparing a tank, so that no scratch lattice is needed
 * and no timing runs on the thread that drives the batch); no-op when the shape
 * is known or autotuning is off */
int tdlb_batch_tune(tdlb_batch_t b, tdlb_cu_t cu);
/* add a member at RunningParams (step, angle) with a budget of nsteps further steps */
int tdlb_batch_add(tdlb_batch_t b, tdlb_cu_t cu, uint64_t step, double angle, int64_t nsteps);
int tdlb_batch_remove(tdlb_batch_t b, tdlb_cu_t cu);
/* every member takes min(nsteps, its remaining budget) steps; *steps_run = the most any member took */
int tdlb_batch_run(tdlb_batch_t b, int64_t nsteps, int64_t* steps_run);
/* a member's RunningParams and remaining budget */
int tdlb_batch_member(tdlb_batch_t b, tdlb_cu_t cu, uint64_t* step, double* angle, int64_t* remaining);
/* members, kernel launches of a step (recorded alone: a graph of several advances the
 * members' state once), and each member's tile (0 row, 1 plane, 2 flat) */
int tdlb_batch_info(tdlb_batch_t b, int64_t* n_members, int64_t* launches_per_step, int32_t* tiles, int64_t cap);
/* the fused kernel's block size of the last run, the steps one graph replay
 * advances and the workgroup size of the forcing levels (chosen from the members'
 * mean stencil cells per plane task; TDLB_BATCH_FORCE_BLOCK overrides it) */
int tdlb_batch_shape(tdlb_batch_t b, int32_t* block_size, int32_t* graph_steps, int32_t* forcing_block);

/* ---- serving a stream of tank requests (no counterpart in the reference).
 * Requests queue in arrival order and are admitted while their HBM footprint
 * fits the budget; a preparation thread builds admitted tanks while the GPU
 * runs; prepared tanks join the running batch between ticks and leave it when
 * their steps are done (continuous batching).  A tank is the generator's
 * default tank at the request's tip speed, nu from calcNuAndRe_m at the
 * request's Reynolds number, cs0 0.1, LES on, at rest (rho 1), bound at step 1;
 * it advances exactly as tdlb_cu_run would advance it alone. */
typedef struct {
    int64_t edge;          /* grid edge T (cubic grid and tank diameter), >= 12 */
    double tip_speed;      /* impeller tip speed (lattice units) */
    double reynolds;       /* reMNonDimensional */
    int64_t steps;         /* main-loop steps to run */
    int64_t startup_steps; /* impeller start-up ramp */
} tdlb_tank_request;
typedef struct {
    int64_t ticket, edge, steps;
    int32_t error;     /* TDLB_OK or the code the tank failed with */
    double submit_s, admit_s, start_s, finish_s; /* server clock (s since create) */
    double mass, mass_drift, torque, power_number; /* FP64 device sums at the end */
} tdlb_tank_result;
typedef struct tdlb_server* tdlb_server_t;
/* budget <= 0: 90 % of the device memory free at creation (also the cap);
 * max_resident > 0 caps the tanks admitted at once (1: one tank at a time);
 * keep_handles: finished tanks are kept for tdlb_server_take instead of freed */
int tdlb_server_create(int32_t precision, int32_t layout, int32_t streaming, int32_t device_id,
                       double hbm_budget_bytes, int64_t tick_steps, int64_t max_resident, int32_t keep_handles,
                       tdlb_server_t* out);
int tdlb_server_destroy(tdlb_server_t s);
int tdlb_server_submit(tdlb_server_t s, const tdlb_tank_request* req, int64_t* ticket);
/* admit, join, run tick_steps steps, retire; counts after the tick */
int tdlb_server_tick(tdlb_server_t s, int64_t* resident, int64_t* queued, int64_t* steps_run);
/* move up to cap finished results out */
int tdlb_server_poll(tdlb_server_t s, tdlb_tank_result* out, int64_t cap, int64_t* n);
/* the handle of a finished tank (keep_handles); the caller destroys it */
int tdlb_server_take(tdlb_server_t s, int64_t ticket, tdlb_cu_t* cu);
int tdlb_server_stats(tdlb_server_t s, double* now_s, double* reserved_bytes, double* budget_bytes);

/* ---- measurement */
/* Speed of light of the stream-collide access pattern (no counterpart in the
 * reference, which has no bandwidth instrument): `planes` (1..20) planes of
 * `cells` values of elem_bytes (2, 4 or 8) bytes, plane_stride_bytes apart (a
 * multiple of 128 of at least cells * elem_bytes; 0: the plane rounded up to
 * 1 MiB); one pass reads every value of every plane and writes it back in
 * place (bits flipped), one cell per lane in 512-lane blocks, with
 * non-temporal loads and stores when nontemporal != 0.  Two untimed passes,
 * then `passes` passes timed with HIP events on a stream of its own:
 * *ms_per_pass is their average.  Bytes moved per pass: 2 * planes * cells *
 * elem_bytes.  Allocates and frees planes * stride bytes. */
int tdlb_probe_planes(int32_t device_id, int32_t elem_bytes, int64_t cells, int64_t plane_stride_bytes,
                      int32_t planes, int32_t nontemporal, int32_t passes, double* ms_per_pass);

#ifdef __cplusplus
}
#endif

#endif /* TDLB_H */
