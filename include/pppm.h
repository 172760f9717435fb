/*
 * pppm.h -- C ABI of the gfx950 PPPM vortex-velocity library (libpppm_hip.so).
 *
 * Plain pointers and sizes only.  All array arguments are DEVICE pointers
 * unless stated otherwise; all work is enqueued on the context's HIP stream.
 *
 * Reference interfaces replaced (paths relative to the reference repository):
 *   pppm_set_vortices      BiotSavartSolver::setVortParameter
 *                          (hybridFastSummation/hybridFastSummation/BiotSavartSolver.h:33,
 *                           BiotSavartSolverImp.cpp:318-377)
 *   pppm_compute_far_field BiotSavartSolver::computeFarFieldBuffer
 *                          (BiotSavartSolver.h:36, BiotSavartSolverImp.cpp:755-816)
 *   pppm_evaluate          BiotSavartSolver::setEvalParameter + evaluateVelocity + getU
 *                          (BiotSavartSolver.h:23-24,32; BiotSavartSolverImp.cpp:266-316,410-516)
 *   pppm_hash_*            ParticleManager::doSpatialHash / reorderData / deorderData
 *                          (particle_hash/particle_hash/SpaceHashClass.h:42-69,
 *                           SpaceHashClassImp.cpp:18-34)
 *   pppm_mg_*              gf::MultiGridSolver3DPeriod(_double)::m_InitialSystem /
 *                          m_FullMultiGrid / m_Vcycle (multigrid/multigrid/MultiGrid.h:128-209,
 *                          MultiGrid.cpp:128-250)
 * The reference's own extern "C" names (calcHash, FindCellStart, sortParticles,
 * reorder, deorder, setParameters, mg_*, AllocateMemory, ...) are declared in
 * pppm_ref.h and implemented on top of these.
 */
#ifndef PPPM_H
#define PPPM_H
#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef enum pppm_status {
    PPPM_OK = 0,
    PPPM_ERR_INVALID = 1,       /* bad argument or unsupported size            */
    PPPM_ERR_HIP = 2,           /* HIP runtime error (pppm_last_error() says which) */
    PPPM_ERR_NOMEM = 3,         /* device allocation failed                    */
    PPPM_ERR_BUDGET = 4,        /* request larger than the HBM budget (serving) */
    PPPM_ERR_NOT_CONVERGED = 5, /* multigrid stopped above its tolerance       */
    PPPM_ERR_STATE = 6,         /* call out of order (e.g. evaluate before far field) */
    PPPM_ERR_NO_DEVICE = 7      /* no usable GPU                               */
} pppm_status;

/* element types; the values equal the reference's "precision" codes
 * (particle_hash_kernel.cu:143-152: 1 = float, 2 = double) */
enum { PPPM_F32 = 1, PPPM_F64 = 2 };
enum { PPPM_KERNEL_EXPCUBIC = 0, PPPM_KERNEL_GAUSSIAN = 1 };
enum { PPPM_MG_VCYCLE = 0, PPPM_MG_REF_FMG = 1, PPPM_MG_REF_VCYCLE = 2 };
enum { PPPM_PREC_FP32 = 0, PPPM_PREC_MIXED = 1 };

typedef struct pppm_params {
    uint32_t g;             /* grid cells per axis (cubic grid and hash), 8..1024      */
    double h;               /* cell size; the hash keeps (float)h, the path (double)(float)h */
    double origin[3];       /* domain origin; the hash keeps (float)origin              */
    int32_t K;              /* near-field range in cells, 0..4; -1 = vortex-in-cell
                               (no near field, M2P of the grid velocity)           */
    int32_t kernel;         /* PPPM_KERNEL_*                                           */
    double core_a;          /* smoothing core radius (absolute units)                 */
    int32_t mg_schedule;    /* PPPM_MG_VCYCLE (to tolerance) or PPPM_MG_REF_FMG          */
    int32_t nu1, nu2;       /* red+black smoothing iterations before / after          */
    double mg_omega;        /* SOR factor (1 = Gauss-Seidel; the reference uses 1.43f)  */
    double mg_tol;          /* relative residual target (VCYCLE / mixed)                */
    int32_t mg_max_cycles;  /* cap on V-cycles (plain) or outer corrections (mixed)    */
    int32_t precision;      /* PPPM_PREC_FP32 or PPPM_PREC_MIXED                        */
} pppm_params;

typedef struct pppm_stats {
    uint32_t n, m;            /* vortices, evaluation points of the last calls        */
    int32_t mg_cycles;        /* V-cycles run (mixed: total inner V-cycles)           */
    int32_t mg_outer;         /* FP64 defect-correction steps (mixed), else 0         */
    double mg_relres[3];      /* final relative residual per component (FP64 norms) */
    uint32_t strays;          /* vortices whose deposit cell differs from hash cell   */
    int32_t mg_converged;     /* 1 if the tolerance was met (REF_FMG: always 1)       */
} pppm_stats;

typedef struct pppm_ctx pppm_ctx;

/* Defaults for the benchmark configurations: domain [0,1)^3, h = 1/g, K = 2,
 * expcubic core a = 1.5 h, V(2,2) red-black SOR cycles (omega 1.15) to
 * relative residual 1e-6. */
void pppm_params_config_preset(pppm_params *p, uint32_t g);
/* The reference's own settings (BiotSavartSolverImp.cpp, VortexSimulationSystemImp.cpp:890-905):
 * a = 0.08, one FMG pass with V(4,4) SOR 1.43f; origin/h from pppm_reference_domain. */
void pppm_params_reference_preset(pppm_params *p, uint32_t g, int32_t K);
/* BiotSavartSolverImp.cpp:378-409 (setDomain): host positions (float4 rows) ->
 * origin = bbox centre - L/2, L = 3 * largest extent; writes h = L / g. */
pppm_status pppm_reference_domain(const float *host_pos4, uint32_t n, uint32_t g, double origin_out[3],
                                  double *h_out);

pppm_status pppm_create(const pppm_params *p, pppm_ctx **out);
void pppm_destroy(pppm_ctx *ctx);
pppm_status pppm_set_stream(pppm_ctx *ctx, void *hip_stream);
pppm_status pppm_get_stream(const pppm_ctx *ctx, void **hip_stream);
pppm_status pppm_get_params(const pppm_ctx *ctx, pppm_params *out);
/* Move the domain (origin, h) of an existing context without reallocating;
 * the grid size stays.  Invalidates the hashed vortices and the far field. */
pppm_status pppm_set_domain(pppm_ctx *ctx, const double origin[3], double h);
/* Replace all parameters except g and precision (which size the context). */
pppm_status pppm_update_params(pppm_ctx *ctx, const pppm_params *p);
/* Device memory the context holds. */
pppm_status pppm_get_device_bytes(const pppm_ctx *ctx, size_t *bytes);
/* on = 1 (default): each multigrid iteration (V-cycle plus residual/norm work)
 * is captured once into a HIP graph and replayed. */
pppm_status pppm_set_graphs(pppm_ctx *ctx, int32_t on);
/* Order in which the near field walks the sorted points (no counterpart in
 * the reference, whose near field takes one thread per point in sort order).
 * PPPM_NEAR_ORDER_AUTO (default): the sort's order (the potential-flow near
 * fields: renumbered in super-blocks of 8x4x4 cells when there are at least
 * 4,096 points and a quarter as many as x segments, and the near field's
 * sources and cell tables, 32 B a source and 8 B a cell, exceed 64 MiB).
 * _SORT: always the sort's order.  _SUPER_BLOCKS: always renumbered.  On grids
 * of more than 2^29 cells (sort keys without the octant) the order is the
 * sort's in every mode.  The orders differ in FP32 summation order only. */
#define PPPM_NEAR_ORDER_AUTO 0
#define PPPM_NEAR_ORDER_SORT 1
#define PPPM_NEAR_ORDER_SUPER_BLOCKS 2
pppm_status pppm_set_near_order(pppm_ctx *ctx, int32_t order);

/* Vortices: pos4 = float4 rows (x, y, z, unused); strength component c of
 * vortex i at w_c[i * w_stride] with element type w_dtype (PPPM_F32/PPPM_F64).
 * Hashes, sorts and reorders them (device-resident afterwards). */
pppm_status pppm_set_vortices(pppm_ctx *ctx, uint32_t n, const float *pos4, const void *wx, const void *wy,
                              const void *wz, uint32_t w_stride, int32_t w_dtype);
/* P2M, three Poisson solves, curl and far-field buffer. */
pppm_status pppm_compute_far_field(pppm_ctx *ctx);
/* Velocity at m points (float4 rows), written in the caller's order to
 * u_c[i * u_stride] with element type u_dtype.  other_end4 (may be NULL) is the
 * segment mode of the reference: vortices within 1e-12 of the other end are skipped. */
pppm_status pppm_evaluate(pppm_ctx *ctx, uint32_t m, const float *eval_pos4, const float *other_end4, void *ux,
                          void *uy, void *uz, uint32_t u_stride, int32_t u_dtype);
/* Velocity at the vortices themselves (reuses the vortex hash). */
pppm_status pppm_evaluate_self(pppm_ctx *ctx, void *ux, void *uy, void *uz, uint32_t u_stride, int32_t u_dtype);
/* Whole path on the vortices: set_vortices + compute_far_field + evaluate_self. */
pppm_status pppm_solve_self(pppm_ctx *ctx, uint32_t n, const float *pos4, const void *wx, const void *wy,
                            const void *wz, uint32_t w_stride, int32_t w_dtype, void *ux, void *uy, void *uz,
                            uint32_t u_stride, int32_t u_dtype);
pppm_status pppm_get_stats(const pppm_ctx *ctx, pppm_stats *out);
/* Near-field pairs of the vortices with each other that pass the box test
 * |dx|,|dy|,|dz| < (K + 1/2) h and are not coincident (self-evaluation),
 * counted on the device; used for FLOP accounting (synchronous). */
pppm_status pppm_count_near_pairs(pppm_ctx *ctx, uint64_t *pairs);

/* Sorted device views of the last set_vortices (BiotSavartSolver::getSortPos /
 * getVortStartTable / getVortEndTable / getSortVort, BiotSavartSolver.h:25-29).
 * Positions are float4 (x - ox, y - oy, z - oz, w): coordinates relative to
 * the grid origin (FP32 of the FP64 difference), and w holds the bits of the
 * uint32 index of the cell the vortex deposits into (0xFFFFFFFF if outside). */
pppm_status pppm_get_sorted_vortices(pppm_ctx *ctx, const float **pos4, const uint32_t **sorted_index,
                                     const uint32_t **cell_start, const uint32_t **cell_end);
/* Grid fields after compute_far_field: which = 0 vorticity (h^-3 scaled),
 * 1 stream function, 2 far-field velocity; component c; float32 [g^3]
 * (mixed precision: the stream function is float64). */
pppm_status pppm_get_grid(pppm_ctx *ctx, int32_t which, int32_t c, const void **ptr, int32_t *dtype);

/* Device bytes a fresh context with these parameters needs for n vortices and
 * m evaluation points (m = 0: self evaluation; other_end: segment mode). */
pppm_status pppm_estimate_device_bytes(const pppm_params *p, uint32_t n, uint32_t m, int32_t other_end,
                                       size_t *bytes);

/* ---- serving: continuous batching of evaluation requests on one GPU -------
 * No counterpart in the reference, which evaluates one scene at a time from
 * one host thread (VortexSimulationSystemImp.cpp:142-228, 1194-1244).
 * Requests run on `slots` worker threads, each on its own resident context and
 * stream, so their work overlaps on the device.  Contexts stay resident after
 * a request and are reused by the next request with the same g and precision.
 * Admission is FIFO against hbm_budget_bytes (least-recently-used idle
 * contexts are evicted to make room).  Buffers in a request are device
 * pointers owned by the caller: inputs complete before submit, all valid
 * until the request is done. */
typedef struct pppm_server pppm_server;
typedef struct pppm_server_config {
    size_t hbm_budget_bytes; /* device bytes the server's contexts may hold          */
    int32_t slots;           /* requests on the device at once, 1..16               */
    int32_t use_graphs;      /* capture multigrid iterations into HIP graphs        */
    int32_t group_max;       /* small requests solved together, up to 16 (0, 1: none) */
    uint32_t group_max_g;    /* largest grid (cells per axis) solved in a group; 0: 64 */
} pppm_server_config;
typedef struct pppm_request {
    pppm_params params;      /* grid, domain, kernel, schedule, precision            */
    uint32_t n;              /* vortices                                             */
    const float *pos4;       /* float4[n]                                            */
    const void *wx, *wy, *wz;
    uint32_t w_stride;
    int32_t w_dtype;         /* PPPM_F32 / PPPM_F64                                   */
    uint32_t m;              /* evaluation points; 0 = at the vortices               */
    const float *eval_pos4;  /* float4[m] (m > 0)                                    */
    const float *other_end4; /* segment mode (may be NULL)                           */
    void *ux, *uy, *uz;      /* velocity out, caller order                           */
    uint32_t u_stride;
    int32_t u_dtype;
} pppm_request;
typedef struct pppm_request_result {
    int32_t status;          /* pppm_status of the request                          */
    int32_t pad;
    double latency_ms;       /* submit to completion                                 */
    double queue_ms;         /* submit to start                                      */
    pppm_stats stats;        /* solver statistics of the request                     */
    char message[160];       /* pppm_last_error() of the failed call, else empty      */
} pppm_request_result;
typedef struct pppm_server_stats {
    uint64_t submitted, completed, failed, particles;
    uint32_t queued, running, contexts, pad;
    uint64_t ctx_created, ctx_reused, ctx_evicted;
    uint64_t device_bytes, peak_device_bytes;
    double p50_ms, p99_ms, mean_ms; /* request latency (nearest rank)              */
    double wall_s;                  /* first submit to last completion             */
    double particles_per_s;         /* evaluated points / wall_s                   */
    uint64_t grouped;               /* requests whose solve ran in a group of >= 2 */
    uint64_t groups;                /* group solves (of >= 2 requests)             */
} pppm_server_stats;
pppm_status pppm_server_create(const pppm_server_config *cfg, pppm_server **out);
/* Waits for every queued and running request, then frees all contexts. */
void pppm_server_destroy(pppm_server *srv);
pppm_status pppm_request_estimate_bytes(const pppm_request *r, size_t *bytes);
pppm_status pppm_server_submit(pppm_server *srv, const pppm_request *r, uint64_t *ticket);
pppm_status pppm_server_poll(pppm_server *srv, uint64_t ticket, int32_t *done);
/* Blocks until the request is done; releases the ticket. */
pppm_status pppm_server_wait(pppm_server *srv, uint64_t ticket, pppm_request_result *res);
pppm_status pppm_server_drain(pppm_server *srv);
pppm_status pppm_server_get_stats(pppm_server *srv, pppm_server_stats *out);
pppm_status pppm_server_reset_stats(pppm_server *srv);

/* ---- potential-flow solver (PotentialFieldSolver.h:15-60) ------------------
 * The reference's PotentialFieldSolver as a context: point masses in, the
 * gradient (or the potential) of G sum m / (4 pi |x - x_m|) out, by PPPM
 * (PotentialFieldSolver.cpp:409-739).  Device buffers stay resident from call
 * to call and run on the solver's own stream; nothing is allocated once the
 * sizes are reached.  The grid part is FP64 as the reference's (deposit,
 * right-hand side with the monopole Dirichlet values, three FMG passes,
 * gradient and far-field buffers); the near fields run in FP32 on the vortex
 * path's clustered kernel. */
typedef struct pppm_pot pppm_pot;
/* g cells per axis (8..1024), near-field range K (0..8), the solver's G and
 * direction (Potential_PPCorrMN's G and direction). */
pppm_status pppm_pot_create(uint32_t g, int32_t K, double G, double direction, pppm_pot **out);
void pppm_pot_destroy(pppm_pot *pot);
pppm_status pppm_pot_get_stream(pppm_pot *pot, void **hip_stream);
/* computeFarFieldBuffer: device float4 positions (xyz used) and FP64 masses;
 * the domain is setDomain's, a cube of twice the masses' largest extent
 * about the centre of their bounding box (one host wait for it). */
pppm_status pppm_pot_set_masses(pppm_pot *pot, uint32_t n, const float *pos4, const double *mass);
/* The domain of the last pppm_pot_set_masses: corner and cell size. */
pppm_status pppm_pot_domain(const pppm_pot *pot, double origin[3], double *h);
/* evaluateGradient: grad[3 m] (x, y, z per point, FP64) at device points;
 * points outside the domain get zero, as in the reference. */
pppm_status pppm_pot_gradient(pppm_pot *pot, uint32_t m, const float *pos4, double *grad);
/* evaluateScalarPotential: phi[m] (FP64) at device points. */
pppm_status pppm_pot_potential(pppm_pot *pot, uint32_t m, const float *pos4, double *phi);

/* ---- particle hash (ParticleManager, SpaceHashClass.h:10-84) -------------- */
typedef struct pppm_hash pppm_hash;
pppm_status pppm_hash_create(uint32_t capacity, uint32_t g, float h, const float origin[3], pppm_hash **out);
void pppm_hash_destroy(pppm_hash *hs);
pppm_status pppm_hash_set_grid(pppm_hash *hs, uint32_t g, float h, const float origin[3]);
/* keys, stable sort by (key, index), start/end tables (empty cells 0xFFFFFFFF) */
pppm_status pppm_hash_build(pppm_hash *hs, const float *pos4, uint32_t n, void *hip_stream);
pppm_status pppm_hash_tables(pppm_hash *hs, const uint32_t **key_sorted, const uint32_t **index_sorted,
                             const uint32_t **cell_start, const uint32_t **cell_end);
/* out[i*stride+c] = in[index[i]*stride+c] (reorder) and its inverse (deorder) */
pppm_status pppm_hash_reorder(pppm_hash *hs, uint32_t n, const void *in, void *out, uint32_t stride,
                              int32_t dtype, void *hip_stream);
pppm_status pppm_hash_deorder(pppm_hash *hs, uint32_t n, const void *in, void *out, uint32_t stride,
                              int32_t dtype, void *hip_stream);

/* ---- primitives on caller buffers ----------------------------------------- */
/* keys[i] = cell key of pos4[i], idx[i] = i (particle_hash_kernel.cu:32-70) */
pppm_status pppm_calc_keys(const float *pos4, uint32_t n, uint32_t g, float h, const float origin[3],
                           uint32_t *keys, uint32_t *idx, void *hip_stream);
/* stable ascending sort of (keys, vals) pairs by key; scratch sized by
 * pppm_sort_scratch_bytes; key_bits = significant low bits of the keys */
size_t pppm_sort_scratch_bytes(uint32_t n);
pppm_status pppm_sort_pairs(uint32_t *keys, uint32_t *vals, uint32_t n, uint32_t key_bits, void *scratch,
                            void *hip_stream);
pppm_status pppm_cell_tables(const uint32_t *keys_sorted, uint32_t n, uint32_t ncells, uint32_t *start,
                             uint32_t *end, void *hip_stream);
pppm_status pppm_gather(const uint32_t *idx, const void *in, void *out, uint32_t stride, int32_t dtype,
                        uint32_t n, void *hip_stream);
pppm_status pppm_scatter(const uint32_t *idx, const void *in, void *out, uint32_t stride, int32_t dtype,
                         uint32_t n, void *hip_stream);

/* ---- multigrid on caller grids (MultiGrid.h:29-209) ------------------------- */
typedef struct pppm_mg pppm_mg;
/* dtype PPPM_F32 or PPPM_F64; nx,ny,nz arbitrary >= 1 */
pppm_status pppm_mg_create(int32_t nx, int32_t ny, int32_t nz, int32_t dtype, pppm_mg **out);
/* Batched form: x and b hold ncomp (1..48) grids one after another
 * (component-major), solved together with one launch per pass over all of
 * them, as the three vector-potential components of BiotSavartSolverImp.cpp:
 * 603-620 (m_SolvePoisson, there three sequential solves), or several scenes'
 * components at once.  pppm_mg_solve then reports the worst component's
 * relative residual. */
pppm_status pppm_mg_create_batched(int32_t nx, int32_t ny, int32_t nz, int32_t dtype, int32_t ncomp, pppm_mg **out);
void pppm_mg_destroy(pppm_mg *mg);
pppm_status pppm_mg_levels(const pppm_mg *mg, int32_t *levels, int32_t dims_out[][3], int32_t max_levels);
/* Solve sum_nb(x) - 6 x = b (zero ghosts) in place on x.  schedule
 * PPPM_MG_REF_FMG = one full-multigrid pass + one V-cycle (the reference);
 * PPPM_MG_REF_VCYCLE = one V-cycle with the reference's transfers
 * (MultiGrid.cpp:128-201 from level 0);
 * PPPM_MG_VCYCLE = V(nu1,nu2) cycles until ||b - A x|| / ||b|| <= tol.
 * cycles_out / relres_out may be NULL. */
pppm_status pppm_mg_solve(pppm_mg *mg, void *x, const void *b, int32_t schedule, int32_t nu1, int32_t nu2,
                          double omega, double tol, int32_t max_cycles, int32_t *cycles_out,
                          double *relres_out, void *hip_stream);

/* `count` V(nu1,nu2) cycles of the PPPM_MG_VCYCLE form in place on x
 * (x_zero: x holds no starting value), asynchronous on the stream, with no
 * residual norms in between: MultiGrid.cpp:128-201 (m_Vcycle) repeated. */
pppm_status pppm_mg_vcycles(pppm_mg *mg, void *x, const void *b, int32_t nu1, int32_t nu2, double omega,
                            int32_t count, int32_t x_zero, void *hip_stream);

/* iters red-black SOR iterations (odd colour first, MultiGrid_kernel.cu:722-820)
 * on the finest level, in place on x.  blocked (PPPM_F32 only): 0 one launch
 * per half-sweep; 1 temporally blocked LDS passes; 2 colour-split blocked
 * passes (four-plane ring); 3 the same with a six-plane ring; 4 passes of two
 * iterations, an odd one by kind 2.  Kinds 2 to 4 take kind 1's kernel when nx
 * is odd.  The results are the same, bit for bit, whichever it is.  Kinds 1 to
 * 4 pass through the handle's buffers: their calls on one handle must not
 * overlap.  Kind 0 touches x and b alone, in PPPM_F64 always. */
pppm_status pppm_mg_smooth(pppm_mg *mg, void *x, const void *b, int32_t iters, double omega, int32_t blocked,
                           void *hip_stream);
/* PPPM_F32 V-cycles on levels at or above the blocked threshold (below):
 * blocked = 1..4 (the kinds of pppm_mg_smooth; default 4) use fused blocked
 * passes, 0 one launch per half-sweep, residual, restriction and
 * prolongation. */
pppm_status pppm_mg_set_blocked(pppm_mg *mg, int32_t blocked);
/* Levels of even dimensions with at least this many cells per component take
 * the blocked passes in PPPM_F32 V-cycles (default 327680: 70^3 and larger);
 * at that default also smaller ones where the components together keep the
 * chip busy (from 851968 cells, or 294912 where tiles would be filled badly).
 * Other levels of even dimensions with fewer than 524288 cells take tile
 * passes (two red-black iterations with the residual or the prolongation in
 * one launch) unless a dimension is below 8 and the components hold 98304
 * cells or more; all others one launch per half-sweep or, with odd
 * dimensions, the blocked smoothing alone.  The results are the same, bit for
 * bit, whichever it is. */
pppm_status pppm_mg_set_blocked_min_cells(pppm_mg *mg, uint64_t cells);
/* PPPM_F32 V-cycles: one_launch = 1 (the default) runs the level above the
 * coarsest (when it is below that threshold and has at most 4096 cells, as
 * 16^3) with the coarsest solve in one launch, one workgroup per component
 * with the iterates in LDS; 0 runs them as one launch per half-sweep,
 * residual, restriction, coarsest solve and prolongation.  Both give the
 * same results, bit for bit.  PPPM_F64 cycles always take the one launch. */
pppm_status pppm_mg_set_small_levels(pppm_mg *mg, int32_t one_launch);

/* ---- device memory (MemoryOperation.cuh:13-29 semantics) -------------------- */
pppm_status pppm_device_count(int32_t *n);
pppm_status pppm_malloc(void **ptr, size_t bytes);
pppm_status pppm_free(void *ptr);
pppm_status pppm_memcpy_htod(void *dst, const void *src, size_t bytes);
pppm_status pppm_memcpy_dtoh(void *dst, const void *src, size_t bytes);
pppm_status pppm_memcpy_dtod(void *dst, const void *src, size_t bytes);
pppm_status pppm_memset(void *dst, int value, size_t bytes);
pppm_status pppm_synchronize(void);
const char *pppm_last_error(void);

/* Tracer evaluation as the simulation's caller runs it
 * (VortexSimulationSystemImp.cpp:1194-1244 evaluateBiotSavart): the m points
 * in batches of at most `batch`, each batch's velocity (evaluated like
 * pppm_evaluate, FP64) added into vel4 (double4 per point,
 * GPU_kernel.cu:3589-3606 AddURotation); when move != 0 each point is then
 * advanced by forward Euler, pos = (float)((double)pos + vel dt) with w = 0
 * (GPU_kernel.cu:3118-3140 move_particle).  pos4 and vel4 are device
 * pointers, updated in place on the context's stream.  The reference's batch
 * is 163,840 points; any batch gives the same velocities to FP32 rounding.
 * Requires pppm_compute_far_field. */
pppm_status pppm_evaluate_tracers(pppm_ctx *ctx, uint32_t m, float *pos4, double *vel4, uint32_t batch, double dt,
                                  int32_t move);

/* ---- frame output (newTest.cpp:23-37 output()) ------------------------------ */
/* Writes dir/Particle_data%04d.bin: n particles as raw float4 (x, y, z, w),
 * w = 1 as the reference writes it, or w[i] when w is given (the reference
 * renderer reads w as the particle's density, read_particles.cpp:55-70).
 * pos4 (float4 per particle) and w are device pointers; the copy runs on
 * hip_stream (null: the default stream) in chunks of 2^20 particles through
 * pinned host memory.  PPPM_ERR_INVALID if the file cannot be written. */
pppm_status pppm_write_frame(const char *dir, int32_t frame, const float *pos4, const float *w, uint32_t n,
                             void *hip_stream);

/* ---- time step of the vortex-segment method --------------------------------
 * VortexSimulationSystemImp.cpp:90-125 (solveTimeStep) and its kernels,
 * GPU_kernel.cu:3118-3254, 3327-3460, 3589-3606.  Device pointers; positions
 * are float4 (x, y, z, w), velocities double4; enqueued on hip_stream (null:
 * the default stream).  FP64 arithmetic rounded through float where the
 * reference's is, with no fused multiply-adds.  n = 0 does nothing. */

/* ComputePosb (GPU_kernel.cu:3182-3235): segment ends enda = c - s/2,
 * endb = c + s/2 about each centre, s = w when |w| < h (kappa = 1), else
 * s = w h / |w| (kappa = |w| / h).  The ends' w fields are not written. */
pppm_status pppm_segments_from_vortices(const float *cent4, float *enda4, float *endb4, const double *wx,
                                        const double *wy, const double *wz, double *kappa, double h, uint32_t n,
                                        void *hip_stream);
/* move_particle (GPU_kernel.cu:3118-3140): pos += u dt in FP64, w = 0. */
pppm_status pppm_move_points(float *pos4, const double *u4, double dt, uint32_t n, void *hip_stream);
/* ComputePosa (GPU_kernel.cu:3237-3254): cent.xyz = 0.5 (enda + endb), the
 * sum in float; cent.w is not written. */
pppm_status pppm_segment_centres(const float *enda4, const float *endb4, float *cent4, uint32_t n,
                                 void *hip_stream);
/* applyFlow without a boundary (VortexSimulationSystemImp.cpp:277-300): both
 * ends moved by their velocities and the centre re-formed, in one pass; the
 * same results as two pppm_move_points and one pppm_segment_centres. */
pppm_status pppm_apply_flow(float *enda4, float *endb4, float *cent4, const double *ua4, const double *ub4,
                            double dt, uint32_t n, void *hip_stream);
/* ComputeVortex (GPU_kernel.cu:3143-3180): dw = kappa (endb - enda) - w, the
 * difference of positions in float. */
pppm_status pppm_vortices_from_segments(const float *enda4, const float *endb4, const double *wx,
                                        const double *wy, const double *wz, double *dwx, double *dwy,
                                        double *dwz, const double *kappa, uint32_t n, void *hip_stream);
/* VectorAdd (GPU_kernel.cu:3442-3460): C = a A + b B (C may be A or B). */
pppm_status pppm_vector_add(const double *A, const double *B, double *C, double a, double b, uint32_t n,
                            void *hip_stream);
/* AddURotation (GPU_kernel.cu:3589-3606): U.xyz += (u, v, w). */
pppm_status pppm_add_velocity(double *U4, const double *u, const double *v, const double *w, uint32_t n,
                              void *hip_stream);
/* computeStretching's smoothing (VortexSimulationSystemImp.cpp:466-520,
 * ParticleGaussianSmooth GPU_kernel.cu:3327-3438) over the vortices of the
 * last pppm_set_vortices: o[i] = sum_p e^{-d^2/(2 nu^2)} v[p] / sum_p
 * e^{-d^2/(2 nu^2)} over the vortices p of the hash cells within +-2 of i's
 * cell (the reference passes nu = 0.1).  v and o are caller-order FP64 with
 * strides (in elements); o may be v.  Runs on the context stream; the
 * context keeps n double4 of scratch. */
pppm_status pppm_smooth_vorticity(pppm_ctx *ctx, const double *vx, const double *vy, const double *vz,
                                  uint32_t v_stride, double *ox, double *oy, double *oz, uint32_t o_stride,
                                  double nu);

/* setDomain (BiotSavartSolverImp.cpp:378-409, run by sortVort and
 * computeFarFieldBuffer, 731-770) over device positions: the bounding box
 * by a device reduction (min and max are exact), then origin = box centre -
 * L/2, h = L / g with L = 3 * the largest extent -- the same numbers as
 * pppm_reference_domain on a host copy.  Synchronises the context stream. */
pppm_status pppm_domain_device(pppm_ctx *ctx, const float *pos4, uint32_t n, double origin_out[3], double *h_out);
/* One step of solveTimeStep (VortexSimulationSystemImp.cpp:90-125) for a
 * flow without boundary, heat or density: convertVortToSeg (segment ends
 * about the centres, length min(|w|, seg_h)); computeURotation (the centres
 * hashed on their own domain, the far field, the velocity at each end with
 * the own vortex excluded, in the context's precision); applyFlow (forward
 * Euler of both ends, centres re-formed); convertSegToVort; computeStretching
 * (w + dw smoothed with pppm_smooth_vorticity's Gaussian over the new
 * centres, nu as given; the reference uses seg_h = 0.1, nu = 0.1).  cent4
 * and w (FP64, n each) are updated in place; the context keeps 128 bytes per
 * vortex of step state.  The domain follows the reference: before each
 * hashing (velocities, smoothing) it is set from the centres by
 * pppm_domain_device.  flags PPPM_STEP_KEEP_DOMAIN keeps the context's
 * domain instead (a fixed grid, as a long run on a given grid uses; vortices
 * outside it are handled as by pppm_set_vortices).  PPPM_STEP_RK2 replaces
 * the reference's forward Euler of the ends by Heun's method: the ends are
 * predicted with the first velocities, the predicted segments give centres
 * and strengths w + dw, the velocities at the predicted ends are taken from
 * those vortices, and the ends move with the mean of the two velocities
 * (two velocity evaluations per step; 96 more bytes per vortex). */
enum { PPPM_STEP_KEEP_DOMAIN = 1, PPPM_STEP_RK2 = 2 };
pppm_status pppm_time_step(pppm_ctx *ctx, uint32_t n, float *cent4, double *wx, double *wy, double *wz, double dt,
                           double seg_h, double nu, int32_t flags);

/* ---- baroclinic source (addBaroclinicForce) ---------------------------------
 * VortexSimulationSystemImp.cpp:369-465 with setDensityDomain (320-367) and
 * the kernels AssignDensity, GradDensity, ParticleGetBaroclinic
 * (GPU_kernel.cu:3655-3898).  The smoke particles (float4 positions, float
 * values) get a density grid over 1.2 x their extent with dim =
 * min(floor(L / cell_target) + 1, max_dim) cells per axis (the reference:
 * cell_target 0.2, max_dim 200); the grid value is the (1 - d^2)^4-weighted
 * mean of the particles within one cell (an empty cell counts its own centre
 * with value 0); its periodic central differences are interpolated at each
 * vortex with hat weights, and w += dt_beta * 0.1 * (grad rho x g) (the
 * reference: dt_beta = 5 dt, g = (0, 10, 0)).  A density object keeps its
 * buffers between calls.  Device pointers; enqueued on hip_stream, with one
 * synchronisation for the smoke's bounding box.  nheat = 0 does nothing.
 * Before pppm_time_step on the same strengths, pass the context's stream
 * (pppm_get_stream) or synchronise: the two are not ordered otherwise. */
typedef struct pppm_density pppm_density;
pppm_status pppm_density_create(pppm_density **out);
void pppm_density_destroy(pppm_density *d);
pppm_status pppm_add_baroclinic(pppm_density *d, const float *heat_pos4, const float *heat_rho, uint32_t nheat,
                                const float *cent4, double *wx, double *wy, double *wz, uint32_t n, double dt_beta,
                                const double gvec[3], double cell_target, uint32_t max_dim, void *hip_stream);
/* The last call's grid: density (dim^3 floats), gradient (3 floats per cell),
 * dim, origin and cell size; device pointers owned by the object. */
pppm_status pppm_density_grid(const pppm_density *d, const float **rho, const float **grad3, uint32_t *dim,
                              double origin[3], double *h);

/* ---- timing on the library's streams --------------------------------------- */
typedef struct pppm_timer pppm_timer;
pppm_status pppm_timer_create(pppm_timer **out);
void pppm_timer_destroy(pppm_timer *t);
pppm_status pppm_timer_start(pppm_timer *t, void *hip_stream);
pppm_status pppm_timer_stop(pppm_timer *t, void *hip_stream);
pppm_status pppm_timer_elapsed_ms(pppm_timer *t, float *ms);

#ifdef __cplusplus
}
#endif
#endif
