// Internal declarations shared by the library's translation units.
#pragma once
#include <mutex>

#include "pppm_common.hpp"
#include "../../include/pppm.h"

namespace pppm {

// Serialises HIP graph capture against device allocation, release and
// synchronous copies anywhere in the process: the runtime may invalidate a
// capture (or refuse the call) when they overlap, and the request server runs
// captures and context creation or eviction on different threads.
std::mutex& runtime_mutex();

// ---- scan ----------------------------------------------------------------
size_t scan_scratch_words(uint64_t n);
pppm_status exclusive_scan_u32(const uint32_t* in, uint32_t n, uint32_t* out, uint32_t* scratch, hipStream_t st);
pppm_status cell_offsets_from_tables(const uint32_t* start, const uint32_t* end, uint32_t ncells, uint32_t* off,
                                     uint32_t* scratch, hipStream_t st);

// ---- hash / sort ---------------------------------------------------------
struct HashGeom {
    uint32_t g;
    float hf;
    float of[3];
};
size_t sort_scratch_bytes(uint32_t n);
uint32_t key_bits_for(uint64_t ncells);
// octant: key = 8 * cell + octant of the point within its cell (the
// halves in x, y and z of the hash quotient; needs 8 * cells <= 2^32), so a
// sort orders each cell's points by octant.
// clamp: evaluation-point keys (eval_cell_key), cells clamped into the grid.
pppm_status launch_calc_keys(const float4* pos, uint32_t n, const HashGeom& hg, uint32_t* keys, uint32_t* idx,
                             hipStream_t st, bool octant = false, bool clamp = false);
// Sorts (keys, vals) by key, stable; on return *keys_out/*vals_out point at
// whichever buffer pair holds the result.  vals_identity: the input values
// are 0..n-1 and vals is not read.
pppm_status radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt, uint32_t n,
                             uint32_t key_bits, bool vals_identity, void* scratch, uint32_t** keys_out,
                             uint32_t** vals_out, hipStream_t st);
pppm_status launch_fill_u32(uint32_t* a, uint64_t n, uint32_t v, hipStream_t st);
// cell = key >> shift (3 for octant keys); off (null: not wanted): the cells'
// first keys, ncells + 1, with scan_scratch of scan_scratch_words(ncells)
pppm_status launch_cell_tables(const uint32_t* keys_sorted, uint32_t n, uint32_t ncells, uint32_t* start,
                               uint32_t* end, hipStream_t st, uint32_t shift = 0, uint32_t* off = nullptr,
                               uint32_t* scan_scratch = nullptr);
pppm_status launch_gather(const uint32_t* idx, const void* in, void* out, uint32_t stride, int dtype, uint32_t n,
                          hipStream_t st);
pppm_status launch_scatter(const uint32_t* idx, const void* in, void* out, uint32_t stride, int dtype, uint32_t n,
                           hipStream_t st);

// Geometry of the PPPM path as the reference uses it: hash in float,
// P2M/M2P/near field with the double origin and (double)(float)h.
struct PathGeom {
    HashGeom hash;
    double origin[3];
    double h;      // (double)(float)h
    double invh;   // 1 / h
};

// Sorted vortex arrays: spos = origin-shifted float coords + deposit-cell key
// in .w (as bits; 0xFFFFFFFF outside the grid); somg = strengths (x,y,z,0).
// idx: sorted slot -> caller index; inv (n words of scratch) receives its
// inverse.
pppm_status launch_reorder_vortices_scatter(const uint32_t* idx, uint32_t* inv, const float4* pos, const void* wx,
                                            const void* wy, const void* wz, uint32_t w_stride, int w_dtype,
                                            uint32_t n, const PathGeom& pg, float4* spos, float4* somg,
                                            uint32_t* strays, hipStream_t st);
// Sorted evaluation points: shifted coords, optional other end (shifted).
pppm_status launch_reorder_eval(const uint32_t* idx, const float4* pos, const float4* other, uint32_t m,
                                const PathGeom& pg, float4* epos, float4* eoth, hipStream_t st);

// ---- P2M -----------------------------------------------------------------
// sflag: one byte per cell, zero on entry; P2M sets the deposit cells of
// strays and the stray pass clears them again.
pppm_status launch_p2m(const uint32_t* off, const float4* spos, const float4* somg, uint32_t g, double invh,
                       float* wgrid /*[3][G]*/, double* b64 /*[3][G] or null*/, double bscale64, uint8_t* sflag,
                       hipStream_t st);
// adds the strays' strengths when *strays (device) is non-zero; a no-op launch otherwise
pppm_status launch_p2m_strays(const uint32_t* off, const float4* spos, const float4* somg, uint32_t g, double invh,
                              float* wgrid, double* b64, double bscale64, const uint32_t* strays, uint8_t* sflag,
                              hipStream_t st);

// The reference's FP64 deposit (ParticleToMesh, GPU_kernel.cu:218-271) on a
// cubic grid and a scale (ComputeRHS), on a stream.
pppm_status launch_pm_p2m(const uint32_t* start, const uint32_t* end, const float4* pos, const double* mass,
                          double cell_h, double* grid, uint32_t g, uint32_t n, double ox, double oy, double oz,
                          hipStream_t st);
pppm_status launch_pm_scale(double* a, uint32_t n, double s, hipStream_t st);

// ---- far field -----------------------------------------------------------
pppm_status launch_curl_far(const void* psi /*[3][G]*/, int psi_dtype, const float* wgrid, float* far, uint32_t g,
                            int K, double h, hipStream_t st);

// ---- M2P + near field ------------------------------------------------------
struct NearArgs {
    const float4* epos;      // sorted shifted eval coords
    const float4* eoth;      // sorted shifted other ends or null
    const uint32_t* eidx;    // eval sorted -> caller index
    uint32_t m;
    const uint32_t* off;     // vortex cell offsets [G+1]
    uint32_t nsrc;           // vortex count (off[G])
    const float4* spos;      // sorted shifted vortex coords
    const float4* somg;      // sorted vortex strengths
    const float* far;        // [3][G]
    uint32_t g;
    int K;
    int kernel;
    double invh;
    double core_a;
    void* ux;
    void* uy;
    void* uz;
    uint32_t u_stride;
    int u_dtype;
    const uint32_t* tperm = nullptr;  // evaluation slot -> sorted point, or null
    double pot_g = 1.0;               // potential kernels: G times the direction
};
// Near-field kernels of the potential-flow solver (not public kernel ids):
// the gradient G m (x_m - x) / (4 pi max(r, a)^3) and the potential
// G m / (4 pi max(r, a)), with the mass in the strength's x component.
constexpr int kNearPotGrad = 100;
constexpr int kNearPotScalar = 101;
// Octant order of sorted points within their hash cells (see nearfield.hip).
// Evaluation order in super-blocks of cells (nearfield.hip): a slot per x
// segment of a row; tperm maps evaluation slot -> sorted point.
struct SbGeom {
    uint32_t g, nX, nY, nslots;
};
struct SbBuffers {
    uint32_t *start, *len, *pre, *scratch;  // nslots each; scratch: scan_scratch_words(nslots)
};
SbGeom sb_geom(uint32_t g);
pppm_status launch_sb_order(const uint32_t* keys, uint32_t osh, uint32_t n, const SbGeom& s, SbBuffers b,
                            uint32_t* tperm, hipStream_t st);
pppm_status launch_octant_order(const uint32_t* ks, const float4* pos, uint32_t n, double invh, uint32_t* perm,
                                hipStream_t st);
pppm_status launch_m2p_near(const NearArgs& a, hipStream_t st);
pppm_status launch_count_pairs(const NearArgs& a, unsigned long long* d_total, hipStream_t st);

// ---- time step (timestep.hip) ----------------------------------------------
// Gaussian smoothing of caller-order FP64 values over the sorted vortices
// (spos, coff, idx of the context's hash); scratch holds n double4.
pppm_status launch_gaussian_smooth(const float4* spos, const uint32_t* coff, const uint32_t* idx, uint32_t n,
                                   const PathGeom& pg, double nu, const double* vx, const double* vy,
                                   const double* vz, uint32_t v_stride, double* ox, double* oy, double* oz,
                                   uint32_t o_stride, double4* scratch, hipStream_t st);
// The same over a caller's start/end tables and sorted arrays.
void launch_gaussian_smooth_tables(const uint32_t* start, const uint32_t* end, const float4* pos,
                                   const float4* pos_sort, double nu, double* ox, double* oy, double* oz,
                                   const double* ix, const double* iy, const double* iz, double h, uint3 hd,
                                   uint32_t n, double4 origin, hipStream_t st);

// Bounding box of device positions into scratch (bbox_scratch_floats()
// floats): the six results (min xyz, max xyz) at scratch + 6 * 1024.
size_t bbox_scratch_floats();
pppm_status launch_bbox(const float4* pos, uint32_t n, float* scratch, hipStream_t st);

}  // namespace pppm

// Request-server groups (csrc/api.hip): several small scenes with identical
// parameters (mixed precision, V-cycle schedule, grids of at most max_g cells
// per axis) have their Poisson solves run in one set of launches.
struct pppm_group;
size_t group_bytes(uint32_t g, int cap);
bool group_eligible(const pppm_params& p, uint32_t max_g);
pppm_status group_create(uint32_t g, int cap, pppm_group** out);
void group_destroy(pppm_group* q);
size_t group_device_bytes(const pppm_group* q);
// The far field of `count` contexts whose vortices are set: P2M on each
// context's stream, the solves together on the group's stream, then curl and
// far field on each context's stream (no host wait after the last launches).
pppm_status group_compute_far_field(pppm_group* q, pppm_ctx* const* ctxs, int count);

// A context's sorted sources, for solvers built on its hash (the potential-flow
// solver): its stream, the cell start/end tables, the sorted slot -> caller
// index map and the count.
struct CtxSources {
    hipStream_t st;
    const uint32_t* start;
    const uint32_t* end;
    const uint32_t* idx;
    uint32_t n;
};
pppm_status ctx_sources(pppm_ctx* c, CtxSources* out);
// The sorted-segment deposit of the context's strengths (no atomics; FP64
// sums of the FP32 sorted strengths, strays added): out[3][g^3] = h^-3 sum w
// per cell and component; wg_scratch is a [3][g^3] float array it also fills.
pppm_status ctx_p2m_x64(pppm_ctx* c, float* wg_scratch, double* out);
// pppm_evaluate with another near-field kernel (kNearPotGrad, kNearPotScalar),
// core radius, FP32 [3][g^3] far-field buffer and kernel factor.
pppm_status ctx_evaluate_with(pppm_ctx* c, uint32_t m, const float* eval_pos4, int kernel, double core_a,
                              const float* far, double pot_g, void* ux, void* uy, void* uz, uint32_t u_stride,
                              int32_t u_dtype);

