// Geometric multigrid hierarchy for the cell-centred 7-point Poisson problem
// sum_nb(x) - 6 x = b with zero ghost values (multigrid/multigrid/MultiGrid.h,
// MultiGrid.cpp, MultiGrid_kernel.cu).  Several independent components (the
// three stream-function components) are solved together: arrays are
// component-major [ncomp][nx*ny*nz].
#pragma once
#include "pppm_internal.hpp"
#include <vector>

namespace pppm {

enum { PROLONG_CONSTANT = 0, PROLONG_TRILINEAR = 1 };

// Ghost factor of level l of the tolerance-driven cycle (l = 0: 0).
double mg_beta(int level);

template <typename T>
class MGHier {
   public:
    MGHier() = default;
    ~MGHier() { release(); }
    MGHier(const MGHier&) = delete;
    MGHier& operator=(const MGHier&) = delete;

    pppm_status init(int nx, int ny, int nz, int ncomp);
    void release();
    // whether every dimension of level l is even
    bool even(int l) const { return !((d_[l][0] | d_[l][1] | d_[l][2]) & 1); }
    int levels() const { return L_; }
    int ncomp() const { return ncomp_; }
    // Work on the first n of the components the hierarchy was made for (n <=
    // that count).  Arrays are component-major, so the first n components of
    // every level are a prefix of the same arrays; a server solving several
    // small scenes together sets the count of scenes in the batch.
    pppm_status set_active(int n) {
        if (n < 1 || n > cap_) return PPPM_ERR_INVALID;
        ncomp_ = n;
        return PPPM_OK;
    }
    int capacity() const { return cap_; }
    const int* dims(int l) const { return d_[l]; }
    size_t cells(int l) const { return (size_t)d_[l][0] * d_[l][1] * d_[l][2]; }
    size_t device_bytes() const { return bytes_; }
    // device bytes init(nx, ny, nz, ncomp) allocates
    static size_t bytes_for(int nx, int ny, int nz, int ncomp);

    // One V(nu1,nu2) cycle from level l0 on (x0, b0 * bscale0) at level 0.
    // consistent: trilinear prolongation and boundary-consistent coarse
    // operators (tolerance-driven cycle); otherwise the reference pair
    // (piecewise-constant prolongation, zero ghosts on every level).
    // x0_zero: x0 holds no starting value (treated as zero; its contents are
    // not read)
    pppm_status vcycle(T* x0, const T* b0, T bscale0, int nu1, int nu2, T omega, bool consistent, hipStream_t st,
                       bool x0_zero = false);
    // MultiGrid.cpp:202-250 (m_FullMultiGrid): one FMG pass plus one V-cycle.
    pppm_status ref_fmg(T* x0, const T* b0, T bscale0, int nu1, int nu2, T omega, hipStream_t st);
    // ||b*bscale - A x||_2 and ||b*bscale||_2 per component (FP64 sums), synchronous.
    pppm_status norms(const T* x0, const T* b0, T bscale0, double* rn, double* bn, hipStream_t st);
    // the same in two halves: device reduction only (capturable), then the
    // synchronous readback of the reduced sums
    pppm_status norms_launch(const T* x0, const T* b0, T bscale0, hipStream_t st);
    pppm_status norms_read(double* rn, double* bn, hipStream_t st);
    // Repeated V-cycles until max relative residual <= tol or max_cycles.
    pppm_status solve(T* x0, const T* b0, T bscale0, int nu1, int nu2, T omega, double tol, int max_cycles,
                      int* cycles, double* relres /*[ncomp]*/, hipStream_t st);

    // raw pieces (also used by the reference-named entry points)
    pppm_status smooth(int l, T* x, const T* b, T bscale, int iters, T omega, T beta, hipStream_t st);
    // red-black iterations with one launch per colour, in place
    pppm_status smooth_colour(int l, T* x, const T* b, T bscale, int iters, T omega, T beta, hipStream_t st);
    pppm_status residual_restrict(int l, const T* x, const T* b, T bscale, T beta, T* bnext, hipStream_t st);
    pppm_status prolong(int l, T* x, const T* xc, int mode, T betac, hipStream_t st);
    pppm_status coarse(T* x, const T* b, T bscale, bool consistent, hipStream_t st);
    pppm_status fill(T* p, size_t n, hipStream_t st);
    pppm_status copy(T* d, const T* s, size_t n, hipStream_t st);
    // out-of-place target of the blocked passes at level l (null where
    // has_temp is false)
    T* temp(int l) { return t_[l]; }
    // whether level l of L has an out-of-place target: every float level
    // (blocked smoother, tile passes), the double ones that take tile passes
    // (below kTileCells) or k_rb4 (even nx, up to 256^3) but not the small
    // levels' one launch.  +134 MB a component at 256^3 in FP64.
    static bool has_temp(const int (*d)[3], int L, int l);
    double* partials() { return part_; }
    // the reduced norms, 2 per component (||r||^2, ||b||^2), after the partials
    double* norm_out() { return part_ + (size_t)kNormBlocks * ncomp_ * 2; }
    double* host_norms() { return hnorm_; }
    // partial-sum slots per component (the defect-correction step uses one
    // per workgroup: up to 4096 at 1024^3); the residual norm uses kResBlocks
    static constexpr int kNormBlocks = 4096;
    // components a hierarchy can hold (several requests' three components
    // when the server solves small scenes together)
    static constexpr int kMaxComp = 48;
    static constexpr int kResBlocks = 2048;
    // float smoothing on large levels: 0 one launch per colour, 1 blocked
    // passes (k_rb2), 2 colour-split blocked passes with a four-plane ring,
    // 3 the same with a six-plane ring, 4 (the default) two iterations in one
    // pass (k_rb4) wherever two follow each other, and kind 2 for the rest
    void set_blocked_smoother(int kind) { tb_ = kind; }
    int blocked_smoother() const { return tb_; }
    // V-cycles run the blocked passes on levels with at least this many cells
    // per component (blocked_level), the tile passes below
    void set_blocked_min_cells(size_t n) { tb_min_cells_ = n; }
    size_t blocked_min_cells() const { return tb_min_cells_; }
    // V-cycles: the level above the coarsest and the coarsest solve in one
    // launch (k_vtail) where they fit, or apart
    void set_small_one_launch(bool on) { tail_ = on; }
    bool small_one_launch() const { return tail_; }
    // the level L - 2 of that launch, or -1 where it does not apply
    int tail_level() const;
    // that launch, on that level's iterate x (xin: its start, null: zero),
    // its right-hand side b (times bscale) and the coarsest one's b1 (written)
    pppm_status tail(const T* xin, T* x, const T* b, T* b1, T bscale, int nu1, int nu2, T omega, bool consistent,
                     hipStream_t st);
    // whether level l takes passes of two iterations over the whole level in
    // FP64 (k_rb4)
    bool wide_level(int l) const {
        return sizeof(T) == 8 && tb_ && cells(l) * (size_t)ncomp_ >= kRb4Doubles && t_[l] && !(d_[l][0] & 1);
    }
    // whether level l of a V-cycle takes the FP32 blocked passes (if its
    // dimensions let it)
    bool blocked_level(int l) const;
    // a dimension of fewer than 8 cells
    bool thin(int l) const { return d_[l][0] < 8 || d_[l][1] < 8 || d_[l][2] < 8; }
    // edge of level l's tiles
    int tile_size(int l) const {
        return sizeof(T) == 4 && cells(l) * (size_t)ncomp_ >= kTile16Cells ? 16 : 8;
    }
    // whether level l of a V-cycle takes the tile passes (k_tile)
    bool tile_level(int l, bool consistent) const;
    // one tile pass, xin (null: zero) -> x: the prolongation of xc added
    // (null: none), 1 or 2 red-black iterations, the residual restricted into
    // bnext (null: none; not with xc)
    pppm_status tile(int l, const T* xin, T* x, const T* b, T bscale, int iters, T omega, T beta, T* bnext,
                     const T* xc, int mode, T betac, hipStream_t st);

   private:
    void release_locked();  // release() with runtime_mutex() already held
    int L_ = 0, ncomp_ = 1, cap_ = 1;
    int d_[16][3];
    std::vector<T*> x_, b_;       // levels >= 1, in xbase_
    T* xbase_ = nullptr;
    std::vector<T*> t_;           // out-of-place targets (has_temp), in tbase_
    T* tbase_ = nullptr;
    double* tab_cons_ = nullptr;  // coarse eigenbasis, consistent ghosts
    double* tab_ref_ = nullptr;   // coarse eigenbasis, zero ghosts
    double* part_ = nullptr;      // norm partial sums
    double* hnorm_ = nullptr;     // pinned host copy of the reduced norms
    size_t bytes_ = 0;
    int tb_ = 4;
    // Tile passes below kTileCells cells a component, in 16^3 tiles from
    // kTile16Cells cells over all components: fewer cells leave CUs without a
    // workgroup, more are worth the smaller halo (us of a V(2,2) cycle, all
    // levels in 8^3 / 16^3 tiles: 48^3 43 / 58, x 3 59 / 70, x 6 76 / 72; 64^3 55 /
    // 74, x 2 79 / 75, x 6 151 / 105; 32^3 x 6 36 / 39, x 16 61 / 41).
    static constexpr size_t kTileCells = (size_t)1 << 19;
    static constexpr size_t kTile16Cells = (size_t)1 << 19;
    // FP32 blocked passes (blocked_level) from kBlockedMin cells (us down and up,
    // tile against blocked: 64^3 10.4 against 13.8; 72^3 17 against 14, three
    // components 26 against 16), and below where the components together keep
    // the chip busy, as the tiles recompute more of their halo: from
    // kBlockedCells over all of them, or kBlockedPartial where the level fills its
    // tiles badly (us of four V(2,2) cycles, tile / blocked: 64^3 x 3 265 / 274,
    // x 6 404 / 333, x 48 1769 / 875; 52^3 x 6 449 / 308, x 3 302 / 254; 40^3 x 3
    // 196 / 231, x 12 325 / 246; 34^3 x 12 296 / 230).
    static constexpr size_t kBlockedMin = (size_t)5 << 16;
    static constexpr size_t kBlockedCells = (size_t)13 << 16, kBlockedPartial = (size_t)9 << 15;
    size_t tb_min_cells_ = kBlockedMin;
    // Levels with a dimension below 8 take no FP32 tiles from this many cells over
    // all components (us, tiles / a launch per half-sweep: 86 x 4 x 52 x 48 394 /
    // 315; 98 x 2 x 44 x 24 252 / 182; 64 x 64 x 2 x 12 127 / 116; below 98K tiles
    // are the faster).
    static constexpr size_t kThinCells = (size_t)3 << 15;
    // FP64 levels of at least this many cells over all components take k_rb4
    // (us of a full multigrid V(4,4), tiles against k_rb4: 32^3 x 3 183 against
    // 205, 48^3 289 against 302, 40^3 x 3 336 against 301, 56^3 355 against 325,
    // 64^3 374 against 338, 64^3 x 3 598 against 388).
    static constexpr size_t kRb4Doubles = (size_t)1 << 17;
    // FP64 levels with odd nx, which k_rb4 does not take, run a launch per
    // half-sweep from this many cells over all components, as their tiles
    // recompute more of the halo than the launches cost (us of two full
    // multigrid solves V(4,4), tiles / launches: 71^3 468 / 560, x 2 629 / 697,
    // x 3 842 / 834; 63^3 x 2 474 / 480, x 6 980 / 729; 45^3 x 12 828 / 700; 65^3
    // x 12 2050 / 1365).
    static constexpr size_t kOddTileDoubles = (size_t)3 << 18;
    bool tail_ = true;
};

// FP64 defect-correction step of the mixed-precision solve:
// x_out = x_in + e (x_in, e may be null = 0), r32 = (float)(b - A x_out),
// block partial sums of r^2 and b^2 into partials; reduced per component into
// out[2*c] = ||r||^2, out[2*c+1] = ||b||^2 (device, FP64).
pppm_status launch_dc_step(const double* x_in, const float* e, const double* b64, double* x_out, float* r32, int nx,
                           int ny, int nz, int ncomp, double* partials, double* out, hipStream_t st);

// Coarse eigenbasis tables: E_x, E_y, E_z (row k = eigenvector k), lam_x, lam_y,
// lam_z of the 1-D second difference with out-of-grid neighbour = beta * end value.
std::vector<double> coarse_tables(int nx, int ny, int nz, double beta);

// Single-array primitives of the reference's mg_* entry points.
template <typename T>
pppm_status ref_rbgs(T* x, const T* b, int iters, int nx, int ny, int nz, T omega, hipStream_t st);
template <typename T>
pppm_status ref_residual(const T* x, const T* b, T* r, int nx, int ny, int nz, hipStream_t st);
template <typename T>
pppm_status ref_restrict(T* bc, const T* rf, int cx, int cy, int cz, hipStream_t st);
template <typename T>
pppm_status ref_prolong(T* xf, const T* xc, int fx, int fy, int fz, hipStream_t st);
template <typename T>
pppm_status ref_coarse(T* res, const T* b, int nx, int ny, int nz, hipStream_t st);

}  // namespace pppm
