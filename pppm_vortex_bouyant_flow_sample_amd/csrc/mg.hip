// Multigrid kernels and hierarchy driver (see mg.hpp).
//   smoother      MultiGrid_kernel.cu:722-820, Multigrid.cu:202-239 (red/black SOR)
//   residual      MultiGrid_kernel.cu:821-871
//   restriction   MultiGrid_kernel.cu:873-910 (fused with the residual here)
//   prolongation  MultiGrid_kernel.cu:912-934 (piecewise constant) + trilinear
//   coarse solve  MultiGrid_kernel.cu:422-498 replaced by an exact eigenbasis solve
//   schedules     MultiGrid.cpp:128-250
#include "mg.hpp"
#include <cmath>
#include <cstring>
#include <type_traits>

namespace pppm {

double mg_beta(int level) {
    double s = std::ldexp(1.0, -level);
    return -(1.0 - s) / (1.0 + s);
}

// ---------------------------------------------------------------------------
template <typename T>
__device__ inline T nb_sum(const T* __restrict__ x, size_t t, int i, int j, int k, int nx, int ny, int nz,
                           int& nout) {
    const size_t sy = (size_t)nx, sz = (size_t)nx * ny;
    T lv = i > 0 ? x[t - 1] : (T)0;
    T rv = i < nx - 1 ? x[t + 1] : (T)0;
    T uv = j < ny - 1 ? x[t + sy] : (T)0;
    T dv = j > 0 ? x[t - sy] : (T)0;
    T fv = k > 0 ? x[t - sz] : (T)0;
    T bv = k < nz - 1 ? x[t + sz] : (T)0;
    nout = (i == 0) + (i == nx - 1) + (j == 0) + (j == ny - 1) + (k == 0) + (k == nz - 1);
    T r = lv + rv;
    r += uv + dv;
    r += fv + bv;
    return r;
}

// What k_rbgs, k_tile, k_vtail, k_rb2, k_rbc and k_rb4 do to a cell, to a residual and to
// a coarse value is written here once, with its fused multiply-adds spelt out
// and no others, so that a level's values are bitwise the same whichever of
// them runs it: the choice may go by the work of all components together, and a
// component solved with others is bitwise the one solved alone.
__device__ inline float fma_(float a, float b, float c) { return fmaf(a, b, c); }
__device__ inline double fma_(double a, double b, double c) { return fma(a, b, c); }
// relaxation factor over the diagonal 6 - beta nout of a cell with nout
// neighbours outside and a ghost factor beta; w6 = omega / 6 (from the
// host: a division a thread made k_rbgs<double> 2% slower)
template <typename T>
__device__ inline T relax_weight(int nout, T omega, T beta, T w6) {
    return beta == (T)0 || nout == 0 ? w6 : omega / fma_(-beta, (T)nout, (T)6);
}
// SOR update of a cell: x from the sum s of its neighbours, bscale times its
// right-hand side b, its relax_weight w and om1 = 1 - omega
template <typename T>
__device__ inline T relax(T x, T s, T b, T bscale, T w, T om1) {
#pragma clang fp contract(off)
    return fma_(w, fma_(-bscale, b, s), om1 * x);
}
// the same with om1 x formed in x's register once the sum is there: the blocked
// passes, which have few registers to spare, spill where it is formed early
__device__ inline double relax_late(double x, double s, double b, double bscale, double w, double om1) {
    return relax(x, s, b, bscale, w, om1);
}
__device__ inline float relax_late(float x, float s, float b, float bscale, float w, float om1) {
    const float r = fmaf(-bscale, b, s);
    __asm__("v_mul_f32 %0, %1, %0" : "+v"(x) : "s"(om1), "v"(r));
    return fmaf(w, r, x);
}
// residual of a cell, s the sum of its neighbours
template <typename T>
__device__ inline T residual_of(T x, T s, T b, T bscale, int nout, T beta) {
#pragma clang fp contract(off)
    s = fma_((T)-6, x, s);
    if (beta != (T)0) s = fma_(beta * (T)nout, x, s);
    return fma_(bscale, b, -s);
}
// 1 - w and w of a parent and its neighbour
template <typename T>
__device__ inline T lerp_(T w, T parent, T neighbour) {
#pragma clang fp contract(off)
    return fma_(w, neighbour, ((T)1 - w) * parent);
}
// coarse value c outside the coarse grid: ghost factors of the three axes
template <typename T>
__device__ inline T ghost(T fi, T fj, T fk, T c) {
#pragma clang fp contract(off)
    return ((fi * fj) * fk) * c;
}
// the 8 children's residuals of a coarse cell, p[y][z] the sums of the pairs
// along x: over z, then y
template <typename T>
__device__ inline T restrict_sum(T p00, T p10, T p01, T p11) {
    return ((p00 + p01) + (p10 + p11)) * (T)0.5;
}

// One colour of red-black SOR.  color 1 = (i+j+k) odd (swept first, as the
// reference's "red" kernel), 0 = even.  BETA: a ghost factor that is not zero.
template <typename T, bool BETA>
__global__ void __launch_bounds__(256) k_rbgs(T* __restrict__ x, const T* __restrict__ b, size_t G, int nx, int ny,
                                              int nz, int color, T bscale, T w6, T om1, T omega, T beta) {
    const int i2 = blockIdx.x * 64 + threadIdx.x;
    const int j = blockIdx.y * 4 + threadIdx.y;
    const int comp = blockIdx.z / nz, k = blockIdx.z - comp * nz;
    if (j >= ny) return;
    const int i = 2 * i2 + ((j + k + color) & 1);
    if (i >= nx) return;
    const size_t t = ((size_t)k * ny + j) * nx + i;
    T* xc = x + (size_t)comp * G;
    int nout;
    const T s = nb_sum(xc, t, i, j, k, nx, ny, nz, nout);
    xc[t] = relax(xc[t], s, b[(size_t)comp * G + t], bscale, BETA ? relax_weight(nout, omega, beta, w6) : w6, om1);
}

// one colour of ncomp components
template <typename T>
static void launch_rbgs(T* x, const T* b, T bscale, int nx, int ny, int nz, int ncomp, int color, T omega, T beta,
                        hipStream_t st) {
    dim3 blk(64, 4), grid(div_up(div_up(nx, 2), 64), div_up(ny, 4), nz * ncomp);
    const size_t G = (size_t)nx * ny * nz;
    const T w6 = omega / (T)6, om1 = (T)1 - omega;
    if (beta != (T)0)
        hipLaunchKernelGGL((k_rbgs<T, true>), grid, blk, 0, st, x, b, G, nx, ny, nz, color, bscale, w6, om1, omega, beta);
    else
        hipLaunchKernelGGL((k_rbgs<T, false>), grid, blk, 0, st, x, b, G, nx, ny, nz, color, bscale, w6, om1, omega, beta);
}

// Tile of the blocked smoother k_rb2 (below): 64 x 16 cells per workgroup.
constexpr int kTbTX = 64;
constexpr int kTbTY = 16;

template <typename T>
struct TbArgsT {
    const T* xin;    // level array before the pass (read only)
    T* x;            // level array after the pass (a different buffer)
    const T* b;      // right-hand side (times bscale)
    T bscale;
    int nx, ny, nz;
    size_t G;            // cells per component
    T omega, beta;   // SOR factor, ghost factor of this level
    T w6, om1;       // omega / 6, 1 - omega
    int zc;              // z planes per workgroup chunk (even)
    // RESTRICT: residual restricted into bn (coarse dims cx, cy, cz = n / 2)
    T* bn;
    int cx, cy, cz;
    size_t Gc;
    // PROLONG: x += trilinear(xc) on load (coarse dims cx, cy, cz, fine dims
    // even), ghost betac
    const T* xc;
    T betac;
};
using TbArgs = TbArgsT<float>;

// Trilinear prolongation (k_prolong's weights) at fine cell (i, j, k) from a
// coarse window held in LDS: cw[slot(c)][cy - cy0][cx - cx0] for coarse planes
// c, rows cy and columns cx; a neighbour outside the coarse grid is betac times
// the parent value.  Fine dimensions are even here, so parents are i / 2.
template <int CLX, int CLY>
__device__ inline float tb_prolong_lds(const float (*cw)[CLY][CLX], int i, int j, int k, int cx0, int cy0, int cx,
                                       int cy, int cz, float betac) {
    const int pi = i >> 1, pj = j >> 1, pk = k >> 1;
    int ni = (i & 1) ? pi + 1 : pi - 1, nj = (j & 1) ? pj + 1 : pj - 1, nk = (k & 1) ? pk + 1 : pk - 1;
    float fi = 1.f, fj = 1.f, fk = 1.f;
    if (ni < 0 || ni > cx - 1) { ni = pi; fi = betac; }
    if (nj < 0 || nj > cy - 1) { nj = pj; fj = betac; }
    if (nk < 0 || nk > cz - 1) { nk = pk; fk = betac; }
    const int sp = pk % 3, sn = nk % 3;
    const int ip = pi - cx0, in_ = ni - cx0, jp = pj - cy0, jn = nj - cy0;
    // the parent's or the neighbour's value on each axis
    auto C = [&](bool x, bool y, bool z) {
        return ghost(x ? fi : 1.f, y ? fj : 1.f, z ? fk : 1.f, cw[z ? sn : sp][y ? jn : jp][x ? in_ : ip]);
    };
    const float p0 = lerp_(0.25f, C(0, 0, 0), C(1, 0, 0)), p1 = lerp_(0.25f, C(0, 1, 0), C(1, 1, 0));
    const float p2 = lerp_(0.25f, C(0, 0, 1), C(1, 0, 1)), p3 = lerp_(0.25f, C(0, 1, 1), C(1, 1, 1));
    return lerp_(0.25f, lerp_(0.25f, p0, p1), lerp_(0.25f, p2, p3));
}

// Blocked red-black smoother: one red-black iteration (two half-sweeps) per
// pass over the grid.  A workgroup owns a 64 x 16 tile plus an H-cell halo in
// x and y and a chunk of z planes plus an H-plane halo; it streams the planes
// through LDS rings and applies half-sweep t to plane k - t right after plane
// k arrives.  In place in LDS is exact for red-black ordering: half-sweep t
// reads only the colour written by half-sweep t - 1, and in step k plane
// k - t has received half-sweeps 1..t-1 while its neighbours have not yet
// received t + 1.  Halo cells are recomputed redundantly; a cell at distance
// d from the loaded region's edge is valid for half-sweeps t <= d (sides on
// the grid boundary use the exact ghost rule).  H = 2, or 3 when the pass
// also forms the residual (which needs final values one cell beyond the
// tile).  Cells outside the grid hold zero in LDS and are never updated, and
// each LDS plane has one spare zero column and row, so neighbour reads need
// no bounds tests.  The pass reads xin and writes x: halos are loaded by other
// workgroups while this one writes its tile, so the two must not alias.
// BETA: coarse level, out-of-grid neighbours are beta times the cell value.
template <bool RESTRICT, bool PROLONG, bool XZERO, bool BETA>
__global__ void __launch_bounds__(256) k_rb2(TbArgs a) {
    constexpr int H = RESTRICT ? 3 : 2;
    constexpr int LX = kTbTX + 2 * H, LY = kTbTY + 2 * H;
    constexpr int LXP = LX + 1, LYP = LY + 1, PL = LXP * LYP;  // padded plane
    constexpr int NR = RESTRICT ? 5 : 4;  // planes of x alive at once
    constexpr int NB = RESTRICT ? 4 : 3;  // planes of b alive at once
    constexpr int NL = (LX * LY + 255) / 256;
    constexpr int HX = LX / 2;                    // cell pairs per row
    constexpr int NP = (HX * LY + 255) / 256;     // pair slots per thread
    constexpr int CLX = PROLONG ? LX / 2 + 3 : 1, CLY = PROLONG ? LY / 2 + 3 : 1;
    constexpr int NC = (CLX * CLY + 255) / 256;
    __shared__ float xs[NR * PL];
    __shared__ float bs[NB * PL];
    __shared__ float cw[PROLONG ? 3 : 1][CLY][CLX];
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    // tiles in x-fastest order, a contiguous range of them per XCD
    const uint32_t tile = xcd_block(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z),
                                    gridDim.x * gridDim.y * gridDim.z);
    const int bx = (int)(tile % gridDim.x), by = (int)((tile / gridDim.x) % gridDim.y);
    const int bz = (int)(tile / (gridDim.x * gridDim.y));
    const int gx0 = bx * kTbTX - H, gy0 = by * kTbTY - H;
    const int nzc = (nz + a.zc - 1) / a.zc;
    const int comp = bz / nzc, zi = bz - comp * nzc;
    const int z0 = zi * a.zc, z1 = min(z0 + a.zc, nz);
    const float* xsrc = a.xin + (size_t)comp * a.G;
    float* xc = a.x + (size_t)comp * a.G;
    const float* bcp = a.b + (size_t)comp * a.G;
    const float* xcoarse = PROLONG ? a.xc + (size_t)comp * a.Gc : nullptr;
    const int cx0 = (gx0 >> 1) - 1, cy0 = (gy0 >> 1) - 1;  // coarse window origin
    const int klo = max(z0 - H, 0), khi = min(z1 + H, nz);
    const bool xl_ghost = gx0 <= 0, xr_ghost = gx0 + LX >= nx;
    const bool yl_ghost = gy0 <= 0, yr_ghost = gy0 + LY >= ny;
    const float omega = a.omega, beta = a.beta;
    const int tid = threadIdx.x;

    // zero everything once: spare column / row and out-of-grid cells stay 0
    for (int q = tid; q < NR * PL; q += 256) xs[q] = 0.f;
    for (int q = tid; q < NB * PL; q += 256) bs[q] = 0.f;

    // this thread's pair slots: row ly, pair lx2 (cells 2 lx2 and 2 lx2 + 1)
    int sbase[NP], sly[NP], slx2[NP], spar[NP];
#pragma unroll
    for (int u = 0; u < NP; u++) {
        const int q = tid + 256 * u;
        const int ly = q < HX * LY ? q / HX : LY + 8;  // out of every update range
        const int lx2 = q < HX * LY ? q - ly * HX : 0;
        sly[u] = ly;
        slx2[u] = lx2;
        sbase[u] = ly * LXP + 2 * lx2;
        spar[u] = (gx0 + gy0 + ly) & 1;
    }

    // Plane k + 1 is fetched into registers while plane k is swept, so the
    // global loads overlap the sweeps; the coarse planes the prolongation
    // needs go through a three-plane LDS ring the same way.
    float px[NL], pb[NL], pc[NC];
    auto fetch = [&](int k) {
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int q = tid + 256 * u;
            const int ly = q / LX, lx = q - ly * LX;
            const int i = gx0 + lx, j = gy0 + ly;
            float xv = 0.f, bv = 0.f;
            if (q < LX * LY && i >= 0 && i < nx && j >= 0 && j < ny) {
                const size_t t = ((size_t)k * ny + j) * nx + i;
                if (!XZERO) xv = xsrc[t];
                bv = bcp[t];
            }
            px[u] = xv;
            pb[u] = bv;
        }
    };
    auto fetch_coarse = [&](int c) {
#pragma unroll
        for (int u = 0; u < NC; u++) {
            const int q = tid + 256 * u;
            const int cyl = q / CLX, cxl = q - cyl * CLX;
            const int ci = cx0 + cxl, cj = cy0 + cyl;
            float v = 0.f;
            if (q < CLX * CLY && c >= 0 && c < a.cz && ci >= 0 && ci < a.cx && cj >= 0 && cj < a.cy)
                v = xcoarse[((size_t)c * a.cy + cj) * a.cx + ci];
            pc[u] = v;
        }
    };
    auto store_coarse = [&](int c) {
        if (c < 0 || c >= a.cz) return;
#pragma unroll
        for (int u = 0; u < NC; u++) {
            const int q = tid + 256 * u;
            if (q < CLX * CLY) cw[c % 3][q / CLX][q % CLX] = pc[u];
        }
    };
    if (PROLONG) {
        // coarse planes of the first fine plane, synchronously
        for (int c = (klo >> 1) - 1; c <= (klo >> 1) + 1; c++) {
            fetch_coarse(c);
            store_coarse(c);
        }
    }
    fetch(klo);
    __syncthreads();  // zeroed rings before the first stores
    float rsum[2] = {0.f, 0.f};  // RESTRICT: this thread's coarse cell, its rows of the even plane
    for (int k = klo; k < khi + 2 + (RESTRICT ? 1 : 0); k++) {
        if (PROLONG) {
            if (k < khi && k > klo && (k & 1) == 0) store_coarse((k >> 1) + 1);  // fetched during plane k - 1
            __syncthreads();
        }
        if (k < khi) {
            float* xr = xs + (k % NR) * PL;
            float* br = bs + (k % NB) * PL;
#pragma unroll
            for (int u = 0; u < NL; u++) {
                const int q = tid + 256 * u;
                if (q < LX * LY) {
                    const int ly = q / LX, lx = q - ly * LX;
                    float xv = px[u];
                    if (PROLONG) {
                        const int i = gx0 + lx, j = gy0 + ly;
                        if (i >= 0 && i < nx && j >= 0 && j < ny)
                            xv += tb_prolong_lds<CLX, CLY>(cw, i, j, k, cx0, cy0, a.cx, a.cy, a.cz, a.betac);
                    }
                    xr[ly * LXP + lx] = xv;
                    br[ly * LXP + lx] = pb[u];
                }
            }
        }
        __syncthreads();
        if (k + 1 < khi) {
            fetch(k + 1);
            if (PROLONG && ((k + 1) & 1) == 0) fetch_coarse(((k + 1) >> 1) + 1);
        }
#pragma unroll
        for (int t = 1; t <= 2; t++) {
            const int p = k - t;
            const int plo = klo > 0 ? klo + t : 0;
            const int phi = khi < nz ? khi - 1 - t : nz - 1;
            if (p >= plo && p <= phi) {
                const int col = t & 1;  // odd colour first, as the reference
                const int ax = xl_ghost ? -gx0 : t, bxl = xr_ghost ? nx - 1 - gx0 : LX - 1 - t;
                const int ay = yl_ghost ? -gy0 : t, byl = yr_ghost ? ny - 1 - gy0 : LY - 1 - t;
                const float* xm = xs + ((p + NR - 1) % NR) * PL;
                float* x0 = xs + (p % NR) * PL;
                const float* xp = xs + ((p + 1) % NR) * PL;
                const float* b0 = bs + (p % NB) * PL;
                const bool zlo = p == 0, zhi = p == nz - 1;
                const int pc_ = (col + p) & 1;
#pragma unroll
                for (int u = 0; u < NP; u++) {
                    const int bit = spar[u] ^ pc_;
                    const int lx = 2 * slx2[u] + bit, ly = sly[u];
                    if (lx < ax || lx > bxl || ly < ay || ly > byl) continue;
                    const int o = sbase[u] + bit;
                    float r = x0[o - 1] + x0[o + 1];
                    r += x0[o - LXP] + x0[o + LXP];
                    r += (zlo ? 0.f : xm[o]) + (zhi ? 0.f : xp[o]);
                    float w = a.w6;
                    if (BETA) {
                        const int i = gx0 + lx, j = gy0 + ly;
                        const int nout = (i == 0) + (i == nx - 1) + (j == 0) + (j == ny - 1) + zlo + zhi;
                        w = relax_weight(nout, omega, beta, a.w6);
                    }
                    x0[o] = relax(x0[o], r, b0[o], a.bscale, w, a.om1);
                }
            }
            __syncthreads();
        }
        // plane k - 2 is final: write its tile interior
        const int pw = k - 2;
        if (pw >= z0 && pw < z1 && pw < khi) {
            const float* xr = xs + (pw % NR) * PL;
            for (int q = tid; q < kTbTX * kTbTY; q += 256) {
                const int ly = H + q / kTbTX, lx = H + (q % kTbTX);
                const int i = gx0 + lx, j = gy0 + ly;
                if (i < nx && j < ny) xc[((size_t)pw * ny + j) * nx + i] = xr[ly * LXP + lx];
            }
        }
        if (RESTRICT) {
            // residual of plane pr = k - 3 (its neighbours are final), summed
            // into the coarse cell (I, J) owned by this thread: 32 x 8 per tile
            const int pr = k - 3;
            if (pr >= z0 && pr < z1) {
                const int I = tid % (kTbTX / 2), J = tid / (kTbTX / 2);
                const float* xm = xs + ((pr + NR - 1) % NR) * PL;
                const float* x0 = xs + (pr % NR) * PL;
                const float* xp = xs + ((pr + 1) % NR) * PL;
                const float* b0 = bs + (pr % NB) * PL;
                const bool zlo = pr == 0, zhi = pr == nz - 1;
                float part[2] = {0.f, 0.f};  // the two rows
#pragma unroll
                for (int dj = 0; dj < 2; dj++)
#pragma unroll
                    for (int di = 0; di < 2; di++) {
                        const int lx = H + 2 * I + di, ly = H + 2 * J + dj;
                        const int i = gx0 + lx, j = gy0 + ly;
                        if (i >= nx || j >= ny) continue;
                        const int o = ly * LXP + lx;
                        float sres = x0[o - 1] + x0[o + 1];
                        sres += x0[o - LXP] + x0[o + LXP];
                        sres += (zlo ? 0.f : xm[o]) + (zhi ? 0.f : xp[o]);
                        const int nout = BETA ? (i == 0) + (i == nx - 1) + (j == 0) + (j == ny - 1) + zlo + zhi : 0;
                        const float r = residual_of(x0[o], sres, b0[o], a.bscale, nout, BETA ? beta : 0.f);
                        part[dj] = di == 0 ? r : part[dj] + r;
                    }
                if ((pr & 1) == 0) {
                    rsum[0] = part[0];
                    rsum[1] = part[1];
                } else {
                    const int gI = bx * (kTbTX / 2) + I, gJ = by * (kTbTY / 2) + J, gK = pr / 2;
                    if (gI < a.cx && gJ < a.cy && gK < a.cz)
                        a.bn[(size_t)comp * a.Gc + ((size_t)gK * a.cy + gJ) * a.cx + gI] =
                            restrict_sum(rsum[0], rsum[1], part[0], part[1]);
                }
            }
            // the next load reuses the ring slots of planes pr - 1 (x) and pr (b)
            __syncthreads();
        }
    }
}

// Colour-split blocked smoother: the pass of k_rb2 (z planes streamed through
// LDS rings, halos recomputed, out of place; one red-black iteration) with
// each LDS plane split by colour.  Row ly of colour c holds at index m the
// colour-c cell of the cell pair (2m, 2m + 1) of that row.  Every
// neighbour of a colour-c cell is of colour 1 - c: at index m in the rows
// above and below and in the planes before and after, and at m + s - 1 and
// m + s in its own row (s = 1 if the cell is the pair's second), so the reads
// of a half-sweep are contiguous across lanes.  A thread owns whole pairs: it
// loads them with 8-byte loads, keeps their right-hand side in registers and
// writes its own cells out.  The z loop is unrolled over the ring (NR planes,
// even, the loop aligned to multiples of NR), so ring slots and plane
// parities are compile-time and every LDS address is a per-slot register plus
// an immediate.  Planes outside the grid in z read as zero: the ring slot
// before the first plane is still zero while the first plane is swept, and a
// zero plane is stored after the last one.  Cells outside the grid in x and y
// are loaded as zero and keep zero (their relaxation factor is 0).  Rows
// beyond the loaded region read zero rows, and an x neighbour beyond a row's
// end reads the adjacent row's cell (rows are not padded, so a wave's reads
// cover 64 consecutive words); the values these produce at the loaded
// region's edge reach at most one cell further inward per half-sweep, which
// the halo absorbs.  Requires nx even: pairs never cross the x boundary, and
// the x halo is even for the same reason.
constexpr int kRcTX = 64;
constexpr int kRcTY = 16;

// The passes that also restrict or prolong hold up to ~190 VGPRs when left
// alone, which allows two workgroups per CU; they are latency-bound, so their
// registers are capped for three waves per SIMD (<= 168; no spills), the
// occupancy their LDS allows.
template <bool RESTRICT, bool PROLONG, bool XZERO, bool BETA, int NR>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RESTRICT || PROLONG ? 3 : 1)))
k_rbc(TbArgs a) {
    constexpr int S = 2;                         // half-sweeps
    constexpr int H = S + (RESTRICT ? 1 : 0);    // halo: one cell per half-sweep, +1 for the residual
    constexpr int HXC = H + (H & 1);             // x halo in cells (even)
    constexpr int HY = H;                        // y and z halo
    constexpr int LX = kRcTX + 2 * HXC, LY = kRcTY + 2 * HY;
    constexpr int HX = LX / 2, HXP = HX;         // pairs per row (no padding: a wave's reads stay in one bank set)
    constexpr int CP = (LY + 2) * HXP;           // one colour of one plane: rows -1 .. LY
    constexpr int PS = 2 * CP;                   // one plane, both colours
    constexpr int NSLOT = HX * LY;
    constexpr int NP = (NSLOT + 255) / 256;      // pair slots per thread
    constexpr int CLX = PROLONG ? LX / 2 + 3 : 1, CLY = PROLONG ? LY / 2 + 3 : 1;
    constexpr int NC = (CLX * CLY + 255) / 256;
    constexpr int RW = kRcTX / 2;                // restriction: coarse cells per tile row
    // the next step's store reuses a ring slot this step reads, or the
    // residual reads what the last half-sweep wrote: barrier after it
    constexpr bool kBarAfter = RESTRICT || NR < S + 3;
    static_assert(NR % 2 == 0 && NR >= S + (RESTRICT ? 3 : 2), "ring too short");
    static_assert(256 * (NP - 1) <= NSLOT, "only the last slot may be partial");
    __shared__ float xs[NR * PS];
    __shared__ float rs[RESTRICT ? kRcTY * RW : 1];
    __shared__ float cw[PROLONG ? 3 : 1][CLY][CLX];
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const uint32_t tile = xcd_block(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z),
                                    gridDim.x * gridDim.y * gridDim.z);
    const int bx = (int)(tile % gridDim.x), by = (int)((tile / gridDim.x) % gridDim.y);
    const int bz = (int)(tile / (gridDim.x * gridDim.y));
    const int gx0 = bx * kRcTX - HXC, gy0 = by * kRcTY - HY;
    const int nzc = (nz + a.zc - 1) / a.zc;
    const int comp = bz / nzc, zi = bz - comp * nzc;
    const int z0 = zi * a.zc, z1 = min(z0 + a.zc, nz);
    const float* xsrc = a.xin + (size_t)comp * a.G;
    float* xdst = a.x + (size_t)comp * a.G;
    const float* bcp = a.b + (size_t)comp * a.G;
    const float* xcoarse = PROLONG ? a.xc + (size_t)comp * a.Gc : nullptr;
    const int cx0 = (gx0 >> 1) - 1, cy0 = (gy0 >> 1) - 1;  // coarse window origin
    const int klo = max(z0 - HY, 0), khi = min(z1 + HY, nz);
    const int kend = khi + S + (RESTRICT ? 1 : 0);
    const size_t plane = (size_t)nx * ny;
    const float omega = a.omega, beta = a.beta, bscale = a.bscale, w6 = a.w6;
    const int tid = threadIdx.x;

    for (int q = tid; q < NR * PS; q += 256) xs[q] = 0.f;

    // Pair slots of this thread: q = tid + 256 u -> row ly, pair m.
    //   e:      index of the pair in a colour plane
    //   ea[v]:  the pair's first cell in its colour plane when the plane
    //           parity is v (that cell's colour is (gy0 + ly + v) & 1)
    //   exn[w]: first x neighbour of the pair's colour-c cell in the other
    //           colour's plane, w = c ^ plane parity
    //   goff:   the pair's offset in a grid plane (0 off the grid)
    int e[NP], ea[NP][2], exn[NP][2], rsi[NP];
    uint32_t gob[NP];  // byte offset of the pair in a grid plane (0 off the grid)
    float wu[NP];
    bool sv[NP], gin[NP], io[NP], swp[NP];
#pragma unroll
    for (int u = 0; u < NP; u++) {
        const int q = tid + 256 * u;
        const bool valid = q < NSLOT;
        const int ly = valid ? q / HX : 0, m = valid ? q - ly * HX : 0;
        const int i0 = gx0 + 2 * m, j = gy0 + ly;
        const bool in = valid && i0 >= 0 && i0 < nx && j >= 0 && j < ny;
        const int sp = j & 1;
        e[u] = (ly + 1) * HXP + m;
        ea[u][0] = e[u] + (sp ? CP : 0);
        ea[u][1] = e[u] + (sp ? 0 : CP);
        exn[u][0] = e[u] + sp - 1;
        exn[u][1] = e[u] - sp;
        gob[u] = in ? 4u * (uint32_t)(j * nx + i0) : 0u;
        wu[u] = in ? (BETA ? omega : w6) : 0.f;
        sv[u] = valid;
        gin[u] = in;
        swp[u] = sp != 0;
        io[u] = in && ly >= HY && ly < HY + kRcTY && m >= HXC / 2 && m < HXC / 2 + kRcTX / 2;
        rsi[u] = (ly - HY) * RW + (m - HXC / 2);
    }

    float2 px[NP], pb[NP], bq[NR][NP];
    float pc[NC];
    float rsum[NP];
#pragma unroll
    for (int u = 0; u < NP; u++) {
        px[u] = pb[u] = make_float2(0.f, 0.f);
        rsum[u] = 0.f;
#pragma unroll
        for (int r = 0; r < NR; r++) bq[r][u] = make_float2(0.f, 0.f);
    }
    // plane k into px, pb (loaded during the step before its store); k >=
    // khi gives the zero plane (the plane index goes through readfirstlane so
    // the compiler keeps one scalar base per plane instead of per-slot 64-bit
    // pointers)
    auto fetch = [&](int k) {
        const size_t ko = (size_t)__builtin_amdgcn_readfirstlane(k) * plane;
        const char* xp_ = reinterpret_cast<const char*>(xsrc + ko);
        const char* bp_ = reinterpret_cast<const char*>(bcp + ko);
        const bool real = k < khi;
#pragma unroll
        for (int u = 0; u < NP; u++) {
            float2 xv = make_float2(0.f, 0.f), bv = make_float2(0.f, 0.f);
            if (real && gin[u]) {
                if (!XZERO) xv = *reinterpret_cast<const float2*>(xp_ + gob[u]);
                bv = *reinterpret_cast<const float2*>(bp_ + gob[u]);
            }
            px[u] = xv;
            pb[u] = bv;
        }
    };
    // Coarse window for the prolongation, ghost-extended: a coarse cell
    // outside the grid holds betac times its nearest in-grid cell per axis
    // it lies out on, so the trilinear weights need no boundary cases (the
    // consistent transfer of k_prolong); plane c in {-1 .. cz} lives in ring
    // slot (c + 3) % 3.
    auto fetch_coarse = [&](int c) {
        const int cc = min(max(c, 0), a.cz - 1);
        const float fz = cc != c ? a.betac : 1.f;
#pragma unroll
        for (int u = 0; u < NC; u++) {
            const int q = tid + 256 * u;
            const int cyl = q / CLX, cxl = q - cyl * CLX;
            const int ci = cx0 + cxl, cj = cy0 + cyl;
            const int cic = min(max(ci, 0), a.cx - 1), cjc = min(max(cj, 0), a.cy - 1);
            float v = 0.f;
            if (q < CLX * CLY)
                v = xcoarse[((size_t)cc * a.cy + cjc) * a.cx + cic] * ((cic != ci ? a.betac : 1.f) *
                                                                         (cjc != cj ? a.betac : 1.f) * fz);
            pc[u] = v;
        }
    };
    auto store_coarse = [&](int c) {
#pragma unroll
        for (int u = 0; u < NC; u++) {
            const int q = tid + 256 * u;
            if (q < CLX * CLY) cw[(c + 3) % 3][q / CLX][q % CLX] = pc[u];
        }
    };
    if (PROLONG) {
        for (int c = (klo >> 1) - 1; c <= (klo >> 1) + 1; c++) {
            fetch_coarse(c);
            store_coarse(c);
        }
    }
    fetch(klo);
    __syncthreads();  // zeroed rings before the first stores

    for (int k0 = klo - klo % NR; k0 < kend; k0 += NR) {
#pragma unroll
        for (int j = 0; j < NR; j++) {
            const int k = k0 + j;  // k % NR == j, k & 1 == j & 1
            if (k < klo || k >= kend) continue;
            if (PROLONG) {
                if (k < khi && k > klo && (j & 1) == 0) store_coarse((k >> 1) + 1);  // fetched during plane k - 1
                __syncthreads();
            }
            // plane k into ring slot j (the zero plane at k == khi)
            if (k <= khi) {
                float* P = xs + j * PS;
#pragma unroll
                for (int u = 0; u < NP; u++) {
                    if (u == NP - 1 && !sv[u]) continue;
                    float2 xv = px[u];
                    if (PROLONG && k < khi && gin[u]) {
                        // trilinear prolongation of the pair: parent column m + 1
                        // of the window, neighbours m (first cell) and m + 2
                        // (second); parent row (ly >> 1) + 1, neighbour one
                        // up (ly odd) or down; parent plane k >> 1, neighbour
                        // one up (k odd) or down
                        const int m = e[u] % HXP, ly = e[u] / HXP - 1;
                        const int rp = (ly >> 1) + 1, rn = rp + ((ly & 1) ? 1 : -1);
                        const int pk = k >> 1, nk = pk + ((j & 1) ? 1 : -1);
                        const float* cp0 = &cw[(pk + 3) % 3][0][0];
                        const float* cn0 = &cw[(nk + 3) % 3][0][0];
                        float ye[2], yo[2];
#pragma unroll
                        for (int z = 0; z < 2; z++) {
                            const float* cz_ = z ? cn0 : cp0;
                            const float* a0 = cz_ + rp * CLX + m;
                            const float* a1 = cz_ + rn * CLX + m;
                            ye[z] = lerp_(0.25f, lerp_(0.25f, a0[1], a0[0]), lerp_(0.25f, a1[1], a1[0]));
                            yo[z] = lerp_(0.25f, lerp_(0.25f, a0[1], a0[2]), lerp_(0.25f, a1[1], a1[2]));
                        }
                        xv.x += lerp_(0.25f, ye[0], ye[1]);
                        xv.y += lerp_(0.25f, yo[0], yo[1]);
                    }
                    P[ea[u][j & 1]] = xv.x;
                    P[ea[u][(j & 1) ^ 1]] = xv.y;
                    // b in colour order: .x colour 0, .y colour 1
                    const bool sw = swp[u] != ((j & 1) != 0);
                    bq[j][u] = sw ? make_float2(pb[u].y, pb[u].x) : pb[u];
                }
            }
            __syncthreads();
            if (k + 1 <= khi) {
                fetch(k + 1);
                if (PROLONG && k + 1 < khi && (j & 1) == 1) fetch_coarse(((k + 1) >> 1) + 1);
            }
#pragma unroll
            for (int t = 1; t <= S; t++) {
                const int p = k - t;
                const int plo = klo > 0 ? klo + t : 0;
                const int phi = khi < nz ? khi - 1 - t : nz - 1;
                if (p >= plo && p <= phi) {
                    const int jp = (j - t + 2 * NR) % NR, jm = (jp + NR - 1) % NR, jq = (jp + 1) % NR;
                    const int c = t & 1;  // odd colour first, as the reference
                    const int w = c ^ (jp & 1);
                    const float* PB = xs + jp * PS + (1 - c) * CP;
                    const float* PM = xs + jm * PS + (1 - c) * CP;
                    const float* PQ = xs + jq * PS + (1 - c) * CP;
                    float* PC = xs + jp * PS + c * CP;
                    // all reads of the half-sweep before its writes: the
                    // slots' cells are distinct and no update reads another
                    // slot's cell of the colour being written
                    float xos[NP], rr[NP];
#pragma unroll
                    for (int u = 0; u < NP; u++) {
                        if (u == NP - 1 && !sv[u]) continue;
                        const int o = e[u], ox = exn[u][w];
                        xos[u] = PC[o];
                        float r = PB[ox] + PB[ox + 1];
                        r += PB[o - HXP] + PB[o + HXP];
                        r += PM[o] + PQ[o];
                        rr[u] = r;
                    }
#pragma unroll
                    for (int u = 0; u < NP; u++) {
                        if (u == NP - 1 && !sv[u]) continue;
                        const int o = e[u];
                        const float xo = xos[u];
                        float wq = wu[u];
                        if (BETA) {
                            const int m = o % HXP, ly = o / HXP - 1;
                            const int i = gx0 + 2 * m + ((swp[u] ? 1 : 0) ^ w), jj = gy0 + ly;
                            const int nout = (i == 0) + (i == nx - 1) + (jj == 0) + (jj == ny - 1) + (p == 0) +
                                             (p == nz - 1);
                            wq = nout == 0 ? (gin[u] ? w6 : 0.f) : wu[u] / fmaf(-beta, (float)nout, 6.f);
                        }
                        PC[o] = relax_late(xo, rr[u], c ? bq[jp][u].y : bq[jp][u].x, bscale, wq, a.om1);
                    }
                }
                if (t < S || kBarAfter) __syncthreads();
            }
            // plane k - S is final: write this thread's interior pairs
            {
                const int pw = k - S;
                if (pw >= z0 && pw < z1) {
                    const int jw = (j + 2 * NR - S) % NR;
                    const float* P = xs + jw * PS;
                    char* dst = reinterpret_cast<char*>(xdst + (size_t)__builtin_amdgcn_readfirstlane(pw) * plane);
#pragma unroll
                    for (int u = 0; u < NP; u++)
                        if (io[u])
                            *reinterpret_cast<float2*>(dst + gob[u]) =
                                make_float2(P[ea[u][jw & 1]], P[ea[u][(jw & 1) ^ 1]]);
                }
            }
            if (RESTRICT) {
                // residual of plane pr = k - 3 (its neighbours are final) at this
                // thread's interior pairs, summed over the pair and the plane
                // pair, then over the two rows of a coarse cell through rs
                const int pr = k - S - 1;
                if (pr >= z0 && pr < z1) {
                    const int jr = (j + 2 * NR - S - 1) % NR, jm = (jr + NR - 1) % NR, jq = (jr + 1) % NR;
#pragma unroll
                    for (int u = 0; u < NP; u++) {
                        if (!io[u]) continue;
                        float part = 0.f;
#pragma unroll
                        for (int c = 0; c < 2; c++) {
                            const int w = c ^ (jr & 1);
                            const float* PB = xs + jr * PS + (1 - c) * CP;
                            const float* PM = xs + jm * PS + (1 - c) * CP;
                            const float* PQ = xs + jq * PS + (1 - c) * CP;
                            const float* PC = xs + jr * PS + c * CP;
                            const int o = e[u], ox = exn[u][w];
                            const float xo = PC[o];
                            float sres = PB[ox] + PB[ox + 1];
                            sres += PB[o - HXP] + PB[o + HXP];
                            sres += PM[o] + PQ[o];
                            int nout = 0;
                            if (BETA) {
                                const int m = o % HXP, ly = o / HXP - 1;
                                const int i = gx0 + 2 * m + ((swp[u] ? 1 : 0) ^ w), jj = gy0 + ly;
                                nout = (i == 0) + (i == nx - 1) + (jj == 0) + (jj == ny - 1) + (pr == 0) +
                                       (pr == nz - 1);
                            }
                            const float r = residual_of(xo, sres, c ? bq[jr][u].y : bq[jr][u].x, bscale, nout,
                                                        BETA ? beta : 0.f);
                            part = c == 0 ? r : part + r;
                        }
                        if ((jr & 1) == 0) rsum[u] = part;
                        else rs[rsi[u]] = rsum[u] + part;
                    }
                    if (jr & 1) {
                        __syncthreads();
                        const int I = tid % RW, J = tid / RW;
                        const int gI = bx * RW + I, gJ = by * (kRcTY / 2) + J, gK = pr / 2;
                        if (gI < a.cx && gJ < a.cy && gK < a.cz)
                            a.bn[(size_t)comp * a.Gc + ((size_t)gK * a.cy + gJ) * a.cx + gI] =
                                (rs[(2 * J) * RW + I] + rs[(2 * J + 1) * RW + I]) * 0.5f;
                    }
                }
            }
        }
    }
}

// Two red-black iterations (four half-sweeps) in one pass over the grid.  A
// workgroup streams z planes of a 64 x 64 cell region; a thread owns the cell
// pair m of two rows (2 rg, 2 rg + 1) and keeps its cells and right-hand side
// of the planes in flight in registers, so that neighbours in z, in the own
// pair and in the other row are registers, the neighbouring pair is a lane
// shift, and only the rows above and below come through LDS: one cell of one
// colour a row and half-sweep.  In step k plane k arrives (state 0) and
// half-sweep t updates plane k - t, t ascending.  What half-sweep t reads of
// other threads (plane k - t after t - 1) was written in step k - 1, and
// what it reads of its own thread's planes k - t + 1 (after t - 1, this step)
// and k - t - 1 (before t + 1) is in program order: one barrier a plane, where
// k_rbc needs one or two a half-sweep.  The region's outer cells become wrong
// by one cell a half-sweep (and one for the residual): a halo of 4 cells, 6
// (5, even) for the residual from a start that is not zero; a zero start is
// exact beyond the region, which saves one.  Planes outside the grid are
// zero and stay so, as cells outside it in x and y.  Needs nx even.
//
// One workgroup of 16 waves a CU, bound
// by its planes' loads and by vector issue at once.  256^3 x 3, V(2,2) (us):
// down from zero 107 + 179 (two k_rbc passes) -> 128, up 203 + 151 -> 205;
// 96^3 x 3: 39 -> 18, 41 -> 22.
constexpr int kR4Region = 64;

// 1024 threads take a region of 64 x 64 floats; of doubles 512 threads one of
// 64 x 32, whose planes in flight need the registers of two waves per SIMD.
template <typename T>
constexpr int r4_threads() { return sizeof(T) == 4 ? 1024 : 512; }

// value of the lane that DPP control C selects (0x130: lane + 1, 0x138: lane - 1)
template <int C>
__device__ inline float lane_shift(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), C, 0xf, 0xf, false));
}
template <int C>
__device__ inline double lane_shift(double v) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), C, 0xf, 0xf, false),
                            __builtin_amdgcn_update_dpp(0, __double2loint(v), C, 0xf, 0xf, false));
}

// A cell pair through a buffer: one 8- or 16-byte access.
template <typename T>
struct R4Pair;
template <>
struct R4Pair<float> {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    u32x2 v = {0u, 0u};
    R4Pair() = default;
    __device__ R4Pair(float a, float b) : v{__float_as_uint(a), __float_as_uint(b)} {}
    template <typename R>
    __device__ void load(R r, uint32_t off) { v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0); }
    template <typename R>
    __device__ void store(R r, uint32_t off) const { __builtin_amdgcn_raw_buffer_store_b64(v, r, off, 0, 0); }
    __device__ float first() const { return __uint_as_float(v[0]); }
    __device__ float second() const { return __uint_as_float(v[1]); }
};
template <>
struct R4Pair<double> {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 v = {0u, 0u, 0u, 0u};
    R4Pair() = default;
    __device__ R4Pair(double a, double b)
        : v{(uint32_t)__double2loint(a), (uint32_t)__double2hiint(a), (uint32_t)__double2loint(b),
            (uint32_t)__double2hiint(b)} {}
    template <typename R>
    __device__ void load(R r, uint32_t off) { v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0); }
    template <typename R>
    __device__ void store(R r, uint32_t off) const { __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, 0); }
    __device__ double first() const { return __hiloint2double((int)v[1], (int)v[0]); }
    __device__ double second() const { return __hiloint2double((int)v[3], (int)v[2]); }
};

template <typename T, bool RESTRICT, bool PROLONG, bool XZERO, bool BETA>
__global__ void __launch_bounds__(r4_threads<T>()) k_rb4(TbArgsT<T> a) {
    constexpr int NT = r4_threads<T>(), RG = NT / 32;  // row groups of the region
    constexpr bool kWide = RESTRICT && !XZERO;
    constexpr int HXY = kWide ? 6 : 4, HZ = kWide ? 5 : 4;
    constexpr int TW = kR4Region - 2 * HXY, TH = 2 * RG - 2 * HXY;  // tile
    constexpr int NR = RESTRICT ? 8 : 6;     // planes in flight
    constexpr int ES = (RG + 2) * 32;        // row groups -1 .. RG of one row parity
    // exchanged rows: state t of plane k - t, stored in step j, goes to slot
    // xslot(t, j); states 0 .. 3 are read one step later (two buffers), the
    // residual also reads state 4 one step and state 3 two steps later (four)
    constexpr int NE = RESTRICT ? 12 : 8;
    auto xslot = [](int t, int j) {
        return t < 3 ? 2 * t + (j & 1) : t == 3 ? 6 + (j & (RESTRICT ? 3 : 1)) : 10 + (j & 1);
    };
    constexpr int CW = 34, CN = CW * (RG + 2);  // coarse window of the prolongation
    __shared__ T ex[NE][2][ES];
    __shared__ T cw[PROLONG ? 3 : 1][PROLONG ? CN : 1];
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const uint32_t tile = xcd_block(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z),
                                    gridDim.x * gridDim.y * gridDim.z);
    const int bx = (int)(tile % gridDim.x), by = (int)((tile / gridDim.x) % gridDim.y);
    const int bz = (int)(tile / (gridDim.x * gridDim.y));
    const int gx0 = bx * TW - HXY, gy0 = by * TH - HXY;
    const int nzc = (nz + a.zc - 1) / a.zc;
    const int comp = bz / nzc, zi = bz - comp * nzc;
    const int z0 = zi * a.zc, z1 = min(z0 + a.zc, nz);
    const T* xsrc = XZERO ? nullptr : a.xin + (size_t)comp * a.G;
    T* xdst = a.x + (size_t)comp * a.G;
    const T* bcp = a.b + (size_t)comp * a.G;
    const T* xcoarse = PROLONG ? a.xc + (size_t)comp * a.Gc : nullptr;
    T* bnext = RESTRICT ? a.bn + (size_t)comp * a.Gc : nullptr;
    const int klo = max(z0 - HZ, 0), khi = min(z1 + HZ, nz);
    const int kend = z1 + 4 + (RESTRICT ? 1 : 0);
    const int kbeg = klo & ~1;  // ring slots and plane parities by the step count
    const size_t plane = (size_t)nx * ny;
    const T omega = a.omega, beta = a.beta, bscale = a.bscale;
    const int tid = threadIdx.x, m = tid & 31, rg = tid >> 5;
    const int i0 = gx0 + 2 * m;
    const bool xin = i0 >= 0 && i0 < nx;
    for (int q = tid; q < NE * 2 * ES; q += NT) (&ex[0][0][0])[q] = (T)0;

    // Planes are read and written as buffers of plane bytes (0 bytes: none),
    // so that loads off the grid give zero and stores outside the tile are
    // dropped without a branch: a step is straight-line code, and its loads
    // are waited for a whole step later.
    constexpr uint32_t kOff = 0x80000000u;  // beyond any plane
    const uint32_t pbytes = (uint32_t)(plane * sizeof(T));
    uint32_t lofs[2], sofs[2];
    bool gin[2];
    // cells outside the grid next to a cell in the plane, and its relaxation
    // factor off and on the first and last plane (0: a cell outside the grid,
    // which is 0 and stays so)
    int nxy[2][2];
    T wr[2], d0[2][2], d1[2][2];  // BETA: d0, d1
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int j = gy0 + 2 * rg + r, ly = 2 * rg + r;
        gin[r] = xin && j >= 0 && j < ny;
        wr[r] = gin[r] ? a.w6 : (T)0;
        lofs[r] = gin[r] ? (uint32_t)sizeof(T) * (uint32_t)(j * nx + i0) : kOff;
        sofs[r] = ly >= HXY && ly < HXY + TH && 2 * m >= HXY && 2 * m < HXY + TW ? lofs[r] : kOff;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int i = i0 + e;
            const int no = (i == 0) + (i == nx - 1) + (j == 0) + (j == ny - 1), noz = no + (nz == 1 ? 2 : 1);
            nxy[r][e] = no;
            d0[r][e] = gin[r] ? relax_weight(no, omega, beta, a.w6) : (T)0;
            d1[r][e] = gin[r] ? relax_weight(noz, omega, beta, a.w6) : (T)0;
        }
    }
    const int gI = i0 >> 1, gJ = (gy0 >> 1) + rg;
    const uint32_t cofs = RESTRICT && sofs[0] != kOff && gI < a.cx && gJ < a.cy ? (uint32_t)sizeof(T) * (uint32_t)(gJ * a.cx + gI) : kOff;
    auto buffer = [](const void* p, uint32_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00027000);
    };

    // [slot][row][pair cell]
    T X[NR][2][2], B[NR][2][2];
    R4Pair<T> px[2], pb[2];
    T pc[2], pf = (T)0, rsum[2] = {(T)0, (T)0};
#pragma unroll
    for (int q = 0; q < NR; q++)
#pragma unroll
        for (int r = 0; r < 2; r++) X[q][r][0] = X[q][r][1] = B[q][r][0] = B[q][r][1] = (T)0;
    auto fetch = [&](int k) {
        k = __builtin_amdgcn_readfirstlane(k);
        const bool real = k >= klo && k < khi;
        const size_t ko = real ? (size_t)k * plane : 0;
        const auto rb = buffer(bcp + ko, real ? pbytes : 0u);
#pragma unroll
        for (int r = 0; r < 2; r++) {
            px[r] = R4Pair<T>{};
            if (!XZERO) {
                const auto rx = buffer(xsrc + ko, real ? pbytes : 0u);
                px[r].load(rx, lofs[r]);
            }
            pb[r].load(rb, lofs[r]);
        }
    };
    // the coarse window, ghost-extended as k_rbc's; plane c in slot (c + 3) % 3.
    // A thread's two cells (the last of them beyond the window: not stored)
    const int cx0 = (gx0 >> 1) - 1, cy0 = (gy0 >> 1) - 1;
    uint32_t cq[2];  // byte offsets
    T cf[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int q = min(tid + NT * u, CN - 1);
        const int ci = cx0 + q % CW, cj = cy0 + q / CW;
        const int cic = PROLONG ? min(max(ci, 0), a.cx - 1) : 0, cjc = PROLONG ? min(max(cj, 0), a.cy - 1) : 0;
        cq[u] = (uint32_t)sizeof(T) * (uint32_t)(cjc * a.cx + cic);
        cf[u] = (cic != ci ? a.betac : (T)1) * (cjc != cj ? a.betac : (T)1);
    }
    auto fetch_coarse = [&](int c) {
        const int cc = min(max(c, 0), a.cz - 1);
        pf = cc != c ? a.betac : (T)1;
        const char* p = reinterpret_cast<const char*>(xcoarse + (size_t)__builtin_amdgcn_readfirstlane(cc) * a.cy * a.cx);
        pc[0] = *reinterpret_cast<const T*>(p + cq[0]);
        pc[1] = *reinterpret_cast<const T*>(p + cq[1]);
    };
    auto store_coarse = [&](int c) {
        T* w = cw[(c + 3) % 3];
        w[tid] = pc[0] * (cf[0] * pf);
        if (tid + NT < CN) w[tid + NT] = pc[1] * (cf[1] * pf);
    };
    if (PROLONG) {
        // (klo is even: the first step stores plane klo / 2 + 1)
        for (int c = (klo >> 1) - 1; c <= (klo >> 1); c++) {
            fetch_coarse(c);
            store_coarse(c);
        }
        fetch_coarse((klo >> 1) + 1);
    }
    fetch(kbeg);
    __syncthreads();

    // the neighbouring pair's cell: lane - 1's (m > 0) or lane + 1's; the
    // region's edge lanes read a row that is not theirs, inside the halo
    auto from_left = [](T v) { return lane_shift<0x138>(v); };
    auto from_right = [](T v) { return lane_shift<0x130>(v); };
    const int lo = rg * 32 + m;  // row group rg - 1 in an exchanged row; rg + 1 at lo + 64

    for (int k0 = kbeg;; k0 += NR) {
#pragma unroll
        for (int j = 0; j < NR; j++) {
            const int k = k0 + j;  // k & 1 == j & 1
            if (k >= kend) return;
            // ---- the exchanged rows of this step (with the coarse window's
            // cells in registers too, spills: the prolongation goes first)
            T y[4][2];
            auto exchanged = [&]() {
#pragma unroll
                for (int t = XZERO ? 2 : 1; t <= 4; t++) {
                    y[t - 1][0] = ex[xslot(t - 1, j + 3)][1][lo];
                    y[t - 1][1] = ex[xslot(t - 1, j + 3)][0][lo + 64];
                }
            };
            // of the residual: [row][colour]; colour 1 was last written by
            // half-sweep 3, colour 0 by 4
            T yr[2][2];
            if (RESTRICT) {
                yr[0][0] = ex[xslot(3, j + 2)][1][lo];
                yr[1][0] = ex[xslot(3, j + 2)][0][lo + 64];
                yr[0][1] = ex[xslot(4, j + 3)][1][lo];
                yr[1][1] = ex[xslot(4, j + 3)][0][lo + 64];
            }
            if (!PROLONG) exchanged();
            // ---- state 0 of plane k (zero from khi on)
            {
                T v[2][2] = {{px[0].first(), px[0].second()}, {px[1].first(), px[1].second()}};
                if (PROLONG) {
                    // trilinear: parent column m + 1 of the window, neighbour m
                    // (first cell) or m + 2; parent row rg + 1, neighbour rg
                    // (first row) or rg + 2; parent plane k >> 1, neighbour one
                    // up (k odd) or down
                    const int pk = k >> 1, nk = pk + ((j & 1) ? 1 : -1);
                    T w[2][2][2];
                    // opaque: the slots repeat with the unrolled steps, and their
                    // addresses would all be kept in registers (spills)
                    int c00 = rg * CW + m;
                    __asm__ volatile("" : "+v"(c00));
#pragma unroll
                    for (int z = 0; z < 2; z++) {
                        const T* c0 = &cw[((z ? nk : pk) + 3) % 3][c00];
                        T xe[3], xo[3];
#pragma unroll
                        for (int q = 0; q < 3; q++) {
                            const T* c = c0 + q * CW;
                            xe[q] = lerp_((T)0.25, c[1], c[0]);
                            xo[q] = lerp_((T)0.25, c[1], c[2]);
                        }
#pragma unroll
                        for (int r = 0; r < 2; r++) {
                            w[z][r][0] = lerp_((T)0.25, xe[1], xe[2 * r]);
                            w[z][r][1] = lerp_((T)0.25, xo[1], xo[2 * r]);
                        }
                    }
                    const bool real = k < khi;
#pragma unroll
                    for (int r = 0; r < 2; r++)
#pragma unroll
                        for (int e = 0; e < 2; e++) {
                            const T f = v[r][e] + lerp_((T)0.25, w[0][r][e], w[1][r][e]);
                            v[r][e] = gin[r] && real ? f : v[r][e];
                        }
                }
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    X[j][r][0] = v[r][0];
                    X[j][r][1] = v[r][1];
                    B[j][r][0] = pb[r].first();
                    B[j][r][1] = pb[r].second();
                    // half-sweep 1 updates colour 1 and reads colour 0
                    if (!XZERO) ex[xslot(0, j)][r][lo + 32] = X[j][r][(r ^ j) & 1];
                }
            }
            if (PROLONG) {
                if ((j & 1) == 0) store_coarse((k >> 1) + 1);  // fetched in step k - 1
                else fetch_coarse(((k + 1) >> 1) + 1);
            }
            fetch(k + 1);
            if (PROLONG) {
                __builtin_amdgcn_sched_barrier(0);
                exchanged();
            }
            // ---- half-sweep t on plane k - t
#pragma unroll
            for (int t = 1; t <= 4; t++) {
                const int jp = (j - t + NR) % NR, jm = (jp + NR - 1) % NR, jq = (jp + 1) % NR;
                const int p = k - t, c = t & 1;  // odd colour first, as the reference
                const bool in = p >= 0 && p < nz, zb = p == 0 || p == nz - 1;
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const int e = (c ^ r ^ jp) & 1;
                    T s = (T)0;
                    if (!(XZERO && t == 1)) {
                        const T other = X[jp][r][1 - e];
                        s = e ? other + from_right(X[jp][r][0]) : from_left(X[jp][r][1]) + other;
                        s += r ? X[jp][0][e] + y[t - 1][1] : y[t - 1][0] + X[jp][1][e];
                        s += X[jm][r][e] + X[jq][r][e];
                    }
                    const T xo = X[jp][r][e];
                    const T w = BETA ? (zb ? d1[r][e] : d0[r][e]) : wr[r];
                    const T xn = relax_late(xo, s, B[jp][r][e], bscale, in ? w : (T)0, a.om1);
                    X[jp][r][e] = xn;
                    if (t < 4 || RESTRICT) ex[xslot(t, j)][r][lo + 32] = xn;
                }
            }
            // ---- plane k - 4 is final
            {
                const int jw = (j + NR - 4) % NR, pw = __builtin_amdgcn_readfirstlane(k - 4);
                const bool mine = pw >= z0 && pw < z1;
                const auto rd = buffer(xdst + (mine ? (size_t)pw * plane : 0), mine ? pbytes : 0u);
#pragma unroll
                for (int r = 0; r < 2; r++) R4Pair<T>(X[jw][r][0], X[jw][r][1]).store(rd, sofs[r]);
            }
            // ---- residual of plane k - 5 and its restriction: this thread's
            // 2 x 2 cells of a plane pair are one coarse cell
            if (RESTRICT) {
                const int jr = (j + NR - 5) % NR, jm = (jr + NR - 1) % NR, jq = (jr + 1) % NR, pr = k - 5;
                const int zb = (pr == 0) + (pr == nz - 1);
                T part[2];
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    part[r] = (T)0;
#pragma unroll
                    for (int c = 0; c < 2; c++) {
                        const int e = (c ^ r ^ jr) & 1;
                        const T xo = X[jr][r][e], other = X[jr][r][1 - e];
                        T s = e ? other + from_right(X[jr][r][0]) : from_left(X[jr][r][1]) + other;
                        s += r ? X[jr][0][e] + yr[1][c] : yr[0][c] + X[jr][1][e];
                        s += X[jm][r][e] + X[jq][r][e];
                        const T v = residual_of(xo, s, B[jr][r][e], bscale, nxy[r][e] + zb, BETA ? beta : (T)0);
                        part[r] = c == 0 ? v : part[r] + v;
                    }
                }
                if ((jr & 1) == 0) {
                    rsum[0] = part[0];
                    rsum[1] = part[1];
                } else {
                    const int gK = __builtin_amdgcn_readfirstlane(pr >> 1);
                    const bool mine = pr >= z0 && pr < z1 && gK < a.cz;
                    const auto rn = buffer(bnext + (mine ? (size_t)gK * a.cy * a.cx : 0),
                                           mine ? (uint32_t)sizeof(T) * (uint32_t)(a.cy * a.cx) : 0u);
                    const T c = restrict_sum(rsum[0], rsum[1], part[0], part[1]);
                    static_assert(!RESTRICT || sizeof(T) == 4, "the restriction stores floats");
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint((float)c), rn, cofs, 0, 0);
                }
            }
            __syncthreads();
        }
    }
}

template <typename T>
__device__ inline T residual_at(const T* __restrict__ x, const T* __restrict__ b, T bscale, int i, int j, int k,
                                int nx, int ny, int nz, T beta) {
    const size_t t = ((size_t)k * ny + j) * nx + i;
    int nout;
    const T s = nb_sum(x, t, i, j, k, nx, ny, nz, nout);
    return residual_of(x[t], s, b[t], bscale, nout, beta);
}

// r = b - A x at the 8 children of coarse cell (ci, cj, ck), summed and
// halved (the sum of MultiGrid_kernel.cu:897-904).
template <typename T>
__device__ inline T restrict_point(const T* xc, const T* bc, T bscale, int ci, int cj, int ck, int nx, int ny, int nz,
                                   T beta) {
    const int i = 2 * ci, j = 2 * cj, k = 2 * ck;
    // children beyond a fine dimension of 1 do not exist
    const bool hi = i + 1 < nx, hj = j + 1 < ny, hk = k + 1 < nz;
    auto pair = [&](int jj, int kk) {
        const T r = residual_at(xc, bc, bscale, i, jj, kk, nx, ny, nz, beta);
        return hi ? r + residual_at(xc, bc, bscale, i + 1, jj, kk, nx, ny, nz, beta) : r;
    };
    const T p00 = pair(j, k), p10 = hj ? pair(j + 1, k) : (T)0;
    const T p01 = hk ? pair(j, k + 1) : (T)0, p11 = hj && hk ? pair(j + 1, k + 1) : (T)0;
    return restrict_sum(p00, p10, p01, p11);
}

// b_c = restrict_point at every coarse cell.
template <typename T>
__global__ void __launch_bounds__(256) k_residual_restrict(const T* __restrict__ x, const T* __restrict__ b, T bscale,
                                                           T* __restrict__ bn, int nx, int ny, int nz, int cx,
                                                           int cy, int cz, size_t G, size_t Gc, T beta) {
    const int ci = blockIdx.x * 64 + threadIdx.x;
    const int cj = blockIdx.y * 4 + threadIdx.y;
    const int comp = blockIdx.z / cz, ck = blockIdx.z - comp * cz;
    if (ci >= cx || cj >= cy) return;
    bn[(size_t)comp * Gc + ((size_t)ck * cy + cj) * cx + ci] =
        restrict_point(x + (size_t)comp * G, b + (size_t)comp * G, bscale, ci, cj, ck, nx, ny, nz, beta);
}

// Coarse correction at fine cell (i, j, k) from the coarse component c.
template <typename T>
__device__ inline T prolong_point(const T* c, int i, int j, int k, int nx, int ny, int nz, int cx, int cy, int cz,
                                  int mode, T betac) {
    int pi = min(i / 2, cx - 1), pj = min(j / 2, cy - 1), pk = min(k / 2, cz - 1);
    T v;
    if (mode == PROLONG_CONSTANT) {
        v = c[((size_t)pk * cy + pj) * cx + pi];
    } else {
        // 1-D weights 3/4 (parent) and 1/4 (neighbour on the fine cell's side);
        // a neighbour outside the coarse grid is betac * parent value
        int ni = (i & 1) ? pi + 1 : pi - 1, nj = (j & 1) ? pj + 1 : pj - 1, nk = (k & 1) ? pk + 1 : pk - 1;
        T wi = nx == 1 ? (T)0 : (T)0.25, wj = ny == 1 ? (T)0 : (T)0.25, wk = nz == 1 ? (T)0 : (T)0.25;
        T fi = (T)1, fj = (T)1, fk = (T)1;
        if (ni < 0 || ni > cx - 1) { ni = pi; fi = betac; }
        if (nj < 0 || nj > cy - 1) { nj = pj; fj = betac; }
        if (nk < 0 || nk > cz - 1) { nk = pk; fk = betac; }
        // the parent's or the neighbour's value on each axis
        auto C = [&](bool x, bool y, bool z) {
            return ghost(x ? fi : (T)1, y ? fj : (T)1, z ? fk : (T)1,
                         c[((size_t)(z ? nk : pk) * cy + (y ? nj : pj)) * cx + (x ? ni : pi)]);
        };
        const T p0 = lerp_(wi, C(0, 0, 0), C(1, 0, 0)), p1 = lerp_(wi, C(0, 1, 0), C(1, 1, 0));
        const T p2 = lerp_(wi, C(0, 0, 1), C(1, 0, 1)), p3 = lerp_(wi, C(0, 1, 1), C(1, 1, 1));
        v = lerp_(wk, lerp_(wj, p0, p1), lerp_(wj, p2, p3));
    }
    return v;
}

template <typename T>
__global__ void __launch_bounds__(256) k_prolong(T* __restrict__ x, const T* __restrict__ xc, int nx, int ny, int nz,
                                                 int cx, int cy, int cz, size_t G, size_t Gc, int mode, T betac) {
    const int i = blockIdx.x * 64 + threadIdx.x;
    const int j = blockIdx.y * 4 + threadIdx.y;
    const int comp = blockIdx.z / nz, k = blockIdx.z - comp * nz;
    if (i >= nx || j >= ny) return;
    x[(size_t)comp * G + ((size_t)k * ny + j) * nx + i] +=
        prolong_point(xc + (size_t)comp * Gc, i, j, k, nx, ny, nz, cx, cy, cz, mode, betac);
}

// ---- small levels: up to two red-black iterations of a 3-D tile in LDS -------
// One launch does what used to take a launch per half-sweep (and one each for
// the zero fill, the residual with its restriction and the prolongation): on
// levels of up to a million cells such launches are latency (4 to 5 us each
// for a level of 32^3, whatever it holds).  A workgroup loads its TI^3 tile
// with an H-cell halo (H = one cell per half-sweep, one more for the residual;
// clipped at the grid), applies the half-sweeps in LDS with the halo
// recomputed, and writes its tile: out of place, as the halos are other
// workgroups' tiles.  A cell at distance d from a side of the loaded region
// that is not a grid boundary is right for the first d half-sweeps.
//
// LDS holds the two colours apart: colour c of plane z, row y has at index m
// the colour-c cell of the pair (2m, 2m + 1), x counted from the region's even
// lower corner, with one zero row, plane and index around it for the ghosts
// (and for what a region side that is no boundary reads: those cells are in
// the discarded halo).  A thread owns the pairs (m, y) of a run of planes, in
// registers with their right-hand sides.  Of the six neighbours of a cell,
// all of the other colour, the pair's other cell and the same cell of the
// planes above and below are the thread's own; the other x neighbour and the
// two in y come from LDS (three reads and a write an update, at immediate
// offsets from three registers).  Vector issue and LDS are about even.
//
// us of one V(2,2) cycle's level, three components, before -> here: 32^3 50
// (11 launches) -> 16.5 (2), 64^3 51 (k_rbc) -> 34; FP64, one component: V(4,4)
// at 64^3 and below 19 launches of 4.2 -> 4 of 11.  Where the FP32 blocked
// passes (k_rb4) are the faster: MGHier::blocked_level.  1024 threads take a
// 16^3 tile, 576 an 8^3 one.
template <typename T>
struct TileArgs {
    const T* xin;  // level before the pass (null: zero)
    T* x;          // level after the pass (another buffer)
    const T* b;
    T bscale;
    int nx, ny, nz;
    size_t G;
    T omega, beta, w6;  // w6 = omega / 6
    int iters;  // 1 or 2
    int tx, ty, tz;
    // residual restricted into bn (null: none), coarse dims n / 2
    T* bn;
    int cx, cy, cz;
    size_t Gc;
    // x += prolongation of xc on load (null: none)
    const T* xc;
    T betac;
    int mode;
};

constexpr int tile_threads(int TI) { return TI == 16 ? 1024 : 576; }

template <typename T, int TI, bool BETA>
__global__ void __launch_bounds__(tile_threads(TI)) k_tile(TileArgs<T> a) {
    constexpr int NT = tile_threads(TI);
    constexpr int HP = TI / 2 + 6;                // pairs per row: TI + 5 above, TI - 6 below, even
    constexpr int RY = TI + 10;                   // rows and planes
    constexpr int PX = HP + 1, PY = RY + 2, PZ = PY * PX;
    constexpr int PC = (RY + 2) * PZ + 1;         // a colour, with the ghosts
    constexpr int NGMIN = NT / (HP * RY);         // column groups when the region is largest
    constexpr int KQ = (RY + NGMIN - 1) / NGMIN;  // planes per thread
    constexpr int CW = TI / 2 + 6;                // coarse window per axis
    constexpr int RW = TI / 2;
    constexpr int AUX = CW * CW * CW > TI * TI * RW ? CW * CW * CW : TI * TI * RW;
    __shared__ T xs[2 * PC];
    __shared__ T aux[AUX];  // coarse window while loading, pair residuals at the end
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int bx = blockIdx.x % a.tx, by = (blockIdx.x / a.tx) % a.ty, bz = blockIdx.x / (a.tx * a.ty);
    const int comp = blockIdx.y;
    const int H = 2 * a.iters + (a.bn ? 1 : 0);
    const int t0x = bx * TI, t0y = by * TI, t0z = bz * TI;
    const int x0 = max(t0x - H, 0) & ~1, x1 = min(t0x + TI + H, nx);
    const int y0 = max(t0y - H, 0), y1 = min(t0y + TI + H, ny);
    const int z0 = max(t0z - H, 0), z1 = min(t0z + TI + H, nz);
    const int hp = (x1 - x0 + 1) >> 1, ry = y1 - y0, rz = z1 - z0;
    const T* xin = a.xin ? a.xin + (size_t)comp * a.G : nullptr;
    const T* b = a.b + (size_t)comp * a.G;
    const int tid = threadIdx.x;
    // thread -> column (m, yy), planes zb .. zb + nq - 1 of the region
    const int ncol = hp * ry, NG = NT / ncol;    // NG >= NGMIN
    const int kq = (rz + NG - 1) / NG;           // <= KQ
    const int col = tid % ncol, grp = tid / ncol;
    const int m = col % hp, yy = col / hp;
    const int zb = grp * kq;
    const int nq = grp < NG ? min(kq, rz - zb) : 0;  // <= 0: no planes
    const int gi = x0 + 2 * m, gj = y0 + yy, gk0 = z0 + zb;
    const bool two = gi + 1 < x1;  // the pair's second cell exists
    // colour of the first cell of plane zb + q: p ^ (q & 1)
    const int p = (gj + gk0) & 1;

    // right-hand sides and starting values by colour, all loads in flight
    // together (a pair that does not exist reads the component's first cells)
    T bc[2][KQ], xr[2][KQ];
    const int o1 = two ? 1 : 0;
#pragma unroll
    for (int q = 0; q < KQ; q++) {
        const bool ok = q < nq;
        const size_t t = ok ? ((size_t)(gk0 + q) * ny + gj) * nx + gi : 0;
        bc[0][q] = b[t];
        bc[1][q] = b[t + (ok ? o1 : 0)];
    }
    if (xin) {
#pragma unroll
        for (int q = 0; q < KQ; q++) {
            const bool ok = q < nq;
            const size_t t = ok ? ((size_t)(gk0 + q) * ny + gj) * nx + gi : 0;
            xr[0][q] = xin[t];
            xr[1][q] = xin[t + (ok ? o1 : 0)];
        }
    } else {
#pragma unroll
        for (int q = 0; q < KQ; q++) xr[0][q] = xr[1][q] = (T)0;
    }
    for (int q = tid; q < 2 * PC; q += NT) xs[q] = (T)0;
    const int c0x = (x0 >> 1) - 1, c0y = (y0 >> 1) - 1, c0z = (z0 >> 1) - 1;
    if (a.xc) {
        // window c0 .. of the coarse level; a cell outside holds its nearest
        // in-grid cell, betac times per axis for the trilinear transfer
        const T* xc = a.xc + (size_t)comp * a.Gc;
        const T gb = a.mode == PROLONG_TRILINEAR ? a.betac : (T)1;
        constexpr int NC = (CW * CW * CW + NT - 1) / NT;
        T cv[NC];
#pragma unroll
        for (int u = 0; u < NC; u++) {
            const int q = min(tid + NT * u, CW * CW * CW - 1);
            const int cx_ = c0x + q % CW, cy_ = c0y + (q / CW) % CW, cz_ = c0z + q / (CW * CW);
            const int ix = min(max(cx_, 0), a.cx - 1), iy = min(max(cy_, 0), a.cy - 1), iz = min(max(cz_, 0), a.cz - 1);
            cv[u] = ghost(ix != cx_ ? gb : (T)1, iy != cy_ ? gb : (T)1, iz != cz_ ? gb : (T)1,
                          xc[((size_t)iz * a.cy + iy) * a.cx + ix]);
        }
#pragma unroll
        for (int u = 0; u < NC; u++) aux[min(tid + NT * u, CW * CW * CW - 1)] = cv[u];
    }
    __syncthreads();
    // index of the pair in a plane of one colour; a thread without planes
    // stays at the first ghost row, which it neither reads nor writes
    T* const X = xs + (nq > 0 ? (zb + 1) * PZ + (yy + 1) * PX + m + 1 : PZ + 1);
#pragma unroll
    for (int q = 0; q < KQ; q++) {
        if (q >= nq) continue;
        if (a.xc) {
            const int px = (gi >> 1) - c0x, py = (gj >> 1) - c0y, gk = gk0 + q, pz = (gk >> 1) - c0z;
            if (a.mode == PROLONG_CONSTANT) {
                const T v = aux[(pz * CW + py) * CW + px];
                xr[0][q] += v;
                xr[1][q] += v;
            } else {
                // 3/4 the parent, 1/4 its neighbour on the cell's side
                const int qy = py + ((gj & 1) ? 1 : -1), qz = pz + ((gk & 1) ? 1 : -1);
                const T w4 = (T)0.25;
                T ye[2], yo[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const T* r0 = aux + ((h ? qz : pz) * CW + py) * CW + px;
                    const T* r1 = aux + ((h ? qz : pz) * CW + qy) * CW + px;
                    ye[h] = lerp_(w4, lerp_(w4, r0[0], r0[-1]), lerp_(w4, r1[0], r1[-1]));
                    yo[h] = lerp_(w4, lerp_(w4, r0[0], r0[1]), lerp_(w4, r1[0], r1[1]));
                }
                xr[0][q] += lerp_(w4, ye[0], ye[1]);
                xr[1][q] += lerp_(w4, yo[0], yo[1]);
            }
        }
        // first, second cell -> colour 0, 1; a second cell that does not
        // exist stays 0 (its relaxation factor is 0)
        const T u0 = xr[0][q], u1 = two ? xr[1][q] : (T)0, d0 = bc[0][q], d1 = bc[1][q];
        const bool sw = (p ^ (q & 1)) != 0;
        xr[0][q] = sw ? u1 : u0;
        xr[1][q] = sw ? u0 : u1;
        bc[0][q] = sw ? d1 : d0;
        bc[1][q] = sw ? d0 : d1;
        X[q * PZ] = xr[0][q];
        X[PC + q * PZ] = xr[1][q];
    }
    __syncthreads();
    // The colour-c cell of plane q is the pair's cell e = p ^ c ^ (q & 1): its
    // x neighbour outside the pair is the other colour's at index e ? + 1 : - 1.
    // Xn[v]: that index for e = p ^ v.
    const T* const Xn[2] = {X + (p ? 1 : -1), X + (p ? -1 : 1)};
    // relax_weight of cell e = p ^ v, wz in the first and last grid plane (0
    // for a second cell that does not exist)
    const int nout_y = (gj == 0) + (gj == ny - 1);
    T w[2], wz[2];
#pragma unroll
    for (int v = 0; v < 2; v++) {
        const int e = p ^ v, i = gi + e;
        const int no = nout_y + (i == 0) + (i == nx - 1);
        const bool cell = e == 0 || two;
        w[v] = cell ? relax_weight(no, a.omega, BETA ? a.beta : (T)0, a.w6) : (T)0;
        wz[v] = BETA && cell ? relax_weight(no + 1, a.omega, a.beta, a.w6) : w[v];
    }
    const int qlo = -gk0, qhi = nz - 1 - gk0;  // plane indices of the z boundaries
    const T om1 = (T)1 - a.omega;
    for (int h = 0; h < 2 * a.iters; h += 2) {
#pragma unroll
        for (int c = 1; c >= 0; c--) {  // odd colour first
            const T* const O = X + (1 - c) * PC;
            // the run's end neighbours in z
            T zlo = (T)0, zhi = (T)0;
            if (nq > 0) {
                zlo = O[-PZ];
                zhi = O[nq * PZ];
            }
#pragma unroll
            for (int q = 0; q < KQ; q++) {
                if (q >= nq) continue;
                const int v = c ^ (q & 1);
                const T zm = q == 0 ? zlo : xr[1 - c][q > 0 ? q - 1 : 0];
                const T zp = q == nq - 1 ? zhi : (q + 1 < KQ ? xr[1 - c][q + 1 < KQ ? q + 1 : q] : zhi);
                T r = xr[1 - c][q] + Xn[v][(1 - c) * PC + q * PZ];
                r += O[q * PZ + PX] + O[q * PZ - PX];
                r += zm + zp;
                const T wq = BETA && (q == qlo || q == qhi) ? wz[v] : w[v];
                xr[c][q] = relax(xr[c][q], r, bc[c][q], a.bscale, wq, om1);
                X[c * PC + q * PZ] = xr[c][q];
            }
            __syncthreads();
        }
    }
    T* x = a.x + (size_t)comp * a.G;
    const bool own = nq > 0 && gi >= t0x && gi < t0x + TI && gj >= t0y && gj < t0y + TI;
    const bool res = a.bn && two && (gi >> 1) < a.cx;
#pragma unroll
    for (int q = 0; q < KQ; q++) {
        const int gk = gk0 + q;
        if (!own || q >= nq || gk < t0z || gk >= t0z + TI) continue;
        const bool sw = (p ^ (q & 1)) != 0;
        const size_t t = ((size_t)gk * ny + gj) * nx + gi;
        x[t] = sw ? xr[1][q] : xr[0][q];
        if (two) x[t + 1] = sw ? xr[0][q] : xr[1][q];
        if (!res) continue;
        // residual of the pair, summed
        T part = (T)0;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const T* const O = X + (1 - c) * PC;
            const int v = c ^ (q & 1);
            T r = xr[1 - c][q] + Xn[v][(1 - c) * PC + q * PZ];
            r += O[q * PZ + PX] + O[q * PZ - PX];
            r += O[q * PZ - PZ] + O[q * PZ + PZ];
            const int i = gi + (p ^ v);
            const int no = nout_y + (i == 0) + (i == nx - 1) + (gk == 0) + (gk == nz - 1);
            r = residual_of(xr[c][q], r, bc[c][q], a.bscale, no, BETA ? a.beta : (T)0);
            part = c == 0 ? r : part + r;
        }
        aux[((gk - t0z) * TI + (gj - t0y)) * RW + ((gi - t0x) >> 1)] = part;
    }
    if (a.bn) {
        __syncthreads();
        T* bn = a.bn + (size_t)comp * a.Gc;
        for (int q = tid; q < RW * RW * RW; q += NT) {
            const int I = q % RW, J = (q / RW) % RW, K = q / (RW * RW);
            const int ci = (t0x >> 1) + I, cj = (t0y >> 1) + J, ck = (t0z >> 1) + K;
            if (ci >= a.cx || cj >= a.cy || ck >= a.cz) continue;
            const T* r = aux + ((2 * K) * TI + 2 * J) * RW + I;
            bn[((size_t)ck * a.cy + cj) * a.cx + ci] =
                restrict_sum(r[0], r[RW], r[TI * RW], r[TI * RW + RW]);
        }
    }
}

// Exact solve of the <= 512-cell coarsest level in the separable eigenbasis,
// FP64: v holds bscale b on entry (t < n = nx ny nz; every thread of the
// workgroup calls it, as it synchronises), thread t < n gets x at cell t.
// N > 0: nx = ny = nz = N, the loops unrolled; N = 0: any dimensions.
template <int N>
__device__ inline double coarse_solve_n(double* v, double* w, const double* tab, int nx_, int ny_, int nz_, int t) {
    const int nx = N ? N : nx_, ny = N ? N : ny_, nz = N ? N : nz_;
    const int n = nx * ny * nz;
    const double* Ex = tab;
    const double* Ey = Ex + nx * nx;
    const double* Ez = Ey + ny * ny;
    const double* lx = Ez + nz * nz;
    const double* ly = lx + nx;
    const double* lz = ly + ny;
    const int i = t % nx, j = (t / nx) % ny, k = t / (nx * ny);
    auto dot = [](int n_, auto term) {
        double s = 0;
        if (N) {
#pragma unroll
            for (int q = 0; q < N; q++) s += term(q);
        } else {
            for (int q = 0; q < n_; q++) s += term(q);
        }
        return s;
    };
    __syncthreads();
    // forward: v <- E v along x, y, z
    if (t < n) w[t] = dot(nx, [&](int q) { return Ex[i * nx + q] * v[(k * ny + j) * nx + q]; });
    __syncthreads();
    if (t < n) v[t] = dot(ny, [&](int q) { return Ey[j * ny + q] * w[(k * ny + q) * nx + i]; });
    __syncthreads();
    if (t < n)
        w[t] = dot(nz, [&](int q) { return Ez[k * nz + q] * v[(q * ny + j) * nx + i]; }) / (lx[i] + ly[j] + lz[k]);
    __syncthreads();
    // backward: v <- E^T v along x, y, z
    if (t < n) v[t] = dot(nx, [&](int q) { return Ex[q * nx + i] * w[(k * ny + j) * nx + q]; });
    __syncthreads();
    if (t < n) w[t] = dot(ny, [&](int q) { return Ey[q * ny + j] * v[(k * ny + q) * nx + i]; });
    __syncthreads();
    double s = 0;
    if (t < n) s = dot(nz, [&](int q) { return Ez[q * nz + k] * w[(q * ny + j) * nx + i]; });
    return s;
}

// The eigenbasis tables of levels whose edges add up to little (8^3: 216
// numbers) are first copied to LDS: the six products of a solve read them one
// after another, at L2's latency (k_vtail 18 -> 15 us with the level in LDS by colours).
constexpr int kCoarseTab = 1024;
__device__ inline int coarse_tab_size(int nx, int ny, int nz) { return nx * nx + ny * ny + nz * nz + nx + ny + nz; }
// ltab: kCoarseTab doubles of LDS, filled here (before coarse_solve, which
// synchronises)
__device__ inline void coarse_stage(double* ltab, const double* __restrict__ tab, int nx, int ny, int nz) {
    const int n = coarse_tab_size(nx, ny, nz);
    if (n <= kCoarseTab)
        for (int q = threadIdx.x; q < n; q += blockDim.x) ltab[q] = tab[q];
}
__device__ inline double coarse_solve(double* v, double* w, const double* ltab, const double* __restrict__ tab, int nx,
                                      int ny, int nz, int t) {
    if (nx == 8 && ny == 8 && nz == 8) return coarse_solve_n<8>(v, w, ltab, nx, ny, nz, t);
    if (coarse_tab_size(nx, ny, nz) <= kCoarseTab) return coarse_solve_n<0>(v, w, ltab, nx, ny, nz, t);
    return coarse_solve_n<0>(v, w, tab, nx, ny, nz, t);
}

// Exact solve of the coarsest level, one workgroup per component.
template <typename T>
__global__ void __launch_bounds__(512) k_coarse(T* __restrict__ x, const T* __restrict__ b, T bscale, int nx, int ny,
                                                int nz, size_t G, const double* __restrict__ tab) {
    __shared__ double v[512];
    __shared__ double w[512];
    __shared__ double ltab[kCoarseTab];
    const int comp = blockIdx.x;
    const int n = nx * ny * nz;
    const int t = threadIdx.x;
    coarse_stage(ltab, tab, nx, ny, nz);
    if (t < n) v[t] = (double)bscale * (double)b[(size_t)comp * G + t];
    const double s = coarse_solve(v, w, ltab, tab, nx, ny, nz, t);
    if (t < n) x[(size_t)comp * G + t] = (T)s;
}

// The two smallest levels of a V-cycle in one launch: level l0 (at most 4096
// cells, 16^3) and the coarsest below it, one component per workgroup, the
// iterate in LDS, the same operations in the same order as the launches they
// replace: the starting x, nu1 red-black iterations, residual and restriction,
// the exact coarsest solve, prolongation, nu2 iterations, and x of level l0
// written for the level above.  A barrier separates the phases (a half-sweep
// reads only the other colour, so its cells update in any order).  Larger
// levels stay on launches over the whole device: one compute unit per
// component sweeps 32^3 in about 115 us.  LDS issue bounds it (eight accesses
// an update); x by colours with ghosts and the relaxation factors formed once
// took the four half-sweeps from 8.9 to 6.1 thousand cycles, the residuals
// through LDS the restriction from 5.8 to 4.1.
constexpr int kTailMax = 4096;
constexpr int kTailThreads = 1024;
// cell pairs (2 i2, 2 i2 + 1) per thread on level l0
constexpr int kTailPairs = 4;
template <typename T>
struct TailArgs {
    const T* xin;         // level l0 iterate before (null: zero)
    T* x0;                // level l0 iterate out [ncomp][G0]
    const T* b0;          // level l0 right-hand side [ncomp][G0]
    T* b1;                // coarsest right-hand side [ncomp][G1] (written)
    T bscale;             // times b0
    int d0[3], d1[3];     // dims of level l0 and of the coarsest
    size_t G0, G1;
    T beta0, beta1;       // ghost factors of the two levels
    int mode;             // prolongation
    int nu1, nu2;
    T omega, w6;          // w6 = omega / 6
    const double* tab;    // coarsest eigenbasis
};

// Level l0 in LDS by colours, as a tile of k_tile with the whole level as its
// region: pair (m, y) of plane z at index ((z + 1) (ny + 2) + y + 1) (hx + 1) +
// m + 1 of each colour, hx = ceil(nx / 2), zeros around.
// Values of a colour that LDS holds: in FP32 those of whatever shape stands two
// levels above nothing but the coarsest ((1, 1024, 4): 2 x 1026 x 6), in FP64 of
// the usual ones.
template <typename T>
constexpr int tail_lds() { return sizeof(T) == 4 ? 12320 : 4096; }
inline int tail_pairs(const int* d) { return ((d[0] + 1) / 2 + 1) * (d[1] + 2) * (d[2] + 2) + 1; }
// the fit test of level l0 (host side): thread t owns column (m, y) = t mod P
// (P = hx ny columns) at kq = ceil(nz / (threads / P)) planes
template <typename T>
inline bool tail_fits(const int* d) {
    const int P = ((d[0] + 1) / 2) * d[1];
    if (P > kTailThreads || tail_pairs(d) > tail_lds<T>()) return false;
    const int R = kTailThreads / P;
    return (d[2] + R - 1) / R <= kTailPairs;
}

template <typename T>
__global__ void __launch_bounds__(kTailThreads) k_vtail(TailArgs<T> a) {
    __shared__ T xa[2][tail_lds<T>()];
    __shared__ T rs[kTailMax];  // residuals of level l0, in grid order
    __shared__ T xc[512];
    __shared__ double cv[512], cw[512], ltab[kCoarseTab];
    const int comp = blockIdx.x, tid = threadIdx.x;
    const int nx = a.d0[0], ny = a.d0[1], nz = a.d0[2];
    const int cx = a.d1[0], cy = a.d1[1], cz = a.d1[2];
    const int n1 = cx * cy * cz;
    const T* b0 = a.b0 + (size_t)comp * a.G0;
    const T* xi = a.xin ? a.xin + (size_t)comp * a.G0 : nullptr;
    T* b1 = a.b1 + (size_t)comp * a.G1;
    // thread -> pair column (m, j), planes k0 .. k0 + nq - 1
    const int hx = (nx + 1) >> 1, P = hx * ny, R = kTailThreads / P;
    const int kq = (nz + R - 1) / R;
    const int col = tid % P, grp = tid / P;
    const int m = col % hx, j = col / hx, i = 2 * m, k0 = grp * kq;
    const int nq = grp < R ? min(kq, nz - k0) : 0;  // <= 0: no planes
    const bool two = i + 1 < nx;
    const int p = (j + k0) & 1;  // colour of the first cell in plane k0
    const int PX = hx + 1, PZ = PX * (ny + 2);
    // the thread's right-hand sides and starting x into registers, by cell
    // (first, second); planes past nq read the first cells
    T be[kTailPairs], bo[kTailPairs], xe[kTailPairs], xo[kTailPairs];
#pragma unroll
    for (int q = 0; q < kTailPairs; q++) {
        const size_t t = q < nq ? ((size_t)(k0 + q) * ny + j) * nx + i : 0;
        const size_t t1 = t + (q < nq && two ? 1 : 0);
        be[q] = b0[t];
        bo[q] = b0[t1];
        xe[q] = xi ? xi[t] : (T)0;
        xo[q] = xi ? xi[t1] : (T)0;
    }
    coarse_stage(ltab, a.tab, cx, cy, cz);
    const int nl = PZ * (nz + 2) + 1;
    for (int q = tid; q < nl; q += kTailThreads) xa[0][q] = xa[1][q] = (T)0;
    __syncthreads();
    const int o0 = nq > 0 ? (k0 + 1) * PZ + (j + 1) * PX + m + 1 : 0;
#pragma unroll
    for (int q = 0; q < kTailPairs; q++)
        if (q < nq) {
            const int s = p ^ (q & 1), o = o0 + q * PZ;
            xa[s][o] = xe[q];
            if (two) xa[1 - s][o] = xo[q];
        }
    __syncthreads();
    // sum of the neighbours of cell e of the pair at o (colour c), added as
    // nb_sum does
    auto nbr = [&](int c, int o, int e) {
        const T* O = xa[1 - c];
        T r = O[o - 1 + e] + O[o + e];
        r += O[o + PX] + O[o - PX];
        r += O[o - PZ] + O[o + PZ];
        return r;
    };
    const int nout_y = (j == 0) + (j == ny - 1);
    auto outside = [&](int e, int k) {
        return (i + e == 0) + (i + e == nx - 1) + nout_y + (k == 0) + (k == nz - 1);
    };
    T we[kTailPairs], wo[kTailPairs];
#pragma unroll
    for (int q = 0; q < kTailPairs; q++) {
        we[q] = relax_weight(outside(0, k0 + q), a.omega, a.beta0, a.w6);
        wo[q] = relax_weight(outside(1, k0 + q), a.omega, a.beta0, a.w6);
    }
    const T om1 = (T)1 - a.omega;
    auto smooth = [&](int iters) {
        for (int h = 0; h < iters; h++)
#pragma unroll
            for (int c = 1; c >= 0; c--) {  // odd colour first
#pragma unroll
                for (int q = 0; q < kTailPairs; q++) {
                    const int e = p ^ c ^ (q & 1), o = o0 + q * PZ;
                    if (q < nq && (e == 0 || two))
                        xa[c][o] = relax(xa[c][o], nbr(c, o, e), e ? bo[q] : be[q], a.bscale, e ? wo[q] : we[q],
                                         om1);
                }
                __syncthreads();
            }
    };
    smooth(a.nu1);
    // residuals (residual_at), then their sums over the children of each
    // coarse cell in restrict_point's order: the coarsest right-hand side
#pragma unroll
    for (int q = 0; q < kTailPairs; q++)
        if (q < nq) {
            const int o = o0 + q * PZ, t = ((k0 + q) * ny + j) * nx + i;
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int c = p ^ e ^ (q & 1);
                if (e == 1 && !two) continue;
                const T xv = xa[c][o];
                rs[t + e] = residual_of(xv, nbr(c, o, e), e ? bo[q] : be[q], a.bscale, outside(e, k0 + q), a.beta0);
            }
        }
    __syncthreads();
    for (int q = tid; q < n1; q += kTailThreads) {
        const int ci = q % cx, cj = (q / cx) % cy, ck = q / (cx * cy);
        const bool hi = 2 * ci + 1 < nx, hj = 2 * cj + 1 < ny, hk = 2 * ck + 1 < nz;
        const T* f = rs + ((2 * ck) * ny + 2 * cj) * nx + 2 * ci;
        auto pair = [&](int o) { return hi ? f[o] + f[o + 1] : f[o]; };
        const T r = restrict_sum(pair(0), hj ? pair(nx) : (T)0, hk ? pair(nx * ny) : (T)0,
                                 hj && hk ? pair(nx * ny + nx) : (T)0);
        b1[q] = r;
        cv[q] = (double)1.0f * (double)r;
    }
    const double s = coarse_solve(cv, cw, ltab, a.tab, cx, cy, cz, tid);
    if (tid < n1) xc[tid] = (T)s;
    __syncthreads();
    // prolongation of the coarse correction, then nu2 iterations
#pragma unroll
    for (int q = 0; q < kTailPairs; q++)
        if (q < nq) {
#pragma unroll
            for (int e = 0; e < 2; e++)
                if (e == 0 || two)
                    xa[p ^ e ^ (q & 1)][o0 + q * PZ] +=
                        prolong_point((const T*)xc, i + e, j, k0 + q, nx, ny, nz, cx, cy, cz, a.mode, a.beta1);
        }
    __syncthreads();
    smooth(a.nu2);
    T* x = a.x0 + (size_t)comp * a.G0;
#pragma unroll
    for (int q = 0; q < kTailPairs; q++)
        if (q < nq) {
            const int sc = p ^ (q & 1), o = o0 + q * PZ, t = ((k0 + q) * ny + j) * nx + i;
            x[t] = xa[sc][o];
            if (two) x[t + 1] = xa[1 - sc][o];
        }
}

template <typename T>
__global__ void k_fill_zero(T* __restrict__ p, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = (T)0;
}

__device__ inline double block_sum_256(double v, double* lds) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) lds[wave] = v;
    __syncthreads();
    double s = 0;
    if (threadIdx.x == 0)
        for (int w2 = 0; w2 < (int)(blockDim.x >> 6); w2++) s += lds[w2];
    __syncthreads();
    return s;
}

// Residual and right-hand-side norms, block partials in a fixed order.
constexpr int kResRows = 4;  // x rows a thread of k_resnorm has in flight

template <typename T>
__global__ void __launch_bounds__(256) k_resnorm(const T* __restrict__ x, const T* __restrict__ b, T bscale, int nx,
                                                 int ny, int nz, size_t G, int rw, double* __restrict__ part) {
    __shared__ double lds[4];
    const int comp = blockIdx.y;
    const T* xc = x + (size_t)comp * G;
    const T* bc = b + (size_t)comp * G;
    double rr = 0, bb = 0;
    // block b takes a contiguous run of x rows, RU rows per step and group of
    // 2^rw threads so that their loads are in flight together (rows past the
    // run read its last row and are not summed); lanes run along x.  Short
    // rows share a block: with one row a step and 2048 blocks 32^3 x 3 took
    // 11.6 us (now 4.6), all of it launching blocks of a row each, and their
    // reduction 4.3 (3.3).
    constexpr int RU = kResRows;
    const int rows = ny * nz, per = (rows + gridDim.x - 1) / gridDim.x;
    const int r0 = blockIdx.x * per, r1 = min(r0 + per, rows);
    const int rg = threadIdx.x >> rw, nrg = blockDim.x >> rw;
    for (int row = r0 + rg * RU; row < r1; row += nrg * RU) {
        for (int i = threadIdx.x & ((1 << rw) - 1); i < nx; i += 1 << rw) {
            T r[RU], bv[RU];
#pragma unroll
            for (int u = 0; u < RU; u++) {
                const int rw_ = min(row + u, r1 - 1);
                const int j = rw_ % ny, k = rw_ / ny;
                r[u] = residual_at(xc, bc, bscale, i, j, k, nx, ny, nz, (T)0);
                bv[u] = bc[(size_t)rw_ * nx + i];
            }
#pragma unroll
            for (int u = 0; u < RU; u++) {
                if (row + u < r1) {
                    const double bd = (double)bscale * (double)bv[u];
                    rr += (double)r[u] * (double)r[u];
                    bb += bd * bd;
                }
            }
        }
    }
    double s1 = block_sum_256(rr, lds);
    double s2 = block_sum_256(bb, lds);
    if (threadIdx.x == 0) {
        part[((size_t)comp * gridDim.x + blockIdx.x) * 2] = s1;
        part[((size_t)comp * gridDim.x + blockIdx.x) * 2 + 1] = s2;
    }
}

// out[2c], out[2c+1] = sums of the partials of component c (fixed order).
__global__ void __launch_bounds__(256) k_reduce_partials(const double* __restrict__ part, int nblk,
                                                         double* __restrict__ out) {
    __shared__ double lds[4];
    const int comp = blockIdx.x;
    double a = 0, b2 = 0;
    for (int q = threadIdx.x; q < nblk; q += blockDim.x) {
        a += part[((size_t)comp * nblk + q) * 2];
        b2 += part[((size_t)comp * nblk + q) * 2 + 1];
    }
    double s1 = block_sum_256(a, lds);
    double s2 = block_sum_256(b2, lds);
    if (threadIdx.x == 0) {
        out[2 * comp] = s1;
        out[2 * comp + 1] = s2;
    }
}

// FP64 defect-correction step (see mg.hpp).  A workgroup owns a 64 x 4 tile
// of x columns and a run of z planes; each thread marches its column in z
// with x at k-1, k, k+1 in registers (x = x_in + e, formed once per cell) and
// takes the in-plane neighbours from an LDS plane with a one-cell halo (the
// first 140 threads also form the halo cells).  Norm partial sums are per
// workgroup, reduced afterwards in a fixed order.
constexpr int kDcTX = 64, kDcTY = 4;

__global__ void __launch_bounds__(256) k_dc_step(const double* __restrict__ xin, const float* __restrict__ e,
                                                 const double* __restrict__ b64, double* __restrict__ xout,
                                                 float* __restrict__ r32, int nx, int ny, int nz, size_t G, int zc,
                                                 double* __restrict__ part) {
    __shared__ double pl[kDcTY + 2][kDcTX + 2];
    __shared__ double lds[4];
    const int tilesx = (nx + kDcTX - 1) / kDcTX, tilesy = (ny + kDcTY - 1) / kDcTY;
    const int nzc = (nz + zc - 1) / zc;
    const int blk = blockIdx.x;  // ((comp * nzc + zchunk) * tilesy + ty) * tilesx + tx
    const int tx = blk % tilesx, ty = (blk / tilesx) % tilesy, zq = (blk / (tilesx * tilesy)) % nzc;
    const int comp = blk / (tilesx * tilesy * nzc);
    const int lx = threadIdx.x % kDcTX, ly = threadIdx.x / kDcTX;
    const int i = tx * kDcTX + lx, j = ty * kDcTY + ly;
    const int z0 = zq * zc, z1 = min(z0 + zc, nz);
    const size_t cb = (size_t)comp * G;
    const bool own = i < nx && j < ny;
    auto X = [&](int ii, int jj, int kk) -> double {
        if (ii < 0 || ii >= nx || jj < 0 || jj >= ny || kk < 0 || kk >= nz) return 0.0;
        const size_t q = cb + ((size_t)kk * ny + jj) * nx + ii;
        return (xin ? xin[q] : 0.0) + (e ? (double)e[q] : 0.0);
    };
    // halo cell of this thread (threads 0..139): the ring around the tile
    int hx = -2, hy = -2;
    {
        const int h = threadIdx.x;
        if (h < kDcTX + 2) { hx = h - 1; hy = -1; }
        else if (h < 2 * (kDcTX + 2)) { hx = h - (kDcTX + 2) - 1; hy = kDcTY; }
        else if (h < 2 * (kDcTX + 2) + kDcTY) { hx = -1; hy = h - 2 * (kDcTX + 2); }
        else if (h < 2 * (kDcTX + 2) + 2 * kDcTY) { hx = kDcTX; hy = h - 2 * (kDcTX + 2) - kDcTY; }
    }
    const bool halo = hx > -2;
    const int hi = tx * kDcTX + hx, hj = ty * kDcTY + hy;
    double xm = own ? X(i, j, z0 - 1) : 0.0, xc = own ? X(i, j, z0) : 0.0;
    double rr = 0, bb = 0;
    for (int k = z0; k < z1; k++) {
        const double xp = own ? X(i, j, k + 1) : 0.0;
        pl[ly + 1][lx + 1] = xc;
        if (halo) pl[hy + 1][hx + 1] = X(hi, hj, k);
        __syncthreads();
        if (own) {
            double s = pl[ly + 1][lx] + pl[ly + 1][lx + 2];
            s += pl[ly][lx + 1] + pl[ly + 2][lx + 1];
            s += xm + xp;
            s -= 6.0 * xc;
            const size_t q = cb + ((size_t)k * ny + j) * nx + i;
            const double bval = b64[q];
            const double r = bval - s;
            xout[q] = xc;
            r32[q] = (float)r;
            rr += r * r;
            bb += bval * bval;
        }
        __syncthreads();
        xm = xc;
        xc = xp;
    }
    const double s1 = block_sum_256(rr, lds);
    const double s2 = block_sum_256(bb, lds);
    if (threadIdx.x == 0) {
        const int per = tilesx * tilesy * nzc, b = blk - comp * per;
        part[((size_t)comp * per + b) * 2] = s1;
        part[((size_t)comp * per + b) * 2 + 1] = s2;
    }
}

pppm_status launch_dc_step(const double* x_in, const float* e, const double* b64, double* x_out, float* r32, int nx,
                           int ny, int nz, int ncomp, double* partials, double* out, hipStream_t st) {
    const size_t G = (size_t)nx * ny * nz;
    const int tiles = ((nx + kDcTX - 1) / kDcTX) * ((ny + kDcTY - 1) / kDcTY);
    // as many z chunks as fit the partial-sum slots of one component
    const int nzc = std::max(1, std::min(nz, MGHier<float>::kNormBlocks / tiles));
    if (tiles > MGHier<float>::kNormBlocks) return PPPM_ERR_INVALID;
    const int zc = (nz + nzc - 1) / nzc;
    const int nzc_eff = (nz + zc - 1) / zc;
    const int per = tiles * nzc_eff;
    hipLaunchKernelGGL(k_dc_step, dim3(per * ncomp), dim3(256), 0, st, x_in, e, b64, x_out, r32, nx, ny, nz, G, zc,
                       partials);
    PPPM_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_reduce_partials, dim3(ncomp), dim3(256), 0, st, partials, per, out);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

// ---------------------------------------------------------------------------
// host side
static void dst_basis(int n, double* E, double* lam) {
    const double pi = 3.14159265358979323846;
    for (int k = 0; k < n; k++) {
        double s = std::sin(pi * (k + 1) / (2.0 * (n + 1)));
        lam[k] = -4.0 * s * s;
        for (int i = 0; i < n; i++) E[k * n + i] = std::sqrt(2.0 / (n + 1)) * std::sin(pi * (double)(k + 1) * (i + 1) / (n + 1));
    }
}

// cyclic Jacobi eigen-decomposition of a symmetric matrix (rows of E = vectors)
static void eig_sym(int n, std::vector<double>& A, double* E, double* lam) {
    for (int i = 0; i < n; i++)
        for (int j = 0; j < n; j++) E[i * n + j] = i == j ? 1.0 : 0.0;
    for (int sweep = 0; sweep < 100; sweep++) {
        double off = 0;
        for (int p = 0; p < n; p++)
            for (int q = p + 1; q < n; q++) off += A[p * n + q] * A[p * n + q];
        if (off < 1e-300) break;
        for (int p = 0; p < n; p++)
            for (int q = p + 1; q < n; q++) {
                double apq = A[p * n + q];
                if (apq == 0.0) continue;
                double theta = (A[q * n + q] - A[p * n + p]) / (2.0 * apq);
                double t = (theta >= 0 ? 1.0 : -1.0) / (std::fabs(theta) + std::sqrt(theta * theta + 1.0));
                double c = 1.0 / std::sqrt(t * t + 1.0), s = t * c;
                for (int i = 0; i < n; i++) {
                    double aip = A[i * n + p], aiq = A[i * n + q];
                    A[i * n + p] = c * aip - s * aiq;
                    A[i * n + q] = s * aip + c * aiq;
                }
                for (int i = 0; i < n; i++) {
                    double api = A[p * n + i], aqi = A[q * n + i];
                    A[p * n + i] = c * api - s * aqi;
                    A[q * n + i] = s * api + c * aqi;
                }
                for (int i = 0; i < n; i++) {
                    double ep = E[p * n + i], eq = E[q * n + i];
                    E[p * n + i] = c * ep - s * eq;
                    E[q * n + i] = s * ep + c * eq;
                }
            }
    }
    for (int i = 0; i < n; i++) lam[i] = A[i * n + i];
}

static void axis_basis(int n, double beta, double* E, double* lam) {
    if (beta == 0.0) {
        dst_basis(n, E, lam);
        return;
    }
    std::vector<double> A((size_t)n * n, 0.0);
    for (int i = 0; i < n; i++) {
        A[i * n + i] = -2.0;
        if (i > 0) A[i * n + i - 1] = 1.0;
        if (i < n - 1) A[i * n + i + 1] = 1.0;
    }
    A[0] += beta;
    A[(size_t)(n - 1) * n + (n - 1)] += beta;
    eig_sym(n, A, E, lam);
}

std::vector<double> coarse_tables(int nx, int ny, int nz, double beta) {
    std::vector<double> t((size_t)nx * nx + ny * ny + nz * nz + nx + ny + nz);
    double* Ex = t.data();
    double* Ey = Ex + nx * nx;
    double* Ez = Ey + ny * ny;
    double* lx = Ez + nz * nz;
    double* ly = lx + nx;
    double* lz = ly + ny;
    axis_basis(nx, beta, Ex, lx);
    axis_basis(ny, beta, Ey, ly);
    axis_basis(nz, beta, Ez, lz);
    return t;
}

// Halvings of MultiGrid.h:115-127 (m_ComputeLevels): the levels' dimensions,
// their number returned.
static int level_dims(int x, int y, int z, int (*d)[3]) {
    int L = 0;
    for (;; L++) {
        d[L][0] = x;
        d[L][1] = y;
        d[L][2] = z;
        if ((long)x * y * z <= 512 || L + 1 >= 16) return L + 1;
        x = x / 2 > 0 ? x / 2 : 1;
        y = y / 2 > 0 ? y / 2 : 1;
        z = z / 2 > 0 ? z / 2 : 1;
    }
}

template <typename T>
bool MGHier<T>::has_temp(const int (*d)[3], int L, int l) {
    if (sizeof(T) == 4) return true;
    const size_t n = (size_t)d[l][0] * d[l][1] * d[l][2];
    const bool tail = l == L - 2 && L >= 3 && n <= (size_t)kTailMax && tail_fits<T>(d[l]);
    const bool tiles = n < kTileCells && d[l][0] > 1 && d[l][1] > 1 && d[l][2] > 1;
    const bool wide = n <= (size_t)1 << 24 && !(d[l][0] & 1);
    return l < L - 1 && !tail && (tiles || wide);
}

template <typename T>
size_t MGHier<T>::bytes_for(int nx, int ny, int nz, int ncomp) {
    int d[16][3];
    const int L = level_dims(nx, ny, nz, d);
    size_t b = 0;
    for (int l = 0; l < L; l++) {
        const size_t n = ((size_t)d[l][0] * d[l][1] * d[l][2] * ncomp + 63) & ~(size_t)63;
        b += ((l > 0 ? 2 : 0) + (has_temp(d, L, l) ? 1 : 0)) * n * sizeof(T);
    }
    const int x = d[L - 1][0], y = d[L - 1][1], z = d[L - 1][2];
    // coarse tables (two bases, <= 3 * 512^2 doubles each at most) and norm partials
    b += 2 * (size_t)(x * x + y * y + z * z + x + y + z) * sizeof(double);
    b += (size_t)kNormBlocks * ncomp * 2 * sizeof(double) + 2 * (size_t)ncomp * sizeof(double);
    return b;
}

static void rbc_prime();
static int cu_count();

template <typename T>
pppm_status MGHier<T>::init(int nx, int ny, int nz, int ncomp) {
    release();
    std::lock_guard<std::mutex> lk(runtime_mutex());
    if (nx < 1 || ny < 1 || nz < 1 || ncomp < 1 || ncomp > kMaxComp) return PPPM_ERR_INVALID;
    ncomp_ = ncomp;
    cap_ = ncomp;
    // MultiGrid.h:93-98
    L_ = level_dims(nx, ny, nz, d_);
    x_.assign(L_, nullptr);
    b_.assign(L_, nullptr);
    t_.assign(L_, nullptr);
    bytes_ = 0;
    {
        if (std::is_same<T, float>::value) rbc_prime();
        else (void)cu_count();
    }
    // out-of-place targets; the FP64 passes run in place without (the same
    // values, more launches), so a card that has no room for them serves the
    // hierarchy all the same
    auto temps = [&]() {
        // one allocation (each takes about 40 us)
        size_t all = 0;
        auto each = [&](auto f) {
            for (int l = 0; l < L_; l++)
                if (has_temp(d_, L_, l)) f(l, (cells(l) * ncomp_ + 63) & ~(size_t)63);
        };
        each([&](int, size_t n) { all += n; });
        if (all == 0) return true;
        if (hipMalloc(&tbase_, all * sizeof(T)) != hipSuccess) {
            (void)hipGetLastError();
            tbase_ = nullptr;
            return false;
        }
        bytes_ += all * sizeof(T);
        T* p = tbase_;
        each([&](int l, size_t n) {
            t_[l] = p;
            p += n;
        });
        return true;
    };
    if (std::is_same<T, float>::value && !temps()) {
        release_locked();
        return PPPM_ERR_NOMEM;
    }
    if (L_ > 1) {
        auto room = [&](int l) { return (cells(l) * ncomp_ + 63) & ~(size_t)63; };
        size_t all = 0;
        for (int l = 1; l < L_; l++) all += 2 * room(l);
        if (hipMalloc(&xbase_, all * sizeof(T)) != hipSuccess) {
            xbase_ = nullptr;
            release_locked();
            return PPPM_ERR_NOMEM;
        }
        bytes_ += all * sizeof(T);
        T* p = xbase_;
        for (int l = 1; l < L_; l++) {
            x_[l] = p;
            b_[l] = p + room(l);
            p += 2 * room(l);
        }
    }
    const int* dc = d_[L_ - 1];
    std::vector<double> tc = coarse_tables(dc[0], dc[1], dc[2], mg_beta(L_ - 1));
    std::vector<double> tr = coarse_tables(dc[0], dc[1], dc[2], 0.0);
    if (hipMalloc(&tab_cons_, tc.size() * sizeof(double)) != hipSuccess ||
        hipMalloc(&tab_ref_, tr.size() * sizeof(double)) != hipSuccess ||
        hipMalloc(&part_, (size_t)kNormBlocks * ncomp_ * 2 * sizeof(double) + 2 * (size_t)ncomp_ * sizeof(double)) !=
            hipSuccess ||
        hipHostMalloc(&hnorm_, (2 * (size_t)ncomp_ + 2) * sizeof(double)) != hipSuccess) {
        release_locked();
        return PPPM_ERR_NOMEM;
    }
    bytes_ += (tc.size() + tr.size()) * sizeof(double) + (size_t)kNormBlocks * ncomp_ * 2 * sizeof(double) +
              2 * (size_t)ncomp_ * sizeof(double);
    PPPM_HIP_TRY(hipMemcpy(tab_cons_, tc.data(), tc.size() * sizeof(double), hipMemcpyHostToDevice));
    PPPM_HIP_TRY(hipMemcpy(tab_ref_, tr.data(), tr.size() * sizeof(double), hipMemcpyHostToDevice));
    if (std::is_same<T, double>::value) (void)temps();
    return PPPM_OK;
}

template <typename T>
void MGHier<T>::release() {
    std::lock_guard<std::mutex> lk(runtime_mutex());
    release_locked();
}

template <typename T>
void MGHier<T>::release_locked() {
    if (xbase_) (void)hipFree(xbase_);
    if (tbase_) (void)hipFree(tbase_);
    xbase_ = tbase_ = nullptr;
    x_.clear();
    b_.clear();
    t_.clear();
    if (tab_cons_) (void)hipFree(tab_cons_);
    if (tab_ref_) (void)hipFree(tab_ref_);
    if (part_) (void)hipFree(part_);
    if (hnorm_) (void)hipHostFree(hnorm_);
    tab_cons_ = tab_ref_ = part_ = hnorm_ = nullptr;
    L_ = 0;
}

template <typename T>
pppm_status MGHier<T>::fill(T* p, size_t n, hipStream_t st) {
    if (n == 0) return PPPM_OK;
    size_t blocks = div_up64(n, 256);
    if (blocks > 16384) blocks = 16384;
    hipLaunchKernelGGL(k_fill_zero<T>, dim3((uint32_t)blocks), dim3(256), 0, st, p, n);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

template <typename T>
__global__ void k_copy(T* __restrict__ d, const T* __restrict__ s, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) d[i] = s[i];
}

template <typename T>
pppm_status MGHier<T>::copy(T* d, const T* s, size_t n, hipStream_t st) {
    if (n == 0) return PPPM_OK;
    size_t blocks = div_up64(n, 256);
    if (blocks > 16384) blocks = 16384;
    hipLaunchKernelGGL(k_copy<T>, dim3((uint32_t)blocks), dim3(256), 0, st, d, s, n);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

// z planes per workgroup of k_rb2: even (restriction pairs), at least 2,
// and small enough that a pass has about 1024 workgroups; the coarse levels
// are latency-bound, so parallelism beats the extra halo planes there.
static int tb_zchunk(int nx, int ny, int nz, int ncomp) {
    const int tiles = (int)(div_up(nx, kTbTX) * div_up(ny, kTbTY)) * ncomp;
    const int want = std::max(1, (1024 + tiles - 1) / tiles);
    int zc = (nz + want - 1) / want;
    zc += zc & 1;
    return std::max(2, std::min(zc, nz + (nz & 1)));
}

// Compute units of the current device (cached per device).
static int cu_count() {
    static int n[16] = {0};
    int d = 0;
    if (hipGetDevice(&d) != hipSuccess || d < 0 || d >= 16) d = 0;
    if (n[d] == 0) {
        int c = 0;
        if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, d) != hipSuccess || c < 1) c = 256;
        n[d] = c;
    }
    return n[d];
}

// Launch one k_rbc instantiation with z chunks sized so the whole grid is
// resident at once (one round of workgroups: no tail), when the tiles leave
// room for at least two chunks; otherwise the caller's chunking.
template <bool R, bool P, bool Z, bool B, int NR>
static int rbc_per_cu() {
    static int per_cu = [] {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(&k_rbc<R, P, Z, B, NR>),
                                                         256, 0) != hipSuccess ||
            n < 1)
            n = 1;
        return n;
    }();
    return per_cu;
}

// The occupancy queries run once, when a hierarchy is set up, not inside a
// stream capture.
static void rbc_prime() {
    (void)cu_count();
    (void)rbc_per_cu<false, false, false, false, 4>();
    (void)rbc_per_cu<false, false, false, true, 4>();
    (void)rbc_per_cu<false, false, true, false, 4>();
    (void)rbc_per_cu<false, false, true, true, 4>();
    (void)rbc_per_cu<false, true, false, false, 4>();
    (void)rbc_per_cu<false, true, false, true, 4>();
    (void)rbc_per_cu<false, false, false, false, 6>();
    (void)rbc_per_cu<false, false, false, true, 6>();
    (void)rbc_per_cu<false, false, true, false, 6>();
    (void)rbc_per_cu<false, false, true, true, 6>();
    (void)rbc_per_cu<false, true, false, false, 6>();
    (void)rbc_per_cu<false, true, false, true, 6>();
    (void)rbc_per_cu<true, false, false, false, 6>();
    (void)rbc_per_cu<true, false, false, true, 6>();
    (void)rbc_per_cu<true, false, true, false, 6>();
    (void)rbc_per_cu<true, false, true, true, 6>();
}

template <bool R, bool P, bool Z, bool B, int NR>
static void launch_rbc(TbArgs a, int ncomp, hipStream_t st) {
    const int per_cu = rbc_per_cu<R, P, Z, B, NR>();
    const int tiles = (int)(div_up(a.nx, kRcTX) * div_up(a.ny, kRcTY)) * ncomp;
    const int chunks = per_cu * cu_count() / tiles;
    if (chunks >= 2) {
        int zc = (a.nz + chunks - 1) / chunks;
        zc += zc & 1;
        a.zc = std::max(2, zc);
    }
    const int nzc = (a.nz + a.zc - 1) / a.zc;
    dim3 grid(div_up(a.nx, kRcTX), div_up(a.ny, kRcTY), nzc * ncomp), blk(256);
    hipLaunchKernelGGL((k_rbc<R, P, Z, B, NR>), grid, blk, 0, st, a);
}

// k_rb4 over all components, one workgroup a CU at a time: the number of z
// chunks that needs the fewest steps, rounds of workgroups times a chunk's
// planes with its halo.
template <typename T, bool R, bool P, bool Z, bool B>
static void launch_rb4(TbArgsT<T> a, int ncomp, hipStream_t st) {
    constexpr int rim = R && !Z ? 12 : 8, tw = kR4Region - rim, th = r4_threads<T>() / 16 - rim, halo = (R && !Z ? 10 : 8) + 4;
    const int tx = (a.nx + tw - 1) / tw, ty = (a.ny + th - 1) / th;
    const int64_t tiles = (int64_t)tx * ty * ncomp, cus = cu_count();
    int64_t best = INT64_MAX;
    for (int c = 1; c <= 64; c++) {
        int zc = (a.nz + c - 1) / c;
        zc += zc & 1;
        const int64_t n = (a.nz + zc - 1) / zc, cost = (tiles * n + cus - 1) / cus * (zc + halo);
        if (cost < best) {
            best = cost;
            a.zc = zc;
        }
    }
    dim3 grid(tx, ty, (a.nz + a.zc - 1) / a.zc * ncomp);
    hipLaunchKernelGGL((k_rb4<T, R, P, Z, B>), grid, dim3(r4_threads<T>()), 0, st, a);
}

// One blocked pass over all components: kind 1 = k_rb2, 2 = k_rbc with a
// four-plane ring, 3 = k_rbc with a six-plane ring (the residual pass always
// uses six); k_rbc needs nx even, k_rb2 takes any size.
// two_iter: two red-black iterations in the pass (k_rb4; nx even, kind 4
// only), else one.
template <bool R, bool P, bool Z>
static pppm_status launch_rb2(const TbArgs& a, int ncomp, int kind, hipStream_t st, bool two_iter = false) {
    static_assert(kTbTX == kRcTX && kTbTY == kRcTY, "both blocked kernels use the same tiles");
    const int nzc = (a.nz + a.zc - 1) / a.zc;
    dim3 grid(div_up(a.nx, kTbTX), div_up(a.ny, kTbTY), nzc * ncomp), blk(256);
    const bool beta = a.beta != 0.f;
    if (two_iter && (kind < 4 || (a.nx & 1) != 0)) return PPPM_ERR_INVALID;
    if (two_iter) {
        // from zero only with the residual, and with it from an iterate only
        // on the finest level, which has no ghost factor
        if constexpr (!R && Z) return PPPM_ERR_INVALID;
        else if constexpr (R && !Z) {
            if (beta) return PPPM_ERR_INVALID;
            launch_rb4<float, R, P, Z, false>(a, ncomp, st);
        } else {
            if (beta) launch_rb4<float, R, P, Z, true>(a, ncomp, st);
            else launch_rb4<float, R, P, Z, false>(a, ncomp, st);
        }
    } else if (kind >= 2 && (a.nx & 1) == 0) {
        if (R || kind == 3) {
            if (beta) launch_rbc<R, P, Z, true, 6>(a, ncomp, st);
            else launch_rbc<R, P, Z, false, 6>(a, ncomp, st);
        } else {
            constexpr int NR4 = R ? 6 : 4;
            if (beta) launch_rbc<R, P, Z, true, NR4>(a, ncomp, st);
            else launch_rbc<R, P, Z, false, NR4>(a, ncomp, st);
        }
    } else if (beta) {
        hipLaunchKernelGGL((k_rb2<R, P, Z, true>), grid, blk, 0, st, a);
    } else {
        hipLaunchKernelGGL((k_rb2<R, P, Z, false>), grid, blk, 0, st, a);
    }
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

// k_rb4 addresses a plane of floats by 31-bit byte offsets (of doubles: levels
// of at most 2^24 cells).
static bool r4_plane(int nx, int ny) { return (size_t)nx * ny * sizeof(float) <= (size_t)1 << 31; }

template <typename T>
static pppm_status smooth_tb(const T*, T*, const T*, T, int, int, int, int, size_t, T, T, int, bool, hipStream_t) {
    return PPPM_ERR_INVALID;
}
// one red-black iteration (two with two_iter), xin -> x
template <>
pppm_status smooth_tb<float>(const float* xin, float* x, const float* b, float bscale, int nx, int ny, int nz,
                             int ncomp, size_t G, float omega, float beta, int kind, bool two_iter, hipStream_t st) {
    TbArgs a{};
    a.xin = xin;
    a.x = x;
    a.b = b;
    a.bscale = bscale;
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    a.G = G;
    a.omega = omega;
    a.beta = beta;
    a.w6 = omega / 6.0f;
    a.om1 = 1.0f - omega;
    a.zc = tb_zchunk(nx, ny, nz, ncomp);
    return launch_rb2<false, false, false>(a, ncomp, kind, st, two_iter);
}

template <typename T>
pppm_status MGHier<T>::smooth_colour(int l, T* x, const T* b, T bscale, int iters, T omega, T beta, hipStream_t st) {
    for (int it = 0; it < iters; it++)
        for (int color = 1; color >= 0; color--) {
            launch_rbgs(x, b, bscale, d_[l][0], d_[l][1], d_[l][2], ncomp_, color, omega, beta, st);
            PPPM_LAUNCH_CHECK();
        }
    return PPPM_OK;
}

template <typename T>
pppm_status MGHier<T>::smooth(int l, T* x, const T* b, T bscale, int iters, T omega, T beta, hipStream_t st) {
    const int nx = d_[l][0], ny = d_[l][1], nz = d_[l][2];
    if (std::is_same<T, float>::value && tb_ && iters > 0) {
        // out-of-place passes of one iteration (two under kind 4 while two
        // remain), x -> t -> x ...; an odd pass count ends in t, copied back
        T* tmp = t_[l];
        const bool pairs = tb_ == 4 && !(nx & 1) && r4_plane(nx, ny);
        int q = 0;
        for (int done = 0; done < iters; q++) {
            const bool two = pairs && iters - done >= 2;
            const T* src = (q & 1) ? tmp : x;
            T* dst = (q & 1) ? x : tmp;
            pppm_status s =
                smooth_tb<T>(src, dst, b, bscale, nx, ny, nz, ncomp_, cells(l), omega, beta, tb_, two, st);
            if (s != PPPM_OK) return s;
            done += two ? 2 : 1;
        }
        if (q & 1) return copy(x, tmp, cells(l) * ncomp_, st);
        return PPPM_OK;
    }
    T* cur = x;
    if constexpr (std::is_same<T, double>::value) {
        // large levels: two iterations a pass while two remain, x -> t -> x
        if (wide_level(l))
            for (; iters >= 2; iters -= 2) {
                T* dst = cur == x ? t_[l] : x;
                TbArgsT<T> a{};
                a.xin = cur;
                a.x = dst;
                a.b = b;
                a.bscale = bscale;
                a.nx = nx;
                a.ny = ny;
                a.nz = nz;
                a.G = cells(l);
                a.omega = omega;
                a.beta = beta;
                a.w6 = omega / (T)6;
                a.om1 = (T)1 - omega;
                if (beta != 0) launch_rb4<T, false, false, false, true>(a, ncomp_, st);
                else launch_rb4<T, false, false, false, false>(a, ncomp_, st);
                PPPM_LAUNCH_CHECK();
                cur = dst;
            }
    }
    pppm_status s = smooth_colour(l, cur, b, bscale, iters, omega, beta, st);
    if (s != PPPM_OK || cur == x) return s;
    return copy(x, cur, cells(l) * ncomp_, st);
}

template <typename T>
pppm_status MGHier<T>::residual_restrict(int l, const T* x, const T* b, T bscale, T beta, T* bnext, hipStream_t st) {
    const int* f = d_[l];
    const int* c = d_[l + 1];
    dim3 blk(64, 4), grid(div_up(c[0], 64), div_up(c[1], 4), c[2] * ncomp_);
    hipLaunchKernelGGL(k_residual_restrict<T>, grid, blk, 0, st, x, b, bscale, bnext, f[0], f[1], f[2], c[0], c[1],
                       c[2], cells(l), cells(l + 1), beta);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

template <typename T>
pppm_status MGHier<T>::prolong(int l, T* x, const T* xc, int mode, T betac, hipStream_t st) {
    const int* f = d_[l];
    const int* c = d_[l + 1];
    dim3 blk(64, 4), grid(div_up(f[0], 64), div_up(f[1], 4), f[2] * ncomp_);
    hipLaunchKernelGGL(k_prolong<T>, grid, blk, 0, st, x, xc, f[0], f[1], f[2], c[0], c[1], c[2], cells(l),
                       cells(l + 1), mode, betac);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

template <typename T>
pppm_status MGHier<T>::coarse(T* x, const T* b, T bscale, bool consistent, hipStream_t st) {
    const int* c = d_[L_ - 1];
    hipLaunchKernelGGL(k_coarse<T>, dim3(ncomp_), dim3(512), 0, st, x, b, bscale, c[0], c[1], c[2], cells(L_ - 1),
                       consistent ? tab_cons_ : tab_ref_);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

template <typename T>
int MGHier<T>::tail_level() const {
    if (!tb_ || !tail_ || L_ < 3) return -1;
    // the level above the coarsest, below the blocked levels
    const int l0 = L_ - 2;
    if (cells(l0) >= tb_min_cells_ || cells(l0) > (size_t)kTailMax || cells(L_ - 1) > 512 || !tail_fits<T>(d_[l0]))
        return -1;
    return l0;
}

template <typename T>
pppm_status MGHier<T>::tail(const T* xin, T* x, const T* b, T* b1, T bscale, int nu1, int nu2, T omega,
                            bool consistent, hipStream_t st) {
    const int l0 = L_ - 2;
    TailArgs<T> a{};
    a.xin = xin;
    a.x0 = x;
    a.b0 = b;
    a.b1 = b1;
    a.bscale = bscale;
    for (int c = 0; c < 3; c++) {
        a.d0[c] = d_[l0][c];
        a.d1[c] = d_[l0 + 1][c];
    }
    a.G0 = cells(l0);
    a.G1 = cells(l0 + 1);
    a.beta0 = consistent ? (T)mg_beta(l0) : (T)0;
    a.beta1 = consistent ? (T)mg_beta(l0 + 1) : (T)0;
    a.mode = consistent ? PROLONG_TRILINEAR : PROLONG_CONSTANT;
    a.nu1 = nu1;
    a.nu2 = nu2;
    a.omega = omega;
    a.w6 = omega / (T)6;
    a.tab = consistent ? tab_cons_ : tab_ref_;
    hipLaunchKernelGGL(k_vtail<T>, dim3(ncomp_), dim3(kTailThreads), 0, st, a);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

template <typename T>
bool MGHier<T>::blocked_level(int l) const {
    const size_t n = cells(l), all = n * (size_t)ncomp_;
    if (n >= tb_min_cells_) return true;
    if (tb_ < 2 || tb_min_cells_ > kBlockedMin) return false;
    if (n >= tb_min_cells_ / 5 * 4 && (all >= kBlockedCells || thin(l))) return true;
    if (thin(l) || d_[l][0] < 20) return false;  // regions of 64 cells along x
    if (all >= kBlockedCells) return true;
    // tiles that the level fills badly: by a quarter more cells than it has,
    // three fifths for those of 16^3
    const int TI = tile_size(l);
    size_t in_tiles = 1;
    for (int c = 0; c < 3; c++) in_tiles *= (size_t)((d_[l][c] + TI - 1) / TI * TI);
    return all >= kBlockedPartial && (TI == 8 ? in_tiles * 4 >= n * 5 : in_tiles * 5 >= n * 8);
}

template <typename T>
bool MGHier<T>::tile_level(int l, bool consistent) const {
    if (!tb_ || l >= L_ - 1 || !t_[l] || cells(l) >= kTileCells) return false;
    if (sizeof(T) == 8 ? wide_level(l) : blocked_level(l) && !(d_[l][0] & 1)) return false;  // k_rb4, k_rbc
    if (sizeof(T) == 8 && (d_[l][0] & 1) && cells(l) * (size_t)ncomp_ >= kOddTileDoubles) return false;
    // thin levels leave most of a tile empty
    if (sizeof(T) == 4 && thin(l) && cells(l) * (size_t)ncomp_ >= kThinCells) return false;
    for (int c = 0; c < 3; c++)
        // without the one launch of the smallest levels the one above the
        // coarsest runs a launch per half-sweep, with bitwise its results
        if (d_[l][c] < 2 || (!tail_ && l == L_ - 2) || (consistent && (d_[l][c] & 1))) return false;  // trilinear parents are i / 2
    return true;
}

template <typename T>
pppm_status MGHier<T>::tile(int l, const T* xin, T* x, const T* b, T bscale, int iters, T omega, T beta, T* bnext,
                            const T* xc, int mode, T betac, hipStream_t st) {
    if (iters < 1 || iters > 2 || (bnext && xc) || xin == x) return PPPM_ERR_INVALID;
    const int* d = d_[l];
    const int* c = d_[l + 1];
    TileArgs<T> a{};
    a.xin = xin;
    a.x = x;
    a.b = b;
    a.bscale = bscale;
    a.nx = d[0];
    a.ny = d[1];
    a.nz = d[2];
    a.G = cells(l);
    a.omega = omega;
    a.beta = beta;
    a.w6 = omega / (T)6;
    a.iters = iters;
    a.bn = bnext;
    a.cx = c[0];
    a.cy = c[1];
    a.cz = c[2];
    a.Gc = cells(l + 1);
    a.xc = xc;
    a.betac = betac;
    a.mode = mode;
    // 16^3 tiles recompute less halo (26^3 cells against 18^3 for an eighth
    // of the tile) where they still fill the chip; doubles of them do not fit
    // LDS with a second workgroup
    const int TI = tile_size(l);
    const bool big = TI == 16;
    a.tx = (d[0] + TI - 1) / TI;
    a.ty = (d[1] + TI - 1) / TI;
    a.tz = (d[2] + TI - 1) / TI;
    dim3 grid(a.tx * a.ty * a.tz, ncomp_);
    if constexpr (std::is_same<T, float>::value) {
        if (big) {
            if (beta != 0.f) hipLaunchKernelGGL((k_tile<float, 16, true>), grid, dim3(tile_threads(16)), 0, st, a);
            else hipLaunchKernelGGL((k_tile<float, 16, false>), grid, dim3(tile_threads(16)), 0, st, a);
            PPPM_LAUNCH_CHECK();
            return PPPM_OK;
        }
    }
    if (beta != (T)0) hipLaunchKernelGGL((k_tile<T, 8, true>), grid, dim3(tile_threads(8)), 0, st, a);
    else hipLaunchKernelGGL((k_tile<T, 8, false>), grid, dim3(tile_threads(8)), 0, st, a);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

// A tile level of a V-cycle on the way down: nu1 iterations, two a launch,
// from src (null: zero; else X[l] itself), the last launch with the residual
// and its restriction; fold (with more than two iterations): coarse iterate
// whose prolongation is added first.  The launches alternate between X and the
// level's temporary so that the nu2 iterations on the way up end in X (a start
// from X itself and an odd number of launches ends in the temporary, copied
// by tile_up).
template <typename T>
static pppm_status tile_down(MGHier<T>& m, int l, T* X, const T* src, const T* b, T bs, int nu1, int nu2, T omega,
                             T beta, T* bnext, const T* fold, int mode, T betac, T** cur, hipStream_t st) {
    const int np1 = (nu1 + 1) / 2, total = np1 + (nu2 + 1) / 2;
    T* dst = (!src && (total & 1)) ? X : m.temp(l);
    for (int q = 0; q < np1; q++) {
        const bool last = q == np1 - 1;
        pppm_status s = m.tile(l, src, dst, b, bs, last ? nu1 - 2 * q : 2, omega, beta, last ? bnext : nullptr,
                               q == 0 ? fold : nullptr, mode, betac, st);
        if (s != PPPM_OK) return s;
        src = dst;
        dst = dst == X ? m.temp(l) : X;
    }
    *cur = const_cast<T*>(src);
    return PPPM_OK;
}
// ... and on the way up: the prolongation of xc, then nu2 iterations, into X.
template <typename T>
static pppm_status tile_up(MGHier<T>& m, int l, T* X, T* cur, const T* b, T bs, int nu2, T omega, T beta, const T* xc,
                           int mode, T betac, hipStream_t st) {
    for (int done = 0; done < nu2; done += 2) {
        T* dst = cur == X ? m.temp(l) : X;
        pppm_status s = m.tile(l, cur, dst, b, bs, std::min(2, nu2 - done), omega, beta, nullptr,
                               done == 0 ? xc : nullptr, mode, betac, st);
        if (s != PPPM_OK) return s;
        cur = dst;
    }
    return cur == X ? PPPM_OK : m.copy(X, cur, m.cells(l) * m.ncomp(), st);
}

// MultiGrid.cpp:128-201 (m_Vcycle) from level l0 on X[l0]; fold: level l0 + 1
// iterate whose (constant) prolongation is added to X[l0] first.
template <typename T>
static pppm_status vcycle_from(MGHier<T>& m, std::vector<T*>& X, std::vector<T*>& B, int l0, T bscale0, int nu1,
                               int nu2, T omega, bool consistent, hipStream_t st, const T* fold = nullptr) {
    const int L = m.levels(), mode = consistent ? PROLONG_TRILINEAR : PROLONG_CONSTANT;
    const bool relax = nu1 > 0 && nu2 > 0;
    const int lt = m.tail_level();
    const bool tail = lt >= l0 && lt >= 0;
    const int lend = tail ? lt : L - 1;
    std::vector<T*> cur(L, nullptr);
    pppm_status s;
    auto beta_of = [&](int l) { return consistent ? (T)mg_beta(l) : (T)0; };
    if (fold && !(l0 < lend && relax && nu1 > 2 && m.tile_level(l0, consistent))) {
        if ((s = m.prolong(l0, X[l0], fold, mode, beta_of(l0 + 1), st)) != PPPM_OK) return s;
        fold = nullptr;
    }
    for (int l = l0; l < lend; l++) {
        const T beta = beta_of(l), bs = l == 0 ? bscale0 : (T)1;
        if (relax && m.tile_level(l, consistent)) {
            if ((s = tile_down(m, l, X[l], l > l0 ? (const T*)nullptr : (const T*)X[l], (const T*)B[l], bs, nu1, nu2,
                               omega, beta, B[l + 1], l == l0 ? fold : (const T*)nullptr, mode, beta_of(l + 1), &cur[l],
                               st)) != PPPM_OK)
                return s;
            continue;
        }
        if (l > l0 && (s = m.fill(X[l], m.cells(l) * m.ncomp(), st)) != PPPM_OK) return s;
        if ((s = m.smooth(l, X[l], B[l], bs, nu1, omega, beta, st)) != PPPM_OK) return s;
        if ((s = m.residual_restrict(l, X[l], B[l], bs, beta, B[l + 1], st)) != PPPM_OK) return s;
    }
    if (tail) {
        if ((s = m.tail(lt > l0 ? (const T*)nullptr : (const T*)X[lt], X[lt], B[lt], B[lt + 1],
                        lt == 0 ? bscale0 : (T)1, nu1, nu2, omega, consistent, st)) != PPPM_OK)
            return s;
    } else {
        T bs = (L - 1) == 0 ? bscale0 : (T)1;
        if ((s = m.coarse(X[L - 1], B[L - 1], bs, consistent, st)) != PPPM_OK) return s;
    }
    for (int l = lend - 1; l >= l0; l--) {
        const T beta = beta_of(l), betac = beta_of(l + 1), bs = l == 0 ? bscale0 : (T)1;
        if (cur[l]) {
            if ((s = tile_up(m, l, X[l], cur[l], (const T*)B[l], bs, nu2, omega, beta, (const T*)X[l + 1], mode, betac,
                             st)) != PPPM_OK)
                return s;
            continue;
        }
        if ((s = m.prolong(l, X[l], X[l + 1], mode, betac, st)) != PPPM_OK) return s;
        if ((s = m.smooth(l, X[l], B[l], bs, nu2, omega, beta, st)) != PPPM_OK) return s;
    }
    return PPPM_OK;
}

// Fused V-cycle (float, consistent transfers): per level nu1 blocked passes
// of one red-black iteration each, the last also forming the residual and its
// restriction, and nu2 passes on the way up, the first adding the prolonged
// coarse correction as it loads x.
template <typename T>
static pppm_status vcycle_fused(MGHier<T>&, std::vector<T*>&, std::vector<T*>&, T, int, int, T, bool, hipStream_t) {
    return PPPM_ERR_INVALID;
}
template <>
pppm_status vcycle_fused<float>(MGHier<float>& m, std::vector<float*>& X, std::vector<float*>& B, float bscale0,
                                int nu1, int nu2, float omega, bool x0_zero, hipStream_t st) {
    const int L = m.levels(), nc = m.ncomp(), kind = m.blocked_smoother();
    pppm_status s;
    auto level_args = [&](int l) {
        const int* d = m.dims(l);
        const int* c = m.dims(l + 1);
        TbArgs a{};
        a.b = B[l];
        a.bscale = l == 0 ? bscale0 : 1.0f;
        a.nx = d[0];
        a.ny = d[1];
        a.nz = d[2];
        a.G = m.cells(l);
        a.omega = omega;
        a.beta = (float)mg_beta(l);
        a.w6 = omega / 6.0f;
        a.om1 = 1.0f - omega;
        a.zc = tb_zchunk(d[0], d[1], d[2], nc);
        a.cx = c[0];
        a.cy = c[1];
        a.cz = c[2];
        a.Gc = m.cells(l + 1);
        return a;
    };
    // Blocked passes pay a fixed latency per plane that small levels cannot
    // amortise: levels below the hierarchy's threshold run the tile passes
    // (k_tile), or with odd dimensions the one-launch-per-colour kernels in
    // place.
    auto blocked = [&](int l) { return m.blocked_level(l) && m.even(l); };
    // smoothing where odd dimensions keep the transfers apart: two iterations out
    // of place on levels large enough for blocked passes; one (copied back), and
    // any for odd nx (k_rb2), on a large level with many components only (us of
    // four V(2,2) cycles, a launch per half-sweep / k_rb2: 145 x 13 x 191 x 12 1278 /
    // 1027, 129 x 145 x 26 x 24 2539 / 1883; 65^3 x 12 842 / 887)
    auto sweeps = [&](int l, float bs, int nu, float beta) {
        const size_t n = m.cells(l);
        const bool pass = (nu == 2 && m.dims(l)[0] % 2 == 0 && m.blocked_level(l)) ||
                          (n >= m.blocked_min_cells() / 5 * 4 && n * nc >= (size_t)1 << 22);
        return pass ? m.smooth(l, X[l], B[l], bs, nu, omega, beta, st)
                    : m.smooth_colour(l, X[l], B[l], bs, nu, omega, beta, st);
    };
    // the small levels in one launch where they fit (l0 >= 1: X and B of
    // those levels are the hierarchy's own)
    const int l0 = m.tail_level();
    const int lend = l0 > 0 ? l0 : L - 1;  // levels below lend: the tail
    // down: nu1 passes per level, x from X (or zero below the finest level)
    // ping-ponging with the level's temporary; the last pass also restricts
    std::vector<float*> cur(L, nullptr);
    for (int l = 0; l < lend; l++) {
        if (m.tile_level(l, true)) {
            const bool zero = l > 0 || x0_zero;
            if ((s = tile_down(m, l, X[l], zero ? (const float*)nullptr : (const float*)X[l], (const float*)B[l],
                               l == 0 ? bscale0 : 1.0f, nu1, nu2, omega, (float)mg_beta(l), B[l + 1],
                               (const float*)nullptr, (int)PROLONG_TRILINEAR, 0.f, &cur[l], st)) != PPPM_OK)
                return s;
            continue;
        }
        if (!blocked(l)) {
            const float bs = l == 0 ? bscale0 : 1.0f, beta = (float)mg_beta(l);
            if ((l > 0 || x0_zero) && (s = m.fill(X[l], m.cells(l) * nc, st)) != PPPM_OK) return s;
            if ((s = sweeps(l, bs, nu1, beta)) != PPPM_OK) return s;
            if ((s = m.residual_restrict(l, X[l], B[l], bs, beta, B[l + 1], st)) != PPPM_OK) return s;
            cur[l] = X[l];
            continue;
        }
        float* src = X[l];
        float* dst = m.temp(l);
        // kind 4 runs nu = 2 as one pass of two iterations
        const bool two1 = kind == 4 && nu1 == 2 && r4_plane(m.dims(l)[0], m.dims(l)[1]);
        for (int q = 0; q < (two1 ? 1 : nu1); q++) {
            TbArgs a = level_args(l);
            a.xin = src;
            a.x = dst;
            a.bn = B[l + 1];
            const bool zero = (l > 0 || x0_zero) && q == 0, last = two1 || q == nu1 - 1;
            if (last)
                s = zero ? launch_rb2<true, false, true>(a, nc, kind, st, two1)
                         : launch_rb2<true, false, false>(a, nc, kind, st, two1);
            else
                s = zero ? launch_rb2<false, false, true>(a, nc, kind, st)
                         : launch_rb2<false, false, false>(a, nc, kind, st);
            if (s != PPPM_OK) return s;
            std::swap(src, dst);
        }
        cur[l] = src;
    }
    if (l0 > 0) {
        if ((s = m.tail(nullptr, X[l0], B[l0], B[l0 + 1], 1.0f, nu1, nu2, omega, true, st)) != PPPM_OK) return s;
        cur[l0] = X[l0];
    } else if ((s = m.coarse(X[L - 1], B[L - 1], L == 1 ? bscale0 : 1.0f, true, st)) != PPPM_OK) {
        return s;
    }
    // up: nu2 passes per level, the first adds the prolonged correction on load
    for (int l = l0 > 0 ? l0 - 1 : L - 2; l >= 0; l--) {
        if (m.tile_level(l, true)) {
            if ((s = tile_up(m, l, X[l], cur[l], (const float*)B[l], l == 0 ? bscale0 : 1.0f, nu2, omega,
                             (float)mg_beta(l), (const float*)X[l + 1], (int)PROLONG_TRILINEAR, (float)mg_beta(l + 1),
                             st)) != PPPM_OK)
                return s;
            continue;
        }
        if (!blocked(l)) {
            const float bs = l == 0 ? bscale0 : 1.0f, beta = (float)mg_beta(l);
            if ((s = m.prolong(l, X[l], X[l + 1], PROLONG_TRILINEAR, (float)mg_beta(l + 1), st)) != PPPM_OK)
                return s;
            if ((s = sweeps(l, bs, nu2, beta)) != PPPM_OK) return s;
            continue;
        }
        float* src = cur[l];
        float* dst = src == X[l] ? m.temp(l) : X[l];
        const bool two2 = kind == 4 && nu2 == 2 && r4_plane(m.dims(l)[0], m.dims(l)[1]);
        for (int q = 0; q < (two2 ? 1 : nu2); q++) {
            TbArgs a = level_args(l);
            a.xin = src;
            a.x = dst;
            a.xc = X[l + 1];
            a.betac = (float)mg_beta(l + 1);
            s = q == 0 ? launch_rb2<false, true, false>(a, nc, kind, st, two2)
                       : launch_rb2<false, false, false>(a, nc, kind, st);
            if (s != PPPM_OK) return s;
            std::swap(src, dst);
        }
        if (src != X[l] && (s = m.copy(X[l], src, m.cells(l) * nc, st)) != PPPM_OK) return s;
    }
    return PPPM_OK;
}

template <typename T>
pppm_status MGHier<T>::vcycle(T* x0, const T* b0, T bscale0, int nu1, int nu2, T omega, bool consistent,
                              hipStream_t st, bool x0_zero) {
    // the blocked prolongation takes parents as i / 2; a small odd level runs
    // a launch per colour inside the fused cycle
    bool even = true;
    for (int l = 0; l + 1 < L_; l++)
        if (cells(l) >= std::max(tb_min_cells_, kTileCells)) even = even && this->even(l);
    if (std::is_same<T, float>::value && consistent && tb_ && (nu1 == 1 || nu1 == 2) && (nu2 == 1 || nu2 == 2) &&
        L_ > 1 && even) {
        std::vector<T*> X = x_, B = b_;
        X[0] = x0;
        B[0] = const_cast<T*>(b0);
        return vcycle_fused<T>(*this, X, B, bscale0, nu1, nu2, omega, x0_zero, st);
    }
    std::vector<T*> X = x_, B = b_;
    X[0] = x0;
    B[0] = const_cast<T*>(b0);
    if (x0_zero) {
        pppm_status s = fill(x0, cells(0) * ncomp_, st);
        if (s != PPPM_OK) return s;
    }
    return vcycle_from(*this, X, B, 0, bscale0, nu1, nu2, omega, consistent, st);
}

template <typename T>
pppm_status MGHier<T>::ref_fmg(T* x0, const T* b0, T bscale0, int nu1, int nu2, T omega, hipStream_t st) {
    std::vector<T*> X = x_, B = b_;
    X[0] = x0;
    B[0] = const_cast<T*>(b0);
    pppm_status s;
    for (int l = 1; l < L_; l++)
        if ((s = fill(X[l], cells(l) * ncomp_, st)) != PPPM_OK) return s;
    for (int l = 0; l < L_ - 1; l++) {
        T bs = l == 0 ? bscale0 : (T)1;
        if ((s = residual_restrict(l, X[l], B[l], bs, (T)0, B[l + 1], st)) != PPPM_OK) return s;
    }
    if ((s = coarse(X[L_ - 1], B[L_ - 1], L_ == 1 ? bscale0 : (T)1, false, st)) != PPPM_OK) return s;
    for (int l = L_ - 2; l >= 0; l--) {
        if ((s = vcycle_from(*this, X, B, l, bscale0, nu1, nu2, omega, false, st, (const T*)X[l + 1])) != PPPM_OK)
            return s;
    }
    return vcycle_from(*this, X, B, 0, bscale0, nu1, nu2, omega, false, st);
}

template <typename T>
pppm_status MGHier<T>::norms_launch(const T* x0, const T* b0, T bscale0, hipStream_t st) {
    const int nx = d_[0][0], ny = d_[0][1], nz = d_[0][2];
    double* out = norm_out();
    int rw = 0;  // threads of a row: the power of two at or above nx, at most the block
    while (rw < 8 && (1 << rw) < nx) rw++;
    const int rows = ny * nz, step = kResRows << (8 - rw);
    const int blocks = std::min(kResBlocks, (rows + step - 1) / step);
    hipLaunchKernelGGL(k_resnorm<T>, dim3(blocks, ncomp_), dim3(256), 0, st, x0, b0, bscale0, nx, ny, nz, cells(0), rw,
                       part_);
    PPPM_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_reduce_partials, dim3(ncomp_), dim3(256), 0, st, part_, blocks, out);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

template <typename T>
pppm_status MGHier<T>::norms_read(double* rn, double* bn, hipStream_t st) {
    double* out = norm_out();
    PPPM_HIP_TRY(hipMemcpyAsync(hnorm_, out, 2 * ncomp_ * sizeof(double), hipMemcpyDeviceToHost, st));
    PPPM_HIP_TRY(hipStreamSynchronize(st));
    for (int c = 0; c < ncomp_; c++) {
        rn[c] = std::sqrt(hnorm_[2 * c]);
        bn[c] = std::sqrt(hnorm_[2 * c + 1]);
    }
    return PPPM_OK;
}

template <typename T>
pppm_status MGHier<T>::norms(const T* x0, const T* b0, T bscale0, double* rn, double* bn, hipStream_t st) {
    pppm_status s = norms_launch(x0, b0, bscale0, st);
    if (s != PPPM_OK) return s;
    return norms_read(rn, bn, st);
}

template <typename T>
pppm_status MGHier<T>::solve(T* x0, const T* b0, T bscale0, int nu1, int nu2, T omega, double tol, int max_cycles,
                             int* cycles, double* relres, hipStream_t st) {
    double rn[kMaxComp], bn[kMaxComp];
    pppm_status s;
    int cyc = 0;
    auto worst = [&]() {
        double w = 0;
        for (int c = 0; c < ncomp_; c++) {
            double r = bn[c] > 0 ? rn[c] / bn[c] : rn[c];
            relres[c] = r;
            if (r > w) w = r;
        }
        return w;
    };
    if ((s = norms(x0, b0, bscale0, rn, bn, st)) != PPPM_OK) return s;
    double w = worst();
    while (cyc < max_cycles && w > tol) {
        if ((s = vcycle(x0, b0, bscale0, nu1, nu2, omega, true, st)) != PPPM_OK) return s;
        cyc++;
        if ((s = norms(x0, b0, bscale0, rn, bn, st)) != PPPM_OK) return s;
        double prev = w;
        w = worst();
        // rounding floor of the working precision reached: stop
        if (cyc >= 3 && w > 0.9 * prev) break;
    }
    *cycles = cyc;
    return w <= tol ? PPPM_OK : PPPM_ERR_NOT_CONVERGED;
}

template class MGHier<float>;
template class MGHier<double>;

// ---------------------------------------------------------------------------
// Single-array primitives behind the reference's mg_* entry points
// (Multigrid.cu:46-60, 202-330).
template <typename T>
__global__ void __launch_bounds__(256) k_residual_full(const T* __restrict__ x, const T* __restrict__ b,
                                                       T* __restrict__ r, int nx, int ny, int nz) {
    const int i = blockIdx.x * 64 + threadIdx.x;
    const int j = blockIdx.y * 4 + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= nx || j >= ny) return;
    r[((size_t)k * ny + j) * nx + i] = residual_at(x, b, (T)1, i, j, k, nx, ny, nz, (T)0);
}

template <typename T>
__global__ void __launch_bounds__(256) k_restrict_full(T* __restrict__ bc, const T* __restrict__ rf, int cx, int cy,
                                                       int cz) {
    const int i = blockIdx.x * 64 + threadIdx.x;
    const int j = blockIdx.y * 4 + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= cx || j >= cy) return;
    const size_t nx = 2 * (size_t)cx, ny = 2 * (size_t)cy;
    const size_t a = ((size_t)(2 * k) * ny + 2 * j) * nx + 2 * i;
    const size_t ay = a + nx, az = a + nx * ny, ayz = az + nx;
    T r = 0;
    r += rf[a];
    r += rf[a + 1];
    r += rf[ay];
    r += rf[ay + 1];
    r += rf[az];
    r += rf[az + 1];
    r += rf[ayz];
    r += rf[ayz + 1];
    bc[((size_t)k * cy + j) * cx + i] = r * (T)0.5;
}

template <typename T>
pppm_status ref_rbgs(T* x, const T* b, int iters, int nx, int ny, int nz, T omega, hipStream_t st) {
    for (int it = 0; it < iters; it++)
        for (int color = 1; color >= 0; color--) {
            launch_rbgs(x, b, (T)1, nx, ny, nz, 1, color, omega, (T)0, st);
            PPPM_LAUNCH_CHECK();
        }
    return PPPM_OK;
}

template <typename T>
pppm_status ref_residual(const T* x, const T* b, T* r, int nx, int ny, int nz, hipStream_t st) {
    hipLaunchKernelGGL(k_residual_full<T>, dim3(div_up(nx, 64), div_up(ny, 4), nz), dim3(64, 4), 0, st, x, b, r, nx,
                       ny, nz);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

template <typename T>
pppm_status ref_restrict(T* bc, const T* rf, int cx, int cy, int cz, hipStream_t st) {
    hipLaunchKernelGGL(k_restrict_full<T>, dim3(div_up(cx, 64), div_up(cy, 4), cz), dim3(64, 4), 0, st, bc, rf, cx,
                       cy, cz);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

template <typename T>
pppm_status ref_prolong(T* xf, const T* xc, int fx, int fy, int fz, hipStream_t st) {
    int cx = fx / 2 > 0 ? fx / 2 : 1, cy = fy / 2 > 0 ? fy / 2 : 1, cz = fz / 2 > 0 ? fz / 2 : 1;
    hipLaunchKernelGGL(k_prolong<T>, dim3(div_up(fx, 64), div_up(fy, 4), fz), dim3(64, 4), 0, st, xf, xc, fx, fy, fz,
                       cx, cy, cz, (size_t)fx * fy * fz, (size_t)cx * cy * cz, (int)PROLONG_CONSTANT, (T)0);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

template <typename T>
pppm_status ref_coarse(T* res, const T* b, int nx, int ny, int nz, hipStream_t st) {
    if ((long)nx * ny * nz > 512) {
        pppm_set_last_error("coarse solve needs <= 512 cells", __FILE__, __LINE__);
        return PPPM_ERR_INVALID;
    }
    std::vector<double> t = coarse_tables(nx, ny, nz, 0.0);
    double* d = nullptr;
    PPPM_HIP_TRY(hipMalloc(&d, t.size() * sizeof(double)));
    hipError_t e = hipMemcpyAsync(d, t.data(), t.size() * sizeof(double), hipMemcpyHostToDevice, st);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_coarse<T>, dim3(1), dim3(512), 0, st, res, b, (T)1, nx, ny, nz, (size_t)nx * ny * nz, d);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    (void)hipFree(d);
    PPPM_HIP_TRY(e);
    return PPPM_OK;
}

#define PPPM_INST_REF(T)                                                                                  \
    template pppm_status ref_rbgs<T>(T*, const T*, int, int, int, int, T, hipStream_t);                    \
    template pppm_status ref_residual<T>(const T*, const T*, T*, int, int, int, hipStream_t);              \
    template pppm_status ref_restrict<T>(T*, const T*, int, int, int, hipStream_t);                        \
    template pppm_status ref_prolong<T>(T*, const T*, int, int, int, hipStream_t);                         \
    template pppm_status ref_coarse<T>(T*, const T*, int, int, int, hipStream_t);
PPPM_INST_REF(float)
PPPM_INST_REF(double)

}  // namespace pppm
