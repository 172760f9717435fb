// M2P interpolation of the far-field buffer and the near-field Biot-Savart
// correction added onto it, both written in the caller's order
// (GPU_kernel.cu:2886-2964 BiotSavartInterpolate_far_field_kernel2,
//  2262-2436 BiotSavartPPCorrScaleMN_kernel, BiotSavartSolverImp.cpp:452-484).
#include "pppm_internal.hpp"
#include <algorithm>
#include <type_traits>

namespace pppm {

struct NearConst {
    float rbox;        // largest float r with (double)r < (K + 1/2) h
    float inv_a;       // 1 / core radius
    float inv_a3;      // 1 / a^3
    float inv4pi;      // 1 / (4 pi) with the reference's 4 pi
    float kexp2;       // -log2(e) / a^3: exp(-(r/a)^3) = exp2(kexp2 r^3)
    float r3_series;   // 0.1 a^3: below it (x = (r/a)^3 < 0.1) the series form
    float sc[5];       // series coefficients of (1 - e^-x) / x, times 1 / a^3
    // potential-flow kernels: core radius, the coefficient inside it
    // (1 / (4 pi a^3) for the gradient, 1 / (4 pi a) for the potential) and
    // G times the direction
    float pa, pc, pg;
};

// q(rho) / r^3 for the expcubic core, q = 1 - exp(-(r/a)^3)
// (GPU_kernel.cu:2389-2402), 1 / (4 pi) left to the caller.  For x = (r/a)^3 <
// 0.1 a series of (1 - e^-x) / x avoids the cancellation.  Pairs that close
// are rare: every lane takes the exponential form (r^-3 - e r^-3 as one fused
// multiply-add), and the series runs only in waves where some lane needs it (a
// wave-uniform branch, so other waves issue none of its instructions).
__device__ inline float coeff_expcubic_4pi(float r2, const NearConst& nc) {
    const float rinv = __frsqrt_rn(r2);
    const float r3 = r2 * (r2 * rinv);
    const float e = __builtin_amdgcn_exp2f(nc.kexp2 * r3);
    const float ri3 = rinv * rinv * rinv;
    float c = fmaf(-e, ri3, ri3);
    const bool small = r3 < nc.r3_series;
    if (__ballot(small) != 0) {
        __asm__ volatile("");  // not speculated: keeps the branch a branch
        const float x = r3 * nc.inv_a3;
        if (small)
            c = fmaf(x, fmaf(x, fmaf(x, fmaf(x, nc.sc[4], nc.sc[3]), nc.sc[2]), nc.sc[1]), nc.sc[0]);
    }
    return c;
}

// Gaussian core: q = erf(rho/sqrt2) - sqrt(2/pi) rho exp(-rho^2/2)
__device__ inline float coeff_gaussian(float r2, const NearConst& nc) {
    float rinv = __frsqrt_rn(r2);
    float r = r2 * rinv;
    float rho = r * nc.inv_a;
    float q;
    if (rho < 0.5f) {
        float p2 = rho * rho;
        float s = 1.0f / 3.0f + p2 * (-1.0f / 10.0f + p2 * (1.0f / 56.0f + p2 * (-1.0f / 432.0f + p2 * (1.0f / 3840.0f))));
        q = 0.7978845608f * rho * p2 * s;
    } else {
        q = erff(rho * 0.7071067812f) - 0.7978845608f * rho * __expf(-0.5f * rho * rho);
    }
    return q * (rinv * rinv * rinv) * nc.inv4pi;
}

// Float bounds of a double: the largest float <= x, the smallest float >= x.
__device__ inline float float_down(double x) {
    float f = (float)x;
    return (double)f > x ? nextafterf(f, -3.4e38f) : f;
}
__device__ inline float float_up(double x) {
    float f = (float)x;
    return (double)f < x ? nextafterf(f, 3.4e38f) : f;
}

// Cell bound along one axis of the range holding every vortex whose
// coordinate is within rb of v: the upper cell floor((v + rb)/h + 1e-3)
// (up) or the lower floor((v - rb)/h - 1e-3).  A vortex's hash cell equals
// floor of its coordinate over h up to FP32 rounding of the hash (far below
// 1e-3 cells), so the margin keeps the range a superset of the box; the box
// test decides.  The clamp runs in FP64 before the conversion (lower to
// [0, 2^31 - 1], upper to [-1, gi - 1]), which gives the saturating
// conversion's cell for every non-NaN input; a NaN bound yields 0 or -1, an
// empty or rejected range either way.
__device__ inline int near_cell_bound(float v, double rb, double invh, int gi, bool up) {
    const double sg = up ? 1.0 : -1.0;
    const double x = floor(fma(fma(sg, rb, (double)v), invh, sg * 1e-3));
    return (int)fmin(fmax(x, up ? -1.0 : 0.0), up ? (double)(gi - 1) : 2147483647.0);
}
// Staging bound: v + rw rounded up (up) or v - rw rounded down, as a float.
__device__ inline float near_stage_bound(float v, double rw, bool up) {
    const double x = fma(up ? 1.0 : -1.0, rw, (double)v);
    return up ? float_up(x) : float_down(x);
}

// Wave-level exchanges through DPP.  quad_perm [1,0,3,2] and [2,3,0,1] swap
// within each quad of lanes; row_ror 4 and 8 rotate within a row of 16.
template <int CTRL>
__device__ inline float dpp_mov(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ inline float quad_min(float v) {
    float t = dpp_mov<0xB1>(v);
    v = t < v ? t : v;
    t = dpp_mov<0x4E>(v);
    return t < v ? t : v;
}
__device__ inline float quad_max(float v) {
    float t = dpp_mov<0xB1>(v);
    v = t > v ? t : v;
    t = dpp_mov<0x4E>(v);
    return t > v ? t : v;
}
// Inclusive prefix sum over the wave: row_shr 1, 2, 4, 8 within rows of 16
// (lanes past a row's start add 0), then row 15's total into rows 1 and 3
// (row_bcast:15) and lane 31's into rows 2 and 3 (row_bcast:31).
__device__ inline uint32_t wave_inclusive_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);
    return v;
}

// M2P (GPU_kernel.cu:2886-2964): the far-field buffer interpolated at
// each sorted evaluation point with hat weights about cell centres (in-grid
// cells only, corners summed in x-fastest order), into the point's output
// slot.  Vortex-in-cell mode (no near field) only: with a near field the
// near-field kernel interpolates the same corners itself.
template <typename TO>
__global__ void __launch_bounds__(256) k_m2p_points(const float4* __restrict__ epos, const uint32_t* __restrict__ eidx,
                                                    uint32_t m, const float* __restrict__ far, uint32_t g, double invh,
                                                    TO* __restrict__ ux, TO* __restrict__ uy,
                                                    TO* __restrict__ uz, uint32_t u_stride) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= m) return;
    const float4 a = epos[t];
    const int gi = (int)g;
    const size_t G = (size_t)g * g * g;
    float sx = 0.f, sy = 0.f, sz = 0.f;
    const int i = cell_of(a.x, invh), j = cell_of(a.y, invh), k = cell_of(a.z, invh);
    // a NaN coordinate counts as outside the grid (cell_of maps it to 0)
    const bool fin = a.x == a.x && a.y == a.y && a.z == a.z;
    if (fin && i >= 0 && i < gi && j >= 0 && j < gi && k >= 0 && k < gi) {
        const double xh = (double)a.x * invh - 0.5, yh = (double)a.y * invh - 0.5, zh = (double)a.z * invh - 0.5;
        const int i0 = (int)floor(xh), j0 = (int)floor(yh), k0 = (int)floor(zh);
        const float fx = (float)(xh - i0), fy = (float)(yh - j0), fz = (float)(zh - k0);
        // the lower corner is at most one cell outside the grid per axis and
        // the upper one inside, so per axis: lower valid iff >= 0, upper iff
        // < gi.  Cell indices fit 32 bits (g <= 1024); a lower corner at -1
        // wraps and the +1 of the upper corner brings it back.
        const bool lx = i0 >= 0, ux = i0 + 1 < gi, ly = j0 >= 0, uy = j0 + 1 < gi, lz = k0 >= 0, uz = k0 + 1 < gi;
        const uint32_t q0 = ((uint32_t)k0 * g + (uint32_t)j0) * g + (uint32_t)i0, gg = g * g;
        const char* Fx = reinterpret_cast<const char*>(far);
        const char* Fy = reinterpret_cast<const char*>(far + G);
        const char* Fz = reinterpret_cast<const char*>(far + 2 * G);
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const int a2 = c & 1, b2 = (c >> 1) & 1, c2 = c >> 2;
            if ((a2 ? ux : lx) && (b2 ? uy : ly) && (c2 ? uz : lz)) {
                const uint32_t ob = 4u * (q0 + (uint32_t)a2 + (b2 ? g : 0u) + (c2 ? gg : 0u));
                const float wgt = (a2 ? fx : 1.f - fx) * (b2 ? fy : 1.f - fy) * (c2 ? fz : 1.f - fz);
                sx += wgt * *reinterpret_cast<const float*>(Fx + ob);
                sy += wgt * *reinterpret_cast<const float*>(Fy + ob);
                sz += wgt * *reinterpret_cast<const float*>(Fz + ob);
            }
        }
    }
    const uint32_t dt = eidx[t];
    if (dt >= m) return;
    const size_t dst = (size_t)dt * u_stride;
    ux[dst] = (TO)sx;
    uy[dst] = (TO)sy;
    uz[dst] = (TO)sz;
}

// Potential-flow near fields, in clusters: one wave takes kNearTI consecutive sorted evaluation points
// (usually one hash cell) and splits the vortices among kNearSJ lanes per
// point (lane = point + kNearTI * slice).  It scans the hash rows covering the
// union of the points' boxes (consecutive x cells of a row are consecutive
// sorted vortices).  The rows' vortex ranges are read in one vector load (a
// row per lane) and packed into one stream, which is staged 64 vortices at a
// time into LDS with the next chunk's loads in flight; each lane tests its
// slice of the chunk against its point and evaluates the kernel where the box
// test passes.  The point's M2P interpolation (k_m2p_points' corners and
// weights, corner c on slice c) joins the partial sums, which are reduced
// over the slices at the end (fixed order, deterministic).  All loop bounds
// are wave-uniform.  The vortex kernels have a layout of their own
// (k_m2p_near); the potential's FP64 outputs hold these FP32 sums and keep
// this order of summation.
constexpr int kNearTI = 4;
constexpr int kNearSJ = 64 / kNearTI;
static_assert(kNearTI == 4, "the union box is a min / max over a quad of lanes (quad_min, quad_max)");

// WIDE: 64-bit vortex addressing; otherwise (fewer than 2^28 vortices) a
// vortex's byte offset fits 32 bits and the loads take a scalar base plus a
// 32-bit lane offset.
template <int KERNEL, typename TO, bool WIDE>
__global__ void __launch_bounds__(256) k_pot_near(const float4* __restrict__ epos,
                                                  const uint32_t* __restrict__ eidx, uint32_t m,
                                                  const uint32_t* __restrict__ off, const float4* __restrict__ spos,
                                                  const float4* __restrict__ somg, const float* __restrict__ far,
                                                  uint32_t g, int K, double invh, NearConst nc, TO* __restrict__ ux,
                                                  TO* __restrict__ uy, TO* __restrict__ uz, uint32_t u_stride,
                                                  const uint32_t* __restrict__ tperm) {
    // per wave: a ring of 128 staged vortices (two windows of 64), positions
    // then strengths, so one address serves both (the second at +2048 bytes)
    __shared__ float4 ring[4][2][128];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ti = lane % kNearTI, sj = lane / kNearTI;
    // Workgroup -> cluster range: groups of 256 consecutive workgroups per
    // XCD (an XCD holds 32 CUs x 8 workgroups of this kernel at once), so
    // each L2 serves one run of about 4,096 consecutive points, whose boxes
    // share most of their hash rows (HBM traffic 21 -> 8.4 GB and -3% time
    // at 8M/256^3; groups of 64, 128, 512, 1024 gained less)
    const uint32_t wg = xcd_group<256>(blockIdx.x, gridDim.x);
    const uint32_t t0 = (wg * 4 + w) * kNearTI;
    if (t0 >= m) return;  // the whole wave leaves together; no block barriers below
    // evaluation slot -> sorted point (octant order within cells, or itself)
    const uint32_t slot = t0 + ti;
    const bool tv = slot < m;
    const uint32_t t = tperm ? tperm[tv ? slot : t0] : (tv ? slot : t0);
    const float4 a = epos[t];
    const int gi = (int)g;
    const size_t G = (size_t)g * g * g;

    float vx = 0.f, vy = 0.f, vz = 0.f;
    {
        // ---- union of the points' boxes -> scanned cell range (wave-uniform)
        // Every quad of lanes holds the wave's four points, so the union is a
        // min / max over the quad.  A NaN coordinate stays out of the union
        // (as fminf would leave it; all-NaN gives an empty range).
        const bool okx = tv && a.x == a.x, oky = tv && a.y == a.y, okz = tv && a.z == a.z;
        const float mnx = quad_min(okx ? a.x : 3.0e38f), mny = quad_min(oky ? a.y : 3.0e38f),
                    mnz = quad_min(okz ? a.z : 3.0e38f);
        const float mxx = quad_max(okx ? a.x : -3.0e38f), mxy = quad_max(oky ? a.y : -3.0e38f),
                    mxz = quad_max(okz ? a.z : -3.0e38f);
        const double rb = (double)nc.rbox;
        const float rbox = nc.rbox;
        // Lane j < 6 computes one axis's bounds (j = axis: lower, 3 + axis:
        // upper): the cell range and the staging bound.
        // Staging bounds per axis: every vortex the box test can accept for a
        // point of the cluster lies strictly inside (lo, hi).  The test keeps
        // fl(|p - s|) <= rbox, so |p - s| <= rbox (1 + 2^-23) exactly, and s >
        // min - rbox (1 + 2^-21) >= lo, with lo that bound rounded down (hi:
        // max + rbox (1 + 2^-21) rounded up).  Vortices outside are not staged.
        const int bj = lane < 6 ? lane : 0;
        const bool bup = bj >= 3;
        const int bax = bup ? bj - 3 : bj;
        const float bvv = bax == 0 ? (bup ? mxx : mnx) : bax == 1 ? (bup ? mxy : mny) : (bup ? mxz : mnz);
        const int cbnd = near_cell_bound(bvv, rb, invh, gi, bup);
        const float sbnd = near_stage_bound(bvv, rb * (1.0 + 0x1p-21), bup);
        const int xlo = __builtin_amdgcn_readlane(cbnd, 0), ylo = __builtin_amdgcn_readlane(cbnd, 1),
                  zlo = __builtin_amdgcn_readlane(cbnd, 2);
        const int xhi = __builtin_amdgcn_readlane(cbnd, 3), yhi = __builtin_amdgcn_readlane(cbnd, 4),
                  zhi = __builtin_amdgcn_readlane(cbnd, 5);
        auto sb = [&](int j) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sbnd), j)); };
        const float lox = sb(0), loy = sb(1), loz = sb(2), hix = sb(3), hiy = sb(4), hiz = sb(5);
        const uint32_t nsrc = off[G];
        const int ny_ = yhi - ylo + 1;
        const int nrows = (xlo <= xhi && ylo <= yhi && zlo <= zhi) ? (zhi - zlo + 1) * ny_ : 0;
        // row r -> (z, y) = (r / ny_, r % ny_) through a float reciprocal
        // (within 1 ulp): exact while r < 2^21 (nrows <= g^2 <= 2^20)
        const float inv_ny = __builtin_amdgcn_rcpf((float)max(ny_, 1));
        // Evaluate the window [wh, wh + n) of the ring (wh is 0 or 64): lane
        // (point, slice) tests ring entries wh + slice + kNearSJ j, j <
        // kNearTI.  (A ring of 256 with 128-entry windows halves the
        // occupancy through its LDS and runs half again as long.)
        auto evaluate = [&](uint32_t wh, uint32_t n) {
            // the candidates' positions are read together (eight waves per
            // SIMD still fit; their strengths, read ahead too, ran slower)
            float4 sv[kNearTI];
#pragma unroll
            for (int qq = 0; qq < kNearTI; qq++) sv[qq] = ring[w][0][wh + sj + qq * kNearSJ];
#pragma unroll
            for (int qq = 0; qq < kNearTI; qq++) {
                const uint32_t q = sj + qq * kNearSJ;
                const float4 s = sv[qq];
                const float dx = a.x - s.x, dy = a.y - s.y, dz = a.z - s.z;
                const float r2 = fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, 0.f)));
                // |d|inf <= rbox as one max3 of absolute values; a point
                // past the end of the evaluation set (tv false) computes on
                // a copy of its cluster's first point and is not stored
                // (the potential keeps coincident masses: they add G m 1e-14)
                const bool acc = q < n && fmaxf(fmaxf(fabsf(dx), fabsf(dy)), fabsf(dz)) <= rbox &&
                                 (KERNEL == kNearPotScalar || r2 >= 1e-24f);
                if (acc) {
                    const float4 o = ring[w][1][wh + q];
                    if constexpr (KERNEL == kNearPotGrad) {
                        // Potential_PPCorrMN_kernel (GPU_kernel.cu:750-870):
                        // G m (x_m - x) / (4 pi max(r, a)^3), the mass in o.x
                        const float rinv = __frsqrt_rn(r2);
                        const float c =
                            nc.pg * o.x * (r2 * rinv > nc.pa ? nc.inv4pi * (rinv * rinv * rinv) : nc.pc);
                        vx = fmaf(-c, dx, vx);
                        vy = fmaf(-c, dy, vy);
                        vz = fmaf(-c, dz, vz);
                    } else {
                        // Potential_PPCorrMNScalar_kernel (GPU_kernel.cu:1301-1419):
                        // G m / (4 pi max(r, a)), G m 1e-14 for r < 1e-12
                        const float rinv = __frsqrt_rn(r2);
                        const float c = r2 < 1e-24f ? 1e-14f : (r2 * rinv > nc.pa ? nc.inv4pi * rinv : nc.pc);
                        vx = fmaf(nc.pg * o.x, c, vx);
                    }
                }
            }
            // the next staging may overwrite these entries
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        };
        // ring state (wave-uniform): window head (0 or 64) and entries held
        uint32_t qh = 0, qn = 0;
        for (int r0 = 0; r0 < nrows; r0 += 64) {
            // lane l holds the vortex range [lp0, lp1) of row r0 + l (z outer,
            // y inner), loaded in one pass instead of row after row
            uint32_t lp0 = 0, lp1 = 0;
            if (r0 + lane < nrows) {
                const int r = r0 + lane;
                const int rz = (int)(((float)r + 0.5f) * inv_ny);
                const uint32_t kk = (uint32_t)(zlo + rz), jj = (uint32_t)(ylo + r - rz * ny_);
                const uint32_t rowc = (kk * g + jj) * g;
                lp0 = off[rowc + xlo];
                lp1 = min(off[rowc + xhi + 1], nsrc);
            }
            const int rn = min(64, nrows - r0);
            // The rows are packed into one stream of vortices: chunk c holds
            // stream positions 64 c .. 64 c + 63 across row boundaries.  pre
            // is a row's first stream position (exclusive prefix of the row
            // lengths), roff maps stream position to vortex index.
            const uint32_t len = lp1 > lp0 ? lp1 - lp0 : 0u;
            const uint32_t incl = wave_inclusive_scan(len);
            const uint32_t pre = incl - len, roff = lp0 - pre;
            const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
            // vortex index of this lane's position in the chunk at S0; rcur
            // (wave-uniform) is a row at or before the one holding S0 and is
            // advanced to the last row starting at or before S0 + 64
            auto locate = [&](uint32_t S0, int& rcur) {
                const uint32_t S = S0 + (uint32_t)lane;
                uint32_t mo = __builtin_amdgcn_readlane(roff, rcur);
                int rnext = rcur;
                for (int rr = rcur + 1; rr < rn; rr++) {
                    const uint32_t p = __builtin_amdgcn_readlane(pre, rr);
                    if (p > S0 + 64) break;
                    rnext = rr;
                    if (S >= p) mo = __builtin_amdgcn_readlane(roff, rr);
                }
                rcur = rnext;
                return S + mo;
            };
            int rc = 0;
            // The next chunk is loaded into registers while this one is
            // staged.  Slots past the end of the stream (pin false) read
            // vortex 0 and are not staged.
            float4 pp = make_float4(0.f, 0.f, 0.f, 0.f), po = pp;
            float lxl = __builtin_inff();
            auto load = [&](uint32_t S0) {
                const uint32_t vi = locate(S0, rc);
                const bool pin = S0 + (uint32_t)lane < total;
                lxl = pin ? lox : __builtin_inff();  // a slot past the end fails the filter
                const uint32_t v = pin ? vi : 0u;
                if (WIDE) {
                    pp = spos[v];
                    po = somg[v];
                } else {
                    const uint32_t ob = v << 4;
                    pp = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(spos) + ob);
                    po = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(somg) + ob);
                }
            };
            if (total > 0) load(0u);
            for (uint32_t S0 = 0; S0 < total; S0 += 64) {
                // Stage only the vortices some point's box may accept (inside
                // the staging bounds on every axis; a NaN coordinate fails).
                // the lane masks of the six compares (ordered: NaN fails)
                // ANDed on the scalar unit, then the mask as the predicate
                const uint64_t bal =
                    __builtin_amdgcn_fcmpf(pp.x, lxl, 2) & __builtin_amdgcn_fcmpf(pp.x, hix, 4) &
                    __builtin_amdgcn_fcmpf(pp.y, loy, 2) & __builtin_amdgcn_fcmpf(pp.y, hiy, 4) &
                    __builtin_amdgcn_fcmpf(pp.z, loz, 2) & __builtin_amdgcn_fcmpf(pp.z, hiz, 4);
                const bool use = __builtin_amdgcn_inverse_ballot_w64(bal);
                // ring slot: the head plus the kept lanes below this one
                const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32),
                                                              __builtin_amdgcn_mbcnt_lo((uint32_t)bal, qh + qn));
                if (use) {
                    const uint32_t e = at & 127u;
                    ring[w][0][e] = pp;
                    ring[w][1][e] = po;
                }
                qn += (uint32_t)__popcll(bal);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if (S0 + 64 < total) load(S0 + 64);
                // a full window: evaluate it and move the head to the other
                if (qn >= 64) {
                    evaluate(qh, 64u);
                    qh ^= 64u;
                    qn -= 64u;
                }
            }
        }
        if (qn > 0) evaluate(qh, qn);  // the last, partial window
    }
    // ---- M2P: the point's 8 interpolation corners, corner sj on slice sj
    // (the weights and validity of k_m2p_points), into the slice sums
    if (sj < 8 && tv) {
        const int i = cell_of(a.x, invh), j = cell_of(a.y, invh), k = cell_of(a.z, invh);
        const bool fin = a.x == a.x && a.y == a.y && a.z == a.z;
        if (fin && i >= 0 && i < gi && j >= 0 && j < gi && k >= 0 && k < gi) {
            const double xh = (double)a.x * invh - 0.5, yh = (double)a.y * invh - 0.5, zh = (double)a.z * invh - 0.5;
            const int i0 = (int)floor(xh), j0 = (int)floor(yh), k0 = (int)floor(zh);
            const float fx = (float)(xh - i0), fy = (float)(yh - j0), fz = (float)(zh - k0);
            const int a2 = sj & 1, b2 = (sj >> 1) & 1, c2 = sj >> 2;
            const bool ok = (a2 ? i0 + 1 < gi : i0 >= 0) && (b2 ? j0 + 1 < gi : j0 >= 0) && (c2 ? k0 + 1 < gi : k0 >= 0);
            if (ok) {
                const uint32_t q = (((uint32_t)k0 + (uint32_t)c2) * g + (uint32_t)j0 + (uint32_t)b2) * g + (uint32_t)i0 +
                                   (uint32_t)a2;
                const float wgt = (a2 ? fx : 1.f - fx) * (b2 ? fy : 1.f - fy) * (c2 ? fz : 1.f - fz);
                vx = fmaf(wgt, far[q], vx);
                if (KERNEL != kNearPotScalar) {
                    vy = fmaf(wgt, far[G + q], vy);
                    vz = fmaf(wgt, far[2 * G + q], vz);
                }
            }
        }
    }
    // ---- reduce over the slices of each point
    // (lanes ti + 4 sj: within a row of 16 by rotations of 4 and 8, then
    // across the rows; a fixed order)
    float rx = vx, ry = vy, rz = vz;
    rx += dpp_mov<0x124>(rx);
    ry += dpp_mov<0x124>(ry);
    rz += dpp_mov<0x124>(rz);
    rx += dpp_mov<0x128>(rx);
    ry += dpp_mov<0x128>(ry);
    rz += dpp_mov<0x128>(rz);
    for (int o = 16; o < 64; o <<= 1) {
        rx += __shfl_xor(rx, o, 64);
        ry += __shfl_xor(ry, o, 64);
        rz += __shfl_xor(rz, o, 64);
    }
    // plus the point's M2P value
    if (sj == 0 && tv) {
        const uint32_t dt = eidx[t];
        if (dt < m) {
            const size_t dst = (size_t)dt * u_stride;
            ux[dst] = (TO)rx;
            if (KERNEL != kNearPotScalar) {  // a scalar has one output
                uy[dst] = (TO)ry;
                uz[dst] = (TO)rz;
            }
        }
    }
}

// ---- vortex near field -----------------------------------------------------
// min / max over the T points that every T consecutive lanes hold
template <int T>
__device__ inline float group_min(float v) {
    if (T == 1) return v;
    if (T == 2) return fminf(v, dpp_mov<0xB1>(v));
    v = quad_min(v);
    if (T == 8) v = fminf(v, dpp_mov<0x124>(v));
    return v;
}
template <int T>
__device__ inline float group_max(float v) {
    if (T == 1) return v;
    if (T == 2) return fmaxf(v, dpp_mov<0xB1>(v));
    v = quad_max(v);
    if (T == 8) v = fmaxf(v, dpp_mov<0x124>(v));
    return v;
}
// v[0..T) per lane -> in lane l the sum, over the lanes that differ from l in
// their low log2(T) bits only, of v[l % T].  Each step exchanges half of the
// values with the lane whose next bit differs (for the third bit the lane four
// below in the row of 16, whose higher bits are summed over later anyway).
template <int T>
__device__ inline float transpose_reduce(float (&v)[T], int lane) {
#pragma unroll
    for (int q = 0; q < T / 2; q++) {
        const bool b = lane & 1;
        const float keep = b ? v[2 * q + 1] : v[2 * q], give = b ? v[2 * q] : v[2 * q + 1];
        v[q] = keep + dpp_mov<0xB1>(give);
    }
#pragma unroll
    for (int q = 0; q < T / 4; q++) {
        const bool b = lane & 2;
        const float keep = b ? v[2 * q + 1] : v[2 * q], give = b ? v[2 * q] : v[2 * q + 1];
        v[q] = keep + dpp_mov<0x4E>(give);
    }
    if (T == 8) {
        const bool b = lane & 4;
        const float keep = b ? v[1] : v[0], give = b ? v[0] : v[1];
        v[0] = keep + dpp_mov<0x124>(give);
    }
    return v[0];
}

// When a group of points is given up for its halves: beyond vlim cells, and where
// few vortices share a cell (SPARSE) only if that costs less.
struct NearSplit {
    int vlim, edge;           // edge: of a point's own box
    float pass, row, vortex;  // instructions of a pass, of a grid row and a vortex in it
    float mean;               // vortices a cell
};

// One wave takes T consecutive sorted evaluation points.  Their coordinates
// sit in scalar registers and the sources in lanes: the hash rows covering the
// union of the points' boxes are packed into one stream of sources, those inside
// the union box are compacted into a ring of 128, and every full window of 64 is
// read back one source a lane and tested against the T points in turn.  A source is read from LDS once for T points
// (one read per pair in k_pot_near's point-by-slice layout), and a point
// whose box holds few of a window's sources costs little, since the sources of
// a window follow the hash rows and the lanes that fail the box test come in
// runs.  What bounds it is the vector issue rate: 6 instructions a source and
// point, 20 more where some lane passes.
// A union box of more than split.vlim cells (points around the end of a grid row
// or plane, or far apart) is given up for two halves of the points, down to
// single ones: before, one wave at the end of a plane walked all of its rows and
// ran on alone (0.79 -> 0.45 ms at 700,001 uniform vortices on 96^3).  In sparse
// scenes (SPARSE) eight points stretch over a large part of a grid row, whose
// halves hold the same vortices in all: they stay together unless the halves or
// the single points cost less (uniform on 256^3, ms, split beyond vlim / by cost:
// 1/8 a cell 1.77 / 1.29, 1/16 1.14 / 0.55; 512^3 of 1/16 8.97 / 5.26).
// Measured, ms a launch, k_pot_near -> here (same box, in the sort's order):
// 8M plume 256^3 16.4 -> 11.6, 33.5M plume 512^3 45.9 -> 30.3, 2M ring 128^3
// 28.8 -> 22.6, 1M plume 128^3 1.87 -> 1.43, 700k uniform 96^3 0.79 -> 0.37,
// 65,536 uniform 32^3 0.153 -> 0.073; the Gaussian core's 1M plume 2.65 -> 2.61,
// 700k uniform 0.92 -> 0.49.  T = 16 needs 96 VGPRs: 12.4 ms at the 8M plume.  At
// eight points and seven waves a SIMD the compiler keeps 2 VGPRs in scratch (12
// bytes a lane; 4 to 10 in the SPARSE and Gaussian forms); six waves without
// scratch are slower: 4M plume 256^3 3.49 / 3.61, ring of 500k 96^3 3.07 / 3.11.
template <int KERNEL, bool SEGMENT, typename TO, bool WIDE, int T, bool SPARSE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(T == 8 || KERNEL == PPPM_KERNEL_GAUSSIAN ? 7 : 8)))
k_m2p_near(const float4* __restrict__ epos, const float4* __restrict__ eoth, const uint32_t* __restrict__ eidx, uint32_t m,
       const uint32_t* __restrict__ off, const float4* __restrict__ spos, const float4* __restrict__ somg,
       const float* __restrict__ far, uint32_t g, double invh, NearConst nc, NearSplit split, TO* __restrict__ ux,
       TO* __restrict__ uy, TO* __restrict__ uz, uint32_t u_stride, const uint32_t* __restrict__ tperm) {
    static_assert(T == 1 || T == 2 || T == 4 || T == 8, "group_min, group_max and transpose_reduce");
    __shared__ float4 ring[4][2][128];
    const int lane0 = threadIdx.x & 63, w = threadIdx.x >> 6;
    // groups of 256 consecutive workgroups per XCD, so each L2 serves one run
    // of points whose boxes share most of their hash rows
    const uint32_t wg = xcd_group<256>(blockIdx.x, gridDim.x);
    const uint32_t t0 = (wg * 4 + w) * T;
    if (t0 >= m) return;  // the whole wave leaves together; no block barriers below
    const uint32_t slot = t0 + lane0 % T;
    const bool tv = slot < m;
    // evaluation slot -> sorted point; a slot past the end takes the first
    // slot's point and is neither in a group nor stored
    const uint32_t t = tperm ? tperm[tv ? slot : t0] : (tv ? slot : t0);
    const float4 a0 = epos[t];
    const int gi = (int)g;
    const size_t G = (size_t)g * g * g;
    auto lanef = [](float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
    const double rb = (double)nc.rbox;
    const float rbox = nc.rbox;
    // the points' y and z (and other ends), in scalar registers
    constexpr int TS = SEGMENT ? T : 1;
    float py[T], pz[T], qx[TS], qy[TS], qz[TS];
#pragma unroll
    for (int p = 0; p < T; p++) {
        py[p] = lanef(a0.y, p);
        pz[p] = lanef(a0.z, p);
    }
    if (SEGMENT) {
        const float4 bp = eoth[t];
#pragma unroll
        for (int p = 0; p < TS; p++) {
            qx[p] = lanef(bp.x, p);
            qy[p] = lanef(bp.y, p);
            qz[p] = lanef(bp.z, p);
        }
    }
    const uint32_t nsrc = off[G];
    int sz = T;
    for (int s0 = 0; s0 < T; s0 += sz) {
        // group [s0, s0 + sz) of the points; after the first, aligned powers
        // of two
        if (s0 > 0) sz = s0 & -s0;
        // opaque in every pass, so that nothing of a pass is kept in registers
        // for the next (there is one pass in most waves)
        float4 a = a0;
        int lane = lane0;
        __asm__ volatile("" : "+v"(a.x), "+v"(a.y), "+v"(a.z), "+v"(lane));
        const int ti = lane % T, sj = lane / T;
        // ---- union of the group's boxes -> scanned cell range (wave-uniform).
        // A NaN coordinate stays out of the union (all-NaN: an empty range).
        // Lane j < 6 computes one axis's bounds (j = axis: lower, 3 + axis:
        // upper): the cell range and the staging bound.  Every vortex the box
        // test can accept lies strictly inside the staging bounds: the test
        // keeps fl(|p - s|) <= rbox, so |p - s| <= rbox (1 + 2^-23) exactly, and
        // s > min - rbox (1 + 2^-21) >= lo, with lo that bound rounded down (hi:
        // max + rbox (1 + 2^-21) rounded up).
        int xlo, ylo, zlo, xhi, yhi, zhi, ny_, nrows;
        float lox, loy, loz, hix, hiy, hiz;
        for (;;) {
            const bool in = tv && ti >= s0 && ti < s0 + sz;
            const bool okx = in && a.x == a.x, oky = in && a.y == a.y, okz = in && a.z == a.z;
            const float mnx = group_min<T>(okx ? a.x : 3.0e38f), mny = group_min<T>(oky ? a.y : 3.0e38f),
                        mnz = group_min<T>(okz ? a.z : 3.0e38f);
            const float mxx = group_max<T>(okx ? a.x : -3.0e38f), mxy = group_max<T>(oky ? a.y : -3.0e38f),
                        mxz = group_max<T>(okz ? a.z : -3.0e38f);
            const int bj = lane < 6 ? lane : 0;
            const bool bup = bj >= 3;
            const int bax = bup ? bj - 3 : bj;
            const float bvv = bax == 0 ? (bup ? mxx : mnx) : bax == 1 ? (bup ? mxy : mny) : (bup ? mxz : mnz);
            const int cbnd = near_cell_bound(bvv, rb, invh, gi, bup);
            xlo = __builtin_amdgcn_readlane(cbnd, 0);
            ylo = __builtin_amdgcn_readlane(cbnd, 1);
            zlo = __builtin_amdgcn_readlane(cbnd, 2);
            xhi = __builtin_amdgcn_readlane(cbnd, 3);
            yhi = __builtin_amdgcn_readlane(cbnd, 4);
            zhi = __builtin_amdgcn_readlane(cbnd, 5);
            ny_ = yhi - ylo + 1;
            nrows = (xlo <= xhi && ylo <= yhi && zlo <= zhi) ? (zhi - zlo + 1) * ny_ : 0;
            if (T > 1 && sz > 1 && nrows * (xhi - xlo + 1) > split.vlim) {
                bool pays = true;
                if constexpr (SPARSE) {
                    // the boxes of the two halves, in lanes 0 .. 5 and 6 .. 11
                    const int hj = lane < 12 ? lane % 6 : 0, p0 = s0 + (lane < 6 ? 0 : sz >> 1), p1 = p0 + (sz >> 1);
                    float hv = hj < 3 ? 3.0e38f : -3.0e38f;
                    for (int p = 0; p < T; p++) {
                        const float v = hj % 3 == 0 ? lanef(a.x, p) : hj % 3 == 1 ? lanef(a.y, p) : lanef(a.z, p);
                        if (p >= p0 && p < p1 && v == v) hv = hj < 3 ? fminf(hv, v) : fmaxf(hv, v);
                    }
                    const int hb = near_cell_bound(hv, rb, invh, gi, hj >= 3);
                    // vortices a cell: the mean, or more in the first point's row
                    const int cy = min(max(cell_of(lanef(a.y, s0), invh), 0), gi - 1),
                              cz = min(max(cell_of(lanef(a.z, s0), invh), 0), gi - 1);
                    const uint32_t row0 = __builtin_amdgcn_readfirstlane(((uint32_t)cz * g + (uint32_t)cy) * g);
                    const float here = (float)(off[row0 + xhi + 1] - off[row0 + xlo]);
                    const float cell = split.vortex * fmaxf(split.mean, here / (float)(xhi - xlo + 1));
                    auto cost = [&](int nr, int nx_) { return split.row * (float)nr + cell * ((float)nr * (float)nx_); };
                    auto half_cost = [&](int l) {
                        const int nx_ = __builtin_amdgcn_readlane(hb, l + 3) - __builtin_amdgcn_readlane(hb, l) + 1,
                                  ny = __builtin_amdgcn_readlane(hb, l + 4) - __builtin_amdgcn_readlane(hb, l + 1) + 1,
                                  nz = __builtin_amdgcn_readlane(hb, l + 5) - __builtin_amdgcn_readlane(hb, l + 2) + 1;
                        return nx_ > 0 && ny > 0 && nz > 0 ? cost(ny * nz, nx_) : 0.f;
                    };
                    const float halves = half_cost(0) + half_cost(6) + split.pass;
                    const float singles = (float)sz * (cost(split.edge * split.edge, split.edge) + split.pass) - split.pass;
                    pays = __builtin_amdgcn_readfirstlane(fminf(halves, singles) < cost(nrows, xhi - xlo + 1));
                }
                if (pays) {
                    sz >>= 1;
                    continue;
                }
            }
            const float sbnd = near_stage_bound(bvv, rb * (1.0 + 0x1p-21), bup);
            lox = lanef(sbnd, 0);
            loy = lanef(sbnd, 1);
            loz = lanef(sbnd, 2);
            hix = lanef(sbnd, 3);
            hiy = lanef(sbnd, 4);
            hiz = lanef(sbnd, 5);
            break;
        }
        // row r -> (z, y) = (r / ny_, r % ny_) through a float reciprocal
        // (within 1 ulp): exact while r < 2^21 (nrows <= g^2 <= 2^20)
        const float inv_ny = __builtin_amdgcn_rcpf((float)max(ny_, 1));
        // x of the points, -inf outside the group: no source passes their box
        // test (a lane past the window's end holds +inf in all coordinates)
        float px[T], vx[T], vy[T], vz[T];
#pragma unroll
        for (int p = 0; p < T; p++) {
            px[p] = p >= s0 && p < s0 + sz ? lanef(a.x, p) : -__builtin_inff();
            vx[p] = vy[p] = vz[p] = 0.f;
        }
        // Evaluate the window [wh, wh + n) of the ring (wh is 0 or 64).
        auto evaluate = [&](uint32_t wh, uint32_t n) {
            float4 s = ring[w][0][wh + lane];
            const float4 o = ring[w][1][wh + lane];
            if ((uint32_t)lane >= n) s.x = s.y = s.z = __builtin_inff();
#pragma unroll
            for (int p = 0; p < T; p++) {
                const float dx = px[p] - s.x, dy = py[p] - s.y, dz = pz[p] - s.z;
                // |d|inf <= rbox as one max3 of absolute values
                bool acc = fmaxf(fmaxf(fabsf(dx), fabsf(dy)), fabsf(dz)) <= rbox;
                if (SEGMENT) {
                    const int ps = SEGMENT ? p : 0;
                    const float ex = qx[ps] - s.x, ey = qy[ps] - s.y, ez = qz[ps] - s.z;
                    acc = acc && ex * ex + ey * ey + ez * ez >= 1e-24f;
                }
                if (acc) {
                    // r^2 carries 1e-24, so a coincident pair has a finite
                    // coefficient and adds omega x 0 = 0 (the reference zeroes
                    // r < 1e-12) with no compare per pair
                    const float r2 = fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, 1e-24f)));
                    const float cf =
                        KERNEL == PPPM_KERNEL_GAUSSIAN ? coeff_gaussian(r2, nc) : coeff_expcubic_4pi(r2, nc);
                    vx[p] += (o.y * dz - o.z * dy) * cf;
                    vy[p] += (o.z * dx - o.x * dz) * cf;
                    vz[p] += (o.x * dy - o.y * dx) * cf;
                }
            }
            // the next staging may overwrite these entries
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        };
        // ring state (wave-uniform): window head (0 or 64) and entries held
        uint32_t qh = 0, qn = 0;
        for (int r0 = 0; r0 < nrows; r0 += 64) {
            // lane l holds the vortex range [lp0, lp1) of row r0 + l (z outer,
            // y inner), loaded in one pass
            uint32_t lp0 = 0, lp1 = 0;
            if (r0 + lane < nrows) {
                const int r = r0 + lane;
                const int rz = (int)(((float)r + 0.5f) * inv_ny);
                const uint32_t kk = (uint32_t)(zlo + rz), jj = (uint32_t)(ylo + r - rz * ny_);
                const uint32_t rowc = (kk * g + jj) * g;
                lp0 = off[rowc + xlo];
                lp1 = min(off[rowc + xhi + 1], nsrc);
            }
            const int rn = min(64, nrows - r0);
            // The rows are packed into one stream of vortices: chunk c holds
            // stream positions 64 c .. 64 c + 63 across row boundaries.  pre
            // is a row's first stream position (exclusive prefix of the row
            // lengths), roff maps stream position to vortex index.
            const uint32_t len = lp1 > lp0 ? lp1 - lp0 : 0u;
            const uint32_t incl = wave_inclusive_scan(len);
            const uint32_t pre = incl - len, roff = lp0 - pre;
            const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
            // vortex index of this lane's position in the chunk at S0; rcur
            // (wave-uniform) is a row at or before the one holding S0 and is
            // advanced to the last row starting at or before S0 + 64
            auto locate = [&](uint32_t S0, int& rcur) {
                const uint32_t S = S0 + (uint32_t)lane;
                uint32_t mo = __builtin_amdgcn_readlane(roff, rcur);
                int rnext = rcur;
                for (int rr = rcur + 1; rr < rn; rr++) {
                    const uint32_t p = __builtin_amdgcn_readlane(pre, rr);
                    if (p > S0 + 64) break;
                    rnext = rr;
                    if (S >= p) mo = __builtin_amdgcn_readlane(roff, rr);
                }
                rcur = rnext;
                return S + mo;
            };
            int rc = 0;
            // The next chunk is loaded into registers while this one is
            // staged.  Slots past the end of the stream (pin false) read
            // vortex 0 and are not staged.
            float4 pp = make_float4(0.f, 0.f, 0.f, 0.f), po = pp;
            float lxl = __builtin_inff();
            auto load = [&](uint32_t S0) {
                const uint32_t vi = locate(S0, rc);
                const bool pin = S0 + (uint32_t)lane < total;
                lxl = pin ? lox : __builtin_inff();  // a slot past the end fails the filter
                const uint32_t v = pin ? vi : 0u;
                if (WIDE) {
                    pp = spos[v];
                    po = somg[v];
                } else {
                    const uint32_t ob = v << 4;
                    pp = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(spos) + ob);
                    po = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(somg) + ob);
                }
            };
            if (total > 0) load(0u);
            for (uint32_t S0 = 0; S0 < total; S0 += 64) {
                // Stage only the vortices inside the staging bounds on every
                // axis: the lane masks of the six compares (ordered: NaN
                // fails) ANDed on the scalar unit, then the mask as the
                // predicate
                const uint64_t bal =
                    __builtin_amdgcn_fcmpf(pp.x, lxl, 2) & __builtin_amdgcn_fcmpf(pp.x, hix, 4) &
                    __builtin_amdgcn_fcmpf(pp.y, loy, 2) & __builtin_amdgcn_fcmpf(pp.y, hiy, 4) &
                    __builtin_amdgcn_fcmpf(pp.z, loz, 2) & __builtin_amdgcn_fcmpf(pp.z, hiz, 4);
                const bool use = __builtin_amdgcn_inverse_ballot_w64(bal);
                // ring slot: the head plus the kept lanes below this one
                const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32),
                                                              __builtin_amdgcn_mbcnt_lo((uint32_t)bal, qh + qn));
                if (use) {
                    const uint32_t e = at & 127u;
                    ring[w][0][e] = pp;
                    ring[w][1][e] = po;
                }
                qn += (uint32_t)__popcll(bal);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if (S0 + 64 < total) load(S0 + 64);
                // a full window: evaluate it and move the head to the other
                if (qn >= 64) {
                    evaluate(qh, 64u);
                    qh ^= 64u;
                    qn -= 64u;
                }
            }
        }
        if (qn > 0) evaluate(qh, qn);  // the last, partial window
        // ---- lane l: point l % T.  1 / (4 pi) is applied here, once a point
        // (the Gaussian coefficient holds it)
        float rx = transpose_reduce<T>(vx, lane), ry = transpose_reduce<T>(vy, lane),
              rz = transpose_reduce<T>(vz, lane);
        if (KERNEL != PPPM_KERNEL_GAUSSIAN) {
            rx *= nc.inv4pi;
            ry *= nc.inv4pi;
            rz *= nc.inv4pi;
        }
        // ---- M2P: the point's 8 interpolation corners, corner sj on slice sj
        // (the weights and validity of k_m2p_points), into the sums
        if (sj < 8 && tv) {
            const int i = cell_of(a.x, invh), j = cell_of(a.y, invh), k = cell_of(a.z, invh);
            const bool fin = a.x == a.x && a.y == a.y && a.z == a.z;
            if (fin && i >= 0 && i < gi && j >= 0 && j < gi && k >= 0 && k < gi) {
                const double xh = (double)a.x * invh - 0.5, yh = (double)a.y * invh - 0.5,
                             zh = (double)a.z * invh - 0.5;
                const int i0 = (int)floor(xh), j0 = (int)floor(yh), k0 = (int)floor(zh);
                const float fx = (float)(xh - i0), fy = (float)(yh - j0), fz = (float)(zh - k0);
                const int a2 = sj & 1, b2 = (sj >> 1) & 1, c2 = sj >> 2;
                const bool ok =
                    (a2 ? i0 + 1 < gi : i0 >= 0) && (b2 ? j0 + 1 < gi : j0 >= 0) && (c2 ? k0 + 1 < gi : k0 >= 0);
                if (ok) {
                    const uint32_t q = (((uint32_t)k0 + (uint32_t)c2) * g + (uint32_t)j0 + (uint32_t)b2) * g +
                                       (uint32_t)i0 + (uint32_t)a2;
                    const float wgt = (a2 ? fx : 1.f - fx) * (b2 ? fy : 1.f - fy) * (c2 ? fz : 1.f - fz);
                    rx = fmaf(wgt, far[q], rx);
                    ry = fmaf(wgt, far[G + q], ry);
                    rz = fmaf(wgt, far[2 * G + q], rz);
                }
            }
        }
        // ---- the lanes of a point (a fixed order)
        if (T == 1) {
            rx += dpp_mov<0xB1>(rx);
            ry += dpp_mov<0xB1>(ry);
            rz += dpp_mov<0xB1>(rz);
        }
        if (T <= 2) {
            rx += dpp_mov<0x4E>(rx);
            ry += dpp_mov<0x4E>(ry);
            rz += dpp_mov<0x4E>(rz);
        }
        if (T <= 4) {
            rx += dpp_mov<0x124>(rx);
            ry += dpp_mov<0x124>(ry);
            rz += dpp_mov<0x124>(rz);
        }
        rx += dpp_mov<0x128>(rx);
        ry += dpp_mov<0x128>(ry);
        rz += dpp_mov<0x128>(rz);
        for (int o = 16; o < 64; o <<= 1) {
            rx += __shfl_xor(rx, o, 64);
            ry += __shfl_xor(ry, o, 64);
            rz += __shfl_xor(rz, o, 64);
        }
        if (lane < T && tv && lane >= s0 && lane < s0 + sz) {
            const uint32_t dt = eidx[t];
            if (dt < m) {
                const size_t dst = (size_t)dt * u_stride;
                ux[dst] = (TO)rx;
                uy[dst] = (TO)ry;
                uz[dst] = (TO)rz;
            }
        }
    }
}

// two rounds of resident waves (256 CUs x 28) of eight points
constexpr uint32_t kNearMany = 8u * 2u * 256u * 28u;

template <int KERNEL, bool SEGMENT, bool WIDE, int T>
static void launch_near_sized(const NearArgs& a, const NearConst& nc, hipStream_t st) {
    // A group's union box stays up to five times a single point's cells (a box
    // of 2K + 1 cells, one more where it straddles).  Limits of 2, 3, 5, 7 and
    // 12 boxes: 0.71, 0.55, 0.37, 0.36 and 0.37 ms at 700,001 uniform vortices
    // on 96^3; 16.3, 15.5 at the 8M plume (2, 3), then unchanged; 65,536
    // uniform on 32^3: 0.073 ms at 5, 0.083 at 7.
    NearSplit split;
    const int edge = 2 * a.K + 2;
    split.vlim = 5 * edge * edge * edge;
    split.pass = 200.f;
    split.row = 8.f;
    split.vortex = 2.5f;
    split.mean = (float)(a.nsrc / ((double)a.g * a.g * a.g));
    split.edge = edge;
    auto run = [&](auto to, auto sparse) {
        using TO = decltype(to);
        hipLaunchKernelGGL((k_m2p_near<KERNEL, SEGMENT, TO, WIDE, T, decltype(sparse)::value>),
                           dim3(div_up(div_up(a.m, T), 4)), dim3(256), 0, st, a.epos, a.eoth, a.eidx, a.m, a.off, a.spos,
                           a.somg, a.far, a.g, a.invh, nc, split, (TO*)a.ux, (TO*)a.uy, (TO*)a.uz, a.u_stride, a.tperm);
    };
    // Sparse: groups stretch beyond vlim along a row, not only around its end.
    // Weighing costs takes 3 to 5% of the dense scenes' time in registers (plume
    // of 8M on 256^3 11.6 / 11.9 ms, of 1/4 vortex a cell 3.75 / 3.87).
    const float line = edge < 6 ? 7.2f / (float)(edge * edge) : 0.2f;
    const bool sparse = T > 1 && split.mean < line;
    if (a.u_dtype == PPPM_F64) sparse ? run(double(), std::bool_constant<(T > 1)>()) : run(double(), std::false_type());
    else sparse ? run(float(), std::bool_constant<(T > 1)>()) : run(float(), std::false_type());
}
template <int KERNEL, bool SEGMENT>
static void launch_near(const NearArgs& a, const NearConst& nc, hipStream_t st) {
    // Eight points a wave once that is two rounds of resident waves; below, four
    // keep more waves in flight (10,007 points: 0.031 against 0.050 ms; 65,536:
    // 0.073 against 0.079; 1M: 1.57 against 1.43), and two or one where four
    // leave SIMDs without a wave (us, four / two / one: 306 points 26 / 14 / 10,
    // 2,000 25 / 19 / 10, 20,000 35 / 30, 65,536 67 / 74).  The Gaussian core's costly
    // pairs ask for small unions of boxes: four points however many (2M plume on
    // 128^3 8.74 against 9.14 ms, 133,613 ring on 160^3 0.43 against 0.59), but
    // for K = 0, whose waves are mostly set-up.
    const bool wide = a.nsrc >= (1u << 28);
    auto run = [&](auto t) {
        if (wide) launch_near_sized<KERNEL, SEGMENT, true, decltype(t)::value>(a, nc, st);
        else launch_near_sized<KERNEL, SEGMENT, false, decltype(t)::value>(a, nc, st);
    };
    if (a.m > kNearMany && (KERNEL != PPPM_KERNEL_GAUSSIAN || a.K < 1)) run(std::integral_constant<int, 8>());
    else if (a.m > 3u << 12) run(std::integral_constant<int, 4>());
    else if (a.m > 1u << 11) run(std::integral_constant<int, 2>());
    else run(std::integral_constant<int, 1>());
}

template <int KERNEL, bool WIDE>
static void launch_pot_sized(const NearArgs& a, const NearConst& nc, hipStream_t st) {
    const uint32_t waves = div_up(a.m, kNearTI);
    dim3 grid(div_up(waves, 4)), blk(256);
    if (a.u_dtype == PPPM_F64)
        hipLaunchKernelGGL((k_pot_near<KERNEL, double, WIDE>), grid, blk, 0, st, a.epos, a.eidx, a.m, a.off, a.spos, a.somg, a.far, a.g, a.K, a.invh, nc, (double*)a.ux, (double*)a.uy,
                           (double*)a.uz, a.u_stride, a.tperm);
    else
        hipLaunchKernelGGL((k_pot_near<KERNEL, float, WIDE>), grid, blk, 0, st, a.epos, a.eidx, a.m, a.off, a.spos, a.somg, a.far, a.g, a.K, a.invh, nc, (float*)a.ux, (float*)a.uy,
                           (float*)a.uz, a.u_stride, a.tperm);
}
template <int KERNEL>
static void launch_pot(const NearArgs& a, const NearConst& nc, hipStream_t st) {
    if (a.nsrc >= (1u << 28)) launch_pot_sized<KERNEL, true>(a, nc, st);
    else launch_pot_sized<KERNEL, false>(a, nc, st);
}

// ---- evaluation order in super-blocks ------------------------------------
// The sorted points (cell-major, octant order within each cell) are
// renumbered so that consecutive evaluation slots walk one super-block of
// kSbX x kSbY x kSbZ cells (its rows z, then y, each an x segment of kSbX
// cells) before the next super-block (blocks in z, y, x order).  Consecutive
// clusters go to one XCD in groups of 256 workgroups, about 4,096 points of
// k_pot_near, and in this order such a run is a compact region whose hash rows
// fit that XCD's L2 (17.4 -> 14.5 ms at 8M/256^3 for waves of four points that
// do not split their union box; blocks of 4x4x4 and 16x4x4 the same, 8x2x2
// 16.8 ms, 8x8x8 17.9 ms).
constexpr uint32_t kSbX = 8, kSbY = 4, kSbZ = 4;

SbGeom sb_geom(uint32_t g) {
    SbGeom s;
    s.g = g;
    s.nX = (g + kSbX - 1) / kSbX;
    s.nY = (g + kSbY - 1) / kSbY;
    s.nslots = s.nX * s.nY * ((g + kSbZ - 1) / kSbZ) * kSbY * kSbZ;
    return s;
}

// slot of a cell: its x segment's place in super-block order
__device__ inline uint32_t sb_slot(uint32_t cell, const SbGeom& s) {
    const uint32_t x = cell % s.g, y = (cell / s.g) % s.g, z = cell / (s.g * s.g);
    return (((z / kSbZ) * s.nY + y / kSbY) * s.nX + x / kSbX) * (kSbY * kSbZ) + (z % kSbZ) * kSbY + y % kSbY;
}

// The points of one slot (one x segment of one row) are consecutive in the
// sort: start[] and len[] (zero beforehand) get the first of them and one
// past the last.
__global__ void __launch_bounds__(256) k_sb_bounds(const uint32_t* __restrict__ keys, uint32_t osh, uint32_t n,
                                                   SbGeom s, uint32_t* __restrict__ start, uint32_t* __restrict__ len) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const uint32_t sl = sb_slot(keys[p] >> osh, s);
    if (p == 0 || sb_slot(keys[p - 1] >> osh, s) != sl) start[sl] = p;
    if (p + 1 == n || sb_slot(keys[p + 1] >> osh, s) != sl) len[sl] = p + 1;
}

// one past the last -> count
__global__ void __launch_bounds__(256) k_sb_len(const uint32_t* __restrict__ start, uint32_t* __restrict__ len,
                                                uint32_t nslots) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nslots) len[i] -= start[i];
}

// slot of sorted point p: its slot's first slot plus its place in the slot
__global__ void __launch_bounds__(256) k_sb_perm(const uint32_t* __restrict__ keys, uint32_t osh, uint32_t n,
                                                 SbGeom s, const uint32_t* __restrict__ start,
                                                 const uint32_t* __restrict__ pre, uint32_t* __restrict__ tperm) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const uint32_t sl = sb_slot(keys[p] >> osh, s);
    tperm[pre[sl] + (p - start[sl])] = p;
}

pppm_status launch_sb_order(const uint32_t* keys, uint32_t osh, uint32_t n, const SbGeom& s, SbBuffers b,
                            uint32_t* tperm, hipStream_t st) {
    if (n == 0) return PPPM_OK;
    pppm_status r = launch_fill_u32(b.start, s.nslots, 0u, st);
    if (r == PPPM_OK) r = launch_fill_u32(b.len, s.nslots, 0u, st);
    if (r != PPPM_OK) return r;
    hipLaunchKernelGGL(k_sb_bounds, dim3(div_up(n, 256)), dim3(256), 0, st, keys, osh, n, s, b.start, b.len);
    PPPM_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_sb_len, dim3(div_up(s.nslots, 256)), dim3(256), 0, st, b.start, b.len, s.nslots);
    PPPM_LAUNCH_CHECK();
    r = exclusive_scan_u32(b.len, s.nslots, b.pre, b.scratch, st);
    if (r != PPPM_OK) return r;
    hipLaunchKernelGGL(k_sb_perm, dim3(div_up(n, 256)), dim3(256), 0, st, keys, osh, n, s, b.start, b.pre, tperm);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

// Evaluation order within each hash cell: by octant of the cell (the halves
// of x, y and z), original order within an octant, so the points of a
// cluster share a half-cell and their union box is smaller.  ks: sorted cell
// keys, pos: sorted origin-shifted points.  A thread ranks its point among
// its cell's segment; segments longer than kOctMax keep their order (the
// ranking is quadratic in the segment length).
constexpr uint32_t kOctMax = 256;

__device__ inline uint32_t octant_of(float4 p, float invh) {
    const float fx = p.x * invh, fy = p.y * invh, fz = p.z * invh;
    return (uint32_t)(fx - floorf(fx) >= 0.5f) | ((uint32_t)(fy - floorf(fy) >= 0.5f) << 1) |
           ((uint32_t)(fz - floorf(fz) >= 0.5f) << 2);
}

__global__ void __launch_bounds__(256) k_octant_order(const uint32_t* __restrict__ ks, const float4* __restrict__ pos,
                                                      uint32_t n, float invh, uint32_t* __restrict__ perm) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const uint32_t k = ks[p];
    uint32_t s = p, e = p + 1;
    while (s > 0 && ks[s - 1] == k && p - s < kOctMax) s--;
    while (e < n && ks[e] == k && e - p <= kOctMax) e++;
    if (e - s > kOctMax || (s > 0 && ks[s - 1] == k)) {
        perm[p] = p;  // long segment: original order
        return;
    }
    const uint32_t o = octant_of(pos[p], invh);
    uint32_t r = 0;
    for (uint32_t q = s; q < e; q++) {
        const uint32_t oq = octant_of(pos[q], invh);
        r += (oq < o || (oq == o && q < p)) ? 1u : 0u;
    }
    perm[s + r] = p;
}

pppm_status launch_octant_order(const uint32_t* ks, const float4* pos, uint32_t n, double invh, uint32_t* perm,
                                hipStream_t st) {
    if (n == 0) return PPPM_OK;
    hipLaunchKernelGGL(k_octant_order, dim3(div_up(n, 256)), dim3(256), 0, st, ks, pos, n, (float)invh, perm);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

// largest float f with (double)f < x (x > 0; returns -1 otherwise)
static float float_below(double x) {
    if (!(x > 0)) return -1.0f;
    float f = (float)x;
    while ((double)f >= x) f = nextafterf(f, 0.0f);
    while ((double)nextafterf(f, 3.4e38f) < x) f = nextafterf(f, 3.4e38f);
    return f;
}

pppm_status launch_m2p_near(const NearArgs& a, hipStream_t st) {
    if (a.m == 0) return PPPM_OK;
    NearConst nc;
    const double h = 1.0 / a.invh;
    nc.rbox = float_below(((double)a.K + 0.5) / a.invh);
    nc.inv_a = (float)(1.0 / a.core_a);
    nc.inv_a3 = (float)(1.0 / (a.core_a * a.core_a * a.core_a));
    nc.inv4pi = (float)(1.0 / kRefFourPi);
    nc.kexp2 = (float)(-1.4426950408889634 / (a.core_a * a.core_a * a.core_a));
    nc.r3_series = (float)(0.1 * a.core_a * a.core_a * a.core_a);
    {
        const double c[5] = {1.0, -0.5, 1.0 / 6.0, -1.0 / 24.0, 1.0 / 120.0};
        for (int k = 0; k < 5; k++) nc.sc[k] = (float)(c[k] / (a.core_a * a.core_a * a.core_a));
    }
    (void)h;
    if (a.K < 0) {
        // vortex-in-cell: M2P alone writes the outputs
        dim3 grid(div_up(a.m, 256)), blk(256);
        if (a.u_dtype == PPPM_F64)
            hipLaunchKernelGGL(k_m2p_points<double>, grid, blk, 0, st, a.epos, a.eidx, a.m, a.far, a.g, a.invh,
                               (double*)a.ux, (double*)a.uy, (double*)a.uz, a.u_stride);
        else
            hipLaunchKernelGGL(k_m2p_points<float>, grid, blk, 0, st, a.epos, a.eidx, a.m, a.far, a.g, a.invh,
                               (float*)a.ux, (float*)a.uy, (float*)a.uz, a.u_stride);
        PPPM_LAUNCH_CHECK();
        return PPPM_OK;
    }
    const bool seg = a.eoth != nullptr;
    if (a.kernel == kNearPotGrad || a.kernel == kNearPotScalar) {
        // potential-flow solver: a = core_a (absolute), G direction in pot_g
        const double ca = a.core_a;
        nc.pa = (float)ca;
        nc.pc = (float)(a.kernel == kNearPotGrad ? 1.0 / (kRefFourPi * ca * ca * ca) : 1.0 / (kRefFourPi * ca));
        nc.pg = (float)a.pot_g;
        if (seg) return PPPM_ERR_INVALID;
        if (a.kernel == kNearPotGrad) launch_pot<kNearPotGrad>(a, nc, st);
        else launch_pot<kNearPotScalar>(a, nc, st);
        PPPM_LAUNCH_CHECK();
        return PPPM_OK;
    }
    if (a.kernel == PPPM_KERNEL_GAUSSIAN) {
        if (seg) launch_near<PPPM_KERNEL_GAUSSIAN, true>(a, nc, st);
        else launch_near<PPPM_KERNEL_GAUSSIAN, false>(a, nc, st);
    } else {
        if (seg) launch_near<PPPM_KERNEL_EXPCUBIC, true>(a, nc, st);
        else launch_near<PPPM_KERNEL_EXPCUBIC, false>(a, nc, st);
    }
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

// Accepted near-field pairs (box test passed, r^2 >= 1e-24) of the evaluation
// points against the vortices, for FLOP accounting; one atomic per wave.
__global__ void __launch_bounds__(256) k_count_pairs(const float4* __restrict__ epos, uint32_t m,
                                                     const uint32_t* __restrict__ off, const float4* __restrict__ spos,
                                                     uint32_t g, int K, double invh, float rbox,
                                                     unsigned long long* __restrict__ total) {
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long cnt = 0;
    if (t < m) {
        const int gi = (int)g;
        const size_t G = (size_t)g * g * g;
        const float4 a = epos[t];
        const int i = cell_of(a.x, invh), j = cell_of(a.y, invh), k = cell_of(a.z, invh);
        const int R = K + 1;
        const uint32_t nsrc = off[G];
        const int ilo = max(i - R, 0), ihi = min(i + R, gi - 1);
        if (K >= 0 && ilo <= ihi)
            for (int kk = max(k - R, 0); kk <= min(k + R, gi - 1); kk++)
                for (int jj = max(j - R, 0); jj <= min(j + R, gi - 1); jj++) {
                    const uint32_t rowc = ((uint32_t)kk * g + (uint32_t)jj) * g;
                    const uint32_t p0 = off[rowc + ilo], p1 = min(off[rowc + ihi + 1], nsrc);
                    for (uint32_t p = p0; p < p1; p++) {
                        const float4 s = spos[p];
                        const float dx = a.x - s.x, dy = a.y - s.y, dz = a.z - s.z;
                        if (fabsf(dx) <= rbox && fabsf(dy) <= rbox && fabsf(dz) <= rbox &&
                            dx * dx + dy * dy + dz * dz >= 1e-24f)
                            cnt++;
                    }
                }
    }
    for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
    if ((threadIdx.x & 63) == 0 && cnt) atomicAdd(total, cnt);
}

pppm_status launch_count_pairs(const NearArgs& a, unsigned long long* d_total, hipStream_t st) {
    if (a.m == 0) return PPPM_OK;
    float rbox = float_below(((double)a.K + 0.5) / a.invh);
    hipLaunchKernelGGL(k_count_pairs, dim3(div_up(a.m, 256)), dim3(256), 0, st, a.epos, a.m, a.off, a.spos, a.g, a.K,
                       a.invh, rbox, d_total);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

}  // namespace pppm
