// Curl of the stream function fused with the far-field correction
// (GPU_kernel.cu:1750-1805 compute_curl_kernel, 2487-2564 Step1, 1976-2001
// compute_diag_Psi_kernel, 2566-2630 subtract_diagonal_grid_kernel, host
// orchestration 2634-2734):
//   far[c] = curl(psi)[c]
//          - sum_{D != 0, |D|inf <= K, c+D in grid} dir[D] x (w[c+D] h^3)
//          - curl(0.250580605913965 h^2 w)[c]
// with clamp-to-edge central differences.  The reference's D2H/H2D stash of
// grid_U and its per-call host table upload are gone: dir[] is built once per
// (K, h) and read with wave-uniform (scalar) loads.
#include "pppm_internal.hpp"
#include <algorithm>
#include <type_traits>

namespace pppm {

// What each plane of the grid vorticity w adds to the sum is formed once, when
// the plane arrives, for the 2K+1 output planes it reaches (their sums sit in
// registers while a workgroup marches along z), so LDS holds one plane and the
// next.  dir[D] has component a odd in D_a and even in the other two (a central
// difference along a of 1/(4 pi |r|)), so the (2K+1)^2 neighbours of a plane are
// folded to sums and differences over +-y and +-x first and the planes at +-dz
// share their products.
// No sum may hold more than differences of w: dir is odd, so a mean of w over
// the neighbourhood cancels, and would do so in FP32 after rounding.  Along x
// and y the differences are formed first.  Along z the planes meet only in the
// output's sum, so dir_2 takes w less a base value of the plane (the mean of
// the pair's four cells at +-1 in y, rounding nothing where w is smooth), and what the
// bases would have added, dir_2's plane sums C_dz times their differences
// over +-dz, joins at the end (C follows dir in the table).  RMS error against 64
// bits, K = 2, relative to that of one FP32 sum over the pairs w[c+D] - w[c-D]:
// 0.63 for white noise, 0.14 for 1 + 2% ripple, 0.3 for a sine over the box;
// with sums in place of the differences 0.7, 9.9 and 1.6.
// The curl of the diagonal term (face neighbours, clamped to the edge) has its
// own sums, joined in FP64.  A thread owns two cells along x.  The curl of psi
// reads global memory at the end of a plane.  Bound by vector issue and the
// loads of psi; us a launch, sum over pairs with a ring of 2K+1 planes -> here,
// K = 2: 32^3 (FP64 psi) 80 -> 18, 64^3 85 -> 21, 96^3 89 -> 45, 128^3 101 -> 69,
// 256^3 503 -> 336 (FP32 psi 467 -> 302); at 128^3 K = 1 51 -> 48, K = 0 83 -> 32.
// Held to 3 or 4 waves per SIMD the compiler spills.
constexpr int kCfThreads = 256;

template <typename TP, typename TC, int K, int TX, bool EVEN>
__global__ void __launch_bounds__(kCfThreads) k_curl_far(const TP* __restrict__ psi, const float* __restrict__ wg,
                                                         float* __restrict__ far, const float* __restrict__ dir,
                                                         uint32_t g, float h3, TC half_invh, float cdiag_half_invh,
                                                         int zc) {
    constexpr bool kSum = K >= 0;           // else the grid velocity alone
    constexpr int KC = K < 1 ? 1 : K;       // reach of the sum with the diagonal term
    constexpr int KE = KC + (KC & 1);       // x halo, even
    constexpr int W = 2 * KC + 1;
    constexpr int TXT = TX / 2, TY = kCfThreads / TXT;
    constexpr int LX = TX + 2 * KE, LY = TY + 2 * KC, PL = LX * LY, NV = 2 + 2 * KE;
    constexpr int NL = (3 * PL + kCfThreads - 1) / kCfThreads;
    __shared__ float2 pl[2][kSum ? 3 * PL / 2 : 1];
    const int gi = (int)g, tid = threadIdx.x;
    const size_t G = (size_t)g * g * g;
    const int tilesx = (gi + TX - 1) / TX;
    const int bx = blockIdx.x % tilesx, by = blockIdx.x / tilesx;
    const int z0 = blockIdx.y * zc, z1 = min(z0 + zc, gi);
    const int tx = tid % TXT, ty = tid / TXT;
    const int i = bx * TX + 2 * tx, j = by * TY + ty;
    const int gx0 = bx * TX - KE, gy0 = by * TY - KC;
    auto at = [&](int a, int b, int c) { return ((size_t)c * g + (size_t)b) * g + (size_t)a; };

    // by slot: the sums of the output planes in flight, their diagonal terms
    // (over 0.5 c h), and of the planes of w the bases and the own x and y
    // components
    float acc[W][3][2], dg[W][3][2], bs[W][2], own[W][2][2];
#pragma unroll
    for (int s = 0; s < W; s++) {
        bs[s][0] = bs[s][1] = 0.f;
#pragma unroll
        for (int c = 0; c < 3; c++) acc[s][c][0] = acc[s][c][1] = dg[s][c][0] = dg[s][c][1] = 0.f;
        own[s][0][0] = own[s][0][1] = own[s][1][0] = own[s][1][1] = 0.f;
    }

    // plane p of w into registers (zero outside the grid), then LDS
    float ld[NL];
    auto fetch = [&](int p) {
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int q = tid + kCfThreads * u, c = q / PL, r = q - c * PL, yy = r / LX, xx = r - yy * LX;
            const int ii = gx0 + xx, jj = gy0 + yy;
            const bool ok = c < 3 && p >= 0 && p < gi && ii >= 0 && ii < gi && jj >= 0 && jj < gi;
            ld[u] = ok ? wg[c * G + at(ii, jj, p)] : 0.f;
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int u = 0; u < NL; u++)
            if (tid + kCfThreads * u < 3 * PL) reinterpret_cast<float*>(pl[buf])[tid + kCfThreads * u] = ld[u];
    };
    // component a of dir at (dx, dy, dz) >= 0
    auto coef = [&](int a, int dx, int dy, int dz) { return dir[3 * (((dz + KC) * W + dy + KC) * W + dx + KC) + a]; };
    // outputs z0 .. z1 - 1; plane p = z0 - KC + s, output p - KC complete
    // after it.  Slot of output or plane k: (k - z0 + KC) mod W.
    const int steps = (kSum ? z1 - z0 + 2 * KC : z1 - z0);
    if (kSum) {
        fetch(z0 - KC);
        store(0);
        __syncthreads();
    }
    for (int s0 = 0; s0 < steps; s0 += W) {
#pragma unroll
        for (int sj = 0; sj < W; sj++) {
            const int s = s0 + sj;
            if (s >= steps) continue;
            const int p = kSum ? z0 - KC + s : z0 + s;
            const int k = kSum ? p - KC : p;  // the output that ends here
            if (kSum) {
                if (s + 1 < steps) fetch(p + 1);
                bs[sj][0] = bs[sj][1] = 0.f;
                if (p >= 0 && p < gi) {
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        // the pair's row and those r above and below
                        float r0[NV], up[KC][NV], dn[KC][NV];
#pragma unroll
                        for (int r = 0; r <= KC; r++) {
                            const float2* a = &pl[s & 1][(c * PL + (ty + KC + r) * LX) / 2 + tx];
                            const float2* b = &pl[s & 1][(c * PL + (ty + KC - r) * LX) / 2 + tx];
#pragma unroll
                            for (int q = 0; q < NV / 2; q++) {
                                const float2 va = a[q];
                                if (r == 0) {
                                    r0[2 * q] = va.x;
                                    r0[2 * q + 1] = va.y;
                                } else {
                                    const float2 vb = b[q];
                                    up[r ? r - 1 : 0][2 * q] = va.x;
                                    up[r ? r - 1 : 0][2 * q + 1] = va.y;
                                    dn[r ? r - 1 : 0][2 * q] = vb.x;
                                    dn[r ? r - 1 : 0][2 * q + 1] = vb.y;
                                }
                            }
                        }
                        // the diagonal term's differences in the plane, clamped
#pragma unroll
                        for (int e = 0; e < 2; e++) {
                            const int m = KE + e;
                            const float o = r0[m];
                            const float xm = e == 0 && i == 0 ? o : r0[m - 1], xp = i + e == gi - 1 ? o : r0[m + 1];
                            const float ym = j == 0 ? o : dn[0][m], yp = j == gi - 1 ? o : up[0][m];
                            if (c < 2) own[sj][c][e] = o;
                            if (c == 0) dg[sj][2][e] = ym - yp;
                            if (c == 1) dg[sj][2][e] += xp - xm;
                            if (c == 2) {
                                dg[sj][0][e] = yp - ym;
                                dg[sj][1][e] = xm - xp;
                            }
                        }
                        if constexpr (K >= 1) {
                            // folded over +-y: less the base, and differences
                            float bb = 0.f;
                            if (c < 2) {
                                bb = 0.25f * ((up[0][KE] + dn[0][KE]) + (up[0][KE + 1] + dn[0][KE + 1]));
                                bs[sj][c] = bb;
                            }
                            float E[KC + 1][NV], O[KC + 1][NV];
#pragma unroll
                            for (int q = 0; q < NV; q++) {
                                E[0][q] = r0[q] - bb;
#pragma unroll
                                for (int r = 1; r <= KC; r++) {
                                    E[r][q] = (up[r - 1][q] - bb) + (dn[r - 1][q] - bb);
                                    O[r][q] = up[r - 1][q] - dn[r - 1][q];
                                }
                            }
#pragma unroll
                            for (int e = 0; e < 2; e++) {
                                const int m = KE + e;
                                // sums over the plane for |dz| = 0 .. KC: with
                                // dir_2 (even in x and y; odd in z, so none at
                                // dz = 0), dir_0 (odd in x), dir_1 (odd in y)
                                float s2[KC + 1], s0_[KC + 1], s1[KC + 1];
#pragma unroll
                                for (int dz = 0; dz <= KC; dz++) s2[dz] = s0_[dz] = s1[dz] = 0.f;
#pragma unroll
                                for (int dy = 0; dy <= KC; dy++)
#pragma unroll
                                    for (int dx = 0; dx <= KC; dx++) {
                                        const int y = dy ? dy - 1 : 0;
                                        const float ee = dx == 0 ? E[dy][m] : E[dy][m + dx] + E[dy][m - dx];
                                        // (z has no base: its differences first)
                                        const float oe = dx == 0  ? 0.f
                                                         : c < 2  ? E[dy][m + dx] - E[dy][m - dx]
                                                         : dy == 0 ? r0[m + dx] - r0[m - dx]
                                                                   : (up[y][m + dx] - up[y][m - dx]) +
                                                                         (dn[y][m + dx] - dn[y][m - dx]);
                                        const float eo = dy == 0   ? 0.f
                                                         : dx == 0 ? O[dy][m]
                                                                   : O[dy][m + dx] + O[dy][m - dx];
#pragma unroll
                                        for (int dz = 0; dz <= KC; dz++) {
                                            if (c != 2 && dz > 0) s2[dz] = fmaf(coef(2, dx, dy, dz), ee, s2[dz]);
                                            if (c != 0 && dx > 0) s0_[dz] = fmaf(coef(0, dx, dy, dz), oe, s0_[dz]);
                                            if (c != 1 && dy > 0) s1[dz] = fmaf(coef(1, dx, dy, dz), eo, s1[dz]);
                                        }
                                    }
                                // dir x w: x = d1 wz - d2 wy, y = d2 wx - d0 wz,
                                // z = d0 wy - d1 wx, of outputs p - dz (D_z = dz)
                                // and p + dz (dir_2 turned round)
#pragma unroll
                                for (int dz = 0; dz <= KC; dz++) {
                                    const int sl = (sj - dz + W) % W, sh = (sj + dz) % W;
                                    if (c == 0) {
                                        if (dz > 0) {
                                            acc[sl][1][e] += s2[dz];
                                            acc[sh][1][e] -= s2[dz];
                                            acc[sh][2][e] -= s1[dz];
                                        }
                                        acc[sl][2][e] -= s1[dz];
                                    } else if (c == 1) {
                                        if (dz > 0) {
                                            acc[sl][0][e] -= s2[dz];
                                            acc[sh][0][e] += s2[dz];
                                            acc[sh][2][e] += s0_[dz];
                                        }
                                        acc[sl][2][e] += s0_[dz];
                                    } else {
                                        acc[sl][0][e] += s1[dz];
                                        acc[sl][1][e] -= s0_[dz];
                                        if (dz > 0) {
                                            acc[sh][0][e] += s1[dz];
                                            acc[sh][1][e] -= s0_[dz];
                                        }
                                    }
                                }
                            }
                        }
                    }
                }
                // the diagonal term of output p - 1: differences along z, clamped
                {
                    const int q = p - 1, sq = (sj - 1 + W) % W, sm = (sj - 2 + W) % W;
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const float xm = q == 0 ? own[sq][0][e] : own[sm][0][e];
                        const float ym = q == 0 ? own[sq][1][e] : own[sm][1][e];
                        const float xp = q == gi - 1 ? own[sq][0][e] : own[sj][0][e];
                        const float yp = q == gi - 1 ? own[sq][1][e] : own[sj][1][e];
                        dg[sq][0][e] += ym - yp;
                        dg[sq][1][e] += xp - xm;
                    }
                }
            }
            constexpr int KO = kSum ? KC : 0;
            const int so = (sj - KO + W) % W;
            if constexpr (K >= 1) {
                // what the bases of the planes at +-dz stand for
                const float* c2 = dir + 3 * W * W * W;
#pragma unroll
                for (int dz = 1; dz <= KC; dz++) {
                    const int sl = (so - dz + W) % W, sh = (so + dz) % W;
                    const float tx_ = c2[dz - 1] * (bs[sh][0] - bs[sl][0]), ty_ = c2[dz - 1] * (bs[sh][1] - bs[sl][1]);
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        acc[so][1][e] += tx_;
                        acc[so][0][e] -= ty_;
                    }
                }
            }
            if (k >= z0 && k < z1 && i < gi && j < gi) {
                const int jm = j > 0 ? j - 1 : 0, jp = j < gi - 1 ? j + 1 : gi - 1;
                const int km = k > 0 ? k - 1 : 0, kp = k < gi - 1 ? k + 1 : gi - 1;
                const TP* Px = psi;
                const TP* Py = psi + G;
                const TP* Pz = psi + 2 * G;
                // psi at the pair's neighbours; pairs in one access when the rows
                // keep them aligned (g even)
                const bool have1 = i + 1 < gi;
                TC zp_[2], zm_[2], xp_[2], xm_[2], yzm[2], yzp[2], xzm[2], xzp[2], zx[4], yx[4];
                auto pair = [&](const TP* P, size_t t, TC* v) {
                    if (EVEN) {
                        struct alignas(2 * sizeof(TP)) P2 { TP a, b; };
                        const P2 q = *reinterpret_cast<const P2*>(P + t);
                        v[0] = (TC)q.a;
                        v[1] = (TC)q.b;
                    } else {
                        v[0] = (TC)P[t];
                        v[1] = (TC)P[t + (have1 ? 1 : 0)];
                    }
                };
                pair(Pz, at(i, jp, k), zp_);
                pair(Pz, at(i, jm, k), zm_);
                pair(Py, at(i, j, km), yzm);
                pair(Py, at(i, j, kp), yzp);
                pair(Px, at(i, j, kp), xzp);
                pair(Px, at(i, j, km), xzm);
                pair(Px, at(i, jm, k), xm_);
                pair(Px, at(i, jp, k), xp_);
                pair(Pz, at(i, j, k), zx + 1);
                pair(Py, at(i, j, k), yx + 1);
                const size_t tl = at(i > 0 ? i - 1 : 0, j, k), tr = at(min(i + 2, gi - 1), j, k);
                zx[0] = (TC)Pz[tl];
                zx[3] = (TC)Pz[tr];
                yx[0] = (TC)Py[tl];
                yx[3] = (TC)Py[tr];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    if (e == 1 && !have1) continue;
                    // curl(psi), GPU_kernel.cu:1770-1786 (evaluation order kept)
                    const TC ux = half_invh * (zp_[e] - zm_[e] + yzm[e] - yzp[e]);
                    const TC uy = half_invh * (xzp[e] - xzm[e] + zx[e] - zx[e + 2]);
                    const TC uz = half_invh * (yx[e + 2] - yx[e] + xm_[e] - xp_[e]);
                    const size_t c = at(i + e, j, k);
                    const double u[3] = {(double)ux, (double)uy, (double)uz};
#pragma unroll
                    for (int q = 0; q < 3; q++) {
                        const float v = acc[so][q][e] * h3, d = cdiag_half_invh * dg[so][q][e];
                        far[q * G + c] = (float)(kSum ? u[q] - (double)v - (double)d : u[q]);
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < 3; c++) acc[so][c][0] = acc[so][c][1] = 0.f;  // output p + KC + 1 takes the slot
            if (kSum) {
                if (s + 1 < steps) store((s + 1) & 1);
                __syncthreads();
            }
        }
    }
}

// K = 3 and 4: the sums of seven or nine planes do not fit the registers of
// k_curl_far (us, k_curl_far against here: 32^3 50 / 28, 128^3 228 / 177, 256^3
// 1020 / 1232 at K = 3; K = 4 at 128^3 1.0 to 1.7 ms / 645), so the sum runs over
// pairs of neighbours.
// A workgroup owns a 32 x 8 tile of cells and a run of z planes.  The grid
// vorticity streams through an LDS ring of 2K+1 planes with a K-cell halo
// (zero outside the grid, which is the reference's in-grid-only sum), so the
// (2K+1)^3 sum reads LDS; the curl of psi reads global memory (12 loads,
// mostly L2 hits).
constexpr int kCfTX = 32, kCfTY = 8;

template <typename TP, typename TC, int K>
__global__ void __launch_bounds__(256) k_curl_far_pairs(const TP* __restrict__ psi, const float* __restrict__ wg,
                                                  float* __restrict__ far, const float* __restrict__ dir, uint32_t g,
                                                  float h3, TC half_invh, float cdiag_half_invh, int zc) {
    constexpr int W = 2 * K + 1, LXW = kCfTX + 2 * K, LYW = kCfTY + 2 * K, PLW = LXW * LYW;
    __shared__ float ring[W][3][PLW];
    const uint32_t G = g * g * g;
    const int gi = (int)g;
    const int tilesx = (gi + kCfTX - 1) / kCfTX, tilesy = (gi + kCfTY - 1) / kCfTY;
    const int bx = blockIdx.x % tilesx, by = blockIdx.x / tilesx;
    const int z0 = blockIdx.y * zc, z1 = min(z0 + zc, gi);
    const int lx = threadIdx.x % kCfTX, ly = threadIdx.x / kCfTX;
    const int i = bx * kCfTX + lx, j = by * kCfTY + ly;
    const int gx0 = bx * kCfTX - K, gy0 = by * kCfTY - K;
    auto at = [&](int a, int b, int cc) { return ((size_t)cc * g + (size_t)b) * g + (size_t)a; };
    const float* Wx = wg;
    const float* Wy = wg + G;
    const float* Wz = wg + 2 * (size_t)G;
    auto load_plane = [&](int kk) {
        float* rp = &ring[((kk % W) + W) % W][0][0];
        for (int q = threadIdx.x; q < PLW; q += 256) {
            const int yy = q / LXW, xx = q - yy * LXW;
            const int ii = gx0 + xx, jj = gy0 + yy;
            float vx = 0.f, vy = 0.f, vz = 0.f;
            if (kk >= 0 && kk < gi && ii >= 0 && ii < gi && jj >= 0 && jj < gi) {
                const size_t t = at(ii, jj, kk);
                vx = Wx[t];
                vy = Wy[t];
                vz = Wz[t];
            }
            rp[q] = vx;
            rp[PLW + q] = vy;
            rp[2 * PLW + q] = vz;
        }
    };
    for (int kk = z0 - K; kk < z0 + K; kk++) load_plane(kk);
    for (int k = z0; k < z1; k++) {
        load_plane(k + K);
        __syncthreads();
        if (i < gi && j < gi) {
            const int im = i > 0 ? i - 1 : 0, ip = i < gi - 1 ? i + 1 : gi - 1;
            const int jm = j > 0 ? j - 1 : 0, jp = j < gi - 1 ? j + 1 : gi - 1;
            const int km = k > 0 ? k - 1 : 0, kp = k < gi - 1 ? k + 1 : gi - 1;
            const TP* Px = psi;
            const TP* Py = psi + G;
            const TP* Pz = psi + 2 * (size_t)G;
            // curl(psi), GPU_kernel.cu:1770-1786 (evaluation order kept)
            TC ux = half_invh * ((TC)Pz[at(i, jp, k)] - (TC)Pz[at(i, jm, k)] + (TC)Py[at(i, j, km)] -
                                 (TC)Py[at(i, j, kp)]);
            TC uy = half_invh * ((TC)Px[at(i, j, kp)] - (TC)Px[at(i, j, km)] + (TC)Pz[at(im, j, k)] -
                                 (TC)Pz[at(ip, j, k)]);
            TC uz = half_invh * ((TC)Py[at(ip, j, k)] - (TC)Py[at(im, j, k)] + (TC)Px[at(i, jm, k)] -
                                 (TC)Px[at(i, jp, k)]);
            // diagonal term: curl of 0.2505806 h^2 w with the same clamped
            // stencil; the ring holds the neighbours (the clamp reads the edge
            // cell itself, which the ring holds too)
            auto wr = [&](int comp, int ii, int jj, int kk) {
                return ring[((kk % W) + W) % W][comp][(jj - gy0) * LXW + (ii - gx0)];
            };
            const float dx = cdiag_half_invh * (wr(2, i, jp, k) - wr(2, i, jm, k) + (wr(1, i, j, km) - wr(1, i, j, kp)));
            const float dy = cdiag_half_invh * (wr(0, i, j, kp) - wr(0, i, j, km) + (wr(2, im, j, k) - wr(2, ip, j, k)));
            const float dz = cdiag_half_invh * (wr(1, ip, j, k) - wr(1, im, j, k) + (wr(0, i, jm, k) - wr(0, i, jp, k)));
            // local correction over the (2K+1)^3 block.  dir is odd,
            // dir[-D] = -dir[D] (a central difference of the even 1/(4 pi |r|),
            // computed so in FP64 and rounded), so D and -D are taken
            // together: dir[D] x (w[c+D] - w[c-D]); h^3 is applied once.
            float vx = 0.f, vy = 0.f, vz = 0.f;
#pragma unroll
            for (int a = 0; a <= K; a++) {
                const float* rp = &ring[(((k + a) % W) + W) % W][0][0];
                const float* rm = &ring[(((k - a) % W) + W) % W][0][0];
#pragma unroll
                for (int b = -K; b <= K; b++) {
                    if (a == 0 && b < 0) continue;
                    const float* drow = dir + 3 * (size_t)(((a + K) * W + (b + K)) * W);
                    const int rowp = (ly + K + b) * LXW + lx + K, rowm = (ly + K - b) * LXW + lx + K;
#pragma unroll
                    for (int e = -K; e <= K; e++) {
                        if (a == 0 && b == 0 && e <= 0) continue;
                        const float d0 = drow[3 * (e + K)], d1 = drow[3 * (e + K) + 1], d2 = drow[3 * (e + K) + 2];
                        const float ox = rp[rowp + e] - rm[rowm - e];
                        const float oy = rp[PLW + rowp + e] - rm[PLW + rowm - e];
                        const float oz = rp[2 * PLW + rowp + e] - rm[2 * PLW + rowm - e];
                        vx += d1 * oz - d2 * oy;
                        vy += d2 * ox - d0 * oz;
                        vz += d0 * oy - d1 * ox;
                    }
                }
            }
            vx *= h3;
            vy *= h3;
            vz *= h3;
            const size_t c = at(i, j, k);
            far[c] = (float)((double)ux - (double)vx - (double)dx);
            far[(size_t)G + c] = (float)((double)uy - (double)vy - (double)dy);
            far[2 * (size_t)G + c] = (float)((double)uz - (double)vz - (double)dz);
        }
        __syncthreads();  // the next plane load reuses the slot of plane k - K
    }
}

template <typename TP, typename TC, int TX, bool EVEN>
static void launch_curl_far_k(const TP* psi, const float* wgrid, float* far, const float* dir, uint32_t g, int K,
                              float h3, TC half_invh, float cd, hipStream_t st) {
    constexpr int TY = kCfThreads / (TX / 2);
    const uint32_t tiles = div_up(g, TX) * div_up(g, TY);
    // planes per workgroup: about three workgroups per CU (of 256) in all; longer runs
    // (up to 32) repeat fewer of the 2K planes around them, shorter ones (down
    // to 2) keep the chip busy on small grids
    const int zc = std::max(2, std::min(32, (int)div_up(g * tiles, 768)));
    dim3 grid(tiles, div_up(g, zc)), blk(kCfThreads);
    switch (K) {
        case 0: hipLaunchKernelGGL((k_curl_far<TP, TC, 0, TX, EVEN>), grid, blk, 0, st, psi, wgrid, far, dir, g, h3, half_invh, cd, zc); break;
        case 1: hipLaunchKernelGGL((k_curl_far<TP, TC, 1, TX, EVEN>), grid, blk, 0, st, psi, wgrid, far, dir, g, h3, half_invh, cd, zc); break;
        case 2: hipLaunchKernelGGL((k_curl_far<TP, TC, 2, TX, EVEN>), grid, blk, 0, st, psi, wgrid, far, dir, g, h3, half_invh, cd, zc); break;
        case 3:
        case 4: {
            // as many workgroups as fit the LDS of 256 CUs at once: three of
            // 45 KB a CU (K = 3), two of 69 KB (K = 4)
            const uint32_t tp = div_up(g, kCfTX) * div_up(g, kCfTY);
            const int zp = std::max(2, std::min(16, (int)div_up(g * tp, K == 3 ? 768 : 512)));
            const dim3 gp(tp, div_up(g, zp));
            if (K == 3) hipLaunchKernelGGL((k_curl_far_pairs<TP, TC, 3>), gp, blk, 0, st, psi, wgrid, far, dir, g, h3, half_invh, cd, zp);
            else hipLaunchKernelGGL((k_curl_far_pairs<TP, TC, 4>), gp, blk, 0, st, psi, wgrid, far, dir, g, h3, half_invh, cd, zp);
            break;
        }
        default: hipLaunchKernelGGL((k_curl_far<TP, TC, -1, TX, EVEN>), grid, blk, 0, st, psi, wgrid, far, dir, g, h3, half_invh, cd, zc); break;
    }
}

pppm_status launch_curl_far_impl(const void* psi, int psi_dtype, const float* wgrid, float* far, const float* dir,
                                 uint32_t g, int K, double h, hipStream_t st) {
    const float h3 = (float)(h * h * h);
    const double half_invh = 0.5 * (1.0 / h);
    // vortex-in-cell (K < 0): the far-field buffer is the grid velocity itself
    const float cd = K < 0 ? 0.0f : (float)(kRefDiagPsi * h * h * half_invh);
    // 64-cell tiles along x, or 32 where one of two would be partial (us, FP64
    // psi, 64 / 32: 66^3 38 / 25, 80^3 44 / 39, 96^3 47 / 45, 120^3 61 / 62).  Past
    // 128 cells 64 throughout: even where the last is well filled (200^3 253 /
    // 253), behind where it is not (160^3 129 / 114, 288^3 580 / 486)
    const bool t64 = g % 64 == 0 || g > 128;
    auto run = [&](auto* ps, auto hi, auto t64_, auto even) {
        using TP = std::remove_const_t<std::remove_pointer_t<decltype(ps)>>;
        launch_curl_far_k<TP, TP, decltype(t64_)::value ? 64 : 32, decltype(even)::value>(ps, wgrid, far, dir, g, K, h3,
                                                                                        hi, cd, st);
    };
    auto by_size = [&](auto* ps, auto hi) {
        using std::true_type;
        using std::false_type;
        if (g % 2 == 0) t64 ? run(ps, hi, true_type(), true_type()) : run(ps, hi, false_type(), true_type());
        else t64 ? run(ps, hi, true_type(), false_type()) : run(ps, hi, false_type(), false_type());
    };
    if (psi_dtype == PPPM_F64) by_size((const double*)psi, half_invh);
    else by_size((const float*)psi, (float)half_invh);
    PPPM_LAUNCH_CHECK();
    return PPPM_OK;
}

}  // namespace pppm
