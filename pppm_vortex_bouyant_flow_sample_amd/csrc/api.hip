// C ABI: context, pipeline orchestration, hash / multigrid objects, memory.
// Pipeline = BiotSavartSolver::computeFarFieldBuffer + evaluateVelocity
// (hybridFastSummation/hybridFastSummation/BiotSavartSolverImp.cpp:410-816)
// with the device-resident layout of this library: sorted float4 vortex
// coordinates (origin-shifted, deposit cell in .w) and strengths, component-
// major [3][g^3] grids, cell offsets [g^3 + 1].
#include "mg.hpp"
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

using namespace pppm;

static thread_local std::string g_last_error;

extern "C" void pppm_set_last_error(const char* msg, const char* file, int line) {
    char buf[512];
    snprintf(buf, sizeof(buf), "%s (%s:%d)", msg ? msg : "?", file ? file : "?", line);
    g_last_error = buf;
}

extern "C" const char* pppm_last_error(void) { return g_last_error.c_str(); }

#define FAIL(code, msg)                                  \
    do {                                                 \
        pppm_set_last_error((msg), __FILE__, __LINE__);  \
        return (code);                                   \
    } while (0)
#define TRY(expr)                            \
    do {                                     \
        pppm_status _s = (expr);             \
        if (_s != PPPM_OK) return _s;        \
    } while (0)

namespace pppm {
std::mutex& runtime_mutex() {
    static std::mutex m;
    return m;
}
}  // namespace pppm

namespace {

template <typename T>
pppm_status dev_alloc(T** p, size_t count) {
    *p = nullptr;
    if (count == 0) count = 1;
    std::lock_guard<std::mutex> lk(pppm::runtime_mutex());
    if (hipMalloc((void**)p, count * sizeof(T)) != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
        FAIL(PPPM_ERR_NOMEM, "device allocation failed");
    }
    return PPPM_OK;
}
template <typename T>
void dev_free(T*& p) {
    if (p) {
        std::lock_guard<std::mutex> lk(pppm::runtime_mutex());
        (void)hipFree((void*)p);
    }
    p = nullptr;
}

// Sorted-particle buffers: keys / values ping-pong + radix scratch.
struct SortBufs {
    uint32_t cap = 0;
    uint32_t *k0 = nullptr, *v0 = nullptr, *k1 = nullptr, *v1 = nullptr;
    void* scratch = nullptr;
    uint32_t *ks = nullptr, *vs = nullptr;  // result views
    pppm_status ensure(uint32_t n) {
        if (n <= cap && k0) return PPPM_OK;
        release();
        uint32_t c = n < 1024 ? 1024 : n;
        TRY(dev_alloc(&k0, c));
        TRY(dev_alloc(&v0, c));
        TRY(dev_alloc(&k1, c));
        TRY(dev_alloc(&v1, c));
        uint8_t* s;
        TRY(dev_alloc(&s, sort_scratch_bytes(c)));
        scratch = s;
        cap = c;
        return PPPM_OK;
    }
    void release() {
        dev_free(k0);
        dev_free(v0);
        dev_free(k1);
        dev_free(v1);
        uint8_t* s = (uint8_t*)scratch;
        dev_free(s);
        scratch = nullptr;
        cap = 0;
        ks = vs = nullptr;
    }
};

pppm_status validate_params(const pppm_params* p) {
    if (!p) FAIL(PPPM_ERR_INVALID, "null params");
    if (p->g < 2 || p->g > 1024) FAIL(PPPM_ERR_INVALID, "g must be in [2, 1024]");
    if (!(p->h > 0) || !std::isfinite(p->h)) FAIL(PPPM_ERR_INVALID, "h must be positive");
    if (p->K < -1 || p->K > 4) FAIL(PPPM_ERR_INVALID, "K must be in [-1, 4]");
    if (p->kernel != PPPM_KERNEL_EXPCUBIC && p->kernel != PPPM_KERNEL_GAUSSIAN) FAIL(PPPM_ERR_INVALID, "kernel");
    if (!(p->core_a > 0)) FAIL(PPPM_ERR_INVALID, "core_a must be positive");
    if (p->mg_schedule != PPPM_MG_VCYCLE && p->mg_schedule != PPPM_MG_REF_FMG) FAIL(PPPM_ERR_INVALID, "schedule");
    if (p->nu1 < 0 || p->nu2 < 0 || p->nu1 + p->nu2 == 0) FAIL(PPPM_ERR_INVALID, "smoothing counts");
    if (p->mg_max_cycles < 1) FAIL(PPPM_ERR_INVALID, "mg_max_cycles");
    if (p->precision != PPPM_PREC_FP32 && p->precision != PPPM_PREC_MIXED) FAIL(PPPM_ERR_INVALID, "precision");
    return PPPM_OK;
}

PathGeom make_geom(const pppm_params& p) {
    PathGeom pg;
    pg.hash.g = p.g;
    pg.hash.hf = (float)p.h;
    for (int i = 0; i < 3; i++) {
        pg.hash.of[i] = (float)p.origin[i];
        pg.origin[i] = p.origin[i];
    }
    pg.h = (double)pg.hash.hf;  // the path uses the hash's float cell size
    pg.invh = 1.0 / pg.h;
    return pg;
}

// dir table of the far-field correction (GPU_kernel.cu:2646-2677), FP64 on the
// host, stored as float3 rows in ((dz+M)(2M+1)+(dy+M))(2M+1)+(dx+M) order, M =
// max(K, 1) (zero for K < 1), then for dz = 1 .. M the sum of component 2 over
// the plane at dz.
constexpr size_t kDirFloats = 3 * 9 * 9 * 9 + 4;  // the largest K, 4
std::vector<float> far_dir_table(int K, double h) {
    const int M = K < 1 ? 1 : K;
    const int W = 2 * M + 1;
    std::vector<float> out((size_t)W * W * W * 3 + M, 0.f);
    if (K < 1) return out;
    auto R = [](double ax, double ay, double az, double bx, double by, double bz) {
        double r2 = (ax - bx) * (ax - bx) + (ay - by) * (ay - by) + (az - bz) * (az - bz);
        return r2 > 1e-12 ? kRefFourPi * std::sqrt(r2) : 1e24;
    };
    std::vector<double> plane(M + 1, 0.0);
    for (int kk = -M; kk <= M; kk++)
        for (int jj = -M; jj <= M; jj++)
            for (int ii = -M; ii <= M; ii++) {
                if (ii == 0 && jj == 0 && kk == 0) continue;
                double px = (ii + 0.5) * h, py = (jj + 0.5) * h, pz = (kk + 0.5) * h, X = 0.5 * h;
                double dx = 0.5 * ((1.0 / R(X + h, X, X, px, py, pz)) - (1.0 / R(X - h, X, X, px, py, pz))) / h;
                double dy = 0.5 * ((1.0 / R(X, X + h, X, px, py, pz)) - (1.0 / R(X, X - h, X, px, py, pz))) / h;
                double dz = 0.5 * ((1.0 / R(X, X, X + h, px, py, pz)) - (1.0 / R(X, X, X - h, px, py, pz))) / h;
                size_t o = 3 * (size_t)(((kk + M) * W + (jj + M)) * W + (ii + M));
                out[o] = (float)dx;
                out[o + 1] = (float)dy;
                out[o + 2] = (float)dz;
                if (kk > 0) plane[kk] += (double)out[o + 2];
            }
    for (int kk = 1; kk <= M; kk++) out[(size_t)W * W * W * 3 + kk - 1] = (float)plane[kk];
    return out;
}

}  // namespace

namespace pppm {
pppm_status launch_curl_far_impl(const void* psi, int psi_dtype, const float* wgrid, float* far, const float* dir,
                                 uint32_t g, int K, double h, hipStream_t st);
}

// Device bytes of a context: the allocations of pppm_ctx::init, plus the
// vortex buffers for capacity capN and the evaluation buffers for capM (0 =
// none), as ensure_vort / ensure_eval allocate them.
static size_t ctx_bytes(const pppm_params& p, uint32_t capN, uint32_t capM) {
    const size_t G = (size_t)p.g * p.g * p.g;
    size_t b = 0;
    b += 4 * G * 2 + 4 * (G + 1) + 4 * (scan_scratch_words(G) + 16) + 16;  // tables, scan, stray counter
    {
        const SbGeom sg = sb_geom(p.g);  // evaluation order in super-blocks
        b += 4 * (3 * ((size_t)sg.nslots + 16) + scan_scratch_words(sg.nslots) + 16);
    }
    b += 4 * ((G + 3) / 4);                                                  // stray flags
    b += 4 * 3 * G * 2;                                                      // vorticity, far field
    if (p.precision == PPPM_PREC_MIXED)
        b += 3 * G * (8 + 8 + 8 + 4 + 4);  // psi64 x2, b64, r32, e32
    else
        b += 3 * G * 4;  // psi32
    if (p.precision == PPPM_PREC_MIXED && p.mg_schedule == PPPM_MG_REF_FMG)
        b += MGHier<double>::bytes_for((int)p.g, (int)p.g, (int)p.g, 3);  // the FP64 hierarchy
    b += 4 * kDirFloats;  // direction table
    b += MGHier<float>::bytes_for((int)p.g, (int)p.g, (int)p.g, 3);
    if (capN) b += (size_t)capN * (4 * 4 + 16 + 16) + sort_scratch_bytes(capN);
    if (capM) b += (size_t)capM * (4 * 4 + 16 + 16) + sort_scratch_bytes(capM);
    return b;
}

// Records body() on stream st into an executable graph.  Captures are
// thread-local and hold the process-wide lock shared with device allocation,
// so serving threads can capture side by side.
template <typename F>
static pppm_status capture_graph(hipStream_t st, hipGraphExec_t* exec, F body) {
    std::lock_guard<std::mutex> lk(runtime_mutex());
    PPPM_HIP_TRY(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    pppm_status s = body();
    hipGraph_t gr = nullptr;
    hipError_t e = hipStreamEndCapture(st, &gr);
    if (s != PPPM_OK || e != hipSuccess) {
        if (gr) (void)hipGraphDestroy(gr);
        (void)hipGetLastError();
        if (s != PPPM_OK) return s;
        PPPM_HIP_TRY(e);
    }
    e = hipGraphInstantiate(exec, gr, nullptr, nullptr, 0);
    (void)hipGraphDestroy(gr);
    PPPM_HIP_TRY(e);
    return PPPM_OK;
}

// Graphs of a mixed-precision solve's geometry: the warm start and the outer
// step per psi ping-pong parity.
struct MixedGraphs {
    hipGraphExec_t warm = nullptr, step[2] = {nullptr, nullptr};
    void drop() {
        for (hipGraphExec_t* e : {&warm, &step[0], &step[1]})
            if (*e) {
                (void)hipGraphExecDestroy(*e);
                *e = nullptr;
            }
    }
};

struct pppm_ctx {
    pppm_params p{};
    PathGeom pg{};
    hipStream_t st = nullptr;
    bool own_stream = false;
    uint32_t g = 0;
    size_t G = 0;
    // vortices
    uint32_t n = 0, capN = 0;
    SortBufs vs;
    float4 *spos = nullptr, *somg = nullptr;
    // tracer batches: FP64 velocities of one batch, [3][capT]
    double* utr = nullptr;
    uint32_t capT = 0;
    // values being smoothed, FP64 in hash order
    double4* sval = nullptr;
    uint32_t capS = 0;
    // time step: segment ends, kappa, vorticity change [3][n], end velocities
    float4 *seg_a = nullptr, *seg_b = nullptr;
    double *kappa = nullptr, *dvort = nullptr;
    double4 *vel_a = nullptr, *vel_b = nullptr;
    uint32_t capStep = 0;
    // RK2's predicted ends, centres, strengths and velocities
    float4 *seg_a2 = nullptr, *seg_b2 = nullptr, *cent2 = nullptr;
    double4 *vel_a2 = nullptr, *vel_b2 = nullptr;
    double* vort2 = nullptr;
    uint32_t capStep2 = 0;
    float* bbox = nullptr;
    uint32_t *cstart = nullptr, *cend = nullptr, *coff = nullptr, *scan_scr = nullptr;
    // evaluation order in super-blocks (slot bounds, prefix, scan scratch)
    SbGeom sbg{};
    uint32_t *sb_start = nullptr, *sb_len = nullptr, *sb_pre = nullptr, *sb_scr = nullptr;
    uint32_t* d_strays = nullptr;
    uint32_t* h_strays = nullptr;
    uint8_t* sflag = nullptr;  // per cell: deposit cell of a stray (P2M sets, the stray pass clears)
    bool have_vort = false;
    // evaluation points
    uint32_t capM = 0;
    SortBufs es;
    float4 *epos = nullptr, *eoth = nullptr;
    // grids
    float *wg = nullptr, *far = nullptr, *psi32 = nullptr, *dir = nullptr;
    double *psi64[2] = {nullptr, nullptr}, *b64 = nullptr;
    float *r32 = nullptr, *e32 = nullptr;
    int psi_cur = 0;
    MGHier<float> mg;
    // FP64 hierarchy of the reference's schedule in mixed precision (the
    // reference's MultiGridSolver3DPeriod_double), made on first use
    MGHier<double>* mg64 = nullptr;
    bool have_far = false;
    pppm_stats stats{};
    // per-iteration multigrid work captured once per geometry and replayed
    bool use_graphs = true;
    int32_t near_order = PPPM_NEAR_ORDER_AUTO;
    MixedGraphs mixg;
    hipGraphExec_t g_plain = nullptr;

    // Sort keys carry each point's octant in its cell (8 G keys fit 32 bits):
    // points come out of the sort in the near field's evaluation order.
    bool octant_keys() const { return G * 8 <= ((size_t)1 << 32); }

    void drop_graphs() {
        mixg.drop();
        if (g_plain) {
            (void)hipGraphExecDestroy(g_plain);
            g_plain = nullptr;
        }
    }

    // Records body() on the context stream into an executable graph.
    template <typename F>
    pppm_status capture(hipGraphExec_t* exec, F body) {
        return capture_graph(st, exec, body);
    }

    size_t device_bytes() const {
        size_t b = ctx_bytes(p, vs.cap, es.cap);
        // a hierarchy made for an earlier schedule stays until release
        if (mg64 && !(p.precision == PPPM_PREC_MIXED && p.mg_schedule == PPPM_MG_REF_FMG))
            b += mg64->device_bytes();
        return b;
    }

    pppm_status ensure_mg64() {
        if (mg64) return PPPM_OK;
        mg64 = new MGHier<double>;
        pppm_status s = mg64->init((int)g, (int)g, (int)g, 3);
        if (s != PPPM_OK) {
            delete mg64;
            mg64 = nullptr;
        }
        return s;
    }

    pppm_status init(const pppm_params& prm) {
        p = prm;
        pg = make_geom(p);
        g = p.g;
        G = (size_t)g * g * g;
        {
            std::lock_guard<std::mutex> lk(runtime_mutex());
            if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess)
                FAIL(PPPM_ERR_HIP, "stream creation failed");
        }
        own_stream = true;
        TRY(dev_alloc(&cstart, G));
        TRY(dev_alloc(&cend, G));
        TRY(dev_alloc(&coff, G + 1));
        TRY(dev_alloc(&scan_scr, scan_scratch_words(G) + 16));
        sbg = sb_geom(g);
        TRY(dev_alloc(&sb_start, (size_t)sbg.nslots + 16));
        TRY(dev_alloc(&sb_len, (size_t)sbg.nslots + 16));
        TRY(dev_alloc(&sb_pre, (size_t)sbg.nslots + 16));
        TRY(dev_alloc(&sb_scr, scan_scratch_words(sbg.nslots) + 16));
        TRY(dev_alloc(&d_strays, 4));
        {
            const size_t words = (G + 3) / 4;
            uint32_t* f = nullptr;
            TRY(dev_alloc(&f, words));
            sflag = reinterpret_cast<uint8_t*>(f);
            TRY(launch_fill_u32(f, words, 0u, st));
        }
        {
            std::lock_guard<std::mutex> lk(runtime_mutex());
            if (hipHostMalloc((void**)&h_strays, 16) != hipSuccess) FAIL(PPPM_ERR_NOMEM, "pinned alloc failed");
        }
        TRY(dev_alloc(&wg, 3 * G));
        TRY(dev_alloc(&far, 3 * G));
        if (p.precision == PPPM_PREC_MIXED) {
            TRY(dev_alloc(&psi64[0], 3 * G));
            TRY(dev_alloc(&psi64[1], 3 * G));
            TRY(dev_alloc(&b64, 3 * G));
            TRY(dev_alloc(&r32, 3 * G));
            TRY(dev_alloc(&e32, 3 * G));
        } else {
            TRY(dev_alloc(&psi32, 3 * G));
        }
        TRY(dev_alloc(&dir, kDirFloats));
        TRY(upload_dir());
        TRY(mg.init((int)g, (int)g, (int)g, 3));
        return PPPM_OK;
    }

    pppm_status upload_dir() {
        if (p.K < 0) return PPPM_OK;
        std::vector<float> dt = far_dir_table(p.K, pg.h);
        PPPM_HIP_TRY(hipMemcpyAsync(dir, dt.data(), dt.size() * sizeof(float), hipMemcpyHostToDevice, st));
        PPPM_HIP_TRY(hipStreamSynchronize(st));
        return PPPM_OK;
    }

    void release() {
        drop_graphs();
        vs.release();
        es.release();
        dev_free(spos);
        dev_free(somg);
        dev_free(utr);
        dev_free(sval);
        dev_free(seg_a);
        dev_free(seg_b);
        dev_free(kappa);
        dev_free(dvort);
        dev_free(vel_a);
        dev_free(vel_b);
        dev_free(seg_a2);
        dev_free(seg_b2);
        dev_free(cent2);
        dev_free(vel_a2);
        dev_free(vel_b2);
        dev_free(vort2);
        dev_free(bbox);
        dev_free(cstart);
        dev_free(cend);
        dev_free(coff);
        dev_free(scan_scr);
        dev_free(sb_start);
        dev_free(sb_len);
        dev_free(sb_pre);
        dev_free(sb_scr);
        dev_free(d_strays);
        dev_free(sflag);
        if (h_strays) {
            std::lock_guard<std::mutex> lk(runtime_mutex());
            (void)hipHostFree(h_strays);
        }
        h_strays = nullptr;
        dev_free(epos);
        dev_free(eoth);
        dev_free(wg);
        dev_free(far);
        dev_free(psi32);
        dev_free(dir);
        dev_free(psi64[0]);
        dev_free(psi64[1]);
        dev_free(b64);
        dev_free(r32);
        dev_free(e32);
        mg.release();
        if (mg64) {
            mg64->release();
            delete mg64;
            mg64 = nullptr;
        }
        if (own_stream && st) {
            std::lock_guard<std::mutex> lk(runtime_mutex());
            (void)hipStreamDestroy(st);
        }
        st = nullptr;
    }

    pppm_status ensure_vort(uint32_t nn) {
        TRY(vs.ensure(nn));
        if (nn > capN || !spos) {
            dev_free(spos);
            dev_free(somg);
            uint32_t c = vs.cap;
            TRY(dev_alloc(&spos, c));
            TRY(dev_alloc(&somg, c));
            capN = c;
        }
        return PPPM_OK;
    }
    pppm_status ensure_eval(uint32_t mm, bool other) {
        TRY(es.ensure(mm));
        if (mm > capM || !epos || (other && !eoth)) {
            dev_free(epos);
            dev_free(eoth);
            uint32_t c = es.cap;
            TRY(dev_alloc(&epos, c));
            TRY(dev_alloc(&eoth, c));
            capM = c;
        }
        return PPPM_OK;
    }
};

// ---------------------------------------------------------------------------
extern "C" void pppm_params_config_preset(pppm_params* p, uint32_t g) {
    if (!p) return;
    memset(p, 0, sizeof(*p));
    p->g = g;
    p->h = 1.0 / (double)g;
    p->origin[0] = p->origin[1] = p->origin[2] = 0.0;
    p->K = 2;
    p->kernel = PPPM_KERNEL_EXPCUBIC;
    p->core_a = 1.5 * (double)(float)p->h;
    p->mg_schedule = PPPM_MG_VCYCLE;
    p->nu1 = 2;
    p->nu2 = 2;
    // red-black SOR with a mild over-relaxation: on the 8M plume at 256^3 a
    // V(2,2) cycle contracts enough more than with Gauss-Seidel (omega 1)
    // that the mixed solve to 1e-7 takes 5 cycles instead of 6 and the FP32
    // solve to 1e-6 takes 4 instead of 5
    p->mg_omega = 1.15;
    p->mg_tol = 1e-6;
    p->mg_max_cycles = 40;
    p->precision = PPPM_PREC_FP32;
}

extern "C" void pppm_params_reference_preset(pppm_params* p, uint32_t g, int32_t K) {
    if (!p) return;
    pppm_params_config_preset(p, g);
    p->K = K;
    p->core_a = 0.08;                       // GPU_kernel.cu:2306
    p->mg_schedule = PPPM_MG_REF_FMG;       // MultiGrid.cpp:202-250
    p->nu1 = p->nu2 = 4;                    // MultiGrid.cpp:149, 186
    p->mg_omega = (double)1.43f;            // MultiGrid_kernel.cu:36
    p->mg_max_cycles = 1;
    p->precision = PPPM_PREC_MIXED;         // FP64 multigrid (BiotSavartSolver.h:57)
}

// setDomain's formula (BiotSavartSolverImp.cpp:378-409): L = 3 * the largest
// extent, origin = bbox centre - L/2, h = L / g.
static pppm_status domain_from_extent(double mx, double Mx, double my, double My, double mz, double Mz, uint32_t g,
                                      double origin_out[3], double* h_out) {
    double L = Mx - mx;
    if (My - my > L) L = My - my;
    if (Mz - mz > L) L = Mz - mz;
    L *= 3;
    origin_out[0] = (mx + 0.5 * (Mx - mx)) - 0.5 * L;
    origin_out[1] = (my + 0.5 * (My - my)) - 0.5 * L;
    origin_out[2] = (mz + 0.5 * (Mz - mz)) - 0.5 * L;
    *h_out = L / (double)g;
    if (!(L > 0)) FAIL(PPPM_ERR_INVALID, "degenerate particle extent");
    return PPPM_OK;
}

extern "C" pppm_status pppm_reference_domain(const float* pos, uint32_t n, uint32_t g, double origin_out[3],
                                             double* h_out) {
    if (!pos || n == 0 || g == 0 || !origin_out || !h_out) FAIL(PPPM_ERR_INVALID, "reference_domain args");
    double mx = pos[0], Mx = pos[0], my = pos[1], My = pos[1], mz = pos[2], Mz = pos[2];
    for (uint32_t i = 1; i < n; i++) {
        double x = pos[4 * (size_t)i], y = pos[4 * (size_t)i + 1], z = pos[4 * (size_t)i + 2];
        if (x < mx) mx = x; else if (x > Mx) Mx = x;
        if (y < my) my = y; else if (y > My) My = y;
        if (z < mz) mz = z; else if (z > Mz) Mz = z;
    }
    return domain_from_extent(mx, Mx, my, My, mz, Mz, g, origin_out, h_out);
}

extern "C" pppm_status pppm_create(const pppm_params* p, pppm_ctx** out) {
    if (!out) FAIL(PPPM_ERR_INVALID, "null out");
    *out = nullptr;
    TRY(validate_params(p));
    int nd = 0;
    if (hipGetDeviceCount(&nd) != hipSuccess || nd < 1) FAIL(PPPM_ERR_NO_DEVICE, "no HIP device");
    pppm_ctx* c = new pppm_ctx();
    pppm_status s = c->init(*p);
    if (s != PPPM_OK) {
        c->release();
        delete c;
        return s;
    }
    *out = c;
    return PPPM_OK;
}

extern "C" void pppm_destroy(pppm_ctx* c) {
    if (!c) return;
    if (c->st) (void)hipStreamSynchronize(c->st);
    c->release();
    delete c;
}

extern "C" pppm_status pppm_set_stream(pppm_ctx* c, void* s) {
    if (!c) FAIL(PPPM_ERR_INVALID, "null ctx");
    PPPM_HIP_TRY(hipStreamSynchronize(c->st));
    if (c->own_stream) (void)hipStreamDestroy(c->st);
    c->st = (hipStream_t)s;
    c->own_stream = false;
    c->drop_graphs();
    return PPPM_OK;
}

extern "C" pppm_status pppm_get_stream(const pppm_ctx* c, void** s) {
    if (!c || !s) FAIL(PPPM_ERR_INVALID, "null arg");
    *s = (void*)c->st;
    return PPPM_OK;
}

extern "C" pppm_status pppm_set_domain(pppm_ctx* c, const double origin[3], double h) {
    if (!c || !origin) FAIL(PPPM_ERR_INVALID, "null arg");
    pppm_params np = c->p;
    np.h = h;
    for (int i = 0; i < 3; i++) np.origin[i] = origin[i];
    TRY(validate_params(&np));
    PPPM_HIP_TRY(hipStreamSynchronize(c->st));
    c->p = np;
    c->pg = make_geom(np);
    c->have_vort = false;
    c->have_far = false;
    c->drop_graphs();
    return c->upload_dir();
}

extern "C" pppm_status pppm_update_params(pppm_ctx* c, const pppm_params* p) {
    if (!c || !p) FAIL(PPPM_ERR_INVALID, "null arg");
    TRY(validate_params(p));
    if (p->g != c->p.g || p->precision != c->p.precision)
        FAIL(PPPM_ERR_INVALID, "grid size and precision are fixed for a context");
    PPPM_HIP_TRY(hipStreamSynchronize(c->st));
    c->p = *p;
    c->pg = make_geom(*p);
    c->have_vort = false;
    c->have_far = false;
    c->drop_graphs();
    return c->upload_dir();
}

extern "C" pppm_status pppm_get_device_bytes(const pppm_ctx* c, size_t* bytes) {
    if (!c || !bytes) FAIL(PPPM_ERR_INVALID, "null arg");
    *bytes = c->device_bytes();
    return PPPM_OK;
}

extern "C" pppm_status pppm_estimate_device_bytes(const pppm_params* p, uint32_t n, uint32_t m, int32_t other_end,
                                                  size_t* bytes) {
    TRY(validate_params(p));
    if (!bytes) FAIL(PPPM_ERR_INVALID, "null arg");
    (void)other_end;  // the segment-end buffer is allocated with the evaluation points
    *bytes = ctx_bytes(*p, n ? std::max(n, 1024u) : 0, m ? std::max(m, 1024u) : 0);
    return PPPM_OK;
}

extern "C" pppm_status pppm_set_graphs(pppm_ctx* c, int32_t on) {
    if (!c) FAIL(PPPM_ERR_INVALID, "null ctx");
    PPPM_HIP_TRY(hipStreamSynchronize(c->st));
    c->use_graphs = on != 0;
    if (!c->use_graphs) c->drop_graphs();
    return PPPM_OK;
}

extern "C" pppm_status pppm_set_near_order(pppm_ctx* c, int32_t order) {
    if (!c) FAIL(PPPM_ERR_INVALID, "null ctx");
    if (order < PPPM_NEAR_ORDER_AUTO || order > PPPM_NEAR_ORDER_SUPER_BLOCKS) FAIL(PPPM_ERR_INVALID, "near order");
    c->near_order = order;
    return PPPM_OK;
}

extern "C" pppm_status pppm_get_params(const pppm_ctx* c, pppm_params* out) {
    if (!c || !out) FAIL(PPPM_ERR_INVALID, "null arg");
    *out = c->p;
    return PPPM_OK;
}

extern "C" pppm_status pppm_set_vortices(pppm_ctx* c, uint32_t n, const float* pos4, const void* wx, const void* wy,
                                         const void* wz, uint32_t w_stride, int32_t w_dtype) {
    if (!c) FAIL(PPPM_ERR_INVALID, "null ctx");
    if (n > 0 && (!pos4 || !wx || !wy || !wz)) FAIL(PPPM_ERR_INVALID, "null vortex array");
    if (w_dtype != PPPM_F32 && w_dtype != PPPM_F64) FAIL(PPPM_ERR_INVALID, "w_dtype");
    if (w_stride == 0) FAIL(PPPM_ERR_INVALID, "w_stride");
    if (n > (1u << 30)) FAIL(PPPM_ERR_INVALID, "too many vortices");
    hipStream_t st = c->st;
    TRY(c->ensure_vort(n));
    c->n = n;
    c->have_far = false;
    const uint32_t osh = c->octant_keys() ? 3u : 0u;
    TRY(launch_calc_keys((const float4*)pos4, n, c->pg.hash, c->vs.k0, nullptr, st, osh != 0));
    TRY(radix_sort_pairs(c->vs.k0, c->vs.v0, c->vs.k1, c->vs.v1, n, key_bits_for(c->G) + osh, true, c->vs.scratch,
                         &c->vs.ks, &c->vs.vs, st));
    TRY(launch_cell_tables(c->vs.ks, n, (uint32_t)c->G, c->cstart, c->cend, st, osh, c->coff, c->scan_scr));
    TRY(launch_fill_u32(c->d_strays, 1, 0u, st));
    {
        // the sort's spare value buffer holds the inverse permutation
        uint32_t* inv = c->vs.vs == c->vs.v0 ? c->vs.v1 : c->vs.v0;
        TRY(launch_reorder_vortices_scatter(c->vs.vs, inv, (const float4*)pos4, wx, wy, wz, w_stride, w_dtype, n,
                                            c->pg, c->spos, c->somg, c->d_strays, st));
    }
    c->have_vort = true;
    c->stats.n = n;
    return PPPM_OK;
}

// FP32 V-cycles before the first FP64 defect correction of a mixed solve.
constexpr int kMixedWarmCycles = 4;

// One mixed-precision solve over `scenes` scenes of three components each
// (component-major [3 scenes][g^3] arrays): a context's own scene, or several
// small scenes with identical parameters that the request server solves in
// one set of launches.  Every kernel works per component, so each scene goes
// through exactly the operations a solve of that scene alone would run.
struct MixedSolve {
    MGHier<float>* mg = nullptr;
    float *e32 = nullptr, *wg = nullptr, *r32 = nullptr;
    double *b64 = nullptr, *psi64[2] = {nullptr, nullptr};
    int g = 0, scenes = 1;
    const pppm_params* p = nullptr;
    double h = 0;
    hipStream_t st = nullptr;
    MixedGraphs* graphs = nullptr;  // null: launch eagerly
};

// A scene's solve ended: its FP64 solution is in psi64[psi] (component-major,
// scene j's three components at 3 j), valid until the next outer step is
// enqueued on the solve's stream.
struct SceneResult {
    int inner = 0, outer = 0, psi = 0;
    double rel[3] = {0, 0, 0};
    bool converged = false;
};

// Warm start: the first V-cycles run in FP32 in place on e from e = 0, on the
// FP32 vorticity grid with the scale -h^2 (the FP32 path's right-hand side,
// equal to (float)b to FP32 rounding), as far as they contract the residual
// before FP32 rounding stalls them (about 2e-5 after four V(2,2) cycles,
// against a floor near 1e-6); then psi = e with its FP64 defect r = b - A psi
// and the FP64 norms of r and b.  Each later outer step is one V-cycle on the
// FP64 defect.  A scene ends at the first check where its worst component's
// relative residual meets the tolerance (done(j, result) is called before any
// later step is enqueued), or when the cycle limit stops the solve.
template <typename Done>
static pppm_status mixed_solve(const MixedSolve& a, Done done) {
    hipStream_t st = a.st;
    const int g = a.g, nc = 3 * a.scenes;
    TRY(a.mg->set_active(nc));
    double* outn = a.mg->norm_out();
    double* hn = a.mg->host_norms();
    std::vector<double> rel(4 * (size_t)a.scenes);
    auto read_rel = [&]() -> pppm_status {
        PPPM_HIP_TRY(hipMemcpyAsync(hn, outn, 2 * (size_t)nc * sizeof(double), hipMemcpyDeviceToHost, st));
        PPPM_HIP_TRY(hipStreamSynchronize(st));
        for (int j = 0; j < a.scenes; j++) {
            double w = 0;
            for (int k = 0; k < 3; k++) {
                const int q = 3 * j + k;
                const double rr = std::sqrt(hn[2 * q]), bb = std::sqrt(hn[2 * q + 1]);
                rel[4 * j + k] = bb > 0 ? rr / bb : rr;
                if (rel[4 * j + k] > w) w = rel[4 * j + k];
            }
            rel[4 * j + 3] = w;
        }
        return PPPM_OK;
    };
    const pppm_params& p = *a.p;
    int cur = 0, outer = 0, inner = 0;
    const int warm = std::min(kMixedWarmCycles, p.mg_max_cycles);
    const float bs = (float)(-a.h * a.h);
    MGHier<float>* mg = a.mg;
    auto warmup = [&]() -> pppm_status {
        for (int q = 0; q < warm; q++)
            TRY(mg->vcycle(a.e32, a.wg, bs, p.nu1, p.nu2, (float)p.mg_omega, true, st, q == 0));
        return launch_dc_step(nullptr, a.e32, a.b64, a.psi64[0], a.r32, g, g, g, nc, mg->partials(), outn, st);
    };
    if (warm > 0) {
        if (a.graphs) {
            if (!a.graphs->warm) TRY(capture_graph(st, &a.graphs->warm, warmup));
            PPPM_HIP_TRY(hipGraphLaunch(a.graphs->warm, st));
        } else {
            TRY(warmup());
        }
        inner += warm;
        outer++;
    } else {
        // r32 = b (psi = 0) and the norms of b
        TRY(launch_dc_step(nullptr, nullptr, a.b64, a.psi64[0], a.r32, g, g, g, nc, mg->partials(), outn, st));
    }
    // one outer step: e = V-cycle(A e = r32, e = 0); psi_next = psi + e;
    // r32 = b - A psi_next and its FP64 norms
    auto step = [&](int c0) -> pppm_status {
        TRY(mg->vcycle(a.e32, a.r32, 1.0f, p.nu1, p.nu2, (float)p.mg_omega, true, st, true));
        return launch_dc_step(a.psi64[c0], a.e32, a.b64, a.psi64[1 - c0], a.r32, g, g, g, nc, mg->partials(), outn,
                              st);
    };
    std::vector<char> fin((size_t)a.scenes, 0);
    int left = a.scenes;
    auto finish = [&](bool last) -> pppm_status {
        for (int j = 0; j < a.scenes; j++) {
            if (fin[j] || !(last || rel[4 * j + 3] <= p.mg_tol)) continue;
            SceneResult r;
            r.inner = inner;
            r.outer = outer;
            r.psi = cur;
            for (int k = 0; k < 3; k++) r.rel[k] = rel[4 * j + k];
            r.converged = rel[4 * j + 3] <= p.mg_tol;
            TRY(done(j, r));
            fin[j] = 1;
            left--;
        }
        return PPPM_OK;
    };
    TRY(read_rel());
    TRY(finish(false));
    while (outer < p.mg_max_cycles && left > 0) {
        const int c0 = cur;
        if (a.graphs) {
            if (!a.graphs->step[c0]) TRY(capture_graph(st, &a.graphs->step[c0], [&]() { return step(c0); }));
            PPPM_HIP_TRY(hipGraphLaunch(a.graphs->step[c0], st));
        } else {
            TRY(step(c0));
        }
        inner++;
        cur = 1 - c0;
        outer++;
        TRY(read_rel());
        TRY(finish(false));
    }
    return finish(true);
}

static pppm_status solve_mixed(pppm_ctx* c) {
    MixedSolve a;
    a.mg = &c->mg;
    a.e32 = c->e32;
    a.wg = c->wg;
    a.r32 = c->r32;
    a.b64 = c->b64;
    a.psi64[0] = c->psi64[0];
    a.psi64[1] = c->psi64[1];
    a.g = (int)c->g;
    a.scenes = 1;
    a.p = &c->p;
    a.h = c->pg.h;
    a.st = c->st;
    a.graphs = c->use_graphs ? &c->mixg : nullptr;
    return mixed_solve(a, [c](int, const SceneResult& r) -> pppm_status {
        c->psi_cur = r.psi;
        c->stats.mg_cycles = r.inner;
        c->stats.mg_outer = r.outer;
        for (int k = 0; k < 3; k++) c->stats.mg_relres[k] = r.rel[k];
        c->stats.mg_converged = r.converged;
        return PPPM_OK;
    });
}

// P2M and the right-hand side on the context's stream.  The stray counter
// gates the neighbourhood pass on the device; its host copy (for the
// statistics) is read after the solve's first synchronisation.
static pppm_status far_p2m(pppm_ctx* c) {
    hipStream_t st = c->st;
    const bool mixed = c->p.precision == PPPM_PREC_MIXED;
    const double h = c->pg.h;
    PPPM_HIP_TRY(hipMemcpyAsync(c->h_strays, c->d_strays, 4, hipMemcpyDeviceToHost, st));
    TRY(launch_p2m(c->coff, c->spos, c->somg, c->g, c->pg.invh, c->wg, mixed ? c->b64 : nullptr, -h * h, c->sflag,
                   st));
    return launch_p2m_strays(c->coff, c->spos, c->somg, c->g, c->pg.invh, c->wg, mixed ? c->b64 : nullptr, -h * h,
                             c->d_strays, c->sflag, st);
}

extern "C" pppm_status pppm_compute_far_field(pppm_ctx* c) {
    if (!c) FAIL(PPPM_ERR_INVALID, "null ctx");
    if (!c->have_vort) FAIL(PPPM_ERR_STATE, "set_vortices first");
    hipStream_t st = c->st;
    const bool mixed = c->p.precision == PPPM_PREC_MIXED;
    const double h = c->pg.h;
    TRY(far_p2m(c));
    const void* psi;
    int pdt;
    if (mixed && c->p.mg_schedule == PPPM_MG_REF_FMG) {
        // the reference's schedule in FP64 throughout (MultiGridSolver3DPeriod_double,
        // BiotSavartSolver.h:57; MultiGrid.cpp:202-250) on the FP64 right-hand
        // side -h^2 w from P2M
        TRY(c->ensure_mg64());
        TRY(c->mg64->fill(c->psi64[0], 3 * c->G, st));
        TRY(c->mg64->ref_fmg(c->psi64[0], c->b64, 1.0, c->p.nu1, c->p.nu2, c->p.mg_omega, st));
        double rn[3], bn[3];
        TRY(c->mg64->norms(c->psi64[0], c->b64, 1.0, rn, bn, st));
        for (int k = 0; k < 3; k++) c->stats.mg_relres[k] = bn[k] > 0 ? rn[k] / bn[k] : rn[k];
        c->stats.mg_cycles = 1;
        c->stats.mg_outer = 0;
        c->stats.mg_converged = 1;
        c->psi_cur = 0;
        psi = c->psi64[0];
        pdt = PPPM_F64;
    } else if (mixed) {
        TRY(solve_mixed(c));
        psi = c->psi64[c->psi_cur];
        pdt = PPPM_F64;
    } else {
        const float bscale = (float)(-h * h);
        TRY(c->mg.fill(c->psi32, 3 * c->G, st));
        if (c->p.mg_schedule == PPPM_MG_REF_FMG) {
            TRY(c->mg.ref_fmg(c->psi32, c->wg, bscale, c->p.nu1, c->p.nu2, (float)c->p.mg_omega, st));
            double rn[3], bn[3];
            TRY(c->mg.norms(c->psi32, c->wg, bscale, rn, bn, st));
            for (int k = 0; k < 3; k++) c->stats.mg_relres[k] = bn[k] > 0 ? rn[k] / bn[k] : rn[k];
            c->stats.mg_cycles = 1;
            c->stats.mg_converged = 1;
        } else {
            // V-cycles until the FP64-accumulated relative residual meets the
            // tolerance or stops improving (FP32 rounding floor)
            double rn[3], bn[3], w = 0, prev;
            auto worst = [&]() {
                double m = 0;
                for (int k = 0; k < 3; k++) {
                    c->stats.mg_relres[k] = bn[k] > 0 ? rn[k] / bn[k] : rn[k];
                    if (c->stats.mg_relres[k] > m) m = c->stats.mg_relres[k];
                }
                return m;
            };
            TRY(c->mg.norms(c->psi32, c->wg, bscale, rn, bn, st));
            w = worst();
            int cyc = 0;
            auto cycle = [c, bscale, st]() -> pppm_status {
                TRY(c->mg.vcycle(c->psi32, c->wg, bscale, c->p.nu1, c->p.nu2, (float)c->p.mg_omega, true, st));
                return c->mg.norms_launch(c->psi32, c->wg, bscale, st);
            };
            while (cyc < c->p.mg_max_cycles && w > c->p.mg_tol) {
                if (c->use_graphs) {
                    if (!c->g_plain) TRY(c->capture(&c->g_plain, cycle));
                    PPPM_HIP_TRY(hipGraphLaunch(c->g_plain, st));
                } else {
                    TRY(cycle());
                }
                cyc++;
                TRY(c->mg.norms_read(rn, bn, st));
                prev = w;
                w = worst();
                if (cyc >= 3 && w > 0.9 * prev) break;
            }
            c->stats.mg_cycles = cyc;
            c->stats.mg_converged = w <= c->p.mg_tol;
        }
        c->stats.mg_outer = 0;
        psi = c->psi32;
        pdt = PPPM_F32;
    }
    // every solve path above has synchronised the stream at least once
    c->stats.strays = *c->h_strays;
    TRY(launch_curl_far_impl(psi, pdt, c->wg, c->far, c->dir, c->g, c->p.K, h, st));
    c->have_far = true;
    return PPPM_OK;
}

// ---------------------------------------------------------------------------
// Several small scenes' Poisson solves in one set of launches (request server).
//
// Scenes on grids of up to 64^3 cells leave the device mostly idle during
// their multigrid: every V-cycle is some twenty-five launches of a few
// microseconds over a few hundred thousand cells.  A group stacks the
// right-hand sides of up to `cap` scenes with identical parameters into one
// [3 cap][g^3] hierarchy and runs the mixed-precision solve once for all of
// them: the same launches, each over all the scenes' components.  Every
// kernel works per component and each scene's solution is copied out when its
// own residual meets the tolerance, so each scene gets exactly the solution
// (and iteration counts) it gets when solved alone.
struct pppm_group {
    uint32_t g = 0;
    size_t G = 0;
    int cap = 0;
    hipStream_t st = nullptr;
    MGHier<float> mg;
    float *wg = nullptr, *e32 = nullptr, *r32 = nullptr;
    double *b64 = nullptr, *psi64[2] = {nullptr, nullptr};
    std::vector<MixedGraphs> graphs;  // per scene count (index count - 1)
    std::vector<hipEvent_t> ev;       // one per scene, and one for the solve
    size_t bytes = 0;

    void release() {
        for (MixedGraphs& m : graphs) m.drop();
        graphs.clear();
        dev_free(wg);
        dev_free(e32);
        dev_free(r32);
        dev_free(b64);
        dev_free(psi64[0]);
        dev_free(psi64[1]);
        mg.release();
        std::lock_guard<std::mutex> lk(runtime_mutex());
        for (hipEvent_t e : ev) (void)hipEventDestroy(e);
        ev.clear();
        if (st) (void)hipStreamDestroy(st);
        st = nullptr;
    }
};

size_t group_bytes(uint32_t g, int cap) {
    const size_t G = (size_t)g * g * g, n = 3 * (size_t)cap * G;
    return n * (4 + 4 + 4 + 8 + 8 + 8) + MGHier<float>::bytes_for((int)g, (int)g, (int)g, 3 * cap);
}

bool group_eligible(const pppm_params& p, uint32_t max_g) {
    return p.precision == PPPM_PREC_MIXED && p.mg_schedule == PPPM_MG_VCYCLE && p.g <= max_g && p.g >= 2;
}

pppm_status group_create(uint32_t g, int cap, pppm_group** out) {
    if (!out || g < 2 || cap < 1 || 3 * cap > MGHier<float>::kMaxComp) FAIL(PPPM_ERR_INVALID, "group size");
    pppm_group* q = new pppm_group;
    q->g = g;
    q->G = (size_t)g * g * g;
    q->cap = cap;
    auto fail = [&](pppm_status s) {
        q->release();
        delete q;
        return s;
    };
    {
        std::lock_guard<std::mutex> lk(runtime_mutex());
        if (hipStreamCreateWithFlags(&q->st, hipStreamNonBlocking) != hipSuccess) {
            q->st = nullptr;
            delete q;
            FAIL(PPPM_ERR_HIP, "group stream creation failed");
        }
        q->ev.assign((size_t)cap + 1, nullptr);
        for (hipEvent_t& e : q->ev)
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                e = nullptr;
                pppm_set_last_error("group event creation failed", __FILE__, __LINE__);
                return fail(PPPM_ERR_HIP);
            }
    }
    const size_t n = 3 * (size_t)cap * q->G;
    pppm_status s;
    if ((s = dev_alloc(&q->wg, n)) != PPPM_OK || (s = dev_alloc(&q->e32, n)) != PPPM_OK ||
        (s = dev_alloc(&q->r32, n)) != PPPM_OK || (s = dev_alloc(&q->b64, n)) != PPPM_OK ||
        (s = dev_alloc(&q->psi64[0], n)) != PPPM_OK || (s = dev_alloc(&q->psi64[1], n)) != PPPM_OK)
        return fail(s);
    if ((s = q->mg.init((int)g, (int)g, (int)g, 3 * cap)) != PPPM_OK) {
        pppm_set_last_error("group multigrid allocation failed", __FILE__, __LINE__);
        return fail(s);
    }
    q->graphs.resize((size_t)cap);
    q->bytes = group_bytes(g, cap);
    *out = q;
    return PPPM_OK;
}

void group_destroy(pppm_group* q) {
    if (!q) return;
    if (q->st) (void)hipStreamSynchronize(q->st);
    q->release();
    delete q;
}

size_t group_device_bytes(const pppm_group* q) { return q ? q->bytes : 0; }

pppm_status group_compute_far_field(pppm_group* q, pppm_ctx* const* ctxs, int count) {
    if (!q || !ctxs || count < 1 || count > q->cap) FAIL(PPPM_ERR_INVALID, "group count");
    const pppm_params& p = ctxs[0]->p;
    for (int j = 0; j < count; j++) {
        pppm_ctx* c = ctxs[j];
        if (!c || !c->have_vort) FAIL(PPPM_ERR_STATE, "group: set_vortices first");
        if (c->g != q->g || std::memcmp(&c->p, &p, sizeof(p)) != 0) FAIL(PPPM_ERR_INVALID, "group: parameters differ");
    }
    if (!group_eligible(p, q->g)) FAIL(PPPM_ERR_INVALID, "group: mixed precision with the V-cycle schedule only");
    const size_t G = q->G, G3 = 3 * G;
    // each scene's P2M on its own stream, then its grids into the group's slots
    for (int j = 0; j < count; j++) {
        pppm_ctx* c = ctxs[j];
        TRY(far_p2m(c));
        PPPM_HIP_TRY(hipEventRecord(q->ev[j], c->st));
        PPPM_HIP_TRY(hipStreamWaitEvent(q->st, q->ev[j], 0));
        PPPM_HIP_TRY(hipMemcpyAsync(q->wg + j * G3, c->wg, G3 * sizeof(float), hipMemcpyDeviceToDevice, q->st));
        PPPM_HIP_TRY(hipMemcpyAsync(q->b64 + j * G3, c->b64, G3 * sizeof(double), hipMemcpyDeviceToDevice, q->st));
    }
    MixedSolve a;
    a.mg = &q->mg;
    a.e32 = q->e32;
    a.wg = q->wg;
    a.r32 = q->r32;
    a.b64 = q->b64;
    a.psi64[0] = q->psi64[0];
    a.psi64[1] = q->psi64[1];
    a.g = (int)q->g;
    a.scenes = count;
    a.p = &p;
    a.h = ctxs[0]->pg.h;
    a.st = q->st;
    a.graphs = ctxs[0]->use_graphs ? &q->graphs[(size_t)count - 1] : nullptr;
    // a scene's solution goes to its context as soon as its solve ends, before
    // the next step overwrites that psi buffer
    TRY(mixed_solve(a, [&](int j, const SceneResult& r) -> pppm_status {
        pppm_ctx* c = ctxs[j];
        PPPM_HIP_TRY(hipMemcpyAsync(c->psi64[0], q->psi64[r.psi] + j * G3, G3 * sizeof(double),
                                    hipMemcpyDeviceToDevice, q->st));
        c->psi_cur = 0;
        c->stats.mg_cycles = r.inner;
        c->stats.mg_outer = r.outer;
        for (int k = 0; k < 3; k++) c->stats.mg_relres[k] = r.rel[k];
        c->stats.mg_converged = r.converged;
        return PPPM_OK;
    }));
    PPPM_HIP_TRY(hipEventRecord(q->ev[(size_t)q->cap], q->st));
    for (int j = 0; j < count; j++) {
        pppm_ctx* c = ctxs[j];
        PPPM_HIP_TRY(hipStreamWaitEvent(c->st, q->ev[(size_t)q->cap], 0));
        // the group stream has synchronised after every scene's P2M
        c->stats.strays = *c->h_strays;
        TRY(launch_curl_far_impl(c->psi64[0], PPPM_F64, c->wg, c->far, c->dir, c->g, c->p.K, c->pg.h, c->st));
        c->have_far = true;
    }
    return PPPM_OK;
}

// Kernel, core radius, far-field buffer and kernel factor of an evaluation
// other than the context's own (the potential-flow solver's near fields).
struct NearOverride {
    int kernel;
    double core_a;
    const float* far;
    double pot_g;
};

// Evaluation slot -> sorted point in super-block order (nearfield.hip),
// written into the sort's spare index buffer, when the sort keys carry the
// octant (so the spare buffer is free).  Null otherwise: the slots follow the
// sort.  The automatic order renumbers for the potential-flow near fields only,
// and where it pays there: points many enough for the slot pass (at least a
// quarter of the slots, and 4,096) and more gathered bytes (positions and
// strengths, 32 B a source, and the cell tables, 8 B a cell) than twice the
// chip's L2 (8 XCDs x 4 MiB); at 1M sources on 128^3 the sort's order is 7%
// faster.  The vortex near field, whose waves split a union box that wraps
// around a row or plane, takes the sort's order: plumes of 8M on 256^3 11.6
// against 12.9 ms, 33.5M on 512^3 30.3 against 34.4, 1M on 128^3 1.43 against
// 1.62; scattered vortices (uniform, 256^3, 1 / 0.5 / 0.25 / 0.06 a cell) 7.7 / 4.1 /
// 2.6 / 0.55 against 8.7 / 4.0 / 2.1 / 0.57.
static pppm_status super_block_order(pppm_ctx* c, const uint32_t* keys, uint32_t m, uint32_t* spare, bool potential,
                                     uint32_t** perm) {
    *perm = nullptr;
    if (!c->octant_keys() || m == 0 || c->near_order == PPPM_NEAR_ORDER_SORT) return PPPM_OK;
    if (c->near_order == PPPM_NEAR_ORDER_AUTO) {
        constexpr size_t kSbMinGather = (size_t)64 << 20;
        const size_t gather = 32 * (size_t)c->n + 8 * c->G;
        if (!potential || m < 4096 || m < c->sbg.nslots / 4 || gather <= kSbMinGather) return PPPM_OK;
    }
    TRY(launch_sb_order(keys, 3u, m, c->sbg, SbBuffers{c->sb_start, c->sb_len, c->sb_pre, c->sb_scr}, spare, c->st));
    *perm = spare;
    return PPPM_OK;
}

static pppm_status near_common(pppm_ctx* c, uint32_t m, const float4* epos, const float4* eoth,
                               const uint32_t* eidx, const uint32_t* tperm, void* ux, void* uy, void* uz,
                               uint32_t u_stride, int32_t u_dtype, const NearOverride* ov = nullptr) {
    NearArgs a;
    a.tperm = tperm;
    a.epos = epos;
    a.eoth = eoth;
    a.eidx = eidx;
    a.m = m;
    a.off = c->coff;
    a.nsrc = c->n;
    a.spos = c->spos;
    a.somg = c->somg;
    a.far = c->far;
    a.g = c->g;
    a.K = c->p.K;
    a.kernel = c->p.kernel;
    a.invh = c->pg.invh;
    a.core_a = c->p.core_a;
    a.ux = ux;
    a.uy = uy;
    a.uz = uz;
    a.u_stride = u_stride;
    a.u_dtype = u_dtype;
    if (ov) {
        a.kernel = ov->kernel;
        a.core_a = ov->core_a;
        a.far = ov->far;
        a.pot_g = ov->pot_g;
    }
    return launch_m2p_near(a, c->st);
}

extern "C" pppm_status pppm_evaluate_self(pppm_ctx* c, void* ux, void* uy, void* uz, uint32_t u_stride,
                                          int32_t u_dtype) {
    if (!c) FAIL(PPPM_ERR_INVALID, "null ctx");
    if (!c->have_far) FAIL(PPPM_ERR_STATE, "compute_far_field first");
    if (c->n > 0 && (!ux || !uy || !uz)) FAIL(PPPM_ERR_INVALID, "null output");
    if (u_dtype != PPPM_F32 && u_dtype != PPPM_F64) FAIL(PPPM_ERR_INVALID, "u_dtype");
    if (u_stride == 0) FAIL(PPPM_ERR_INVALID, "u_stride");
    c->stats.m = c->n;
    // octant order within cells: from the sort when the keys carry the
    // octant, else ranked into the sort's spare index buffer
    uint32_t* perm = nullptr;
    uint32_t* spare = c->vs.vs == c->vs.v0 ? c->vs.v1 : c->vs.v0;
    if (!c->octant_keys()) {
        perm = spare;
        TRY(launch_octant_order(c->vs.ks, c->spos, c->n, c->pg.invh, perm, c->st));
    } else {
        TRY(super_block_order(c, c->vs.ks, c->n, spare, false, &perm));
    }
    return near_common(c, c->n, c->spos, nullptr, c->vs.vs, perm, ux, uy, uz, u_stride, u_dtype);
}

static pppm_status eval_points(pppm_ctx* c, uint32_t m, const float* eval_pos4, const float* other_end4, void* ux,
                               void* uy, void* uz, uint32_t u_stride, int32_t u_dtype, const NearOverride* ov);

extern "C" pppm_status pppm_evaluate(pppm_ctx* c, uint32_t m, const float* eval_pos4, const float* other_end4,
                                     void* ux, void* uy, void* uz, uint32_t u_stride, int32_t u_dtype) {
    if (!c) FAIL(PPPM_ERR_INVALID, "null ctx");
    if (!c->have_far) FAIL(PPPM_ERR_STATE, "compute_far_field first");
    if (m > 0 && (!eval_pos4 || !ux || !uy || !uz)) FAIL(PPPM_ERR_INVALID, "null array");
    if (u_dtype != PPPM_F32 && u_dtype != PPPM_F64) FAIL(PPPM_ERR_INVALID, "u_dtype");
    if (u_stride == 0) FAIL(PPPM_ERR_INVALID, "u_stride");
    if (m > (1u << 30)) FAIL(PPPM_ERR_INVALID, "too many points");
    return eval_points(c, m, eval_pos4, other_end4, ux, uy, uz, u_stride, u_dtype, nullptr);
}

pppm_status ctx_sources(pppm_ctx* c, CtxSources* out) {
    if (!c || !out || !c->have_vort) FAIL(PPPM_ERR_STATE, "set_vortices first");
    out->st = c->st;
    out->start = c->cstart;
    out->end = c->cend;
    out->idx = c->vs.vs;
    out->n = c->n;
    return PPPM_OK;
}

pppm_status ctx_p2m_x64(pppm_ctx* c, float* wg_scratch, double* out) {
    if (!c || !c->have_vort) FAIL(PPPM_ERR_STATE, "set_vortices first");
    TRY(launch_p2m(c->coff, c->spos, c->somg, c->g, c->pg.invh, wg_scratch, out, 1.0, c->sflag, c->st));
    return launch_p2m_strays(c->coff, c->spos, c->somg, c->g, c->pg.invh, wg_scratch, out, 1.0, c->d_strays, c->sflag,
                             c->st);
}

pppm_status ctx_evaluate_with(pppm_ctx* c, uint32_t m, const float* eval_pos4, int kernel, double core_a,
                              const float* far, double pot_g, void* ux, void* uy, void* uz, uint32_t u_stride,
                              int32_t u_dtype) {
    if (!c || !c->have_vort) FAIL(PPPM_ERR_STATE, "set_vortices first");
    if (m > (1u << 30)) FAIL(PPPM_ERR_INVALID, "too many points");
    NearOverride ov{kernel, core_a, far, pot_g};
    return eval_points(c, m, eval_pos4, nullptr, ux, uy, uz, u_stride, u_dtype, &ov);
}

static pppm_status eval_points(pppm_ctx* c, uint32_t m, const float* eval_pos4, const float* other_end4, void* ux,
                               void* uy, void* uz, uint32_t u_stride, int32_t u_dtype, const NearOverride* ov) {
    hipStream_t st = c->st;
    TRY(c->ensure_eval(m, other_end4 != nullptr));
    const bool ok8 = c->octant_keys();
    TRY(launch_calc_keys((const float4*)eval_pos4, m, c->pg.hash, c->es.k0, nullptr, st, ok8, true));
    TRY(radix_sort_pairs(c->es.k0, c->es.v0, c->es.k1, c->es.v1, m, key_bits_for(c->G) + (ok8 ? 3u : 0u), true,
                         c->es.scratch, &c->es.ks, &c->es.vs, st));
    TRY(launch_reorder_eval(c->es.vs, (const float4*)eval_pos4, (const float4*)other_end4, m, c->pg, c->epos,
                            other_end4 ? c->eoth : nullptr, st));
    c->stats.m = m;
    uint32_t* perm = nullptr;
    uint32_t* spare = c->es.vs == c->es.v0 ? c->es.v1 : c->es.v0;
    if (!ok8) {
        perm = spare;
        TRY(launch_octant_order(c->es.ks, c->epos, m, c->pg.invh, perm, st));
    } else {
        TRY(super_block_order(c, c->es.ks, m, spare, ov != nullptr, &perm));
    }
    return near_common(c, m, c->epos, other_end4 ? c->eoth : nullptr, c->es.vs, perm, ux, uy, uz, u_stride,
                       u_dtype, ov);
}

// add_u_rotation_kernel (GPU_kernel.cu:3589-3606): vel.xyz += u; then, when
// dt is applied, move_particle_kernel (GPU_kernel.cu:3118-3140): the position
// advanced by vel dt in FP64 and stored as float with w = 0.
__global__ void __launch_bounds__(256) k_tracer_update(float4* __restrict__ pos, double4* __restrict__ vel,
                                                       const double* __restrict__ u, uint32_t n, uint32_t cap,
                                                       double dt, int move) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double4 v = vel[i];
    v.x += u[i];
    v.y += u[(size_t)cap + i];
    v.z += u[2 * (size_t)cap + i];
    vel[i] = v;
    if (move) {
        const float4 p = pos[i];
        pos[i] = make_float4((float)((double)p.x + v.x * dt), (float)((double)p.y + v.y * dt),
                             (float)((double)p.z + v.z * dt), 0.0f);
    }
}

extern "C" pppm_status pppm_evaluate_tracers(pppm_ctx* c, uint32_t m, float* pos4, double* vel4, uint32_t batch,
                                             double dt, int32_t move) {
    if (!c) FAIL(PPPM_ERR_INVALID, "null ctx");
    if (!c->have_far) FAIL(PPPM_ERR_STATE, "compute_far_field first");
    if (m > 0 && (!pos4 || !vel4)) FAIL(PPPM_ERR_INVALID, "null array");
    if (batch == 0) FAIL(PPPM_ERR_INVALID, "batch must be > 0");
    const uint32_t cap = batch < m ? batch : (m > 0 ? m : 1);
    if (cap > c->capT || !c->utr) {
        dev_free(c->utr);
        TRY(dev_alloc(&c->utr, 3 * (size_t)cap));
        c->capT = cap;
    }
    for (uint32_t b0 = 0; b0 < m; b0 += cap) {
        const uint32_t nb = m - b0 < cap ? m - b0 : cap;
        double* u = c->utr;
        TRY(pppm_evaluate(c, nb, pos4 + 4 * (size_t)b0, nullptr, u, u + c->capT, u + 2 * (size_t)c->capT, 1,
                          PPPM_F64));
        hipLaunchKernelGGL(k_tracer_update, dim3(div_up(nb, 256)), dim3(256), 0, c->st,
                           reinterpret_cast<float4*>(pos4) + b0, reinterpret_cast<double4*>(vel4) + b0, u, nb,
                           c->capT, dt, move ? 1 : 0);
        PPPM_LAUNCH_CHECK();
    }
    return PPPM_OK;
}

extern "C" pppm_status pppm_smooth_vorticity(pppm_ctx* c, const double* vx, const double* vy, const double* vz,
                                             uint32_t v_stride, double* ox, double* oy, double* oz,
                                             uint32_t o_stride, double nu) {
    if (!c) FAIL(PPPM_ERR_INVALID, "null ctx");
    if (!c->have_vort) FAIL(PPPM_ERR_STATE, "set_vortices first");
    if (v_stride == 0 || o_stride == 0) FAIL(PPPM_ERR_INVALID, "stride");
    if (!(nu > 0)) FAIL(PPPM_ERR_INVALID, "nu must be > 0");
    const uint32_t n = c->n;
    if (n == 0) return PPPM_OK;
    if (!vx || !vy || !vz || !ox || !oy || !oz) FAIL(PPPM_ERR_INVALID, "null array");
    if (n > c->capS || !c->sval) {
        dev_free(c->sval);
        c->capS = 0;
        TRY(dev_alloc(&c->sval, n));
        c->capS = n;
    }
    return launch_gaussian_smooth(c->spos, c->coff, c->vs.vs, n, c->pg, nu, vx, vy, vz, v_stride, ox, oy, oz,
                                  o_stride, c->sval, c->st);
}

extern "C" pppm_status pppm_domain_device(pppm_ctx* c, const float* pos4, uint32_t n, double origin_out[3],
                                          double* h_out) {
    if (!c || !pos4 || n == 0 || !origin_out || !h_out) FAIL(PPPM_ERR_INVALID, "domain_device args");
    if (!c->bbox) TRY(dev_alloc(&c->bbox, bbox_scratch_floats()));
    TRY(launch_bbox((const float4*)pos4, n, c->bbox, c->st));
    float b[6];
    PPPM_HIP_TRY(hipMemcpyAsync(b, c->bbox + bbox_scratch_floats() - 6, sizeof b, hipMemcpyDeviceToHost, c->st));
    PPPM_HIP_TRY(hipStreamSynchronize(c->st));
    return domain_from_extent(b[0], b[3], b[1], b[4], b[2], b[5], c->g, origin_out, h_out);
}

extern "C" pppm_status pppm_time_step(pppm_ctx* c, uint32_t n, float* cent4, double* wx, double* wy, double* wz,
                                      double dt, double seg_h, double nu, int32_t flags) {
    if (!c) FAIL(PPPM_ERR_INVALID, "null ctx");
    if (n == 0) return PPPM_OK;
    if (!cent4 || !wx || !wy || !wz) FAIL(PPPM_ERR_INVALID, "null array");
    if (!(seg_h > 0) || !(nu > 0)) FAIL(PPPM_ERR_INVALID, "seg_h and nu must be > 0");
    if (flags & ~(PPPM_STEP_KEEP_DOMAIN | PPPM_STEP_RK2)) FAIL(PPPM_ERR_INVALID, "unknown step flags");
    const bool move_domain = !(flags & PPPM_STEP_KEEP_DOMAIN);
    const bool rk2 = (flags & PPPM_STEP_RK2) != 0;
    if (n > c->capStep) {
        for (float4** q : {&c->seg_a, &c->seg_b}) dev_free(*q);
        dev_free(c->kappa);
        dev_free(c->dvort);
        dev_free(c->vel_a);
        dev_free(c->vel_b);
        c->capStep = 0;
        TRY(dev_alloc(&c->seg_a, n));
        TRY(dev_alloc(&c->seg_b, n));
        TRY(dev_alloc(&c->kappa, n));
        TRY(dev_alloc(&c->dvort, 3 * (size_t)n));
        TRY(dev_alloc(&c->vel_a, n));
        TRY(dev_alloc(&c->vel_b, n));
        c->capStep = n;
    }
    if (rk2 && n > c->capStep2) {
        for (float4** q : {&c->seg_a2, &c->seg_b2, &c->cent2}) dev_free(*q);
        for (double4** q : {&c->vel_a2, &c->vel_b2}) dev_free(*q);
        dev_free(c->vort2);
        c->capStep2 = 0;
        for (float4** q : {&c->seg_a2, &c->seg_b2, &c->cent2}) TRY(dev_alloc(q, n));
        for (double4** q : {&c->vel_a2, &c->vel_b2}) TRY(dev_alloc(q, n));
        TRY(dev_alloc(&c->vort2, 3 * (size_t)n));
        c->capStep2 = n;
    }
    hipStream_t st = c->st;
    float* a = (float*)c->seg_a;
    float* b = (float*)c->seg_b;
    double* ua = (double*)c->vel_a;
    double* ub = (double*)c->vel_b;
    double* dw[3] = {c->dvort, c->dvort + n, c->dvort + 2 * (size_t)n};
    double* w[3] = {wx, wy, wz};
    // computeURotation: the vortices (centres cc, strengths ww) hashed on
    // their own domain, the far field, then both ends in segment mode (the
    // own vortex excluded), into double4 velocities
    auto end_velocities = [&](const float* cc, double* const* ww, const float* ea, const float* eb, double* va,
                              double* vb) -> pppm_status {
        if (move_domain) {
            double o[3], h;
            TRY(pppm_domain_device(c, cc, n, o, &h));
            TRY(pppm_set_domain(c, o, h));
        }
        TRY(pppm_set_vortices(c, n, cc, ww[0], ww[1], ww[2], 1, PPPM_F64));
        TRY(pppm_compute_far_field(c));
        TRY(pppm_evaluate(c, n, eb, cc, vb, vb + 1, vb + 2, 4, PPPM_F64));
        return pppm_evaluate(c, n, ea, cc, va, va + 1, va + 2, 4, PPPM_F64);
    };
    // convertVortToSeg
    TRY(pppm_segments_from_vortices(cent4, a, b, wx, wy, wz, c->kappa, seg_h, n, st));
    TRY(end_velocities(cent4, w, a, b, ua, ub));
    if (rk2) {
        // Heun: ends predicted with the first velocities, the predicted
        // segments' centres and strengths w + dw (computeStretching's sum),
        // the velocities there, then both ends move with the mean of the two
        float* a2 = (float*)c->seg_a2;
        float* b2 = (float*)c->seg_b2;
        float* c2 = (float*)c->cent2;
        double* w1[3] = {c->vort2, c->vort2 + n, c->vort2 + 2 * (size_t)n};
        PPPM_HIP_TRY(hipMemcpyAsync(a2, a, 16 * (size_t)n, hipMemcpyDeviceToDevice, st));
        PPPM_HIP_TRY(hipMemcpyAsync(b2, b, 16 * (size_t)n, hipMemcpyDeviceToDevice, st));
        PPPM_HIP_TRY(hipMemcpyAsync(c2, cent4, 16 * (size_t)n, hipMemcpyDeviceToDevice, st));
        TRY(pppm_apply_flow(a2, b2, c2, ua, ub, dt, n, st));
        TRY(pppm_vortices_from_segments(a2, b2, wx, wy, wz, dw[0], dw[1], dw[2], c->kappa, n, st));
        for (int q = 0; q < 3; q++) TRY(pppm_vector_add(w[q], dw[q], w1[q], 1.0, 1.0, n, st));
        double* ua2 = (double*)c->vel_a2;
        double* ub2 = (double*)c->vel_b2;
        TRY(end_velocities(c2, w1, a2, b2, ua2, ub2));
        // 4 doubles per velocity, in pieces that fit the 32-bit count
        const size_t n4 = 4 * (size_t)n, piece = (size_t)1 << 30;
        for (size_t o = 0; o < n4; o += piece) {
            const uint32_t m = (uint32_t)std::min(piece, n4 - o);
            TRY(pppm_vector_add(ua + o, ua2 + o, ua + o, 0.5, 0.5, m, st));
            TRY(pppm_vector_add(ub + o, ub2 + o, ub + o, 0.5, 0.5, m, st));
        }
    }
    // applyFlow, convertSegToVort
    TRY(pppm_apply_flow(a, b, cent4, ua, ub, dt, n, st));
    TRY(pppm_vortices_from_segments(a, b, wx, wy, wz, dw[0], dw[1], dw[2], c->kappa, n, st));
    // computeStretching: w + dw smoothed over the new centres' neighbourhoods
    for (int q = 0; q < 3; q++) TRY(pppm_vector_add(w[q], dw[q], dw[q], 1.0, 1.0, n, st));
    if (move_domain) {
        double o[3], h;
        TRY(pppm_domain_device(c, cent4, n, o, &h));
        TRY(pppm_set_domain(c, o, h));
    }
    TRY(pppm_set_vortices(c, n, cent4, dw[0], dw[1], dw[2], 1, PPPM_F64));
    return pppm_smooth_vorticity(c, dw[0], dw[1], dw[2], 1, wx, wy, wz, 1, nu);
}

extern "C" pppm_status pppm_solve_self(pppm_ctx* c, uint32_t n, const float* pos4, const void* wx, const void* wy,
                                       const void* wz, uint32_t w_stride, int32_t w_dtype, void* ux, void* uy,
                                       void* uz, uint32_t u_stride, int32_t u_dtype) {
    TRY(pppm_set_vortices(c, n, pos4, wx, wy, wz, w_stride, w_dtype));
    TRY(pppm_compute_far_field(c));
    return pppm_evaluate_self(c, ux, uy, uz, u_stride, u_dtype);
}

extern "C" pppm_status pppm_count_near_pairs(pppm_ctx* c, uint64_t* pairs) {
    if (!c || !pairs) FAIL(PPPM_ERR_INVALID, "null arg");
    if (!c->have_vort) FAIL(PPPM_ERR_STATE, "set_vortices first");
    unsigned long long* d = nullptr;
    PPPM_HIP_TRY(hipMalloc(&d, sizeof(unsigned long long)));
    NearArgs a{};
    a.epos = c->spos;
    a.m = c->n;
    a.off = c->coff;
    a.nsrc = c->n;
    a.spos = c->spos;
    a.g = c->g;
    a.K = c->p.K;
    a.invh = c->pg.invh;
    hipError_t e = hipMemsetAsync(d, 0, sizeof(unsigned long long), c->st);
    pppm_status s = e == hipSuccess ? launch_count_pairs(a, d, c->st) : PPPM_ERR_HIP;
    unsigned long long h = 0;
    if (s == PPPM_OK) e = hipMemcpyAsync(&h, d, sizeof(h), hipMemcpyDeviceToHost, c->st);
    if (s == PPPM_OK && e == hipSuccess) e = hipStreamSynchronize(c->st);
    (void)hipFree(d);
    if (s != PPPM_OK) return s;
    PPPM_HIP_TRY(e);
    *pairs = h;
    return PPPM_OK;
}

extern "C" pppm_status pppm_get_stats(const pppm_ctx* c, pppm_stats* out) {
    if (!c || !out) FAIL(PPPM_ERR_INVALID, "null arg");
    *out = c->stats;
    return PPPM_OK;
}

extern "C" pppm_status pppm_get_sorted_vortices(pppm_ctx* c, const float** pos4, const uint32_t** sorted_index,
                                                const uint32_t** cell_start, const uint32_t** cell_end) {
    if (!c) FAIL(PPPM_ERR_INVALID, "null ctx");
    if (!c->have_vort) FAIL(PPPM_ERR_STATE, "set_vortices first");
    if (pos4) *pos4 = (const float*)c->spos;
    if (sorted_index) *sorted_index = c->vs.vs;
    if (cell_start) *cell_start = c->cstart;
    if (cell_end) *cell_end = c->cend;
    return PPPM_OK;
}

extern "C" pppm_status pppm_get_grid(pppm_ctx* c, int32_t which, int32_t comp, const void** ptr, int32_t* dtype) {
    if (!c || !ptr || !dtype || comp < 0 || comp > 2) FAIL(PPPM_ERR_INVALID, "get_grid args");
    if (!c->have_far) FAIL(PPPM_ERR_STATE, "compute_far_field first");
    switch (which) {
        case 0:
            *ptr = c->wg + comp * c->G;
            *dtype = PPPM_F32;
            break;
        case 1:
            if (c->p.precision == PPPM_PREC_MIXED) {
                *ptr = c->psi64[c->psi_cur] + comp * c->G;
                *dtype = PPPM_F64;
            } else {
                *ptr = c->psi32 + comp * c->G;
                *dtype = PPPM_F32;
            }
            break;
        case 2:
            *ptr = c->far + comp * c->G;
            *dtype = PPPM_F32;
            break;
        default:
            FAIL(PPPM_ERR_INVALID, "which");
    }
    return PPPM_OK;
}

// ---------------------------------------------------------------------------
// device memory
extern "C" pppm_status pppm_device_count(int32_t* n) {
    int d = 0;
    if (hipGetDeviceCount(&d) != hipSuccess) d = 0;
    (void)hipGetLastError();
    if (n) *n = d;
    return d > 0 ? PPPM_OK : PPPM_ERR_NO_DEVICE;
}
extern "C" pppm_status pppm_malloc(void** ptr, size_t bytes) {
    if (!ptr) FAIL(PPPM_ERR_INVALID, "null ptr");
    std::lock_guard<std::mutex> lk(runtime_mutex());
    if (hipMalloc(ptr, bytes ? bytes : 1) != hipSuccess) {
        *ptr = nullptr;
        (void)hipGetLastError();
        FAIL(PPPM_ERR_NOMEM, "hipMalloc failed");
    }
    return PPPM_OK;
}
extern "C" pppm_status pppm_free(void* ptr) {
    std::lock_guard<std::mutex> lk(runtime_mutex());
    if (ptr) PPPM_HIP_TRY(hipFree(ptr));
    return PPPM_OK;
}
extern "C" pppm_status pppm_memcpy_htod(void* dst, const void* src, size_t bytes) {
    std::lock_guard<std::mutex> lk(runtime_mutex());
    if (bytes) PPPM_HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return PPPM_OK;
}
extern "C" pppm_status pppm_memcpy_dtoh(void* dst, const void* src, size_t bytes) {
    std::lock_guard<std::mutex> lk(runtime_mutex());
    if (bytes) PPPM_HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return PPPM_OK;
}
extern "C" pppm_status pppm_memcpy_dtod(void* dst, const void* src, size_t bytes) {
    std::lock_guard<std::mutex> lk(runtime_mutex());
    if (bytes) PPPM_HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToDevice));
    return PPPM_OK;
}
extern "C" pppm_status pppm_memset(void* dst, int value, size_t bytes) {
    std::lock_guard<std::mutex> lk(runtime_mutex());
    if (bytes) PPPM_HIP_TRY(hipMemset(dst, value, bytes));
    return PPPM_OK;
}
extern "C" pppm_status pppm_synchronize(void) {
    PPPM_HIP_TRY(hipDeviceSynchronize());
    return PPPM_OK;
}

// ---------------------------------------------------------------------------
// timers
struct pppm_timer {
    hipEvent_t a = nullptr, b = nullptr;
};
extern "C" pppm_status pppm_timer_create(pppm_timer** out) {
    if (!out) FAIL(PPPM_ERR_INVALID, "null out");
    pppm_timer* t = new pppm_timer();
    if (hipEventCreate(&t->a) != hipSuccess || hipEventCreate(&t->b) != hipSuccess) {
        delete t;
        FAIL(PPPM_ERR_HIP, "event create failed");
    }
    *out = t;
    return PPPM_OK;
}
extern "C" void pppm_timer_destroy(pppm_timer* t) {
    if (!t) return;
    (void)hipEventDestroy(t->a);
    (void)hipEventDestroy(t->b);
    delete t;
}
extern "C" pppm_status pppm_timer_start(pppm_timer* t, void* s) {
    PPPM_HIP_TRY(hipEventRecord(t->a, (hipStream_t)s));
    return PPPM_OK;
}
extern "C" pppm_status pppm_timer_stop(pppm_timer* t, void* s) {
    PPPM_HIP_TRY(hipEventRecord(t->b, (hipStream_t)s));
    return PPPM_OK;
}
extern "C" pppm_status pppm_timer_elapsed_ms(pppm_timer* t, float* ms) {
    PPPM_HIP_TRY(hipEventSynchronize(t->b));
    PPPM_HIP_TRY(hipEventElapsedTime(ms, t->a, t->b));
    return PPPM_OK;
}
