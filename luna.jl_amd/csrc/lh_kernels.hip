// lh_kernels.hip -- C ABI of the propagation hot path on MI355X (gfx950): contexts,
// batches, streaming, plans; and the kernels that are not in lh_gang.h.
//
// Mode-averaged instances run on gangs of four workgroups (lh_gang.h), those
// with a z-dependent fill on one workgroup (lh_solo_kernel.h), radial ones as a
// launch sequence (lh_radial.hip).  A right-hand side keeps its time series in
// LDS:
//   stage prologue (ȳ = y + Δz Σ B k, ·exp(LΔ)) → c2r pre-pack → inverse
//   Stockham FFT → Kerr + PPT spline + three cumtrapz block scans + towin →
//   forward FFT → r2c post-step, crop, normalisation → stage epilogue
//   (·exp(-LΔ)) written to HBM.
// The adaptive Dormand–Prince loop (controller, window filter, dense-output
// saves) runs inside the same launch, so a whole propagation is one launch and
// a batch of independent instances is one launch per grid size.
//
// Reference semantics (file:line in the reference tree):
//   TransModeAvg              src/NonlinearRHS.jl:362-387
//   to_time!/to_freq!         src/NonlinearRHS.jl:16-53
//   Kerr_field, PlasmaCumtrapz src/Nonlinear.jl:8-10, 24-34, 88-177
//   makePPTaccel + CSpline    src/Ionisation.jl:247-271, src/Maths.jl:771-775, 840-848
//   cumtrapz!                 src/Maths.jl:299-327
//   PreconStepper/step!/evaluate!/interpolate, weaknorm, stepcontrolPI!
//                             src/RK45.jl:128-309, 343-406; tableau src/dopri.jl
//   Luna.run stepfun filter   src/Luna.jl:366-372
//   GridCondition saves       src/Output.jl:65-81, 490-502
#include <hip/hip_runtime.h>

#include <math.h>
#include <pthread.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <functional>
#include <mutex>
#include <queue>
#include <string>
#include <time.h>
#include <vector>

#include "../../include/luna_hip.h"
#include "lh_core.h"
#include "lh_gang_launch.h"
#include "lh_hostcopy.h"
#include "lh_solo.h"

static const long long LH_MAX_STEPS = 500000;  // default cap on step attempts per instance

// hω·δt on the big grid: h zero-padded to 2·NO reals, packed into NO complex
// points in W, transformed, post-stepped into hwdt[0..NO].  One workgroup.
template <int NO>
__global__ __launch_bounds__(LH_T) void lh_raman_hw_big_kernel(const double* __restrict__ h, double dt,
                                                               const double2* __restrict__ twg, double2* work,
                                                               double2* hwdt) {
    __shared__ SmemT<NO / 2> sm;
    tw_load(sm.tw, twg);
    double2* W = work;
    double2* T = work + NO;
    for (int j = threadIdx.x; j < NO; j += LH_T)
        W[j] = (j < NO / 2) ? make_double2(h[2 * j], h[2 * j + 1]) : make_double2(0.0, 0.0);
    fft_big<NO / 2, false>(W, T, sm);
    for (int k = threadIdx.x; k <= NO; k += LH_T) {
        const double2 X = r2c_bin_big<NO>(W, sm, k);
        hwdt[k] = make_double2(X.x * dt, X.y * dt);
    }
}

// hω·δt for the Raman convolution: rfft of h(t) zero-padded to 2·Nto reals
// (the reference's FT * h on the doubled grid, src/Nonlinear.jl:307-312).
template <int NO>
__global__ __launch_bounds__(LH_T) void lh_raman_hw_kernel(const double* __restrict__ h, double dt,
                                                           const double2* __restrict__ twg, double2* hwdt) {
    __shared__ SmemT<NO> sm;
    tw_load(sm.tw, twg);
    for (int j = threadIdx.x; j < NO; j += LH_T)
        sm.buf[pad(j)] = (j < NO / 2) ? make_double2(h[2 * j], h[2 * j + 1]) : make_double2(0.0, 0.0);
    __syncthreads();
    fft_lds<NO, false>(sm.buf, sm.tw);
    for (int k = threadIdx.x; k <= NO; k += LH_T) {
        double2 X = r2c_bin<NO>(sm.buf, sm.tw, k);
        hwdt[k] = make_double2(X.x * dt, X.y * dt);
    }
}

static int size_class_of(int grid_kind, int n_to, int n_t) {
    if (grid_kind == LH_GRID_REAL) {
        if (n_to == 32768 && n_t == 16384) return LH_CLASS_32768;
        if (n_to == 16384 && n_t == 8192) return LH_CLASS_16384;
        if (n_to == 8192 && n_t == 4096) return LH_CLASS_8192;
        if (n_to == 4096 && n_t == 2048) return LH_CLASS_4096;
    } else if (grid_kind == LH_GRID_ENV) {
        if (n_to == 16384 && n_t == 16384) return LH_CLASS_ENV16384;
        if (n_to == 8192 && n_t == 8192) return LH_CLASS_ENV8192;
        if (n_to == 4096 && n_t == 4096) return LH_CLASS_ENV4096;
    }
    return -1;
}

static void launch_raman_hw(int n_to, const double* h, double dt, const double2* tw, double2* hwdt, double2* work,
                            hipStream_t s) {
    if (n_to == 16384) {
        hipLaunchKernelGGL((lh_raman_hw_big_kernel<16384>), dim3(1), dim3(LH_T), 0, s, h, dt, tw, work, hwdt);
        return;
    }
    if (n_to == 8192)
        hipLaunchKernelGGL((lh_raman_hw_kernel<8192>), dim3(1), dim3(LH_T), 0, s, h, dt, tw, hwdt);
    else
        hipLaunchKernelGGL((lh_raman_hw_kernel<4096>), dim3(1), dim3(LH_T), 0, s, h, dt, tw, hwdt);
}

// The gang kernels of a class (raman: its field-grid instances carry a Raman
// response).
static bool is_env_class(int cls) { return cls == LH_CLASS_ENV16384 || cls == LH_CLASS_ENV8192 || cls == LH_CLASS_ENV4096; }
static bool launch_solve(const GangLaunch& l, bool raman, bool stream) {
    if (is_env_class(l.cls)) return lg_env_solve(l, stream);
    return raman ? lg_raman_solve(l, stream) : lg_field_solve(l, stream);
}
static bool launch_rhs(const GangLaunch& l, bool raman, int* status) {
    if (is_env_class(l.cls)) return lg_env_rhs(l, status);
    return raman ? lg_raman_rhs(l, status) : lg_field_rhs(l, status);
}
static bool launch_stats(const GangLaunch& l, double z, double dz, int* status) {
    return is_env_class(l.cls) ? lg_env_stats(l, z, dz, status) : lg_field_stats(l, z, dz, status);
}

// Radially symmetric transform: per-column kernels and FP64 MFMA contraction.
#include "lh_radial.hip"

// ==========================================================================
// Host side: contexts, constant upload, launches (C ABI, include/luna_hip.h)
// ==========================================================================
static const double EPS0 = 8.854187817620389e-12;  // CODATA 2014 ε0
static const double ECHARGE = 1.6021766208e-19;
static const double MELEC = 9.10938356e-31;
static const double CLIGHT = 299792458.0;

// What the single right-hand sides and statistics records launched on one
// stream use: a control block (which each launch leaves ready for the next), a
// status word, an exchange area and, on a field grid with Raman, its series; in
// z, the operator and output factor of a z-dependent fill.  A set belongs to
// one stream, so launches on different streams share nothing, and launches on
// one follow each other.  Launches under capture have one of their own: which
// streams replay a graph, and beside what, is not known when it is recorded.
// That set and one more are there from the start.
struct RhsSet {
    hipStream_t s;
    unsigned long long thread;  // of hipStreamPerThread, one handle for every thread's stream
    unsigned long long used;    // of the context's launches, the last here
    unsigned char* block;
    double2* z;
};
enum { RHS_CAPTURED, RHS_FIRST, RHS_SETS = RHS_FIRST + 5 };

struct lh_ctx {
    int device;
    hipStream_t stream;
    lh_desc d;  // scalars only; host pointers cleared after upload
    int n_state;
    double ppt_emin, ppt_emax;
    double* omega_win;
    double* t_win;
    double* to_win;
    double2* linop;
    double2* outfac;
    double4* ppt;
    double2* hwdt;  // envelope Raman: rfft(h, 2·Nto)·δt
    double2* escr;  // field-grid Raman: E(t) and P(t), Nto/2 points each, of solves
    double2* gx;    // exchange area of the gang, of solves
    // solver buffers (allocated on first use)
    double2* Yin;
    int have_state;
    double amp;  // root of the initial field's energy (in its time units), for solve_cost
    int have_result;
    int result_save_n;
    double2* Y;
    double2* YN;
    double2* K;   // work block: vector j at K + j·kstride (radial: 7 and one, gangs: LgVec)
    long long kstride;
    double2* K1;  // the nine vectors of a solver with one workgroup, at K1 + j·k1stride
    long long k1stride;
    double2* saves;
    int saves_cap;
    double* zgrid;
    int zgrid_cap;
    double* zgrid_h;  // host copy of the save grid in zgrid (an unchanged grid is not uploaded again)
    int zgrid_hn;
    RunStats* dstats;
    unsigned char* launch1;  // one instance's solve: control block, then its DInst
    unsigned* beat;          // the device's
    RhsSet rset[RHS_SETS];
    unsigned long long rhs_calls;
    hipStream_t cap_stream;      // of the last launch under capture, and its capture
    unsigned long long cap_id;
    hipEvent_t cap_ev;
    double2* rhs_in;
    double2* rhs_out;
    int* dstatus;                // of the last right-hand side or record (mode-averaged: its set's)
    int last_status;
    int rhs_pending;
    hipStream_t rhs_stream;
    // radial transform
    double* Mt;          // transposed QDHT matrix
    double* Ek;          // [Nr][Nto] time series per k column
    double* Er;          // [Nr][Nto] time series per r column
    double* partial;     // [Nr][3] weaknorm partial sums
    DInst* pw;           // pointwise parameters (e_scale = 1)
    RadArgs* rargs;      // [0]: solver, [1]: single RHS
    RadCtl* rctl;        // [0]: solver, [1]: single RHS
    hipGraphExec_t rgraph;
    RadPlan rplan;       // variant of the RHS launch sequence
    int rplan_own;       // from the wisdom or lh_set_plan, else the default
    // per-step statistics
    double* omega;       // [Nω] ω (shared)
    double* st_ew;       // [Nω] energy weights (shared)
    double* st_t;        // [Nt] grid.t (shared)
    double* st_win;      // [st_nwin][Nω] window weights (shared)
    int st_nwin;
    double st_aeff, st_ediv;
    int st_on, st_cap;
    double* steprec;     // [st_cap][LH_NSTAT]
    double* st_rec1;     // [LH_NSTAT], lh_stats_eval
    int result_nrec;     // records kept by the last solve
    int have_records;    // the last solve (lh_batch_solve* or lh_solve_noalloc) ran
    // gradient fill
    int zg_on, zg_np, zg_two, zg_model, zg_loss, zd_n;
    double zsqrt_aeff, zfd_h;
    double *zg_Z, *zg_P, *zfd, *zgam;  // shared
    double4* zd;                       // shared
    double2 *znwg, *zpre;              // shared
    unsigned char* zsidx;              // shared
    double2 *zL, *zOF;                 // per context, of solves
    int zg_taper;                      // 1 linear, 2 piecewise-linear taper
    double zg_a0, zg_a1, zg_aL, zg_sqrt_intg;
    int zt_n;
    double *zt_Z, *zt_A;               // shared
    double *zU, *zfdt;                 // shared
    double2* zV;                       // shared
};

static std::mutex g_mu;
static double2* g_tw[64] = {nullptr};
static double2* g_gtw[64] = {nullptr};

// Working memory of lh_solve_noalloc: one fixed array per GPU, held until the
// process ends.  Its name is a host-side stand-in, not a device address; host
// code uses only the per-device address that hipGetSymbolAddress returns
// (g_scratch, set once per device by lh_create with that device current).
static constexpr size_t SCRATCH_BYTES = LH_NOALLOC_SCRATCH_BYTES + (1024u * 1024u);
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];
static unsigned char* g_scratch[64] = {nullptr};
// The word of each GPU that its solvers change as they get on (GangCtl::beat).
static __device__ unsigned beat;
static unsigned* g_beat[64] = {nullptr};
// HIP-event durations of the last resident batch and its kernels (LH_KIND_*), per size class
static float g_last_ms[8] = {0};
static int g_last_n[8] = {0};
static int g_last_kind[8] = {0};

#define HIPCK(x)                                                                     \
    do {                                                                             \
        hipError_t e_ = (x);                                                         \
        if (e_ != hipSuccess) {                                                      \
            fprintf(stderr, "luna_hip: %s failed: %s\n", #x, hipGetErrorString(e_)); \
            return (e_ == hipErrorOutOfMemory) ? LH_E_NOMEM : LH_E_HIP;              \
        }                                                                            \
    } while (0)

// cos and sin of 2π m/N built from the first octant, so values on the axes are
// exact (0, ±1) and the table is symmetric to the last bit.
static void sincos_frac(long m, long N, double* c, double* s) {
    const long double tau = 6.283185307179586476925286766559005768L;
    m %= N;
    if (m < 0) m += N;
    long oct = (8 * m) / N;
    long f = m - oct * (N / 8);
    if (f == 0 && oct % 2 == 0) {
        const double ax[4][2] = {{1, 0}, {0, 1}, {-1, 0}, {0, -1}};
        *c = ax[oct / 2][0];
        *s = ax[oct / 2][1];
        return;
    }
    long double phi = tau * (long double)f / (long double)N;
    long double phip = tau * (long double)(N / 8 - f) / (long double)N;
    long double cp = cosl(phi), sp = sinl(phi), cq = cosl(phip), sq = sinl(phip);
    long double C, S;
    switch (oct) {
        case 0: C = cp; S = sp; break;
        case 1: C = sq; S = cq; break;
        case 2: C = -sp; S = cp; break;
        case 3: C = -cq; S = sq; break;
        case 4: C = -cp; S = -sp; break;
        case 5: C = -sq; S = -cq; break;
        case 6: C = sp; S = -cp; break;
        default: C = cq; S = -sq; break;
    }
    *c = (double)C;
    *s = (double)S;
}

// Device addresses of `scratch` and `beat` on dev (the current device), looked up once.
static int scratch_init(int dev) {
    std::lock_guard<std::mutex> g(g_mu);
    if (dev < 0 || dev >= 64) return LH_E_ARG;
    if (!g_scratch[dev]) {
        void* p = nullptr;
        HIPCK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        void* b = nullptr;
        HIPCK(hipGetSymbolAddress(&b, HIP_SYMBOL(beat)));
        if (!p || !b) return LH_E_HIP;
        g_beat[dev] = (unsigned*)b;
        g_scratch[dev] = (unsigned char*)p;
    }
    return LH_OK;
}

// Global twiddle tables exp(-2πi m/n), one of each length per device: LH_TWN
// for the column transforms, LG_TWN for the gangs'.
static int twiddle_table(double2** table, int dev, int n, const double2** out) {
    std::lock_guard<std::mutex> g(g_mu);
    if (dev < 0 || dev >= 64) return LH_E_ARG;
    if (!table[dev]) {
        std::vector<double2> h(n);
        for (int m = 0; m < n; m++) {
            double c, s;
            sincos_frac(m, n, &c, &s);
            h[m] = make_double2(c, -s);
        }
        double2* d = nullptr;
        HIPCK(hipMalloc(&d, sizeof(double2) * n));
        HIPCK(hipMemcpy(d, h.data(), sizeof(double2) * n, hipMemcpyHostToDevice));
        table[dev] = d;
    }
    *out = table[dev];
    return LH_OK;
}
static int twiddles(int dev, const double2** out) { return twiddle_table(g_tw, dev, LH_TWN, out); }
static int gang_twiddles(int dev, const double2** out) { return twiddle_table(g_gtw, dev, LG_TWN, out); }

// Constants that many contexts share (a scan's PPT table, the windows of one
// grid) are uploaded once per device and reference-counted: identical content
// maps to one device buffer, which then stays resident in the L2/MALL caches
// for every instance of a batch instead of one private copy each.
// A twiddle table and the scratch address of dev as the set-up left them; null
// if there is none (nothing is allocated here).
static const double2* table_existing(double2* const* table, int dev) {
    std::lock_guard<std::mutex> g(g_mu);
    return (dev >= 0 && dev < 64) ? table[dev] : nullptr;
}
static unsigned char* scratch_existing(int dev) {
    std::lock_guard<std::mutex> g(g_mu);
    return (dev >= 0 && dev < 64) ? g_scratch[dev] : nullptr;
}

struct SharedBuf {
    int device;
    uint64_t hash;
    std::vector<unsigned char> host;  // content, for an exact match
    void* dev;
    int refs;
};
static std::vector<SharedBuf*> g_shared;

static uint64_t fnv1a(const void* p, size_t n) {
    const unsigned char* b = (const unsigned char*)p;
    uint64_t h = 1469598103934665603ULL;
    for (size_t i = 0; i < n; i++) h = (h ^ b[i]) * 1099511628211ULL;
    return h;
}

template <class T>
static int shared_upload(int device, T** dst, const void* src, size_t count) {
    *dst = nullptr;
    if (!src || count == 0) return LH_OK;
    const size_t bytes = sizeof(T) * count;
    const uint64_t h = fnv1a(src, bytes);
    std::lock_guard<std::mutex> g(g_mu);
    for (SharedBuf* e : g_shared)
        if (e->device == device && e->hash == h && e->host.size() == bytes && !memcmp(e->host.data(), src, bytes)) {
            e->refs++;
            *dst = (T*)e->dev;
            return LH_OK;
        }
    void* d = nullptr;
    HIPCK(hipMalloc(&d, bytes));
    if (hipMemcpy(d, src, bytes, hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(d);
        return LH_E_HIP;
    }
    SharedBuf* e = new SharedBuf{device, h, std::vector<unsigned char>((const unsigned char*)src, (const unsigned char*)src + bytes), d, 1};
    g_shared.push_back(e);
    *dst = (T*)d;
    return LH_OK;
}

static void shared_release(const void* dev) {
    if (!dev) return;
    std::lock_guard<std::mutex> g(g_mu);
    for (size_t i = 0; i < g_shared.size(); i++)
        if (g_shared[i]->dev == dev) {
            if (--g_shared[i]->refs == 0) {
                (void)hipFree(g_shared[i]->dev);
                delete g_shared[i];
                g_shared.erase(g_shared.begin() + i);
            }
            return;
        }
}

template <class T>
static int upload(T** dst, const void* src, size_t count) {
    *dst = nullptr;
    if (!src || count == 0) return LH_OK;
    HIPCK(hipMalloc((void**)dst, sizeof(T) * count));
    HIPCK(hipMemcpy(*dst, src, sizeof(T) * count, hipMemcpyHostToDevice));
    return LH_OK;
}


static int ctx_class(const lh_ctx* c);

static bool supported(const lh_desc* d) {
    if (d->transform == LH_TRANS_RADIAL) {
        // Nr a multiple of the 64-wide contraction tile; field grid with Kerr and
        // PPT plasma, or envelope grid (Nt = Nto) with Kerr_env
        if (d->n_r < 64 || d->n_r > 4096 || d->n_r % 64 != 0 || d->raman || d->qdht == nullptr) return false;
        if (d->grid_kind == LH_GRID_ENV)
            return rad_env_size_ok(d->n_to) && d->n_t == d->n_to && d->n_omega == d->n_t && !d->plasma &&
                   d->kerr != LH_KERR_FIELD;
        return d->grid_kind == LH_GRID_REAL && rad_size_ok(d->n_to) && d->n_t == d->n_to / 2 &&
               d->n_omega == d->n_t / 2 + 1 && d->kerr != LH_KERR_ENV;
    }
    if (d->transform != LH_TRANS_MODEAVG || d->n_r != 1) return false;
    if (size_class_of(d->grid_kind, d->n_to, d->n_t) < 0) return false;
    if (d->grid_kind == LH_GRID_REAL) {
        if (d->n_omega != d->n_t / 2 + 1) return false;
        if ((d->raman && !d->raman_h) || d->kerr == LH_KERR_ENV) return false;
    } else {
        if (d->n_omega != d->n_t) return false;
        if (d->plasma || d->kerr == LH_KERR_FIELD) return false;
        if (d->raman && !d->raman_h) return false;
    }
    return true;
}

// to_time!/to_freq! length-ratio scales, src/NonlinearRHS.jl:16-53.
static double scale_to_time(const lh_desc& d) {
    if (d.grid_kind == LH_GRID_REAL) return (double)(d.n_to / 2) / (double)(d.n_omega - 1);
    return (double)d.n_to / (double)d.n_omega;
}
static double scale_to_freq(const lh_desc& d) {
    if (d.grid_kind == LH_GRID_REAL) return (double)(d.n_omega - 1) / (double)(d.n_to / 2);
    return (double)d.n_omega / (double)d.n_to;
}

static int ctx_class(const lh_ctx* c) {
    if (c->d.transform == LH_TRANS_RADIAL) return LH_CLASS_RADIAL;
    return size_class_of(c->d.grid_kind, c->d.n_to, c->d.n_t);
}

static DInst base_inst(const lh_ctx* c) {
    DInst in;
    memset(&in, 0, sizeof(in));
    const lh_desc& d = c->d;
    in.grid_kind = d.grid_kind;
    in.transform = d.transform;
    in.n_omega = d.n_omega;
    in.n_t = d.n_t;
    in.n_to = d.n_to;
    in.n_r = d.n_r;
    in.kerr = d.kerr;
    in.plasma = d.plasma;
    in.raman = d.raman;
    in.ppt_n = d.ppt_n;
    in.density = d.density;
    in.kerr_fac = d.density * EPS0 * d.gamma3;  // (ρ ε0) γ3, Nonlinear.jl:30
    in.kerr34 = 0.75 * in.kerr_fac;             // 3/4·fac, Nonlinear.jl:48
    in.inv_2n = 1.0 / (2.0 * (double)d.n_to);
    in.hwdt = c->hwdt;
    in.escr = c->escr;
    in.gx = c->gx;
    in.gx_len = (int)lg_exchange_len(d);
    in.beat = c->beat;
    in.ionpot = d.ionpot;
    in.preion_p1 = d.preionfrac + 1;
    in.e_ratio = ECHARGE * ECHARGE / MELEC;
    in.dt_o = d.dt_o;
    in.e_scale = (1.0 / (double)d.n_to) / d.field_div;  // E = c2r/Nto/(nlscale·√Aeff)
    in.inv_nt = 1.0 / (double)d.n_t;
    in.sc_t = scale_to_time(d);
    in.ppt_emin = c->ppt_emin;
    in.ppt_emax = c->ppt_emax;
    in.omega_win = c->omega_win;
    in.t_win = c->t_win;
    in.to_win = c->to_win;
    in.linop = c->linop;
    in.outfac = c->outfac;
    in.ppt = c->ppt;
    in.st_omega = c->omega;
    in.st_ew = c->st_ew;
    in.st_t = c->st_t;
    in.st_aeff = c->st_aeff;
    in.st_ediv = c->st_ediv;
    in.st_win = c->st_win;
    in.st_nwin = c->st_nwin;
    in.steprec = c->st_on ? c->steprec : nullptr;
    in.steprec_cap = c->st_on ? c->st_cap : 0;
    in.sc_f = scale_to_freq(d);
    in.kerr_gamma3 = (d.kerr == LH_KERR_FIELD) ? d.gamma3 : 0.0;
    if (c->zg_on) {
        in.zg_np = c->zg_np;
        in.zg_two = c->zg_two;
        in.zg_model = c->zg_model;
        in.zg_loss = c->zg_loss;
        in.zd_n = c->zd_n;
        in.zsqrt_aeff = c->zsqrt_aeff;
        in.zfd_h = c->zfd_h;
        in.zg_Z = c->zg_Z;
        in.zg_P = c->zg_P;
        in.zd = c->zd;
        in.zgam = c->zgam;
        in.znwg = c->znwg;
        in.zpre = c->zpre;
        in.zsidx = c->zsidx;
        in.zfd = c->zfd;
        in.ztaper = c->zg_taper;
        in.za0 = c->zg_a0;
        in.za1 = c->zg_a1;
        in.zaL = c->zg_aL;
        in.zsqrt_intg = c->zg_sqrt_intg;
        in.zt_n = c->zt_n;
        in.zt_Z = c->zt_Z;
        in.zt_A = c->zt_A;
        in.zU = c->zU;
        in.zV = c->zV;
        in.zfdt = c->zfdt;
        in.zL = c->zL;
        in.zOF = c->zOF;
        in.linop = c->zL;  // refreshed in place at every new z (lh_solo_kernel.h)
        in.outfac = c->zOF;
    }
    return in;
}

// The counters of an instance until its solver writes them: what a launch whose
// gangs never form leaves.
__host__ __device__ static RunStats unsolved(const DInst& in) {
    return RunStats{{0, 0, 0, 0, LH_E_HIP, in.save_first, in.z0, in.init_dz}, 0, 0};
}
static lh_stats solved(const RunStats& r) {
    lh_stats s = r.s;
    if (r.lost) s.status = LH_E_HIP;
    return s;
}

// A launch over one instance: its control block, then its DInst.  A kernel that
// has them by value puts them there, in stream order, so no host memory has to
// outlive the call.
static constexpr size_t LAUNCH1_CTL = (lg_ctl_bytes(1, LG_MIN_WG) + 255) / 256 * 256;
static constexpr size_t LAUNCH1_BYTES = LAUNCH1_CTL + (sizeof(DInst) + 255) / 256 * 256;
__device__ __forceinline__ void lg_ctl_clear(unsigned* ctl, size_t bytes, const unsigned* beat) {
    for (int i = threadIdx.x; i < (int)(bytes / sizeof(unsigned)); i += 64) ctl[i] = 0u;
    __syncthreads();
    if (threadIdx.x != 0) return;
    ((GangCtl*)ctl)->njobs = 1;
    ((GangCtl*)ctl)->n_wg = LG_MIN_WG;
    ((GangCtl*)ctl)->beat = beat;
}
__global__ __launch_bounds__(64) void lh_set_launch1(DInst in, unsigned char* at) {
    lg_ctl_clear((unsigned*)at, LAUNCH1_CTL, in.beat);
    if (threadIdx.x != 0) return;
    *(DInst*)(at + LAUNCH1_CTL) = in;
    *in.stats = unsolved(in);
}
static int set_launch1(unsigned char* at, const DInst& in, hipStream_t s) {
    hipLaunchKernelGGL(lh_set_launch1, dim3(1), dim3(64), 0, s, in, at);
    HIPCK(hipGetLastError());
    return LH_OK;
}

static GangLaunch launch1_of(const lh_ctx* c, unsigned char* at, const double2* tw, hipStream_t s) {
    return {ctx_class(c), LG_MIN_WG, (GangCtl*)at, (const DInst*)(at + LAUNCH1_CTL), tw, s};
}

static bool field_raman(const lh_desc& d) {
    return d.transform == LH_TRANS_MODEAVG && d.grid_kind == LH_GRID_REAL && d.raman;
}
static constexpr size_t RHS_STATUS = LAUNCH1_CTL, RHS_GX = LAUNCH1_CTL + 256;
__global__ __launch_bounds__(64) void lh_clear_ctl(unsigned* ctl, const unsigned* beat) {
    lg_ctl_clear(ctl, LAUNCH1_CTL, beat);
}
static size_t rhs_block_bytes(const lh_ctx* c) {
    return RHS_GX + sizeof(double2) * (lg_area_len(c->d) + (field_raman(c->d) ? (size_t)c->d.n_to : 0));
}
// Makes a set ready for launches on s (ordered on s; allocates what is missing).
static int rhs_set_ready(lh_ctx* c, RhsSet* r, hipStream_t s) {
    if (!r->block) {
        HIPCK(hipMalloc(&r->block, rhs_block_bytes(c)));
        hipLaunchKernelGGL(lh_clear_ctl, dim3(1), dim3(64), 0, s, (unsigned*)r->block, c->beat);
        HIPCK(hipGetLastError());
    }
    if (c->zg_on && !r->z) HIPCK(hipMalloc(&r->z, sizeof(double2) * 2 * lg_stride(c->d)));
    return LH_OK;
}
// The first two sets.  Their control blocks are copied: a kernel would bind the
// context's stream to a hardware queue, which takes a millisecond.
static int rhs_sets_init(lh_ctx* c) {
    alignas(256) unsigned char h[RHS_GX] = {};
    lg_ctl_init(h, 1, LG_MIN_WG, c->beat);
    for (const int i : {RHS_FIRST, RHS_CAPTURED}) {
        if (hipMalloc(&c->rset[i].block, rhs_block_bytes(c)) != hipSuccess) return LH_E_NOMEM;
        HIPCK(hipMemcpy(c->rset[i].block, h, sizeof(h), hipMemcpyHostToDevice));
    }
    return LH_OK;
}

// The set of a launch on s.  A capture that forks runs its branches side by
// side: a launch on another of its streams than the last one follows that one
// inside the graph.
static int rhs_set_of(lh_ctx* c, hipStream_t s, RhsSet** out) {
    if (s != c->stream) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        unsigned long long id = 0;
        HIPCK(hipStreamGetCaptureInfo(s, &cs, &id));
        if (cs != hipStreamCaptureStatusNone) {
            if (c->cap_stream && c->cap_id == id && c->cap_stream != s) {
                if (!c->cap_ev) HIPCK(hipEventCreateWithFlags(&c->cap_ev, hipEventDisableTiming));
                HIPCK(hipEventRecord(c->cap_ev, c->cap_stream));
                HIPCK(hipStreamWaitEvent(s, c->cap_ev, 0));
            }
            c->cap_stream = s;
            c->cap_id = id;
            *out = &c->rset[RHS_CAPTURED];
            return LH_OK;  // ready since lh_create or lh_set_gradient
        }
    }
    const unsigned long long thread = s == hipStreamPerThread ? (unsigned long long)pthread_self() : 0;
    RhsSet* r = nullptr;
    for (int i = RHS_FIRST; i < RHS_SETS && !r; i++)
        if (c->rset[i].used && c->rset[i].s == s && c->rset[i].thread == thread) r = &c->rset[i];
    if (!r) {  // a stream not seen yet: an unused set, or the one unused for longest once its launches are done
        r = &c->rset[RHS_FIRST];
        for (int i = RHS_FIRST + 1; i < RHS_SETS; i++)
            if (c->rset[i].used < r->used) r = &c->rset[i];
        if (r->used) HIPCK(hipDeviceSynchronize());
        r->s = s;
        r->thread = thread;
    }
    r->used = ++c->rhs_calls;
    *out = r;
    return rhs_set_ready(c, r, s);
}

// A single right-hand side or record on stream s: *in gets the memory of the
// stream's set.
static int rhs_launch_of(lh_ctx* c, DInst* in, const double2* tw, hipStream_t s, GangLaunch* l) {
    RhsSet* r;
    const int st = rhs_set_of(c, s, &r);
    if (st) return st;
    in->gx = (double2*)(r->block + RHS_GX);
    if (in->escr) in->escr = in->gx + lg_area_len(c->d);
    if (c->zg_on) {
        in->zL = r->z;
        in->zOF = r->z + lg_stride(c->d);
    }
    c->dstatus = (int*)(r->block + RHS_STATUS);
    *l = {ctx_class(c), LG_MIN_WG, (GangCtl*)r->block, in, tw, s};
    return LH_OK;
}

// Per-context solver buffers sized for n_state and save_n.
// alone: for a solver with one workgroup (lh_solo_kernel.h), whose vectors have a
// block of their own: in the first nine slots of the gang's, with its unused rest
// between the instances, 256 envelope instances of 4096 points took 12.6 to
// 13.1 ms instead of 11.9 (such a batch just fills the last-level cache).
static int ensure_solver_buffers(lh_ctx* c, int save_n, bool want_saves, bool alone) {
    const size_t NS = (size_t)c->n_state, NS16 = (NS + 15) & ~(size_t)15;  // vectors on 256-byte boundaries
    const bool radial = c->d.transform == LH_TRANS_RADIAL;
    if (!c->Y) {
        HIPCK(hipMalloc(&c->Yin, sizeof(double2) * NS));
        HIPCK(hipMalloc(&c->Y, sizeof(double2) * NS));
        if (radial) HIPCK(hipMalloc(&c->YN, sizeof(double2) * NS));
    }
    if (alone && !c->K1) {
        HIPCK(hipMalloc(&c->K1, sizeof(double2) * NS16 * 9));
        c->k1stride = (long long)NS16;
    }
    if (!alone && !c->K) {
        const size_t stride = radial ? NS16 : lg_stride(c->d);
        HIPCK(hipMalloc(&c->K, sizeof(double2) * stride * (radial ? 8 : LG_SLOTS)));
        c->kstride = (long long)stride;
    }
    if (want_saves && save_n > c->saves_cap) {
        if (c->saves) HIPCK(hipFree(c->saves));
        c->saves = nullptr;
        HIPCK(hipMalloc(&c->saves, sizeof(double2) * NS * (size_t)save_n));
        c->saves_cap = save_n;
    }
    int zn = save_n > 0 ? save_n : 1;
    if (zn > c->zgrid_cap) {
        if (c->zgrid) HIPCK(hipFree(c->zgrid));
        c->zgrid = nullptr;
        c->zgrid_hn = 0;
        HIPCK(hipMalloc(&c->zgrid, sizeof(double) * (size_t)zn));
        c->zgrid_cap = zn;
    }
    return LH_OK;
}

// range(save_z0, stop=zmax, length=n) as Julia evaluates it (correctly rounded
// lerp): GridCondition(tmin, tmax, saveN), src/Output.jl:490-496.
static double save_grid_at(const lh_rk_opts* o, int i) {
    const int n = o->save_n;
    const long double a = o->save_z0, b = o->zmax;
    if (n <= 1) return o->save_z0;
    return (double)((a * (long double)(n - 1 - i) + b * (long double)i) / (long double)(n - 1));
}

static void save_grid_into(const lh_rk_opts* o, double* g) {
    const int n = o->save_n > 0 ? o->save_n : 1;
    for (int i = 0; i < n; i++) g[i] = save_grid_at(o, i);
}

static void save_grid(const lh_rk_opts* o, std::vector<double>& g) {
    g.assign(o->save_n > 0 ? o->save_n : 1, o->save_z0);
    save_grid_into(o, g.data());
}

static bool opts_ok(const lh_rk_opts* o) {
    return o->save_n >= 0 && o->repeat_limit >= 0 && o->rtol > 0 && o->zmax >= o->z0 && o->save_first >= 0 &&
           o->save_first <= o->save_n && o->max_steps >= 0 && o->zstop >= 0 && (o->every_step == 0 || o->every_step == 1);
}

static void inst_options(DInst* in, const lh_rk_opts* o) {
    in->z0 = o->z0;
    in->zmax = o->zmax;
    in->rtol = o->rtol;
    in->atol = o->atol;
    in->safety = o->safety;
    in->max_dz = o->max_dz;
    in->min_dz = o->min_dz;
    in->init_dz = o->init_dz;
    in->repeat_limit = o->repeat_limit;
    in->save_n = o->save_n;
    in->save_first = o->save_first;
    in->zstop = o->zstop;
    in->max_steps = o->max_steps > 0 ? o->max_steps : LH_MAX_STEPS;
}

// Expected cost of a solve relative to others, for the order of a batch only:
// the nonlinear phase per length and the class's time per right-hand side.  The
// steps of a capillary sweep (256 points over energy and pressure) correlate
// with amplitude·density to 0.9996.
static double class_us(int cls) {
    switch (cls) {
        case LH_CLASS_32768: return 50.0;
        case LH_CLASS_16384: return 28.0;
        case LH_CLASS_8192: return 21.0;
        case LH_CLASS_ENV16384: return 42.0;
        case LH_CLASS_ENV8192: return 26.0;
        default: return 18.0;
    }
}
static double solve_cost(const lh_ctx* c, const lh_rk_opts* o) {
    const double x = fabs(c->amp * c->d.density * c->d.gamma3) * (o->zmax - o->z0);
    return isfinite(x) ? x * class_us(ctx_class(c)) : 0.0;
}

// Whether the constant-fill instances of a batch run on one workgroup each
// (lh_solo_kernel.h) instead of on gangs.  Both ways are priced with the
// estimated lengths of their runs (a run without nonlinear phase still takes a
// tenth of the longest one's steps), dealt longest first to the places there
// are: 256 workgroups alone, 64 gangs or 128 dense ones.  Equal instances come in
// rounds: 65 to 128 of them occupy 64 gangs as long as 128 do.  µs per
// right-hand side, one workgroup 23.4, 37.4, 63.7 at Nto = 4096, 8192, 16384;
// gangs, per instance on the whole chip, 0.275, 0.31, 0.455 at one workgroup per
// CU and 0.241, 0.26, 0.382 on dense kernels; the other entries of solo_price
// likewise (with a Raman response; the envelope grid of 4096 points).  Field
// grids without an entry, and envelope grids of 8192 points and more, have no
// kernel for one workgroup: at 16 to 512 equal instances gangs took 0.2 to 0.97
// of the time that one did when it had.  The estimates of field grids, of those
// with a Raman response and of envelope grids cannot be compared, so a batch with
// more than one of them stays on gangs.
// Equal instances, ms alone / on gangs: Nto = 4096, 72 3.3/5.9; 8192, 72 5.3/6.5;
// 16384, 72 9.8/9.7; Raman 4096, 72 12.2/14.7, 8192, 72 21.9/17.9, 176 24.2/28.5;
// envelope 4096, 72 10.5/9.0; 256 of each field grid 3.8, 6.1, 10.4 against 10.1,
// 10.9, 16.0.  Energies and pressures at random: 8192, 160 10.5/10.0, 176
// 10.6/11.3, 256 11.1/14.8; 16384, 224 19.4/18.9, 256 20.0/20.3; 4096, 128
// 6.1/8.4; sweeps over both, 256 20.9/17.2, 300 21.6/20.2, 384 22.1/25.1, 512
// 24.0/31.9: the rule takes the faster way in each.  It depends on the batch
// alone, so a batch gives the same bits every time; what the two ways differ by
// is with lh_batch_solve in luna_hip.h.
struct SoloPrice {
    double alone, gang, dense;  // µs: alone per right-hand side, on gangs per instance
};
static bool solo_price(const lh_ctx* c, SoloPrice* p) {
    if (c->d.transform != LH_TRANS_MODEAVG || c->zg_on) return false;
    const int cls = ctx_class(c);
    if (cls == LH_CLASS_ENV4096) return *p = {53.5, 0.341, 0}, true;
    if (c->d.grid_kind != LH_GRID_REAL) return false;
    if (c->d.raman) {
        if (cls == LH_CLASS_8192) return *p = {90.0, 0.511, 0}, true;
        if (cls == LH_CLASS_4096) return *p = {48.4, 0.404, 0}, true;
        return false;
    }
    if (cls == LH_CLASS_16384) return *p = {63.7, 0.455, 0.382}, true;
    if (cls == LH_CLASS_8192) return *p = {37.4, 0.31, 0.26}, true;
    if (cls == LH_CLASS_4096) return *p = {23.4, 0.275, 0.241}, true;
    return false;
}
// When the last of these runs ends, dealt longest first to so many places.
static double dealt(std::vector<double>& w, int places) {
    std::sort(w.begin(), w.end(), std::greater<double>());
    std::priority_queue<double, std::vector<double>, std::greater<double>> free_at;
    double end = 0.0;
    for (double x : w) {
        if ((int)free_at.size() == places) {
            x += free_at.top();
            free_at.pop();
        }
        free_at.push(x);
        end = std::max(end, x);
    }
    return end;
}
static bool solo_pays(lh_ctx* const* ctxs, const lh_rk_opts* const* op, int n) {
    constexpr int GANGS = LG_MAX_WG / LG_G;
    std::vector<double> cost;
    std::vector<SoloPrice> price;
    SoloPrice p;
    bool kind[3] = {false, false, false};
    int n_dense = 0;
    for (int i = 0; i < n; i++) {
        const lh_desc& d = ctxs[i]->d;
        if (d.transform == LH_TRANS_MODEAVG && !ctxs[i]->zg_on) kind[d.grid_kind == LH_GRID_ENV ? 2 : field_raman(d) ? 1 : 0] = true;
        if (!solo_price(ctxs[i], &p)) continue;
        cost.push_back(solve_cost(ctxs[i], op[i]) / class_us(ctx_class(ctxs[i])));
        price.push_back(p);
        n_dense += p.dense > 0;
    }
    if (cost.empty() || kind[0] + kind[1] + kind[2] > 1) return false;
    const double longest = *std::max_element(cost.begin(), cost.end());
    std::vector<double> alone, gang, dense;
    double work = 0.0;
    for (size_t i = 0; i < cost.size(); i++) {
        const double c = longest > 0.0 ? cost[i] + 0.1 * longest : 1.0;  // linear runs: equal lengths
        const bool d = n_dense > LG_DENSE_ABOVE && price[i].dense > 0;
        alone.push_back(c * price[i].alone);
        (d ? dense : gang).push_back(c * (d ? 2 * GANGS * price[i].dense : GANGS * price[i].gang));
        work += c * (d ? price[i].dense : price[i].gang);
    }
    // the gangs' tails and the estimates' errors: a tenth of the work, 7 % of the dealing
    return dealt(alone, LG_MAX_WG) < std::max(1.1 * work, 1.07 * std::max(dealt(gang, GANGS), dealt(dense, 2 * GANGS)));
}

static int prepare_instance(lh_ctx* c, const lh_rk_opts* o, bool want_saves, bool alone, DInst* in,
                            RunStats* dstats_slot, hipStream_t s) {
    if (!opts_ok(o)) return LH_E_ARG;
    if (!c->have_state) return LH_E_ARG;
    int st = ensure_solver_buffers(c, o->save_n, want_saves, alone);
    if (st) return st;
    std::vector<double> g;
    save_grid(o, g);
    // the kernels only read the grid: a sweep repeated with the same options
    // skips the upload (and its synchronisation) for every instance
    const bool same = c->zgrid_h && c->zgrid_hn == (int)g.size() &&
                      memcmp(c->zgrid_h, g.data(), sizeof(double) * g.size()) == 0;
    if (!same) {
        HIPCK(hipMemcpyAsync(c->zgrid, g.data(), sizeof(double) * g.size(), hipMemcpyHostToDevice, s));
        HIPCK(hipStreamSynchronize(s));  // g is a local buffer
        double* h = (double*)realloc(c->zgrid_h, sizeof(double) * g.size());
        if (h) {
            memcpy(h, g.data(), sizeof(double) * g.size());
            c->zgrid_h = h;
            c->zgrid_hn = (int)g.size();
        } else {
            c->zgrid_hn = 0;
        }
    }
    *in = base_inst(c);
    in->Yin = c->Yin;
    in->Y = c->Y;
    in->K = alone ? c->K1 : c->K;
    in->kstride = alone ? c->k1stride : c->kstride;
    in->saves = want_saves ? c->saves : nullptr;
    in->zgrid = c->zgrid;
    in->stats = dstats_slot;
    inst_options(in, o);
    c->have_result = 0;
    c->have_records = 0;
    c->result_save_n = want_saves ? o->save_n : 0;
    return LH_OK;
}

// --------------------------------------------------------------------------
// Plan wisdom: measured radial plans keyed by (n_to, n_r)
// --------------------------------------------------------------------------
// The role of FFTW's wisdom in the reference (src/Utils.jl:84-108 imports it
// before planning and exports it after): a context created for a shape with
// wisdom takes the recorded plan without measuring; any other takes
// RAD_DEFAULT_PLAN (with the tiles of rad_default_tiles).  Process-wide, guarded
// by g_wisdom_mu.
struct WisdomEntry {
    int n_to, n_r;
    RadPlan plan;
    double us;
};
static std::mutex g_wisdom_mu;
static std::vector<WisdomEntry> g_wisdom;

static bool wisdom_lookup(int n_to, int n_r, RadPlan* p) {
    std::lock_guard<std::mutex> lk(g_wisdom_mu);
    for (const WisdomEntry& w : g_wisdom)
        if (w.n_to == n_to && w.n_r == n_r) return *p = w.plan, true;
    return false;
}

static void wisdom_record(int n_to, int n_r, RadPlan p, double us) {
    std::lock_guard<std::mutex> lk(g_wisdom_mu);
    for (WisdomEntry& w : g_wisdom)
        if (w.n_to == n_to && w.n_r == n_r) {
            w.plan = p;
            w.us = us;
            return;
        }
    g_wisdom.push_back({n_to, n_r, p, us});
}

// --------------------------------------------------------------------------
// Radial transform: set-up, one RHS, solve
// --------------------------------------------------------------------------
static int rad_setup(lh_ctx* c, const lh_desc* d) {
    const size_t nr = (size_t)d->n_r, nto = (size_t)d->n_to;
    std::vector<double> mt(nr * nr);
    for (size_t k = 0; k < nr; k++)
        for (size_t n = 0; n < nr; n++) mt[k * nr + n] = d->qdht[n * nr + k];
    int st = upload(&c->Mt, mt.data(), mt.size());
    if (st) return st;
    const size_t col = (d->grid_kind == LH_GRID_ENV) ? 2 * nto : nto;  // complex samples on the envelope grid
    HIPCK(hipMalloc(&c->Ek, sizeof(double) * col * nr));
    HIPCK(hipMalloc(&c->Er, sizeof(double) * col * nr));
    HIPCK(hipMalloc(&c->partial, sizeof(double) * 3 * nr));
    HIPCK(hipMalloc(&c->rargs, sizeof(RadArgs) * 2));
    HIPCK(hipMalloc(&c->rctl, sizeof(RadCtl) * 2));
    c->rplan = RAD_DEFAULT_PLAN;
    c->rplan_own = wisdom_lookup(d->n_to, d->n_r, &c->rplan);
    DInst pw = base_inst(c);
    pw.e_scale = 1.0;  // the 1/Nto of the inverse transform is folded into the k→r contraction
    return upload(&c->pw, &pw, 1);
}

static void rad_ctl_init(RadCtl* h, const lh_rk_opts* o) {
    memset(h, 0, sizeof(*h));
    if (o) {
        h->t = h->tn = o->z0;
        h->dt = h->dtn = o->init_dz;
        h->saved = o->save_first;
    }
    for (int j = 0; j < 8; j++) h->perm[j] = j;
    h->status = LH_OK;
}

// The plan that the context's launches follow (rgraph is captured with it).
static RadPlan rad_plan_run(const lh_ctx* c) {
    if (c->rplan_own) return c->rplan;
    return {c->rplan.fft, rad_default_tiles((c->d.grid_kind == LH_GRID_ENV ? 2 : 1) * c->d.n_to, c->d.n_r)};
}

static RadArgs rad_args(const lh_ctx* c, int slot) {
    RadArgs a;
    memset(&a, 0, sizeof(a));
    const lh_desc& d = c->d;
    a.n_omega = d.n_omega;
    a.n_t = d.n_t;
    a.n_to = d.n_to;
    a.n_r = d.n_r;
    a.col = (d.grid_kind == LH_GRID_ENV) ? 2 * d.n_to : d.n_to;
    a.sc_t = scale_to_time(d);
    a.gemm_kr = d.qdht_inv / (double)d.n_to;  // ldiv!(Eto, QDHT, Eto) with irfft's 1/Nto
    a.gemm_rk = d.qdht_fwd;                   // mul!(Pto, QDHT, Pto)
    a.linop = c->linop;
    a.outfac = c->outfac;
    a.Mt = c->Mt;
    a.pw = c->pw;
    a.Ek = c->Ek;
    a.Er = c->Er;
    a.partial = c->partial;
    a.ctl = c->rctl + slot;
    return a;
}

// Per-step output of a radial run (lh_solve_stream): the steps are replayed
// one at a time and each accepted step that saves (every accepted step with
// every) is handed to cb with the saves since the previous call and the state,
// copied out of device memory into page-locked host buffers.
struct RadHook {
    lh_output_cb cb;
    void* user;
    bool every;
    double2* y_h;          // [n_state]
    double2* sv_h;         // [save_n][n_state]
    const double* zgrid;   // [save_n] host save grid
};

// Full propagation of one radial context on stream s (buffers and save grid
// prepared by prepare_instance).  The per-step launch sequence is captured
// once per context as a graph and replayed until the control block says done.
static int rad_solve(lh_ctx* c, const lh_rk_opts* o, bool want_saves, hipStream_t s, lh_stats* out,
                     const RadHook* hook = nullptr) {
    const double2* tw;
    int st = twiddles(c->device, &tw);
    if (st) return st;
    const int n_to = c->d.n_to, n_r = c->d.n_r;
    RadArgs a = rad_args(c, 0);
    a.Y[0] = c->Y;
    a.Y[1] = c->YN;
    for (int j = 0; j < 7; j++) a.K[j] = c->K + j * c->kstride;
    a.kstride = c->kstride;
    a.saves = want_saves ? c->saves : nullptr;
    a.zgrid = c->zgrid;
    a.zmax = o->zmax;
    a.rtol = o->rtol;
    a.atol = o->atol;
    a.safety = o->safety;
    a.max_dz = o->max_dz;
    a.min_dz = o->min_dz;
    a.repeat_limit = o->repeat_limit;
    a.save_n = o->save_n;
    a.zstop = o->zstop;
    a.max_steps = o->max_steps > 0 ? o->max_steps : LH_MAX_STEPS;
    RadCtl h;
    rad_ctl_init(&h, o);
    h.rhs_evals = 1;
    hipLaunchKernelGGL(rad_set, dim3(1), dim3(64), 0, s, a, h, c->rargs);
    HIPCK(hipMemcpyAsync(c->Y, c->Yin, sizeof(double2) * (size_t)c->n_state, hipMemcpyDeviceToDevice, s));
    rad_rhs_dispatch(rad_plan_run(c), c->d.grid_kind == LH_GRID_ENV, n_to, n_r, c->rargs, tw, -1, s);  // PreconStepper init: k1 = fbar(y0)
    HIPCK(hipGetLastError());
    HIPCK(hipMemcpyAsync(&h, c->rctl, sizeof(h), hipMemcpyDeviceToHost, s));
    HIPCK(hipStreamSynchronize(s));
    if (h.status != LH_OK) {
        h.done = 1;
        HIPCK(hipMemcpy(c->rctl, &h, sizeof(h), hipMemcpyHostToDevice));
    }
    if (!h.done && !c->rgraph) {
        hipGraph_t g = nullptr;
        HIPCK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        rad_step_dispatch(rad_plan_run(c), c->d.grid_kind == LH_GRID_ENV, n_to, n_r, c->rargs, tw, s);
        hipError_t e1 = hipGetLastError();
        hipError_t e2 = hipStreamEndCapture(s, &g);
        if (e1 != hipSuccess || e2 != hipSuccess || !g) {
            if (g) (void)hipGraphDestroy(g);
            return LH_E_HIP;
        }
        hipError_t e3 = hipGraphInstantiate(&c->rgraph, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e3 != hipSuccess) {
            c->rgraph = nullptr;
            return LH_E_HIP;
        }
    }
    // replay in chunks (one step at a time with a hook); steps after
    // completion return at once
    int chunk = hook ? 1 : 4;
    long long acc_done = 0;
    int saves_done = o->save_first;
    bool stop_req = false;
    const size_t NS = (size_t)c->n_state;
    while (!h.done) {
        for (int i = 0; i < chunk; i++) HIPCK(hipGraphLaunch(c->rgraph, s));
        HIPCK(hipMemcpyAsync(&h, c->rctl, sizeof(h), hipMemcpyDeviceToHost, s));
        HIPCK(hipStreamSynchronize(s));
        if (!hook) {
            if (chunk < 16) chunk *= 2;
            continue;
        }
        if (h.accepted == acc_done) continue;
        acc_done = h.accepted;
        if (!stop_req && (hook->every || h.saved > saves_done)) {
            const int nsv = h.saved - saves_done;
            if (nsv > 0)
                HIPCK(hipMemcpyAsync(hook->sv_h + (size_t)saves_done * NS, c->saves + (size_t)saves_done * NS,
                                     sizeof(double2) * NS * (size_t)nsv, hipMemcpyDeviceToHost, s));
            HIPCK(hipMemcpyAsync(hook->y_h, h.ycur ? c->YN : c->Y, sizeof(double2) * NS, hipMemcpyDeviceToHost, s));
            HIPCK(hipStreamSynchronize(s));
            lh_step_out so;
            memset(&so, 0, sizeof(so));
            so.first_save = saves_done;
            so.n_saves = nsv;
            so.saves = (const double*)(hook->sv_h + (size_t)saves_done * NS);
            so.zsaves = hook->zgrid + saves_done;
            so.z = h.tn;
            so.dz = h.dtn;
            so.y = (const double*)hook->y_h;
            so.accepted = h.accepted;
            if (hook->cb(hook->user, &so) != 0) stop_req = true;
        }
        saves_done = h.saved;
        if (stop_req && !h.done) {
            // nothing more is handed over; the run ends here
            h.status = LH_E_STOPPED;
            h.done = 1;
            HIPCK(hipMemcpy(c->rctl, &h, sizeof(h), hipMemcpyHostToDevice));
        }
    }
    if (h.ycur == 1)  // the final state s.yn lives in YN
        HIPCK(hipMemcpyAsync(c->Y, c->YN, sizeof(double2) * (size_t)c->n_state, hipMemcpyDeviceToDevice, s));
    HIPCK(hipStreamSynchronize(s));
    out->steps = h.steps;
    out->accepted = h.accepted;
    out->rejected = h.rejected;
    out->rhs_evals = h.rhs_evals;
    out->status = h.status;
    out->saved = h.saved;
    out->z = h.tn;
    out->dz = h.dtn;
    return LH_OK;
}

extern "C" {

const char* lh_strerror(int status) {
    switch (status) {
        case LH_OK: return "ok";
        case LH_E_ARG: return "invalid argument or unsupported configuration";
        case LH_E_HIP: return "HIP runtime error";
        case LH_E_PPT_RANGE: return "field strength exceeds maximum for PPT ionisation rate";
        case LH_E_REPEAT_LIMIT: return "reached limit for step repetition";
        case LH_E_NONFINITE: return "non-finite state";
        case LH_E_NOMEM: return "device allocation failed";
        case LH_E_NODEVICE: return "no HIP device";
        case LH_E_MAXSTEPS: return "reached the cap on step attempts";
        case LH_E_STOPPED: return "stopped before the end of the propagation (zstop)";
        case LH_E_TOO_LARGE: return "problem exceeds the fixed working memory of lh_solve_noalloc";
        case LH_E_HOST_WAIT: return "the host fell behind the per-step output by more than its ring of slots";
        default: return "unknown status";
    }
}

int lh_device_count(int* count) {
    if (!count) return LH_E_ARG;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
    *count = n;
    return LH_OK;
}

int lh_destroy(lh_ctx* c) {
    if (!c) return LH_OK;
    hipSetDevice(c->device);
    if (c->stream) hipStreamSynchronize(c->stream);
    for (const void* p : {(const void*)c->omega_win, (const void*)c->t_win, (const void*)c->to_win, (const void*)c->ppt,
                          (const void*)c->omega, (const void*)c->st_ew, (const void*)c->st_t, (const void*)c->st_win,
                          (const void*)c->zg_Z,
                          (const void*)c->zg_P, (const void*)c->zfd, (const void*)c->zgam, (const void*)c->zd,
                          (const void*)c->znwg, (const void*)c->zpre, (const void*)c->zsidx})
        shared_release(p);
    void* ptrs[] = {c->linop, c->outfac, c->hwdt, c->escr, c->gx, c->Yin, c->Y, c->YN,
                    c->saves, c->zgrid, c->dstats, c->launch1, c->rhs_in, c->rhs_out,
                    c->steprec, c->st_rec1, c->zL, c->zOF};
    for (void* p : ptrs)
        if (p) hipFree(p);
    if (c->K) hipFree(c->K);
    if (c->K1) hipFree(c->K1);
    void* rptrs[] = {c->Mt, c->Ek, c->Er, c->partial, c->pw, c->rargs, c->rctl};
    for (void* p : rptrs)
        if (p) hipFree(p);
    if (c->rgraph) hipGraphExecDestroy(c->rgraph);
    for (RhsSet& r : c->rset) {
        if (r.block) hipFree(r.block);
        if (r.z) hipFree(r.z);
    }
    if (c->cap_ev) hipEventDestroy(c->cap_ev);
    free(c->zgrid_h);
    if (c->stream) hipStreamDestroy(c->stream);
    free(c);
    return LH_OK;
}

int lh_create(lh_ctx** out, const lh_desc* d) {
    if (!out || !d) return LH_E_ARG;
    *out = nullptr;
    if (!supported(d)) return LH_E_ARG;
    if (!d->omega_win || !d->sidx || !d->t_win || !d->to_win || !d->norm) return LH_E_ARG;
    if (d->plasma && (!d->ppt_x || !d->ppt_y || !d->ppt_d || d->ppt_n < 4)) return LH_E_ARG;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return LH_E_NODEVICE;
    lh_ctx* c = (lh_ctx*)calloc(1, sizeof(lh_ctx));
    if (!c) return LH_E_NOMEM;
    c->d = *d;
    c->n_state = d->n_omega * d->n_r;
    int st = LH_OK;
    if (hipGetDevice(&c->device) != hipSuccess) st = LH_E_HIP;
    if (!st) st = scratch_init(c->device);
    if (!st) c->beat = g_beat[c->device];
    if (!st && hipStreamCreate(&c->stream) != hipSuccess) st = LH_E_HIP;
    const size_t N = (size_t)d->n_omega, NS = (size_t)c->n_state;
    if (!st) st = shared_upload(c->device, &c->omega_win, d->omega_win, N);
    if (!st && d->omega) st = shared_upload(c->device, &c->omega, d->omega, N);
    if (!st && d->transform == LH_TRANS_MODEAVG)
        st = shared_upload(c->device, &c->zsidx, d->sidx, N);
    if (!st) st = shared_upload(c->device, &c->t_win, d->t_win, (size_t)d->n_t);
    if (!st) st = shared_upload(c->device, &c->to_win, d->to_win, (size_t)d->n_to);
    if (!st) {
        // Output factor per bin: to_freq! crop scale, then norm! and ×ωwin on
        // sidx bins (mode-average, src/NonlinearRHS.jl:368-387), or the radial
        // factor on every bin (:473).
        const double sf = scale_to_freq(*d);
        const double2* nf = (const double2*)d->norm;
        std::vector<double2> of(NS);
        for (size_t i = 0; i < NS; i++) {
            size_t k = i % N;
            if (d->transform == LH_TRANS_RADIAL)
                of[i] = make_double2(sf * nf[i].x, sf * nf[i].y);
            else if (d->sidx[k])
                of[i] = make_double2((sf * nf[i].x) * d->omega_win[k], (sf * nf[i].y) * d->omega_win[k]);
            else
                of[i] = make_double2(sf, 0.0);
        }
        st = upload(&c->outfac, of.data(), NS);
    }
    if (!st) {
        std::vector<double2> lin(NS, make_double2(0.0, 0.0));
        if (d->linop) memcpy(lin.data(), d->linop, sizeof(double2) * NS);
        st = upload(&c->linop, lin.data(), NS);
    }
    if (!st && d->plasma) {
        std::vector<double4> p((size_t)d->ppt_n);
        for (int i = 0; i < d->ppt_n; i++) p[i] = make_double4(d->ppt_x[i], d->ppt_y[i], d->ppt_d[i], 0.0);
        c->ppt_emin = d->ppt_x[0];
        c->ppt_emax = d->ppt_x[d->ppt_n - 1];
        st = shared_upload(c->device, &c->ppt, p.data(), p.size());
    }
    const bool modeavg = d->transform == LH_TRANS_MODEAVG;
    if (!st && ctx_class(c) == LH_CLASS_32768 && d->raman) st = LH_E_ARG;  // no Raman convolution on the largest field grid
    if (!st && field_raman(*d) && hipMalloc(&c->escr, sizeof(double2) * (size_t)d->n_to) != hipSuccess) st = LH_E_NOMEM;
    if (!st && modeavg && hipMalloc(&c->gx, sizeof(double2) * lg_area_len(*d)) != hipSuccess) st = LH_E_NOMEM;
    if (!st && d->raman) {
        const double2* tw;
        double* dh = nullptr;
        double2* work = nullptr;
        st = twiddles(c->device, &tw);
        if (!st) st = upload(&dh, d->raman_h, (size_t)d->n_to);
        if (!st && d->n_to == 16384 && hipMalloc(&work, sizeof(double2) * (size_t)d->n_to * 3 / 2) != hipSuccess)
            st = LH_E_NOMEM;
        if (!st && hipMalloc(&c->hwdt, sizeof(double2) * (size_t)(d->n_to + 1)) != hipSuccess) st = LH_E_NOMEM;
        if (!st) {
            launch_raman_hw(d->n_to, dh, d->dt_o, tw, c->hwdt, work, c->stream);
            if (hipGetLastError() != hipSuccess || hipStreamSynchronize(c->stream) != hipSuccess) st = LH_E_HIP;
        }
        if (dh) (void)hipFree(dh);
        if (work) (void)hipFree(work);
    }
    if (!st && d->transform == LH_TRANS_RADIAL) st = rad_setup(c, d);
    // host pointers inside the copied descriptor belong to the caller
    c->d.omega = nullptr; c->d.sidx = nullptr; c->d.omega_win = nullptr; c->d.t_win = nullptr;
    c->d.to_win = nullptr; c->d.linop = nullptr; c->d.norm = nullptr; c->d.ppt_x = nullptr;
    c->d.ppt_y = nullptr; c->d.ppt_d = nullptr; c->d.raman_h = nullptr; c->d.qdht = nullptr;
    if (!st) {
        const double2* tw;
        st = modeavg ? gang_twiddles(c->device, &tw) : twiddles(c->device, &tw);
    }
    if (!st && modeavg && hipMalloc(&c->launch1, LAUNCH1_BYTES) != hipSuccess) st = LH_E_NOMEM;
    if (!st && modeavg) st = rhs_sets_init(c);
    if (!st && hipMalloc(&c->dstats, sizeof(RunStats)) != hipSuccess) st = LH_E_NOMEM;
    if (st) {
        lh_destroy(c);
        return st;
    }
    *out = c;
    return LH_OK;
}

int lh_ctx_status(lh_ctx* c) {
    if (!c) return LH_E_ARG;
    if (c->rhs_pending) {  // status of the last lh_rhs_device launch
        int kst = LH_OK;
        HIPCK(hipSetDevice(c->device));
        HIPCK(hipStreamSynchronize(c->rhs_stream ? c->rhs_stream : c->stream));
        const int* sp = (c->d.transform == LH_TRANS_RADIAL) ? &c->rctl[1].status : c->dstatus;
        HIPCK(hipMemcpy(&kst, sp, sizeof(int), hipMemcpyDeviceToHost));
        c->last_status = kst;
        c->rhs_pending = 0;
    }
    return c->last_status;
}

int lh_rhs_device(lh_ctx* c, void* nl_dev, const void* Ew_dev, double z, void* stream) {
    if (!c || !nl_dev || !Ew_dev) return LH_E_ARG;
    HIPCK(hipSetDevice(c->device));
    hipStream_t s = stream ? (hipStream_t)stream : c->stream;
    const double2* tw;
    const bool radial = c->d.transform == LH_TRANS_RADIAL;
    int st = radial ? twiddles(c->device, &tw) : gang_twiddles(c->device, &tw);
    if (st) return st;
    if (radial) {
        RadArgs a = rad_args(c, 1);
        a.rhs_in = (const double2*)Ew_dev;
        a.rhs_out = (double2*)nl_dev;
        RadOne one;
        one.a = a;
        rad_ctl_init(&one.h, nullptr);
        const bool env = c->d.grid_kind == LH_GRID_ENV;
        if (env) hipLaunchKernelGGL(rad_set, dim3(1), dim3(64), 0, s, one.a, one.h, c->rargs + 1);
        rad_rhs_dispatch(rad_plan_run(c), env, c->d.n_to, c->d.n_r, c->rargs + 1, tw, -1, s, &one);
    } else {
        DInst in = base_inst(c);
        in.rhs_in = (const double2*)Ew_dev;
        in.rhs_out = (double2*)nl_dev;
        in.z0 = z;  // a gradient fill evaluates its constants at z
        GangLaunch l;
        st = rhs_launch_of(c, &in, tw, s, &l);
        if (st) return st;
        if (!launch_rhs(l, c->d.raman != 0, c->dstatus)) return LH_E_ARG;
    }
    HIPCK(hipGetLastError());
    c->rhs_pending = 1;
    c->rhs_stream = s;
    return LH_OK;
}

int lh_rhs(lh_ctx* c, double* nl, const double* Ew, double z) {
    if (!c || !nl || !Ew) return LH_E_ARG;
    HIPCK(hipSetDevice(c->device));
    const size_t bytes = sizeof(double2) * (size_t)c->n_state;
    if (!c->rhs_in) {
        HIPCK(hipMalloc(&c->rhs_in, bytes));
        HIPCK(hipMalloc(&c->rhs_out, bytes));
    }
    HIPCK(hipMemcpyAsync(c->rhs_in, Ew, bytes, hipMemcpyHostToDevice, c->stream));
    int st = lh_rhs_device(c, c->rhs_out, c->rhs_in, z, c->stream);
    if (st) return st;
    int kst = LH_OK;
    HIPCK(hipMemcpyAsync(nl, c->rhs_out, bytes, hipMemcpyDeviceToHost, c->stream));
    const int* sp = (c->d.transform == LH_TRANS_RADIAL) ? &c->rctl[1].status : c->dstatus;
    HIPCK(hipMemcpyAsync(&kst, sp, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HIPCK(hipStreamSynchronize(c->stream));
    c->last_status = kst;
    c->rhs_pending = 0;
    return kst;
}

int lh_solve(lh_ctx* c, double* Ew, const lh_rk_opts* o, double* saves, double* zsaves, lh_stats* stats) {
    lh_ctx* cs[1] = {c};
    double* ews[1] = {Ew};
    double* svs[1] = {saves};
    double* zss[1] = {zsaves};
    lh_stats tmp;
    lh_stats* sp = stats ? stats : &tmp;
    int st = lh_batch_solve(cs, 1, ews, o, saves ? svs : nullptr, zss, sp);
    if (st) return st;
    return sp->status;
}

// lh_solve_stream of a radial context: the host replays the steps (RadHook).
static int rad_solve_stream(lh_ctx* c, double* Ew, const lh_rk_opts* o, lh_output_cb cb, void* user,
                            lh_stats* stats) {
    const size_t NS = (size_t)c->n_state;
    const size_t nsave = (size_t)(o->save_n > 0 ? o->save_n : 0);
    double2* y_h = nullptr;
    double2* sv_h = nullptr;
    HIPCK(hipHostMalloc((void**)&y_h, sizeof(double2) * NS, 0));
    if (nsave && hipHostMalloc((void**)&sv_h, sizeof(double2) * NS * nsave, 0) != hipSuccess) {
        (void)hipHostFree(y_h);
        return LH_E_NOMEM;
    }
    std::vector<double> zg;
    save_grid(o, zg);
    DInst in;
    int st = prepare_instance(c, o, true, false, &in, c->dstats, c->stream);
    RadHook hk{cb, user, o->every_step != 0, y_h, sv_h, zg.data()};
    if (!st) st = rad_solve(c, o, true, c->stream, stats, &hk);
    if (!st && hipMemcpy(Ew, c->Y, sizeof(double2) * NS, hipMemcpyDeviceToHost) != hipSuccess) st = LH_E_HIP;
    (void)hipHostFree(y_h);
    if (sv_h) (void)hipHostFree(sv_h);
    if (st) return st;
    c->last_status = stats->status;
    c->have_result = 1;
    c->result_save_n = 0;  // the saves went to the callback
    c->result_nrec = 0;
    c->have_records = 1;
    return stats->status;
}

// Page-locked bytes of the every-step ring of state slots (clamped to 64..4096
// slots): 1023 slots of a 4097-bin state.
static constexpr size_t LH_RING_BYTES = (size_t)64 << 20;

int lh_solve_stream(lh_ctx* c, double* Ew, const lh_rk_opts* o, lh_output_cb cb, void* user, lh_stats* stats) {
    if (!c || !Ew || !o || !cb || !stats || !opts_ok(o)) return LH_E_ARG;
    const int cls = ctx_class(c);
    if (cls < 0 || c->zg_on) return LH_E_ARG;
    int st = lh_set_state(c, Ew);
    if (st) return st;
    if (cls == LH_CLASS_RADIAL) return rad_solve_stream(c, Ew, o, cb, user, stats);
    const double2* tw;
    st = gang_twiddles(c->device, &tw);
    if (st) return st;
    // one page-locked, device-mapped, coherent block: publication counter and
    // stop flag, slot info and state slots (two, or the every-step ring), every
    // save and its position, the statistics records
    const size_t NS = (size_t)c->n_state;
    const size_t nsave = (size_t)(o->save_n > 0 ? o->save_n : 0);
    const size_t ncap = (size_t)(c->st_on ? c->st_cap : 0);
    const bool every = o->every_step != 0;
    size_t nslot = 2;
    if (every) {
        nslot = LH_RING_BYTES / (NS * sizeof(double2));
        nslot = nslot < 64 ? 64 : nslot > 4096 ? 4096 : nslot;
    }
    const size_t off_info = 256, off_y = (off_info + nslot * 4 * sizeof(double) + 255) / 256 * 256,
                 off_sv = off_y + nslot * NS * sizeof(double2), off_rec = off_sv + nsave * NS * sizeof(double2),
                 total = off_rec + ncap * LH_NSTAT * sizeof(double);
    unsigned char* hb = nullptr;
    HIPCK(hipHostMalloc((void**)&hb, total, hipHostMallocMapped | hipHostMallocCoherent));
    unsigned char* db = nullptr;
    if (hipHostGetDevicePointer((void**)&db, hb, 0) != hipSuccess) {
        (void)hipHostFree(hb);
        return LH_E_HIP;
    }
    memset(hb, 0, 256);
    unsigned long long* pub = (unsigned long long*)hb;
    int* stop = (int*)(hb + 64);
    const double* info = (const double*)(hb + off_info);
    const double2* ys = (const double2*)(hb + off_y);
    const double2* sv = (const double2*)(hb + off_sv);
    const double* recs = (const double*)(hb + off_rec);
    DInst in;
    st = prepare_instance(c, o, false, false, &in, c->dstats, c->stream);
    std::vector<double> zg;
    save_grid(o, zg);
    if (!st) {
        in.saves = nsave ? (double2*)(db + off_sv) : nullptr;
        if (ncap) in.steprec = (double*)(db + off_rec);
        in.pub = (unsigned long long*)db;
        in.pub_stop = (const int*)(db + 64);
        in.pub_info = (double*)(db + off_info);
        in.pub_y = (double2*)(db + off_y);
        in.pub_ring = every ? (int)nslot : 0;
        st = set_launch1(c->launch1, in, c->stream);
    }
    if (!st) {
        if (!launch_solve(launch1_of(c, c->launch1, tw, c->stream), c->d.raman != 0, true)) st = LH_E_ARG;
        if (hipGetLastError() != hipSuccess) st = LH_E_HIP;
    }
    // Drain the publications while the kernel runs.  A publication's state
    // slot is rewritten two publications later, so a copy of it counts only
    // if the counter has not moved on meanwhile; saves and records have slots
    // of their own.  In every-step mode each publication is handed over in
    // turn from the ring, which the kernel rewrites nslot publications later:
    // the copy of publication q counts if the counter has not passed
    // q + nslot − 2 after it (the kernel writes publication j into its slot
    // only once j publications are out), else the host has fallen behind and
    // the run ends with LH_E_HOST_WAIT.  After the callback asks to stop,
    // nothing more is handed over (the run ends at its next publication).
    std::vector<double2> ycopy(NS);
    unsigned long long done = 0;
    int saves_done = o->save_first;
    long long recs_done = 0;
    bool stop_req = false, lapped = false;
    while (!st) {
        const hipError_t q = hipStreamQuery(c->stream);
        if (q != hipSuccess && q != hipErrorNotReady) {
            st = LH_E_HIP;
            break;
        }
        unsigned long long p = __atomic_load_n(pub, __ATOMIC_ACQUIRE);
        while (every && p > done && !lapped) {
            const unsigned long long q = done + 1;
            const int slot = (int)((q - 1) % nslot);
            const double z = info[4 * slot], dz = info[4 * slot + 1];
            const int nsaved = (int)info[4 * slot + 2];
            const long long nacc = (long long)info[4 * slot + 3];
            memcpy(ycopy.data(), ys + (size_t)slot * NS, NS * sizeof(double2));
            if (__atomic_load_n(pub, __ATOMIC_ACQUIRE) > q + nslot - 2) {
                lapped = true;
                __atomic_store_n(stop, 1, __ATOMIC_RELEASE);
                break;
            }
            const long long nrec = ncap ? (nacc < (long long)ncap ? nacc : (long long)ncap) : 0;
            if (!stop_req) {
                lh_step_out out;
                out.first_save = saves_done;
                out.n_saves = nsaved - saves_done;
                out.saves = (const double*)(sv + (size_t)saves_done * NS);
                out.zsaves = zg.data() + saves_done;
                out.z = z;
                out.dz = dz;
                out.y = (const double*)ycopy.data();
                out.accepted = nacc;
                out.first_record = (int32_t)recs_done;
                out.n_records = (int32_t)(nrec - recs_done);
                out.records = recs + (size_t)recs_done * LH_NSTAT;
                if (cb(user, &out) != 0) {
                    stop_req = true;
                    __atomic_store_n(stop, 1, __ATOMIC_RELEASE);
                }
            }
            done = q;
            saves_done = nsaved;
            recs_done = nrec;
        }
        if (!every && p > done && !stop_req) {
            double z = 0, dz = 0, fsaved = 0, facc = 0;
            for (;;) {
                const int slot = (int)((p - 1) & 1);
                z = info[4 * slot];
                dz = info[4 * slot + 1];
                fsaved = info[4 * slot + 2];
                facc = info[4 * slot + 3];
                memcpy(ycopy.data(), ys + (size_t)slot * NS, NS * sizeof(double2));
                const unsigned long long p2 = __atomic_load_n(pub, __ATOMIC_ACQUIRE);
                if (p2 == p) break;
                p = p2;
            }
            const int nsaved = (int)fsaved;
            const long long nacc = (long long)facc;
            const long long nrec = ncap ? (nacc < (long long)ncap ? nacc : (long long)ncap) : 0;
            lh_step_out out;
            out.first_save = saves_done;
            out.n_saves = nsaved - saves_done;
            out.saves = (const double*)(sv + (size_t)saves_done * NS);
            out.zsaves = zg.data() + saves_done;
            out.z = z;
            out.dz = dz;
            out.y = (const double*)ycopy.data();
            out.accepted = nacc;
            out.first_record = (int32_t)recs_done;
            out.n_records = (int32_t)(nrec - recs_done);
            out.records = recs + (size_t)recs_done * LH_NSTAT;
            if (cb(user, &out) != 0) {
                stop_req = true;
                __atomic_store_n(stop, 1, __ATOMIC_RELEASE);
            }
            done = p;
            saves_done = nsaved;
            recs_done = nrec;
        }
        if (q == hipSuccess) break;  // p was read after the kernel had ended
        struct timespec ts = {0, 20000};
        nanosleep(&ts, nullptr);
    }
    if (!st) {
        RunStats rs;
        if (hipMemcpy(&rs, c->dstats, sizeof(rs), hipMemcpyDeviceToHost) != hipSuccess) st = LH_E_HIP;
        if (!st) *stats = solved(rs);
        if (!st && lapped) stats->status = LH_E_HOST_WAIT;
    } else {
        (void)hipStreamSynchronize(c->stream);  // never free a block the kernel may still write
    }
    if (!st && hipMemcpy(Ew, c->Y, sizeof(double2) * NS, hipMemcpyDeviceToHost) != hipSuccess) st = LH_E_HIP;
    if (!st && ncap && c->steprec &&
        hipMemcpy(c->steprec, recs, sizeof(double) * LH_NSTAT * ncap, hipMemcpyHostToDevice) != hipSuccess)
        st = LH_E_HIP;
    (void)hipHostFree(hb);
    if (st) return st;
    c->last_status = stats->status;
    c->have_result = 1;
    c->result_save_n = 0;  // the saves went to the callback
    c->result_nrec = ncap ? (int)(stats->accepted < (long long)ncap ? stats->accepted : (long long)ncap) : 0;
    c->have_records = 1;
    return stats->status;
}

int lh_set_state(lh_ctx* c, const double* Ew) {
    if (!c || !Ew) return LH_E_ARG;
    HIPCK(hipSetDevice(c->device));
    int st = ensure_solver_buffers(c, 0, false, c->zg_on != 0);
    if (st) return st;
    HIPCK(hipMemcpy(c->Yin, Ew, sizeof(double2) * (size_t)c->n_state, hipMemcpyHostToDevice));
    c->have_state = 1;
    if (c->d.transform == LH_TRANS_MODEAVG) {
        // sums of their own, so that the additions don't wait for each other (a
        // batch spent 1 to 13 µs of host time an instance on one serial sum over
        // 2049 to 16384 bins; now 0.2 to 1.7)
        double part[8] = {0}, e = 0.0;
        const int n = 2 * c->n_state;
        for (int i = 0; i + 8 <= n; i += 8)
            for (int j = 0; j < 8; j++) part[j] += Ew[i + j] * Ew[i + j];
        for (int i = n & ~7; i < n; i++) e += Ew[i] * Ew[i];
        for (int j = 0; j < 8; j++) e += part[j];
        c->amp = scale_to_time(c->d) * sqrt(e * c->d.dt_o / (double)c->d.n_to) / c->d.field_div;
    }
    return LH_OK;
}

int lh_get_state(lh_ctx* c, double* Ew) {
    if (!c || !Ew || !c->have_result) return LH_E_ARG;
    HIPCK(hipSetDevice(c->device));
    HIPCK(hipMemcpy(Ew, c->Y, sizeof(double2) * (size_t)c->n_state, hipMemcpyDeviceToHost));
    return LH_OK;
}

int lh_get_saves(lh_ctx* c, double* saves, double* zsaves) {
    if (!c || !c->have_result) return LH_E_ARG;
    HIPCK(hipSetDevice(c->device));
    int n = c->result_save_n;
    if (saves && n > 0)
        HIPCK(copy_to_host(saves, c->saves, sizeof(double2) * (size_t)c->n_state * n, c->device, c->stream));
    if (zsaves && n > 0) HIPCK(hipMemcpy(zsaves, c->zgrid, sizeof(double) * n, hipMemcpyDeviceToHost));
    return LH_OK;
}

// One stream per (device, size class and kernel) for the batched launches, created on
// first use and kept for the process (default priority).
static std::mutex g_cls_mu;
static hipStream_t g_cls_stream[64][3 * LH_NCLASS];

static int class_stream(int dev, int c, hipStream_t* out) {
    if (dev < 0 || dev >= 64) return LH_E_ARG;
    std::lock_guard<std::mutex> lk(g_cls_mu);
    if (!g_cls_stream[dev][c] && hipStreamCreate(&g_cls_stream[dev][c]) != hipSuccess) {
        g_cls_stream[dev][c] = nullptr;
        return LH_E_HIP;
    }
    *out = g_cls_stream[dev][c];
    return LH_OK;
}

// The resident batch with options per instance: op[i] for instance i.
static int batch_resident(lh_ctx* const* ctxs, int n, const lh_rk_opts* const* op, int want_saves, lh_stats* stats) {
    if (!ctxs || n <= 0 || !op || !stats) return LH_E_ARG;
    for (int i = 0; i < n; i++)
        if (!op[i]) return LH_E_ARG;
    const int dev = ctxs[0]->device;
    for (int i = 0; i < n; i++)
        if (!ctxs[i] || ctxs[i]->device != dev || ctx_class(ctxs[i]) < 0) return LH_E_ARG;
    for (int i = 0; i < n; i++)  // the same context twice would share buffers
        for (int j = i + 1; j < n; j++)
            if (ctxs[i] == ctxs[j]) return LH_E_ARG;
    HIPCK(hipSetDevice(dev));
    hipStream_t s0 = ctxs[0]->stream;
    const double2 *tw, *tw16;
    int st = gang_twiddles(dev, &tw);
    if (!st) st = twiddles(dev, &tw16);
    if (st) return st;
    // group instances by size class and kernel (gangs, gangs with a field-grid
    // Raman response, one workgroup for z-dependent fills and for even batches);
    // each group is one
    // persistent launch on its own stream so the groups run concurrently.  The
    // larger grids come first: their gangs take the CUs, the others' workgroups
    // follow as those run out of jobs.  Radial contexts block the host and come
    // last.
    const bool solo = solo_pays(ctxs, op, n);
    enum { V_GANG, V_RAMAN, V_ZDEP, V_SOLO, V_SOLOR, N_VAR };
    constexpr int NG = N_VAR * LH_NCLASS;
    static const int order[LH_NCLASS] = {LH_CLASS_32768, LH_CLASS_ENV16384, LH_CLASS_16384, LH_CLASS_ENV8192,
                                         LH_CLASS_8192,  LH_CLASS_ENV4096,  LH_CLASS_4096,  LH_CLASS_RADIAL};
    auto group_of = [&](const lh_ctx* c) {
        const bool fr = c->d.transform == LH_TRANS_MODEAVG && c->d.grid_kind == LH_GRID_REAL && c->d.raman;
        SoloPrice p;
        const bool one = solo && solo_price(c, &p);
        return (c->zg_on ? V_ZDEP : fr ? (one ? V_SOLOR : V_RAMAN) : (one ? V_SOLO : V_GANG)) * LH_NCLASS + ctx_class(c);
    };
    int count[NG] = {0}, first[NG] = {0};
    for (int i = 0; i < n; i++) count[group_of(ctxs[i])]++;
    for (int c = 0; c < LH_NCLASS; c++)  // refused as before: both in one class
        if ((count[V_RAMAN * LH_NCLASS + c] || count[V_SOLOR * LH_NCLASS + c]) && count[V_ZDEP * LH_NCLASS + c])
            return LH_E_ARG;
    for (int c = 1; c < NG; c++) first[c] = first[c - 1] + count[c - 1];
    // Within a group the expensive instances come first (the gangs take them in
    // order), so the last ones to run are short: a 256-point sweep ends 10 ms
    // earlier than in the caller's order.  Every group asks for as many gangs as
    // it has instances, up to the whole chip: those of the groups behind take the
    // CUs that the ones in front leave.  (Shares of the CUs that followed the
    // groups' estimated costs left CUs idle where the estimates were off: 40
    // instances at 16384, 40 with Raman at 8192 and 40 at 4096 20.9 ms, now 10.1;
    // 60 envelope instances beside 120 at 16384 90 ms, now 13; equal for sweeps.)
    std::vector<int> pos(n), by_cost(n);
    std::vector<double> cost(n);
    for (int i = 0; i < n; i++) {
        cost[i] = solve_cost(ctxs[i], op[i]);
        by_cost[i] = i;
    }
    std::stable_sort(by_cost.begin(), by_cost.end(), [&](int a, int b) { return cost[a] > cost[b]; });
    int nwg[NG] = {0}, n_dense = 0;
    bool dense[NG] = {false};
    const auto is_gang = [](int c) { return c < V_ZDEP * LH_NCLASS && c != LH_CLASS_RADIAL; };
    const auto has_dense = [&](int c) { return is_gang(c) && lg_has_dense(c % LH_NCLASS, c >= V_RAMAN * LH_NCLASS); };
    {
        int fill[NG] = {0};
        for (int i : by_cost) {
            const int c = group_of(ctxs[i]);
            pos[i] = first[c] + fill[c]++;
        }
    }
    for (int c = 0; c < NG; c++)
        if (has_dense(c)) n_dense += count[c];
    for (int c = 0; c < NG; c++) {
        dense[c] = has_dense(c) && n_dense > LG_DENSE_ABOVE;
        if (count[c] && is_gang(c)) nwg[c] = lg_workgroups(count[c], dense[c]);
    }
    // one device block: the instances' records, each class's control block, the
    // run counters
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    size_t ctl_off[NG], total = up(sizeof(DInst) * (size_t)n);
    for (int c = 0; c < NG; c++) {
        ctl_off[c] = total;
        if (count[c] && c < V_ZDEP * LH_NCLASS && c != LH_CLASS_RADIAL)
            total += up(lg_ctl_bytes(count[c], nwg[c]));
    }
    const size_t st_off = total, in_bytes = st_off + sizeof(RunStats) * (size_t)n;
    unsigned char* dblk = nullptr;
    HIPCK(hipMalloc(&dblk, in_bytes));
    const DInst* dinst = (const DInst*)dblk;
    RunStats* dstats = (RunStats*)(dblk + st_off);
    std::vector<unsigned char> hblk(in_bytes);
    DInst* h = (DInst*)hblk.data();
    for (int c = 0; c < V_ZDEP * LH_NCLASS; c++)
        if (count[c] && c != LH_CLASS_RADIAL) lg_ctl_init(hblk.data() + ctl_off[c], count[c], nwg[c], ctxs[0]->beat);
    for (int i = 0; i < n && !st; i++)
        st = prepare_instance(ctxs[i], op[i], want_saves != 0, pos[i] >= first[V_ZDEP * LH_NCLASS], &h[pos[i]],
                              dstats + pos[i], s0);
    for (int i = 0; i < n && !st; i++) ((RunStats*)(hblk.data() + st_off))[i] = unsolved(h[i]);
    if (!st && hipMemcpyAsync(dblk, hblk.data(), in_bytes, hipMemcpyHostToDevice, s0) != hipSuccess) st = LH_E_HIP;
    std::vector<lh_stats> rad_stats(n);
    hipEvent_t ready = nullptr, done[NG] = {nullptr}, t0[NG] = {nullptr}, t1[NG] = {nullptr};
    if (!st && hipEventCreateWithFlags(&ready, hipEventDisableTiming) != hipSuccess) st = LH_E_HIP;
    if (!st && hipEventRecord(ready, s0) != hipSuccess) st = LH_E_HIP;
    for (int gi = 0; gi < NG && !st; gi++) {
        const int cls = order[gi / N_VAR], var = gi % N_VAR, c = var * LH_NCLASS + cls;
        if (!count[c]) continue;
        hipStream_t cs;
        // a class is on gangs or alone, never both: one stream, so the classes'
        // launches keep the hardware queues that let them run side by side
        if (class_stream(dev, var == V_SOLO ? cls : var == V_SOLOR ? V_RAMAN * LH_NCLASS + cls : c, &cs) != LH_OK || hipEventCreateWithFlags(&done[c], hipEventDisableTiming) != hipSuccess ||
            hipStreamWaitEvent(cs, ready, 0) != hipSuccess || hipEventCreate(&t0[c]) != hipSuccess ||
            hipEventCreate(&t1[c]) != hipSuccess || hipEventRecord(t0[c], cs) != hipSuccess) {
            st = LH_E_HIP;
            break;
        }
        if (cls == LH_CLASS_RADIAL) {
            // context by context (each fills the GPU)
            for (int i = 0; i < n && !st; i++)
                if (ctx_class(ctxs[i]) == LH_CLASS_RADIAL)
                    st = rad_solve(ctxs[i], op[i], want_saves != 0, cs, &rad_stats[i]);
            if (st) break;
        } else if (var >= V_ZDEP) {
            if (!launch_solo(cls, count[c], dinst + first[c], tw16, cs, var == V_ZDEP, var == V_SOLOR)) st = LH_E_ARG;
        } else {
            const GangLaunch l{cls, nwg[c], (GangCtl*)(dblk + ctl_off[c]), dinst + first[c], tw, cs};
            if (!(dense[c] ? lg_dense_solve(l) : launch_solve(l, var == V_RAMAN, false))) st = LH_E_ARG;
        }
        if (st || hipGetLastError() != hipSuccess || hipEventRecord(t1[c], cs) != hipSuccess ||
            hipEventRecord(done[c], cs) != hipSuccess || hipStreamWaitEvent(s0, done[c], 0) != hipSuccess)
            st = st ? st : LH_E_HIP;
    }
    std::vector<RunStats> hs(n);
    if (!st && hipMemcpyAsync(hs.data(), dstats, sizeof(RunStats) * (size_t)n, hipMemcpyDeviceToHost, s0) != hipSuccess)
        st = LH_E_HIP;
    if (hipStreamSynchronize(s0) != hipSuccess && !st) st = LH_E_HIP;
    float cls_ms[LH_NCLASS] = {0};
    int cls_n[LH_NCLASS] = {0}, cls_kind[LH_NCLASS] = {0};
    for (int c = 0; c < NG; c++) {
        float ms = 0.0f;
        cls_n[c % LH_NCLASS] += count[c];
        if (count[c])
            cls_kind[c % LH_NCLASS] |= c == LH_CLASS_RADIAL         ? LH_KIND_RADIAL
                                       : c >= V_ZDEP * LH_NCLASS    ? LH_KIND_ALONE
                                       : dense[c]                   ? LH_KIND_GANG_DENSE
                                                                    : LH_KIND_GANG;
        if (!st && t0[c] && t1[c] && hipEventElapsedTime(&ms, t0[c], t1[c]) == hipSuccess && ms > cls_ms[c % LH_NCLASS])
            cls_ms[c % LH_NCLASS] = ms;
        if (t0[c]) (void)hipEventDestroy(t0[c]);
        if (t1[c]) (void)hipEventDestroy(t1[c]);
        if (done[c]) (void)hipEventDestroy(done[c]);
    }
    for (int c = 0; c < LH_NCLASS && !st; c++) {
        g_last_ms[c] = cls_ms[c];
        g_last_n[c] = cls_n[c];
        g_last_kind[c] = cls_kind[c];
    }
    if (ready) (void)hipEventDestroy(ready);
    (void)hipFree(dblk);
    if (st) return st;
    for (int i = 0; i < n; i++) {
        stats[i] = (ctx_class(ctxs[i]) == LH_CLASS_RADIAL) ? rad_stats[i] : solved(hs[pos[i]]);
        ctxs[i]->last_status = stats[i].status;
        ctxs[i]->have_result = 1;
        ctxs[i]->result_nrec = ctxs[i]->st_on ? (int)(stats[i].accepted < ctxs[i]->st_cap ? stats[i].accepted : ctxs[i]->st_cap) : 0;
        ctxs[i]->have_records = 1;
    }
    return LH_OK;
}

int lh_batch_solve_resident(lh_ctx* const* ctxs, int n, const lh_rk_opts* o, int want_saves, lh_stats* stats) {
    if (!o || n <= 0) return LH_E_ARG;
    std::vector<const lh_rk_opts*> op((size_t)n, o);
    return batch_resident(ctxs, n, op.data(), want_saves, stats);
}

int lh_batch_solve_opts(lh_ctx* const* ctxs, int n, double* const* Ew, const lh_rk_opts* opts, double* const* saves,
                        double* const* zsaves, lh_stats* stats) {
    if (!ctxs || n <= 0 || !Ew || !opts || !stats) return LH_E_ARG;
    for (int i = 0; i < n; i++) {
        if (!ctxs[i] || !Ew[i]) return LH_E_ARG;
        int st = lh_set_state(ctxs[i], Ew[i]);
        if (st) return st;
    }
    int want = 0;
    HostPages pages;
    for (int i = 0; i < n; i++)
        if (saves && saves[i]) {
            want = 1;
            pages.add(saves[i], sizeof(double2) * (size_t)ctxs[i]->n_state * (size_t)std::max(opts[i].save_n, 0));
        }
    std::vector<const lh_rk_opts*> op((size_t)n);
    for (int i = 0; i < n; i++) op[i] = opts + i;
    pages.start();
    int st = batch_resident(ctxs, n, op.data(), want, stats);
    pages.wait();
    if (st) return st;
    for (int i = 0; i < n && !st; i++) {
        st = lh_get_state(ctxs[i], Ew[i]);
        if (!st && ((saves && saves[i]) || (zsaves && zsaves[i])))
            st = lh_get_saves(ctxs[i], saves ? saves[i] : nullptr, zsaves ? zsaves[i] : nullptr);
    }
    return st;
}

int lh_set_step_stats(lh_ctx* c, const lh_stats_desc* sd) {
    if (!c) return LH_E_ARG;
    if (!sd) {
        c->st_on = 0;
        return LH_OK;
    }
    if (c->d.transform != LH_TRANS_MODEAVG || ctx_class(c) == LH_CLASS_ENV16384 || ctx_class(c) == LH_CLASS_32768)
        return LH_E_ARG;
    HIPCK(hipSetDevice(c->device));
    if (sd->capacity < 0 || !sd->energy_w || !sd->t || !(sd->aeff > 0) || !c->omega) return LH_E_ARG;
    if (sd->n_windows < 0 || sd->n_windows > LH_STAT_MAX_WINDOWS || (sd->n_windows > 0 && !sd->window_w))
        return LH_E_ARG;
    double* ew = nullptr;
    double* tg = nullptr;
    double* wn = nullptr;
    int st = shared_upload(c->device, &ew, sd->energy_w, (size_t)c->d.n_omega);
    if (!st) st = shared_upload(c->device, &tg, sd->t, (size_t)c->d.n_t);
    if (!st && sd->n_windows > 0)
        st = shared_upload(c->device, &wn, sd->window_w, (size_t)sd->n_windows * (size_t)c->d.n_omega);
    if (!st && !c->st_rec1 && hipMalloc(&c->st_rec1, sizeof(double) * LH_NSTAT) != hipSuccess) st = LH_E_NOMEM;
    if (!st && sd->capacity > c->st_cap) {
        if (c->steprec) (void)hipFree(c->steprec);
        c->steprec = nullptr;
        c->st_cap = 0;
        if (hipMalloc(&c->steprec, sizeof(double) * LH_NSTAT * (size_t)sd->capacity) != hipSuccess) st = LH_E_NOMEM;
    }
    if (st) {
        shared_release(ew);
        shared_release(tg);
        shared_release(wn);
        return st;
    }
    shared_release(c->st_ew);
    shared_release(c->st_t);
    shared_release(c->st_win);
    c->st_ew = ew;
    c->st_t = tg;
    c->st_win = wn;
    c->st_nwin = sd->n_windows;
    c->st_cap = sd->capacity;
    c->st_aeff = sd->aeff;
    c->st_ediv = sqrt(EPS0 * CLIGHT * sd->aeff / 2);  // sqrt(ε_0*c*aeff(z)/2), src/Stats.jl:236
    c->st_on = 1;
    c->result_nrec = 0;
    return LH_OK;
}

static void zg_release(lh_ctx* c) {
    for (const void* p : {(const void*)c->zg_Z, (const void*)c->zg_P, (const void*)c->zfd, (const void*)c->zgam,
                          (const void*)c->zd, (const void*)c->znwg, (const void*)c->zpre, (const void*)c->zU,
                          (const void*)c->zV, (const void*)c->zfdt, (const void*)c->zt_Z, (const void*)c->zt_A})
        shared_release(p);
    c->zt_Z = c->zt_A = nullptr;
    c->zt_n = 0;
    c->zg_Z = c->zg_P = c->zfd = c->zgam = nullptr;
    c->zd = nullptr;
    c->znwg = c->zpre = nullptr;
    c->zU = c->zfdt = nullptr;
    c->zV = nullptr;
    c->zg_taper = 0;
}

int lh_set_gradient(lh_ctx* c, const lh_gradient_desc* g) {
    if (!c) return LH_E_ARG;
    HIPCK(hipSetDevice(c->device));
    if (!g) {
        c->zg_on = 0;
        zg_release(c);
        return LH_OK;
    }
    const lh_desc& d = c->d;
    // (a Raman response depends on the density; with ρ(z) it would change along z)
    if (d.transform != LH_TRANS_MODEAVG || d.grid_kind != LH_GRID_REAL || !c->omega || !c->zsidx || d.raman ||
        ctx_class(c) == LH_CLASS_32768)
        return LH_E_ARG;
    if (g->n_points < 2 || !g->Z || !g->P || g->dens_n < 4 || !g->dens_p || !g->dens_rho || !g->dens_d ||
        !g->gamma || !g->nwg || !g->pre || !g->fd || !(g->fd_h > 0) || !(g->sqrt_aeff > 0) ||
        (g->model != 0 && g->model != 1) || (g->two_point && g->n_points != 2) || g->taper < 0 || g->taper > 2)
        return LH_E_ARG;
    if (g->taper && (!(g->sqrt_aeff_intg > 0) || !g->wgU || !g->wgV || !g->fdt)) return LH_E_ARG;
    if (g->taper == 1 && (!(g->taper_a0 > 0) || !(g->taper_a1 > 0) || !(g->taper_L > 0))) return LH_E_ARG;
    if (g->taper == 2) {
        if (g->taper_n < 2 || !g->taper_Z || !g->taper_A) return LH_E_ARG;
        for (int i = 0; i < g->taper_n; i++)
            if (!(g->taper_A[i] > 0) || (i > 0 && !(g->taper_Z[i - 1] < g->taper_Z[i]))) return LH_E_ARG;
    }
    for (int i = 0; i + 1 < g->n_points; i++)
        if (!(g->Z[i] < g->Z[i + 1])) return LH_E_ARG;
    if (g->two_point && !(g->Z[0] == 0.0)) return LH_E_ARG;
    const size_t N = (size_t)d.n_omega;
    std::vector<double4> spl((size_t)g->dens_n);
    for (int i = 0; i < g->dens_n; i++) spl[i] = make_double4(g->dens_p[i], g->dens_rho[i], g->dens_d[i], 0.0);
    zg_release(c);
    const double2* tw;
    int st = twiddles(c->device, &tw);
    if (!st) st = shared_upload(c->device, &c->zg_Z, g->Z, (size_t)g->n_points);
    if (!st) st = shared_upload(c->device, &c->zg_P, g->P, (size_t)g->n_points);
    if (!st) st = shared_upload(c->device, &c->zd, spl.data(), spl.size());
    if (!st) st = shared_upload(c->device, &c->zgam, g->gamma, N);
    if (!st) st = shared_upload(c->device, &c->znwg, g->nwg, N);
    if (!st) st = shared_upload(c->device, &c->zpre, g->pre, N);
    if (!st) st = shared_upload(c->device, &c->zfd, g->fd, (size_t)36);
    if (!st && g->taper) st = shared_upload(c->device, &c->zU, g->wgU, N);
    if (!st && g->taper) st = shared_upload(c->device, &c->zV, g->wgV, N);
    if (!st && g->taper) st = shared_upload(c->device, &c->zfdt, g->fdt, (size_t)27);
    if (!st && g->taper == 2) st = shared_upload(c->device, &c->zt_Z, g->taper_Z, (size_t)g->taper_n);
    if (!st && g->taper == 2) st = shared_upload(c->device, &c->zt_A, g->taper_A, (size_t)g->taper_n);
    if (!st && !c->zL && hipMalloc(&c->zL, sizeof(double2) * lg_stride(d)) != hipSuccess) st = LH_E_NOMEM;
    if (!st && !c->zOF && hipMalloc(&c->zOF, sizeof(double2) * lg_stride(d)) != hipSuccess) st = LH_E_NOMEM;
    if (st) {
        zg_release(c);
        c->zg_on = 0;
        return st;
    }
    c->zg_np = g->n_points;
    c->zg_two = g->two_point;
    c->zg_model = g->model;
    c->zg_loss = g->loss;
    c->zd_n = g->dens_n;
    c->zsqrt_aeff = g->sqrt_aeff;
    c->zfd_h = g->fd_h;
    c->zg_taper = g->taper;
    c->zg_a0 = g->taper_a0;
    c->zg_a1 = g->taper_a1;
    c->zg_aL = g->taper_L;
    c->zg_sqrt_intg = g->sqrt_aeff_intg;
    c->zt_n = (g->taper == 2) ? g->taper_n : 0;
    c->zg_on = 1;
    st = rhs_set_ready(c, &c->rset[RHS_CAPTURED], c->stream);
    if (st) {
        zg_release(c);
        c->zg_on = 0;
    }
    return st;
}

int lh_stats_eval(lh_ctx* c, const double* Ew, double z, double dz, double* rec) {
    if (!c || !Ew || !rec || !c->st_on) return LH_E_ARG;
    HIPCK(hipSetDevice(c->device));
    const size_t bytes = sizeof(double2) * (size_t)c->n_state;
    if (!c->rhs_in) {
        HIPCK(hipMalloc(&c->rhs_in, bytes));
        HIPCK(hipMalloc(&c->rhs_out, bytes));
    }
    const double2* tw;
    int st = gang_twiddles(c->device, &tw);
    if (st) return st;
    DInst in = base_inst(c);
    in.rhs_in = c->rhs_in;
    in.steprec = c->st_rec1;
    HIPCK(hipMemcpyAsync(c->rhs_in, Ew, bytes, hipMemcpyHostToDevice, c->stream));
    GangLaunch l;
    st = rhs_launch_of(c, &in, tw, c->stream, &l);
    if (st) return st;
    if (!launch_stats(l, z, dz, c->dstatus)) return LH_E_ARG;
    HIPCK(hipGetLastError());
    int kst = LH_OK;
    HIPCK(hipMemcpyAsync(rec, c->st_rec1, sizeof(double) * LH_NSTAT, hipMemcpyDeviceToHost, c->stream));
    HIPCK(hipMemcpyAsync(&kst, c->dstatus, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HIPCK(hipStreamSynchronize(c->stream));
    return kst;
}

int lh_get_step_stats(lh_ctx* c, double* rec, int capacity, int* n) {
    if (!c || !n || capacity < 0 || (!rec && capacity > 0) || !c->have_records) return LH_E_ARG;
    HIPCK(hipSetDevice(c->device));
    int k = c->result_nrec < capacity ? c->result_nrec : capacity;
    if (k > 0) HIPCK(hipMemcpy(rec, c->steprec, sizeof(double) * LH_NSTAT * (size_t)k, hipMemcpyDeviceToHost));
    *n = k;
    return LH_OK;
}

int lh_last_launch_times(double* ms, int* n_inst, int nclass) {
    if (!ms || !n_inst || nclass < LH_NCLASS) return LH_E_ARG;
    for (int c = 0; c < LH_NCLASS; c++) {
        ms[c] = g_last_ms[c];
        n_inst[c] = g_last_n[c];
    }
    return LH_OK;
}

int lh_last_launch_kinds(int* kinds, int nclass) {
    if (!kinds || nclass < LH_NCLASS) return LH_E_ARG;
    for (int c = 0; c < LH_NCLASS; c++) kinds[c] = g_last_kind[c];
    return LH_OK;
}

int lh_host_alloc(size_t bytes, void** ptr) {
    if (!ptr || bytes == 0) return LH_E_ARG;
    *ptr = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return LH_E_NODEVICE;
    if (hipHostMalloc(ptr, bytes, hipHostMallocDefault) != hipSuccess) {
        *ptr = nullptr;
        return LH_E_NOMEM;
    }
    return LH_OK;
}

int lh_host_free(void* ptr) {
    if (!ptr) return LH_OK;
    return hipHostFree(ptr) == hipSuccess ? LH_OK : LH_E_HIP;
}

int lh_get_plan(const lh_ctx* c, lh_plan* p) {
    if (!c || !p) return LH_E_ARG;
    if (c->d.transform != LH_TRANS_RADIAL) return LH_E_ARG;
    p->fft_radix_plan = c->rplan.fft;
    p->gemm_tiles = c->rplan.mt;
    p->rhs_us = 0.0;
    p->agrees = 1;
    return LH_OK;
}

int lh_set_plan(lh_ctx* c, const lh_plan* p) {
    if (!c || !p || c->d.transform != LH_TRANS_RADIAL) return LH_E_ARG;
    const RadPlan np = {p->fft_radix_plan, p->gemm_tiles};
    if (!rad_plan_ok(np)) return LH_E_ARG;
    const RadPlan run = rad_plan_run(c);
    if (np.fft != run.fft || np.mt != run.mt) {
        HIPCK(hipSetDevice(c->device));
        HIPCK(hipStreamSynchronize(c->stream));
        if (c->rgraph) {  // captured with the old plan
            (void)hipGraphExecDestroy(c->rgraph);
            c->rgraph = nullptr;
        }
    }
    c->rplan = np;
    c->rplan_own = 1;
    return LH_OK;
}

int lh_plan_tiles(const lh_ctx* c, int* tiles) {
    if (!c || !tiles || c->d.transform != LH_TRANS_RADIAL) return LH_E_ARG;
    *tiles = rad_plan_run(c).mt;
    return LH_OK;
}

// Measures every plan on one RHS of ctx's shape (the field Ew, or zero when
// NULL) and installs the fastest in ctx and in the wisdom.  Each plan runs
// once untimed, then reps times between two events on the context's stream;
// a plan whose RHS differs from the default plan's by more than 1e-12
// (relative L2) is never chosen.
int lh_autotune(lh_ctx* c, const double* Ew, int reps, lh_plan* tried, int cap, int* n_tried) {
    if (!c || reps < 1 || (cap > 0 && !tried) || c->d.transform != LH_TRANS_RADIAL) return LH_E_ARG;
    HIPCK(hipSetDevice(c->device));
    const double2* tw;
    int st = twiddles(c->device, &tw);
    if (st) return st;
    hipStream_t s = c->stream;
    const size_t n = (size_t)c->n_state;
    double2 *din = nullptr, *dout = nullptr;
    if (hipMalloc(&din, sizeof(double2) * n) != hipSuccess) return LH_E_NOMEM;
    if (hipMalloc(&dout, sizeof(double2) * n) != hipSuccess) {
        (void)hipFree(din);
        return LH_E_NOMEM;
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    std::vector<double2> ref(n), out(n);
    RadPlan plans[6];
    int np = 0;
    plans[np++] = RAD_DEFAULT_PLAN;
    for (int f = 0; f < 2; f++)
        for (int mt : {1, 2, 4})
            if (!(f == RAD_DEFAULT_PLAN.fft && mt == RAD_DEFAULT_PLAN.mt)) plans[np++] = {f, mt};
    RadPlan best = RAD_DEFAULT_PLAN;
    double best_us = 0.0;
    st = LH_OK;
    do {
        if (Ew) {
            if (hipMemcpy(din, Ew, sizeof(double2) * n, hipMemcpyHostToDevice) != hipSuccess) { st = LH_E_HIP; break; }
        } else if (hipMemset(din, 0, sizeof(double2) * n) != hipSuccess) { st = LH_E_HIP; break; }
        if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) { st = LH_E_HIP; break; }
        RadArgs a = rad_args(c, 1);
        a.rhs_in = din;
        a.rhs_out = dout;
        RadCtl h;
        rad_ctl_init(&h, nullptr);
        if (hipStreamSynchronize(s) != hipSuccess ||
            hipMemcpy(c->rargs + 1, &a, sizeof(a), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(c->rctl + 1, &h, sizeof(h), hipMemcpyHostToDevice) != hipSuccess) { st = LH_E_HIP; break; }
        double refn = 0.0;
        for (int i = 0; i < np && !st; i++) {
            const RadPlan p = plans[i];
            rad_rhs_dispatch(p, c->d.grid_kind == LH_GRID_ENV, c->d.n_to, c->d.n_r, c->rargs + 1, tw, -1, s);
            if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) { st = LH_E_HIP; break; }
            if (hipMemcpy(i == 0 ? ref.data() : out.data(), dout, sizeof(double2) * n, hipMemcpyDeviceToHost) !=
                hipSuccess) { st = LH_E_HIP; break; }
            double dn = 0.0;
            if (i == 0) {
                for (size_t k = 0; k < n; k++) refn += ref[k].x * ref[k].x + ref[k].y * ref[k].y;
            } else {
                for (size_t k = 0; k < n; k++) {
                    const double dx = out[k].x - ref[k].x, dy = out[k].y - ref[k].y;
                    dn += dx * dx + dy * dy;
                }
            }
            const bool agrees = !(dn > 1e-24 * refn);
            (void)hipEventRecord(e0, s);
            for (int r = 0; r < reps; r++) rad_rhs_dispatch(p, c->d.grid_kind == LH_GRID_ENV, c->d.n_to, c->d.n_r, c->rargs + 1, tw, -1, s);
            (void)hipEventRecord(e1, s);
            float ms = 0.0f;
            if (hipGetLastError() != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                hipEventElapsedTime(&ms, e0, e1) != hipSuccess) { st = LH_E_HIP; break; }
            const double us = 1e3 * (double)ms / reps;
            if (i < cap) {
                tried[i].fft_radix_plan = p.fft;
                tried[i].gemm_tiles = p.mt;
                tried[i].rhs_us = us;
                tried[i].agrees = agrees ? 1 : 0;
            }
            if (agrees && (i == 0 || us < best_us)) {
                best = p;
                best_us = us;
            }
        }
    } while (0);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(din);
    (void)hipFree(dout);
    if (st) return st;
    if (n_tried) *n_tried = np;
    lh_plan bp = {best.fft, best.mt, best_us, 1};
    st = lh_set_plan(c, &bp);
    if (!st) wisdom_record(c->d.n_to, c->d.n_r, best, best_us);
    return st;
}

// Wisdom as text: a header line, then one line per shape
// "radial <n_to> <n_r> <fft_radix_plan> <gemm_tiles> <rhs_us>".
int lh_wisdom_export(char* buf, size_t cap, size_t* len) {
    std::string t = "luna-hip-wisdom 1\n";
    {
        std::lock_guard<std::mutex> lk(g_wisdom_mu);
        char line[128];
        for (const WisdomEntry& w : g_wisdom) {
            snprintf(line, sizeof(line), "radial %d %d %d %d %.3f\n", w.n_to, w.n_r, w.plan.fft, w.plan.mt, w.us);
            t += line;
        }
    }
    if (len) *len = t.size() + 1;
    if (!buf) return LH_OK;
    if (cap < t.size() + 1) return LH_E_ARG;
    memcpy(buf, t.c_str(), t.size() + 1);
    return LH_OK;
}

int lh_wisdom_import(const char* text) {
    if (!text) return LH_E_ARG;
    std::vector<WisdomEntry> got;
    const char* p = text;
    int lineno = 0;
    while (*p) {
        const char* e = strchr(p, '\n');
        std::string line = e ? std::string(p, e - p) : std::string(p);
        p = e ? e + 1 : p + line.size();
        if (lineno++ == 0) {
            if (line != "luna-hip-wisdom 1") return LH_E_ARG;
            continue;
        }
        if (line.empty()) continue;
        WisdomEntry w;
        char kind[16];
        int used = 0;
        if (sscanf(line.c_str(), "%15s %d %d %d %d %lf%n", kind, &w.n_to, &w.n_r, &w.plan.fft, &w.plan.mt, &w.us,
                   &used) != 6 || strcmp(kind, "radial") != 0 || (size_t)used != line.size() || !rad_plan_ok(w.plan) ||
            !rad_size_ok(w.n_to) || w.n_r < 64 || w.n_r % 64 != 0)
            return LH_E_ARG;
        got.push_back(w);
    }
    if (lineno == 0) return LH_E_ARG;
    for (const WisdomEntry& w : got) wisdom_record(w.n_to, w.n_r, w.plan, w.us);
    return LH_OK;
}

int lh_wisdom_forget(void) {
    std::lock_guard<std::mutex> lk(g_wisdom_mu);
    g_wisdom.clear();
    return LH_OK;
}

// Offsets of the working memory of one lh_solve_noalloc call inside `scratch`
// (each part 256-byte aligned): control block and instance record, run
// counters, save grid, the gang's work block.  The exchange area is the
// context's.
struct NoallocLayout {
    size_t inst, stats, zgrid, k, total;
};
static NoallocLayout noalloc_layout(const lh_desc& d, int save_n) {
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    NoallocLayout L;
    L.inst = 0;
    L.stats = up(LAUNCH1_BYTES);
    L.zgrid = L.stats + up(sizeof(RunStats));
    L.k = L.zgrid + up(sizeof(double) * (size_t)(save_n > 0 ? save_n : 1));
    L.total = L.k + sizeof(double2) * lg_stride(d) * LG_SLOTS;
    return L;
}

// The problems lh_solve_noalloc takes.  The bound is what a solver with one
// workgroup needs: record (1 KB), counters, save grid, a second state, eight
// stage vectors and the series of a Raman response or of the largest grids within
// LH_NOALLOC_SCRATCH_BYTES; the gangs' layout (noalloc_layout) of every such
// problem fits the array.
static bool noalloc_fits(const lh_ctx* c, int save_n) {
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const lh_desc& d = c->d;
    const size_t ns = (size_t)c->n_state, nto = (size_t)d.n_to;
    const int cls = ctx_class(c);
    const size_t series = cls == LH_CLASS_ENV16384 ? nto * 5 / 2
                          : cls == LH_CLASS_32768  ? nto * 3 / 4
                          : !d.raman               ? 0
                          : d.grid_kind == LH_GRID_REAL ? nto * 2
                                                        : nto;
    return 1024 + up(sizeof(lh_stats)) + up(sizeof(double) * (size_t)(save_n > 0 ? save_n : 1)) +
               up(sizeof(double2) * ns) + sizeof(double2) * ((ns + 15) & ~(size_t)15) * 8 + up(sizeof(double2) * series) <=
           LH_NOALLOC_SCRATCH_BYTES;
}

int lh_solve_noalloc(lh_ctx* c, void* Ew_dev, const lh_rk_opts* o, void* saves_dev, double* zsaves, lh_stats* stats,
                     void* stream) {
    if (!c || !Ew_dev || !o || !stats || !opts_ok(o)) return LH_E_ARG;
    const int cls = ctx_class(c);
    if (c->d.transform != LH_TRANS_MODEAVG || cls < 0 || cls == LH_CLASS_RADIAL) return LH_E_ARG;
    const NoallocLayout L = noalloc_layout(c->d, o->save_n);
    if (!noalloc_fits(c, o->save_n) || L.total > SCRATCH_BYTES) return LH_E_TOO_LARGE;
    HIPCK(hipSetDevice(c->device));
    unsigned char* base = scratch_existing(c->device);
    const double2* tw = table_existing(g_gtw, c->device);
    const double2* tw16 = table_existing(g_tw, c->device);  // there for a z-dependent fill (lh_set_gradient)
    if (!base || !tw || (c->zg_on && !tw16)) return LH_E_HIP;  // set by lh_create on this device
    hipStream_t s = stream ? (hipStream_t)stream : c->stream;
    DInst in = base_inst(c);
    in.Yin = (const double2*)Ew_dev;  // read once into Y, the same buffer
    in.Y = (double2*)Ew_dev;          // receives the final state
    in.K = (double2*)(base + L.k);
    in.kstride = (long long)lg_stride(c->d);
    in.saves = (double2*)saves_dev;
    in.zgrid = (const double*)(base + L.zgrid);
    in.stats = (RunStats*)(base + L.stats);
    inst_options(&in, o);
    // Nothing in the working memory needs clearing: the kernel writes every
    // state and stage vector before reading it, and the counters at the end.
    // The save grid is staged on this stack frame; each copy is waited for
    // before the frame's buffer is reused or left.
    const int st = set_launch1(base + L.inst, in, s);
    if (st) return st;
    const int zn = o->save_n > 0 ? o->save_n : 1;
    double chunk[256];
    for (int i0 = 0; i0 < zn; i0 += 256) {
        const int m = (zn - i0 < 256) ? zn - i0 : 256;
        for (int i = 0; i < m; i++) chunk[i] = save_grid_at(o, i0 + i);
        HIPCK(hipMemcpyAsync(base + L.zgrid + sizeof(double) * (size_t)i0, chunk, sizeof(double) * (size_t)m,
                             hipMemcpyHostToDevice, s));
        HIPCK(hipStreamSynchronize(s));
    }
    const GangLaunch l = launch1_of(c, base + L.inst, tw, s);
    if (c->zg_on)
        (void)launch_solo(cls, 1, l.d, tw16, s, true, false);
    else if (!launch_solve(l, c->d.raman != 0, false))
        return LH_E_ARG;
    HIPCK(hipGetLastError());
    RunStats rs;
    HIPCK(hipMemcpyAsync(&rs, base + L.stats, sizeof(rs), hipMemcpyDeviceToHost, s));
    HIPCK(hipStreamSynchronize(s));
    const lh_stats hs = solved(rs);
    if (zsaves && o->save_n > 0) save_grid_into(o, zsaves);
    *stats = hs;
    c->last_status = hs.status;
    // the state and saves went to the caller's buffers, not the context's
    c->have_result = 0;
    c->result_nrec = c->st_on ? (int)(hs.accepted < c->st_cap ? hs.accepted : c->st_cap) : 0;
    c->have_records = 1;
    return hs.status;
}

int lh_batch_solve(lh_ctx* const* ctxs, int n, double* const* Ew, const lh_rk_opts* o, double* const* saves,
                   double* const* zsaves, lh_stats* stats) {
    if (!ctxs || n <= 0 || !Ew || !o || !stats) return LH_E_ARG;
    for (int i = 0; i < n; i++) {
        if (!ctxs[i] || !Ew[i]) return LH_E_ARG;
        int st = lh_set_state(ctxs[i], Ew[i]);
        if (st) return st;
    }
    int want = 0;
    HostPages pages;
    for (int i = 0; i < n; i++)
        if (saves && saves[i]) {
            want = 1;
            pages.add(saves[i], sizeof(double2) * (size_t)ctxs[i]->n_state * (size_t)std::max(o->save_n, 0));
        }
    pages.start();
    int st = lh_batch_solve_resident(ctxs, n, o, want, stats);
    pages.wait();
    if (st) return st;
    for (int i = 0; i < n && !st; i++) {
        st = lh_get_state(ctxs[i], Ew[i]);
        if (!st && ((saves && saves[i]) || (zsaves && zsaves[i])))
            st = lh_get_saves(ctxs[i], saves ? saves[i] : nullptr, zsaves ? zsaves[i] : nullptr);
    }
    return st;
}

}  // extern "C"
