// lh_core.h -- what the propagation kernels share: the instance record, the
// Dormand–Prince tableau, the PPT spline, workgroup scans, the pointwise plasma
// and Kerr responses, stage prologue and window filter of one column, the
// z-dependent fill's functions and the size classes.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "../../include/luna_hip.h"
#include "lh_device.h"

// --------------------------------------------------------------------------
// Device-side instance description
// --------------------------------------------------------------------------
// An instance's counters, and a word that any workgroup sets which lost another
// one of its gang (lh_gang_proto.h): the run's status is then LH_E_HIP, whatever
// the one that wrote the counters knew.
struct RunStats {
    lh_stats s;
    int lost, pad;
};

struct DInst {
    int grid_kind, transform, n_omega, n_t, n_to, n_r;
    int kerr, plasma, raman, ppt_n;
    double density, kerr_fac, ionpot, preion_p1, e_ratio;
    double dt_o, e_scale, inv_nt, sc_t, ppt_emin, ppt_emax;
    const double* omega_win;
    const double* t_win;
    const double* to_win;
    const double2* linop;
    const double2* outfac;  // per-bin output factor: sc_f·norm·ωwin (sidx) or sc_f
    const double4* ppt;     // (x, y, D, 0) per spline node
    // envelope grid
    double kerr34;          // ¾·ρ·ε0·γ3 (Kerr_env)
    double inv_2n;          // 1/(2·Nto): inverse of the zero-padded Raman transform
    const double2* hwdt;    // rfft of h(t) zero-padded to 2·Nto, times δt: bins 0..Nto
    double2* escr;          // field-grid Raman: E(t) and P(t) of the member's times
    double2* gx;            // exchange area of the gang (lh_gang.h)
    int gx_len;             // points of one of its two series
    // solver state
    const double2* Yin;  // initial field (never written)
    double2* Y;          // receives the final state s.yn
    double2* K;          // work block: vector j at K + j·kstride (LgVec)
    long long kstride;
    double2* saves;       // [save_n][n_state] or null
    const double* zgrid;  // [save_n]
    RunStats* stats;
    double z0, zmax, rtol, atol, safety, max_dz, min_dz, init_dz;
    int repeat_limit, save_n;
    int save_first;       // saves already written (a resumed run continues at this index)
    double zstop;         // > 0: stop after the first accepted step with tn > zstop
    long long max_steps;  // cap on step attempts
    // single-RHS I/O
    const double2* rhs_in;
    double2* rhs_out;
    // per-step statistics (steprec null: off)
    const double* st_omega;  // [Nω] ω
    const double* st_ew;     // [Nω] energy quadrature weights
    const double* st_t;      // [Nt] grid.t
    double st_aeff;          // Aeff
    double st_ediv;          // sqrt(ε0·c·Aeff/2)
    const double* st_win;    // [st_nwin][Nω] energy_w·window² of each energy window
    int st_nwin;
    double* steprec;         // [steprec_cap][LH_NSTAT]
    int steprec_cap;
    // z-dependent fill (pressure gradient); zg_np = 0: constant fill
    int zg_np, zg_two, zg_model, zg_loss, zd_n;
    double sc_f;             // to_freq! crop scale (Nω-1)/(No-1)
    double kerr_gamma3;      // γ3 of Kerr_field (0 without Kerr)
    double zsqrt_aeff, zfd_h;
    const double* zg_Z;      // [zg_np] profile positions
    const double* zg_P;      // [zg_np] profile pressures
    const double4* zd;       // [zd_n] density spline (P, ρ, D, 0)
    const double* zgam;      // [Nω] γ(λ)
    const double2* znwg;     // [Nω] neff_wg
    const double2* zpre;     // [Nω] norm prefactor
    const unsigned char* zsidx;  // [Nω]
    const double* zfd;       // [9][4] β1 stencil (ω, γ, nwg)
    int ztaper;              // 1: linear taper a(z), 2: piecewise linear; neff_wg from zU, zV
    double za0, za1, zaL, zsqrt_intg;
    int zt_n;                // taper = 2: nodes
    const double* zt_Z;      // [zt_n] positions
    const double* zt_A;      // [zt_n] radii
    const double* zU;        // [Nω] u_nm/k
    const double2* zV;       // [Nω] v_n/k
    const double* zfdt;      // [9][3] U, V at the β1 stencil points
    double2* zL;             // operator at the last refresh (in the members' order in lh_gang.h)
    double2* zOF;            // output factor at the last refresh, likewise
    // streaming output (lh_solve_stream; pub null: off): device-mapped,
    // page-locked host memory.  A step that writes saves publishes itself:
    // its filtered state and (z, dz, saved, accepted) go to slot k & 1 of
    // publication k, then pub is set to k + 1 with a system-scope release.
    unsigned long long* pub;
    double* pub_info;        // [2][4]
    double2* pub_y;          // [2][n_state]
    const int* pub_stop;     // set by the host: end with LH_E_STOPPED at the next publication
    // every-step mode (pub_ring > 0): every accepted step publishes, into
    // slot k % pub_ring of pub_ring slots (pub_info and pub_y hold that many);
    // the kernel never waits, the host checks that it has not been lapped
    int pub_ring;
    unsigned* beat;          // a word of the device that every solver changes at each step attempt
};

// Dormand–Prince tableau, src/dopri.jl:1-28 (rational literals evaluated in double).
static __constant__ double c_B[6][6] = {
    {1.0 / 5, 0, 0, 0, 0, 0},
    {3.0 / 40, 9.0 / 40, 0, 0, 0, 0},
    {44.0 / 45, -56.0 / 15, 32.0 / 9, 0, 0, 0},
    {19372.0 / 6561, -25360.0 / 2187, 64448.0 / 6561, -212.0 / 729, 0, 0},
    {9017.0 / 3168, -355.0 / 33, 46732.0 / 5247, 49.0 / 176, -5103.0 / 18656, 0},
    {35.0 / 384, 0, 500.0 / 1113, 125.0 / 192, -2187.0 / 6784, 11.0 / 84}};
static __constant__ double c_nodes[6] = {1.0 / 5, 3.0 / 10, 4.0 / 5, 8.0 / 9, 1, 1};
static __constant__ double c_b5[7] = {5179.0 / 57600, 0, 7571.0 / 16695, 393.0 / 640, -92097.0 / 339200, 187.0 / 2100, 1.0 / 40};
static __constant__ double c_b4[7] = {35.0 / 384, 0, 500.0 / 1113, 125.0 / 192, -2187.0 / 6784, 11.0 / 84, 0};
static __constant__ double c_iC[4][7] = {
    {1, 0, 0, 0, 0, 0, 0},
    {-183.0 / 64, 0, 1500.0 / 371, -125.0 / 32, 9477.0 / 3392, -11.0 / 7, 3.0 / 2},
    {37.0 / 12, 0, -1000.0 / 159, 125.0 / 12, -729.0 / 106, 11.0 / 3, -4},
    {-145.0 / 128, 0, 1000.0 / 371, -375.0 / 64, 25515.0 / 6784, -55.0 / 28, 5.0 / 2}};

// LDS of one workgroup: the padded transform buffer sized for the largest
// transform it runs (MO complex points + Nyquist), twiddles, scan scratch.
// plist: the rates of the samples that need one (the few hundred under the
// pulse), so that every thread takes one or two of them instead of the
// threads owning the pulse doing all of that work: a compacted list up to
// Nto = 8192, a window [lo, hi] of the round for Nto = 16384, whose 149 KB of
// other buffers leave 11 KB (1408 samples) for it.
template <int MO>
struct PList {
    // what the largest class's LDS leaves after the buffer, twiddles and the
    // per-wave reduction and scan slots
    static constexpr int CAP = (MO >= 8192) ? 1344 - 19 * (LH_NW - 8) : 4096;
};

template <int MO>
struct SmemT {
    double2 buf[padded_len(MO)];
    TwLds tw;
    double wsum[5 * LH_NW];      // block_sum3/block_sum4 and the statistics reductions
    double scan[2][7 * LH_NW];   // one-barrier scans and min/max, used in alternation
    double plist[PList<MO>::CAP];
    double zs[3];  // gradient fill: ρ(z), β1(z), taper radius a(z) from thread 0
    int flag;
};

// Number of state bins each thread owns for an oversampled half-length MO.
template <int MO>
struct Bins {
    static constexpr int N = MO / 2 + 1;  // Nω of a real grid with Nto = 2·MO, Nt = MO
    static constexpr int NPT = (N + LH_T - 1) / LH_T;
};

// --------------------------------------------------------------------------
// Maths.CSpline evaluation on uniform nodes (x, y, D) with the uniform index
// rule (src/Maths.jl:771-775, 840-848).  The PPT table (log rate) and the
// density-vs-pressure spline of a gradient fill use it.
// --------------------------------------------------------------------------
__device__ __forceinline__ double cspline_uniform(const double4* nodes, int n, double xmin, double xmax, double x) {
    int i;
    if (x <= xmin)
        i = 2;
    else if (x >= xmax)
        i = n;
    else
        i = (int)ceil((x - xmin) / (xmax - xmin) * (double)(n - 1)) + 1;
    i = min(max(i, 2), n);
    const double4 pc = nodes[i - 1], pm = nodes[i - 2];
    if (x == pc.x) return pc.y;
    if (x == pm.x) return pm.y;
    const double t = (x - pm.x) / (pc.x - pm.x);
    return (pm.y + pm.z * t + (3 * (pc.y - pm.y) - 2 * pm.z - pc.z) * (t * t) +
            (2 * (pm.y - pc.y) + pm.z + pc.z) * (t * t * t));
}

// The same for Q samples at once: every index first, then all table loads,
// then the splines, so the loads of a thread's samples are in flight together
// instead of forming one dependent load-and-wait chain per sample.  Inactive
// samples (below the table, or out of range) load the first interval and are
// discarded.
template <int Q>
__device__ __forceinline__ void ppt_rates(const DInst& in, const double* aE, double* rate, int& bad) {
    const double xmin = in.ppt_emin, xmax = in.ppt_emax;
    const int n = in.ppt_n;
    int idx[Q];
    bool act[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const double x = aE[q];
        const bool below = x < xmin;
        const bool out = !below && !(x <= xmax);  // above the table, or NaN
        if (out) bad = (x > xmax) ? LH_E_PPT_RANGE : LH_E_NONFINITE;
        act[q] = !below && !out;
        int i = 2;
        if (act[q]) {
            if (x <= xmin)
                i = 2;
            else if (x >= xmax)
                i = n;
            else
                i = (int)ceil((x - xmin) / (xmax - xmin) * (double)(n - 1)) + 1;
            i = min(max(i, 2), n);
        }
        idx[q] = i;
    }
    double4 pc[Q], pm[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        pc[q] = gl(in.ppt)[idx[q] - 1];
        pm[q] = gl(in.ppt)[idx[q] - 2];
    }
#pragma unroll
    for (int q = 0; q < Q; q++) {
        double r = 0.0;
        if (act[q]) {
            const double x = aE[q];
            double v;
            if (x == pc[q].x) {
                v = pc[q].y;
            } else if (x == pm[q].x) {
                v = pm[q].y;
            } else {
                const double t = (x - pm[q].x) / (pc[q].x - pm[q].x);
                v = (pm[q].y + pm[q].z * t + (3 * (pc[q].y - pm[q].y) - 2 * pm[q].z - pc[q].z) * (t * t) +
                     (2 * (pm[q].y - pc[q].y) + pm[q].z + pc[q].z) * (t * t * t));
            }
            r = exp(v);
        }
        rate[q] = r;
    }
}

// cumtrapz over the workgroup for one round of QR samples per thread (global
// index g0+q), with a single barrier.  The trapezoid joining a thread's first
// sample to its predecessor's last comes from a lane move inside a
// wavefront; for lane 0 of waves ≥ 1 it is added after the barrier from the
// previous wave's last sample in LDS.  S: a scan slot of 3·LH_NW doubles (wave
// totals, first and last samples of each wave); consecutive calls alternate
// between the two slots, so a slot is rewritten only after a further barrier
// has passed all of its readers.  carry: running integral before this round;
// prev0: the integrand at the sample just before the round (thread 0 only).
// On return y[q] holds the running integral and carry the round's final value;
// returns the round's last integrand value.
template <int QR>
__device__ __forceinline__ double block_cumtrapz(double* y, double dx, int g0, double* S, double& carry,
                                                 double prev0) {
    const int tid = fresh_tid();
    const int lane = tid & 63, wid = tid >> 6;
    const double first = y[0], lastv = y[QR - 1];
    double prev = dpp_f64<DPP_WAVE_SHR1>(lastv);
    if (tid == 0) prev = prev0;
    const bool joined = (g0 != 0) && !(lane == 0 && wid > 0);
    double acc = 0.0;
    double last = prev;
#pragma unroll
    for (int q = 0; q < QR; q++) {
        const double cur = y[q];
        const double term = (q == 0) ? (joined ? (0.5 * (last + cur)) * dx : 0.0) : (0.5 * (last + cur)) * dx;
        last = cur;
        acc += term;
        y[q] = acc;
    }
    const double x = wave_incl_scan(acc);
    const double ex = dpp_f64<DPP_WAVE_SHR1>(x);  // exclusive (0 in lane 0)
    if (lane == 63) {
        S[wid] = x;
        S[2 * LH_NW + wid] = lastv;
    }
    if (lane == 0) S[LH_NW + wid] = first;
    __syncthreads();
    // lane w < LH_NW: wave w's joining trapezoid and total, scanned over those lanes
    double Ww = 0.0, c = 0.0;
    if (lane < LH_NW) {
        Ww = S[lane];
        c = (lane > 0) ? (0.5 * (S[2 * LH_NW + lane - 1] + S[LH_NW + lane])) * dx + Ww : Ww;
    }
    c = lanes_incl_scan(c);
    const double off = (carry + (lane_value(c, wid) - lane_value(Ww, wid))) + ex;
#pragma unroll
    for (int q = 0; q < QR; q++) y[q] = off + y[q];
    carry = carry + lane_value(c, LH_NW - 1);
    return S[3 * LH_NW - 1];
}

// Two chained cumtrapz over the workgroup with a single barrier: J = ∫a and
// P = ∫(J + l) for one round of QR samples per thread (global index g0+q).
// A run of samples acts on the integrals at the sample before it as
// J ← J + SJ, P ← P + n·dx·J + SP (n: its trapezoids; SJ, SP: its integrals
// from J = P = 0), and runs compose as
//   (n1, SJ1, SP1)·(n2, SJ2, SP2) = (n1 + n2, SJ1 + SJ2, SP1 + SP2 + n2·dx·SJ1),
// which the wave scan (DPP) and the cross-wave step apply in that order.  The
// trapezoid joining lane 0 of wave w ≥ 1 to wave w−1's last sample is a run
// of its own, formed after the barrier from the first and last samples in S
// (7·LH_NW doubles: wave totals n, SJ, SP; first a, l; last a, l).
// cJ, cP: J and P at the sample before the round; pa0, pl0: a and l there
// (thread 0).  On return a[q] = P at the sample, cJ, cP, pa0, pl0 those of the
// round's last sample.
struct Run2 {
    int n;
    double sj, sp;
};
__device__ __forceinline__ Run2 run2_cat(const Run2& x, const Run2& y, double dx) {
    return Run2{x.n + y.n, x.sj + y.sj, (x.sp + y.sp) + ((double)y.n * dx) * x.sj};
}

template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ Run2 dpp_run2(const Run2& x) {
    return Run2{dpp_i32<CTRL, ROW_MASK>(x.n, 0), dpp_f64<CTRL, ROW_MASK>(x.sj), dpp_f64<CTRL, ROW_MASK>(x.sp)};
}

template <int QR>
__device__ __forceinline__ void block_cumtrapz2(double* a, const double* l, double dx, int g0, double* S, double& cJ,
                                                double& cP, double& pa0, double& pl0) {
    const int tid = fresh_tid();
    const int lane = tid & 63, wid = tid >> 6;
    const double afirst = a[0], lfirst = l[0], alast = a[QR - 1], llast = l[QR - 1];
    double aprev = dpp_f64<DPP_WAVE_SHR1>(alast), pprev = dpp_f64<DPP_WAVE_SHR1>(llast);
    if (tid == 0) {
        aprev = pa0;
        pprev = pl0;
    }
    const bool joined = (g0 != 0) && !(lane == 0 && wid > 0);
    // this thread's run; a[q] := its SP up to sample q
    double sj = 0.0, sp = 0.0;
#pragma unroll
    for (int q = 0; q < QR; q++) {
        const double cur = a[q];
        if (q > 0 || joined) {
            sj += (0.5 * (aprev + cur)) * dx;
            const double pc = sj + l[q];
            sp += (0.5 * (pprev + pc)) * dx;
            pprev = pc;
        } else {
            pprev = l[q];
        }
        aprev = cur;
        a[q] = sp;
    }
    const int nt = QR - (joined ? 0 : 1);
    // inclusive scan of the runs over the wave (DPP), then exclusive by one lane
    Run2 x{nt, sj, sp};
    x = run2_cat(dpp_run2<DPP_ROW_SHR1>(x), x, dx);
    x = run2_cat(dpp_run2<DPP_ROW_SHR2>(x), x, dx);
    x = run2_cat(dpp_run2<DPP_ROW_SHR4>(x), x, dx);
    x = run2_cat(dpp_run2<DPP_ROW_SHR8>(x), x, dx);
    x = run2_cat(dpp_run2<DPP_ROW_BCAST15, 0xa>(x), x, dx);
    x = run2_cat(dpp_run2<DPP_ROW_BCAST31, 0xc>(x), x, dx);
    const Run2 ex = dpp_run2<DPP_WAVE_SHR1>(x);
    if (lane == 63) {
        S[wid] = (double)x.n;
        S[LH_NW + wid] = x.sj;
        S[2 * LH_NW + wid] = x.sp;
        S[5 * LH_NW + wid] = alast;
        S[6 * LH_NW + wid] = llast;
    }
    if (lane == 0) {
        S[3 * LH_NW + wid] = afirst;
        S[4 * LH_NW + wid] = lfirst;
    }
    __syncthreads();
    // lane w < LH_NW: the join into wave w (w ≥ 1), then wave w's total
    Run2 e{0, 0.0, 0.0}, jn{0, 0.0, 0.0};
    if (lane < LH_NW) {
        if (lane > 0) {
            const double ta = (0.5 * (S[5 * LH_NW + lane - 1] + S[3 * LH_NW + lane])) * dx;
            const double sp1 = (0.5 * (S[6 * LH_NW + lane - 1] + (ta + S[4 * LH_NW + lane]))) * dx;
            jn = Run2{1, ta, sp1};
        }
        e = run2_cat(jn, Run2{(int)S[lane], S[LH_NW + lane], S[2 * LH_NW + lane]}, dx);
    }
    Run2 c = e;  // inclusive over lanes 0..LH_NW-1
    c = run2_cat(dpp_run2<DPP_ROW_SHR1>(c), c, dx);
    c = run2_cat(dpp_run2<DPP_ROW_SHR2>(c), c, dx);
    c = run2_cat(dpp_run2<DPP_ROW_SHR4>(c), c, dx);
    if constexpr (LH_NW > 8) c = run2_cat(dpp_run2<DPP_ROW_SHR8>(c), c, dx);
    const Run2 win = run2_cat(dpp_run2<DPP_ROW_SHR1>(c), jn, dx);  // runs before wave w's first lane
    // runs before this thread: the wave's, then the lanes' before it in the wave
    const Run2 w_in{__builtin_amdgcn_readlane(win.n, __builtin_amdgcn_readfirstlane(wid)), lane_value(win.sj, wid),
                    lane_value(win.sp, wid)};
    const Run2 t_in = run2_cat(w_in, ex, dx);
    const double J = cJ + t_in.sj;
    const double P = (cP + ((double)t_in.n * dx) * cJ) + t_in.sp;
#pragma unroll
    for (int q = 0; q < QR; q++) {
        const int nq = q + (joined ? 1 : 0);
        a[q] = (P + ((double)nq * dx) * J) + a[q];
    }
    const Run2 all{__builtin_amdgcn_readlane(c.n, LH_NW - 1), lane_value(c.sj, LH_NW - 1),
                   lane_value(c.sp, LH_NW - 1)};
    cP = (cP + ((double)all.n * dx) * cJ) + all.sp;
    cJ = cJ + all.sj;
    pa0 = S[6 * LH_NW - 1];
    pl0 = S[7 * LH_NW - 1];
}

// Exclusive prefix sum of one value per thread with a single barrier (scan
// slot S as for block_cumtrapz); also returns the workgroup total.
__device__ __forceinline__ double block_exscan1(double v, double* S, double* total) {
    const int tid = fresh_tid();
    const int lane = tid & 63, wid = tid >> 6;
    const double x = wave_incl_scan(v);
    const double ex = dpp_f64<DPP_WAVE_SHR1>(x);
    if (lane == 63) S[wid] = x;
    __syncthreads();
    const double Ww = (lane < LH_NW) ? S[lane] : 0.0;
    const double c = lanes_incl_scan(Ww);
    *total = lane_value(c, LH_NW - 1);
    return (lane_value(c, wid) - lane_value(Ww, wid)) + ex;
}

// Workgroup min of lo and max of hi with a single barrier (scan slot S).
__device__ __forceinline__ void block_minmax(int& lo, int& hi, double* S) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    wave_minmax(lo, hi);
    if (lane == 0) {
        S[2 * wid] = (double)lo;
        S[2 * wid + 1] = (double)hi;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < LH_NW; w++) {
        lo = min(lo, (int)S[2 * w]);
        hi = max(hi, (int)S[2 * w + 1]);
    }
}

template <class Smem>
__device__ __forceinline__ double field_at(const Smem& sm, int g, double e_scale) {
    double2 v = sm.buf[pad(g >> 1)];
    return ((g & 1) ? v.y : v.x) * e_scale;
}

// Pointwise field responses on the packed real series in LDS (in place):
// E = c2r/Nto/field_div; P = ρε0γ3 E³ + ρ·Plasma(E); P *= towin.
// The series is processed in rounds of QR samples per thread (contiguous
// chunks), with the three cumtrapz integrals carried from round to round;
// each thread's samples are touched only by that thread.
// RAMAN: praman holds P(t) of the Raman response, packed pairs.
template <int MO, class Smem, bool RAMAN = false>
__device__ __forceinline__ void pointwise_field(const DInst& in, Smem& sm, double rho, double kfac,
                                                const double2* praman = nullptr) {
    constexpr int QT = 2 * MO / LH_T;          // samples per thread over all rounds
    constexpr int QR = (QT > 16) ? 16 : QT;    // samples per thread per round
    constexpr int NR = QT / QR;                // rounds
    const int tid = fresh_tid();
    const double es = in.e_scale;
    const bool kerr = (in.kerr == LH_KERR_FIELD), plasma = in.plasma;
    const double* tw = gl(in.to_win);
    const double dt = in.dt_o, pp1 = in.preion_p1, er = in.e_ratio, ip = in.ionpot;
    double cF = 0.0, cJ = 0.0, cP = 0.0;           // carried integrals
    double lastRate = 0.0, lastPhi = 0.0, lastLoss = 0.0;
    double Fprev = 0.0, fprev = pp1 - 1.0;         // exp(-0) = 1
    int sl = 0;                                    // scan slot of the next workgroup scan
#pragma unroll 1
    for (int r = 0; r < NR; r++) {
        const int g0 = r * (LH_T * QR) + QR * tid;
        double a[QR];
        if (plasma) {
            double jf[QR];
            int bad = 0;
            constexpr int QC = (QR < 4) ? QR : 4;
            constexpr int PCAP = PList<MO>::CAP;
#pragma unroll
            for (int q = 0; q < QR; q++) jf[q] = fabs(field_at(sm, g0 + q, es));
            if constexpr (MO <= 4096) {
                // samples inside the table's range get a rate; above it (or NaN) raise the flag
                unsigned mask = 0;
                int cnt = 0;
#pragma unroll
                for (int q = 0; q < QR; q++) {
                    const double x = jf[q];
                    const bool below = x < in.ppt_emin;
                    const bool out = !below && !(x <= in.ppt_emax);
                    if (out) bad = (x > in.ppt_emax) ? LH_E_PPT_RANGE : LH_E_NONFINITE;
                    if (!below && !out) {
                        mask |= 1u << q;
                        cnt++;
                    }
                }
                double ntot;
                const int off = (int)block_exscan1((double)cnt, sm.scan[sl], &ntot);
                sl ^= 1;
                const int total = (int)ntot;
                if (total <= PCAP) {  // compacted: one or two samples per thread
                    // sample q of this thread sits at off + (set bits of mask below q)
#pragma unroll
                    for (int q = 0; q < QR; q++)
                        if ((mask >> q) & 1u) sm.plist[off + __popc(mask & ((1u << q) - 1u))] = jf[q];
                    __syncthreads();
                    int unused = 0;
                    for (int i = tid; i < total; i += LH_T) {
                        double r;
                        ppt_rates<1>(in, &sm.plist[i], &r, unused);
                        sm.plist[i] = r;
                    }
                    __syncthreads();
#pragma unroll
                    for (int q = 0; q < QR; q++)
                        a[q] = ((mask >> q) & 1u) ? sm.plist[off + __popc(mask & ((1u << q) - 1u))] : 0.0;
                } else {
#pragma unroll
                    for (int c = 0; c < QR; c += QC) ppt_rates<QC>(in, jf + c, a + c, bad);
                }
            } else {
                // The samples that need a rate (the few hundred under the
                // pulse) lie in a window [lo, hi] of the round; when it fits the
                // LDS list, all threads take its samples in turn (one or two
                // each) instead of the ~16 threads that own them doing all of it.
                int lo = 0x7fffffff, hi = -1;
#pragma unroll
                for (int q = 0; q < QR; q++)
                    if (!(jf[q] < in.ppt_emin)) {
                        lo = min(lo, g0 + q);
                        hi = max(hi, g0 + q);
                    }
                block_minmax(lo, hi, sm.scan[sl]);
                sl ^= 1;
                if (hi < lo) {
#pragma unroll
                    for (int q = 0; q < QR; q++) a[q] = 0.0;
                } else if (hi - lo < PCAP) {
                    for (int g = lo + tid; g <= hi; g += LH_T) {
                        double ae = fabs(field_at(sm, g, es)), rr = 0.0;
                        if (!(ae < in.ppt_emin)) ppt_rates<1>(in, &ae, &rr, bad);
                        sm.plist[g - lo] = rr;
                    }
                    __syncthreads();
#pragma unroll
                    for (int q = 0; q < QR; q++) {
                        const int g = g0 + q;
                        a[q] = (g >= lo && g <= hi) ? sm.plist[g - lo] : 0.0;
                    }
                } else {
#pragma unroll
                    for (int c = 0; c < QR; c += QC) ppt_rates<QC>(in, jf + c, a + c, bad);
                }
            }
#pragma unroll
            for (int q = 0; q < QR; q++) jf[q] = a[q];  // rate, kept for the loss term
            if (bad) sm.flag = bad;
            lastRate = block_cumtrapz<QR>(a, dt, g0, sm.scan[sl], cF, lastRate);  // a = ∫rate
            sl ^= 1;
#pragma unroll
            for (int q = 0; q < QR; q++) {
                double E = field_at(sm, g0 + q, es);
                double F = a[q];
                double f = (F == Fprev) ? fprev : pp1 - exp(-F);  // F is flat outside the pulse
                Fprev = F;
                fprev = f;
                double rate = jf[q];
                a[q] = (f * er) * E;                                                     // phase
                jf[q] = (rate != 0.0 && E != 0.0) ? ((ip * rate) * (1 - f)) / E : 0.0;  // loss current
            }
            // a = P = ∫(J + loss), J = ∫(phase term)
            block_cumtrapz2<QR>(a, jf, dt, g0, sm.scan[sl], cJ, cP, lastPhi, lastLoss);
            sl ^= 1;
        }
#pragma unroll
        for (int s2 = 0; s2 < QR / 2; s2++) {
            const int g = g0 + 2 * s2;
            double2 v = sm.buf[pad(g >> 1)];
            double E0 = v.x * es, E1 = v.y * es;
            double p0 = kerr ? kfac * (E0 * E0 * E0) : 0.0;
            double p1 = kerr ? kfac * (E1 * E1 * E1) : 0.0;
            if (plasma) {
                p0 = p0 + rho * a[2 * s2];
                p1 = p1 + rho * a[2 * s2 + 1];
            }
            if constexpr (RAMAN) {  // RamanPolarField: Pout = ρ·E·P (src/Nonlinear.jl:323-325)
                const double2 pr = gl(praman)[g >> 1];
                p0 = p0 + (rho * E0) * pr.x;
                p1 = p1 + (rho * E1) * pr.y;
            }
            sm.buf[pad(g >> 1)] = make_double2(p0 * tw[g], p1 * tw[g + 1]);
        }
    }
}

// exp(−2πi k/L) for the zero-padded Raman transforms: L up to LH_TWN from
// the table; L = 2·LH_TWN gives even k from the table and odd k one more
// factor exp(−2πi/L).
template <int L>
__device__ __forceinline__ double2 tw_frac(const TwLds& tw, int k) {
    if constexpr (L <= LH_TWN) {
        return tw_get(tw, k * (LH_TWN / L));
    } else {
        static_assert(L == 2 * LH_TWN, "tw_frac: L up to 2·LH_TWN");
        double2 w = tw_get(tw, k >> 1);
        if (k & 1) {
            double sn, cs;
            sincos(-6.283185307179586476925286766559 / (double)L, &sn, &cs);
            w = cmul(w, make_double2(cs, sn));
        }
        return w;
    }
}

// Unnormalised complex FFT of NO = 2·M points held in HBM (natural order, in
// place in g); tmp: M points of HBM.  X[k] = E[k] + w^k O[k], X[k+M] =
// E[k] − w^k O[k], with E, O the transforms of the even and odd samples and
// w = exp(∓2πi/NO).  Starts and ends with a workgroup barrier.
template <int M, bool INV, class Smem>
__device__ __forceinline__ void fft_big(double2* g, double2* tmp, Smem& sm) {
    const int tid = fresh_tid();
    __syncthreads();
    for (int j = tid; j < M; j += LH_T) sm.buf[pad(j)] = g[2 * j];
    __syncthreads();
    fft_lds<M, INV>(sm.buf, sm.tw);
    for (int j = tid; j < M; j += LH_T) tmp[j] = sm.buf[pad(j)];
    __syncthreads();
    for (int j = tid; j < M; j += LH_T) sm.buf[pad(j)] = g[2 * j + 1];
    __syncthreads();
    fft_lds<M, INV>(sm.buf, sm.tw);
    constexpr int TS = LH_TWN / (2 * M);
    for (int k = tid; k < M; k += LH_T) {
        double2 w = tw_get(sm.tw, k * TS);
        if (INV) w.y = -w.y;
        const double2 o = cmul(w, sm.buf[pad(k)]), e = tmp[k];
        g[k] = cadd(e, o);
        g[k + M] = csub(e, o);
    }
    __syncthreads();
}

// r2c post-step of a 2·NO-point real transform whose packed NO-point
// transform Z is in HBM: X[k] = E + w^k O (as r2c_bin).
template <int NO, class Smem>
__device__ __forceinline__ double2 r2c_bin_big(const double2* Z, const Smem& sm, int k) {
    double2 zk = Z[k == NO ? 0 : k];
    double2 zc = cconj(Z[k == 0 ? 0 : NO - k]);
    double2 E = cscal(0.5, cadd(zk, zc));
    double2 d = csub(zk, zc);
    double2 O = make_double2(0.5 * d.y, -(0.5 * d.x));
    double2 w = (k == NO) ? make_double2(-1.0, 0.0) : tw_frac<2 * NO>(sm.tw, k);
    return cadd(E, cmul(w, O));
}

// The seven stage vectors k1..k7, addressed arithmetically: a loop over j
// computes the address of k_j in registers (the index is uniform over the
// workgroup) instead of reading a pointer array from private memory before
// every vector's loads.
struct KSet {
    double2* base;     // the vectors lie in one block, `stride` elements apart; slot 7:
                       // the envelope stage's exp(L·(t − t2))
    long long stride;
    int s0, s6;        // slots of k1 and k7 (swapped by FSAL); k2..k6 keep slots 1..5
    __device__ __forceinline__ gptr<double2> operator[](int j) const {
        const int s = (j == 0) ? s0 : (j == 6) ? s6 : j;
        return gl(base + (long long)s * stride);
    }
    __device__ __forceinline__ void swap06() {  // FSAL: ks[1] .= ks[7] as a pointer swap
        const int t = s0;
        s0 = s6;
        s6 = t;
    }
};

// Stage prologue: buf[k] = sc_t · (y + Σ_j Δz B_ij k_j)·exp(L hf); k1 first
// propagated by h0 (evaluate!, src/RK45.jl:209-223).  Loops run over the
// k-vectors outside and this thread's bins inside, so each vector's loads
// for all bins are in flight together; with nine bins per thread and FOLD,
// chunks of three bins instead load every vector a chunk needs in one round
// (three rounds per stage instead of three to five: 125.3 → 122.2 ms for the
// Nto = 16384 class of the sweep, bit-identical results).
// FOLD (field grid): also stores the stage epilogue's factor
// outfac·exp(L·(t − t2)) = outfac·exp(−L·hf) into slot 7 of K, from the same
// exp and sincos as exp(L·hf) (the epilogue then needs neither a
// transcendental pass nor the output factor held across the forward FFT).
template <int MO, class Smem, class KS, bool PACK, bool FOLD = false>
__device__ __forceinline__ void stage_prologue_cols(const double2* __restrict__ linop, double sc_t, Smem& sm,
                                                    const double2* Y, const KS& K, int stage, double dt,
                                                    double h0, double hf, const double2* outfac = nullptr);

// Same on explicit per-column pointers (one column of a radial state).
template <int MO, class Smem, class KS, bool PACK, bool FOLD>
__device__ __forceinline__ void stage_prologue_cols(const double2* __restrict__ linop, double sc_t, Smem& sm,
                                                    const double2* Y, const KS& K, int stage, double dt,
                                                    double h0, double hf, const double2* outfac) {
    constexpr int N = Bins<MO>::N, NPT = Bins<MO>::NPT;
    const int tid = fresh_tid();
    if constexpr (FOLD && NPT == 9) {
        // chunks of three bins per thread, each with every vector it needs
        // (y, L, the output factor and k1..k_{stage+1}) loaded in one round
        constexpr int CB = 3;
        double2* F = K[7];
#pragma unroll 1
        for (int c = 0; c < NPT; c += CB) {
            double2 yb[CB], L[CB], of[CB], kk[6][CB];
#pragma unroll
            for (int i = 0; i < CB; i++) {
                const int k = tid + (c + i) * LH_T;
                const bool v = k < N;
                yb[i] = v ? Y[k] : make_double2(0.0, 0.0);
                L[i] = v ? linop[k] : make_double2(0.0, 0.0);
                of[i] = v ? outfac[k] : make_double2(0.0, 0.0);
            }
#pragma unroll
            for (int j = 0; j < 6; j++) {
                const double2* Kj = K[j];
                const bool use = j <= stage && c_B[stage][j] != 0.0;
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    const int k = tid + (c + i) * LH_T;
                    kk[j][i] = (use && k < N) ? Kj[k] : make_double2(0.0, 0.0);
                }
            }
            if (stage == 0 && h0 != 0.0) {
                double2* K0 = K[0];
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    const int k = tid + (c + i) * LH_T;
                    kk[0][i] = cmul(kk[0][i], cexp_lh(L[i], h0));
                    if (k < N) K0[k] = kk[0][i];
                }
            }
#pragma unroll
            for (int j = 0; j < 6; j++) {
                const double cj = dt * c_B[stage][j];
                if (j <= stage && cj != 0.0) {
#pragma unroll
                    for (int i = 0; i < CB; i++) yb[i] = cadd(yb[i], cscal(cj, kk[j][i]));
                }
            }
#pragma unroll
            for (int i = 0; i < CB; i++) {
                const int k = tid + (c + i) * LH_T;
                if (k < N) {
                    double2 yp = yb[i], inv = make_double2(1.0, 0.0);
                    if (hf != 0.0) yp = cmul(yb[i], cexp_lh_inv(L[i], hf, inv));
                    c2r_pack_bin<MO>(sm.buf, sm.tw, k, cscal(sc_t, yp));
                    F[k] = cmul(of[i], inv);
                }
            }
        }
        return;
    }
    double2 yb[NPT], L[NPT];
#pragma unroll
    for (int i = 0; i < NPT; i++) {
        int k = tid + i * LH_T;
        bool v = k < N;
        yb[i] = v ? Y[k] : make_double2(0.0, 0.0);
        L[i] = v ? linop[k] : make_double2(0.0, 0.0);
    }
    if (stage == 0 && h0 != 0.0) {
        double2* K0 = K[0];
        constexpr int CH = (NPT > 9) ? 8 : NPT;  // a chunk's loads before its first store
        static_assert(NPT % CH == 0, "prologue chunks");
#pragma unroll
        for (int c = 0; c < NPT; c += CH) {
            double2 kv[CH];
#pragma unroll
            for (int i = 0; i < CH; i++) {
                int k = tid + (c + i) * LH_T;
                kv[i] = (k < N) ? K0[k] : make_double2(0.0, 0.0);
            }
#pragma unroll
            for (int i = 0; i < CH; i++) {
                int k = tid + (c + i) * LH_T;
                if (k < N) K0[k] = cmul(kv[i], cexp_lh(L[c + i], h0));
            }
        }
    }
    // two k-vectors per iteration: both vectors' loads are in flight together
    // (the sum still runs over j in order)
#pragma unroll 1
    for (int j = 0; j <= stage; j += 2) {
        const double c0 = dt * c_B[stage][j];
        const double c1 = (j + 1 <= stage) ? dt * c_B[stage][j + 1] : 0.0;
        const double2* K0j = K[j];
        const double2* K1j = K[j + 1];
        double2 a[NPT], b[NPT];
#pragma unroll
        for (int i = 0; i < NPT; i++) {
            int k = tid + i * LH_T;
            a[i] = (k < N && c0 != 0.0) ? K0j[k] : make_double2(0.0, 0.0);
            b[i] = (k < N && c1 != 0.0) ? K1j[k] : make_double2(0.0, 0.0);
        }
#pragma unroll
        for (int i = 0; i < NPT; i++) {
            if (c0 != 0.0) yb[i] = cadd(yb[i], cscal(c0, a[i]));
            if (c1 != 0.0) yb[i] = cadd(yb[i], cscal(c1, b[i]));
        }
    }
    if constexpr (FOLD) {
        double2* F = K[7];
#pragma unroll
        for (int i = 0; i < NPT; i++) {
            int k = tid + i * LH_T;
            if (k < N) {
                const double2 of = outfac[k];
                double2 yp = yb[i], inv = make_double2(1.0, 0.0);
                if (hf != 0.0) yp = cmul(yb[i], cexp_lh_inv(L[i], hf, inv));
                c2r_pack_bin<MO>(sm.buf, sm.tw, k, cscal(sc_t, yp));
                F[k] = cmul(of, inv);
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < NPT; i++) {
            int k = tid + i * LH_T;
            if (k < N) {
                double2 yp = (hf != 0.0) ? cmul(yb[i], cexp_lh(L[i], hf)) : yb[i];
                if constexpr (PACK)  // the c2r pre-pack of the RHS, bin by bin (N − 1 = MO/2)
                    c2r_pack_bin<MO>(sm.buf, sm.tw, k, cscal(sc_t, yp));
                else
                    sm.buf[pad(k)] = cscal(sc_t, yp);
            }
        }
    }
    if constexpr (!PACK)
        for (int k = N + tid; k <= MO; k += LH_T) sm.buf[pad(k)] = make_double2(0.0, 0.0);
}

// Statistics of the spectrum held in LDS (defined with the statistics below).
// Partial energies Σ_k window_w[w][k]·|Eω_k|² of a thread's bins for the
// energy windows (energy_window: energyfun_ω(Eω .* window), src/Stats.jl:69-79).
struct WinSums {
    double s[LH_STAT_MAX_WINDOWS];
};
__device__ __forceinline__ void win_add(const DInst& in, WinSums& w, int k, double a) {
#pragma unroll
    for (int q = 0; q < LH_STAT_MAX_WINDOWS; q++)
        if (q < in.st_nwin) w.s[q] += gl(in.st_win)[(size_t)q * in.n_omega + k] * a;
}

template <int KIND, int NT, class Smem>
__device__ __forceinline__ void stats_time(const DInst& in, Smem& sm, double s0, double s1, double se,
                                           const WinSums& ws, double z, double dz, double rho, double* rec);

// Accepted-step window filter (stepfun, src/Luna.jl:366-370) on the coarse
// grid: YN ← rfft(twin · irfft(ωwin · YN·exp(L h))).  With STATS and a
// record pointer, the statistics of the filtered YN follow from the values
// still in registers (no read-back of YN).
template <int MC, class Smem, bool STATS = false>
__device__ __forceinline__ void stepfun_filter_cols(const DInst& in, const double2* __restrict__ linop, Smem& sm,
                                                    double2* YN, double h, double* rec = nullptr, double z = 0.0,
                                                    double dz = 0.0, double rho = 0.0);

template <int MC, class Smem>
__device__ __forceinline__ void stepfun_filter(const DInst& in, Smem& sm, double2* YN, double h, double* rec,
                                               double z, double dz, double rho) {
    stepfun_filter_cols<MC, Smem, true>(in, gl(in.linop), sm, YN, h, rec, z, dz, rho);
}

template <int MC, class Smem, bool STATS>
__device__ __forceinline__ void stepfun_filter_cols(const DInst& in, const double2* __restrict__ linop, Smem& sm,
                                                    double2* YN, double h, double* rec, double z, double dz,
                                                    double rho) {
    constexpr int N = MC + 1;
    constexpr int NPT = (N + LH_T - 1) / LH_T;
#pragma unroll
    for (int i = 0; i < NPT; i++) {
        int k = fresh_tid() + i * LH_T;
        if (k < N) {
            double2 v = YN[k];
            if (h != 0.0) v = cmul(v, cexp_lh(linop[k], h));
            sm.buf[pad(k)] = cscal(gl(in.omega_win)[k], v);
        }
    }
    __syncthreads();
    c2r_prepack<MC>(sm.buf, sm.tw);
    __syncthreads();
    fft_lds<MC, true>(sm.buf, sm.tw);
    const double inv_nt = in.inv_nt;
    for (int j = fresh_tid(); j < MC; j += LH_T) {
        double2 z = sm.buf[pad(j)];
        double x0 = (inv_nt * z.x) * gl(in.t_win)[2 * j];
        double x1 = (inv_nt * z.y) * gl(in.t_win)[2 * j + 1];
        sm.buf[pad(j)] = make_double2(x0, x1);
    }
    __syncthreads();
    fft_lds<MC, false>(sm.buf, sm.tw);
    if constexpr (STATS) {
        if (rec) {
            // analytic spectrum (copyto_fft!, src/Stats.jl:441-448): bins
            // 0..Nω-2 doubled, the +fs/2 bin dropped, zero up to Nt = 2·MC
            double2 yv[NPT];
            double wv[NPT], ev[NPT];
#pragma unroll
            for (int i = 0; i < NPT; i++) {
                int k = fresh_tid() + i * LH_T;
                wv[i] = (k < N) ? gl(in.st_omega)[k] : 0.0;
                ev[i] = (k < N) ? gl(in.st_ew)[k] : 0.0;
                yv[i] = make_double2(0.0, 0.0);
                if (k < N) {
                    yv[i] = r2c_bin<MC>(sm.buf, sm.tw, k);
                    YN[k] = yv[i];
                }
            }
            __syncthreads();  // every bin read before the buffer is reused
            double s0 = 0.0, s1 = 0.0, se = 0.0;
            WinSums ws = {{0.0, 0.0, 0.0, 0.0}};
#pragma unroll
            for (int i = 0; i < NPT; i++) {
                int k = fresh_tid() + i * LH_T;
                double a = yv[i].x * yv[i].x + yv[i].y * yv[i].y;
                s0 += a;
                s1 += wv[i] * a;
                se += ev[i] * a;
                if (k < N) win_add(in, ws, k, a);
                if (k < N - 1) sm.buf[pad(k)] = make_double2(2.0 * yv[i].x, 2.0 * yv[i].y);
            }
            for (int k = N - 1 + fresh_tid(); k < 2 * MC; k += LH_T) sm.buf[pad(k)] = make_double2(0.0, 0.0);
            stats_time<0, 2 * MC, Smem>(in, sm, s0, s1, se, ws, z, dz, rho, rec);
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < NPT; i++) {
        int k = fresh_tid() + i * LH_T;
        if (k < N) YN[k] = r2c_bin<MC>(sm.buf, sm.tw, k);
    }
    __syncthreads();
}

// ==========================================================================
// z-dependent gas fill (Capillary.gradient + LinearOps.make_linop)
// ==========================================================================
#define LH_EPS0 8.854187817620389e-12  // CODATA 2014 ε0
#define LH_CLIGHT 299792458.0

// 8th-order central first-derivative weights at offsets -4..4 (times 1/h)
static __constant__ double c_fd8[9] = {1.0 / 280, -4.0 / 105, 1.0 / 5, -4.0 / 5, 0.0, 4.0 / 5, -1.0 / 5, 4.0 / 105, -1.0 / 280};

// Pressure profile p(z) of Capillary.gradient, src/Capillary.jl:306-340.
__device__ __forceinline__ double zg_pressure(const DInst& in, double z) {
    const double* Z = gl(in.zg_Z);
    const double* P = gl(in.zg_P);
    const int n = in.zg_np;
    if (in.zg_two) {
        const double L = Z[1], p0 = P[0], p1 = P[1];
        if (z > L) return p1;
        if (z <= 0) return p0;
        return sqrt(p0 * p0 + z / L * (p1 * p1 - p0 * p0));
    }
    if (z <= Z[0]) return P[0];
    if (z >= Z[n - 1]) return P[n - 1];
    int i = 0;
    for (int j = 0; j < n; j++)
        if (Z[j] < z) i = j;  // findlast(x -> x < z, Z)
    return sqrt(P[i] * P[i] + (z - Z[i]) / (Z[i + 1] - Z[i]) * (P[i + 1] * P[i + 1] - P[i] * P[i]));
}

// Principal square root of x + iy.
__device__ __forceinline__ double2 csqrt_lh(double x, double y) {
    if (x == 0.0 && y == 0.0) return make_double2(0.0, y);
    const double t = sqrt((fabs(x) + hypot(x, y)) * 0.5);
    if (x >= 0.0) return make_double2(t, y / (2.0 * t));
    return make_double2(fabs(y) / (2.0 * t), copysign(t, y));
}

// neff(mode, εco, nwg) of a Marcatili mode, src/Capillary.jl:216-234.
__device__ __forceinline__ double2 zg_neff(const DInst& in, double eco, double2 nwg) {
    double2 n;
    if (in.zg_model == 0)
        n = csqrt_lh(eco - nwg.x, -nwg.y);
    else
        n = make_double2(1 + (eco - 1) / 2 - nwg.x, -nwg.y);
    if (!in.zg_loss) n.y = 0.0;
    return n;
}

// Radius of the taper at z: linear a0 + (a1 - a0)·clamp(z/L, 0, 1), or the
// piecewise-linear profile through (zt_Z, zt_A), constant outside.
__device__ __forceinline__ double zg_radius(const DInst& in, double z) {
    if (in.ztaper == 2) {
        const double *Z = gl(in.zt_Z), *A = gl(in.zt_A);
        const int n = in.zt_n;
        if (z <= Z[0]) return A[0];
        if (z >= Z[n - 1]) return A[n - 1];
        // the segment [Z[i], Z[i+1]] with Z[i] < z <= Z[i+1] (nodes strictly
        // increasing), by bisection: Z[lo] < z <= Z[hi] throughout
        int lo = 0, hi = n - 1;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (Z[mid] < z)
                lo = mid;
            else
                hi = mid;
        }
        const int i = lo;
        return A[i] + (A[i + 1] - A[i]) * ((z - Z[i]) / (Z[i + 1] - Z[i]));
    }
    double f = z / in.zaL;
    f = f < 0.0 ? 0.0 : (f > 1.0 ? 1.0 : f);
    return in.za0 + (in.za1 - in.za0) * f;
}

// neff_wg(mode, ω; z) at radius a from U = u_nm/k and V = v_n/k
// (src/Capillary.jl:188-214): (U/a)²(1 - iV/a)² (:full); (U/a)²/2, plus
// i(U/a)²V/a with loss (:reduced).
__device__ __forceinline__ double2 zg_nwg_taper(const DInst& in, double U, double2 V, double a) {
    const double q = U / a, q2 = q * q;
    if (in.zg_model == 0) {
        const double tr = 1.0 + V.y / a, ti = -(V.x / a);  // 1 - iV/a
        return make_double2(q2 * (tr * tr - ti * ti), q2 * (2.0 * tr * ti));
    }
    double2 r = make_double2(q2 / 2, 0.0);
    if (in.zg_loss) {
        r.x += -(q2 * (V.y / a));
        r.y += q2 * (V.x / a);
    }
    return r;
}

// ρ(z), β1(z) and the taper's radius at z into zs[0..2], by one wavefront: a
// stencil point per lane, the sum in the points' order.  β1 =
// Modes.dispersion(mode, 1, ω0, z): β(ω) = ω/c·Re neff(mode, ω; z) with neff's
// own clamp (src/Capillary.jl:162-186).
__device__ __forceinline__ void zg_constants(const DInst& in, double* zs, double z) {
    const double p = zg_pressure(in, z);
    const double r = cspline_uniform(gl(in.zd), in.zd_n, gl(in.zd)[0].x, gl(in.zd)[in.zd_n - 1].x, p);
    const double a = in.ztaper ? zg_radius(in, z) : 0.0;
    const int lane = threadIdx.x & 63, j = min(lane, 8);
    const double* f = gl(in.zfd) + 4 * j;
    const double sc = sqrt(1 + f[1] * r);
    double2 nwj = make_double2(f[2], f[3]);
    if (in.ztaper) {
        const double* t = gl(in.zfdt) + 3 * j;
        nwj = zg_nwg_taper(in, t[0], make_double2(t[1], t[2]), a);
    }
    double nr = zg_neff(in, sc * sc, nwj).x;
    if (in.zg_model == 0 && nr < 1e-3) nr = 1e-3;
    const double beta = f[0] / LH_CLIGHT * nr;
    double acc = 0.0;
#pragma unroll
    for (int i = 0; i < 9; i++) acc = fma(c_fd8[i], lane_value(beta, i), acc);
    if (lane == 0) {
        zs[0] = r;
        zs[1] = acc / in.zfd_h;
        zs[2] = a;
    }
}

// ==========================================================================
// Per-step statistics (Stats.default + collect_stats, src/Stats.jl:454-532)
// ==========================================================================
// Maths.linterpx, src/Maths.jl:248-252.
__device__ __forceinline__ double linterpx(double x1, double x2, double y1, double y2, double val) {
    double slope = (y2 - y1) / (x2 - x1);
    double icpt = y1 - slope * x1;
    return (val - icpt) / slope;
}

// Size classes with a compiled kernel.
enum {
    LH_CLASS_16384 = 0,    // field grid, Nto = 16384, Nt = 8192
    LH_CLASS_8192 = 1,     // field grid, Nto = 8192, Nt = 4096
    LH_CLASS_4096 = 2,     // field grid, Nto = 4096, Nt = 2048
    LH_CLASS_ENV8192 = 3,  // envelope grid, Nto = Nt = 8192
    LH_CLASS_ENV4096 = 4,  // envelope grid, Nto = Nt = 4096
    LH_CLASS_RADIAL = 5,   // radial transform (solved context by context)
    LH_CLASS_ENV16384 = 6, // envelope grid, Nto = Nt = 16384
    LH_CLASS_32768 = 7,    // field grid, Nto = 32768, Nt = 16384
    LH_NCLASS = 8
};
