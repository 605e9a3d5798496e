// lh_solo_kernel.h -- propagation with one workgroup per instance (gfx950),
// compiled by lh_solo.hip and lh_solo_8192.hip.
//
// Two kinds of instances run here instead of on gangs of workgroups (lh_gang.h).
//
// z-dependent fills (pressure gradient, taper) stay on this order of operations,
// because their operator amplifies rounding: β1(z) is a 9-point difference of
// β ≈ 8e6 rad/m over a step h, so one unit in the last place of a single β moves
// the phase of the field by 1e-9 to 1e-8 over a propagation.  Any other order of
// operations in the right-hand side shifts the step positions z by a relative
// 1e-13 through the error estimate, which is enough to flip such a unit at some
// z: the same solver on gangs took 19.4 ms instead of 42.6 for a 0.5 m
// propagation at Nto = 16384, but landed 5e-8 away.  Field grids only.
//
// Large even batches: a gang exchanges its series through the L2 and waits at
// barriers, a workgroup alone does neither, so with an instance for every CU and
// about equal lengths one workgroup each does 1.5 to 2.6 times as much per
// second (solo_pays in lh_kernels.hip has the rule).
#pragma once
#include "lh_core.h"
#include "lh_solo.h"

// Epilogues of a transform: called with v[i] = the RHS of bin
// k = (the thread's index) + i·LH_T.
struct EpiStore {  // out[k] = v
    static constexpr bool FOLDS_OUTFAC = false;
    double2* out;
    template <int NP>
    __device__ __forceinline__ void operator()(const double2 (&v)[NP], int n) const {
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int k = fresh_tid() + i * LH_T;
            if (k < n) gl(out)[k] = v[i];
        }
    }
};
// out[k] = v·F[k], F = outfac·exp(L·(t − t2)) stored by the stage prologue.
struct EpiStageFO {
    static constexpr bool FOLDS_OUTFAC = true;
    double2* out;
    const double2* F;
    template <int NP>
    __device__ __forceinline__ void operator()(const double2 (&v)[NP], int n) const {
        static_assert(NP <= 9, "epilogue chunk");
        double2 f[NP];  // the chunk's loads before its first store (out may alias F as far as the compiler knows)
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int k = fresh_tid() + i * LH_T;
            f[i] = (k < n) ? static_cast<const double2*>(gl(F))[k] : make_double2(0.0, 0.0);
        }
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int k = fresh_tid() + i * LH_T;
            if (k < n) gl(out)[k] = cmul(v[i], f[i]);
        }
    }
};

// The convolution step of the zero-padded Raman transform (2·NO reals packed
// into the NO-point transform Z in HBM): r2c post-step, ×hω·δt, and the c2r
// pre-pack of the product, pairwise (k, NO − k) in place.
template <int NO, class Smem>
__device__ __forceinline__ void raman_spectrum_big(const DInst& in, const Smem& sm, double2* W) {
    const int tid = fresh_tid();
    for (int k = tid; k <= NO / 2; k += LH_T) {
        const int m = NO - k;
        if (k == 0) {
            double2 Y0 = cmul(gl(in.hwdt)[0], r2c_bin_big<NO>(W, sm, 0));
            double2 YM = cmul(gl(in.hwdt)[NO], r2c_bin_big<NO>(W, sm, NO));
            Y0.y = 0.0;
            YM.y = 0.0;
            const double2 A = cadd(Y0, cconj(YM)), B = csub(Y0, cconj(YM));
            W[0] = cadd(A, cmul_pi(B));
        } else if (k == NO / 2) {
            const double2 Yk = cmul(gl(in.hwdt)[k], r2c_bin_big<NO>(W, sm, k));
            const double2 A = cadd(Yk, cconj(Yk));
            const double2 B = cmul(csub(Yk, cconj(Yk)), cconj(tw_frac<2 * NO>(sm.tw, k)));
            W[k] = cadd(A, cmul_pi(B));
        } else {
            const double2 Yk = cmul(gl(in.hwdt)[k], r2c_bin_big<NO>(W, sm, k));
            const double2 Ym = cmul(gl(in.hwdt)[m], r2c_bin_big<NO>(W, sm, m));
            const double2 wk = cconj(tw_frac<2 * NO>(sm.tw, k)), wm = cconj(tw_frac<2 * NO>(sm.tw, m));
            const double2 Ak = cadd(Yk, cconj(Ym)), Bk = cmul(csub(Yk, cconj(Ym)), wk);
            const double2 Am = cadd(Ym, cconj(Yk)), Bm = cmul(csub(Ym, cconj(Yk)), wm);
            W[k] = cadd(Ak, cmul_pi(Bk));
            W[m] = cadd(Am, cmul_pi(Bm));
        }
    }
}

// RamanPolarField with third-harmonic terms (src/Nonlinear.jl:183-247,
// 284-333, thg = true) for a series of Nto = 2·MO reals held packed in LDS
// (before the e_scale factor).  E² over the zero-padded 2·Nto reals is one
// 2·MO-point complex transform, run through HBM as two MO-point LDS transforms
// (fft_big); ×hω·δt; back; P(t) lands in the last MO points of the exchange area
// (4·MO) as packed pairs.  The LDS series is restored from its copy in the first.
template <int MO, class Smem>
__device__ __forceinline__ void raman_field(const DInst& in, Smem& sm) {
    constexpr int NR = 2 * MO;
    double2* S = gl(in.gx);
    double2* W = gl(in.gx) + MO;
    double2* T = gl(in.gx) + 3 * MO;
    const int tid = fresh_tid();
    const double es = in.e_scale;
    for (int j = tid; j < MO; j += LH_T) {
        const double2 z = sm.buf[pad(j)];
        const double e0 = z.x * es, e1 = z.y * es;
        S[j] = z;
        W[j] = make_double2(e0 * e0, e1 * e1);  // E² (thg: E.^2), reals packed in pairs
        W[j + MO] = make_double2(0.0, 0.0);     // zero padding to 2·Nto reals
    }
    fft_big<MO, false>(W, T, sm);
    raman_spectrum_big<NR>(in, sm, W);
    fft_big<MO, true>(W, T, sm);
    const double inv2n = in.inv_2n;
    for (int j = tid; j < MO; j += LH_T) {
        const double2 p = W[j];
        T[j] = make_double2(p.x * inv2n, p.y * inv2n);
        sm.buf[pad(j)] = S[j];
    }
    __syncthreads();
}

// Field-grid mode-averaged transform on LDS data.  On entry buf holds the c2r
// pre-pack of sc_t·Eω.  Hands the output bins k < N to epi.
template <int MO, bool RAMAN, class Smem, class Epi>
__device__ __forceinline__ void rhs_field(const DInst& in, Smem& sm, Epi epi, double rho, double kfac) {
    __syncthreads();
    fft_lds<MO, true>(sm.buf, sm.tw);
    if constexpr (RAMAN) raman_field<MO, Smem>(in, sm);
    pointwise_field<MO, Smem, RAMAN>(in, sm, rho, kfac, RAMAN ? in.gx + 3 * MO : nullptr);
    constexpr int N = Bins<MO>::N, NPT = Bins<MO>::NPT;
    static_assert(NPT <= 9, "one epilogue chunk");
    double2 res[NPT];
    if constexpr (Epi::FOLDS_OUTFAC) {
        __syncthreads();
        fft_lds<MO, false>(sm.buf, sm.tw);
#pragma unroll
        for (int i = 0; i < NPT; i++) {
            int k = fresh_tid() + i * LH_T;
            res[i] = (k < N) ? r2c_bin<MO>(sm.buf, sm.tw, k) : make_double2(0.0, 0.0);
        }
    } else {
        double2 of[NPT];  // loads in flight during the forward FFT
#pragma unroll
        for (int i = 0; i < NPT; i++) {
            int k = fresh_tid() + i * LH_T;
            of[i] = (k < N) ? static_cast<const double2*>(gl(in.outfac))[k] : make_double2(0.0, 0.0);
        }
        __syncthreads();
        fft_lds<MO, false>(sm.buf, sm.tw);
#pragma unroll
        for (int i = 0; i < NPT; i++) {
            int k = fresh_tid() + i * LH_T;
            res[i] = (k < N) ? cmul(r2c_bin<MO>(sm.buf, sm.tw, k), of[i]) : make_double2(0.0, 0.0);
        }
    }
    epi(res, N);
}

template <int MO, class Smem>
__device__ __forceinline__ void stage_prologue(const DInst& in, Smem& sm, const double2* Y, const KSet& K,
                                               int stage, double dt, double h0, double hf) {
    stage_prologue_cols<MO, Smem, KSet, true, true>(gl(in.linop), in.sc_t, sm, Y, K, stage, dt, h0, hf, gl(in.outfac));
}

// Re-evaluate the z-dependent constants at z (make_prop!(linop!) evaluates
// linop!(out, t2) whenever t2 changes): ρ(z) and β1(z) on the first wavefront,
// one stencil point per lane and the sum in the points' order, then per
// bin the operator -i(ω/c·conj_clamp(neff) - ω β1) (src/LinearOps.jl:337-358,
// 254) and the output factor sc_f·pre/β·√Aeff·ωwin (β = ω/c·Re neff),
// written to gl(in.zL) / gl(in.zOF).  Returns ρ(z) and the Kerr factor ρ ε0 γ3.
template <class Smem>
__device__ __forceinline__ void zg_refresh(const DInst& in, Smem& sm, double z, double& rho, double& kfac) {
    const int tid = fresh_tid();
    if (tid < 64) zg_constants(in, sm.zs, z);
    __syncthreads();
    rho = sm.zs[0];
    const double b1 = sm.zs[1];
    const double a = sm.zs[2];
    const double sqrt_aeff = in.ztaper ? a * in.zsqrt_intg : in.zsqrt_aeff;  // Aeff(z) = a(z)²·aeff_intg
    kfac = rho * LH_EPS0 * in.kerr_gamma3;
    // three bins per round: their loads are in flight together (a bin at a time
    // waited for zsidx, then for the rest, nine times per refresh at Nto = 16384:
    // 40.9 → 38.2 ms for a 0.5 m propagation; one stencil point per lane above
    // instead of nine in a row: 42.9 → 40.9 ms; the same bits)
    constexpr int CB = 3;
    const int N = in.n_omega;
#pragma unroll 1
    for (int k0 = tid; k0 < N; k0 += CB * LH_T) {
        double w[CB], gam[CB], win[CB], U[CB];
        double2 nw[CB], pre[CB];
        bool live[CB];
#pragma unroll
        for (int i = 0; i < CB; i++) {
            const int k = min(k0 + i * LH_T, N - 1);
            live[i] = gl(in.zsidx)[k];
            w[i] = gl(in.st_omega)[k];
            gam[i] = gl(in.zgam)[k];
            win[i] = gl(in.omega_win)[k];
            pre[i] = static_cast<const double2*>(gl(in.zpre))[k];
            U[i] = in.ztaper ? gl(in.zU)[k] : 0.0;
            nw[i] = in.ztaper ? static_cast<const double2*>(gl(in.zV))[k] : static_cast<const double2*>(gl(in.znwg))[k];
        }
#pragma unroll
        for (int i = 0; i < CB; i++) {
            const int k = k0 + i * LH_T;
            if (k >= N) break;
            double2 L = make_double2(0.0, 0.0), of = make_double2(in.sc_f, 0.0);
            if (live[i]) {
                const double sc = sqrt(1 + gam[i] * rho);  // coren(ω; z)^2
                const double2 nwk = in.ztaper ? zg_nwg_taper(in, U[i], nw[i], a) : nw[i];
                const double2 n = zg_neff(in, sc * sc, nwk);
                const double ncr = (n.x < 1e-3) ? 1e-3 : n.x;  // conj_clamp
                const double lim = 3000 * LH_CLIGHT / w[i];
                const double nci = -((n.y < 0.0) ? 0.0 : (n.y > lim ? lim : n.y));
                const double wc = w[i] / LH_CLIGHT;
                const double zr = wc * ncr - w[i] * b1, zi = wc * nci;
                L = make_double2(zi, -zr);
                const double beta = wc * n.x;
                const double nfx = pre[i].x / beta * sqrt_aeff, nfy = pre[i].y / beta * sqrt_aeff;
                of = make_double2((in.sc_f * nfx) * win[i], (in.sc_f * nfy) * win[i]);
            }
            gl(in.zL)[k] = L;
            gl(in.zOF)[k] = of;
        }
    }
    __syncthreads();
}

// The analytic spectrum is in LDS (not yet synchronised) and each thread holds
// its partial sums Σ|E|², Σω|E|², Σw|E|²: the record of the state.
template <int KIND, int NT, class Smem>
__device__ __forceinline__ void stats_time(const DInst& in, Smem& sm, double s0, double s1, double se,
                                           const WinSums& ws, double z, double dz, double rho, double* rec) {
    const int tid = fresh_tid();
    const int lane = tid & 63, wid = tid >> 6;
    block_sum3(s0, s1, se, sm.wsum);  // ends synchronised: the spectrum is complete
    // Aeff at this record's z: a taper's a(z)²·aeff_intg from the last refresh
    // (at z: the step's final stage, or lh_stats_eval's own), else the constant
    double st_aeff = in.st_aeff, st_ediv = in.st_ediv;
    if (KIND == 0 && in.zg_np > 0 && in.ztaper) {
        const double sa = sm.zs[2] * in.zsqrt_intg;
        st_aeff = sa * sa;
        st_ediv = sqrt(LH_EPS0 * LH_CLIGHT * st_aeff / 2);
    }
    {
        // energy windows: reduced and written here, so the sums do not stay live
        const double nan = __longlong_as_double(0x7ff8000000000000LL);
        double e[LH_STAT_MAX_WINDOWS] = {nan, nan, nan, nan};
        if (in.st_nwin > 0) {
            double w0 = ws.s[0], w1 = ws.s[1], w2 = ws.s[2], w3 = ws.s[3];
            block_sum4(w0, w1, w2, w3, sm.wsum);
            e[0] = w0;
            e[1] = (in.st_nwin > 1) ? w1 : nan;
            e[2] = (in.st_nwin > 2) ? w2 : nan;
            e[3] = (in.st_nwin > 3) ? w3 : nan;
        }
        if (tid == 0) {
#pragma unroll
            for (int q = 0; q < LH_STAT_MAX_WINDOWS; q++) rec[LH_STAT_WINDOW0 + q] = e[q];
        }
    }
    fft_lds<NT, true>(sm.buf, sm.tw);
    // pass 1: P = |Et|² (kept in .x), rate (kept in .y); argmax, max/sum of
    // rate.  Sample j = tid + m·LH_T; rates in batches of QC (spline-table
    // loads issued together).
    constexpr int MPT = NT / LH_T, QC = (MPT < 4) ? MPT : 4;
    static_assert(NT % LH_T == 0 && MPT % QC == 0, "stats sample split");
    const double inv = 1.0 / (double)NT;  // FFTW's ifft normalisation
    const bool ion = (KIND == 0) && in.plasma;
    double pmax = -1.0, rmax = 0.0, rsum = 0.0;
    int imax = NT, bad = LH_OK;
#pragma unroll 1
    for (int c = 0; c < MPT; c += QC) {
        double p[QC], aE[QC], r[QC];
#pragma unroll
        for (int q = 0; q < QC; q++) {
            const double2 e = sm.buf[pad(tid + (c + q) * LH_T)];
            const double re = e.x * inv, im = e.y * inv;
            p[q] = re * re + im * im;
            aE[q] = fabs(re / st_ediv);
            r[q] = 0.0;
        }
        bool need = false;  // any sample at or above the table start (or NaN)
#pragma unroll
        for (int q = 0; q < QC; q++) need |= !(aE[q] < in.ppt_emin);
        if (ion && need) {  // most of the window is below it: those waves skip the table
            ppt_rates<QC>(in, aE, r, bad);
#pragma unroll
            for (int q = 0; q < QC; q++) {
                rmax = fmax(rmax, r[q]);
                rsum += r[q];
            }
        }
#pragma unroll
        for (int q = 0; q < QC; q++) {
            if (p[q] > pmax) {  // j increases within a thread: the first maximum is kept
                pmax = p[q];
                imax = tid + (c + q) * LH_T;
            }
            sm.buf[pad(tid + (c + q) * LH_T)] = make_double2(p[q], r[q]);
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        double p2 = __shfl_xor(pmax, off, 64);
        int i2 = __shfl_xor(imax, off, 64);
        if (p2 > pmax || (p2 == pmax && i2 < imax)) {
            pmax = p2;
            imax = i2;
        }
        rmax = fmax(rmax, __shfl_xor(rmax, off, 64));
        rsum += __shfl_xor(rsum, off, 64);
    }
    if (lane == 0) {
        sm.wsum[4 * wid + 0] = pmax;
        sm.wsum[4 * wid + 1] = (double)imax;
        sm.wsum[4 * wid + 2] = rmax;
        sm.wsum[4 * wid + 3] = rsum;
    }
    if (bad != LH_OK) sm.flag = bad;
    __syncthreads();
    pmax = sm.wsum[0];
    imax = (int)sm.wsum[1];
    rmax = sm.wsum[2];
    rsum = sm.wsum[3];
    for (int w = 1; w < LH_NW; w++) {
        double p2 = sm.wsum[4 * w];
        int i2 = (int)sm.wsum[4 * w + 1];
        if (p2 > pmax || (p2 == pmax && i2 < imax)) {
            pmax = p2;
            imax = i2;
        }
        rmax = fmax(rmax, sm.wsum[4 * w + 2]);
        rsum += sm.wsum[4 * w + 3];
    }
    __syncthreads();
    // pass 2: level crossings around the maximum at val = 0.5·max (t increasing,
    // so x < xmax ⇔ j < imax):  :min takes the last j < imax with P < val and the
    // first j > imax with P < val; :max the first j < imax with P > val and the
    // last j > imax with P > val.
    const double val = 0.5 * pmax;
    int aL = -1, aR = NT, bL = NT, bR = -1;
#pragma unroll
    for (int m = 0; m < MPT; m++) {
        const int j = tid + m * LH_T;
        const double p = sm.buf[pad(j)].x;
        if (j < imax) {
            if (p < val) aL = max(aL, j);
            if (p > val) bL = min(bL, j);
        } else if (j > imax) {
            if (p < val) aR = min(aR, j);
            if (p > val) bR = max(bR, j);
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        aL = max(aL, __shfl_xor(aL, off, 64));
        aR = min(aR, __shfl_xor(aR, off, 64));
        bL = min(bL, __shfl_xor(bL, off, 64));
        bR = max(bR, __shfl_xor(bR, off, 64));
    }
    if (lane == 0) {
        sm.wsum[4 * wid + 0] = (double)aL;
        sm.wsum[4 * wid + 1] = (double)aR;
        sm.wsum[4 * wid + 2] = (double)bL;
        sm.wsum[4 * wid + 3] = (double)bR;
    }
    __syncthreads();
    if (tid == 0) {
        for (int w = 0; w < LH_NW; w++) {
            aL = max(aL, (int)sm.wsum[4 * w + 0]);
            aR = min(aR, (int)sm.wsum[4 * w + 1]);
            bL = min(bL, (int)sm.wsum[4 * w + 2]);
            bR = max(bR, (int)sm.wsum[4 * w + 3]);
        }
        const double* t = gl(in.st_t);
        const double nan = __longlong_as_double(0x7ff8000000000000LL);
        // a missing crossing or a neighbour off the grid is the reference's
        // caught exception: NaN
        double fmin_ = nan, fmax_ = nan;
        if (imax < NT && aL >= 0 && aR < NT) {
            double left = linterpx(t[aL], t[aL + 1], sm.buf[pad(aL)].x, sm.buf[pad(aL + 1)].x, val);
            double right = linterpx(t[aR - 1], t[aR], sm.buf[pad(aR - 1)].x, sm.buf[pad(aR)].x, val);
            fmin_ = fabs(right - left);
        }
        if (imax < NT && bL >= 1 && bL < NT && bR >= 0 && bR + 1 < NT) {
            double left = linterpx(t[bL - 1], t[bL], sm.buf[pad(bL - 1)].x, sm.buf[pad(bL)].x, val);
            double right = linterpx(t[bR], t[bR + 1], sm.buf[pad(bR)].x, sm.buf[pad(bR + 1)].x, val);
            fmax_ = fabs(right - left);
        }
        double ed = nan, pr = nan;
        if (ion) {
            // cumtrapz!(out, δt) end value: Σ ½(r_{j-1} + r_j)·δt
            const double dt = t[1] - t[0];
            double integral = (rsum - 0.5 * (sm.buf[pad(0)].y + sm.buf[pad(NT - 1)].y)) * dt;
            ed = (1.0 - exp(-integral)) * rho;
            pr = rmax;
        }
        rec[LH_STAT_Z] = z;
        rec[LH_STAT_DZ] = dz;
        rec[LH_STAT_OMEGA0] = s1 / s0;
        rec[LH_STAT_ENERGY] = se;
        rec[LH_STAT_PEAKPOWER] = pmax;
        rec[LH_STAT_PEAKINTENSITY] = pmax / st_aeff;
        rec[LH_STAT_FWHM_T_MIN] = fmin_;
        rec[LH_STAT_FWHM_T_MAX] = fmax_;
        rec[LH_STAT_ELECTRONDENSITY] = ed;
        rec[LH_STAT_PEAK_IONISATION_RATE] = pr;
        rec[LH_STAT_DENSITY] = rho;
    }
    __syncthreads();
}

// Envelope grid of NO points (Nto = Nt).
template <int NO, class Smem>
__device__ __forceinline__ void stage_prologue_env(const DInst& in, Smem& sm, const double2* Y, const KSet& K,
                                                   int stage, double dt, double h0, double hf) {
    constexpr int N = NO, NPT = NO / LH_T;
    const int tid = fresh_tid();
    double2 yb[NPT], L[NPT];
#pragma unroll
    for (int i = 0; i < NPT; i++) {
        int k = tid + i * LH_T;
        bool v = k < N;
        yb[i] = v ? Y[k] : make_double2(0.0, 0.0);
        L[i] = v ? static_cast<const double2*>(gl(in.linop))[k] : make_double2(0.0, 0.0);
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
#pragma unroll 1
    for (int j = 0; j <= stage; j++) {
        const double cj = dt * c_B[stage][j];
        if (cj == 0.0) continue;
        const double2* Kj = K[j];
#pragma unroll
        for (int i = 0; i < NPT; i++) {
            int k = tid + i * LH_T;
            if (k < N) yb[i] = cadd(yb[i], cscal(cj, Kj[k]));
        }
    }
    const double sc_t = in.sc_t;
#pragma unroll
    for (int i = 0; i < NPT; i++) {
        int k = tid + i * LH_T;
        if (k < N) {
            // exp(L·hf), and for the stage epilogue exp(L·(t − t2)) = exp(−L·hf)
            // from the same exp and sincos into slot 7 (saves the envelope
            // epilogue, with 16 bins per thread, its own transcendental pass)
            double2 yp = yb[i], inv = make_double2(1.0, 0.0);
            if (hf != 0.0) yp = cmul(yb[i], cexp_lh_inv(L[i], hf, inv));
            sm.buf[pad(k)] = cscal(sc_t, yp);
            K[7][k] = inv;
        }
    }
}

// TransModeAvg on an envelope grid with Kerr_env and RamanPolarEnv
// (src/NonlinearRHS.jl:25-32, 47-53, 362-373, 389-399; src/Nonlinear.jl:47-49,
// 63-73, 282-333).  The Raman convolution of ½|E|² with h(t) over the
// zero-padded 2·Nto grid is done as a real transform: r2c of 2·Nto reals (a
// length-Nto complex FFT), ×(hω δt), c2r, with E(t) in the exchange area meanwhile.
template <int NO, class Smem, class Epi>
__device__ __forceinline__ void rhs_env(const DInst& in, Smem& sm, Epi epi) {
    constexpr int PER = NO / LH_T;  // complex samples per thread (contiguous chunk)
    const int tid = fresh_tid();
    const int i0 = PER * tid;
    __syncthreads();
    fft_lds<NO, true>(sm.buf, sm.tw);
    const double es = in.e_scale;
    if (in.raman) {
        double2 E[PER];
#pragma unroll
        for (int q = 0; q < PER; q++) {
            double2 z = sm.buf[pad(i0 + q)];
            E[q] = make_double2(z.x * es, z.y * es);
            gl(in.gx)[i0 + q] = E[q];
        }
        __syncthreads();  // every thread has read its E before the packing overwrites
#pragma unroll
        for (int q = 0; q < PER / 2; q++) {
            double a0 = 0.5 * (E[2 * q].x * E[2 * q].x + E[2 * q].y * E[2 * q].y);
            double a1 = 0.5 * (E[2 * q + 1].x * E[2 * q + 1].x + E[2 * q + 1].y * E[2 * q + 1].y);
            sm.buf[pad(i0 / 2 + q)] = make_double2(a0, a1);        // ½|E|², reals packed in pairs
            sm.buf[pad(NO / 2 + i0 / 2 + q)] = make_double2(0.0, 0.0);  // zero padding to 2·Nto
        }
        __syncthreads();
        fft_lds<NO, false>(sm.buf, sm.tw);
        // r2c post-step of the 2·Nto-point transform, ×hω·δt, and the c2r
        // pre-pack of the product, pairwise (k, Nto-k) in place
        constexpr int TS = LH_TWN / (2 * NO);
        for (int k = tid; k <= NO / 2; k += LH_T) {
            int m = NO - k;
            if (k == 0) {
                double2 Y0 = cmul(gl(in.hwdt)[0], r2c_bin<NO>(sm.buf, sm.tw, 0));
                double2 YM = cmul(gl(in.hwdt)[NO], r2c_bin<NO>(sm.buf, sm.tw, NO));
                Y0.y = 0.0;
                YM.y = 0.0;
                double2 A = cadd(Y0, cconj(YM)), B = csub(Y0, cconj(YM));
                sm.buf[pad(0)] = cadd(A, cmul_pi(B));
            } else if (k == NO / 2) {
                double2 Yk = cmul(gl(in.hwdt)[k], r2c_bin<NO>(sm.buf, sm.tw, k));
                double2 A = cadd(Yk, cconj(Yk));
                double2 B = cmul(csub(Yk, cconj(Yk)), cconj(tw_get(sm.tw, k * TS)));
                sm.buf[pad(k)] = cadd(A, cmul_pi(B));
            } else {
                double2 Yk = cmul(gl(in.hwdt)[k], r2c_bin<NO>(sm.buf, sm.tw, k));
                double2 Ym = cmul(gl(in.hwdt)[m], r2c_bin<NO>(sm.buf, sm.tw, m));
                double2 wk = cconj(tw_get(sm.tw, k * TS)), wm = cconj(tw_get(sm.tw, m * TS));
                double2 Ak = cadd(Yk, cconj(Ym)), Bk = cmul(csub(Yk, cconj(Ym)), wk);
                double2 Am = cadd(Ym, cconj(Yk)), Bm = cmul(csub(Ym, cconj(Yk)), wm);
                sm.buf[pad(k)] = cadd(Ak, cmul_pi(Bk));
                sm.buf[pad(m)] = cadd(Am, cmul_pi(Bm));
            }
        }
        __syncthreads();
        fft_lds<NO, true>(sm.buf, sm.tw);  // P(t) on the 2·Nto grid, packed in pairs
        double P[PER];
#pragma unroll
        for (int q = 0; q < PER / 2; q++) {
            double2 z = sm.buf[pad(i0 / 2 + q)];
            P[2 * q] = z.x * in.inv_2n;
            P[2 * q + 1] = z.y * in.inv_2n;
        }
        __syncthreads();
        const double rho = in.density, k34 = in.kerr34;
        const bool kerr = (in.kerr == LH_KERR_ENV);
        const double* tw = gl(in.to_win);
#pragma unroll
        for (int q = 0; q < PER; q++) {
            double2 e = gl(in.gx)[i0 + q];
            double2 p = make_double2(0.0, 0.0);
            if (kerr) {
                double s = k34 * (e.x * e.x + e.y * e.y);
                p = make_double2(s * e.x, s * e.y);
            }
            double2 re = make_double2(rho * e.x, rho * e.y);
            p = cadd(p, make_double2(re.x * P[q], re.y * P[q]));
            sm.buf[pad(i0 + q)] = make_double2(p.x * tw[i0 + q], p.y * tw[i0 + q]);
        }
    } else {
        const double k34 = in.kerr34;
        const bool kerr = (in.kerr == LH_KERR_ENV);
        const double* tw = gl(in.to_win);
#pragma unroll
        for (int q = 0; q < PER; q++) {
            double2 z = sm.buf[pad(i0 + q)];
            double2 e = make_double2(z.x * es, z.y * es);
            double2 p = make_double2(0.0, 0.0);
            if (kerr) {
                double s = k34 * (e.x * e.x + e.y * e.y);
                p = make_double2(s * e.x, s * e.y);
            }
            sm.buf[pad(i0 + q)] = make_double2(p.x * tw[i0 + q], p.y * tw[i0 + q]);
        }
    }
    constexpr int N = NO, NPT = NO / LH_T;
    double2 of[NPT];
#pragma unroll
    for (int i = 0; i < NPT; i++) {
        int k = tid + i * LH_T;
        of[i] = (k < N) ? static_cast<const double2*>(gl(in.outfac))[k] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    fft_lds<NO, false>(sm.buf, sm.tw);
    constexpr int CH = NPT;
    static_assert(NPT <= 9, "one epilogue chunk");
#pragma unroll
    for (int c = 0; c < NPT; c += CH) {
        double2 res[CH];
#pragma unroll
        for (int i = 0; i < CH; i++) {
            int k = tid + (c + i) * LH_T;
            res[i] = (k < N) ? cmul(sm.buf[pad(k)], of[c + i]) : make_double2(0.0, 0.0);
        }
        epi(res, N);
    }
}

// stepfun on the envelope grid (src/Luna.jl:366-370 with a c2c FT).
template <int NT, class Smem>
__device__ __forceinline__ void stepfun_env(const DInst& in, Smem& sm, double2* YN, double h, double* rec, double z,
                                            double dz, double rho) {
    constexpr int NPT = (NT + LH_T - 1) / LH_T;
#pragma unroll
    for (int i = 0; i < NPT; i++) {
        int k = fresh_tid() + i * LH_T;
        if (k < NT) {
            double2 v = YN[k];
            if (h != 0.0) v = cmul(v, cexp_lh(gl(in.linop)[k], h));
            sm.buf[pad(k)] = cscal(gl(in.omega_win)[k], v);
        }
    }
    __syncthreads();
    fft_lds<NT, true>(sm.buf, sm.tw);
    const double inv_nt = in.inv_nt;
    for (int j = fresh_tid(); j < NT; j += LH_T) {
        double2 z = sm.buf[pad(j)];
        double w = gl(in.t_win)[j];
        sm.buf[pad(j)] = make_double2((inv_nt * z.x) * w, (inv_nt * z.y) * w);
    }
    __syncthreads();
    fft_lds<NT, false>(sm.buf, sm.tw);
    double s0 = 0.0, s1 = 0.0, se = 0.0;
    WinSums ws = {{0.0, 0.0, 0.0, 0.0}};
#pragma unroll
    for (int i = 0; i < NPT; i++) {
        int k = fresh_tid() + i * LH_T;
        if (k < NT) {
            double2 v = sm.buf[pad(k)];
            YN[k] = v;
            if (rec) {  // the envelope's analytic field is ifft(Eω): the spectrum stays in place
                double a = v.x * v.x + v.y * v.y;
                s0 += a;
                s1 += gl(in.st_omega)[k] * a;
                se += gl(in.st_ew)[k] * a;
                win_add(in, ws, k, a);
            }
        }
    }
    if (rec)
        stats_time<1, NT, Smem>(in, sm, s0, s1, se, ws, z, dz, rho, rec);
    else
        __syncthreads();
}

template <int KIND, int MO, class Smem>
__device__ __forceinline__ void prologue(const DInst& in, Smem& sm, const double2* Y, const KSet& K, int stage, double dt,
                                         double h0, double hf) {
    if constexpr (KIND == 0)
        stage_prologue<MO, Smem>(in, sm, Y, K, stage, dt, h0, hf);
    else
        stage_prologue_env<MO, Smem>(in, sm, Y, K, stage, dt, h0, hf);
}
template <int KIND, int MO, bool RAMAN, class Smem, class Epi>
__device__ __forceinline__ void rhs(const DInst& in, Smem& sm, Epi epi, double rho, double kfac) {
    if constexpr (KIND == 0)
        rhs_field<MO, RAMAN, Smem, Epi>(in, sm, epi, rho, kfac);
    else
        rhs_env<MO, Smem>(in, sm, epi);
}

// Adaptive solve of one instance (Luna.run → RK45.solve_precon).
template <int KIND, int MO, int MC, bool ZDEP, bool RAMAN, class Smem>
__device__ __forceinline__ void solo_solve(const DInst& in, Smem& sm) {
    constexpr int N = (KIND == 0) ? Bins<MO>::N : MO, NPT = (N + LH_T - 1) / LH_T;
    KSet K{gl(in.K), in.kstride, 0, 6};
    double2* const Y0 = gl(in.Y);
    double2* Y = gl(in.Y);
    double2* YN = K[8];
    for (int k = fresh_tid(); k < N; k += LH_T) Y[k] = gl(in.Yin)[k];
    if (threadIdx.x == 0) sm.flag = LH_OK;
    __syncthreads();

    long long steps = 0, accepted = 0, rejected = 0, rhs_evals = 0;
    int status = LH_OK, saved = in.save_first, repeated = 0;
    double t = in.z0, tn = in.z0, dt = in.init_dz, dtn = in.init_dz, errlast = 0.0;
    // density and Kerr factor of the current z, re-evaluated with the operator at
    // every new z
    double rho = in.density, kfac = in.kerr_fac;
    if constexpr (ZDEP) zg_refresh(in, sm, in.z0, rho, kfac);

    // PreconStepper init: k1 = fbar(y0, t, t)
    prologue<KIND, MO, Smem>(in, sm, Y, K, 0, 0.0, 0.0, 0.0);
    rhs<KIND, MO, RAMAN, Smem>(in, sm, EpiStore{K[0]}, rho, kfac);
    rhs_evals++;
    __syncthreads();
    if (sm.flag != LH_OK) status = sm.flag;

    while (status == LH_OK && tn <= in.zmax) {
        if (steps >= in.max_steps) {
            status = LH_E_MAXSTEPS;
            break;
        }
        // evaluate!
        double h0 = tn - t;
        dt = dtn;
        t = tn;
        if (threadIdx.x == 0)
            __hip_atomic_store(in.beat, (unsigned)steps, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // prop!(ks[1], t, tn) with the operator at tn; each stage then
        // re-evaluates it at its own t2
        if constexpr (ZDEP) {
            zg_refresh(in, sm, t, rho, kfac);
            if (h0 != 0.0) {
                double2* K0 = K[0];
                for (int k = fresh_tid(); k < N; k += LH_T) K0[k] = cmul(K0[k], cexp_lh(gl(in.linop)[k], h0));
                __syncthreads();
            }
            h0 = 0.0;
        }
#pragma unroll 1
        for (int st = 0; st < 6 && status == LH_OK; st++) {
            double t2 = t + c_nodes[st] * dt;
            double hf = t2 - t;
            if (ZDEP && st != 5) zg_refresh(in, sm, t2, rho, kfac);  // stages 5 and 6 share t + dt
            prologue<KIND, MO, Smem>(in, sm, Y, K, st, dt, h0, hf);
            rhs<KIND, MO, RAMAN, Smem>(in, sm, EpiStageFO{K[st + 1], K[7]}, rho, kfac);
            rhs_evals++;
            __syncthreads();
            if (sm.flag != LH_OK) status = sm.flag;
        }
        if (status != LH_OK) break;
        steps++;
        // yn = y + Δz Σ b5 k ; yerr = Σ (Δz k) e ; weaknorm (src/RK45.jl:170-181, 343-354)
        double sy = 0.0, syn = 0.0, se = 0.0;
        if constexpr (NPT == 9) {
            // chunks of three bins, y and the six k-vectors of each loaded in
            // one round (three rounds instead of seven: 123.9 → 121.4 ms for
            // the Nto = 16384 class; results within 1e-13, steps unchanged)
            constexpr int CB = 3;
#pragma unroll 1
            for (int c = 0; c < NPT; c += CB) {
                double2 yv[CB], kk[7][CB];
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    const int k = fresh_tid() + (c + i) * LH_T;
                    yv[i] = (k < N) ? Y[k] : make_double2(0.0, 0.0);
                }
#pragma unroll
                for (int j = 0; j < 7; j++) {
                    if (j == 1) continue;
                    const double2* Kj = K[j];
#pragma unroll
                    for (int i = 0; i < CB; i++) {
                        const int k = fresh_tid() + (c + i) * LH_T;
                        kk[j][i] = (k < N) ? Kj[k] : make_double2(0.0, 0.0);
                    }
                }
                double2 yn[CB], ye[CB];
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    yn[i] = yv[i];
                    ye[i] = make_double2(0.0, 0.0);
                }
#pragma unroll
                for (int j = 0; j < 7; j++) {
                    if (j == 1) continue;  // b5[2] = b4[2] = 0
                    const double cb = dt * c_b5[j], ce = c_b5[j] - c_b4[j];
#pragma unroll
                    for (int i = 0; i < CB; i++) {
                        const int k = fresh_tid() + (c + i) * LH_T;
                        if (k < N) {
                            yn[i] = cadd(yn[i], cscal(cb, kk[j][i]));
                            ye[i] = cadd(ye[i], cscal(ce, cscal(dt, kk[j][i])));
                        }
                    }
                }
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    const int k = fresh_tid() + (c + i) * LH_T;
                    if (k < N) {
                        sy += yv[i].x * yv[i].x + yv[i].y * yv[i].y;
                        syn += yn[i].x * yn[i].x + yn[i].y * yn[i].y;
                        se += ye[i].x * ye[i].x + ye[i].y * ye[i].y;
                        YN[k] = yn[i];
                    }
                }
            }
        } else {
            double2 yv[NPT], yn[NPT], ye[NPT];
#pragma unroll
            for (int i = 0; i < NPT; i++) {
                int k = fresh_tid() + i * LH_T;
                yv[i] = (k < N) ? Y[k] : make_double2(0.0, 0.0);
                yn[i] = yv[i];
                ye[i] = make_double2(0.0, 0.0);
            }
#pragma unroll 1
            for (int j = 0; j < 7; j++) {
                if (j == 1) continue;  // b5[2] = b4[2] = 0
                const double cb = dt * c_b5[j], ce = c_b5[j] - c_b4[j];
                const double2* Kj = K[j];
#pragma unroll
                for (int i = 0; i < NPT; i++) {
                    int k = fresh_tid() + i * LH_T;
                    if (k < N) {
                        double2 kv = Kj[k];
                        yn[i] = cadd(yn[i], cscal(cb, kv));
                        ye[i] = cadd(ye[i], cscal(ce, cscal(dt, kv)));
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < NPT; i++) {
                int k = fresh_tid() + i * LH_T;
                if (k < N) {
                    sy += yv[i].x * yv[i].x + yv[i].y * yv[i].y;
                    syn += yn[i].x * yn[i].x + yn[i].y * yn[i].y;
                    se += ye[i].x * ye[i].x + ye[i].y * ye[i].y;
                    YN[k] = yn[i];
                }
            }
        }
        block_sum3(sy, syn, se, sm.wsum);
        double errwt = fmax(fmax(sqrt(sy), sqrt(syn)), in.atol);
        double err = sqrt(se) / in.rtol / errwt;
        bool ok = err <= 1.0;
        // stepcontrolPI!, src/RK45.jl:374-396, steplims! :399-406
        const double beta1 = 3.0 / 5 / 5, beta2 = -1.0 / 5 / 5, eps = 0.8;
        if (ok) {
            if (errlast == 0.0) errlast = err;
            double fac = (err == 0.0) ? 1.5 : in.safety * pow(eps / err, beta1) * pow(eps / errlast, beta2);
            dtn = fac * dt;
            errlast = err;
        } else {
            if (!isfinite(err))
                dtn = dt / 2;
            else
                dtn = dt * fmax(0.1, in.safety * pow(err, -1.0 / 5));
        }
        if (dtn > in.max_dz)
            dtn = in.max_dz;
        else if (dtn < in.min_dz) {
            dtn = in.min_dz;
            ok = true;
        }
        if (ok) {
            tn = t + dt;
            K.swap06();  // FSAL: ks[1] .= ks[7] (src/RK45.jl:184-186)
            // stepfun, then MemoryOutput's statistics of the filtered state
            // (src/Output.jl:65-67) from the same LDS pass
            double* rec = (gl(in.steprec) && accepted < in.steprec_cap) ? gl(in.steprec) + (size_t)accepted * LH_NSTAT
                                                                      : nullptr;
            if constexpr (KIND == 0)
                stepfun_filter<MC, Smem>(in, sm, YN, tn - t, rec, tn, dtn, rho);
            else
                stepfun_env<MO, Smem>(in, sm, YN, tn - t, rec, tn, dtn, rho);
            if (rec && sm.flag != LH_OK) status = sm.flag;
            // GridCondition saves via dense output; ks[1] and ks[7] both hold k7
            while (saved < in.save_n && gl(in.zgrid)[saved] <= tn) {
                double ti = gl(in.zgrid)[saved];
                if (ZDEP && gl(in.saves) && ti != t && ti != tn) zg_refresh(in, sm, ti, rho, kfac);  // prop!(out, t, ti)
                if (gl(in.saves)) {
                    double2* out = gl(in.saves) + (size_t)saved * N;
                    if (ti == t) {
                        for (int k = fresh_tid(); k < N; k += LH_T) out[k] = Y[k];
                    } else if (ti == tn) {
                        for (int k = fresh_tid(); k < N; k += LH_T) out[k] = YN[k];
                    } else {
                        double sg = (ti - t) / dt;
                        const double sp1 = sg, sp2 = pow(sg, 2.0), sp3 = pow(sg, 3.0), sp4 = pow(sg, 4.0);
                        double h = ti - t;
                        // this thread's bins in registers (chunks of at most 9),
                        // one k-vector at a time, every load of a chunk before
                        // its first store to out
                        constexpr int CH = NPT;
                        if constexpr (NPT == 9) {
                            // chunks of three bins, y, L and the six k-vectors of
                            // each loaded in one round (three rounds per save
                            // instead of seven: 121.9 → 120.1 ms for the Nto =
                            // 16384 class, bit-identical results)
                            constexpr int CB = 3;
#pragma unroll 1
                            for (int c = 0; c < NPT; c += CB) {
                                double2 kk[7][CB], yv[CB], Lv[CB], yi[CB];
#pragma unroll
                                for (int i = 0; i < CB; i++) {
                                    const int k = fresh_tid() + (c + i) * LH_T;
                                    yv[i] = (k < N) ? Y[k] : make_double2(0.0, 0.0);
                                    Lv[i] = (k < N) ? static_cast<const double2*>(gl(in.linop))[k] : make_double2(0.0, 0.0);
                                    yi[i] = make_double2(0.0, 0.0);
                                }
#pragma unroll
                                for (int j = 0; j < 7; j++) {
                                    if (j == 1) continue;
                                    const double2* kj = (j == 6) ? K[0] : K[j];
#pragma unroll
                                    for (int i = 0; i < CB; i++) {
                                        const int k = fresh_tid() + (c + i) * LH_T;
                                        kk[j][i] = (k < N) ? kj[k] : make_double2(0.0, 0.0);
                                    }
                                }
#pragma unroll
                                for (int j = 0; j < 7; j++) {
                                    if (j == 1) continue;
                                    const double bj =
                                        ((sp1 * c_iC[0][j] + sp2 * c_iC[1][j]) + sp3 * c_iC[2][j]) + sp4 * c_iC[3][j];
#pragma unroll
                                    for (int i = 0; i < CB; i++) yi[i] = cadd(yi[i], cscal(bj, kk[j][i]));
                                }
#pragma unroll
                                for (int i = 0; i < CB; i++) {
                                    const int k = fresh_tid() + (c + i) * LH_T;
                                    if (k < N) out[k] = cmul(cadd(yv[i], cscal(dt, yi[i])), cexp_lh(Lv[i], h));
                                }
                            }
                        } else
#pragma unroll 1
                        for (int c = 0; c < NPT; c += CH) {
                            double2 yi[CH], yv[CH], Lv[CH];
#pragma unroll
                            for (int i = 0; i < CH; i++) yi[i] = make_double2(0.0, 0.0);
#pragma unroll 1
                            for (int j = 0; j < 7; j++) {
                                if (j == 1) continue;
                                const double2* kj = (j == 6) ? K[0] : K[j];
                                // weight b_j(σ) = Σ_p σ^p C[p][j] of the dense output
                                const double bj =
                                    ((sp1 * c_iC[0][j] + sp2 * c_iC[1][j]) + sp3 * c_iC[2][j]) + sp4 * c_iC[3][j];
#pragma unroll
                                for (int i = 0; i < CH; i++) {
                                    const int k = fresh_tid() + (c + i) * LH_T;
                                    if (k < N) yi[i] = cadd(yi[i], cscal(bj, kj[k]));
                                }
                            }
#pragma unroll
                            for (int i = 0; i < CH; i++) {
                                const int k = fresh_tid() + (c + i) * LH_T;
                                yv[i] = (k < N) ? Y[k] : make_double2(0.0, 0.0);
                                Lv[i] = (k < N) ? static_cast<const double2*>(gl(in.linop))[k] : make_double2(0.0, 0.0);
                            }
#pragma unroll
                            for (int i = 0; i < CH; i++) {
                                const int k = fresh_tid() + (c + i) * LH_T;
                                if (k < N) out[k] = cmul(cadd(yv[i], cscal(dt, yi[i])), cexp_lh(Lv[i], h));
                            }
                        }
                    }
                }
                saved++;
            }
            double2* tmp2 = Y;
            Y = YN;
            YN = tmp2;
            accepted++;
            repeated = 0;
            if (in.zstop > 0.0 && tn > in.zstop && tn <= in.zmax) status = LH_E_STOPPED;
        } else {
            rejected++;
            repeated++;
            if (repeated > in.repeat_limit) status = LH_E_REPEAT_LIMIT;
        }
        __syncthreads();
    }
    // The final state s.yn lives in whichever buffer Y points to after the
    // swaps; copy it into the caller-visible buffer Y0.
    if (Y != Y0)
        for (int k = fresh_tid(); k < N; k += LH_T) Y0[k] = Y[k];
    if (threadIdx.x == 0 && gl(in.stats)) {
        lh_stats s;
        s.steps = steps;
        s.accepted = accepted;
        s.rejected = rejected;
        s.rhs_evals = rhs_evals;
        s.status = status;
        s.saved = saved;
        s.z = tn;
        s.dz = dtn;
        in.stats->s = s;
    }
    __syncthreads();
}

template <int KIND, int MO, int MC, bool ZDEP, bool RAMAN>
__global__ __launch_bounds__(LH_T) void lh_solo_solve(const DInst* insts, const double2* __restrict__ twg) {
    __shared__ SmemT<MO> sm;
    tw_load(sm.tw, twg);
    __syncthreads();
    solo_solve<KIND, MO, MC, ZDEP, RAMAN, SmemT<MO>>(insts[blockIdx.x], sm);
}

template <int KIND, int MO, int MC, bool ZDEP, bool RAMAN>
static inline void solo_launch(int n, const DInst* d, const double2* tw, hipStream_t s) {
    hipLaunchKernelGGL((lh_solo_solve<KIND, MO, MC, ZDEP, RAMAN>), dim3(n), dim3(LH_T), 0, s, d, tw);
}
