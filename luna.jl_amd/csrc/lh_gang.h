// lh_gang.h -- mode-averaged propagation by gangs of four workgroups (gfx950).
//
// Compiled by lh_gang_field.hip, lh_gang_raman.hip, lh_gang_env.hip and
// lh_gang_dense.hip.  One instance is
// solved by a gang: four workgroups of 512 threads on four CUs of one XCD,
// which exchange data through that XCD's L2.  A transform of M points splits
// as M = 8·S: the bins k ≡ r (mod 8) form one S-point transform, and an
// 8-point transform over r joins them.  Member h of the gang owns
//   bins:  the residues r = ±h mod 8 (member 0: r = 0 and 4), closed under
//          k → M − k, so the packing of real transforms stays inside a member;
//   time:  n ≡ h·S/4 .. (h+1)·S/4 − 1 (mod S): eight runs of S/4 consecutive
//          points, one per wavefront.
// One exchange of the series (each member writes its residues, reads its times)
// turns one into the other.  The cumulative integrals of the plasma response
// exchange one record per run (32 of them), the norms one record per member.
//
// What bounds it: latency.  A right-hand side is a chain of some twenty phases
// (LDS passes, exchanges, scans), each shorter than 2 us; the vector ALUs are
// busy 30 % of the time.  An exchange costs 0.7 to 0.9 us through L2 and a
// right-hand side with plasma has four, whatever the gang's size, so the gain
// per added CU falls: four members are a compromise between one propagation
// alone and a sweep that fills the chip.  Measured against one workgroup per
// instance (one MI355X): a propagation at Nto = 8192 18.4 → 10.6 ms, envelope
// Nt = 8192 with Raman 274 → 87 ms, Nt = 16384 57.4 → 11.8 ms, a single
// right-hand side at Nto = 16384 56 → 38 us; a 64-point sweep 41.6 → 19.6 ms,
// 256 points 47.1 → 45.2 ms.
//
// Gangs form by themselves: every workgroup of a launch takes a ticket of its
// XCD (HW_REG_XCC_ID), and four consecutive tickets are a gang, so members are
// resident and share an L2 whatever the order of dispatch.  Gangs then take
// jobs (instances) from one counter until none is left.  A launch has at least
// 32 workgroups, so that one of at most eight XCDs gets four of them; where
// they don't become resident there, the launch ends with LH_E_HIP
// (lh_gang_proto.h).

#pragma once
#include "lh_core.h"
#include "lh_gang_launch.h"

typedef double lg_d2 __attribute__((ext_vector_type(2)));

static constexpr int LG_MAX_POLL = 1 << 25;  // polls of another member before it counts as lost (some ten seconds)
static_assert(LG_LOST == LH_E_HIP, "the protocol's status of a lost member");

static_assert(LH_T == 512, "a gang member is 8 wavefronts, one per run of its times");

// Slots of the work block in.K (each kstride long, member h at h·GSTR):
// k1..k7, the stage factor F = outfac·exp(−L·hf), member-ordered copies of the
// operator, the output factor and the Raman response, the two states, and
// exp(L·dz) of the step.
enum LgVec { LG_F = 7, LG_L = 8, LG_OF = 9, LG_YA = 10, LG_YB = 11, LG_HW = 12, LG_E = 13 };

template <class T>
__device__ __forceinline__ T lg_ld(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void lg_st(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The protocol's memory operations (lh_gang_proto.h).
struct LgMem {
    template <class T>
    __device__ __forceinline__ static T ld(const T* p) {
        return lg_ld(p);
    }
    __device__ __forceinline__ static void st(unsigned long long* p, unsigned long long v) { lg_st(p, v); }
    __device__ __forceinline__ static unsigned add(unsigned* p, unsigned v) {
        return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ static unsigned long long cas(unsigned long long* p, unsigned long long old,
                                                             unsigned long long v) {
        __hip_atomic_compare_exchange_strong(p, &old, v, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return old;
    }
    __device__ __forceinline__ static void drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
    __device__ __forceinline__ static void pause() { __builtin_amdgcn_s_sleep(8); }
};

// 16-byte loads past the CU's L1 (which may hold a line's earlier content) of
// the series the other members wrote: a buffer descriptor over it and the
// device-scope bit.
struct GxView {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ GxView(const double2* p, int n)
        : r(__builtin_amdgcn_make_buffer_rsrc((void*)p, 0, n * 16, 0x00027000)) {}
    __device__ __forceinline__ double2 operator[](int i) const {
        const lg_d2 v = __builtin_bit_cast(lg_d2, __builtin_amdgcn_raw_buffer_load_b128(r, i * 16, 0, 16));
        return make_double2(v.x, v.y);
    }
};

// Twiddles: W^m = hi[m >> 7] · lo[m & 127], W = exp(-2πi/LG_TWN).
struct GTw {
    double2 lo[128];
    double2 hi[256];
};
__device__ __forceinline__ void gtw_load(GTw& t, const double2* __restrict__ tw) {
    for (int i = threadIdx.x; i < 256; i += LH_T) {
        if (i < 128) t.lo[i] = tw[i];
        t.hi[i] = tw[128 * i];
    }
}
template <int L>
__device__ __forceinline__ double2 gtw(const GTw& t, int k) {  // exp(-2πi k/L), 0 <= k < L
    static_assert(LG_TWN % L == 0, "twiddle length");
    const int m = k * (LG_TWN / L);
    return cmul(t.hi[m >> 7], t.lo[m & 127]);
}

// LDS of a member.  BUF: complex points it holds of the longest transform.
template <int BUF, int CAP>
struct GSmem {
    static constexpr int PCAP = CAP;
    double2 buf[padded_len(BUF + 1)];
    GTw tw;
    double wsum[5 * LH_NW];
    double scan[LH_NW];
    double plist[CAP];
    double zs[3];
    int flag;   // error raised by this member
    int gflag;  // first error of any member, as of the last barrier
    int job, member, slot;
};

struct Gang {
    int h;
    unsigned ep;
    unsigned* flags;
    double* rec;   // [2][32][8]
    double2* X;    // [2][xlen]
    double* P;     // [M] |Et|² of the statistics
    int xlen, xb, rb;
    __device__ __forceinline__ double2* xnext() {
        double2* p = X + (size_t)xb * xlen;
        xb ^= 1;
        return p;
    }
    __device__ __forceinline__ double* rnext() {
        double* p = rec + 256 * rb;
        rb ^= 1;
        return p;
    }
};

// Barrier of the gang: the stores of every member before it are in L2 when it
// ends.  Each wavefront waits for its own stores (the L2 acknowledges them),
// then one lane raises the member's flag to the new epoch and four lanes poll
// all flags.  A flag also carries the member's error status, so all members see
// an error at the first barrier after it.  A member that another one does not
// join within LG_MAX_POLL polls goes on alone with LH_E_HIP and raises its flag
// again with that, which the late one finds there or at its next barrier.
template <class SM>
__device__ __forceinline__ void gang_sync(Gang& g, SM& sm) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    g.ep++;
    const int t = threadIdx.x;
    if (t < 64) {
        if (t == 0) lg_st(g.flags + LG_FLAG_STRIDE * g.h, lg_flag(g.ep, sm.flag));
        if (t < LG_G) {
            // (one that goes on alone looks once)
            const int st = lg_await<LgMem>(g.flags + LG_FLAG_STRIDE * t, g.ep, sm.gflag == LG_LOST ? 1 : LG_MAX_POLL);
            if (__any(st != LH_OK)) {
                if (__any(st == LG_LOST)) {
                    sm.flag = sm.gflag = LG_LOST;
                    if (t == 0) lg_st(g.flags + LG_FLAG_STRIDE * g.h, lg_flag(g.ep, LG_LOST));
                } else if (st != LH_OK && sm.gflag == LH_OK) {
                    sm.gflag = st;
                }
            }
        }
    }
    __syncthreads();
}

// Member geometry for transforms of M points.
template <int M>
struct GGeo {
    static constexpr int S = M / 8;     // points per residue
    static constexpr int RUN = M / 32;  // consecutive complex times per run (S/4)
    __device__ static __forceinline__ int res(int h, int s) { return s == 0 ? h : (h == 0 ? 4 : 8 - h); }
    // LDS index of bin M − k for bin k = res(h, s) + 8q
    __device__ static __forceinline__ int conj_idx(int h, int s, int q) {
        if (h != 0) return (1 - s) * S + (S - 1 - q);
        if (s != 0) return S + (S - 1 - q);
        return q == 0 ? 0 : S - q;
    }
};

// Radix of the pass that has S/NS = REM points left: the fewest passes of
// radix 16 and 8 (radices up to 8 with a pass more: the same time within 1 %).
template <int REM>
struct GRadix {
    static constexpr int R = (REM == 8 || REM == 64 || REM == 512) ? 8 : 16;
};

// v[r] *= w^r, r = 1..R−1, the powers by products of lower ones (depth log2 R).
template <int R>
__device__ __forceinline__ void mul_powers(double2* v, double2 w) {
    double2 p[R];
    p[1] = w;
#pragma unroll
    for (int r = 2; r < R; r++) p[r] = cmul(p[(r + 1) / 2], p[r / 2]);
#pragma unroll
    for (int r = 1; r < R; r++) v[r] = cmul(v[r], p[r]);
}

// One radix-R Stockham pass over the member's two S-point transforms (2·S/R
// butterflies, one thread each).  SRC and DST: 0 the LDS buffer (transform s at
// index s·S), 1 the exchange series (residue r at index r·S).
template <int S, int R, int NS, bool INV, int SRC, int DST, class SM>
__device__ __forceinline__ void gpass(SM& sm, const double2* src, double2* dst, int r0, int r1) {
    constexpr int NB = S / R, TOT = 2 * NB;
    static_assert(TOT <= LH_T, "one butterfly per thread");
    const int tid = fresh_tid();
    const int s = tid / NB, j = tid - s * NB;
    const bool act = tid < TOT;
    double2 v[R];
    if (act) {
        if constexpr (SRC == 0) {
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = sm.buf[pad(s * S + j + r * NB)];
        } else {
            const GxView x(src, 8 * S);
            const int b = (s ? r1 : r0) * S + j;
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = x[b + r * NB];
        }
    }
    if constexpr (SRC == 0 && DST == 0) __syncthreads();
    if (act) {
        const int k = j & (NS - 1);
        if constexpr (NS > 1) {
            double2 w1 = gtw<NS * R>(sm.tw, k);
            if (INV) w1.y = -w1.y;
            mul_powers<R>(v, w1);
        }
        dft<R, INV>(v);
        const int idx = (j - k) * R + k;
        if constexpr (DST == 0) {
#pragma unroll
            for (int r = 0; r < R; r++) sm.buf[pad(s * S + idx + r * NS)] = v[r];
        } else {
            double2* o = gl(dst) + (s ? r1 : r0) * S + idx;
#pragma unroll
            for (int r = 0; r < R; r++) o[r * NS] = v[r];
        }
    }
    if constexpr (DST == 0) __syncthreads();
}

template <int S, int NS, bool INV, class SM>
__device__ __forceinline__ void gpasses(SM& sm, const double2* src, double2* dst, int r0, int r1) {
    if constexpr (NS < S) {
        constexpr int R = GRadix<S / NS>::R;
        constexpr bool LAST = NS * R == S;
        gpass<S, R, NS, INV, (!INV && NS == 1) ? 1 : 0, (INV && LAST) ? 1 : 0>(sm, src, dst, r0, r1);
        gpasses<S, NS * R, INV>(sm, src, dst, r0, r1);
    }
}

// Inverse: the bins in LDS (synchronised) → S-point transforms in the exchange
// series (before the gang's barrier).  Forward: the reverse, after the barrier;
// ends synchronised.
template <int M, class SM>
__device__ __forceinline__ void g_local_inv(SM& sm, const Gang& g, double2* x) {
    gpasses<M / 8, 1, true>(sm, nullptr, x, GGeo<M>::res(g.h, 0), GGeo<M>::res(g.h, 1));
}
template <int M, class SM>
__device__ __forceinline__ void g_local_fwd(SM& sm, const Gang& g, const double2* x) {
    gpasses<M / 8, 1, false>(sm, x, nullptr, GGeo<M>::res(g.h, 0), GGeo<M>::res(g.h, 1));
}

// The 8-point join at time n0 (mod S): inverse reads the eight residues and
// leaves z[n0 + S·n1] in v[n1]; forward takes those and writes the residues.
template <int M, class SM>
__device__ __forceinline__ void g_join_inv(const SM& sm, const double2* xs, int n0, double2 (&v)[8]) {
    constexpr int S = M / 8;
    const GxView x(xs, M);
#pragma unroll
    for (int r = 0; r < 8; r++) v[r] = x[r * S + n0];
    mul_powers<8>(v, cconj(gtw<M>(sm.tw, n0)));
    dft8<true>(v);
}
template <int M, class SM>
__device__ __forceinline__ void g_join_fwd(const SM& sm, double2* xs, int n0, double2 (&v)[8]) {
    constexpr int S = M / 8;
    dft8<false>(v);
    mul_powers<8>(v, gtw<M>(sm.tw, n0));
    double2* o = gl(xs) + n0;
#pragma unroll
    for (int r = 0; r < 8; r++) o[r * S] = v[r];
}

// Inclusive prefix sum over lanes 0..31.
__device__ __forceinline__ double lanes32_incl_scan(double x) {
    x += dpp_f64<DPP_ROW_SHR1>(x);
    x += dpp_f64<DPP_ROW_SHR2>(x);
    x += dpp_f64<DPP_ROW_SHR4>(x);
    x += dpp_f64<DPP_ROW_SHR8>(x);
    x += dpp_f64<DPP_ROW_BCAST15, 0xa>(x);
    return x;
}

// Pointwise field responses on the member's times in LDS (run sg at index
// sg·RUN, packed pairs of reals), in place: E = z·e_scale, P = ρε0γ3 E³ +
// ρ·Plasma(E) + ρ·E·Raman, ×towin.  Wavefront sg owns run sg, which is run
// 4·sg + h of the 32 runs of the whole series; a lane owns M/2048 consecutive
// pairs.  The integrals F = ∫rate and J, P (Run2) run inside the wavefront by
// DPP, then over the 32 runs' records, which every wavefront reads and scans
// itself.
template <int M, bool RAMAN, class SM>
__device__ __forceinline__ void g_pointwise(const DInst& in, SM& sm, Gang& g, double rho, double kfac,
                                            const double2* praman) {
    constexpr int C = M / 2048, QR = 2 * C, RUN = M / 32, S = M / 8;
    const int tid = fresh_tid(), lane = tid & 63, sg = tid >> 6;
    const int i0 = sg * RUN + lane * C;                 // LDS index of the lane's first pair
    const int n0 = sg * S + g.h * RUN + lane * C;       // its place in the series
    const int o = 4 * sg + g.h;                         // its run
    const double es = in.e_scale, dt = in.dt_o;
    const bool kerr = (in.kerr == LH_KERR_FIELD), plasma = in.plasma;
    double a[QR];
    if (plasma) {
        const double pp1 = in.preion_p1, er = in.e_ratio, ip = in.ionpot;
        double jf[QR];
        int bad = 0, cnt = 0;
        unsigned mask = 0;
#pragma unroll
        for (int c = 0; c < C; c++) {
            const double2 v = sm.buf[pad(i0 + c)];
            jf[2 * c] = fabs(v.x * es);
            jf[2 * c + 1] = fabs(v.y * es);
        }
        // samples inside the table's range get a rate; above it (or NaN) raise the flag
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
        if (bad) sm.flag = bad;
        double ntot;
        const int off = (int)block_exscan1((double)cnt, sm.scan, &ntot);
        const int total = (int)ntot;
        if (total == 0) {
#pragma unroll
            for (int q = 0; q < QR; q++) a[q] = 0.0;
        } else if (total <= SM::PCAP) {
            // the few hundred samples under the pulse belong to a few lanes:
            // compacted, they are one or two per thread of the member
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
            constexpr int QC = (QR < 4) ? QR : 4;
            int unused = 0;
#pragma unroll
            for (int c = 0; c < QR; c += QC) ppt_rates<QC>(in, jf + c, a + c, unused);
        }
#pragma unroll
        for (int q = 0; q < QR; q++) jf[q] = a[q];  // rate, kept for the loss term
        // a = F = ∫rate
        {
            double* rec = gl(g.rnext());
            double prev = dpp_f64<DPP_WAVE_SHR1>(a[QR - 1]);
            if (lane == 0) rec[8 * o + 1] = a[0];
            if (lane == 63) rec[8 * o + 2] = a[QR - 1];
            double acc = 0.0;
#pragma unroll
            for (int q = 0; q < QR; q++) {
                const double cur = a[q];
                if (q > 0 || lane > 0) acc += (0.5 * (prev + cur)) * dt;
                prev = cur;
                a[q] = acc;
            }
            const double x = wave_incl_scan(acc);
            const double ex = dpp_f64<DPP_WAVE_SHR1>(x);
            if (lane == 63) rec[8 * o] = x;
            gang_sync(g, sm);
            double W = 0.0, c = 0.0;
            if (lane < 32) {
                W = lg_ld(rec + 8 * lane);
                c = W;
                if (lane > 0) c = (0.5 * (lg_ld(rec + 8 * lane - 6) + lg_ld(rec + 8 * lane + 1))) * dt + W;
            }
            c = lanes32_incl_scan(c);
            const double base = (lane_value(c, o) - lane_value(W, o)) + ex;
#pragma unroll
            for (int q = 0; q < QR; q++) a[q] = base + a[q];
        }
        double Fprev = 0.0, fprev = pp1 - 1.0;  // exp(-0) = 1
#pragma unroll
        for (int q = 0; q < QR; q++) {
            const double2 v = sm.buf[pad(i0 + (q >> 1))];
            const double E = ((q & 1) ? v.y : v.x) * es;
            const double F = a[q];
            const double f = (F == Fprev) ? fprev : pp1 - exp(-F);  // F is flat outside the pulse
            Fprev = F;
            fprev = f;
            const double rate = jf[q];
            a[q] = (f * er) * E;                                                     // phase
            jf[q] = (rate != 0.0 && E != 0.0) ? ((ip * rate) * (1 - f)) / E : 0.0;  // loss current
        }
        // a = P = ∫(J + loss), J = ∫(phase term); runs compose as in Run2
        {
            double* rec = gl(g.rnext());
            double aprev = dpp_f64<DPP_WAVE_SHR1>(a[QR - 1]), pprev = dpp_f64<DPP_WAVE_SHR1>(jf[QR - 1]);
            if (lane == 0) {
                rec[8 * o + 2] = a[0];
                rec[8 * o + 3] = jf[0];
            }
            if (lane == 63) {
                rec[8 * o + 4] = a[QR - 1];
                rec[8 * o + 5] = jf[QR - 1];
            }
            const bool joined = lane > 0;
            double sj = 0.0, sp = 0.0;
#pragma unroll
            for (int q = 0; q < QR; q++) {
                const double cur = a[q];
                if (q > 0 || joined) {
                    sj += (0.5 * (aprev + cur)) * dt;
                    const double pc = sj + jf[q];
                    sp += (0.5 * (pprev + pc)) * dt;
                    pprev = pc;
                } else {
                    pprev = jf[q];
                }
                aprev = cur;
                a[q] = sp;
            }
            Run2 x{QR - (joined ? 0 : 1), sj, sp};
            x = run2_cat(dpp_run2<DPP_ROW_SHR1>(x), x, dt);
            x = run2_cat(dpp_run2<DPP_ROW_SHR2>(x), x, dt);
            x = run2_cat(dpp_run2<DPP_ROW_SHR4>(x), x, dt);
            x = run2_cat(dpp_run2<DPP_ROW_SHR8>(x), x, dt);
            x = run2_cat(dpp_run2<DPP_ROW_BCAST15, 0xa>(x), x, dt);
            x = run2_cat(dpp_run2<DPP_ROW_BCAST31, 0xc>(x), x, dt);
            const Run2 ex = dpp_run2<DPP_WAVE_SHR1>(x);
            if (lane == 63) {
                rec[8 * o] = x.sj;
                rec[8 * o + 1] = x.sp;
            }
            gang_sync(g, sm);
            Run2 e{0, 0.0, 0.0}, jn{0, 0.0, 0.0};
            if (lane < 32) {
                const double* r = rec + 8 * lane;
                if (lane > 0) {
                    const double ta = (0.5 * (lg_ld(r - 4) + lg_ld(r + 2))) * dt;
                    const double sp1 = (0.5 * (lg_ld(r - 3) + (ta + lg_ld(r + 3)))) * dt;
                    jn = Run2{1, ta, sp1};
                }
                e = run2_cat(jn, Run2{2 * RUN - 1, lg_ld(r), lg_ld(r + 1)}, dt);
            }
            Run2 c = e;
            c = run2_cat(dpp_run2<DPP_ROW_SHR1>(c), c, dt);
            c = run2_cat(dpp_run2<DPP_ROW_SHR2>(c), c, dt);
            c = run2_cat(dpp_run2<DPP_ROW_SHR4>(c), c, dt);
            c = run2_cat(dpp_run2<DPP_ROW_SHR8>(c), c, dt);
            c = run2_cat(dpp_run2<DPP_ROW_BCAST15, 0xa>(c), c, dt);
            const Run2 win = run2_cat(dpp_run2<DPP_WAVE_SHR1>(c), jn, dt);  // the runs before run `lane`, and the join
            const Run2 w_in{__builtin_amdgcn_readlane(win.n, __builtin_amdgcn_readfirstlane(o)), lane_value(win.sj, o),
                            lane_value(win.sp, o)};
            const Run2 t_in = run2_cat(w_in, ex, dt);
            const double J = t_in.sj, P = t_in.sp;
#pragma unroll
            for (int q = 0; q < QR; q++) a[q] = (P + ((double)(q + (joined ? 1 : 0)) * dt) * J) + a[q];
        }
    }
    const double* tw = gl(in.to_win);
#pragma unroll
    for (int c = 0; c < C; c++) {
        const double2 v = sm.buf[pad(i0 + c)];
        const double E0 = v.x * es, E1 = v.y * es;
        double p0 = kerr ? kfac * (E0 * E0 * E0) : 0.0;
        double p1 = kerr ? kfac * (E1 * E1 * E1) : 0.0;
        if (plasma) {
            p0 = p0 + rho * a[2 * c];
            p1 = p1 + rho * a[2 * c + 1];
        }
        if constexpr (RAMAN) {  // RamanPolarField: Pout = ρ·E·P (src/Nonlinear.jl:323-325)
            const double2 pr = gl(praman)[i0 + c];
            p0 = p0 + (rho * E0) * pr.x;
            p1 = p1 + (rho * E1) * pr.y;
        }
        const int n = 2 * (n0 + c);
        sm.buf[pad(i0 + c)] = make_double2(p0 * tw[n], p1 * tw[n + 1]);
    }
}

// The convolution step of a zero-padded Raman transform (2·L reals packed into
// L points, bins of the member in LDS): r2c post-step, ×hω·δt, c2r pre-pack,
// pairwise (k, L − k) in place.  hw(s, q) gives hω·δt at k = res(h, s) + 8q,
// hw(0, S) at k = L.  Starts and ends synchronised.
template <int L, class SM, class HW>
__device__ __forceinline__ void g_raman_spectrum(SM& sm, const Gang& g, HW hw) {
    constexpr int S = L / 8;
    const int npair = (g.h != 0) ? S : S / 2 + 1 + S / 2;
    for (int i = fresh_tid(); i < npair; i += LH_T) {
        // members 1..3: (slot 0, q) with (slot 1, S−1−q); member 0: slot 0's
        // q = 0 (alone, with k = L), 1..S/2 with S − q, slot 1's q < S/2 with S−1−q
        const int s = (g.h == 0 && i > S / 2) ? 1 : 0;
        const int q = s ? i - (S / 2 + 1) : i;
        const int ik = s * S + q, im = GGeo<L>::conj_idx(g.h, s, q);
        const int k = GGeo<L>::res(g.h, s) + 8 * q;
        const double2 Zk = sm.buf[pad(ik)], Zm = sm.buf[pad(im)];
        if (k == 0) {
            // X[0] = Re + Im, X[L] = Re − Im
            double2 Y0 = cscal(Zk.x + Zk.y, hw(0, 0)), YL = cscal(Zk.x - Zk.y, hw(0, S));
            Y0.y = 0.0;
            YL.y = 0.0;
            const double2 A = cadd(Y0, cconj(YL)), B = csub(Y0, cconj(YL));
            sm.buf[pad(0)] = cadd(A, cmul_pi(B));
            continue;
        }
        const double2 w = gtw<2 * L>(sm.tw, k);       // exp(-iπk/L)
        const double2 wm = make_double2(-w.x, w.y);   // exp(-iπ(L−k)/L) = −conj(w)
        auto post = [](double2 z, double2 zc, double2 w_) {  // r2c: E + w·O
            const double2 c = cconj(zc);
            const double2 E = cscal(0.5, cadd(z, c)), d = csub(z, c);
            return cadd(E, cmul(w_, make_double2(0.5 * d.y, -(0.5 * d.x))));
        };
        const int sm_ = (im >= S) ? 1 : 0, qm = im - sm_ * S;
        const double2 Yk = cmul(hw(s, q), post(Zk, Zm, w));
        const double2 Ym = (ik == im) ? Yk : cmul(hw(sm_, qm), post(Zm, Zk, wm));
        const double2 Ak = cadd(Yk, cconj(Ym)), Bk = cmul(csub(Yk, cconj(Ym)), cconj(w));
        sm.buf[pad(ik)] = cadd(Ak, cmul_pi(Bk));
        if (ik != im) {
            const double2 Am = cadd(Ym, cconj(Yk)), Bm = cmul(csub(Ym, cconj(Yk)), cconj(wm));
            sm.buf[pad(im)] = cadd(Am, cmul_pi(Bm));
        }
    }
    __syncthreads();
}

// Field-grid transform: the bins' c2r pre-pack is in LDS (synchronised); ends
// with the forward transform's bins in LDS (synchronised), to be post-stepped by
// g_r2c.  Series of Nto = 2·M reals.
template <int M, bool RAMAN, class SM>
__device__ __forceinline__ void g_rhs_field(const DInst& in, SM& sm, Gang& g, double rho, double kfac) {
    constexpr int S = M / 8, RUN = M / 32;
    double2* x = g.xnext();
    g_local_inv<M>(sm, g, x);
    gang_sync(g, sm);
    const int u = fresh_tid();
    const int n0 = g.h * RUN + u;
    double2* praman = nullptr;
    {
        double2 v[8];
        if (u < RUN) g_join_inv<M>(sm, x, n0, v);
        if constexpr (RAMAN) {
            // RamanPolarField with third-harmonic terms (src/Nonlinear.jl:183-247,
            // 284-333): E² over the zero-padded 2·Nto reals is a transform of 2·M
            // points; pair j of the series is point j, its upper half zero.  The
            // thread's pairs n0 + S·n1 are times n0 and n0 + S (mod 2S).
            constexpr int M2 = 2 * M;
            double2* E = gl(in.escr) + (size_t)g.h * (M / 4);
            praman = gl(in.escr) + M + (size_t)g.h * (M / 4);
            double2* x2 = g.xnext();
            if (u < RUN) {
                const double es = in.e_scale;
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    double2 t[8];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const double2 z = v[2 * j + b];
                        const double e0 = z.x * es, e1 = z.y * es;
                        t[j] = make_double2(e0 * e0, e1 * e1);
                        t[j + 4] = make_double2(0.0, 0.0);
                        E[(2 * j + b) * RUN + u] = z;
                    }
                    g_join_fwd<M2>(sm, x2, n0 + S * b, t);
                }
            }
            gang_sync(g, sm);
            g_local_fwd<M2>(sm, g, x2);
            {
                const double2* hw = gl(in.hwdt);
                const int h = g.h;
                g_raman_spectrum<M2>(sm, g, [hw, h](int s, int q) { return hw[GGeo<M2>::res(h, s) + 8 * q]; });
            }
            x2 = g.xnext();
            g_local_inv<M2>(sm, g, x2);
            gang_sync(g, sm);
            if (u < RUN) {
                const double inv2n = in.inv_2n;
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    double2 t[8];
                    g_join_inv<M2>(sm, x2, n0 + S * b, t);
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        praman[(2 * j + b) * RUN + u] = make_double2(t[j].x * inv2n, t[j].y * inv2n);
                }
#pragma unroll
                for (int n1 = 0; n1 < 8; n1++) v[n1] = E[n1 * RUN + u];
            }
        }
        if (u < RUN) {
#pragma unroll
            for (int n1 = 0; n1 < 8; n1++) sm.buf[pad(n1 * RUN + u)] = v[n1];
        }
    }
    __syncthreads();
    g_pointwise<M, RAMAN>(in, sm, g, rho, kfac, praman);
    __syncthreads();
    x = g.xnext();
    const int u2 = fresh_tid();
    if (u2 < RUN) {
        double2 v[8];
#pragma unroll
        for (int n1 = 0; n1 < 8; n1++) v[n1] = sm.buf[pad(n1 * RUN + u2)];
        g_join_fwd<M>(sm, x, g.h * RUN + u2, v);
    }
    gang_sync(g, sm);
    g_local_fwd<M>(sm, g, x);
}

// r2c post-step of bin k = res(h, s) + 8q of a series of 2·M reals whose
// transform's bins are in LDS.
template <int M, class SM>
__device__ __forceinline__ double2 g_r2c(const SM& sm, const Gang& g, int s, int q) {
    constexpr int S = M / 8;
    const int k = GGeo<M>::res(g.h, s) + 8 * q;
    const double2 zk = sm.buf[pad(s * S + q)];
    const double2 zc = cconj(sm.buf[pad(GGeo<M>::conj_idx(g.h, s, q))]);
    const double2 E = cscal(0.5, cadd(zk, zc)), d = csub(zk, zc);
    const double2 O = make_double2(0.5 * d.y, -(0.5 * d.x));
    return cadd(E, cmul(gtw<2 * M>(sm.tw, k), O));
}

// Envelope-grid transform of M points (Kerr_env, RamanPolarEnv; src/Nonlinear.jl:
// 47-73, 282-333): the bins are in LDS (synchronised); ends with the forward
// transform's bins in LDS (synchronised).  The pointwise work happens on the
// eight times a thread holds after the join.
template <int M, class SM, class HW>
__device__ __forceinline__ void g_rhs_env(const DInst& in, SM& sm, Gang& g, HW hw) {
    constexpr int S = M / 8, RUN = M / 32;
    double2* x = g.xnext();
    g_local_inv<M>(sm, g, x);
    gang_sync(g, sm);
    const int u = fresh_tid();
    const int n0 = g.h * RUN + u;
    const double es = in.e_scale;
    double2 v[8];
    if (u < RUN) {
        g_join_inv<M>(sm, x, n0, v);
#pragma unroll
        for (int n1 = 0; n1 < 8; n1++) v[n1] = cscal(es, v[n1]);
    }
    double P[8];
    const bool raman = in.raman;
    if (raman) {
        // ½|E|² as reals packed in pairs (2j, 2j+1) over the zero-padded 2·M
        // grid: pair j of lanes 2i, 2i+1 is time j0 = n0/2 + (S/2)·(n1 & 1),
        // j1 = n1/2.  The even lane takes the even n1, the odd lane the odd ones.
        const int b = u & 1, j0 = (n0 >> 1) + (S / 2) * b;
        double2* x2 = g.xnext();
        if (u < RUN) {
            double a[8];
#pragma unroll
            for (int n1 = 0; n1 < 8; n1++) a[n1] = 0.5 * (v[n1].x * v[n1].x + v[n1].y * v[n1].y);
            double2 t[8];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const double own = b ? a[2 * j + 1] : a[2 * j], give = b ? a[2 * j] : a[2 * j + 1];
                const double got = dpp_f64<0xB1>(give);  // lanes 2i and 2i+1 swap
                t[j] = b ? make_double2(got, own) : make_double2(own, got);
                t[j + 4] = make_double2(0.0, 0.0);
            }
            g_join_fwd<M>(sm, x2, j0, t);
        }
        gang_sync(g, sm);
        g_local_fwd<M>(sm, g, x2);
        g_raman_spectrum<M>(sm, g, hw);
        x2 = g.xnext();
        g_local_inv<M>(sm, g, x2);
        gang_sync(g, sm);
        if (u < RUN) {
            double2 t[8];
            g_join_inv<M>(sm, x2, j0, t);
            const double inv2n = in.inv_2n;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const double own = b ? t[j].y : t[j].x, give = b ? t[j].x : t[j].y;
                const double got = dpp_f64<0xB1>(give);
                P[2 * j] = (b ? got : own) * inv2n;
                P[2 * j + 1] = (b ? own : got) * inv2n;
            }
        }
    }
    x = g.xnext();
    if (u < RUN) {
        const double rho = in.density, k34 = in.kerr34;
        const bool kerr = (in.kerr == LH_KERR_ENV);
        const double* tw = gl(in.to_win);
#pragma unroll
        for (int n1 = 0; n1 < 8; n1++) {
            const double2 e = v[n1];
            double2 p = make_double2(0.0, 0.0);
            if (kerr) p = cscal(k34 * (e.x * e.x + e.y * e.y), e);
            if (raman) p = cadd(p, make_double2((rho * e.x) * P[n1], (rho * e.y) * P[n1]));
            v[n1] = cscal(tw[n0 + S * n1], p);
        }
        g_join_fwd<M>(sm, x, n0, v);
    }
    gang_sync(g, sm);
    g_local_fwd<M>(sm, g, x);
}

// c2r pre-pack of one bin of a spectrum that is zero above M/2 (see
// c2r_pack_bin) into the member's LDS bins.
template <int M, class SM>
__device__ __forceinline__ void g_pack_bin(SM& sm, const Gang& g, int s, int q, double2 Xk) {
    constexpr int S = M / 8;
    const int k = GGeo<M>::res(g.h, s) + 8 * q;
    if (k == 0) {
        sm.buf[pad(0)] = make_double2(Xk.x, Xk.x);
        return;
    }
    const double2 w = gtw<2 * M>(sm.tw, k);
    if (k == M / 2) {
        const double2 A = cadd(Xk, cconj(Xk)), B = cmul(csub(Xk, cconj(Xk)), cconj(w));
        sm.buf[pad(s * S + q)] = cadd(A, cmul_pi(B));
        return;
    }
    const double2 wm = make_double2(-w.x, w.y);
    sm.buf[pad(s * S + q)] = cadd(Xk, cmul_pi(cmul(Xk, cconj(w))));
    const double2 Xc = cconj(Xk);
    sm.buf[pad(GGeo<M>::conj_idx(g.h, s, q))] = csub(Xc, cmul_pi(cmul(Xc, cconj(wm))));
}

// Sizes of a gang's member.  KIND 0: field grid, Nto = 2·M, state bins 0..M/2;
// KIND 1: envelope grid of M points.
template <int KIND, int M>
struct GSizes {
    static constexpr int S = M / 8;
    static constexpr int NB = (KIND == 0) ? S : 2 * S;        // bins of a member (member 0 of a field grid: one more)
    static constexpr int NMAX = (KIND == 0) ? NB + 1 : NB;
    static constexpr int GSTR = NB + 8;                       // elements of a member's part of a vector
    static constexpr int MC = (KIND == 0) ? M / 2 : M;        // filter transform
    static constexpr int N = (KIND == 0) ? M / 2 + 1 : M;     // state bins
    static constexpr int NPT = (NMAX + LH_T - 1) / LH_T;      // bins per thread
    // of them in one round of loads (as many as the registers hold: envelope grids
    // of 16384 points with four instead of two 12.15 → 11.84 ms for 0.15 m)
    static constexpr int CB = NPT <= 4 ? NPT : (KIND == 0) ? 3 : 4;
    static constexpr int CBD = NPT >= 2 ? 2 : 1;              // in a dense kernel (half the registers)
    __device__ static __forceinline__ int count(int h) { return (KIND == 0 && h == 0) ? NB + 1 : NB; }
    // local bin p → (slot, q); k = res + 8q.  Field grids: p < S/2 is slot 0,
    // p < S slot 1, p = S (member 0) bin M/2.
    __device__ static __forceinline__ void bin(int p, int& s, int& q) {
        constexpr int H = (KIND == 0) ? S / 2 : S;
        s = (p >= H && p < 2 * H) ? 1 : 0;
        q = s ? p - H : (p >= H ? p - H : p);
        if (KIND == 0 && p == S) q = S / 2;
    }
    __device__ static __forceinline__ int k_of(int h, int p) {
        int s, q;
        bin(p, s, q);
        return GGeo<M>::res(h, s) + 8 * q;
    }
};

// Whether a wavefront has any bin at or after chunk start c (bins c·LH_T + its
// threads): chunks beyond the member's bins cost their wavefronts nothing.
__device__ __forceinline__ bool lg_none(int tid, int c, int nb) {
    return __builtin_amdgcn_readfirstlane(tid & ~63) + c * LH_T >= nb;
}

// z-dependent fill (see zg_refresh): ρ(z), β1(z) and the taper's radius by the
// first wavefront (one stencil point per lane), then the member's bins of the
// operator and the output factor.
template <int KIND, int M, class SM>
__device__ __forceinline__ void g_zg_refresh(const DInst& in, SM& sm, int h, double2* Lg, double2* OFg, double z,
                                             double& rho, double& kfac) {
    using Z = GSizes<KIND, M>;
    const int tid = fresh_tid();
    if (tid < 64) zg_constants(in, sm.zs, z);
    __syncthreads();
    rho = sm.zs[0];
    const double b1 = sm.zs[1], a = sm.zs[2];
    const double sqrt_aeff = in.ztaper ? a * in.zsqrt_intg : in.zsqrt_aeff;  // Aeff(z) = a(z)²·aeff_intg
    kfac = rho * LH_EPS0 * in.kerr_gamma3;
    const int nb = Z::count(h);
    for (int p = tid; p < nb; p += LH_T) {
        const int k = Z::k_of(h, p);
        double2 L = make_double2(0.0, 0.0), of = make_double2(in.sc_f, 0.0);
        if (gl(in.zsidx)[k]) {
            const double w = gl(in.st_omega)[k];
            const double sc = sqrt(1 + gl(in.zgam)[k] * rho);  // coren(ω; z)^2
            const double2 nw = in.ztaper ? zg_nwg_taper(in, gl(in.zU)[k], gl(in.zV)[k], a)
                                         : static_cast<const double2*>(gl(in.znwg))[k];
            const double2 n = zg_neff(in, sc * sc, nw);
            const double ncr = (n.x < 1e-3) ? 1e-3 : n.x;  // conj_clamp
            const double lim = 3000 * LH_CLIGHT / w;
            const double nci = -((n.y < 0.0) ? 0.0 : (n.y > lim ? lim : n.y));
            const double wc = w / LH_CLIGHT;
            const double zr = wc * ncr - w * b1, zi = wc * nci;
            L = make_double2(zi, -zr);
            const double beta = wc * n.x;
            const double2 pre = gl(in.zpre)[k];
            const double nfx = pre.x / beta * sqrt_aeff, nfy = pre.y / beta * sqrt_aeff;
            of = make_double2((in.sc_f * nfx) * gl(in.omega_win)[k], (in.sc_f * nfy) * gl(in.omega_win)[k]);
        }
        gl(Lg)[p] = L;
        gl(OFg)[p] = of;
    }
    __syncthreads();
}

// One statistics record (see step_stats in the reference order of operations,
// Stats.jl:454-532): the analytic spectrum of M points is in LDS (not yet
// synchronised), each thread holds its partial sums.  Four barriers of the
// gang; member 0 writes the record.
template <int KIND, int M, class SM>
__device__ __forceinline__ void g_stats(const DInst& in, SM& sm, Gang& g, double s0, double s1, double se,
                                        const WinSums& ws, double z, double dz, double rho, double* rec) {
    constexpr int S = M / 8, RUN = M / 32, NT = M;
    const int tid = fresh_tid(), lane = tid & 63, wid = tid >> 6;
    double st_aeff = in.st_aeff, st_ediv = in.st_ediv;
    if (KIND == 0 && in.zg_np > 0 && in.ztaper) {  // Aeff at this record's z, from the last refresh
        const double sa = sm.zs[2] * in.zsqrt_intg;
        st_aeff = sa * sa;
        st_ediv = sqrt(LH_EPS0 * LH_CLIGHT * st_aeff / 2);
    }
    const double* r1;
    {
        block_sum3(s0, s1, se, sm.wsum);  // ends synchronised: the spectrum is complete
        double w0 = ws.s[0], w1 = ws.s[1], w2 = ws.s[2], w3 = ws.s[3];
        if (in.st_nwin > 0) block_sum4(w0, w1, w2, w3, sm.wsum);
        double* r = gl(g.rnext());
        if (tid == 0) {
            double* q = r + 8 * g.h;
            q[0] = s0, q[1] = s1, q[2] = se, q[3] = w0, q[4] = w1, q[5] = w2, q[6] = w3;
        }
        r1 = r;
    }
    double2* x = g.xnext();
    g_local_inv<M>(sm, g, x);
    gang_sync(g, sm);
    double sums[7];
    if (g.h == 0 && tid == 0) {
#pragma unroll
        for (int i = 0; i < 7; i++) {
            sums[i] = lg_ld(r1 + i);
            for (int m = 1; m < LG_G; m++) sums[i] += lg_ld(r1 + 8 * m + i);
        }
    }
    // pass 1: P = |Et|² at the thread's eight times, PPT rate of |Re Et|
    const double inv = 1.0 / (double)NT;  // FFTW's ifft normalisation
    const bool ion = (KIND == 0) && in.plasma;
    const int n0 = g.h * RUN + tid;
    double p[8];
    double pmax = -1.0, rmax = 0.0, rsum = 0.0, edge = 0.0;
    int imax = NT, bad = LH_OK;
    if (tid < RUN) {
        double2 v[8];
        g_join_inv<M>(sm, x, n0, v);
#pragma unroll
        for (int n1 = 0; n1 < 8; n1++) {
            const double re = v[n1].x * inv, im = v[n1].y * inv;
            p[n1] = re * re + im * im;
            v[n1].x = fabs(re / st_ediv);
            gl(g.P)[n0 + S * n1] = p[n1];
            if (p[n1] > pmax) {  // n increases with n1: the first maximum is kept
                pmax = p[n1];
                imax = n0 + S * n1;
            }
        }
        if (ion) {
#pragma unroll 1
            for (int c = 0; c < 8; c += 2) {
                double aE[2], r[2];
                aE[0] = c == 0 ? v[0].x : c == 2 ? v[2].x : c == 4 ? v[4].x : v[6].x;
                aE[1] = c == 0 ? v[1].x : c == 2 ? v[3].x : c == 4 ? v[5].x : v[7].x;
                if (!(aE[0] < in.ppt_emin) || !(aE[1] < in.ppt_emin)) {
                    ppt_rates<2>(in, aE, r, bad);
                    rmax = fmax(rmax, fmax(r[0], r[1]));
                    rsum += r[0];
                    rsum += r[1];
                    if (c == 0 && n0 == 0) edge = r[0];                // sample 0
                    if (c == 6 && n0 == S - 1) edge = r[1];           // sample NT − 1
                }
            }
        }
    }
    rsum -= 0.5 * edge;
    if (bad != LH_OK) sm.flag = bad;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double p2 = __shfl_xor(pmax, off, 64);
        const int i2 = __shfl_xor(imax, off, 64);
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
    __syncthreads();
    double* r2 = gl(g.rnext());
    if (tid == 0) {
        for (int w = 1; w < LH_NW; w++) {
            const double p2 = sm.wsum[4 * w];
            const int i2 = (int)sm.wsum[4 * w + 1];
            if (p2 > pmax || (p2 == pmax && i2 < imax)) {
                pmax = p2;
                imax = i2;
            }
            rmax = fmax(rmax, sm.wsum[4 * w + 2]);
            rsum += sm.wsum[4 * w + 3];
        }
        double* q = r2 + 8 * g.h;
        q[0] = pmax, q[1] = (double)imax, q[2] = rmax, q[3] = rsum;
    }
    gang_sync(g, sm);
    pmax = lg_ld(r2);
    imax = (int)lg_ld(r2 + 1);
    rmax = lg_ld(r2 + 2);
    rsum = lg_ld(r2 + 3);
    for (int m = 1; m < LG_G; m++) {
        const double p2 = lg_ld(r2 + 8 * m);
        const int i2 = (int)lg_ld(r2 + 8 * m + 1);
        if (p2 > pmax || (p2 == pmax && i2 < imax)) {
            pmax = p2;
            imax = i2;
        }
        rmax = fmax(rmax, lg_ld(r2 + 8 * m + 2));
        rsum += lg_ld(r2 + 8 * m + 3);
    }
    // pass 2: level crossings around the maximum at half of it: :min takes the
    // last j < imax with P < val and the first j > imax with P < val; :max the
    // first j < imax with P > val and the last j > imax with P > val
    const double val = 0.5 * pmax;
    int aL = -1, aR = NT, bL = NT, bR = -1;
    if (tid < RUN) {
#pragma unroll
        for (int n1 = 0; n1 < 8; n1++) {
            const int j = n0 + S * n1;
            if (j < imax) {
                if (p[n1] < val) aL = max(aL, j);
                if (p[n1] > val) bL = min(bL, j);
            } else if (j > imax) {
                if (p[n1] < val) aR = min(aR, j);
                if (p[n1] > val) bR = max(bR, j);
            }
        }
    }
    wave_minmax(aR, aL);
    wave_minmax(bL, bR);
    if (lane == 0) {
        sm.wsum[4 * wid + 0] = (double)aL;
        sm.wsum[4 * wid + 1] = (double)aR;
        sm.wsum[4 * wid + 2] = (double)bL;
        sm.wsum[4 * wid + 3] = (double)bR;
    }
    __syncthreads();
    double* r3 = gl(g.rnext());
    if (tid == 0) {
        for (int w = 1; w < LH_NW; w++) {
            aL = max(aL, (int)sm.wsum[4 * w + 0]);
            aR = min(aR, (int)sm.wsum[4 * w + 1]);
            bL = min(bL, (int)sm.wsum[4 * w + 2]);
            bR = max(bR, (int)sm.wsum[4 * w + 3]);
        }
        double* q = r3 + 8 * g.h;
        q[0] = (double)aL, q[1] = (double)aR, q[2] = (double)bL, q[3] = (double)bR;
    }
    gang_sync(g, sm);
    if (g.h == 0 && tid == 0) {
        for (int m = 1; m < LG_G; m++) {
            aL = max(aL, (int)lg_ld(r3 + 8 * m));
            aR = min(aR, (int)lg_ld(r3 + 8 * m + 1));
            bL = min(bL, (int)lg_ld(r3 + 8 * m + 2));
            bR = max(bR, (int)lg_ld(r3 + 8 * m + 3));
        }
        const double* t = gl(in.st_t);
        const double* Pg = gl(g.P);
        const double nan = __longlong_as_double(0x7ff8000000000000LL);
        // a missing crossing or a neighbour off the grid is the reference's
        // caught exception: NaN
        double fmin_ = nan, fmax_ = nan;
        if (imax < NT && aL >= 0 && aR < NT) {
            const double left = linterpx(t[aL], t[aL + 1], lg_ld(Pg + aL), lg_ld(Pg + aL + 1), val);
            const double right = linterpx(t[aR - 1], t[aR], lg_ld(Pg + aR - 1), lg_ld(Pg + aR), val);
            fmin_ = fabs(right - left);
        }
        if (imax < NT && bL >= 1 && bL < NT && bR >= 0 && bR + 1 < NT) {
            const double left = linterpx(t[bL - 1], t[bL], lg_ld(Pg + bL - 1), lg_ld(Pg + bL), val);
            const double right = linterpx(t[bR], t[bR + 1], lg_ld(Pg + bR), lg_ld(Pg + bR + 1), val);
            fmax_ = fabs(right - left);
        }
        double ed = nan, pr = nan;
        if (ion) {
            // cumtrapz!(out, δt) end value: Σ ½(r_{j-1} + r_j)·δt
            const double dt = t[1] - t[0];
            ed = (1.0 - exp(-(rsum * dt))) * rho;
            pr = rmax;
        }
        rec[LH_STAT_Z] = z;
        rec[LH_STAT_DZ] = dz;
        rec[LH_STAT_OMEGA0] = sums[1] / sums[0];
        rec[LH_STAT_ENERGY] = sums[2];
        rec[LH_STAT_PEAKPOWER] = pmax;
        rec[LH_STAT_PEAKINTENSITY] = pmax / st_aeff;
        rec[LH_STAT_FWHM_T_MIN] = fmin_;
        rec[LH_STAT_FWHM_T_MAX] = fmax_;
        rec[LH_STAT_ELECTRONDENSITY] = ed;
        rec[LH_STAT_PEAK_IONISATION_RATE] = pr;
        rec[LH_STAT_DENSITY] = rho;
#pragma unroll
        for (int q = 0; q < LH_STAT_MAX_WINDOWS; q++) rec[LH_STAT_WINDOW0 + q] = (q < in.st_nwin) ? sums[3 + q] : nan;
    }
    __syncthreads();
}

// Accepted-step window filter (stepfun, src/Luna.jl:366-370): YN ← FT(twin ·
// FT⁻¹(ωwin · YN·exp(L dz))) on the member's bins, E = exp(L dz); between the
// transforms each thread holds eight times.  With a record due, its statistics
// follow from the filtered bins.
template <int KIND, int M, bool STATS, class SM>
__device__ __forceinline__ void g_stepfun(const DInst& in, SM& sm, Gang& g, const double2* E, double2* YN, double* rec,
                                          double z, double dz, double rho) {
    using Z = GSizes<KIND, M>;
    constexpr int MC = Z::MC, SC = MC / 8, RUNC = MC / 32;
    const int nb = Z::count(g.h);
    for (int p = fresh_tid(); p < nb; p += LH_T) {
        const double2 v = cmul(gl(YN)[p], static_cast<const double2*>(gl(E))[p]);
        sm.buf[pad(p)] = cscal(gl(in.omega_win)[Z::k_of(g.h, p)], v);
    }
    __syncthreads();
    if constexpr (KIND == 0) {
        // c2r pre-pack in place, pairs (k, MC − k); bin MC sits at index 2·SC
        const int npair = (g.h != 0) ? SC : SC + 1;
        for (int i = fresh_tid(); i < npair; i += LH_T) {
            const int s = (g.h == 0 && i > SC / 2) ? 1 : 0;
            const int q = s ? i - (SC / 2 + 1) : i;
            const int ik = s * SC + q;
            const int k = GGeo<MC>::res(g.h, s) + 8 * q;
            if (k == 0) {
                const double a = sm.buf[pad(0)].x, b = sm.buf[pad(2 * SC)].x;
                sm.buf[pad(0)] = make_double2(a + b, a - b);
                continue;
            }
            const int im = GGeo<MC>::conj_idx(g.h, s, q);
            const double2 Xk = sm.buf[pad(ik)], Xm = sm.buf[pad(im)];
            const double2 w = gtw<2 * MC>(sm.tw, k), wm = make_double2(-w.x, w.y);
            const double2 Ak = cadd(Xk, cconj(Xm)), Bk = cmul(csub(Xk, cconj(Xm)), cconj(w));
            sm.buf[pad(ik)] = cadd(Ak, cmul_pi(Bk));
            if (ik != im) {
                const double2 Am = cadd(Xm, cconj(Xk)), Bm = cmul(csub(Xm, cconj(Xk)), cconj(wm));
                sm.buf[pad(im)] = cadd(Am, cmul_pi(Bm));
            }
        }
        __syncthreads();
    }
    double2* x = g.xnext();
    g_local_inv<MC>(sm, g, x);
    gang_sync(g, sm);
    double2* x2 = g.xnext();
    const int u = fresh_tid();
    if (u < RUNC) {
        const int n0 = g.h * RUNC + u;
        double2 v[8];
        g_join_inv<MC>(sm, x, n0, v);
        const double inv_nt = in.inv_nt;
#pragma unroll
        for (int n1 = 0; n1 < 8; n1++) {
            const int n = n0 + SC * n1;
            if constexpr (KIND == 0) {
                v[n1].x = (inv_nt * v[n1].x) * gl(in.t_win)[2 * n];
                v[n1].y = (inv_nt * v[n1].y) * gl(in.t_win)[2 * n + 1];
            } else {
                const double w = gl(in.t_win)[n];
                v[n1] = make_double2((inv_nt * v[n1].x) * w, (inv_nt * v[n1].y) * w);
            }
        }
        g_join_fwd<MC>(sm, x2, n0, v);
    }
    gang_sync(g, sm);
    g_local_fwd<MC>(sm, g, x2);
    constexpr int NPT = Z::NPT;
    double2 yv[NPT];
    double s0 = 0.0, s1 = 0.0, se = 0.0;
    WinSums ws = {{0.0, 0.0, 0.0, 0.0}};
    const bool stat = STATS && rec != nullptr;
#pragma unroll
    for (int i = 0; i < NPT; i++) {
        const int p = fresh_tid() + i * LH_T;
        if (p < nb) {
            if constexpr (KIND == 0) {
                if (p == Z::NB) {  // bin MC: Re − Im of point 0
                    const double2 z0 = sm.buf[pad(0)];
                    yv[i] = make_double2(z0.x - z0.y, 0.0);
                } else {
                    const int s = (p >= SC) ? 1 : 0;
                    yv[i] = g_r2c<MC>(sm, g, s, p - s * SC);
                }
            } else {
                yv[i] = sm.buf[pad(p)];
            }
            gl(YN)[p] = yv[i];
            if (stat) {
                const int k = Z::k_of(g.h, p);
                const double a = yv[i].x * yv[i].x + yv[i].y * yv[i].y;
                s0 += a;
                s1 += gl(in.st_omega)[k] * a;
                se += gl(in.st_ew)[k] * a;
                win_add(in, ws, k, a);
            }
        }
    }
    __syncthreads();  // every bin read before the buffer is reused
    if (stat) {
        if constexpr (KIND == 0) {
            // analytic spectrum (copyto_fft!, src/Stats.jl:441-448): bins
            // 0..Nω−2 doubled, bin Nω−1 dropped, zero up to M
            constexpr int S = M / 8;
#pragma unroll
            for (int i = 0; i < NPT; i++) {
                const int p = fresh_tid() + i * LH_T;
                if (p < Z::NB) {
                    const int s = (p >= S / 2) ? 1 : 0, q = p - s * (S / 2);
                    sm.buf[pad(s * S + q)] = make_double2(2.0 * yv[i].x, 2.0 * yv[i].y);
                    sm.buf[pad(s * S + S / 2 + q)] = make_double2(0.0, 0.0);
                }
            }
        }
        g_stats<KIND, M>(in, sm, g, s0, s1, se, ws, z, dz, rho, rec);
    }
}

// The right-hand side of the bins in LDS, and its bin p (before the output factor).
template <int KIND, int M, bool RAMAN, class SM, class HW>
__device__ __forceinline__ void g_rhs(const DInst& in, SM& sm, Gang& g, double rho, double kfac, HW hw) {
    if constexpr (KIND == 0)
        g_rhs_field<M, RAMAN>(in, sm, g, rho, kfac);
    else
        g_rhs_env<M>(in, sm, g, hw);
}
template <int KIND, int M, class SM>
__device__ __forceinline__ double2 g_rhs_bin(const SM& sm, const Gang& g, int p) {
    if constexpr (KIND == 0) {
        int s, q;
        GSizes<KIND, M>::bin(p, s, q);
        return g_r2c<M>(sm, g, s, q);
    } else {
        return sm.buf[pad(p)];
    }
}

// Persistent adaptive solve of one instance by a gang (Luna.run →
// RK45.solve_precon).  Every member runs the same step control on the same
// numbers.
template <int KIND, int M, bool STREAM, bool RAMAN, bool DENSE, class SM>
__device__ __forceinline__ void g_solve(const DInst& in, SM& sm, Gang& g) {
    using Z = GSizes<KIND, M>;
    constexpr int N = Z::N, CB = DENSE ? Z::CBD : Z::CB, NC = (Z::NPT + CB - 1) / CB;
    const int h = g.h, nb = Z::count(h);
    KSet K{gl(in.K) + (size_t)h * Z::GSTR, in.kstride, 0, 6};
    double2* const Fv = K[LG_F];
    double2* const Ev = K[LG_E];
    double2* const Lg = K[LG_L];
    double2* const OFg = K[LG_OF];
    double2* Y = K[LG_YA];
    double2* YN = K[LG_YB];
    double2* const hwg = K[LG_HW];
    for (int p = fresh_tid(); p < nb; p += LH_T) {
        const int k = Z::k_of(h, p);
        Y[p] = gl(in.Yin)[k];
        Lg[p] = gl(in.linop)[k];
        OFg[p] = gl(in.outfac)[k];
        if (KIND == 1 && in.raman) hwg[p] = gl(in.hwdt)[k];
    }
    if (KIND == 1 && in.raman && h == 0 && threadIdx.x == 0) hwg[Z::NB] = gl(in.hwdt)[M];
    if (threadIdx.x == 0) sm.flag = sm.gflag = LH_OK;
    __syncthreads();
    auto hw = [hwg](int s, int q) { return static_cast<const double2*>(gl(hwg))[s * (M / 8) + q + (q == M / 8 ? M / 8 : 0)]; };

    long long steps = 0, accepted = 0, rejected = 0, rhs_evals = 0, npub = 0;
    int status = LH_OK, saved = in.save_first, repeated = 0;
    double t = in.z0, tn = in.z0, dt = in.init_dz, dtn = in.init_dz, errlast = 0.0;
    const double rho = in.density, kfac = in.kerr_fac;

    // stage −1 is PreconStepper's initial k1 = fbar(y0, t, t); the stages of a
    // step follow from the same code
    int st = -1;
    double h0 = 0.0;
    while (status == LH_OK && (st < 0 || tn <= in.zmax)) {
        if (st >= 0) {
            if (steps >= in.max_steps) {
                status = LH_E_MAXSTEPS;
                break;
            }
            // evaluate!
            h0 = tn - t;
            dt = dtn;
            t = tn;
            if (h == 0 && threadIdx.x == 0) lg_st(in.beat, (unsigned)steps);
        }
        const int st_end = (st < 0) ? 0 : 6;
#pragma unroll 1
        for (; st < st_end && status == LH_OK; st++) {
            const bool init = st < 0;
            const int sc = init ? 0 : st;
            const double dts = init ? 0.0 : dt;
            const double t2 = t + c_nodes[sc] * dts, hf = t2 - t;
            // prologue: ȳ = y + Δz Σ B k, ·exp(L hf), to the transform's bins;
            // F = outfac·exp(−L hf) from the same exp and sincos.  Every vector of
            // a round's bins is loaded together.  exp(L·dz) is computed once
            // per step, at stage 5: it serves stage 6, the window filter and the
            // next step's propagation of k1.  Bins outside the grid's band have
            // L = 0 and skip the exponential.
            const double sc_t = in.sc_t;
#pragma unroll 1
            for (int c = 0; c < NC; c++) {
                const int tid = fresh_tid();
                if (lg_none(tid, c * CB, nb)) break;
                double2 yb[CB], L[CB], of[CB], ee[CB], kk[6][CB];
                const bool reuse = st == 5;
                const bool carry = st == 0 && h0 != 0.0;
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    const int p = tid + (c * CB + i) * LH_T;
                    const bool v = p < nb;
                    yb[i] = v ? static_cast<const double2*>(gl(Y))[p] : make_double2(0.0, 0.0);
                    L[i] = (v && !reuse) ? static_cast<const double2*>(gl(Lg))[p] : make_double2(0.0, 0.0);
                    of[i] = (v && !reuse) ? static_cast<const double2*>(gl(OFg))[p] : make_double2(0.0, 0.0);
                    ee[i] = (v && (reuse || carry)) ? static_cast<const double2*>(gl(Ev))[p] : make_double2(0.0, 0.0);
                }
#pragma unroll
                for (int j = 0; j < 6; j++) {
                    const bool use = !init && j <= st && c_B[sc][j] != 0.0;
                    const double2* Kj = K[j];
#pragma unroll
                    for (int i = 0; i < CB; i++) {
                        const int p = tid + (c * CB + i) * LH_T;
                        kk[j][i] = (use && p < nb) ? Kj[p] : make_double2(0.0, 0.0);
                    }
                }
                if (carry) {
                    double2* K0 = K[0];
#pragma unroll
                    for (int i = 0; i < CB; i++) {
                        const int p = tid + (c * CB + i) * LH_T;
                        kk[0][i] = cmul(kk[0][i], ee[i]);
                        if (p < nb) K0[p] = kk[0][i];
                    }
                }
#pragma unroll
                for (int j = 0; j < 6; j++) {
                    const double cj = dts * c_B[sc][j];
                    if (j <= st && cj != 0.0) {
#pragma unroll
                        for (int i = 0; i < CB; i++) yb[i] = cadd(yb[i], cscal(cj, kk[j][i]));
                    }
                }
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    const int p = tid + (c * CB + i) * LH_T;
                    if (p < nb) {
                        double2 e = make_double2(1.0, 0.0), inv = make_double2(1.0, 0.0);
                        if (reuse) {
                            e = ee[i];
                        } else if (hf != 0.0 && (L[i].x != 0.0 || L[i].y != 0.0)) {
                            e = cexp_lh_inv(L[i], hf, inv);
                        }
                        const double2 X = cscal(sc_t, cmul(yb[i], e));
                        if constexpr (KIND == 0) {
                            int s, q;
                            Z::bin(p, s, q);
                            g_pack_bin<M>(sm, g, s, q, X);
                        } else {
                            sm.buf[pad(p)] = X;
                        }
                        if (!reuse) {
                            const double2 F = cmul(of[i], inv);
                            if (st == 4) gl(Ev)[p] = e;
                            gl(Fv)[p] = F;
                        }
                    }
                }
            }
            __syncthreads();
            g_rhs<KIND, M, RAMAN>(in, sm, g, rho, kfac, hw);
            // epilogue: k_{i+1} = F · RHS
            double2* out = K[init ? 0 : st + 1];
#pragma unroll 1
            for (int c = 0; c < NC; c++) {
                const int tid = fresh_tid();
                if (lg_none(tid, c * CB, nb)) break;
                double2 f[CB];
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    const int p = tid + (c * CB + i) * LH_T;
                    f[i] = (p < nb) ? static_cast<const double2*>(gl(Fv))[p] : make_double2(0.0, 0.0);
                }
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    const int p = tid + (c * CB + i) * LH_T;
                    if (p < nb) out[p] = cmul(g_rhs_bin<KIND, M>(sm, g, p), f[i]);
                }
            }
            rhs_evals++;
            __syncthreads();
            if (sm.gflag != LH_OK) status = sm.gflag;
        }
        if (status != LH_OK) break;
        if (st_end == 0) continue;  // the initial k1 is there; st is 0 now
        st = 0;
        steps++;
        // yn = y + Δz Σ b5 k ; yerr = Σ (Δz k) e ; weaknorm (src/RK45.jl:170-181, 343-354)
        double sy = 0.0, syn = 0.0, se = 0.0;
#pragma unroll 1
        for (int c = 0; c < NC; c++) {
            const int tid = fresh_tid();
            if (lg_none(tid, c * CB, nb)) break;
            double2 yv[CB], kk[7][CB];
#pragma unroll
            for (int i = 0; i < CB; i++) {
                const int p = tid + (c * CB + i) * LH_T;
                yv[i] = (p < nb) ? static_cast<const double2*>(gl(Y))[p] : make_double2(0.0, 0.0);
            }
#pragma unroll
            for (int j = 0; j < 7; j++) {
                if (j == 1) continue;  // b5[2] = b4[2] = 0
                const double2* Kj = K[j];
#pragma unroll
                for (int i = 0; i < CB; i++) {
                    const int p = tid + (c * CB + i) * LH_T;
                    kk[j][i] = (p < nb) ? Kj[p] : make_double2(0.0, 0.0);
                }
            }
#pragma unroll
            for (int i = 0; i < CB; i++) {
                const int p = tid + (c * CB + i) * LH_T;
                double2 yn = yv[i], ye = make_double2(0.0, 0.0);
#pragma unroll
                for (int j = 0; j < 7; j++) {
                    if (j == 1) continue;
                    const double cb = dt * c_b5[j], ce = c_b5[j] - c_b4[j];
                    yn = cadd(yn, cscal(cb, kk[j][i]));
                    ye = cadd(ye, cscal(ce, cscal(dt, kk[j][i])));
                }
                if (p < nb) {
                    sy += yv[i].x * yv[i].x + yv[i].y * yv[i].y;
                    syn += yn.x * yn.x + yn.y * yn.y;
                    se += ye.x * ye.x + ye.y * ye.y;
                    gl(YN)[p] = yn;
                }
            }
        }
        block_sum3(sy, syn, se, sm.wsum);
        {
            double* r = gl(g.rnext());
            if (threadIdx.x == 0) {
                r[8 * h + 0] = sy;
                r[8 * h + 1] = syn;
                r[8 * h + 2] = se;
            }
            gang_sync(g, sm);
            sy = lg_ld(r + 0);
            syn = lg_ld(r + 1);
            se = lg_ld(r + 2);
            for (int m = 1; m < LG_G; m++) {
                sy += lg_ld(r + 8 * m + 0);
                syn += lg_ld(r + 8 * m + 1);
                se += lg_ld(r + 8 * m + 2);
            }
        }
        const double errwt = fmax(fmax(sqrt(sy), sqrt(syn)), in.atol);
        const double err = sqrt(se) / in.rtol / errwt;
        bool ok = err <= 1.0;
        // stepcontrolPI!, src/RK45.jl:374-396, steplims! :399-406; the two powers of
        // an accepted step run in two lanes at once
        const double beta1 = 3.0 / 5 / 5, beta2 = -1.0 / 5 / 5, eps = 0.8;
        if (ok && errlast == 0.0) errlast = err;
        const bool l0 = (threadIdx.x & 63) == 0;
        const double pw = pow(ok ? eps / (l0 ? err : errlast) : err, ok ? (l0 ? beta1 : beta2) : -1.0 / 5);
        if (ok) {
            const double fac = (err == 0.0) ? 1.5 : in.safety * lane_value(pw, 0) * lane_value(pw, 1);
            dtn = fac * dt;
            errlast = err;
        } else {
            if (!isfinite(err))
                dtn = dt / 2;
            else
                dtn = dt * fmax(0.1, in.safety * lane_value(pw, 0));
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
            // (src/Output.jl:65-67)
            double* rec = (gl(in.steprec) && accepted < in.steprec_cap) ? gl(in.steprec) + (size_t)accepted * LH_NSTAT
                                                                      : nullptr;
            g_stepfun<KIND, M, (M <= 8192)>(in, sm, g, Ev, YN, rec, tn, dtn, rho);
            if (sm.gflag != LH_OK) status = sm.gflag;
            // GridCondition saves via dense output; ks[1] and ks[7] both hold k7
            const int saved_before = saved;
            while (saved < in.save_n && gl(in.zgrid)[saved] <= tn) {
                const double ti = gl(in.zgrid)[saved];
                if (gl(in.saves)) {
                    double2* out = gl(in.saves) + (size_t)saved * N;
                    if (ti == t) {
                        for (int p = fresh_tid(); p < nb; p += LH_T) gl(out)[Z::k_of(h, p)] = gl(Y)[p];
                    } else if (ti == tn) {
                        for (int p = fresh_tid(); p < nb; p += LH_T) gl(out)[Z::k_of(h, p)] = gl(YN)[p];
                    } else {
                        const double sg = (ti - t) / dt;
                        const double sp1 = sg, sp2 = sg * sg, sp3 = sp2 * sg, sp4 = sp2 * sp2;
                        const double hs = ti - t;
#pragma unroll 1
                        for (int c = 0; c < NC; c++) {
                            const int tid = fresh_tid();
                            if (lg_none(tid, c * CB, nb)) break;
                            double2 kk[7][CB], yv[CB], Lv[CB], yi[CB];
#pragma unroll
                            for (int i = 0; i < CB; i++) {
                                const int p = tid + (c * CB + i) * LH_T;
                                yv[i] = (p < nb) ? static_cast<const double2*>(gl(Y))[p] : make_double2(0.0, 0.0);
                                Lv[i] = (p < nb) ? static_cast<const double2*>(gl(Lg))[p] : make_double2(0.0, 0.0);
                                yi[i] = make_double2(0.0, 0.0);
                            }
#pragma unroll
                            for (int j = 0; j < 7; j++) {
                                if (j == 1) continue;
                                const double2* kj = (j == 6) ? K[0] : K[j];
#pragma unroll
                                for (int i = 0; i < CB; i++) {
                                    const int p = tid + (c * CB + i) * LH_T;
                                    kk[j][i] = (p < nb) ? kj[p] : make_double2(0.0, 0.0);
                                }
                            }
#pragma unroll
                            for (int j = 0; j < 7; j++) {
                                if (j == 1) continue;
                                // weight b_j(σ) = Σ_p σ^p C[p][j] of the dense output
                                const double bj =
                                    ((sp1 * c_iC[0][j] + sp2 * c_iC[1][j]) + sp3 * c_iC[2][j]) + sp4 * c_iC[3][j];
#pragma unroll
                                for (int i = 0; i < CB; i++) yi[i] = cadd(yi[i], cscal(bj, kk[j][i]));
                            }
#pragma unroll
                            for (int i = 0; i < CB; i++) {
                                const int p = tid + (c * CB + i) * LH_T;
                                if (p < nb) {
                                    const double2 e = (Lv[i].x != 0.0 || Lv[i].y != 0.0) ? cexp_lh(Lv[i], hs)
                                                                                        : make_double2(1.0, 0.0);
                                    gl(out)[Z::k_of(h, p)] = cmul(cadd(yv[i], cscal(dt, yi[i])), e);
                                }
                            }
                        }
                    }
                }
                saved++;
            }
            if (STREAM && (saved > saved_before || in.pub_ring > 0)) {
                // the output call of this step (src/Output.jl:65-81, 262-302):
                // its saves are in place; hand over the state, then member 0
                // publishes and tells the others whether to stop
                const int slot = (in.pub_ring > 0) ? (int)(npub % in.pub_ring) : (int)(npub & 1);
                double2* py = in.pub_y + (size_t)slot * N;
                for (int p = fresh_tid(); p < nb; p += LH_T) py[Z::k_of(h, p)] = gl(YN)[p];
                if (h == 0 && threadIdx.x == 0) {
                    double* info = in.pub_info + 4 * slot;
                    info[0] = tn;
                    info[1] = dtn;
                    info[2] = (double)saved;
                    info[3] = (double)(accepted + 1);
                }
                __threadfence_system();
                gang_sync(g, sm);
                if (h == 0 && threadIdx.x == 0) {
                    __hip_atomic_store(in.pub, (unsigned long long)(npub + 1), __ATOMIC_RELEASE,
                                       __HIP_MEMORY_SCOPE_SYSTEM);
                    if (__hip_atomic_load(in.pub_stop, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM))
                        sm.flag = LH_E_STOPPED;
                }
                gang_sync(g, sm);
                if (sm.gflag == LH_E_STOPPED && status == LH_OK && tn <= in.zmax) status = LH_E_STOPPED;
                npub++;
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
    for (int p = fresh_tid(); p < nb; p += LH_T) gl(in.Y)[Z::k_of(h, p)] = gl(Y)[p];
    // (a word of its own: agreeing on the status at one more barrier, with the
    // counters in registers, cost a dense kernel 10 spills and a sweep 1.5 %)
    if (sm.gflag == LG_LOST && threadIdx.x == 0) lg_st(&in.stats->lost, 1);
    if (h == 0 && threadIdx.x == 0 && gl(in.stats)) {
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

// LDS of a class: the longest transform is M points, 2·M with the field grid's
// Raman convolution.  The list of ionising samples leaves room for two
// workgroups per CU up to M = 8192.
template <int KIND, int M, bool RAMAN>
struct GLds {
    using T = GSmem<(KIND == 0 && RAMAN) ? M / 2 : M / 4, (KIND == 1) ? 1 : (M >= 16384 || RAMAN) ? 1024 : 2048>;
};

// Forms gangs and hands their members jobs (lg_next_job).  run(job) is called by
// all members of a gang together.  status: null, or where the status of a launch
// of one job goes, whose control block then serves launch after launch (in
// stream order) instead of being set for each.
template <bool RESET, class SM, class F>
__device__ __forceinline__ void gang_loop(GangCtl* ctl, SM& sm, Gang& g, int* status, F run) {
    const int n_gang = (int)(ctl->n_wg / LG_G);
    const unsigned njobs = ctl->njobs;
    unsigned long long* mailbox = (unsigned long long*)((char*)ctl + lg_mail_off(njobs));
    if (threadIdx.x == 0) {
        const unsigned xcc = __builtin_amdgcn_s_getreg((3 << 11) | 20) & (LG_XCC - 1);  // HW_REG_XCC_ID, 4 bits
        const unsigned tk = LgMem::add(&ctl->ticket[xcc], 1u);
        sm.member = (int)(tk % LG_G);
        sm.slot = (int)(xcc * n_gang + tk / LG_G);
        sm.gflag = LH_OK;
    }
    __syncthreads();
    g.h = __builtin_amdgcn_readfirstlane(sm.member);
    unsigned long long* mail = mailbox + __builtin_amdgcn_readfirstlane(sm.slot);
    unsigned seq = 1;
    for (;;) {
        if (threadIdx.x == 0)
            sm.job = (int)lg_next_job<LgMem>(ctl, mail, g.h, seq, sm.gflag == LG_LOST, njobs, LG_MAX_POLL);
        __syncthreads();
        const int job = __builtin_amdgcn_readfirstlane(sm.job);
        __syncthreads();
        if (job < 0) break;
        seq++;
        g.flags = (unsigned*)((char*)ctl + lg_flags_off()) + (size_t)job * LG_G * LG_FLAG_STRIDE;
        g.ep = 0;
        g.xb = g.rb = 0;
        run(job);
    }
    if constexpr (RESET) {
        // the last workgroup to leave has the status of all, and makes the control
        // block ready for the next launch
        if (threadIdx.x == 0) {
            const unsigned mine = lg_leave(g.h, seq - 1, sm.gflag), sum = LgMem::add(&ctl->left, mine) + mine;
            sm.job = (sum & 255u) == ctl->n_wg;
            if (sm.job) *status = lg_left(sum);
        }
        __syncthreads();
        if (sm.job) {
            unsigned* flags = (unsigned*)((char*)ctl + lg_flags_off());
            for (int i = threadIdx.x; i < (int)njobs * LG_G; i += LH_T) lg_st(flags + i * LG_FLAG_STRIDE, 0u);
            for (int i = threadIdx.x; i < LG_XCC * n_gang; i += LH_T) lg_st(mailbox + i, 0ull);
            if (threadIdx.x < LG_XCC) lg_st(ctl->ticket + threadIdx.x, 0u);
            if (threadIdx.x == 0) {
                lg_st(&ctl->next_job, 0u);
                lg_st(&ctl->left, 0u);
            }
        }
    }
}

// Exchange area of an instance: two series, 2·32 records of 8 doubles, M doubles.
__device__ __forceinline__ void gang_area(Gang& g, const DInst& in) {
    g.xlen = in.gx_len;
    g.X = in.gx;
    g.rec = (double*)(in.gx + 2 * (size_t)in.gx_len);
    g.P = g.rec + 512;
}

// DENSE: compiled for two workgroups per CU (128 registers; 128 of the field
// kernel's values at Nto = 16384 spill, most of them around the transform
// passes; 204 with three bins per thread in a round of loads).  The same source,
// so the same bits; the loads of a round alone are grouped differently.
template <int KIND, int M, bool STREAM, bool RAMAN, bool DENSE = false>
__global__ __launch_bounds__(LH_T, DENSE ? 4 : 1) void lh_gang_solve(GangCtl* ctl, const DInst* insts,
                                                                     const double2* __restrict__ twg) {
    using SM = typename GLds<KIND, M, RAMAN>::T;
    __shared__ SM sm;
    gtw_load(sm.tw, twg);
    Gang g;
    gang_loop<false>(ctl, sm, g, nullptr, [&](int job) {
        const DInst& in = insts[job];
        gang_area(g, in);
        g_solve<KIND, M, STREAM, RAMAN, DENSE>(in, sm, g);
    });
}

// One right-hand side of rhs_in into rhs_out (natural order), by one gang.
template <int KIND, int M, bool RAMAN>
__global__ __launch_bounds__(LH_T) void lh_gang_rhs(GangCtl* ctl, const DInst in, const double2* __restrict__ twg,
                                                    int* status) {
    using SM = typename GLds<KIND, M, RAMAN>::T;
    using Z = GSizes<KIND, M>;
    __shared__ SM sm;
    gtw_load(sm.tw, twg);
    Gang g;
    gang_loop<true>(ctl, sm, g, status, [&](int) {
        gang_area(g, in);
        if (threadIdx.x == 0) sm.flag = sm.gflag = LH_OK;
        __syncthreads();
        const int h = g.h, nb = Z::count(h);
        const bool zdep = (KIND == 0) && !RAMAN && in.zg_np > 0;
        double rho = in.density, kfac = in.kerr_fac;
        if (zdep)  // the call's z
            g_zg_refresh<KIND, M>(in, sm, h, in.zL + (size_t)h * Z::GSTR, in.zOF + (size_t)h * Z::GSTR, in.z0, rho, kfac);
        for (int p = threadIdx.x; p < nb; p += LH_T) {
            const double2 v = cscal(in.sc_t, gl(in.rhs_in)[Z::k_of(h, p)]);
            if constexpr (KIND == 0) {
                int s, q;
                Z::bin(p, s, q);
                g_pack_bin<M>(sm, g, s, q, v);
            } else {
                sm.buf[pad(p)] = v;
            }
        }
        __syncthreads();
        const double2* hwn = gl(in.hwdt);
        g_rhs<KIND, M, RAMAN>(in, sm, g, rho, kfac,
                              [hwn, h](int s, int q) { return hwn[GGeo<M>::res(h, s) + 8 * q]; });
        const double2* of = zdep ? gl(in.zOF) + (size_t)h * Z::GSTR : gl(in.outfac);
        for (int p = threadIdx.x; p < nb; p += LH_T) {
            const int k = Z::k_of(h, p);
            gl(in.rhs_out)[k] = cmul(g_rhs_bin<KIND, M>(sm, g, p), of[zdep ? p : k]);
        }
    });
}

// Statistics of one given state (rhs_in) into steprec[0..LH_NSTAT).
template <int KIND, int M>
__global__ __launch_bounds__(LH_T) void lh_gang_stats(GangCtl* ctl, const DInst in, const double2* __restrict__ twg,
                                                      double z, double dz, int* status) {
    using SM = typename GLds<KIND, M, false>::T;
    using Z = GSizes<KIND, M>;
    constexpr int S = M / 8;
    __shared__ SM sm;
    gtw_load(sm.tw, twg);
    Gang g;
    gang_loop<true>(ctl, sm, g, status, [&](int) {
        gang_area(g, in);
        if (threadIdx.x == 0) sm.flag = sm.gflag = LH_OK;
        __syncthreads();
        const int h = g.h, nb = Z::count(h);
        double rho = in.density, kfac = in.kerr_fac;
        if (KIND == 0 && in.zg_np > 0)
            g_zg_refresh<KIND, M>(in, sm, h, in.zL + (size_t)h * Z::GSTR, in.zOF + (size_t)h * Z::GSTR, z, rho, kfac);
        double s0 = 0.0, s1 = 0.0, se = 0.0;
        WinSums ws = {{0.0, 0.0, 0.0, 0.0}};
        for (int p = threadIdx.x; p < nb; p += LH_T) {
            const int k = Z::k_of(h, p);
            const double2 v = gl(in.rhs_in)[k];
            const double a = v.x * v.x + v.y * v.y;
            s0 += a;
            s1 += gl(in.st_omega)[k] * a;
            se += gl(in.st_ew)[k] * a;
            win_add(in, ws, k, a);
            if constexpr (KIND == 0) {  // copyto_fft!: bins 0..Nω−2 doubled, the +fs/2 bin dropped, zero up to M
                if (p < Z::NB) {
                    const int s = (p >= S / 2) ? 1 : 0, q = p - s * (S / 2);
                    sm.buf[pad(s * S + q)] = make_double2(2.0 * v.x, 2.0 * v.y);
                    sm.buf[pad(s * S + S / 2 + q)] = make_double2(0.0, 0.0);
                }
            } else {
                sm.buf[pad(p)] = v;
            }
        }
        g_stats<KIND, M>(in, sm, g, s0, s1, se, ws, z, dz, rho, gl(in.steprec));
    });
}

template <int KIND, int M, bool RAMAN>
static bool lg_launch_solve(const GangLaunch& l, bool stream) {
    if (stream)
        hipLaunchKernelGGL((lh_gang_solve<KIND, M, true, RAMAN>), dim3(l.nwg), dim3(LH_T), 0, l.s, l.ctl, l.d, l.tw);
    else
        hipLaunchKernelGGL((lh_gang_solve<KIND, M, false, RAMAN>), dim3(l.nwg), dim3(LH_T), 0, l.s, l.ctl, l.d, l.tw);
    return true;
}
template <int M>
static bool lg_launch_dense(const GangLaunch& l) {
    static_assert(2 * sizeof(typename GLds<0, M, false>::T) <= 160 * 1024, "two workgroups per CU");
    hipLaunchKernelGGL((lh_gang_solve<0, M, false, false, true>), dim3(l.nwg), dim3(LH_T), 0, l.s, l.ctl, l.d, l.tw);
    return true;
}
template <int KIND, int M, bool RAMAN>
static bool lg_launch_rhs(const GangLaunch& l, int* status) {
    hipLaunchKernelGGL((lh_gang_rhs<KIND, M, RAMAN>), dim3(l.nwg), dim3(LH_T), 0, l.s, l.ctl, *l.d, l.tw, status);
    return true;
}
template <int KIND, int M>
static bool lg_launch_stats(const GangLaunch& l, double z, double dz, int* status) {
    hipLaunchKernelGGL((lh_gang_stats<KIND, M>), dim3(l.nwg), dim3(LH_T), 0, l.s, l.ctl, *l.d, l.tw, z, dz, status);
    return true;
}
