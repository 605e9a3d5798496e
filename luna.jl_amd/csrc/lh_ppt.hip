// lh_ppt.hip -- PPT ionisation-rate table on the GPU (set-up of the plasma
// response: makePPTcache, src/Ionisation.jl:185-200, with ionrate_fun_PPT,
// :317-390, and φ, :403-429).  A group of lanes works on one field value: it
// evaluates that many consecutive terms of the PPT sum at once, adds them with
// a prefix sum and stops at the first term that meets the reference's
// converge_series rule (src/Maths.jl:721-736).
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/luna_hip.h"
#include "lh_device.h"

namespace {

constexpr double kInvSqrtPi = 0.56418958354775628695;  // 1/√π
constexpr double kRybH = 0.25;                         // Rybicki sampling step
constexpr int kRybN = 13;                              // sample pairs
constexpr double kAsym = 10.0;                         // asymptotic series from here on
// odd denominators of the sample pairs for 0 ≤ x < kAsym: n0 = 2 rint(2x) ≤ 40
// gives −(2·kRybN − 1) .. 40 + 2·kRybN − 1
constexpr int kOddLo = -(2 * kRybN - 1), kOddN = (40 + 4 * kRybN) / 2;
constexpr int kPptBlock = 1024;
constexpr int kPptPoints = 256;             // field values per workgroup at most
constexpr int kPptGrid = 256;               // one workgroup per CU while they suffice
constexpr int kPptWide = 16384;         // up to here a whole wave per field value
constexpr long long kMaxTerms = 1LL << 24;  // a series longer than this is reported

struct PptTables {
    double c[kRybN];      // exp(-((2i+1)h)²)
    double rodd[kOddN];   // 1/(kOddLo + 2i)
};

// Dawson's integral D(x) = exp(-x²)∫₀ˣ exp(t²) dt for 0 ≤ x < kAsym.
// x < 0.2: its Taylor series Σ (-2x²)^k x / (2k+1)!!.  Otherwise Rybicki's
// sampling formula D(x) = lim_{h→0} π^{-1/2} Σ_{n odd} exp(-(x - nh)²)/n
// (G. B. Rybicki, Computers in Physics 3, 85 (1989)), summed around the
// nearest even multiple of h; with h = 0.25 the sampling error is of order
// exp(-(π/2h)²) ≈ 7e-18 and 13 pairs leave out terms below exp(-42).  The
// reciprocals of the odd integers come from LDS: the 26 divisions of one value
// were nine tenths of its time.
__device__ __forceinline__ double dawson(double x, const PptTables& tb) {
    if (x < 0.2) {
        const double y = -2.0 * x * x;
        double r = 1.0;
#pragma unroll
        for (int k = 12; k >= 1; k--) r = 1.0 + y * (1.0 / (2 * k + 1)) * r;
        return x * r;
    }
    const double m0 = rint(0.5 * x / kRybH);
    const double xp = x - m0 * (2 * kRybH);
    double e1 = exp(2.0 * xp * kRybH), i1 = exp(-2.0 * xp * kRybH);
    const double e2 = e1 * e1, i2 = i1 * i1;
    const double* r1 = tb.rodd + ((int)m0 + (1 - kOddLo) / 2);  // 1/(n0 + 1), n0 = 2 m0
    double sum = 0.0;
#pragma unroll
    for (int i = 0; i < kRybN; i++) {
        sum += tb.c[i] * (e1 * r1[i] + i1 * r1[-1 - i]);
        e1 *= e2;
        i1 *= i2;
    }
    return kInvSqrtPi * exp(-xp * xp) * sum;
}

// Coefficients in 1/x² of the asymptotic series of 2x·φ_0, c_k = (2k-1)!!/2^k,
// and of 2x·φ_1, c_{k+1} + c_k/2.
constexpr int kAsym0 = 13, kAsym1 = 15;
struct Asym {
    double a[kAsym1], b[kAsym1];
    constexpr Asym() : a(), b() {
        double c = 1.0;
        for (int k = 0; k < kAsym1; k++) {
            const double c1 = c * (2 * k + 1) * 0.5;
            a[k] = c;
            b[k] = c1 + 0.5 * c;
            c = c1;
        }
    }
};

// φ_m(x) = exp(-x²)∫₀ˣ (x² - y²)^|m| exp(y²) dy for m = 0 and |m| = 1 at
// x = √s (PPT, src/Ionisation.jl:403-429).  φ_0 = D(x).  φ_1 = (x² + 1/2) D(x) - x/2
// (integrating y² exp(y²) by parts), which cancels to ~1/(2x) for large x.  From
// x = 10 on both are their asymptotic series φ_0 = (1/2x) Σ_k c_k x^{-2k} and
// φ_1 = (1/2x) Σ_k (c_{k+1} + c_k/2) x^{-2k} (13 and 15 terms; the first
// omitted ones are below 1e-16 of the sums there).
template <bool M1>
__device__ __forceinline__ void ppt_phi(double s, const PptTables& tb, double& p0, double& p1) {
    const double x = sqrt(s);
    if (x < kAsym) {
        p0 = dawson(x, tb);
        if (M1) p1 = (x * x + 0.5) * p0 - 0.5 * x;
    } else {
        const double is = 1.0 / s, h = 0.5 * x * is;
        constexpr Asym as;
        double a = 0.0, b = 0.0;
#pragma unroll
        for (int k = kAsym1 - 1; k >= 0; k--) {
            if (k < kAsym0) a = a * is + as.a[k];
            if (M1) b = b * is + as.b[k];
        }
        p0 = a * h;
        if (M1) p1 = b * h;
    }
}

__device__ __forceinline__ double fact(int n) {
    double f = 1.0;
    for (int i = 2; i <= n; i++) f *= (double)i;
    return f;
}

// What the terms of one field value need, and the factors its sums are multiplied by.
struct PptPoint {
    double n0, v, alpha, beta;  // first term ceil(v); exponents
    double f[2];                // prefactors of the m = 0 and |m| = 1 sums
    double post;                // dipole correction
};

// ionrate_fun_PPT at field E up to its sums (src/Ionisation.jl:330-384), the
// same sequence of operations as the reference.
__device__ PptPoint ppt_point(const lh_ppt_desc& p, double E) {
    PptPoint q;
    const double au_energy = p.au_energy, au_time = p.au_time, au_efield = p.au_efield;
    const double Ip_au = (p.ionpot + p.dalpha / 2 * (E * E)) / au_energy;
    const double ns = p.Z / sqrt(2 * Ip_au);
    const double ls = ns - 1;
    const double Cnl2 = (p.cnl > 0) ? p.cnl * p.cnl : pow(2.0, 2 * ns) / (ns * tgamma(ns + ls + 1) * tgamma(ns - ls));
    const double w0 = 2 * M_PI * p.c / p.lambda0;
    const double w0_au = au_time * w0;
    const double E0_au = pow(2 * Ip_au, 1.5);
    const double E_au = fabs(E) / au_efield;
    const double g = w0_au * sqrt(2 * Ip_au) / E_au;
    const double g2 = g * g;
    q.beta = 2 * g / sqrt(1 + g2);
    q.alpha = 2 * (asinh(g) - g / sqrt(1 + g2));
    const double Up_au = (E_au * E_au) / (4 * (w0_au * w0_au));
    q.v = (Ip_au + Up_au) / w0_au;
    q.n0 = ceil(q.v);
    const int l = p.l, m1 = p.msum ? l : 0;
    for (int mabs = 0; mabs <= 1; mabs++) {
        q.f[mabs] = 0.0;
        if (mabs > m1) continue;
        const double flm = ((2 * l + 1) * fact(l + mabs)) / (pow(2.0, (double)mabs) * fact(mabs) * fact(l - mabs));
        double lret = 4 * sqrt(2.0) / M_PI * Cnl2;
        lret *= pow(2 * E0_au / (E_au * sqrt(1 + g2)), 2 * ns - mabs - 1.5);
        lret *= flm / fact(mabs);
        lret *= exp(-2 * q.v * (asinh(g) - g * sqrt(1 + g2) / (1 + 2 * g2)));
        lret *= Ip_au * g2 / (1 + g2);
        if (!p.cycle_average) lret *= sqrt(M_PI * E0_au / (3 * E_au));
        q.f[mabs] = lret;
    }
    q.post = (p.alpha_ion_au != 0) ? exp(-2 * p.alpha_ion_au * E_au) : 1.0;
    return q;
}

// Inclusive prefix sum over the G lanes of a group (16: a DPP row, 64: the wave).
template <int G>
__device__ __forceinline__ double group_scan(double x) {
    x += dpp_f64<DPP_ROW_SHR1>(x);
    x += dpp_f64<DPP_ROW_SHR2>(x);
    x += dpp_f64<DPP_ROW_SHR4>(x);
    x += dpp_f64<DPP_ROW_SHR8>(x);
    if constexpr (G == 64) {
        x += dpp_f64<DPP_ROW_BCAST15, 0xa>(x);
        x += dpp_f64<DPP_ROW_BCAST31, 0xc>(x);
    }
    return x;
}

// One sum of a group's field value: adds the group's G next terms to x and sets
// done at the first that meets 2|x1 − x0|/|x1 + x0| < tol.
template <int G>
__device__ __forceinline__ void ppt_add(double term, double tol, double& x, bool& done) {
    const int lane = threadIdx.x & 63, g0 = lane & ~(G - 1);
    const double inc = group_scan<G>(term);
    const double ex = (G == 64) ? dpp_f64<DPP_WAVE_SHR1>(inc) : dpp_f64<DPP_ROW_SHR1>(inc);
    const double x1 = x + inc, x0 = x + ex;
    const unsigned long long hit = __ballot(2 * fabs(x1 - x0) < tol * fabs(x1 + x0));
    const unsigned long long mine = (G == 64) ? hit : (hit >> g0) & ((1ull << (G & 63)) - 1);
    const double xn = __shfl(x1, g0 + (mine ? __ffsll(mine) - 1 : G - 1));
    if (!done) {
        x = xn;
        done = (mine != 0);
    }
}

// Workgroup b has the field values b, b + gridDim, ...: the length of the sum
// rises steeply with the field (7 to 300 terms for Ar at 800 nm, 60 to 15000 for
// He at 2 µm), so neighbours are spread over the chip, and the waves of a
// workgroup take groups of values from a counter, from the high end.
// Bound by the FP64 arithmetic of the terms (one exponential, one square root
// and one φ each; a serial sum per lane was bound by the longest sum and by the
// divisions of φ): 65536 values of Ar at 800 nm in 67 µs (756 µs), of He at 2 µm
// in 1.2 ms (16.0 ms).  A wave per value (G = 64) has the shorter chain, 16
// lanes waste fewer terms past the end of short sums: µs at G = 64 / 16, 8192
// values: Ar 22/28, He 34/62, He at 2 µm 175/446, Xe at 400 nm 17/13; 16384:
// 32/29, 56/66, 321/456, 22/13; 65536: 88/67, 175/171, 1082/1184, 56/25.
template <int G, bool M1>
__global__ __launch_bounds__(kPptBlock) void lh_ppt_kernel(lh_ppt_desc p, const double* __restrict__ E, int n,
                                                           double* __restrict__ rate, int* status) {
    __shared__ PptTables tb;
    __shared__ PptPoint pt[kPptPoints];
    __shared__ int next;
    const int tid = threadIdx.x, lane = tid & 63, nb = gridDim.x, b = blockIdx.x;
    const int np = (n - b + nb - 1) / nb;
    if (tid < kPptPoints && tid < np) pt[tid] = ppt_point(p, E[b + (long long)nb * tid]);
    if (tid >= kPptBlock - 64 && lane < kRybN) {
        const double a = (2 * lane + 1) * kRybH;
        tb.c[lane] = exp(-a * a);
    }
    if (tid >= kPptBlock - 128 && tid < kPptBlock - 64 && lane < kOddN) tb.rodd[lane] = 1.0 / (kOddLo + 2 * lane);
    if (tid == kPptBlock - 1) next = 0;
    __syncthreads();
    constexpr int PER = 64 / G;
    const int gl = lane & (G - 1);
    for (;;) {
        int t = 0;
        if (lane == 0) t = atomicAdd(&next, PER);
        t = __builtin_amdgcn_readfirstlane(t);
        if (t >= np) break;
        const int j = np - 1 - t - lane / G;
        const bool live = j >= 0;
        const PptPoint& q = pt[live ? j : 0];
        const double n0 = q.n0, v = q.v, alpha = q.alpha, beta = q.beta;
        // n grows by repeated n += 1.0, which stands still from 2^53 on
        const double cap = fmax(n0 + 1.0, 9007199254740992.0);
        double xa = 0.0, xb = 0.0;
        bool da = !live, db = !live || !M1;
        long long it = 0;
        while (it < kMaxTerms && __any(!(da && db))) {
            const double diff = fmin(n0 + (double)(it + gl), cap) - v;
            const double ex = exp(-alpha * diff);
            double p0, p1 = 0.0;
            ppt_phi<M1>(beta * diff, tb, p0, p1);
            ppt_add<G>(ex * p0, p.sum_tol, xa, da);
            if (M1) ppt_add<G>(ex * p1, p.sum_tol, xb, db);
            it += G;
        }
        if (live && gl == 0) {
            // Σ over m = −l..l: the |m| = 1 sums are equal
            double ret = 0.0;
            if (M1) ret += p.occupancy * (q.f[1] * xb);
            ret += p.occupancy * (q.f[0] * xa);
            if (M1) ret += p.occupancy * (q.f[1] * xb);
            if (p.alpha_ion_au != 0) ret *= q.post;
            rate[b + (long long)nb * j] = ret / p.au_time;
            if (!(da && db)) atomicMax(status, LH_E_NONFINITE);
        }
    }
}

}  // namespace

#define PPT_CK(x)                                                                    \
    do {                                                                             \
        hipError_t e_ = (x);                                                         \
        if (e_ != hipSuccess) {                                                      \
            fprintf(stderr, "luna_hip: %s failed: %s\n", #x, hipGetErrorString(e_)); \
            st = (e_ == hipErrorOutOfMemory) ? LH_E_NOMEM : LH_E_HIP;                \
            goto done;                                                               \
        }                                                                            \
    } while (0)

extern "C" int lh_ppt_table(const lh_ppt_desc* p, int n, const double* E, double* rate, double* ms) {
    if (!p || !E || !rate || n <= 0) return LH_E_ARG;
    if (p->l < 0 || p->l > 1 || !(p->sum_tol > 0) || !(p->lambda0 > 0) || !(p->ionpot > 0)) return LH_E_ARG;
    for (int i = 0; i < n; i++)
        if (!(E[i] > 0)) return LH_E_ARG;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return LH_E_NODEVICE;
    int st = LH_OK, kst = LH_OK;
    double *dE = nullptr, *dR = nullptr;  // one allocation: field values, rates, status
    int* dS = nullptr;
    hipEvent_t t0 = nullptr, t1 = nullptr;
    const size_t bytes = sizeof(double) * (size_t)n;
    PPT_CK(hipMalloc(&dE, 2 * bytes + sizeof(int)));
    dR = dE + n;
    dS = (int*)(dR + n);
    PPT_CK(hipMemsetAsync(dS, 0, sizeof(int), nullptr));
    PPT_CK(hipMemcpy(dE, E, bytes, hipMemcpyHostToDevice));
    PPT_CK(hipEventCreate(&t0));
    PPT_CK(hipEventCreate(&t1));
    PPT_CK(hipEventRecord(t0, nullptr));
    {
        int nb = (n < kPptGrid) ? n : kPptGrid;
        if (n > kPptGrid * kPptPoints) nb = (n - 1) / kPptPoints + 1;
        const bool m1 = p->l == 1 && p->msum;
        auto k = (n <= kPptWide) ? (m1 ? lh_ppt_kernel<64, true> : lh_ppt_kernel<64, false>)
                                 : (m1 ? lh_ppt_kernel<16, true> : lh_ppt_kernel<16, false>);
        hipLaunchKernelGGL(k, dim3(nb), dim3(kPptBlock), 0, nullptr, *p, dE, n, dR, dS);
    }
    PPT_CK(hipGetLastError());
    PPT_CK(hipEventRecord(t1, nullptr));
    PPT_CK(hipMemcpy(rate, dR, bytes, hipMemcpyDeviceToHost));
    PPT_CK(hipMemcpy(&kst, dS, sizeof(int), hipMemcpyDeviceToHost));
    if (ms) {
        float f = 0.0f;
        PPT_CK(hipEventElapsedTime(&f, t0, t1));
        *ms = f;
    }
    st = kst;
done:
    if (t0) (void)hipEventDestroy(t0);
    if (t1) (void)hipEventDestroy(t1);
    if (dE) (void)hipFree(dE);
    return st;
}
