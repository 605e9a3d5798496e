// lh_fno.hip -- 1-D Fourier neural operator surrogate on gfx950.
//
// Every matrix product (lift, the truncated forward/inverse DFTs of the
// spectral convolution, the per-mode complex channel mixing, the pointwise
// channel mixing, and all their gradients) is part of a launch of one strided,
// batched kernel on BF16 matrix cores with FP32 accumulation.  The truncated
// DFT is a dense (2·modes × n_x) product: with 32 modes of a 1024-point series
// it is cheaper as a matrix-core product than as an FFT, and it keeps the whole
// network on the MFMA path.  The projection head runs on FP32 matrix cores in
// kernels of its own; elementwise work (GELU and its derivative, loss) runs in
// FP32 inside the kernels that produce or read its operands, AdamW in one pass.
// Reductions over the batch (bias gradients, split-K partial sums, the loss) use
// fixed orders, so results are deterministic run to run.

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <initializer_list>
#include <utility>
#include <vector>

#include "../../include/luna_fno.h"
#include "../../include/luna_hip.h"

typedef float fno_f4 __attribute__((ext_vector_type(4)));
typedef __bf16 fno_bf8 __attribute__((ext_vector_type(8)));

static const int FNO_MAXL = 8;
static const int FNO_T = 256;

#define FNOCK(x)                                                                     \
    do {                                                                             \
        hipError_t e_ = (x);                                                         \
        if (e_ != hipSuccess) {                                                      \
            fprintf(stderr, "luna_fno: %s failed: %s\n", #x, hipGetErrorString(e_)); \
            return (e_ == hipErrorOutOfMemory) ? LH_E_NOMEM : LH_E_HIP;              \
        }                                                                            \
    } while (0)

// ---------------------------------------------------------------------------
// Elementwise functions
// ---------------------------------------------------------------------------
__device__ __forceinline__ float gelu_f(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_d(float z) {
    return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * expf(-0.5f * z * z) * 0.39894228040143268f;
}

// ---------------------------------------------------------------------------
// Strided, batched products on BF16 matrix cores:
//   acc_p[b] = A_p[b] · B_p[b],  p = 0 (and 1),
//   C[b] = acc_1 + acc_0  (or acc_0 − acc_1; one product: acc_0)  + bias[n],
//   then optionally gelu(C) into a second output, or C · gelu'(zref).
//   A(m, k) = A[b·sa_b + m·sa_m + k·sa_k],  B(k, n) = B[b·sb_b + k·sb_k + n·sb_n],
//   C(m, n) = C[b·sc_b + m·sc_m + n]; each operand is contiguous in one of its
//   two dimensions and holds FP32 or BF16.
// Workgroup tile 64×64, K slab 64; four wave64s, each 32×32 = 2×2 tiles of
// v_mfma_f32_16x16x32_bf16.  Lane l supplies A[l%16][8(l/16)..8(l/16)+7] and
// B[8(l/16)..+7][l%16]; accumulator register r of lane l is D[4(l/16)+r][l%16].
// Operands are converted to BF16 (round to nearest even) on their way to LDS.
// With ksplit > 1 each k range goes into work[] and a second kernel adds the
// ranges in order.  One launch runs up to three independent products (a group).
//
// These products are small (K of 64 to 1024, 8 MB operands): bound by the load
// latency of a slab and by launches, not by the matrix cores.  So a thread
// loads a slab as four 4-element vectors, the next slab's loads are in flight
// while this one multiplies, products that share their output or their input
// share a launch, and the activation is applied where its input is produced.
// Loss and gradient of 32 series of 1024 points, 64 channels, 32 modes, 4
// layers: 39 launches, 370 µs (92 launches of one product or elementwise pass
// each with 4-byte loads, 960 µs; 12 to 20 µs a product, now 7 to 15).
// ---------------------------------------------------------------------------
struct FnoOp {  // one operand: rows m (A) or n (B), k
    const void* p;
    long long s_row, s_k, s_b;
    int bf;   // BF16 elements
    int kc;   // contiguous along k (else along the rows)
    int vec;  // base and strides allow 4-element loads
};
struct GemmArgs {
    int M, N, K[2], batch, ksplit, kchunk, np;
    FnoOp A[2], B[2];
    float sign;  // of product 1 where it is subtracted (−1), else +1
    float* C;
    long long sc_m, sc_b;
    const float* bias;
    float* gelu_out;    // gelu(C), same layout as C
    const float* zref;  // C is multiplied by gelu'(zref), same layout as C
    float* rowsum;      // Σ_k A(m, k) in FP32 (batch 1, A contiguous along its rows)
    float* work;
    int gx, gy, nblk;
    int cvec;  // the outputs allow 4-element accesses
};
struct GemmGroup {
    GemmArgs g[3];
    int n;
};

constexpr int KB = 64;        // K slab
constexpr int LDB = KB + 8;   // LDS row (BF16): 16-byte aligned, rows 36 banks apart
constexpr int LDC = 64 + 4;   // LDS row of a result tile

// Four elements from p, `have` of them inside the operand (the rest are zero).
struct __attribute__((aligned(8))) fno_h4 { __bf16 v[4]; };
__device__ __forceinline__ float4 ld_quad(const float* p, int have) {
    return make_float4(have > 0 ? p[0] : 0.f, have > 1 ? p[1] : 0.f, have > 2 ? p[2] : 0.f, have > 3 ? p[3] : 0.f);
}
__device__ __forceinline__ fno_h4 ld_quad(const __bf16* p, int have) {
    fno_h4 q;
#pragma unroll
    for (int j = 0; j < 4; j++) q.v[j] = (j < have) ? p[j] : (__bf16)0.0f;
    return q;
}

// One thread's part of a 64 × KB slab: k-contiguous, rows tid/16 + 16i, k quad
// tid%16; row-contiguous, k = 4(tid/16) + i, row quad tid%16 (a 4×4 block,
// transposed on its way to LDS).
struct Slab {
    float4 f[4];
    fno_h4 h[4];
    bool zero;  // this thread's k lie past the end
};
// Where extents and alignment are whole quads (vec, and kend, nrow multiples of
// 4) the loads have no branch around them, so all of a slab are in flight: a
// row past the end is read from the last one (its products are not stored), a k
// past the end from the first one and cleared before use.  With a test per quad
// a slab took twice as long.
template <class T, class Q>
__device__ __forceinline__ void slab_load_t(Q r[4], const T* p, const FnoOp& o, int row0, int nrow, int k0, int kend,
                                            bool zero) {
    const int q = threadIdx.x & 15, t = threadIdx.x >> 4;
    if (o.vec && !(kend & 3) && (o.kc || !(nrow & 3))) {
        if (o.kc) {
            p += zero ? k0 : k0 + 4 * q;
#pragma unroll
            for (int i = 0; i < 4; i++) r[i] = *reinterpret_cast<const Q*>(p + min(row0 + t + 16 * i, nrow - 1) * o.s_row);
        } else {
            p += min(row0 + 4 * q, nrow - 4) + (zero ? k0 : k0 + 4 * t) * o.s_k;
#pragma unroll
            for (int i = 0; i < 4; i++) r[i] = *reinterpret_cast<const Q*>(p + i * o.s_k);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int row = o.kc ? row0 + t + 16 * i : row0 + 4 * q;
        const int k = o.kc ? k0 + 4 * q : k0 + 4 * t + i;
        const int have = (row < nrow && k < kend) ? (o.kc ? kend - k : nrow - row) : 0;
        r[i] = ld_quad(p + row * o.s_row + k * o.s_k, have);
    }
}
__device__ __forceinline__ void slab_load(Slab& r, const FnoOp& o, long long boff, int row0, int nrow, int k0, int kend) {
    r.zero = k0 + 4 * (int)(o.kc ? threadIdx.x & 15 : threadIdx.x >> 4) >= kend;
    if (o.bf)
        slab_load_t(r.h, (const __bf16*)o.p + boff, o, row0, nrow, k0, kend, r.zero);
    else
        slab_load_t(r.f, (const float*)o.p + boff, o, row0, nrow, k0, kend, r.zero);
}
__device__ __forceinline__ void slab_store(Slab& r, const FnoOp& o, __bf16 (*S)[LDB], float4& rs) {
    const int q = threadIdx.x & 15, t = threadIdx.x >> 4;
    if (!o.bf) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (r.zero) r.f[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            rs.x += r.f[i].x;
            rs.y += r.f[i].y;
            rs.z += r.f[i].z;
            rs.w += r.f[i].w;
            r.h[i].v[0] = (__bf16)r.f[i].x;
            r.h[i].v[1] = (__bf16)r.f[i].y;
            r.h[i].v[2] = (__bf16)r.f[i].z;
            r.h[i].v[3] = (__bf16)r.f[i].w;
        }
    } else if (r.zero) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) r.h[i].v[j] = (__bf16)0.0f;
    }
    if (o.kc) {
#pragma unroll
        for (int i = 0; i < 4; i++) *reinterpret_cast<fno_h4*>(&S[t + 16 * i][4 * q]) = r.h[i];
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            fno_h4 c;
#pragma unroll
            for (int i = 0; i < 4; i++) c.v[i] = r.h[i].v[j];
            *reinterpret_cast<fno_h4*>(&S[4 * q + j][4 * t]) = c;
        }
    }
}

__global__ __launch_bounds__(FNO_T) void fno_gemm(GemmGroup grp) {
    __shared__ __attribute__((aligned(16))) __bf16 AB[2][64][LDB];  // the B tile as [n][k]
    __bf16(*As)[LDB] = AB[0], (*Bs)[LDB] = AB[1];
    float(*Cs)[LDC] = reinterpret_cast<float(*)[LDC]>(&AB[0][0][0]);  // the result, once the operands are used
    int blk = blockIdx.x, gi = 0;
    while (gi + 1 < grp.n && blk >= grp.g[gi].nblk) blk -= grp.g[gi++].nblk;
    const GemmArgs& g = grp.g[gi];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int bx = blk % g.gx, by = (blk / g.gx) % g.gy, bz = blk / (g.gx * g.gy);
    const int n0 = bx * 64, m0 = by * 64, b = bz / g.ksplit, ks = bz % g.ksplit;
    const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
    const int lr = lane & 15, lq = lane >> 4;
    fno_f4 acc[2][2][2];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[p][i][j] = (fno_f4){0.f, 0.f, 0.f, 0.f};
    float4 rs = make_float4(0.f, 0.f, 0.f, 0.f), unused = rs;
    const bool want_rs = g.rowsum && bx == 0;
    Slab ra, rb;
#pragma unroll
    for (int p = 0; p < 2; p++) {
        if (p >= g.np) break;
        const int kbeg = ks * g.kchunk, kend = min(g.K[p], (p == 0 && g.ksplit > 1) ? kbeg + g.kchunk : g.K[p]);
        const FnoOp &oa = g.A[p], &ob = g.B[p];
        const long long ba = (long long)b * oa.s_b, bb = (long long)b * ob.s_b;
        if (p == 0) {
            slab_load(ra, oa, ba, m0, g.M, kbeg, kend);
            slab_load(rb, ob, bb, n0, g.N, kbeg, kend);
        }
        for (int k0 = kbeg; k0 < kend; k0 += KB) {
            slab_store(ra, oa, As, rs);
            slab_store(rb, ob, Bs, unused);
            __syncthreads();
            if (k0 + KB < kend) {
                slab_load(ra, oa, ba, m0, g.M, k0 + KB, kend);
                slab_load(rb, ob, bb, n0, g.N, k0 + KB, kend);
            } else if (p + 1 < g.np) {  // the second product's first slab
                slab_load(ra, g.A[1], (long long)b * g.A[1].s_b, m0, g.M, 0, g.K[1]);
                slab_load(rb, g.B[1], (long long)b * g.B[1].s_b, n0, g.N, 0, g.K[1]);
            }
#pragma unroll
            for (int s2 = 0; s2 < KB / 32; s2++) {
                fno_bf8 af[2], bfr[2];
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    af[t] = *(const fno_bf8*)&As[wm + 16 * t + lr][32 * s2 + 8 * lq];
                    bfr[t] = *(const fno_bf8*)&Bs[wn + 16 * t + lr][32 * s2 + 8 * lq];
                }
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        acc[p][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfr[j], acc[p][i][j], 0, 0, 0);
            }
            __syncthreads();
        }
    }
    const long long MN = (long long)g.M * g.N;
    const int q = tid & 15, t = tid >> 4;
    if (want_rs) {  // the 16 k groups of each row, in order
        float* red = reinterpret_cast<float*>(&AB[0][0][0]);  // [16][64]
        *reinterpret_cast<float4*>(&red[64 * t + 4 * q]) = rs;
        __syncthreads();
        if (tid < 64 && m0 + tid < g.M) {
            float v = 0.f;
#pragma unroll
            for (int k = 0; k < 16; k++) v += red[64 * k + tid];
            if (g.ksplit > 1)
                g.work[(long long)g.ksplit * MN + (long long)ks * g.M + m0 + tid] = v;
            else
                g.rowsum[m0 + tid] = v;
        }
        __syncthreads();
    }
    // through LDS, so that a thread has four consecutive n: 16-byte stores
    // (4-byte ones in the accumulator layout: 11.8 µs where 8 MB are written, now 9.0)
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float o = acc[0][i][j][r];
                if (g.np > 1) o = (g.sign < 0.f) ? o - acc[1][i][j][r] : acc[1][i][j][r] + o;
                Cs[wm + 16 * i + 4 * lq + r][wn + 16 * j + lr] = o;
            }
    __syncthreads();
    const int n = n0 + 4 * q, have = g.N - n;
    if (have <= 0) return;
    const bool split = g.ksplit > 1, vec = g.cvec && have >= 4;
    float* C = split ? g.work + bz * MN : g.C + (long long)b * g.sc_b;
    const long long ld = split ? g.N : g.sc_m;
    float bn[4] = {0.f, 0.f, 0.f, 0.f};
    if (g.bias) {
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (j < have) bn[j] = g.bias[n + j];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int ml = t + 16 * i, m = m0 + ml;
        if (m >= g.M) break;
        const long long ci = m * ld + n;
        float4 o = *reinterpret_cast<const float4*>(&Cs[ml][4 * q]);
        if (vec) {
            if (g.bias) {
                o.x += bn[0];
                o.y += bn[1];
                o.z += bn[2];
                o.w += bn[3];
            }
            if (g.zref) {
                const float4 z = *reinterpret_cast<const float4*>(g.zref + (C - g.C) + ci);
                o.x *= gelu_d(z.x);
                o.y *= gelu_d(z.y);
                o.z *= gelu_d(z.z);
                o.w *= gelu_d(z.w);
            }
            *reinterpret_cast<float4*>(C + ci) = o;
            if (g.gelu_out)
                *reinterpret_cast<float4*>(g.gelu_out + (C - g.C) + ci) =
                    make_float4(gelu_f(o.x), gelu_f(o.y), gelu_f(o.z), gelu_f(o.w));
        } else {
            for (int j = 0; j < 4 && j < have; j++) {
                float v = Cs[ml][4 * q + j];
                if (g.bias) v += g.bias[n + j];
                if (g.zref) v *= gelu_d(g.zref[(C - g.C) + ci + j]);
                C[ci + j] = v;
                if (g.gelu_out) g.gelu_out[(C - g.C) + ci + j] = gelu_f(v);
            }
        }
    }
}

// The k ranges of 32 outputs per workgroup: eight groups of threads take the
// ranges part, part + 8, ... of each output in order (independent loads, so
// many are in flight), and the eight group sums are added in a fixed tree.
constexpr int RED_OUT = 32, RED_PART = FNO_T / RED_OUT;
static_assert(RED_PART == 8, "the reduction tree below adds eight group sums");
__device__ __forceinline__ float red_sum(const float* w, long long stride, int n, bool live, float (*red)[RED_OUT + 1]) {
    const int ol = threadIdx.x % RED_OUT, part = threadIdx.x / RED_OUT;
    float s = 0.0f;
    if (live) {
#pragma unroll 8
        for (int ks = part; ks < n; ks += RED_PART) s += w[(long long)ks * stride];
    }
    red[part][ol] = s;
    __syncthreads();
    return ((red[0][ol] + red[1][ol]) + (red[2][ol] + red[3][ol])) +
           ((red[4][ol] + red[5][ol]) + (red[6][ol] + red[7][ol]));
}
static inline int red_blocks(const GemmArgs& g) {
    if (g.ksplit <= 1) return 0;
    return (int)(((long long)g.M * g.N * g.batch + (g.rowsum ? g.M : 0) + RED_OUT - 1) / RED_OUT);
}
__global__ __launch_bounds__(FNO_T) void fno_splitk_reduce(GemmGroup grp, int blk1, int blk2) {
    __shared__ float red[RED_PART][RED_OUT + 1];
    const int gi = ((int)blockIdx.x >= blk2) ? 2 : ((int)blockIdx.x >= blk1) ? 1 : 0;
    const int blk = blockIdx.x - (gi == 2 ? blk2 : gi == 1 ? blk1 : 0);
    const GemmArgs& g = grp.g[gi];
    const long long MN = (long long)g.M * g.N, all = MN * g.batch;
    const long long idx = (long long)blk * RED_OUT + threadIdx.x % RED_OUT;
    const bool prod = idx < all, row = !prod && g.rowsum && idx < all + g.M;
    const int b = prod ? (int)(idx / MN) : 0;
    const long long rem = idx - (long long)b * MN;
    const float* w = prod ? g.work + (long long)b * g.ksplit * MN + rem
                          : g.work + (long long)g.ksplit * all + (idx - all);
    const float t = red_sum(w, prod ? MN : g.M, g.ksplit, prod || row, red);
    if (threadIdx.x >= RED_OUT) return;
    if (prod) {
        const int m = (int)(rem / g.N), n = (int)(rem - (long long)m * g.N);
        g.C[(long long)b * g.sc_b + (long long)m * g.sc_m + n] = t;
    } else if (row)
        g.rowsum[idx - all] = t;
}

// ---------------------------------------------------------------------------
// Projection head on FP32 matrix cores: z1 = v Q1ᵀ + bq1, y = gelu(z1)·Q2 + bq2.
// Tile 64×64, K slab 32, v_mfma_f32_16x16x4f32 (lane l supplies A[l%16][l/16]
// and B[l/16][l%16]; accumulator register r of lane l is D[4(l/16)+r][l%16]).
// The hidden activations and their gradients exist only inside these kernels;
// z1 is the one array that the backward pass reads again.
// ---------------------------------------------------------------------------
constexpr int HB = 32;
constexpr int LDH = HB + 4;

// d = y - t;  loss = Σ w d² / n;  dy = 2 w d / n
struct HeadLoss {
    const float *y, *t, *w;
    float n;
    __device__ __forceinline__ float dy(long long i, float& wdd) const {
        const float d = y[i] - t[i], wi = w ? w[i] : 1.0f;
        wdd = wi * d * d;
        return 2.0f * wi * d / n;
    }
};

// A thread's two quads of a 64 × 32 slab: k-contiguous, rows tid/8 + 32i, k
// quad tid%8; row-contiguous, k = 2(tid/16) + i, row quad tid%16.  All extents
// are multiples of 32 along the quads.
__device__ __forceinline__ void head_load_k(float4 r[2], const float* p, long long ld, long long row0, long long nrow, int k0) {
    const int q = threadIdx.x & 7, t = threadIdx.x >> 3;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const long long row = row0 + t + 32 * i;
        r[i] = (row < nrow) ? *reinterpret_cast<const float4*>(p + row * ld + k0 + 4 * q) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
}
__device__ __forceinline__ void head_store_k(const float4 r[2], float (*S)[LDH]) {
    const int q = threadIdx.x & 7, t = threadIdx.x >> 3;
#pragma unroll
    for (int i = 0; i < 2; i++) *reinterpret_cast<float4*>(&S[t + 32 * i][4 * q]) = r[i];
}
__device__ __forceinline__ void head_load_r(float4 r[2], const float* p, long long ld, int row0, int nrow, long long k0, long long kend) {
    const int q = threadIdx.x & 15, t = threadIdx.x >> 4;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const long long k = k0 + 2 * t + i;
        r[i] = (k < kend && row0 + 4 * q < nrow) ? *reinterpret_cast<const float4*>(p + k * ld + row0 + 4 * q)
                                                 : make_float4(0.f, 0.f, 0.f, 0.f);
    }
}
__device__ __forceinline__ void head_store_r(const float4 r[2], float (*S)[LDH]) {
    const int q = threadIdx.x & 15, t = threadIdx.x >> 4;
    *reinterpret_cast<float2*>(&S[4 * q + 0][2 * t]) = make_float2(r[0].x, r[1].x);
    *reinterpret_cast<float2*>(&S[4 * q + 1][2 * t]) = make_float2(r[0].y, r[1].y);
    *reinterpret_cast<float2*>(&S[4 * q + 2][2 * t]) = make_float2(r[0].z, r[1].z);
    *reinterpret_cast<float2*>(&S[4 * q + 3][2 * t]) = make_float2(r[0].w, r[1].w);
}
__device__ __forceinline__ void head_mfma(fno_f4 acc[2][2], float (*As)[LDH], float (*Bs)[LDH]) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32, lr = lane & 15, lq = lane >> 4;
#pragma unroll
    for (int s4 = 0; s4 < HB / 4; s4++) {
        float af[2], bfr[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            af[t] = As[wm + 16 * t + lr][4 * s4 + lq];
            bfr[t] = Bs[wn + 16 * t + lr][4 * s4 + lq];
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i], bfr[j], acc[i][j], 0, 0, 0);
    }
}
__device__ __forceinline__ void head_zero(fno_f4 acc[2][2]) {
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = (fno_f4){0.f, 0.f, 0.f, 0.f};
}

// A 64×64 result tile from LDS to out, `have` of its columns (a multiple of 32).
__device__ __forceinline__ void head_out(float (*Cs)[LDC], float* out, long long ld, int have) {
    const int q = threadIdx.x & 15, t = threadIdx.x >> 4;
    if (4 * q >= have) return;
#pragma unroll
    for (int i = 0; i < 4; i++)
        *reinterpret_cast<float4*>(out + (t + 16 * i) * ld + 4 * q) = *reinterpret_cast<const float4*>(&Cs[t + 16 * i][4 * q]);
}

// 64 rows per workgroup, all hidden units in blocks of 64; Z1 may be null.
__global__ __launch_bounds__(FNO_T) void fno_head_fwd(const float* __restrict__ V, int C, int H, const float* __restrict__ Q1,
                                                      const float* __restrict__ bq1, const float* __restrict__ Q2,
                                                      const float* __restrict__ bq2, float* __restrict__ Z1,
                                                      float* __restrict__ y) {
    __shared__ __attribute__((aligned(16))) float AB[2][64][LDH];
    float(*As)[LDH] = AB[0], (*Bs)[LDH] = AB[1], (*Cs)[LDC] = reinterpret_cast<float(*)[LDC]>(&AB[0][0][0]);
    __shared__ float ys[2][64];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const long long r0 = (long long)blockIdx.x * 64, rows = (long long)gridDim.x * 64;
    const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32, lr = lane & 15, lq = lane >> 4;
    float yp[2][4] = {};
    float4 ra[2], rb[2];
    head_load_k(ra, V, C, r0, rows, 0);
    head_load_k(rb, Q1, C, 0, H, 0);
    for (int h0 = 0; h0 < H; h0 += 64) {
        fno_f4 acc[2][2];
        head_zero(acc);
        for (int k0 = 0; k0 < C; k0 += HB) {
            head_store_k(ra, As);
            head_store_k(rb, Bs);
            __syncthreads();
            const bool more = k0 + HB < C;
            if (more || h0 + 64 < H) {
                head_load_k(ra, V, C, r0, rows, more ? k0 + HB : 0);
                head_load_k(rb, Q1, C, more ? h0 : h0 + 64, H, more ? k0 + HB : 0);
            }
            head_mfma(acc, As, Bs);
            __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int n = h0 + wn + 16 * j + lr;
            if (n >= H) continue;
            const float bn = bq1[n], q2 = Q2[n];
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float z = acc[i][j][r] + bn;
                    if (Z1) Cs[wm + 16 * i + 4 * lq + r][n - h0] = z;
                    yp[i][r] += gelu_f(z) * q2;
                }
        }
        if (Z1) {
            __syncthreads();
            head_out(Cs, Z1 + r0 * H + h0, H, H - h0);
            __syncthreads();
        }
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float v = yp[i][r];
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o);
            if (lr == 0) ys[wave >> 1][wm + 16 * i + 4 * lq + r] = v;
        }
    __syncthreads();
    if (tid < 64) y[r0 + tid] = (ys[0][tid] + ys[1][tid]) + bq2[0];
}

// dv = dz1 · Q1 with dz1[i][j] = dy[i] · Q2[j] · gelu'(z1[i][j]); 64 rows × 64 channels.
__global__ __launch_bounds__(FNO_T) void fno_head_dv(HeadLoss ls, const float* __restrict__ Z1, int H, int C,
                                                     const float* __restrict__ Q1, const float* __restrict__ Q2,
                                                     float* __restrict__ dV) {
    __shared__ __attribute__((aligned(16))) float AB[2][64][LDH];
    float(*As)[LDH] = AB[0], (*Bs)[LDH] = AB[1], (*Cs)[LDC] = reinterpret_cast<float(*)[LDC]>(&AB[0][0][0]);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const long long r0 = (long long)blockIdx.x * 64, rows = (long long)gridDim.x * 64;
    const int n0 = blockIdx.y * 64;
    const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32, lr = lane & 15, lq = lane >> 4;
    float dy[2], unused;
#pragma unroll
    for (int i = 0; i < 2; i++) dy[i] = ls.dy(r0 + (tid >> 3) + 32 * i, unused);
    fno_f4 acc[2][2];
    head_zero(acc);
    float4 ra[2], rb[2];
    head_load_k(ra, Z1, H, r0, rows, 0);
    head_load_r(rb, Q1, C, n0, C, 0, H);
    for (int k0 = 0; k0 < H; k0 += HB) {
        const float4 q2 = *reinterpret_cast<const float4*>(Q2 + k0 + 4 * (tid & 7));
#pragma unroll
        for (int i = 0; i < 2; i++) {
            ra[i].x = dy[i] * q2.x * gelu_d(ra[i].x);
            ra[i].y = dy[i] * q2.y * gelu_d(ra[i].y);
            ra[i].z = dy[i] * q2.z * gelu_d(ra[i].z);
            ra[i].w = dy[i] * q2.w * gelu_d(ra[i].w);
        }
        head_store_k(ra, As);
        head_store_r(rb, Bs);
        __syncthreads();
        if (k0 + HB < H) {
            head_load_k(ra, Z1, H, r0, rows, k0 + HB);
            head_load_r(rb, Q1, C, n0, C, k0 + HB, H);
        }
        head_mfma(acc, As, Bs);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) Cs[wm + 16 * i + 4 * lq + r][wn + 16 * j + lr] = acc[i][j][r];
    __syncthreads();
    head_out(Cs, dV + r0 * C + n0, C, C - n0);
}

// Partial sums over a range of rows: dQ1 = dz1ᵀ v, dbq1 = Σ dz1, dQ2 = Σ dy·gelu(z1),
// dbq2 = Σ dy and Σ w d².  part[ks] = [H·C | H | H | 1 | 1].
__global__ __launch_bounds__(FNO_T) void fno_head_dq(HeadLoss ls, const float* __restrict__ Z1, const float* __restrict__ V,
                                                     int H, int C, const float* __restrict__ Q2, long long rows, int chunk,
                                                     float* __restrict__ part) {
    __shared__ __attribute__((aligned(16))) float As[64][LDH], Bs[64][LDH];
    __shared__ float red[2][16][64];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q = tid & 15, t = tid >> 4;
    const int n0 = blockIdx.x * 64, m0 = blockIdx.y * 64;
    const long long kbeg = (long long)blockIdx.z * chunk;
    const long long kend = (kbeg + chunk < rows) ? kbeg + chunk : rows;
    const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32, lr = lane & 15, lq = lane >> 4;
    const float4 q2 = (m0 + 4 * q < H) ? *reinterpret_cast<const float4*>(Q2 + m0 + 4 * q) : make_float4(0.f, 0.f, 0.f, 0.f);
    float4 sz = make_float4(0.f, 0.f, 0.f, 0.f), sh = sz;
    float sdy = 0.f, sl = 0.f;
    fno_f4 acc[2][2];
    head_zero(acc);
    float4 ra[2], rb[2];
    float dy[2], wdd[2];
    const auto load = [&](long long k0) {
        head_load_r(ra, Z1, H, m0, H, k0, kend);
        head_load_r(rb, V, C, n0, C, k0, kend);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const long long k = k0 + 2 * t + i;
            dy[i] = wdd[i] = 0.f;
            if (k < kend) dy[i] = ls.dy(k, wdd[i]);
        }
    };
    load(kbeg);
    for (long long k0 = kbeg; k0 < kend; k0 += HB) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            sh.x += dy[i] * gelu_f(ra[i].x);
            sh.y += dy[i] * gelu_f(ra[i].y);
            sh.z += dy[i] * gelu_f(ra[i].z);
            sh.w += dy[i] * gelu_f(ra[i].w);
            ra[i].x = dy[i] * q2.x * gelu_d(ra[i].x);
            ra[i].y = dy[i] * q2.y * gelu_d(ra[i].y);
            ra[i].z = dy[i] * q2.z * gelu_d(ra[i].z);
            ra[i].w = dy[i] * q2.w * gelu_d(ra[i].w);
            sz.x += ra[i].x;
            sz.y += ra[i].y;
            sz.z += ra[i].z;
            sz.w += ra[i].w;
            sdy += dy[i];
            sl += wdd[i];
        }
        head_store_r(ra, As);
        head_store_r(rb, Bs);
        __syncthreads();
        if (k0 + HB < kend) load(k0 + HB);
        head_mfma(acc, As, Bs);
        __syncthreads();
    }
    float* out = part + (long long)blockIdx.z * ((long long)H * C + 2 * H + 2);
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + wm + 16 * i + 4 * lq + r, n = n0 + wn + 16 * j + lr;
                if (m < H && n < C) out[(long long)m * C + n] = acc[i][j][r];
            }
    if (blockIdx.x != 0) return;
    *reinterpret_cast<float4*>(&red[0][t][4 * q]) = sz;
    *reinterpret_cast<float4*>(&red[1][t][4 * q]) = sh;
    __syncthreads();
    if (tid < 128) {
        const int which = tid >> 6, m = tid & 63;
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < 16; k++) v += red[which][k][m];
        if (m0 + m < H) out[(long long)H * C + which * H + m0 + m] = v;
    }
    if (blockIdx.y != 0) return;
    __syncthreads();
    if (q == 0) {
        red[0][t][0] = sdy;
        red[1][t][0] = sl;
    }
    __syncthreads();
    if (tid < 2) {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < 16; k++) v += red[tid][k][0];
        out[(long long)H * C + 2 * H + tid] = v;
    }
}
// The parameters Q1, bq1, Q2, bq2 lie behind one another in this order, as do
// the partial sums; the last sum is the loss.
__global__ __launch_bounds__(FNO_T) void fno_head_reduce(const float* __restrict__ part, int nks, long long per,
                                                         float* __restrict__ grad, float n, float* __restrict__ loss) {
    __shared__ float red[RED_PART][RED_OUT + 1];
    const long long idx = (long long)blockIdx.x * RED_OUT + threadIdx.x % RED_OUT;
    const bool live = idx < per;
    const float s = red_sum(part + idx, per, nks, live, red);
    if (threadIdx.x >= RED_OUT || !live) return;
    if (idx < per - 1)
        grad[idx] = s;
    else
        *loss = s / n;
}

__global__ void fno_cvt_bf16(const float* __restrict__ src, __bf16* __restrict__ dst, long long n) {
    long long i = (long long)blockIdx.x * FNO_T + threadIdx.x;
    if (i < n) dst[i] = (__bf16)src[i];
}

// Rblk[m] = [[Rre, Rim], [-Rim, Rre]] (2C × 2C, rows: re/im of the input
// channel, columns: re/im of the output channel), so that one real product
// [Vre, Vim] · Rblk gives [Re(V R), Im(V R)].
__global__ void fno_build_rblk(const float* __restrict__ Rre, const float* __restrict__ Rim, __bf16* __restrict__ Rblk,
                               int C, int modes) {
    const long long n = (long long)modes * 4 * C * C;
    long long i = (long long)blockIdx.x * FNO_T + threadIdx.x;
    if (i >= n) return;
    const int C2 = 2 * C;
    const int m = (int)(i / ((long long)C2 * C2));
    const int rem = (int)(i - (long long)m * C2 * C2);
    const int kr = rem / C2, nc = rem % C2;
    const long long base = (long long)m * C * C;
    float v;
    if (kr < C && nc < C)
        v = Rre[base + kr * C + nc];
    else if (kr < C)
        v = Rim[base + kr * C + (nc - C)];
    else if (nc < C)
        v = -Rim[base + (kr - C) * C + nc];
    else
        v = Rre[base + (kr - C) * C + (nc - C)];
    Rblk[i] = (__bf16)v;
}

// AdamW on the FP32 master copy; refreshes the BF16 copy.
__global__ void fno_adamw(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                          float* __restrict__ v, __bf16* __restrict__ pbf, long long n, const float* __restrict__ lr_sched,
                          int step_idx, float lr0, float b1, float b2, float eps, float wd, float bc1, float bc2) {
    long long i = (long long)blockIdx.x * FNO_T + threadIdx.x;
    if (i >= n) return;
    const float lr = lr_sched ? lr_sched[step_idx] : lr0;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / bc1, vh = vi / bc2;
    const float pi = p[i] - lr * (mh / (sqrtf(vh) + eps) + wd * p[i]);
    p[i] = pi;
    pbf[i] = (__bf16)pi;
}

__global__ void fno_gather(const float* __restrict__ xs, const float* __restrict__ ts, const float* __restrict__ ws,
                           const int32_t* __restrict__ idx, float* __restrict__ xb, float* __restrict__ tb,
                           float* __restrict__ wb, int B, int X, int cin) {
    const long long per_x = (long long)X * cin;
    const long long nx = (long long)B * per_x, nt = (long long)B * X;
    long long i = (long long)blockIdx.x * FNO_T + threadIdx.x;
    if (i < nx) {
        const int b = (int)(i / per_x);
        xb[i] = xs[(long long)idx[b] * per_x + (i - (long long)b * per_x)];
    }
    if (i < nt) {
        const int b = (int)(i / X);
        const long long src = (long long)idx[b] * X + (i - (long long)b * X);
        tb[i] = ts[src];
        if (ws) wb[i] = ws[src];
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
struct FnoLayout {
    long long P, bP, W[FNO_MAXL], b[FNO_MAXL], Rre[FNO_MAXL], Rim[FNO_MAXL], Q1, bq1, Q2, bq2, total;
};

struct lh_fno {
    lh_fno_cfg cfg;
    int device;
    hipStream_t stream;
    hipStream_t copy_stream;     // targets in, gradients out, beside the kernels of lh_fno_loss_grad
    hipEvent_t ready[FNO_MAXL + 1];  // gradients of layer l, of the head
    hipEvent_t targets;
    FnoLayout L;
    float* params;
    float* grads;
    float* adam_m;
    float* adam_v;
    __bf16* pbf;
    __bf16* Rblk;  // [layers][modes][2C][2C]
    __bf16* F;     // [2·modes][n_x]
    __bf16* Ginv;  // [n_x][2·modes]
    float* xb;
    float* tb;
    float* wb;       // loss weights of the batch
    const float* wcur;  // wb, or null for unit weights
    float* V[FNO_MAXL];     // layer inputs v_0 .. v_{L-1}
    float* Z[FNO_MAXL];     // pre-activations z_0 .. z_{L-1}  (v_L = z_{L-1})
    float* Vhat[FNO_MAXL];  // [B][2·modes][C]
    float* Ohat;
    float* Z1;
    float* y;
    float* dVa;
    float* dVb;
    float* dOhat;
    float* dVhat;
    float* work;
    long long work_cap;
    float* loss_dev;  // [max steps per train call]
    int loss_cap;
    float* data_x;
    float* data_t;
    float* data_w;
    int data_n;
    int32_t* idx_dev;
    long long idx_cap;
    float* lr_dev;
    long long adam_t;
    std::vector<std::pair<const char*, size_t>>* allocs;  // every device buffer (base, bytes)
};

// Host-side bounds check of a strided operand before any launch: the largest
// element offset must stay inside the allocation the pointer points into.
static bool fno_in_bounds(const lh_fno* f, const void* p, long long max_off, size_t esize) {
    if (!p || max_off < 0) return false;
    const char* c = (const char*)p;
    for (const auto& a : *f->allocs)
        if (c >= a.first && c < a.first + a.second) return c + (size_t)(max_off + 1) * esize <= a.first + a.second;
    return false;
}

static FnoLayout fno_layout(const lh_fno_cfg& c) {
    FnoLayout L;
    memset(&L, 0, sizeof(L));
    const long long C = c.channels, H = c.hidden, Mo = c.modes;
    long long o = 0;
    L.P = o; o += C * c.cin;
    L.bP = o; o += C;
    for (int l = 0; l < c.layers; l++) {
        L.W[l] = o; o += C * C;
        L.b[l] = o; o += C;
        L.Rre[l] = o; o += Mo * C * C;
        L.Rim[l] = o; o += Mo * C * C;
    }
    L.Q1 = o; o += H * C;
    L.bq1 = o; o += H;
    L.Q2 = o; o += H;
    L.bq2 = o; o += 1;
    L.total = o;
    return L;
}

static inline unsigned nblk(long long n) { return (unsigned)((n + FNO_T - 1) / FNO_T); }

static FnoOp op(const float* p, long long s_row, long long s_k, long long s_b) {
    return FnoOp{p, s_row, s_k, s_b, 0, s_k == 1, 0};
}
static FnoOp op(const __bf16* p, long long s_row, long long s_k, long long s_b) {
    return FnoOp{p, s_row, s_k, s_b, 1, s_k == 1, 0};
}

static GemmArgs G(int M, int N, int batch, int K, FnoOp A, FnoOp B, float* C, long long sc_m, long long sc_b) {
    GemmArgs g;
    memset(&g, 0, sizeof(g));
    g.M = M; g.N = N; g.batch = batch; g.np = 1; g.sign = 1.0f;
    g.K[0] = K; g.A[0] = A; g.B[0] = B;
    g.C = C; g.sc_m = sc_m; g.sc_b = sc_b;
    return g;
}
// ± a second product with the same output
static GemmArgs G2(GemmArgs g, float sign, int K, FnoOp A, FnoOp B) {
    g.np = 2; g.sign = sign; g.K[1] = K; g.A[1] = A; g.B[1] = B;
    return g;
}

// Checks one operand of rows × K × batch and chooses its load width.
static bool op_ok(const lh_fno* f, FnoOp& o, long long rows, long long K, long long batch) {
    if (rows < 1 || K < 1 || o.s_row < 0 || o.s_k < 0 || o.s_b < 0 || (o.s_k != 1 && o.s_row != 1)) return false;
    if (!fno_in_bounds(f, o.p, (batch - 1) * o.s_b + (rows - 1) * o.s_row + (K - 1) * o.s_k, o.bf ? 2 : 4)) return false;
    const long long other = o.kc ? o.s_row : o.s_k;
    o.vec = other % 4 == 0 && o.s_b % 4 == 0 && (uintptr_t)o.p % (o.bf ? 8 : 16) == 0;
    return true;
}

// Launch a group of up to three independent products.
static int fno_launch(lh_fno* f, std::initializer_list<GemmArgs> gs) {
    GemmGroup grp;
    memset(&grp, 0, sizeof(grp));
    if (gs.size() < 1 || gs.size() > 3) return LH_E_ARG;
    for (const GemmArgs& g : gs) grp.g[grp.n++] = g;
    const long long cap = f->work_cap / grp.n & ~3LL;
    long long blocks = 0, red[3] = {0, 0, 0};
    for (int i = 0; i < grp.n; i++) {
        GemmArgs& g = grp.g[i];
        bool ok = g.M >= 1 && g.N >= 1 && g.batch >= 1 && g.sc_m >= 0 && g.sc_b >= 0;
        for (int p = 0; p < g.np && ok; p++)
            ok = op_ok(f, g.A[p], g.M, g.K[p], g.batch) && op_ok(f, g.B[p], g.N, g.K[p], g.batch);
        const long long cmax = (g.batch - 1) * g.sc_b + (g.M - 1) * g.sc_m + (g.N - 1);
        ok = ok && fno_in_bounds(f, g.C, cmax, 4) && (!g.bias || fno_in_bounds(f, g.bias, g.N - 1, 4)) &&
             (!g.gelu_out || fno_in_bounds(f, g.gelu_out, cmax, 4)) && (!g.zref || fno_in_bounds(f, g.zref, cmax, 4)) &&
             (!g.rowsum || (fno_in_bounds(f, g.rowsum, g.M - 1, 4) && g.batch == 1 && !g.A[0].kc && !g.A[0].bf));
        if (!ok) {
            fprintf(stderr, "luna_fno: GEMM operand out of bounds (M=%d N=%d K=%d batch=%d)\n", g.M, g.N, g.K[0], g.batch);
            return LH_E_ARG;
        }
        const long long tiles = (long long)g.batch * ((g.M + 63) / 64) * ((g.N + 63) / 64);
        int ksplit = 1;
        if (tiles < 256 && g.K[0] >= 1024 && g.np == 1 && !g.bias && !g.gelu_out && !g.zref) {
            // at least ~512 workgroups (two per CU) in k ranges of at least 128
            const long long want = 512 / tiles, maxk = (g.K[0] + 127) / 128;
            ksplit = (int)(want < maxk ? want : maxk);
            while (ksplit > 1 && ksplit * ((long long)g.batch * g.M * g.N + g.M) > cap) ksplit--;
        }
        g.kchunk = ((g.K[0] + ksplit - 1) / ksplit + 31) / 32 * 32;
        g.ksplit = (g.K[0] + g.kchunk - 1) / g.kchunk;
        g.work = f->work + i * cap;
        const uintptr_t all = (uintptr_t)g.C | (uintptr_t)g.gelu_out | (uintptr_t)g.zref | (uintptr_t)g.work;
        g.cvec = all % 16 == 0 && g.N % 4 == 0 && g.sc_m % 4 == 0 && g.sc_b % 4 == 0;
        g.gx = (g.N + 63) / 64;
        g.gy = (g.M + 63) / 64;
        const long long nb = (long long)g.gx * g.gy * g.batch * g.ksplit;
        if (nb > 0x7fffffff - blocks) return LH_E_ARG;
        g.nblk = (int)nb;
        blocks += nb;
        red[i] = red_blocks(g);
    }
    hipLaunchKernelGGL(fno_gemm, dim3((unsigned)blocks), dim3(FNO_T), 0, f->stream, grp);
    if (red[0] + red[1] + red[2] > 0)
        hipLaunchKernelGGL(fno_splitk_reduce, dim3((unsigned)(red[0] + red[1] + red[2])), dim3(FNO_T), 0, f->stream, grp,
                           (int)red[0], (int)(red[0] + red[1]));
    FNOCK(hipGetLastError());
    return LH_OK;
}

static void refresh_bf16(lh_fno* f) {
    const lh_fno_cfg& c = f->cfg;
    hipLaunchKernelGGL(fno_cvt_bf16, dim3(nblk(f->L.total)), dim3(FNO_T), 0, f->stream, f->params, f->pbf, f->L.total);
    const long long rb = (long long)c.modes * 4 * c.channels * c.channels;
    for (int l = 0; l < c.layers; l++)
        hipLaunchKernelGGL(fno_build_rblk, dim3(nblk(rb)), dim3(FNO_T), 0, f->stream, f->params + f->L.Rre[l],
                           f->params + f->L.Rim[l], f->Rblk + (long long)l * rb, c.channels, c.modes);
}

// Forward pass on f->xb (batch B) → f->y; keeps every activation for backward.
static int fno_forward_dev(lh_fno* f, int B, bool keep) {
    const lh_fno_cfg& c = f->cfg;
    const int X = c.n_x, C = c.channels, Mo2 = 2 * c.modes, H = c.hidden, cin = c.cin;
    const long long BX = (long long)B * X, XC = (long long)X * C, MC = (long long)Mo2 * C;
    const FnoLayout& L = f->L;
    const __bf16* pb = f->pbf;
    const float* pf = f->params;
    const long long rb = (long long)c.modes * 4 * C * C;
    // lift: v0 = x Pᵀ + bP
    GemmArgs g = G((int)BX, C, 1, cin, op(f->xb, cin, 1, 0), op(pb + L.P, cin, 1, 0), f->V[0], C, 0);
    g.bias = pf + L.bP;
    int st = fno_launch(f, {g});
    for (int l = 0; l < c.layers && !st; l++) {
        const float* v = f->V[l];
        // Vhat_b = F · v_b                              [2·modes × C] per sample
        st = fno_launch(f, {G(Mo2, C, B, X, op(f->F, X, 1, 0), op(v, 1, C, XC), f->Vhat[l], C, MC)});
        // per mode: [B × 2C] · Rblk[m] (2C × 2C)
        if (!st)
            st = fno_launch(f, {G(B, 2 * C, c.modes, 2 * C, op(f->Vhat[l], MC, 1, 2 * C),
                                  op(f->Rblk + (long long)l * rb, 1, 2 * C, 4LL * C * C), f->Ohat, MC, 2 * C)});
        // z_b = Ginv · Ohat_b + v_b Wᵀ + b, next layer's input gelu(z)
        g = G2(G(X, C, B, Mo2, op(f->Ginv, Mo2, 1, 0), op(f->Ohat, 1, C, MC), f->Z[l], C, XC), 1.0f, C, op(v, C, 1, XC),
               op(pb + L.W[l], C, 1, 0));
        g.bias = pf + L.b[l];
        if (l + 1 < c.layers) g.gelu_out = f->V[l + 1];
        if (!st) st = fno_launch(f, {g});
    }
    if (st) return st;
    hipLaunchKernelGGL(fno_head_fwd, dim3((unsigned)(BX / 64)), dim3(FNO_T), 0, f->stream, f->Z[c.layers - 1], C, H,
                       pf + L.Q1, pf + L.bq1, pf + L.Q2, pf + L.bq2, keep ? f->Z1 : nullptr, f->y);
    FNOCK(hipGetLastError());
    return LH_OK;
}

// Loss against f->tb and the full gradient into f->grads; loss → *loss_out (device).
static int fno_backward_dev(lh_fno* f, int B, float* loss_out) {
    const lh_fno_cfg& c = f->cfg;
    const int X = c.n_x, C = c.channels, Mo2 = 2 * c.modes, H = c.hidden, cin = c.cin;
    const long long BX = (long long)B * X, XC = (long long)X * C, MC = (long long)Mo2 * C, CC = (long long)C * C;
    const FnoLayout& L = f->L;
    const __bf16* pb = f->pbf;
    const float* pf = f->params;
    float* gr = f->grads;
    const long long rb = 4 * CC * c.modes;
    hipStream_t s = f->stream;
    const float* vL = f->Z[c.layers - 1];
    // loss and projection head
    const HeadLoss ls{f->y, f->tb, f->wcur, (float)BX};
    const long long per = (long long)H * C + 2 * H + 2;
    const unsigned hx = (C + 63) / 64, hy = (H + 63) / 64;
    long long nks = 512 / ((long long)hx * hy);  // two workgroups per CU, at least 128 rows each
    if (nks > (BX + 127) / 128) nks = (BX + 127) / 128;
    if (nks > f->work_cap / per) nks = f->work_cap / per;
    if (nks < 1) nks = 1;
    const int chunk = (int)(((BX + nks - 1) / nks + HB - 1) / HB * HB);
    nks = (BX + chunk - 1) / chunk;
    if (nks * per > f->work_cap) return LH_E_ARG;
    hipLaunchKernelGGL(fno_head_dq, dim3(hx, hy, (unsigned)nks), dim3(FNO_T), 0, s, ls, f->Z1, vL, H, C, pf + L.Q2, BX,
                       chunk, f->work);
    hipLaunchKernelGGL(fno_head_reduce, dim3((unsigned)((per + RED_OUT - 1) / RED_OUT)), dim3(FNO_T), 0, s, f->work,
                       (int)nks, per, gr + L.Q1, (float)BX, loss_out);
    FNOCK(hipEventRecord(f->ready[c.layers], s));
    float* dz = f->dVa;  // gradient w.r.t. the current layer's pre-activation
    float* dn = f->dVb;
    hipLaunchKernelGGL(fno_head_dv, dim3((unsigned)(BX / 64), hx), dim3(FNO_T), 0, s, ls, f->Z1, H, C, pf + L.Q1,
                       pf + L.Q2, dz);
    FNOCK(hipGetLastError());
    int st = LH_OK;
    for (int l = c.layers - 1; l >= 0 && !st; l--) {
        const float* v = f->V[l];
        // dW = dzᵀ v, db = Σ dz;  dOhat_b = Ginvᵀ dz_b
        GemmArgs g = G(C, C, 1, (int)BX, op(dz, 1, C, 0), op(v, 1, C, 0), gr + L.W[l], C, 0);
        g.rowsum = gr + L.b[l];
        st = fno_launch(f, {g, G(Mo2, C, B, X, op(f->Ginv, 1, Mo2, 0), op(dz, 1, C, XC), f->dOhat, C, MC)});
        // per mode: dRre = Vreᵀ dOre + Vimᵀ dOim, dRim = Vreᵀ dOim − Vimᵀ dOre;
        // dVblk = dOblk Rblkᵀ
        const float* vh = f->Vhat[l];
        const float* dO = f->dOhat;
        if (!st)
            st = fno_launch(f, {G2(G(C, C, c.modes, B, op(vh, 1, MC, 2 * C), op(dO, 1, MC, 2 * C), gr + L.Rre[l], C, CC),
                                   1.0f, B, op(vh + C, 1, MC, 2 * C), op(dO + C, 1, MC, 2 * C)),
                                G2(G(C, C, c.modes, B, op(vh, 1, MC, 2 * C), op(dO + C, 1, MC, 2 * C), gr + L.Rim[l], C, CC),
                                   -1.0f, B, op(vh + C, 1, MC, 2 * C), op(dO, 1, MC, 2 * C)),
                                G(B, 2 * C, c.modes, 2 * C, op(dO, MC, 1, 2 * C),
                                  op(f->Rblk + (long long)l * rb, 2 * C, 1, 4 * CC), f->dVhat, MC, 2 * C)});
        if (!st) FNOCK(hipEventRecord(f->ready[l], s));
        // dv = dz W + Fᵀ dVhat, times gelu' of the layer below
        g = G2(G(X, C, B, C, op(dz, C, 1, XC), op(pb + L.W[l], 1, C, 0), dn, C, XC), 1.0f, Mo2, op(f->F, 1, X, 0),
               op(f->dVhat, 1, C, MC));
        if (l > 0) g.zref = f->Z[l - 1];
        if (!st) st = fno_launch(f, {g});
        std::swap(dz, dn);
    }
    if (st) return st;
    // lift: dP = dv0ᵀ x, dbP = Σ dv0
    GemmArgs g = G(C, cin, 1, (int)BX, op(dz, 1, C, 0), op(f->xb, 1, cin, 0), gr + L.P, cin, 0);
    g.rowsum = gr + L.bP;
    return fno_launch(f, {g});
}

static int fno_adam_step(lh_fno* f, const lh_adam* o, const float* lr_dev, int step_idx) {
    f->adam_t++;
    const float bc1 = 1.0f - powf(o->beta1, (float)f->adam_t);
    const float bc2 = 1.0f - powf(o->beta2, (float)f->adam_t);
    hipLaunchKernelGGL(fno_adamw, dim3(nblk(f->L.total)), dim3(FNO_T), 0, f->stream, f->params, f->grads, f->adam_m,
                       f->adam_v, f->pbf, f->L.total, lr_dev, step_idx, o->lr, o->beta1, o->beta2, o->eps,
                       o->weight_decay, bc1, bc2);
    const lh_fno_cfg& c = f->cfg;
    const long long rb = (long long)c.modes * 4 * c.channels * c.channels;
    for (int l = 0; l < c.layers; l++)
        hipLaunchKernelGGL(fno_build_rblk, dim3(nblk(rb)), dim3(FNO_T), 0, f->stream, f->params + f->L.Rre[l],
                           f->params + f->L.Rim[l], f->Rblk + (long long)l * rb, c.channels, c.modes);
    FNOCK(hipGetLastError());
    return LH_OK;
}

extern "C" {

int lh_fno_destroy(lh_fno* f) {
    if (!f) return LH_OK;
    hipSetDevice(f->device);
    if (f->stream) hipStreamSynchronize(f->stream);
    if (f->copy_stream) hipStreamSynchronize(f->copy_stream);
    void* ptrs[] = {f->params, f->grads, f->adam_m, f->adam_v, f->pbf, f->Rblk, f->F, f->Ginv, f->xb, f->tb, f->wb,
                    f->data_w,
                    f->Ohat, f->Z1, f->y, f->dVa, f->dVb, f->dOhat, f->dVhat, f->work, f->loss_dev,
                    f->data_x, f->data_t, f->idx_dev, f->lr_dev};
    for (void* p : ptrs)
        if (p) hipFree(p);
    for (int l = 0; l < FNO_MAXL; l++) {
        if (f->V[l]) hipFree(f->V[l]);
        if (f->Z[l]) hipFree(f->Z[l]);
        if (f->Vhat[l]) hipFree(f->Vhat[l]);
    }
    for (hipEvent_t e : f->ready)
        if (e) hipEventDestroy(e);
    if (f->targets) hipEventDestroy(f->targets);
    if (f->copy_stream) hipStreamDestroy(f->copy_stream);
    if (f->stream) hipStreamDestroy(f->stream);
    delete f->allocs;
    free(f);
    return LH_OK;
}

int lh_fno_create(lh_fno** out, const lh_fno_cfg* cfg) {
    if (!out || !cfg) return LH_E_ARG;
    *out = nullptr;
    const lh_fno_cfg c = *cfg;
    if (c.n_x < 64 || c.n_x % 64 || c.cin < 1 || c.channels < 32 || c.channels % 32 || c.modes < 1 ||
        2 * c.modes > c.n_x || c.layers < 1 || c.layers > FNO_MAXL || c.hidden < 32 || c.hidden % 32 ||
        c.max_batch < 1)
        return LH_E_ARG;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return LH_E_NODEVICE;
    lh_fno* f = (lh_fno*)calloc(1, sizeof(lh_fno));
    if (!f) return LH_E_NOMEM;
    f->cfg = c;
    f->L = fno_layout(c);
    int st = LH_OK;
    f->allocs = new std::vector<std::pair<const char*, size_t>>();
    auto alloc = [&](void** p, size_t bytes) {
        if (!st && hipMalloc(p, bytes) != hipSuccess) st = LH_E_NOMEM;
        if (!st) f->allocs->push_back({(const char*)*p, bytes});
    };
    if (hipGetDevice(&f->device) != hipSuccess || hipStreamCreate(&f->stream) != hipSuccess ||
        hipStreamCreate(&f->copy_stream) != hipSuccess ||
        hipEventCreateWithFlags(&f->targets, hipEventDisableTiming) != hipSuccess)
        st = LH_E_HIP;
    for (int l = 0; l <= c.layers && !st; l++)
        if (hipEventCreateWithFlags(&f->ready[l], hipEventDisableTiming) != hipSuccess) st = LH_E_HIP;
    const long long P = f->L.total, X = c.n_x, C = c.channels, Mo2 = 2 * c.modes, H = c.hidden, B = c.max_batch;
    const long long BX = B * X;
    alloc((void**)&f->params, 4 * P);
    alloc((void**)&f->grads, 4 * P);
    alloc((void**)&f->adam_m, 4 * P);
    alloc((void**)&f->adam_v, 4 * P);
    alloc((void**)&f->pbf, 2 * P);
    alloc((void**)&f->Rblk, 2 * (size_t)c.layers * c.modes * 4 * C * C);
    alloc((void**)&f->F, 2 * Mo2 * X);
    alloc((void**)&f->Ginv, 2 * Mo2 * X);
    alloc((void**)&f->xb, 4 * BX * c.cin);
    alloc((void**)&f->tb, 4 * BX);
    alloc((void**)&f->wb, 4 * BX);
    for (int l = 0; l < c.layers; l++) {
        alloc((void**)&f->V[l], 4 * BX * C);
        alloc((void**)&f->Z[l], 4 * BX * C);
        alloc((void**)&f->Vhat[l], 4 * B * Mo2 * C);
    }
    alloc((void**)&f->Ohat, 4 * B * Mo2 * C);
    alloc((void**)&f->Z1, 4 * BX * H);
    alloc((void**)&f->y, 4 * BX);
    alloc((void**)&f->dVa, 4 * BX * C);
    alloc((void**)&f->dVb, 4 * BX * C);
    alloc((void**)&f->dOhat, 4 * B * Mo2 * C);
    alloc((void**)&f->dVhat, 4 * B * Mo2 * C);
    f->work_cap = 4LL << 20;  // split-K partials (floats)
    if (f->work_cap < H * C + 2 * H + 2) f->work_cap = H * C + 2 * H + 2;
    alloc((void**)&f->work, 4 * f->work_cap);
    f->loss_cap = 1;
    if (!st && hipMalloc(&f->loss_dev, 4) != hipSuccess) st = LH_E_NOMEM;  // not a GEMM operand
    if (!st) {
        // truncated DFT matrices (exact angles from the integer m·x mod n_x)
        std::vector<float> F(Mo2 * X), Gi(Mo2 * X);
        const long double tau = 6.283185307179586476925286766559005768L;
        for (int m = 0; m < c.modes; m++)
            for (int x = 0; x < X; x++) {
                const long long q = ((long long)m * x) % X;
                const long double ang = tau * (long double)q / (long double)X;
                const double cs = (double)cosl(ang), sn = (double)sinl(ang);
                const double cm = (m == 0) ? 1.0 : 2.0;
                F[(2 * m) * X + x] = (float)cs;
                F[(2 * m + 1) * X + x] = (float)(-sn);
                Gi[x * Mo2 + 2 * m] = (float)(cm * cs / (double)X);
                Gi[x * Mo2 + 2 * m + 1] = (float)(-cm * sn / (double)X);
            }
        float* tmp = nullptr;
        if (hipMalloc(&tmp, 4 * Mo2 * X) != hipSuccess) st = LH_E_NOMEM;
        if (!st && hipMemcpy(tmp, F.data(), 4 * Mo2 * X, hipMemcpyHostToDevice) != hipSuccess) st = LH_E_HIP;
        if (!st) hipLaunchKernelGGL(fno_cvt_bf16, dim3(nblk(Mo2 * X)), dim3(FNO_T), 0, f->stream, tmp, f->F, Mo2 * X);
        if (!st && hipStreamSynchronize(f->stream) != hipSuccess) st = LH_E_HIP;
        if (!st && hipMemcpy(tmp, Gi.data(), 4 * Mo2 * X, hipMemcpyHostToDevice) != hipSuccess) st = LH_E_HIP;
        if (!st) hipLaunchKernelGGL(fno_cvt_bf16, dim3(nblk(Mo2 * X)), dim3(FNO_T), 0, f->stream, tmp, f->Ginv, Mo2 * X);
        if (!st && hipStreamSynchronize(f->stream) != hipSuccess) st = LH_E_HIP;
        if (tmp) hipFree(tmp);
    }
    if (st) {
        lh_fno_destroy(f);
        return st;
    }
    *out = f;
    return LH_OK;
}

int lh_fno_param_count(const lh_fno* f, int64_t* n) {
    if (!f || !n) return LH_E_ARG;
    *n = f->L.total;
    return LH_OK;
}

int lh_fno_set_params(lh_fno* f, const float* params) {
    if (!f || !params) return LH_E_ARG;
    FNOCK(hipSetDevice(f->device));
    const size_t bytes = 4 * (size_t)f->L.total;
    FNOCK(hipMemcpy(f->params, params, bytes, hipMemcpyHostToDevice));
    FNOCK(hipMemset(f->adam_m, 0, bytes));
    FNOCK(hipMemset(f->adam_v, 0, bytes));
    f->adam_t = 0;
    refresh_bf16(f);
    FNOCK(hipGetLastError());
    FNOCK(hipStreamSynchronize(f->stream));
    return LH_OK;
}

int lh_fno_get_params(lh_fno* f, float* params) {
    if (!f || !params) return LH_E_ARG;
    FNOCK(hipSetDevice(f->device));
    FNOCK(hipStreamSynchronize(f->stream));
    FNOCK(hipMemcpy(params, f->params, 4 * (size_t)f->L.total, hipMemcpyDeviceToHost));
    return LH_OK;
}

int lh_fno_forward(lh_fno* f, const float* x, int batch, float* y) {
    if (!f || !x || !y || batch < 1) return LH_E_ARG;
    FNOCK(hipSetDevice(f->device));
    const lh_fno_cfg& c = f->cfg;
    for (int b0 = 0; b0 < batch; b0 += c.max_batch) {
        const int B = (batch - b0 < c.max_batch) ? batch - b0 : c.max_batch;
        const long long BX = (long long)B * c.n_x;
        FNOCK(hipMemcpyAsync(f->xb, x + (long long)b0 * c.n_x * c.cin, 4 * BX * c.cin, hipMemcpyHostToDevice, f->stream));
        int st = fno_forward_dev(f, B, false);
        if (st) return st;
        FNOCK(hipMemcpyAsync(y + (long long)b0 * c.n_x, f->y, 4 * BX, hipMemcpyDeviceToHost, f->stream));
        FNOCK(hipStreamSynchronize(f->stream));
    }
    return LH_OK;
}

int lh_fno_loss_grad(lh_fno* f, const float* x, const float* target, const float* weight, int batch, float* loss,
                     float* grad) {
    if (!f || !x || !target || !loss || batch < 1 || batch > f->cfg.max_batch) return LH_E_ARG;
    FNOCK(hipSetDevice(f->device));
    const lh_fno_cfg& c = f->cfg;
    const long long BX = (long long)batch * c.n_x;
    FNOCK(hipMemcpyAsync(f->xb, x, 4 * BX * c.cin, hipMemcpyHostToDevice, f->stream));
    int st = fno_forward_dev(f, batch, true);
    if (st) return st;
    // the targets arrive while the forward pass runs
    FNOCK(hipMemcpyAsync(f->tb, target, 4 * BX, hipMemcpyHostToDevice, f->copy_stream));
    f->wcur = nullptr;
    if (weight) {
        FNOCK(hipMemcpyAsync(f->wb, weight, 4 * BX, hipMemcpyHostToDevice, f->copy_stream));
        f->wcur = f->wb;
    }
    FNOCK(hipEventRecord(f->targets, f->copy_stream));
    FNOCK(hipStreamWaitEvent(f->stream, f->targets, 0));
    st = fno_backward_dev(f, batch, f->loss_dev);
    if (st) return st;
    // and each layer's gradients leave while the layers below are at work
    if (grad) {
        const auto out = [&](hipEvent_t e, long long from, long long to) {
            if (hipStreamWaitEvent(f->copy_stream, e, 0) != hipSuccess) return false;
            return hipMemcpyAsync(grad + from, f->grads + from, 4 * (size_t)(to - from), hipMemcpyDeviceToHost,
                                  f->copy_stream) == hipSuccess;
        };
        bool ok = out(f->ready[c.layers], f->L.Q1, f->L.total);
        for (int l = c.layers - 1; l >= 0 && ok; l--) ok = out(f->ready[l], f->L.W[l], l + 1 < c.layers ? f->L.W[l + 1] : f->L.Q1);
        if (!ok) {
            (void)hipStreamSynchronize(f->copy_stream);  // nothing in flight into the caller's array
            return LH_E_HIP;
        }
        FNOCK(hipMemcpyAsync(grad, f->grads, 4 * (size_t)f->L.W[0], hipMemcpyDeviceToHost, f->stream));
    }
    FNOCK(hipMemcpyAsync(loss, f->loss_dev, 4, hipMemcpyDeviceToHost, f->stream));
    FNOCK(hipStreamSynchronize(f->stream));
    FNOCK(hipStreamSynchronize(f->copy_stream));
    return LH_OK;
}

int lh_fno_set_data(lh_fno* f, const float* x, const float* target, const float* weight, int n) {
    if (!f || !x || !target || n < 1) return LH_E_ARG;
    FNOCK(hipSetDevice(f->device));
    const lh_fno_cfg& c = f->cfg;
    for (void* old : {(void*)f->data_x, (void*)f->data_t}) {
        if (!old) continue;
        for (size_t i = 0; i < f->allocs->size(); i++)
            if ((*f->allocs)[i].first == (const char*)old) {
                f->allocs->erase(f->allocs->begin() + i);
                break;
            }
        FNOCK(hipFree(old));
    }
    f->data_x = f->data_t = nullptr;
    f->data_n = 0;
    const size_t nx = (size_t)n * c.n_x * c.cin, nt = (size_t)n * c.n_x;
    FNOCK(hipMalloc(&f->data_x, 4 * nx));
    f->allocs->push_back({(const char*)f->data_x, 4 * nx});
    FNOCK(hipMalloc(&f->data_t, 4 * nt));
    f->allocs->push_back({(const char*)f->data_t, 4 * nt});
    FNOCK(hipMemcpy(f->data_x, x, 4 * nx, hipMemcpyHostToDevice));
    FNOCK(hipMemcpy(f->data_t, target, 4 * nt, hipMemcpyHostToDevice));
    if (f->data_w) FNOCK(hipFree(f->data_w));
    f->data_w = nullptr;
    if (weight) {
        FNOCK(hipMalloc(&f->data_w, 4 * nt));
        FNOCK(hipMemcpy(f->data_w, weight, 4 * nt, hipMemcpyHostToDevice));
    }
    f->data_n = n;
    return LH_OK;
}

int lh_fno_train(lh_fno* f, const int32_t* batch_idx, int n_steps, int batch, const lh_adam* opt,
                 const float* lr_sched, float* losses) {
    if (!f || !batch_idx || n_steps < 1 || batch < 1 || batch > f->cfg.max_batch || !opt || !f->data_x) return LH_E_ARG;
    const long long nidx = (long long)n_steps * batch;
    for (long long i = 0; i < nidx; i++)
        if (batch_idx[i] < 0 || batch_idx[i] >= f->data_n) return LH_E_ARG;
    FNOCK(hipSetDevice(f->device));
    const lh_fno_cfg& c = f->cfg;
    if (nidx > f->idx_cap) {
        if (f->idx_dev) FNOCK(hipFree(f->idx_dev));
        f->idx_dev = nullptr;
        FNOCK(hipMalloc(&f->idx_dev, 4 * nidx));
        f->idx_cap = nidx;
    }
    if (n_steps > f->loss_cap) {
        if (f->loss_dev) FNOCK(hipFree(f->loss_dev));
        f->loss_dev = nullptr;
        FNOCK(hipMalloc(&f->loss_dev, 4 * (size_t)n_steps));
        f->loss_cap = n_steps;
    }
    if (f->lr_dev) FNOCK(hipFree(f->lr_dev));
    f->lr_dev = nullptr;
    if (lr_sched) {
        FNOCK(hipMalloc(&f->lr_dev, 4 * (size_t)n_steps));
        FNOCK(hipMemcpy(f->lr_dev, lr_sched, 4 * (size_t)n_steps, hipMemcpyHostToDevice));
    }
    FNOCK(hipMemcpy(f->idx_dev, batch_idx, 4 * nidx, hipMemcpyHostToDevice));
    const long long ng = (long long)batch * c.n_x * (c.cin > 1 ? c.cin : 1);
    for (int s = 0; s < n_steps; s++) {
        hipLaunchKernelGGL(fno_gather, dim3(nblk(ng)), dim3(FNO_T), 0, f->stream, f->data_x, f->data_t, f->data_w,
                           f->idx_dev + (long long)s * batch, f->xb, f->tb, f->wb, batch, c.n_x, c.cin);
        f->wcur = f->data_w ? f->wb : nullptr;
        int st = fno_forward_dev(f, batch, true);
        if (!st) st = fno_backward_dev(f, batch, f->loss_dev + s);
        if (!st) st = fno_adam_step(f, opt, f->lr_dev, s);
        if (st) return st;
    }
    if (losses) FNOCK(hipMemcpyAsync(losses, f->loss_dev, 4 * (size_t)n_steps, hipMemcpyDeviceToHost, f->stream));
    FNOCK(hipStreamSynchronize(f->stream));
    return LH_OK;
}

}  // extern "C"
