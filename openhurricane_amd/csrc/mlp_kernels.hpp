// mlp_kernels.hpp -- BF16 MFMA kernels of the chemistry surrogate (an MLP
// with GELU hidden layers): a tiled GEMM with fused epilogues for training,
// element-wise helpers (normalisation, loss gradient, bias gradient, Adam),
// and the fused inference + gate kernel that advances the cell states.
//
// Matrix-core layout (gfx950, v_mfma_f32_32x32x16_bf16): lane l holds
//   A[i][8*(l/32) + 0..7] with i = l % 32 (a 32x16 tile, K contiguous),
//   B[8*(l/32) + 0..7][j] with j = l % 32 (a 16x32 tile),
//   D[8*(v/4) + 4*(l/32) + v%4][l % 32] in accumulator v = 0..15.
// Activations are row-major [cells][features], weights [out][in] (so both
// GEMM operands of the forward pass have the reduction dimension
// contiguous), all BF16 with FP32 accumulation.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace ohcm {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef unsigned short bf16_t;  // storage type (raw bits)

__device__ __forceinline__ float bf2f(bf16_t h) { return __uint_as_float((unsigned)h << 16); }
// round-to-nearest-even FP32 -> BF16 (NaN kept quiet)
__device__ __forceinline__ bf16_t f2bf(float f) {
    unsigned u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x7fffffu)) return (bf16_t)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}

// GELU, tanh form: 0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3)))
__device__ __forceinline__ float gelu(float x) {
    const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    const float t = 1.0f - 2.0f / (1.0f + __expf(2.0f * u));
    return 0.5f * x * (1.0f + t);
}
__device__ __forceinline__ float gelu_grad(float x) {
    const float x2 = x * x;
    const float u = 0.7978845608028654f * (x + 0.044715f * x2 * x);
    const float t = 1.0f - 2.0f / (1.0f + __expf(2.0f * u));
    const float du = 0.7978845608028654f * (1.0f + 3.0f * 0.044715f * x2);
    return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * du;
}

enum Epi : int {
    EPI_F32 = 0,        // C32 = acc
    EPI_BIAS_GELU = 1,  // Z32 = acc + bias, C16 = bf16(gelu(Z))
    EPI_BIAS_F32 = 2,   // C32 = acc + bias
    EPI_GELU_BWD = 3,   // C16 = bf16(acc * gelu'(Z32))
};

struct GemmArgs {
    int M, N, K;
    const bf16_t *A;  // A(m,k) = A_KC ? A[m*lda + k] : A[k*lda + m]
    int64_t lda;
    const bf16_t *B;  // B(k,n) = B_KC ? B[n*ldb + k] : B[k*ldb + n]
    int64_t ldb;
    float *C32;       // EPI_F32 / EPI_BIAS_F32 output, EPI_BIAS_GELU pre-activation
    bf16_t *C16;      // EPI_BIAS_GELU / EPI_GELU_BWD output
    int64_t ldc;
    const float *bias;  // [N]
    const float *Z;     // EPI_GELU_BWD: saved pre-activation, ld ldc
    // split-K (EPI_F32 only): block z reduces k in [z kc, min(K, (z+1) kc))
    // into C32 + z zstride; splitk_sum then adds the partial results in order
    int kc;
    int64_t zstride;
    float *rowsum;  // EPI_F32: sum over k of A(m, k), at rowsum + z zstride (nullable)
};

constexpr int kTM = 64, kTN = 128, kTK = 64, kLdsK = kTK + 8;  // +8: LDS row padding

// Part of an operand tile in a thread's registers, on its way from global
// memory to LDS as [row][k].  KC: the operand is K-contiguous, and a thread
// moves 16-byte pieces of rows; else rows are contiguous and a thread moves
// blocks of 8 k x 8 rows, transposed in registers (two byte permutes per
// four values; neighbouring threads take neighbouring k, so that their LDS
// rows fall into different banks).  T0: the thread that takes the first piece.  Loads are 16 bytes wide where base and leading dimension
// allow and the piece lies inside, else by element; outside the matrix they
// give zero.
template <bool KC, int R, int T0 = 0>
struct Stage {
    static constexpr int kPieces = KC ? R * kTK / 8 : R * kTK / 64;
    static constexpr int kPer = (kPieces + 255) / 256, kVec = KC ? 1 : 8;
    uint4 v[kPer][kVec];

    static __device__ __forceinline__ uint4 row8(const bf16_t *p, int left, bool wide) {
        if (wide && left >= 8) return *(const uint4 *)p;
        union {
            bf16_t h[8];
            uint4 q;
        } u;
#pragma unroll
        for (int e = 0; e < 8; ++e) u.h[e] = e < left ? p[e] : (bf16_t)0;
        return u.q;
    }
    // rows r0.. of [0, rows), k in [k0, ke)
    __device__ __forceinline__ void load(const bf16_t *X, int64_t ld, bool wide, int rows, int r0,
                                         int k0, int ke) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int c = ((threadIdx.x + 256 - T0) & 255) + 256 * i;
            if (kPieces % 256 != 0 && c >= kPieces) break;
            if constexpr (KC) {
                const int r = r0 + c / (kTK / 8), k = k0 + c % (kTK / 8) * 8;
                v[i][0] = r < rows ? row8(X + (int64_t)r * ld + k, ke - k, wide) : uint4{0, 0, 0, 0};
            } else {
                const int r = r0 + c / (kTK / 8) * 8, k = k0 + c % (kTK / 8) * 8;
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    v[i][e] = k + e < ke ? row8(X + (int64_t)(k + e) * ld + r, rows - r, wide)
                                         : uint4{0, 0, 0, 0};
            }
        }
    }
    __device__ __forceinline__ void store(bf16_t (*s)[kLdsK]) const {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int c = ((threadIdx.x + 256 - T0) & 255) + 256 * i;
            if (kPieces % 256 != 0 && c >= kPieces) break;
            if constexpr (KC) {
                *(uint4 *)&s[c / (kTK / 8)][c % (kTK / 8) * 8] = v[i][0];
            } else {
                const int r = c / (kTK / 8) * 8, k = c % (kTK / 8) * 8;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    uint4 o;
                    unsigned *w = (unsigned *)&o;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        w[j] = __builtin_amdgcn_perm(((const unsigned *)&v[i][2 * j + 1])[e / 2],
                                                     ((const unsigned *)&v[i][2 * j])[e / 2],
                                                     e % 2 ? 0x07060302u : 0x05040100u);
                    *(uint4 *)&s[r + e][k] = o;
                }
            }
        }
    }
};

// C[M x N] = A[M x K] B[K x N] with a fused epilogue.  A 256-thread block
// computes a 64 x 128 tile (each wavefront two 32 x 32 MFMA tiles) from 64-wide
// slices of A and B in LDS; the next slice is on its way to registers while
// the current one is multiplied.  The training batch (16,384 x 256 x 256)
// gives 512 blocks, two per CU.  Bound by the traffic of its outputs (34 MB
// with the saved pre-activation) and the latency of the few slices: 17 us
// forward, 49 us with 64 x 64 tiles and element-wise loads.
template <bool A_KC, bool B_KC, int EPI>
__global__ __launch_bounds__(256) void gemm_bf16(const GemmArgs g) {
    __shared__ __attribute__((aligned(16))) bf16_t sA[kTM][kLdsK], sB[kTN][kLdsK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * kTM, n0 = blockIdx.x * kTN;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 64;
    const int kb = (int)blockIdx.z * g.kc, ke = min(g.K, kb + g.kc);
    const bool wa = g.lda % 8 == 0 && (uintptr_t)g.A % 16 == 0,
               wb = g.ldb % 8 == 0 && (uintptr_t)g.B % 16 == 0;
    const bool sums = EPI == EPI_F32 && g.rowsum && blockIdx.x == 0;
    Stage<A_KC, kTM> ra;
    Stage<B_KC, kTN, B_KC ? 0 : 128> rb;
    f32x16 acc[2] = {};
    float rs = 0.0f;
    ra.load(g.A, g.lda, wa, g.M, m0, kb, ke);
    rb.load(g.B, g.ldb, wb, g.N, n0, kb, ke);
    for (int k0 = kb; k0 < ke; k0 += kTK) {
        __syncthreads();
        ra.store(sA);
        rb.store(sB);
        __syncthreads();
        if (k0 + kTK < ke) {
            ra.load(g.A, g.lda, wa, g.M, m0, k0 + kTK, ke);
            rb.load(g.B, g.ldb, wb, g.N, n0, k0 + kTK, ke);
        }
        const int i = lane & 31, kh = 8 * (lane >> 5);
#pragma unroll
        for (int ks = 0; ks < kTK; ks += 16) {
            const bf16x8 a = *(const bf16x8 *)&sA[wm + i][ks + kh];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const bf16x8 b = *(const bf16x8 *)&sB[wn + 32 * c + i][ks + kh];
                acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[c], 0, 0, 0);
            }
        }
        if (sums) {  // four threads to a row, 16 k each
#pragma unroll
            for (int e = 0; e < 16; ++e) rs += bf2f(sA[tid >> 2][(tid & 3) * 16 + e]);
        }
    }
    // ---- epilogue ----
    if (sums) {
        rs += __shfl_xor(rs, 1);
        rs += __shfl_xor(rs, 2);
        const int m = m0 + (tid >> 2);
        if ((tid & 3) == 0 && m < g.M) g.rowsum[m + (int64_t)blockIdx.z * g.zstride] = rs;
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int j = n0 + wn + 32 * c + (lane & 31);
        if (j >= g.N) continue;
        const float bias = EPI == EPI_BIAS_F32 || EPI == EPI_BIAS_GELU ? g.bias[j] : 0.0f;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int i = m0 + wm + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
            if (i >= g.M) continue;
            const int64_t o = (int64_t)i * g.ldc + j;
            const float x = acc[c][v];
            if (EPI == EPI_F32) {
                g.C32[o + (int64_t)blockIdx.z * g.zstride] = x;
            } else if (EPI == EPI_BIAS_F32) {
                g.C32[o] = x + bias;
            } else if (EPI == EPI_BIAS_GELU) {
                const float z = x + bias;
                if (g.C32) g.C32[o] = z;
                g.C16[o] = f2bf(gelu(z));
            } else {
                g.C16[o] = f2bf(x * gelu_grad(g.Z[o]));
            }
        }
    }
}

// G[e] = sum over z = 0..S-1, in that order, of the split-K partial gradients.
__global__ void splitk_sum(int S, int64_t np, const float *part, float *G) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= np) return;
    float v = part[e];
    for (int z = 1; z < S; ++z) v += part[z * np + e];
    G[e] = v;
}

// ---- element-wise training helpers ----

// X16[i][k] = bf16((X[i][k] - mean[k]) / std[k]) for k < nin, 0 for padding
__global__ void normalize_in(int64_t n, int nin, int kpad, const float *X, const float *mean,
                             const float *rstd, bf16_t *X16) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n * kpad) return;
    const int64_t i = e / kpad;
    const int k = (int)(e % kpad);
    X16[e] = k < nin ? f2bf((X[i * nin + k] - mean[k]) * rstd[k]) : (bf16_t)0;
}

// Weighted mean-square loss on normalised targets t = (Yt - mean) / std:
// loss = sum w_k (out - t)^2 / n, dOut = 2 w (out - t) / n (BF16 for the
// backward GEMMs, rows padded with zeros to ld); per-block partial losses
// into part[].
__global__ void loss_grad(int64_t n, int nout, int ld, const float *out, const float *Yt,
                          const float *mean, const float *rstd, const float *w, bf16_t *dOut,
                          float *part) {
    __shared__ float red[256];
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.0f;
    if (e < n * nout) {
        const int k = (int)(e % nout);
        const float r = out[e] - (Yt[e] - mean[k]) * rstd[k];
        l = w[k] * r * r / (float)n;
        const int64_t i = e / nout;
        dOut[i * ld + k] = f2bf(2.0f * w[k] * r / (float)n);
        if (k < ld - nout) dOut[i * ld + nout + k] = (bf16_t)0;
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// Adam on the flat FP32 master parameters (c1 = 1/(1-b1^t), c2 = 1/(1-b2^t)),
// refreshing their BF16 copy p16 (same layout).
__global__ void adam_step(int64_t np, float *p, const float *g, float *m, float *v, float lr,
                          float b1, float b2, float eps, float c1, float c2, bf16_t *p16) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= np) return;
    const float gi = g[e];
    const float mi = b1 * m[e] + (1.0f - b1) * gi;
    const float vi = b2 * v[e] + (1.0f - b2) * gi * gi;
    m[e] = mi;
    v[e] = vi;
    const float pi = p[e] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
    p[e] = pi;
    p16[e] = f2bf(pi);
}

__global__ void to_bf16(int64_t n, const float *x, bf16_t *y) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n) y[e] = f2bf(x[e]);
}

__global__ void sum_partials(int nb, const float *part, float *out) {
    __shared__ float red[256];
    float s = 0.0f;
    for (int i = threadIdx.x; i < nb; i += 256) s += part[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

}  // namespace ohcm

namespace ohcm {

// ---- fused inference + gate ------------------------------------------------

constexpr double kYFloor = 1e-20;  // mass-fraction floor of the log features
constexpr double kAgreeY = 1e-4;   // species the two-network agreement check covers

typedef __attribute__((__vector_size__(8 * sizeof(int)))) int i32x8;

// OCP FP8 E4M3 (bias 7, no infinities, 0x7f NaN, largest finite 448): round to
// nearest even, saturating.
__host__ __device__ inline uint8_t f2e4m3(float x) {
    const uint8_t sign = x < 0.0f ? 0x80 : 0x00;
    const float a = fabsf(x);
    if (!(a == a)) return 0x7f;
    if (a >= 448.0f) return sign | 0x7e;
    if (a < 0.015625f) {  // subnormal: m * 2^-9
        const int m = (int)rintf(a * 512.0f);
        return sign | (uint8_t)m;  // m == 8 is the smallest normal, 0x08
    }
    int ex;
    const float fr = frexpf(a, &ex);  // a = fr 2^ex, fr in [0.5, 1)
    int e = ex - 1;
    int m = (int)rintf((2.0f * fr - 1.0f) * 8.0f);
    if (m == 8) {
        m = 0;
        ++e;
    }
    const int be = e + 7;
    if (be > 15 || (be == 15 && m == 7)) return sign | 0x7e;
    return sign | (uint8_t)((be << 3) | m);
}
// The same rounding with the hardware conversion (v_cvt_pk_fp8_f32 is OCP
// E4M3 with round to nearest even on this target, NaN above 448, hence the
// clamp; a negative value that rounds to zero gives +0 instead of -0).
__device__ __forceinline__ uint8_t f2e4m3_hw(float x) {
    const float c = fminf(fmaxf(x, -448.0f), 448.0f);
    return (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(c, c, 0, false) & 0xff);
}
__host__ __device__ inline float e4m32f(uint8_t b) {
    const int e = (b >> 3) & 15, m = b & 7;
    const float v = e == 0 ? ldexpf((float)m, -9) : ldexpf(1.0f + 0.125f * (float)m, e - 7);
    return (b & 0x80) ? -v : v;
}

struct InferArgs {
    int64_t n;
    int ns, ne;                 // species, elements
    double *T, *Y;              // state, advanced in place where the gate passes
    const double *p;
    int64_t ldY;
    const double *dt;
    double dtFactor, dt_train;  // cells whose dt*dtFactor differs from dt_train fall back
    const bf16_t *W;            // packed BF16 weights, layer l at woff[l], [rows][K] padded
    const float *b;             // biases, layer l at boff[l] (padded rows zero)
    int woff[8], boff[8];
    int depth;                  // hidden layers
    const uint8_t *W8;          // FP8 copies of the hidden-to-hidden layers l = 1..depth-1
    const float *s8;            // their per-row scales
    int w8off[8], s8off[8];
    const float *in_mean, *in_rstd, *zlo, *zhi;  // input normalisation and OOD box
    const float *out_mean, *out_std;
    const float *delta;         // symmetric-log target scales (nullptr: plain increments)
    const float *peer;          // [n][nout] increments of a second network (nullptr: none)
    double peer_tol;            // largest accepted disagreement with the peer
    const double *elemW;        // [ns][ne]: atoms of element e in species k / W_k
    double gate_tol;            // max relative element-mass change
    double T_low, T_high;
    int *fail_list;             // indices of cells left to the integrator
    unsigned int *fail_count;
    int mode;                   // 0: advance and gate; 1: write increments to out32 only
    float *out32;               // mode 1: [n][nout] increments (dT, dln Y)
};

// network output k (denormalised) -> increment: identity, or the inverse of
// z = sign(d) ln(1 + |d| / delta_k)
// (nrm: output mean, standard deviation and target scale, each [NOUTP])
template <int NOUTP>
__device__ __forceinline__ float out_increment(const InferArgs &a, const float (*nrm)[NOUTP],
                                               const float *o, int k) {
    const float z = o[k] * nrm[1][k] + nrm[0][k];
    if (!a.delta) return z;
    return copysignf(expm1f(fabsf(z)), z) * nrm[2][k];
}

template <int B, int E, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// gelu() for the inference epilogue: the quotient 2 / (1 + e) by the refined
// reciprocal and a remainder step, as an IEEE division without its scaling (the
// divisor is at least 1, and clamped below overflow, where the quotient no
// longer changes 1 - q).
__device__ __forceinline__ float gelu_fast(float x) {
    const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    const float d = fminf(1.0f + __builtin_amdgcn_exp2f(u * 2.885390082f), 1.0e38f);  // 2 / ln 2
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(fmaf(-d, r, 1.0f), r, r);
    float q = r + r;
    q = fmaf(fmaf(-d, q, 2.0f), r, q);
    const float t = 1.0f - q;
    return 0.5f * x * (1.0f + t);
}
// two BF16 values (round to nearest even) in one word, low first
__device__ __forceinline__ unsigned pk_bf16(float a, float b) {
    typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
    const bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(unsigned, v);
}

// ln x to about 1e-14 relative (x positive and normal; else as log): mantissa
// m in [sqrt(1/2), sqrt(2)), s = (m - 1) / (m + 1), and the series of
// 2 artanh(s) to s^19 -- a quarter of the library logarithm's instructions, for
// features that are rounded to FP32 next.
__device__ __forceinline__ double log_feature(double x) {
    double m = __builtin_amdgcn_frexp_mant(x);  // [1/2, 1)
    int e = __builtin_amdgcn_frexp_exp(x);
    const bool low = m < 0.70710678118654752;
    m = low ? m + m : m;
    e -= low ? 1 : 0;
    const double b = m + 1.0;
    double r = __builtin_amdgcn_rcp(b);
    r = fma(fma(-b, r, 1.0), r, r);
    r = fma(fma(-b, r, 1.0), r, r);
    const double s = (m - 1.0) * r, z = s * s;
    double p = 2.0 / 19.0;
    p = fma(p, z, 2.0 / 17.0);
    p = fma(p, z, 2.0 / 15.0);
    p = fma(p, z, 2.0 / 13.0);
    p = fma(p, z, 2.0 / 11.0);
    p = fma(p, z, 2.0 / 9.0);
    p = fma(p, z, 2.0 / 7.0);
    p = fma(p, z, 2.0 / 5.0);
    p = fma(p, z, 2.0 / 3.0);
    p = fma(p, z, 2.0);
    const double l = fma((double)e, 0.69314718055994530942, s * p);
    return x > 0.0 ? l : (x == 0.0 ? -__builtin_huge_val() : __builtin_nan(""));
}

// Hidden layer: out[TM][W] = gelu(in[TM][K] W^T + b), NW wavefronts each
// producing TM rows x W/NW columns.  IN8: FP8 activations and weights on the
// 32x32x64 f8f6f4 MFMA (unit block scales; per-row weight scale applied in
// the epilogue), else BF16 on 32x32x16.  OUT8: the epilogue writes FP8.
// Strides LDI / LDO count elements of the buffer's type.  The weights are the
// first MFMA operand, so that a lane's accumulators hold four consecutive
// features of one cell at a time: the epilogue packs and stores them as one
// word or two.  The layer is bound by that epilogue (24 vector instructions per
// activation), not by the matrix cores.
template <int TM, int WD, int NW, int K, int LDI, int LDO, bool IN8, bool OUT8>
__device__ __forceinline__ void mlp_layer(const void *sin_, void *sout_, const void *Wl_,
                                          const float *ws, const float *bl) {
    constexpr int RT = TM / 32, CT = WD / (32 * NW);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    f32x16 acc[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[r][c] = f32x16{};
    const int i = lane & 31, h = lane >> 5;
    // The weights come from L2: a group of KG steps' fragments is requested ahead
    // of the group before it (one wait per group instead of one per step).
    using W_t = std::conditional_t<IN8, uint8_t, bf16_t>;
    using frag = std::conditional_t<IN8, i32x8, bf16x8>;
    constexpr int KS = IN8 ? 64 : 16, NK = K / KS, KW = IN8 ? 32 : 8;  // k of a step, steps, k of a lane
    constexpr int KG = IN8 ? 2 : (CT > 2 ? 4 : 8);
    const W_t *sin = (const W_t *)sin_ + i * LDI + KW * h;
    const W_t *Wl = (const W_t *)Wl_ + (int64_t)(wave * (CT * 32) + i) * K + KW * h;
    frag b[2][KG][CT];
    auto load = [&](auto gc) __attribute__((always_inline)) {
        constexpr int g = gc;
#pragma unroll
        for (int t = 0; t < KG; ++t)
            if (g * KG + t < NK)
#pragma unroll
                for (int c = 0; c < CT; ++c)
                    b[g % 2][t][c] = *(const frag *)(Wl + (int64_t)c * 32 * K + (g * KG + t) * KS);
    };
    load(std::integral_constant<int, 0>{});
    constexpr int NG = (NK + KG - 1) / KG;
    auto group = [&](auto gc) __attribute__((always_inline)) {
        constexpr int g = gc;
        if constexpr (g + 1 < NG) load(std::integral_constant<int, g + 1>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < KG; ++t)
            if (g * KG + t < NK) {
                frag a[RT];
#pragma unroll
                for (int r = 0; r < RT; ++r)
                    a[r] = *(const frag *)(sin + r * 32 * LDI + (g * KG + t) * KS);
#pragma unroll
                for (int r = 0; r < RT; ++r)
#pragma unroll
                    for (int c = 0; c < CT; ++c) {
                        if constexpr (IN8)
                            acc[r][c] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                                b[g % 2][t][c], a[r], acc[r][c], 0, 0, 0, 127, 0, 127);
                        else
                            acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[g % 2][t][c], a[r],
                                                                                acc[r][c], 0, 0, 0);
                    }
            }
    };
    static_for<0, NG>(group);
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            // features col .. col + 3 of cell r * 32 + i
            const int col = wave * (CT * 32) + c * 32 + 8 * q + 4 * h;
            const float4 b4 = *(const float4 *)(bl + col);
            const float bias[4] = {b4.x, b4.y, b4.z, b4.w};
            float scale[4] = {1.0f, 1.0f, 1.0f, 1.0f};
            if constexpr (IN8) {
                const float4 s4 = *(const float4 *)(ws + col);
                scale[0] = s4.x, scale[1] = s4.y, scale[2] = s4.z, scale[3] = s4.w;
            }
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                float g[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    g[e] = gelu_fast(acc[r][c][4 * q + e] * scale[e] + bias[e]);
                const int o = (r * 32 + i) * LDO + col;
                if constexpr (OUT8)
                    *(unsigned *)((uint8_t *)sout_ + o) =
                        f2e4m3_hw(g[0]) | f2e4m3_hw(g[1]) << 8 | f2e4m3_hw(g[2]) << 16 |
                        (unsigned)f2e4m3_hw(g[3]) << 24;
                else
                    *(uint2 *)((bf16_t *)sout_ + o) = uint2{pk_bf16(g[0], g[1]), pk_bf16(g[2], g[3])};
            }
        }
}

// One block of NW wavefronts advances TM cells: features (T, log p, log Y) ->
// normalised BF16 -> hidden layers -> increments (dT, dlog Y) -> new state,
// gated on the dt match, the input box (OOD), the element-mass change and,
// with a peer network, the two networks' agreement (the state then takes the
// mean of both increments).  FP8: the hidden-to-hidden layers run in FP8.
template <int TM, int WD, int NW, int KIN, int NOUTP, bool FP8>
__global__ __launch_bounds__(64 * NW) void mlp_infer(const InferArgs a) {
    constexpr int NT = 64 * NW;
    constexpr int LD = WD + 8;   // LDS row stride (bf16) of the activation buffers
    constexpr int LD8 = WD + 16; // the same buffers holding FP8 rows (bytes)
    static_assert(TM * LD8 <= TM * LD * 2, "FP8 rows must fit the buffer");
    __shared__ __attribute__((aligned(16))) bf16_t buf[2][TM * LD];
    __shared__ int sfail[TM];
    __shared__ float snorm[4][KIN], sout_n[3][NOUTP];  // input / output normalisation
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t c0 = (int64_t)blockIdx.x * TM;
    const int nin = a.ns + 2, nout = a.ns + 1;
    if (tid < TM) sfail[tid] = 0;
    for (int e = tid; e < 4 * KIN; e += NT) {
        const int q = e / KIN, k = e % KIN;
        const float *src = q == 0 ? a.in_mean : q == 1 ? a.in_rstd : q == 2 ? a.zlo : a.zhi;
        snorm[q][k] = k < nin ? src[k] : 0.0f;
    }
    for (int e = tid; e < 3 * NOUTP; e += NT) {
        const int q = e / NOUTP, k = e % NOUTP;
        const float *src = q == 0 ? a.out_mean : q == 1 ? a.out_std : a.delta;
        sout_n[q][k] = k < nout && src ? src[k] : 0.0f;
    }
    __syncthreads();
    // ---- features, normalised, into buf[0] as [TM][KIN] (stride LD) ----
    // Thread tid takes the features tid / TM + m (256 / TM) of cell tid % TM, all
    // loads first; normalisation and box come from LDS and the box check is one flag
    // per thread (with four table loads and a branch per value the features took
    // 42 k of a block's 97 k cycles).
    {
        constexpr int IT = TM * KIN / NT, KT = NT / TM;
        const int r = tid % TM, k0 = tid / TM;
        const bool in = c0 + r < a.n;
        const int64_t cell = in ? c0 + r : a.n - 1;
        double v[IT];
#pragma unroll
        for (int m = 0; m < IT; ++m) {
            const int k = k0 + KT * m;
            const double *src = k == 0 ? a.T : k == 1 ? a.p : a.Y + (int64_t)min(k - 2, a.ns - 1) * a.ldY;
            v[m] = src[cell];
        }
        bool ood = false;
#pragma unroll
        for (int m = 0; m < IT; ++m) {
            const int k = k0 + KT * m;
            const double l = log_feature(k == 1 ? v[m] : fmax(v[m], kYFloor));
            const float z = ((float)(k == 0 ? v[m] : l) - snorm[0][k]) * snorm[1][k];
            ood = ood || (k < nin && !(z >= snorm[2][k] && z <= snorm[3][k]));
            buf[0][r * LD + k] = f2bf(k < nin && in ? z : 0.0f);
        }
        if (ood && in) atomicOr(&sfail[r], 1);
    }
    __syncthreads();
    // ---- hidden layers (ping-pong between the two buffers) ----
    const bool l1_fp8 = FP8 && a.depth > 1;
    if (l1_fp8) mlp_layer<TM, WD, NW, KIN, LD, LD8, false, true>(buf[0], buf[1], a.W + a.woff[0], nullptr, a.b + a.boff[0]);
    else mlp_layer<TM, WD, NW, KIN, LD, LD, false, false>(buf[0], buf[1], a.W + a.woff[0], nullptr, a.b + a.boff[0]);
    __syncthreads();
    int cur = 1;
    for (int l = 1; l < a.depth; ++l) {
        if constexpr (FP8) {
            if (l + 1 < a.depth)
                mlp_layer<TM, WD, NW, WD, LD8, LD8, true, true>(buf[cur], buf[cur ^ 1], a.W8 + a.w8off[l],
                                                             a.s8 + a.s8off[l], a.b + a.boff[l]);
            else
                mlp_layer<TM, WD, NW, WD, LD8, LD, true, false>(buf[cur], buf[cur ^ 1], a.W8 + a.w8off[l],
                                                             a.s8 + a.s8off[l], a.b + a.boff[l]);
        } else {
            mlp_layer<TM, WD, NW, WD, LD, LD, false, false>(buf[cur], buf[cur ^ 1], a.W + a.woff[l],
                                                         nullptr, a.b + a.boff[l]);
        }
        __syncthreads();
        cur ^= 1;
    }
    // ---- output layer into FP32 (aliasing the free buffer) ----
    float *sout = (float *)buf[cur ^ 1];
    constexpr int LDF = NOUTP + 1;
    static_assert(TM * LDF * 4 <= TM * LD * 2, "output tile must fit the free buffer");
    {
        constexpr int RT = TM / 32, CTO = NOUTP / 32;
        const int i = lane & 31, kh = 8 * (lane >> 5);
        static_assert(RT * CTO <= NW, "one wavefront per output tile");
        if (wave < RT * CTO) {
            const int r = wave / CTO, c = wave % CTO;
            const bf16_t *Wl = a.W + a.woff[a.depth];
            f32x16 acc = {};
#pragma unroll
            for (int k0 = 0; k0 < WD; k0 += 16) {
                const bf16x8 av = *(const bf16x8 *)(buf[cur] + (r * 32 + i) * LD + k0 + kh);
                const bf16x8 bv = *(const bf16x8 *)(Wl + (int64_t)(c * 32 + i) * WD + k0 + kh);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc, 0, 0, 0);
            }
            const float bias = a.b[a.boff[a.depth] + c * 32 + i];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = r * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
                sout[row * LDF + c * 32 + i] = acc[v] + bias;
            }
        }
    }
    __syncthreads();
    if (a.mode == 1) {
        // the block's increments are contiguous: element e of [TM][nout] per thread
        const int ne = (int)min((int64_t)TM, a.n - c0) * nout;
        for (int e = tid; e < ne; e += NT)
            a.out32[c0 * nout + e] = out_increment<NOUTP>(a, sout_n, sout + (e / nout) * LDF, e % nout);
        return;
    }
    // ---- per cell: increments, new state, gate ----
    if (tid >= TM) return;
    const int64_t cell = c0 + tid;
    if (cell >= a.n) return;
    const float *o = sout + tid * LDF;
    bool ok = sfail[tid] == 0;
    ok = ok && fabs(a.dt[cell] * a.dtFactor - a.dt_train) <= 1e-9 * a.dt_train;
    const double T0 = a.T[cell];
    const float *q = a.peer ? a.peer + cell * nout : nullptr;
    double dT = out_increment<NOUTP>(a, sout_n, o, 0);
    if (q) {
        ok = ok && fabs(dT - (double)q[0]) <= a.peer_tol * T0;
        dT = 0.5 * (dT + (double)q[0]);
    }
    const double T1 = T0 + dT;
    ok = ok && T1 >= a.T_low && T1 <= a.T_high;
    // mass fractions from the log increments (kept in the free activation
    // buffer as [TM][64] doubles), then renormalised
    double *y1 = (double *)buf[cur] + tid * 64;
    static_assert(TM * 64 * 8 <= TM * LD * 2, "mass-fraction tile must fit the free buffer");
    double ys = 0.0;
    for (int k = 0; k < a.ns; ++k) {
        const double yk = a.Y[(int64_t)k * a.ldY + cell];
        const double y0 = fmax(yk, kYFloor);
        const double ds = out_increment<NOUTP>(a, sout_n, o, k + 1);
        const double dq = q ? (double)q[k + 1] : ds;
        const double d = q ? 0.5 * (ds + dq) : ds;
        const double v = y0 * exp(d);
        // the networks must agree on every species above kAgreeY before or
        // after the step (a decade below the 1e-3 "major" threshold, so
        // that a species predicted just under it is still checked)
        if (q && (yk >= kAgreeY || v >= kAgreeY)) ok = ok && fabs(ds - dq) <= a.peer_tol;
        y1[k] = v;
        ys += v;
    }
    ok = ok && ys > 0.0 && isfinite(ys);
    const double rys = 1.0 / ys;
    // element-mass change (chemistry conserves element moles per unit mass)
    double emax = 0.0;
    for (int e = 0; e < a.ne && ok; ++e) {
        double e0 = 0.0, e1 = 0.0;
        for (int k = 0; k < a.ns; ++k) {
            const double w = a.elemW[k * a.ne + e];
            e0 += w * a.Y[(int64_t)k * a.ldY + cell];
            e1 += w * y1[k] * rys;
        }
        if (e0 > 1e-12) emax = fmax(emax, fabs(e1 - e0) / e0);
    }
    ok = ok && emax <= a.gate_tol;
    if (ok) {
        a.T[cell] = T1;
        for (int k = 0; k < a.ns; ++k) a.Y[(int64_t)k * a.ldY + cell] = y1[k] * rys;
    } else {
        const unsigned int slot = atomicAdd(a.fail_count, 1u);
        a.fail_list[slot] = (int)cell;
    }
}

}  // namespace ohcm
