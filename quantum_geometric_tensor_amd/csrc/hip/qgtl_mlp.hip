// Training and inference kernels of the learned preconditioner.
//
// The network (feature vector of one parameter point -> diagonal and
// low-rank factor of a preconditioner for the metric solve) is a stack of
// dense layers with BF16 weights, BF16 MFMA operands and FP32 accumulation
// (v_mfma_f32_32x32x16_bf16); activations, gradients and the Adam state are
// FP32; the Kaporin loss and its gradient per sample are FP64.  QGTL has no
// learned component: these kernels precondition the conjugate-gradient
// solve of compute_natural_gradient_cpu
// (src/quantum_geometric/hybrid/classical_optimization_engine.c:543-610).
#include <math.h>

#include "qgtl_hip_common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kThreads = 256;

__device__ __forceinline__ uint16_t bf16_rn(float x) {
    const uint32_t u = __float_as_uint(x);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

// ---- dense layers ----
// C (M x N, fp32) = op(A) op(B): operands rounded to bf16 when staged into LDS,
// fp32 accumulation, one 32 x 32 tile per workgroup.  The layers are small (the
// preconditioner's: 256 x 256 .. 1728 outputs, K = 256 .. 1728), so a product is
// a few memory latencies long and what counts is how many are in a row: a stage
// covers 256 of K (64 KB of fp32 in flight per workgroup), its 16-byte loads go
// out before the previous stage's MFMAs, the four waves take a quarter of the
// stage's K each and add their accumulators at the end, and the small tiles
// give 64 .. 432 workgroups.  The activation, its derivative, the bias and the
// bias gradient (column sums) ride on the products instead of reading and
// writing the layer again, and a layer's weight gradient and the gradient handed
// down are one launch.  Loss and gradient at P = 192, rank 8, 256 samples: 21
// launches of 880 us in all before, 8 of 53 us now; the call 1402 -> 584 us.
constexpr int kTile = 32, kK = 256;
constexpr int kLdsRow = kK + 8;                  // bf16 per LDS row: 528 B (16-B aligned, rows 4 banks apart)
constexpr float kGeluC = 0.7978845608028654f;    // sqrt(2 / pi)

__device__ __forceinline__ float gelu(float x) {
    return 0.5f * x * (1.f + tanhf(kGeluC * (x + 0.044715f * x * x * x)));
}

__device__ __forceinline__ float gelu_grad(float x) {
    const float t = tanhf(kGeluC * (x + 0.044715f * x * x * x));
    return 0.5f * (1.f + t) + 0.5f * x * (1.f - t * t) * kGeluC * (1.f + 3.f * 0.044715f * x * x);
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// An operand tile: 32 rows (of M or N) x 256 of K.  kContig: a row's K values are
// adjacent (element (r, k) at r * ld + k); else its rows are (k * ld + r).
// vec: 16-byte (fp32) or 8-byte (bf16, strided) loads are aligned; without it, and
// at the edges, elements are read one by one.
template <bool BF16, bool CONTIG>
struct Operand;

// n adjacent elements of a row, n = min(COUNT, left) of them real, the rest zero
template <int COUNT, typename Vec, typename Elem>
__device__ __forceinline__ Vec load_run(const Elem *q, int left, bool vec) {
    if (vec && left >= COUNT) return *reinterpret_cast<const Vec *>(q);
    Vec v;
#pragma unroll
    for (int c = 0; c < COUNT; c++) v[c] = c < left ? q[c] : Elem(0);
    return v;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

template <>
struct Operand<false, true> {                    // fp32, K adjacent: 8 lanes per row, 8 loads
    f32x4 v[8];
    __device__ __forceinline__ void load(const void *p, int ld, int r0, int R, int k0, int K, bool vec) {
        const int r = r0 + (int)(threadIdx.x >> 3);
        const float *q = reinterpret_cast<const float *>(p) + (size_t)(r < R ? r : 0) * ld;
        const int lim = r < R ? K : 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int k = k0 + 4 * (int)(threadIdx.x & 7) + 32 * i;
            v[i] = load_run<4, f32x4>(q + k, lim - k, vec);
        }
    }
    __device__ __forceinline__ void store(uint16_t *lds) const {
#pragma unroll
        for (int i = 0; i < 8; i++)
            *reinterpret_cast<uint2 *>(lds + (threadIdx.x >> 3) * kLdsRow + 4 * (threadIdx.x & 7) + 32 * i) =
                make_uint2(pack_bf16(v[i][0], v[i][1]), pack_bf16(v[i][2], v[i][3]));
    }
};

template <>
struct Operand<false, false> {                   // fp32, rows adjacent: 4 rows x 2 of K per thread, 4 times
    f32x4 v[8];
    __device__ __forceinline__ void load(const void *p, int ld, int r0, int R, int k0, int K, bool vec) {
        const int r = r0 + 4 * (int)(threadIdx.x & 7);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int k = k0 + 2 * (int)(threadIdx.x >> 3) + 64 * (i >> 1) + (i & 1);
            const float *q = reinterpret_cast<const float *>(p) + (size_t)(k < K ? k : 0) * ld + r;
            v[i] = load_run<4, f32x4>(q, k < K ? R - r : 0, vec);
        }
    }
    __device__ __forceinline__ void store(uint16_t *lds) const {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int c = 0; c < 4; c++)
                *reinterpret_cast<uint32_t *>(lds + (4 * (threadIdx.x & 7) + c) * kLdsRow + 2 * (threadIdx.x >> 3) +
                                              64 * i) = pack_bf16(v[2 * i][c], v[2 * i + 1][c]);
    }
};

template <>
struct Operand<true, true> {                     // bf16, K adjacent
    u16x8 v[4];
    __device__ __forceinline__ void load(const void *p, int ld, int r0, int R, int k0, int K, bool vec) {
        const int r = r0 + (int)(threadIdx.x >> 3);
        const uint16_t *q = reinterpret_cast<const uint16_t *>(p) + (size_t)(r < R ? r : 0) * ld;
        const int lim = r < R ? K : 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int k = k0 + 8 * (int)(threadIdx.x & 7) + 64 * i;
            v[i] = load_run<8, u16x8>(q + k, lim - k, vec);
        }
    }
    __device__ __forceinline__ void store(uint16_t *lds) const {
#pragma unroll
        for (int i = 0; i < 4; i++)
            *reinterpret_cast<u16x8 *>(lds + (threadIdx.x >> 3) * kLdsRow + 8 * (threadIdx.x & 7) + 64 * i) = v[i];
    }
};

template <>
struct Operand<true, false> {                    // bf16, rows adjacent
    u16x4 v[8];
    __device__ __forceinline__ void load(const void *p, int ld, int r0, int R, int k0, int K, bool vec) {
        const int r = r0 + 4 * (int)(threadIdx.x & 7);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int k = k0 + 2 * (int)(threadIdx.x >> 3) + 64 * (i >> 1) + (i & 1);
            const uint16_t *q = reinterpret_cast<const uint16_t *>(p) + (size_t)(k < K ? k : 0) * ld + r;
            v[i] = load_run<4, u16x4>(q, k < K ? R - r : 0, vec);
        }
    }
    __device__ __forceinline__ void store(uint16_t *lds) const {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int c = 0; c < 4; c++)
                *reinterpret_cast<uint32_t *>(lds + (4 * (threadIdx.x & 7) + c) * kLdsRow + 2 * (threadIdx.x >> 3) +
                                              64 * i) = (uint32_t)v[2 * i][c] | ((uint32_t)v[2 * i + 1][c] << 16);
    }
};

struct Lds {
    uint16_t a[kTile * kLdsRow], b[kTile * kLdsRow];
};

enum { kForward, kWeightGrad, kInputGrad };      // what a product is (see qgtl_mlp_product_t)

template <int KIND>
__device__ __forceinline__ void product(const qgtl_mlp_product_t &g, int tile, Lds &sm) {
    constexpr bool A_CONTIG = KIND != kWeightGrad, B_BF16 = KIND != kWeightGrad, B_CONTIG = KIND == kInputGrad;
    const int tn = (g.N + kTile - 1) / kTile;
    const int m0 = tile / tn * kTile, n0 = tile % tn * kTile;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    f32x16 acc;
#pragma unroll
    for (int e = 0; e < 16; e++) acc[e] = 0.f;
    f32x4 cs = {0.f, 0.f, 0.f, 0.f};               // weight gradient: column sums of B (the bias gradient)
    const bool sums = KIND == kWeightGrad && m0 == 0;

    Operand<false, A_CONTIG> oa;
    Operand<B_BF16, B_CONTIG> ob;
    oa.load(g.A, g.lda, m0, g.M, 0, g.K, g.avec);
    ob.load(g.B, g.ldb, n0, g.N, 0, g.K, g.bvec);
    for (int k0 = 0; k0 < g.K; k0 += kK) {
        oa.store(sm.a);
        ob.store(sm.b);
        if constexpr (KIND == kWeightGrad) {
            if (sums)
#pragma unroll
                for (int i = 0; i < 8; i++) cs += ob.v[i];
        }
        __syncthreads();
        if (k0 + kK < g.K) {
            oa.load(g.A, g.lda, m0, g.M, k0 + kK, g.K, g.avec);
            ob.load(g.B, g.ldb, n0, g.N, k0 + kK, g.K, g.bvec);
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int koff = 64 * wave + 16 * s + 8 * (lane >> 5);
            const bf16x8 fa = *reinterpret_cast<const bf16x8 *>(&sm.a[(lane & 31) * kLdsRow + koff]);
            const bf16x8 fb = *reinterpret_cast<const bf16x8 *>(&sm.b[(lane & 31) * kLdsRow + koff]);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    // the four waves' accumulators, added in wave order; wave w finishes elements 4 w .. 4 w + 3
    float *red = reinterpret_cast<float *>(sm.a);                // 4 x 16 x 64 floats (16 KB of the 16.5 KB tile)
    static_assert(sizeof(sm.a) >= 4 * 16 * 64 * sizeof(float), "accumulators fit the A tile");
#pragma unroll
    for (int e = 0; e < 16; e++) red[(wave * 16 + e) * 64 + lane] = acc[e];
    f32x4 *cred = reinterpret_cast<f32x4 *>(sm.b);               // 32 x 8
    if (sums) cred[threadIdx.x] = cs;
    __syncthreads();
    const int col = n0 + (lane & 31);
#pragma unroll
    for (int e2 = 0; e2 < 4; e2++) {
        const int e = 4 * wave + e2;
        float v = red[e * 64 + lane];
#pragma unroll
        for (int w = 1; w < 4; w++) v += red[(w * 16 + e) * 64 + lane];
        const int row = m0 + wave * 8 + (lane >> 5) * 4 + e2;
        if (row >= g.M || col >= g.N) continue;
        const size_t at = (size_t)row * g.N + col;
        if constexpr (KIND == kForward) {
            v += g.bias[col];
            if (g.act) g.act[at] = gelu(v);
        }
        if constexpr (KIND == kInputGrad) v *= gelu_grad(g.pre[at]);
        g.C[at] = v;
    }
    if (sums && threadIdx.x < 32) {
        const int n = n0 + (int)threadIdx.x;
        const float *c = reinterpret_cast<const float *>(cred) + threadIdx.x;   // (thread kp * 8 + n / 4, n % 4)
        float v = 0.f;
        for (int kp = 0; kp < 32; kp++) v += c[kp * 32];
        if (n < g.N) g.colsum[n] = v;
    }
}

__device__ __forceinline__ int product_tiles(const qgtl_mlp_product_t &g) {
    return ((g.M + kTile - 1) / kTile) * ((g.N + kTile - 1) / kTile);
}

__global__ __launch_bounds__(kThreads) void mlp_forward_kernel(const qgtl_mlp_product_t g) {
    __shared__ __attribute__((aligned(16))) Lds sm;
    product<kForward>(g, blockIdx.x, sm);
}

// a layer's weight gradient w (its tiles first) and, in the same launch, the gradient x of its input
__global__ __launch_bounds__(kThreads) void mlp_backward_kernel(const qgtl_mlp_product_t w, const qgtl_mlp_product_t x) {
    __shared__ __attribute__((aligned(16))) Lds sm;
    const int tw = product_tiles(w);
    if ((int)blockIdx.x < tw) product<kWeightGrad>(w, blockIdx.x, sm);
    else product<kInputGrad>(x, (int)blockIdx.x - tw, sm);
}

__global__ void gather_rows_kernel(const float *__restrict__ src, const int *__restrict__ idx, int rows, int cols,
                                   float *dst) {
    const size_t total = (size_t)rows * cols;
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
        const size_t r = e / cols, c = e % cols;
        dst[e] = src[(size_t)idx[r] * cols + c];
    }
}

// Adam on the FP32 master copy; the BF16 mirror is what the GEMMs read.
__global__ void adam_kernel(float *w, uint16_t *w_bf16, float *m, float *v, const float *__restrict__ g, size_t n,
                            float lr, float b1, float b2, float eps, float c1, float c2) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        w[i] = wi;
        w_bf16[i] = bf16_rn(wi);
    }
}

__global__ void to_bf16_kernel(const float *__restrict__ w, uint16_t *out, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        out[i] = bf16_rn(w[i]);
}

constexpr int kMaxRank = 32;
constexpr int kMaxP = 1024;
constexpr int kMaxPR = 8192;    // P * r: the low-rank factor held in LDS as the network's fp32 outputs (32 KB)

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ double block_sum(double v, double *red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < kThreads / 64; w++) s += red[w];
    return s;
}

__device__ __forceinline__ double lane_value(double v, int lane) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Kaporin loss of sample b and dL/dy (scaled by `scale`), FP64.
//   s_k = y[k(1+r)], u_kj = y[k(1+r)+1+j] / sqrt(P), Mt = diag(e^s) + u u^T,
//   L = P log(tr(Mt As)/P) - sum s - log det(I + u^T e^-s u).
//
// One workgroup per sample.  A_s u, the bulk of the work, and the r x r matrix
// W = I + u^T e^-s u run on v_mfma_f64_16x16x4_f64 (A_s read once, a float4 per
// lane, exact in FP64; u scaled by 1/sqrt(P) in FP64 as it is read from LDS),
// A_s u kept in LDS for the trace and the gradient; W is factored by one wave
// (a row per lane) and inverted a column per lane.  What bounds it: the latency
// of the sample's serial steps (W's factor) and of reading A_s.  P = 192, r = 8,
// 256 samples: 42 us, from 278 us with a row of A_s per thread (uncoalesced),
// twice, an exponential per term of W and one thread factoring and inverting it.
//
// RT: 16-column tiles of the rank (1: r <= 16, 2: r <= 32); PR: bound on P r.
template <int RT, int PR>
__global__ __launch_bounds__(kThreads) void kaporin_kernel(int P, int r, const float *__restrict__ Y,
                                                           const float *__restrict__ As_all, const int *__restrict__ idx,
                                                           double *loss, float *dY, float scale, int vec) {
    constexpr int R = 16 * RT, MP = RT == 1 ? kMaxP : 512;   // r > 16: P <= 8192 / 17
    const int b = blockIdx.x;
    const float *y = Y + (size_t)b * P * (1 + r);
    const float *As = As_all + (size_t)idx[b] * P * P;
    float *dy = dY + (size_t)b * P * (1 + r);
    __shared__ float yu[PR];                      // u sqrt(P), row k at k * r
    __shared__ double au[PR];                     // A_s u, likewise
    __shared__ double es[MP], ems[MP];            // e^s, e^-s
    __shared__ double inv[R];                     // reciprocal diagonal of W's factor
    __shared__ double W[R * (R + 1)], Wi[R * (R + 1)], part[4][RT * RT][256];
    __shared__ double red[kThreads / 64];
    __shared__ double sh_logdet;
    const double us = 1.0 / sqrt((double)P);
    const int st = 1 + r;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int l16 = lane & 15, q4 = lane >> 4;
    for (int e = threadIdx.x; e < P * r; e += kThreads) yu[e] = y[(size_t)(e / r) * st + 1 + e % r];
    double trp = 0.0, ssum = 0.0;
    for (int k = threadIdx.x; k < P; k += kThreads) {
        const double s = y[(size_t)k * st], ek = exp(s);
        es[k] = ek;
        ems[k] = exp(-s);
        ssum += s;
        trp += ek * (double)As[(size_t)k * P + k];
    }
    __syncthreads();
    auto u_at = [&](int k, int j) -> double { return k < P && j < r ? (double)yu[k * r + j] * us : 0.0; };
    // A_s u: 16 rows a wave.  Lane l takes A_s[row l % 16][k .. k + 3], k = k0 + 4 (l / 16); product e
    // of a group of four sums over k0 + e, k0 + 4 + e, k0 + 8 + e, k0 + 12 + e, A and B alike.
    for (int r0 = 16 * wave; r0 < P && r > 0; r0 += 16 * (kThreads / 64)) {
        f64x4 acc[RT];
#pragma unroll
        for (int c = 0; c < RT; c++) acc[c] = f64x4{0.0, 0.0, 0.0, 0.0};
        const bool row_ok = r0 + l16 < P;
        const float *row = As + (size_t)(row_ok ? r0 + l16 : 0) * P;
        const int lim = row_ok ? P : 0;
        f32x4 a = load_run<4, f32x4>(row + 4 * q4, lim - 4 * q4, vec);
        for (int k0 = 0; k0 < P; k0 += 16) {
            const int kn = k0 + 16 + 4 * q4;
            const f32x4 an = load_run<4, f32x4>(row + kn, lim - kn, vec);
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int c = 0; c < RT; c++)
                    acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[e], u_at(k0 + 4 * q4 + e, 16 * c + l16), acc[c], 0, 0, 0);
            a = an;
        }
#pragma unroll
        for (int c = 0; c < RT; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int k = r0 + 4 * e + q4, j = 16 * c + l16;
                if (k < P && j < r) au[k * r + j] = acc[c][e];
            }
    }
    // W - I: each wave a quarter of the rows
    if (r > 0) {
        f64x4 acc[RT * RT];
#pragma unroll
        for (int c = 0; c < RT * RT; c++) acc[c] = f64x4{0.0, 0.0, 0.0, 0.0};
        for (int k0 = 4 * wave; k0 < P; k0 += 4 * (kThreads / 64)) {
            const int k = k0 + q4;
            double uj[RT];
#pragma unroll
            for (int c = 0; c < RT; c++) uj[c] = u_at(k, 16 * c + l16);
            const double ek = k < P ? ems[k] : 0.0;
#pragma unroll
            for (int c = 0; c < RT; c++)
#pragma unroll
                for (int d = 0; d < RT; d++)
                    acc[c * RT + d] = __builtin_amdgcn_mfma_f64_16x16x4f64(ek * uj[c], uj[d], acc[c * RT + d], 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < RT * RT; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) part[wave][c][(4 * e + q4) * 16 + l16] = acc[c][e];
    }
    __syncthreads();
    if (r > 0) {
        for (int e = threadIdx.x; e < P * r; e += kThreads) trp += ((double)yu[e] * us) * au[e];
        for (int e = threadIdx.x; e < R * R; e += kThreads) {
            const int i = e / R, j = e % R, c = (i / 16) * RT + j / 16, o = (i % 16) * 16 + j % 16;
            const double v = ((part[0][c][o] + part[1][c][o]) + part[2][c][o]) + part[3][c][o];
            W[i * (R + 1) + j] = v + (i == j ? 1.0 : 0.0);     // past r: the identity
        }
    }
    const double tr = block_sum(trp, red);                     // (barriers: W is complete after them)
    const double S = block_sum(ssum, red);
    if (wave == 0 && r > 0) {
        // Cholesky of W, a row per lane; then W^-1, a column per lane
        const int row = lane < R ? lane : R - 1;
        double ld = 0.0;
        {
            double a[R];
#pragma unroll
            for (int c = 0; c < R; c++) a[c] = W[row * (R + 1) + c];
#pragma unroll
            for (int j = 0; j < R; j++) {
                const double d = lane_value(a[j], j);
                if (lane == j) ld = log(d);
                const double ri = 1.0 / sqrt(d);
                if (lane == 0) inv[j] = ri;
                const double l = a[j] * ri;
                a[j] = l;
#pragma unroll
                for (int k = j + 1; k < R; k++) a[k] = fma(-l, lane_value(l, k), a[k]);
            }
            if (lane < R)
#pragma unroll
                for (int c = 0; c < R; c++) W[lane * (R + 1) + c] = a[c];
        }
        ld = lane < R ? ld : 0.0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ld += __shfl_xor(ld, o, 64);
        if (lane == 0) sh_logdet = ld;
        qgtl::wave_sync();                                     // inv and W's rows, by other lanes
        if constexpr (RT == 1) {
            double x[R];
#pragma unroll
            for (int i = 0; i < R; i++) {
                double v = i == row ? 1.0 : 0.0;
#pragma unroll
                for (int k = 0; k < i; k++) v = fma(-W[i * (R + 1) + k], x[k], v);
                x[i] = v * inv[i];
            }
            // the same elements of W, read again: kept from above they would spill
            __asm__ volatile("" ::: "memory");
#pragma unroll
            for (int i = R - 1; i >= 0; i--) {
                double v = x[i];
#pragma unroll
                for (int k = i + 1; k < R; k++) v = fma(-W[k * (R + 1) + i], x[k], v);
                x[i] = v * inv[i];
            }
            if (lane < R)
#pragma unroll
                for (int i = 0; i < R; i++) Wi[lane * (R + 1) + i] = x[i];
        } else if (lane < R) {
            // 32 unknowns and their rows do not fit the registers: the column lives in LDS
            double *x = Wi + row * (R + 1);
            for (int i = 0; i < R; i++) {
                double v = i == row ? 1.0 : 0.0;
#pragma unroll 4
                for (int k = 0; k < i; k++) v = fma(-W[i * (R + 1) + k], x[k], v);
                x[i] = v * inv[i];
            }
            for (int i = R - 1; i >= 0; i--) {
                double v = x[i];
#pragma unroll 4
                for (int k = i + 1; k < R; k++) v = fma(-W[k * (R + 1) + i], x[k], v);
                x[i] = v * inv[i];
            }
        }
    }
    if (threadIdx.x == 0 && r == 0) sh_logdet = 0.0;
    __syncthreads();
    if (threadIdx.x == 0) loss[b] = (double)P * log(tr / P) - S - sh_logdet;
    const double g = (double)P / tr;
    for (int k = threadIdx.x; k < P; k += kThreads) {
        double q = 0.0;
        for (int j = 0; j < r; j++) {
            double uw = 0.0;                                   // (u W^-1)_kj
            for (int c = 0; c < r; c++) uw += ((double)yu[k * r + c] * us) * Wi[c * (R + 1) + j];
            q += uw * ((double)yu[k * r + j] * us);
            dy[(size_t)k * st + 1 + j] = (float)(scale * (2.0 * g * au[k * r + j] - 2.0 * ems[k] * uw) * us);
        }
        dy[(size_t)k * st] = (float)(scale * (g * es[k] * (double)As[(size_t)k * P + k] - 1.0 + ems[k] * q));
    }
}

unsigned grid_1d(size_t n) {
    size_t g = (n + 255) / 256;
    if (g < 1) g = 1;
    if (g > 8192) g = 8192;
    return (unsigned)g;
}

}  // namespace

extern "C" {

static int product_ok(const qgtl_mlp_product_t *g) {
    return g && g->M >= 1 && g->N >= 1 && g->K >= 1 && g->A && g->B && g->C;
}

static unsigned product_grid(const qgtl_mlp_product_t *g) {
    return (unsigned)(((g->M + kTile - 1) / kTile) * ((g->N + kTile - 1) / kTile));
}

// whether the operand's vector loads (size bytes of a row start, every elems-th element) are aligned
static int vec_ok(const void *p, int ld, int bytes_per_elem, int bytes) {
    return (uintptr_t)p % (uintptr_t)bytes == 0 && ((size_t)ld * bytes_per_elem) % (size_t)bytes == 0;
}

int qgtl_hip_mlp_forward(const qgtl_mlp_product_t *desc) {
    if (!product_ok(desc) || !desc->bias) return qgtl::set_error_msg(-118, "mlp_forward: empty product");
    qgtl_mlp_product_t g = *desc;
    g.avec = vec_ok(g.A, g.lda, 4, 16);
    g.bvec = vec_ok(g.B, g.ldb, 2, 8);
    hipLaunchKernelGGL(mlp_forward_kernel, dim3(product_grid(&g)), dim3(kThreads), 0, qgtl::stream(), g);
    QGTL_LAUNCH_CHECK("mlp_forward");
    return 0;
}

int qgtl_hip_mlp_backward(const qgtl_mlp_product_t *weight, const qgtl_mlp_product_t *input) {
    if (!product_ok(weight) || !weight->colsum || (input && (!product_ok(input) || !input->pre)))
        return qgtl::set_error_msg(-118, "mlp_backward: empty product");
    qgtl_mlp_product_t w = *weight, x;
    w.avec = vec_ok(w.A, w.lda, 4, 16);
    w.bvec = vec_ok(w.B, w.ldb, 4, 16);
    x = input ? *input : w;
    unsigned grid = product_grid(&w);
    if (input) {
        x.avec = vec_ok(x.A, x.lda, 4, 16);
        x.bvec = vec_ok(x.B, x.ldb, 2, 16);
        grid += product_grid(&x);
    }
    hipLaunchKernelGGL(mlp_backward_kernel, dim3(grid), dim3(kThreads), 0, qgtl::stream(), w, x);
    QGTL_LAUNCH_CHECK("mlp_backward");
    return 0;
}

int qgtl_hip_gather_rows(const float *src, const int *idx, int rows, int cols, float *dst) {
    hipLaunchKernelGGL(gather_rows_kernel, dim3(grid_1d((size_t)rows * cols)), dim3(256), 0, qgtl::stream(), src,
                       idx, rows, cols, dst);
    QGTL_LAUNCH_CHECK("gather_rows");
    return 0;
}

int qgtl_hip_adam(float *w, uint16_t *w_bf16, float *m, float *v, const float *g, size_t n, float lr, float b1,
                  float b2, float eps, int step) {
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(adam_kernel, dim3(grid_1d(n)), dim3(256), 0, qgtl::stream(), w, w_bf16, m, v, g, n, lr, b1,
                       b2, eps, c1, c2);
    QGTL_LAUNCH_CHECK("adam");
    return 0;
}

int qgtl_hip_to_bf16(const float *w, uint16_t *out, size_t n) {
    hipLaunchKernelGGL(to_bf16_kernel, dim3(grid_1d(n)), dim3(256), 0, qgtl::stream(), w, out, n);
    QGTL_LAUNCH_CHECK("to_bf16");
    return 0;
}

int qgtl_hip_kaporin(int P, int r, int B, const float *Y, const float *As_all, const int *idx, double *loss,
                     float *dY, float scale) {
    if (P < 1 || P > kMaxP || r < 0 || r > kMaxRank || P * r > kMaxPR || B < 1)
        return qgtl::set_error_msg(-118, "kaporin: needs P <= 1024, r <= 32, P r <= 8192");
    const int vec = vec_ok(As_all, P, 4, 16);
#define QGTL_KAPORIN(RT, PR)                                                                                      \
    hipLaunchKernelGGL((kaporin_kernel<RT, PR>), dim3((unsigned)B), dim3(kThreads), 0, qgtl::stream(), P, r, Y,    \
                       As_all, idx, loss, dY, scale, vec)
    // up to P r = 2048 two workgroups share a CU's LDS
    if (r <= 16 && P * r <= 2048) QGTL_KAPORIN(1, 2048);
    else if (r <= 16) QGTL_KAPORIN(1, kMaxPR);
    else QGTL_KAPORIN(2, kMaxPR);
#undef QGTL_KAPORIN
    QGTL_LAUNCH_CHECK("kaporin");
    return 0;
}

}  // extern "C"
