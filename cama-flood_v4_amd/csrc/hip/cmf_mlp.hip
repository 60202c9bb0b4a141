// cmf_mlp.hip -- training and inference kernels of the spin-up surrogate, a
// per-cell multilayer perceptron (n_in -> H -> H -> H -> n_out, ReLU) that maps
// catchment attributes and runoff climatology to equilibrium river and
// floodplain storage. No reference counterpart: the reference spins up by
// repeating the forcing year (gosh/test1-glb_15min.sh:311-345).
//
// Arithmetic: BF16 operands on the matrix cores (v_mfma_f32_16x16x32_bf16),
// FP32 accumulation, FP32 master weights and Adam moments. Quantisation points
// (each is a round-to-nearest-even FP32 -> BF16 conversion):
//   forward : X, W_l              -> Z_l = X W_l + b_l (FP32), H_l = bf16(relu(Z_l))
//   output  : Y = H_3 W_4 + b_4 (FP32)
//   backward: G_Y = bf16(dL/dY); dW_l = H_{l-1}^T G_l (FP32); db_l = sum G_l (FP32);
//             G_{l-1} = bf16((G_l W_l^T) * [H_{l-1} > 0])
// The CPU oracle restates the same quantisation points.
//
// Networks of 256 hidden units (and at most 32 inputs, 16 outputs: the surrogate's
// own 24-256-256-256-2 among them) run as fused kernels, other sizes layer by layer.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "cmf_mlp.h"
#include "cmf_xfer.hpp"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

thread_local std::string m_err;
int mfail(int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    m_err = buf;
    return code;
}
#define MCHK(x)                                                                                  \
    do {                                                                                         \
        hipError_t e_ = (x);                                                                     \
        if (e_ != hipSuccess) return mfail(CMF_MLP_EHIP, "%s: %s", #x, hipGetErrorString(e_));   \
    } while (0)
#define MTRY(x)                 \
    do {                        \
        int r_ = (x);           \
        if (r_ != 0) return r_; \
    } while (0)

// FP32 -> BF16, round to nearest even (NaN kept quiet)
__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// ---------------------------------------------------------------------------
// C[M,N] (+)= op(A)[M,K] op(B)[K,N], A and B BF16, C FP32.
// op(A)(m,k) = ta ? A[k*lda+m] : A[m*lda+k];  op(B)(k,n) = tb ? B[n*ldb+k] : B[k*ldb+n].
// Block tile 64x64, K step 32, 256 threads = 4 wavefronts in 2x2, each 32x32 =
// 2x2 MFMA 16x16 tiles. Tiles are staged in LDS with k contiguous for both
// operands, so every lane reads its 8 consecutive k of one row/column with one
// 16-byte LDS load. MFMA 16x16x32 lane layout: lane l supplies A(row l%16,
// k 8*(l/16)..+7) and B(k 8*(l/16)..+7, col l%16) and receives
// D(row 4*(l/16)+r, col l%16), r = 0..3.
constexpr int TM = 64, TN = 64, TK = 32, LDK = TK + 8;   // +8 bf16 pad against bank conflicts

__global__ __launch_bounds__(256) void k_gemm_bf16(int M, int N, int K, const uint16_t* __restrict__ A, int lda,
                                                   int ta, const uint16_t* __restrict__ B, int ldb, int tb,
                                                   float* __restrict__ C, int ldc, int accumulate) {
    __shared__ __attribute__((aligned(16))) uint16_t As[TM * LDK];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[TN * LDK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += TK) {
        // stage op(A)[m0..+64, k0..+32] and op(B)[k0..+32, n0..+64]: 2048 values each
        for (int e = tid; e < TM * TK; e += 256) {
            int r, k;
            if (ta) { r = e % TM; k = e / TM; }     // consecutive threads walk m (contiguous in memory)
            else { r = e / TK; k = e % TK; }        // consecutive threads walk k
            const int gm = m0 + r, gk = k0 + k;
            uint16_t v = 0;
            if (gm < M && gk < K) v = ta ? A[(size_t)gk * lda + gm] : A[(size_t)gm * lda + gk];
            As[r * LDK + k] = v;
        }
        for (int e = tid; e < TN * TK; e += 256) {
            int c, k;
            if (tb) { c = e / TK; k = e % TK; }     // B[n*ldb+k]: k contiguous
            else { c = e % TN; k = e / TN; }        // B[k*ldb+n]: n contiguous
            const int gn = n0 + c, gk = k0 + k;
            uint16_t v = 0;
            if (gn < N && gk < K) v = tb ? B[(size_t)gn * ldb + gk] : B[(size_t)gk * ldb + gn];
            Bs[c * LDK + k] = v;
        }
        __syncthreads();
        const int fr = lane & 15, fk = (lane >> 4) * 8;
        bf16x8 a[2], b[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) a[i] = *reinterpret_cast<const bf16x8*>(&As[(wm + 16 * i + fr) * LDK + fk]);
#pragma unroll
        for (int j = 0; j < 2; ++j) b[j] = *reinterpret_cast<const bf16x8*>(&Bs[(wn + 16 * j + fr) * LDK + fk]);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        __syncthreads();
    }
    const int col = lane & 15, rq = (lane >> 4) * 4;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gm = m0 + wm + 16 * i + rq + r, gn = n0 + wn + 16 * j + col;
                if (gm < M && gn < N) {
                    float* c = &C[(size_t)gm * ldc + gn];
                    *c = accumulate ? *c + acc[i][j][r] : acc[i][j][r];
                }
            }
}

// FP32 -> BF16 copy
__global__ void k_to_bf16(const float* __restrict__ x, uint16_t* __restrict__ y, long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

// rows gathered by index (training batch) and converted to BF16
__global__ void k_gather_bf16(const float* __restrict__ x, const int64_t* __restrict__ idx, int rows, int cols,
                              uint16_t* __restrict__ y) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)rows * cols) return;
    const int r = (int)(i / cols), c = (int)(i % cols);
    y[i] = f2bf(x[(size_t)idx[r] * cols + c]);
}
__global__ void k_gather_f32(const float* __restrict__ x, const int64_t* __restrict__ idx, int rows, int cols,
                             float* __restrict__ y) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)rows * cols) return;
    const int r = (int)(i / cols), c = (int)(i % cols);
    y[i] = x[(size_t)idx[r] * cols + c];
}

// H = bf16(relu(Z + b)) (hidden layers); Y = Z + b (output layer, FP32 in place)
__global__ void k_bias_relu_bf16(const float* __restrict__ z, const float* __restrict__ b, int rows, int cols,
                                 uint16_t* __restrict__ h) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)rows * cols) return;
    const float v = z[i] + b[i % cols];
    h[i] = f2bf(v > 0.f ? v : 0.f);
}
__global__ void k_bias(float* __restrict__ z, const float* __restrict__ b, int rows, int cols) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (long long)rows * cols) z[i] = z[i] + b[i % cols];
}

// weighted mean squared error over rows*cols values, weight w_over where the
// prediction exceeds the target and 1 elsewhere: G = bf16(2 w (Y - T) / (rows*cols)),
// per-block partial sums of w (Y - T)^2 into part[blockIdx.x]
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ y, const float* __restrict__ t, int n,
                                             float w_over, uint16_t* __restrict__ g, float* __restrict__ part) {
    __shared__ float red[256];
    const int i = blockIdx.x * 256 + threadIdx.x;
    float e2 = 0.f;
    if (i < n) {
        const float d = y[i] - t[i];
        const float w = d > 0.f ? w_over : 1.f;
        e2 = w * (d * d);
        g[i] = f2bf((2.f * w) * d / (float)n);
    }
    red[threadIdx.x] = e2;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// G = bf16(D * [H > 0])
__global__ void k_relu_grad(const float* __restrict__ d, const uint16_t* __restrict__ h, long long n,
                            uint16_t* __restrict__ g) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) g[i] = (h[i] & 0x7fffu) != 0 && !(h[i] & 0x8000u) ? f2bf(d[i]) : (uint16_t)0;
}

// db[c] = sum over rows of G[r][c] (BF16 values, FP32 sums in a fixed order):
// chunk sums of COLSUM_CHUNK rows, then the chunk sums in chunk order
constexpr int COLSUM_CHUNK = 128;
__global__ void k_colsum_part(const uint16_t* __restrict__ g, int rows, int cols, float* __restrict__ part) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cols) return;
    const int r0 = blockIdx.y * COLSUM_CHUNK;
    const int r1 = r0 + COLSUM_CHUNK < rows ? r0 + COLSUM_CHUNK : rows;
    float s = 0.f;
    for (int r = r0; r < r1; ++r) s += bf2f(g[(size_t)r * cols + c]);
    part[(size_t)blockIdx.y * cols + c] = s;
}
__global__ void k_colsum_final(const float* __restrict__ part, int nchunk, int cols, float* __restrict__ db) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cols) return;
    float s = 0.f;
    for (int k = 0; k < nchunk; ++k) s += part[(size_t)k * cols + c];
    db[c] = s;
}

// Adam with bias correction, FP32 master parameters
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m1,
                       float* __restrict__ m2, long long n, float lr, float b1, float b2, float eps, float c1,
                       float c2) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float a = b1 * m1[i] + (1.f - b1) * gi;
    const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    p[i] = p[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
}

// ---------------------------------------------------------------------------
// Fused kernels for H = 256. Every layer but the weight gradients maps rows to rows,
// so one workgroup takes a tile of RT rows through the whole network, forward and,
// for a gradient, back again, with the activations in LDS: nothing but the inputs,
// the outputs and what the weight gradients need touches HBM. The products are
// formed transposed (features x rows): a wavefront owns 64 features, its weight
// fragments come straight from L2 with 16-byte loads (two layouts of the weights are
// kept, k contiguous for either direction), and a lane ends with four consecutive
// features of a row, one 8-byte LDS store for the next layer's operand. Each output
// is one accumulator over ascending k in steps of 32, as in k_gemm_bf16.
constexpr int FH = 256, FKI = 32, FNO = 16;     // hidden units, padded inputs and outputs
constexpr int LDX = FKI + 8, LDH = FH + 8;      // LDS rows, padded against bank conflicts

struct FusedNet {
    const uint16_t *wt[4];                      // W_l transposed [dout][din]: forward (rows >= dout and k >= din zero)
    const uint16_t *w[4];                       // W_l [din][dout]: backward (w[3] padded to 32 columns)
    const float* b[4];
    int n_in, n_out;
};
struct FusedTrain {
    const float* t;                             // targets
    const int64_t* idx;                         // rows of x and t, or NULL
    float w_over;
    float* y;                                   // outputs [rows][n_out]
    uint16_t *xt, *ht[3], *gt[4];               // transposed [feature][ld]: inputs, hidden values, gradients
    int ld;
};

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// acc[i][j] = A(16 features i) x B(16 rows j) over NK steps of 32 k. The weights of the
// next D steps are in flight: all of a layer's for the small tiles, whose products
// would otherwise wait for one L2 round trip each.
template <int NJ, int NK>
__device__ __forceinline__ void tile_product(const uint16_t* __restrict__ A, int lda, const uint16_t* Bs, int ldb,
                                             f32x4 (&acc)[4][NJ]) {
    constexpr int D = NK == 1 ? 1 : (NJ <= 2 ? 8 : 2);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int lane = threadIdx.x & 63, fr = lane & 15, fk = (lane >> 4) * 8;
    const uint16_t* a0 = A + (size_t)fr * lda + fk;
    const uint16_t* b0 = Bs + fr * ldb + fk;
    bf16x8 a[D][4];
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i) a[d][i] = *reinterpret_cast<const bf16x8*>(a0 + (size_t)16 * i * lda + 32 * d);
    if (D > 1) asm volatile("" ::: "memory");                       // the loads stay here, ahead of their uses
#pragma unroll
    for (int kb = 0; kb < NK; kb += D) {
        bf16x8 an[D][4];
        if (kb + D < NK)
#pragma unroll
            for (int d = 0; d < D; ++d)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    an[d][i] = *reinterpret_cast<const bf16x8*>(a0 + (size_t)16 * i * lda + 32 * (kb + D + d));
#pragma unroll
        for (int d = 0; d < D; ++d)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const bf16x8 b = *reinterpret_cast<const bf16x8*>(b0 + 16 * j * ldb + 32 * (kb + d));
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i][j] = mfma(a[d][i], b, acc[i][j]);
            }
        if (kb + D < NK)
#pragma unroll
            for (int d = 0; d < D; ++d)
#pragma unroll
                for (int i = 0; i < 4; ++i) a[d][i] = an[d][i];
    }
}

// Workgroup barrier for data in LDS only: the stores of the transposed activations
// stay in flight across it (no other thread of the launch reads them)
__device__ __forceinline__ void sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Measured (24-256-256-256-2): a chunk of the inference, 16,384 rows, 27 us, 169 TFLOP/s,
// one tile of 64 rows per CU (layer kernels: 112 us); a gradient's pass over 1024
// rows 29 us and over 4099 rows 38 us, bound by the chain of seven layers on one
// wavefront per SIMD (layer kernels, forward and backward with k_mlp_dw's part: 860 us
// and 2.4 ms).
template <int RT, bool TRAIN>
__global__ __launch_bounds__(256) void k_mlp_fused(FusedNet N, FusedTrain G, const float* __restrict__ x, int rows,
                                                   float* __restrict__ yout) {
    constexpr int NJ = RT / 16, NM = (NJ * 16 + 31) / 32;
    __shared__ __attribute__((aligned(16))) uint16_t Xs[RT * LDX];
    __shared__ __attribute__((aligned(16))) uint16_t Hs[RT * LDH];
    __shared__ __attribute__((aligned(16))) uint16_t Ys[TRAIN ? RT * LDX : 8];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r0 = blockIdx.x * RT, f0 = 64 * wave;
    const int row_l = lane & 15, q4 = (lane >> 4) * 4;
    // inputs: 8 threads a row, 4 columns each
    for (int e = tid; e < RT * 8; e += 256) {
        const int r = e >> 3, c0 = (e & 7) * 4, gr = r0 + r;
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        if (gr < rows) {
            const float* src = x + (size_t)(TRAIN && G.idx ? G.idx[gr] : gr) * N.n_in + c0;
            if ((N.n_in & 3) == 0) {
                if (c0 < N.n_in) {
                    const float4 u = *reinterpret_cast<const float4*>(src);
                    v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
                }
            } else {
                for (int k = 0; k < 4; ++k) if (c0 + k < N.n_in) v[k] = src[k];
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint16_t u = f2bf(v[k]);
            Xs[r * LDX + c0 + k] = u;
            if (TRAIN) {
                if (c0 + k < N.n_in) G.xt[(size_t)(c0 + k) * G.ld + gr] = u;
                Ys[r * LDX + c0 + k] = 0;
            }
        }
    }
    sync_lds();
    f32x4 acc[4][NJ];
    uint32_t mask[3][NM];
    // forward, hidden layers
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        float4 bias[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) bias[i] = *reinterpret_cast<const float4*>(N.b[l] + f0 + 16 * i + q4);
        asm volatile("" ::: "memory");
        if (l == 0) tile_product<NJ, 1>(N.wt[0] + (size_t)f0 * FKI, FKI, Xs, LDX, acc);
        else tile_product<NJ, FH / 32>(N.wt[l] + (size_t)f0 * FH, FH, Hs, LDH, acc);
        if (l > 0) sync_lds();                                // every wavefront has read the old values
#pragma unroll
        for (int m = 0; m < NM; ++m) mask[l][m] = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n0 = f0 + 16 * i + q4;
            const float4 b = bias[i];
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int r = 16 * j + row_l;
                const float v[4] = {acc[i][j][0] + b.x, acc[i][j][1] + b.y, acc[i][j][2] + b.z, acc[i][j][3] + b.w};
                uint16_t u[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    u[k] = f2bf(v[k] > 0.f ? v[k] : 0.f);
                    if (TRAIN) {
                        const int bit = (i * NJ + j) * 4 + k;
                        if ((u[k] & 0x7fffu) != 0 && !(u[k] & 0x8000u)) mask[l][bit >> 5] |= 1u << (bit & 31);
                        G.ht[l][(size_t)(n0 + k) * G.ld + r0 + r] = r0 + r < rows ? u[k] : (uint16_t)0;
                    }
                }
                uint2 p;
                p.x = (uint32_t)u[0] | ((uint32_t)u[1] << 16);
                p.y = (uint32_t)u[2] | ((uint32_t)u[3] << 16);
                *reinterpret_cast<uint2*>(&Hs[r * LDH + n0]) = p;
            }
        }
        sync_lds();
    }
    // output layer: a wavefront takes every fourth tile of rows
    for (int j = wave; j < NJ; j += 4) {
        f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
        const int fk = (lane >> 4) * 8;
#pragma unroll
        for (int k = 0; k < FH / 32; ++k)
            o = mfma(*reinterpret_cast<const bf16x8*>(N.wt[3] + row_l * FH + 32 * k + fk),
                     *reinterpret_cast<const bf16x8*>(&Hs[(16 * j + row_l) * LDH + 32 * k + fk]), o);
        const int r = 16 * j + row_l, gr = r0 + r;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int n = q4 + k;
            if (n < N.n_out) {
                const float yv = o[k] + N.b[3][n];
                if (gr < rows) yout[(size_t)gr * N.n_out + n] = yv;
                if (TRAIN) {
                    uint16_t u = 0;
                    if (gr < rows) {
                        const float d = yv - G.t[(size_t)(G.idx ? G.idx[gr] : gr) * N.n_out + n];
                        const float w = d > 0.f ? G.w_over : 1.f;
                        u = f2bf((2.f * w) * d / (float)(rows * N.n_out));
                    }
                    Ys[r * LDX + n] = u;
                    G.gt[3][(size_t)n * G.ld + gr] = u;
                }
            }
        }
    }
    if (!TRAIN) return;
    // backward: G_(l-1) = (W_l G_l) where H_(l-1) > 0
    sync_lds();
#pragma unroll
    for (int l = 3; l > 0; --l) {
        if (l == 3) tile_product<NJ, 1>(N.w[3] + (size_t)f0 * FKI, FKI, Ys, LDX, acc);
        else tile_product<NJ, FH / 32>(N.w[l] + (size_t)f0 * FH, FH, Hs, LDH, acc);
        sync_lds();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n0 = f0 + 16 * i + q4;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int r = 16 * j + row_l;
                uint16_t u[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int bit = (i * NJ + j) * 4 + k;
                    const bool on = (mask[l - 1][bit >> 5] >> (bit & 31)) & 1u;
                    u[k] = on && r0 + r < rows ? f2bf(acc[i][j][k]) : (uint16_t)0;
                    G.gt[l - 1][(size_t)(n0 + k) * G.ld + r0 + r] = u[k];
                }
                if (l > 1) {
                    uint2 p;
                    p.x = (uint32_t)u[0] | ((uint32_t)u[1] << 16);
                    p.y = (uint32_t)u[2] | ((uint32_t)u[3] << 16);
                    *reinterpret_cast<uint2*>(&Hs[r * LDH + n0]) = p;
                }
            }
        }
        sync_lds();
    }
}

// Gradients of the weights and biases and the loss, one wavefront per block:
//  * dW_l = H_(l-1)^T G_l, a 32 x 32 tile each; both operands are stored with the rows
//    (the k of this product) contiguous, so fragments are 16-byte loads and need no
//    LDS. Batches of more than DW_ROWS rows are split (blockIdx.y) and summed after.
//  * db_l: chunk sums of COLSUM_CHUNK rows, then the chunk sums in chunk order
//  * partial sums of the loss over 256 values
// 9 us for 1024 rows, 26 us for 4099: bound by the serial sum over the rows on 144
// wavefronts, which keeps the order of the sums; longer batches are split.
constexpr int DW_ROWS = 8192;
constexpr int DW_TILES = 8 + 64 + 64 + 8;
__global__ __launch_bounds__(64) void k_mlp_dw(FusedNet N, FusedTrain G, int rows, int rows_per, float* __restrict__ gw,
                                               size_t g_stride, float* __restrict__ g, const int* __restrict__ off /* w0 b0 w1 ... */,
                                               float* __restrict__ part) {
    const int lane = threadIdx.x, ndb = (3 * FH + N.n_out + 1) / 2;
    if (blockIdx.x < DW_TILES) {
        int t = blockIdx.x, l = 0;
        if (t >= 136) { l = 3; t -= 136; }
        else if (t >= 72) { l = 2; t -= 72; }
        else if (t >= 8) { l = 1; t -= 8; }
        const int nt = l == 3 ? 1 : 8;                              // tiles along the columns
        const int m0 = 32 * (t / nt), n0 = 32 * (t % nt);
        const int din = l == 0 ? N.n_in : FH, dout = l == 3 ? N.n_out : FH;
        const uint16_t* A = l == 0 ? G.xt : G.ht[l - 1];
        const uint16_t* B = G.gt[l];
        const int k0 = blockIdx.y * rows_per;
        const int k1 = k0 + rows_per < rows ? k0 + rows_per : (rows + 31) & ~31;
        const int fr = lane & 15, fk = (lane >> 4) * 8;
        const bool two = l != 3;                                    // 16 output columns at most
        const uint16_t* a0 = A + (size_t)(m0 + fr) * G.ld + fk;
        const uint16_t* b0 = B + (size_t)(n0 + fr) * G.ld + fk;
        const size_t step = (size_t)16 * G.ld, step_b = two ? step : 0;
        f32x4 acc[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        constexpr int U = 8;                                        // steps in flight
        bf16x8 a[U][2], b[U][2];
        auto fetch = [&](int k, bf16x8 (&fa)[2], bf16x8 (&fb)[2]) {
            const int kk = k < k1 ? k : k0;                         // past the end: loaded, not used
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                fa[i] = *reinterpret_cast<const bf16x8*>(a0 + i * step + kk);
                fb[i] = *reinterpret_cast<const bf16x8*>(b0 + i * step_b + kk);
            }
        };
#pragma unroll
        for (int u = 0; u < U; ++u) fetch(k0 + 32 * u, a[u], b[u]);
        for (int k = k0; k < k1; k += 32 * U) {
            bf16x8 an[U][2], bn[U][2];
#pragma unroll
            for (int u = 0; u < U; ++u) fetch(k + 32 * (U + u), an[u], bn[u]);
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k + 32 * u < k1) {
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j) acc[i][j] = mfma(a[u][i], b[u][j], acc[i][j]);
                }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < 2; ++i) { a[u][i] = an[u][i]; b[u][i] = bn[u][i]; }
        }
        float* C = gw + blockIdx.y * g_stride + off[2 * l];
        const int rq = (lane >> 4) * 4;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int gm = m0 + 16 * i + rq + r, gn = n0 + 16 * j + fr;
                    if (gm < din && gn < dout && (two || j == 0)) C[(size_t)gm * dout + gn] = acc[i][j][r];
                }
        return;
    }
    if (blockIdx.y != 0) return;
    const int q = blockIdx.x - DW_TILES;
    if (q < ndb) {                                                  // two features, 32 chunks at a time
        const int f = 2 * q + (lane >> 5), c = lane & 31;
        const int l = f < 3 * FH ? f / FH : 3, n = f - l * FH;
        const bool on = l < 3 || n < N.n_out;
        const uint16_t* src = G.gt[l] + (size_t)(on ? n : 0) * G.ld;
        const int nchunk = (rows + COLSUM_CHUNK - 1) / COLSUM_CHUNK;
        float total = 0.f;
        for (int cb = 0; cb < nchunk; cb += 32) {
            float s = 0.f;
            const int ch = cb + c;
            if (ch < nchunk) {
                const int ra = ch * COLSUM_CHUNK, rb = ra + COLSUM_CHUNK < rows ? ra + COLSUM_CHUNK : rows;
                int r = ra;
                for (; r + 8 <= rb; r += 8) {
                    const uint4 v = *reinterpret_cast<const uint4*>(src + r);
                    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        s += __uint_as_float(w[k] << 16);
                        s += __uint_as_float(w[k] & 0xffff0000u);
                    }
                }
                for (; r < rb; ++r) s += bf2f(src[r]);
            }
            const int last = nchunk - cb < 32 ? nchunk - cb : 32;
            for (int k = 0; k < last; ++k) total += __shfl(s, (lane & 32) + k, 64);
        }
        if (c == 0 && on) g[off[2 * l + 1] + n] = total;
        return;
    }
    // loss: the pairwise tree of k_mse over 256 values, four of them per lane
    const int i0 = (q - ndb) * 256, ny = rows * N.n_out;
    float e[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int i = i0 + 64 * k + lane;
        e[k] = 0.f;
        if (i < ny) {
            const int r = i / N.n_out, n = i % N.n_out;
            const float d = G.y[i] - G.t[(size_t)(G.idx ? G.idx[r] : r) * N.n_out + n];
            const float w = d > 0.f ? G.w_over : 1.f;
            e[k] = w * (d * d);
        }
    }
    float s = (e[0] + e[2]) + (e[1] + e[3]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
    if (lane == 0) part[q - ndb] = s;
}

// the split weight gradients in order
__global__ void k_sum_splits(const float* __restrict__ p, size_t stride, int ns, const int* __restrict__ off, int n_in,
                             int n_out, float* __restrict__ g, long long np) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    for (int l = 0; l < 4; ++l)
        if (i >= off[2 * l + 1] && i < off[2 * l + 1] + (l == 3 ? n_out : FH)) return;   // biases are not split
    float s = 0.f;
    for (int k = 0; k < ns; ++k) s += p[(size_t)k * stride + i];
    g[i] = s;
}

// BF16 copies of the weights in the layouts of the fused kernels; with m1: after an
// Adam step (bias correction c1, c2)
__global__ void k_adam_fused(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m1,
                             float* __restrict__ m2, long long n, float lr, float b1, float b2, float eps, float c1,
                             float c2, const int* __restrict__ off, int n_in, int n_out, uint16_t* __restrict__ wbf,
                             uint16_t* __restrict__ wt, uint16_t* __restrict__ w3) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float v = p[i];
    if (m1) {
        const float gi = g[i];
        const float a = b1 * m1[i] + (1.f - b1) * gi;
        const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
        m1[i] = a;
        m2[i] = b;
        v = v - lr * (a / c1) / (sqrtf(b / c2) + eps);
        p[i] = v;
    }
    const uint16_t u = f2bf(v);
    wbf[i] = u;
    const int l = i < off[2] ? 0 : (i < off[4] ? 1 : (i < off[6] ? 2 : 3));
    const int e = (int)i - off[2 * l], dout = l == 3 ? n_out : FH, din = l == 0 ? n_in : FH;
    if (e >= din * dout) return;                                     // a bias
    const int k = e / dout, m = e % dout;
    const int base = l == 0 ? 0 : FH * FKI + (l - 1) * FH * FH;
    wt[base + m * (l == 0 ? FKI : FH) + k] = u;
    if (l == 3) w3[k * FKI + m] = u;
}

inline unsigned nblk(long long n, int bs = 256) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

// ===========================================================================
struct cmf_mlp {
    int n_in = 0, hid = 0, n_out = 0, max_batch = 0;
    hipStream_t stream = nullptr;
    std::vector<void*> allocs;
    long long np = 0;                      // parameter count
    long long off_w[4], off_b[4];          // offsets in the packed parameter vector
    int din[4], dout[4];
    float *p = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;   // FP32 master, grads, Adam moments
    uint16_t* wbf = nullptr;               // BF16 copy of the parameters (weights used by the GEMMs)
    // batch buffers
    uint16_t* xb = nullptr;                // [B][n_in]
    uint16_t* hb[3] = {nullptr, nullptr, nullptr};   // [B][H]
    float* z = nullptr;                    // [B][max(H, n_out)] FP32 pre-activation / products
    float* y = nullptr;                    // [B][n_out]
    float* t = nullptr;                    // [B][n_out] targets
    uint16_t* gy = nullptr;                // [B][n_out]
    uint16_t* gh[2] = {nullptr, nullptr};  // [B][H] ping-pong
    float* part = nullptr;                 // loss partial sums
    float* colpart = nullptr;              // bias-gradient chunk sums
    int64_t* idx = nullptr;                // batch row indices
    // resident training set
    float *tx = nullptr, *tt = nullptr;
    long long tn = 0;
    float* h_scratch = nullptr;            // pinned
    float w_over = 1.f;                    // loss weight of over-predictions
    // fused kernels (256 hidden units)
    bool fused = false;
    int ld = 0;                            // row length of the transposed arrays
    uint16_t *wt = nullptr, *w3 = nullptr; // weights transposed; W_4 padded to 32 columns
    int* off = nullptr;                    // offsets of W and b in the packed parameters (device)
    uint16_t *xt = nullptr, *ht[3] = {nullptr, nullptr, nullptr};
    uint16_t* gt[4] = {nullptr, nullptr, nullptr, nullptr};
    float* gsplit = nullptr;               // split weight gradients
    float* xd = nullptr;                   // FP32 inputs of a host call
    cmf::Pinned fwd_pin;                   // slots of the chunked inference: x and y; x on the device
    float* fwd_x = nullptr;
    int fwd_slots = 0;
    hipStream_t fwd_stream[4] = {nullptr, nullptr, nullptr, nullptr};
    float* lossbuf = nullptr;              // loss partial sums of every batch of a training call
    size_t loss_cap = 0;
    int64_t* order = nullptr;              // row order of a training call
    size_t order_cap = 0;
};

namespace {

template <class T>
int malloc_t(cmf_mlp* h, T** p, size_t n) {
    void* q = nullptr;
    MCHK(hipMalloc(&q, (n ? n : 1) * sizeof(T)));
    MCHK(hipMemsetAsync(q, 0, (n ? n : 1) * sizeof(T), h->stream));
    MCHK(hipStreamSynchronize(h->stream));
    h->allocs.push_back(q);
    *p = static_cast<T*>(q);
    return 0;
}

void gemm(cmf_mlp* h, int M, int N, int K, const uint16_t* A, int lda, int ta, const uint16_t* B, int ldb, int tb,
          float* C, int ldc, int acc) {
    dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM);
    hipLaunchKernelGGL(k_gemm_bf16, grid, dim3(256), 0, h->stream, M, N, K, A, lda, ta, B, ldb, tb, C, ldc, acc);
}

// forward pass of `rows` BF16 input rows in h->xb; output FP32 in h->y
void forward(cmf_mlp* h, int rows) {
    const uint16_t* in = h->xb;
    for (int l = 0; l < 3; ++l) {
        gemm(h, rows, h->dout[l], h->din[l], in, h->din[l], 0, h->wbf + h->off_w[l], h->dout[l], 0, h->z,
             h->dout[l], 0);
        hipLaunchKernelGGL(k_bias_relu_bf16, dim3(nblk((long long)rows * h->dout[l])), dim3(256), 0, h->stream, h->z,
                           h->p + h->off_b[l], rows, h->dout[l], h->hb[l]);
        in = h->hb[l];
    }
    gemm(h, rows, h->n_out, h->hid, in, h->hid, 0, h->wbf + h->off_w[3], h->n_out, 0, h->y, h->n_out, 0);
    hipLaunchKernelGGL(k_bias, dim3(nblk((long long)rows * h->n_out)), dim3(256), 0, h->stream, h->y,
                       h->p + h->off_b[3], rows, h->n_out);
}

// device buffer of at least n values kept with the handle
template <class T>
int grow(cmf_mlp* h, T** p, size_t* cap, size_t n) {
    if (n <= *cap) return 0;
    if (*p) {
        MCHK(hipStreamSynchronize(h->stream));
        for (void*& q : h->allocs) if (q == (void*)*p) { (void)hipFree(q); q = nullptr; }
        *p = nullptr;
        *cap = 0;
    }
    MTRY(malloc_t(h, p, n));
    *cap = n;
    return 0;
}

int loss_parts(const cmf_mlp* h, int rows) { return (int)nblk((long long)rows * h->n_out); }

FusedNet fused_net(const cmf_mlp* h) {
    FusedNet N{};
    const size_t o[4] = {0, FH * FKI, FH * FKI + FH * FH, FH * FKI + 2 * FH * FH};
    for (int l = 0; l < 4; ++l) {
        N.wt[l] = h->wt + o[l];
        N.w[l] = l == 3 ? h->w3 : h->wbf + h->off_w[l];
        N.b[l] = h->p + h->off_b[l];
    }
    N.n_in = h->n_in; N.n_out = h->n_out;
    return N;
}

// Rows per workgroup: small batches need many workgroups more than large tiles
// (1024 rows fill 64 of them with 16 rows); from 8192 rows on, 64-row tiles keep the
// matrix cores busy and read the weights once per 64 rows. Larger ones have no use: a
// chunk of the inference is 16,384 rows, and the masks and accumulators of a gradient
// would spill.
template <bool TRAIN>
void launch_fused(cmf_mlp* h, const FusedTrain& G, const float* x, int rows, float* y, hipStream_t st) {
    const FusedNet N = fused_net(h);
    const int pad = TRAIN ? (rows + 31) & ~31 : rows;                // the weight gradients read whole 32-row steps
    auto blocks = [&](int rt) { return dim3((pad + rt - 1) / rt); };
    if (rows <= 4096)
        hipLaunchKernelGGL((k_mlp_fused<16, TRAIN>), blocks(16), dim3(256), 0, st, N, G, x, rows, y);
    else if (rows <= 8192)
        hipLaunchKernelGGL((k_mlp_fused<32, TRAIN>), blocks(32), dim3(256), 0, st, N, G, x, rows, y);
    else
        hipLaunchKernelGGL((k_mlp_fused<64, TRAIN>), blocks(64), dim3(256), 0, st, N, G, x, rows, y);
}

// slots of the chunked inference: rows of x and y in pinned memory, x on the device
constexpr int FWD_ROWS = 16384, FWD_STREAMS = 4;
int grow_forward(cmf_mlp* h, int slots) {
    if (slots <= h->fwd_slots) return 0;
    const size_t nx = (size_t)FWD_ROWS * h->n_in, ny = (size_t)FWD_ROWS * h->n_out;
    MCHK(h->fwd_pin.grow((size_t)slots * (nx + ny) * sizeof(float)));
    float* q = nullptr;
    MTRY(malloc_t(h, &q, (size_t)slots * nx));
    if (h->fwd_x) {
        (void)hipFree(h->fwd_x);
        for (size_t k = 0; k < h->allocs.size(); ++k)
            if (h->allocs[k] == (void*)h->fwd_x) { h->allocs.erase(h->allocs.begin() + (long)k); break; }
    }
    h->fwd_x = q;
    h->fwd_slots = slots;
    return 0;
}

int dw_splits(int rows) {
    const int ns = (rows - 1) / DW_ROWS + 1;
    return ns < 64 ? ns : 64;
}

// Buffers of the fused kernels, all of them with the handle: made in the first gradient,
// a failed allocation left some of them to the next call, and that gradient, of 64 rows,
// took 0.25 ms with max_batch 1,024 and 0.9 ms with 65,536 (0.07 ms now)
int alloc_fused(cmf_mlp* h) {
    // whole tiles, and an odd number of 256-byte pieces a row: with a power of two the
    // same rows of all features would meet in one or two L2 channels
    size_t ld = ((size_t)h->max_batch + 127) & ~(size_t)127;
    if (ld / 128 % 2 == 0) ld += 128;
    uint16_t* q = nullptr;                                // one allocation: eight took 0.2 ms longer
    MTRY(malloc_t(h, &q, (size_t)(6 * FH + FNO + FKI) * ld));
    for (auto& p : h->ht) { p = q; q += FH * ld; }
    for (int l = 0; l < 4; ++l) { h->gt[l] = q; q += (l == 3 ? FNO : FH) * ld; }
    h->xt = q;
    if (ld > 0x7fffffff) return mfail(CMF_MLP_EINVAL, "max_batch too large");
    h->ld = (int)ld;
    const int ns = dw_splits(h->max_batch);
    if (ns > 1) MTRY(malloc_t(h, &h->gsplit, (size_t)ns * (size_t)h->np));
    (void)grow_forward(h, 1);                             // inference can do without
    return 0;
}

// forward and backward of a batch by the fused kernels; gradients into h->g, loss
// partial sums into part. x, t: device arrays, rows picked by idx (NULL: in order)
int fused_grad(cmf_mlp* h, const float* x, const float* t, const int64_t* idx, int rows, float* part) {
    FusedTrain G{};
    G.t = t; G.idx = idx; G.w_over = h->w_over; G.y = h->y;
    G.xt = h->xt; G.ld = h->ld;
    for (int l = 0; l < 3; ++l) G.ht[l] = h->ht[l];
    for (int l = 0; l < 4; ++l) G.gt[l] = h->gt[l];
    const int ns = dw_splits(rows);
    const int per = ((rows + ns - 1) / ns + 31) & ~31;
    launch_fused<true>(h, G, x, rows, h->y, h->stream);
    const unsigned nb = DW_TILES + (unsigned)((3 * FH + h->n_out + 1) / 2) + (unsigned)loss_parts(h, rows);
    float* dst = ns > 1 ? h->gsplit : h->g;
    hipLaunchKernelGGL(k_mlp_dw, dim3(nb, ns), dim3(64), 0, h->stream, fused_net(h), G, rows, per, dst, (size_t)h->np,
                       h->g, h->off, part);
    if (ns > 1)
        hipLaunchKernelGGL(k_sum_splits, dim3(nblk(h->np)), dim3(256), 0, h->stream, h->gsplit, (size_t)h->np, ns, h->off,
                           h->n_in, h->n_out, h->g, h->np);
    MCHK(hipGetLastError());
    return 0;
}

// Inference over any number of rows in chunks of FWD_ROWS: copied into a pinned slot
// by one of several threads, sent, computed, written by the kernel into the slot and
// copied out, chunks in flight on FWD_STREAMS streams. Bound by the host's copies and
// PCIe (96 bytes a row): 1,500,120 rows 2.9 ms, 51 GB/s (one pageable copy, kernel and
// copy back after another 7.1; chunks of 8,192 rows 3.9, of 4,096 6.2: the launches of
// a chunk cost about 20 us).
int forward_fused(cmf_mlp* h, const float* x, int64_t n, float* y) {
    const int64_t nc = (n + FWD_ROWS - 1) / FWD_ROWS;
    if (nc > 0x7fffffff) return mfail(CMF_MLP_EINVAL, "too many rows");
    const int slots = (int)std::min<int64_t>(nc, cmf::XFER_SLOTS);
    const size_t nx = (size_t)FWD_ROWS * h->n_in, ny = (size_t)FWD_ROWS * h->n_out;
    if (grow_forward(h, slots) != 0) {
        // no pinned memory: pageable copies, one chunk after another
        (void)hipGetLastError();
        const int64_t most = std::min(FWD_ROWS, h->max_batch);
        for (int64_t r0 = 0; r0 < n; r0 += most) {
            const size_t rows = (size_t)std::min(most, n - r0);
            MCHK(hipMemcpyAsync(h->xd, x + (size_t)r0 * h->n_in, rows * h->n_in * sizeof(float), hipMemcpyHostToDevice, h->stream));
            launch_fused<false>(h, FusedTrain{}, h->xd, (int)rows, h->y, h->stream);
            MCHK(hipGetLastError());
            MCHK(hipMemcpyAsync(y + (size_t)r0 * h->n_out, h->y, rows * h->n_out * sizeof(float), hipMemcpyDeviceToHost, h->stream));
            MCHK(hipStreamSynchronize(h->stream));
        }
        return 0;
    }
    float* const pin = reinterpret_cast<float*>(h->fwd_pin.p);
    auto rows_of = [n](int64_t c) { return (int)std::min<int64_t>(FWD_ROWS, n - c * FWD_ROWS); };
    auto start_on = [&](int c, int slot, hipStream_t st) -> hipError_t {
        const int rows = rows_of(c);
        float *px = pin + (size_t)slot * (nx + ny), *dx = h->fwd_x + (size_t)slot * nx;
        const size_t bytes = (size_t)rows * h->n_in * sizeof(float);
        std::memcpy(px, x + (size_t)c * nx, bytes);
        const hipError_t e = hipMemcpyAsync(dx, px, bytes, hipMemcpyHostToDevice, st);
        if (e != hipSuccess) return e;
        launch_fused<false>(h, FusedTrain{}, dx, rows, px + nx, st);
        return hipGetLastError();
    };
    auto finish = [&](int c, int slot) {
        std::memcpy(y + (size_t)c * ny, pin + (size_t)slot * (nx + ny) + nx, (size_t)rows_of(c) * h->n_out * sizeof(float));
    };
    if (nc == 1) {
        MCHK(start_on(0, 0, h->stream));
        MCHK(hipStreamSynchronize(h->stream));
        finish(0, 0);
        return 0;
    }
    for (hipStream_t& st : h->fwd_stream)
        if (!st) MCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    int device = 0;
    MCHK(hipGetDevice(&device));
    MCHK(hipStreamSynchronize(h->stream));                            // the weights
    const hipError_t e = cmf::run_chunks((int)nc, device, [&](int c, int slot, hipEvent_t ev) -> hipError_t {
        const hipStream_t st = h->fwd_stream[slot % FWD_STREAMS];
        const hipError_t r = start_on(c, slot, st);
        return r != hipSuccess ? r : hipEventRecord(ev, st);
    }, finish);
    if (e != hipSuccess)
        for (hipStream_t st : h->fwd_stream) (void)hipStreamSynchronize(st);   // the slots are the next call's
    MCHK(e);
    return 0;
}

double loss_of(const float* part, int n) {
    double s = 0.0;
    for (int b = 0; b < n; ++b) s += part[b];
    return s;
}

void refresh_bf16(cmf_mlp* h) {
    if (h->fused) {
        hipLaunchKernelGGL(k_adam_fused, dim3(nblk(h->np)), dim3(256), 0, h->stream, h->p, (const float*)nullptr,
                           (float*)nullptr, (float*)nullptr, h->np, 0.f, 0.f, 0.f, 0.f, 1.f, 1.f, h->off, h->n_in, h->n_out,
                           h->wbf, h->wt, h->w3);
        return;
    }
    hipLaunchKernelGGL(k_to_bf16, dim3(nblk(h->np)), dim3(256), 0, h->stream, h->p, h->wbf, h->np);
}

// forward + backward of a batch whose BF16 inputs are in xb and FP32 targets in t;
// gradients into h->g, mean squared error into *loss (host)
int grad_batch(cmf_mlp* h, int rows, float* loss) {
    forward(h, rows);
    const int ny = rows * h->n_out;
    const unsigned nb = nblk(ny);
    hipLaunchKernelGGL(k_mse, dim3(nb), dim3(256), 0, h->stream, h->y, h->t, ny, h->w_over, h->gy, h->part);
    // output layer: dW4 = H3^T GY, db4 = colsum GY, D = GY W4^T
    const uint16_t* G = h->gy;
    int gcols = h->n_out;
    for (int l = 3; l >= 0; --l) {
        const uint16_t* Hin = l == 0 ? h->xb : h->hb[l - 1];
        gemm(h, h->din[l], h->dout[l], rows, Hin, h->din[l], 1, G, gcols, 0, h->g + h->off_w[l], h->dout[l], 0);
        const int nchunk = (rows + COLSUM_CHUNK - 1) / COLSUM_CHUNK;
        hipLaunchKernelGGL(k_colsum_part, dim3(nblk(gcols, 64), nchunk), dim3(64), 0, h->stream, G, rows, gcols,
                           h->colpart);
        hipLaunchKernelGGL(k_colsum_final, dim3(nblk(gcols, 64)), dim3(64), 0, h->stream, h->colpart, nchunk, gcols,
                           h->g + h->off_b[l]);
        if (l == 0) break;
        gemm(h, rows, h->din[l], h->dout[l], G, gcols, 0, h->wbf + h->off_w[l], h->dout[l], 1, h->z, h->din[l], 0);
        uint16_t* Gn = h->gh[l & 1];
        hipLaunchKernelGGL(k_relu_grad, dim3(nblk((long long)rows * h->din[l])), dim3(256), 0, h->stream, h->z,
                           h->hb[l - 1], (long long)rows * h->din[l], Gn);
        G = Gn;
        gcols = h->din[l];
    }
    if (loss) {
        std::vector<float> part(nb);
        MCHK(hipMemcpyAsync(part.data(), h->part, nb * sizeof(float), hipMemcpyDeviceToHost, h->stream));
        MCHK(hipStreamSynchronize(h->stream));
        double s = 0.0;
        for (unsigned b = 0; b < nb; ++b) s += part[b];
        *loss = (float)(s / ny);
    }
    MCHK(hipGetLastError());
    return 0;
}

}  // namespace

extern "C" {

const char* cmf_mlp_last_error(void) { return m_err.c_str(); }

int cmf_mlp_create(int32_t n_in, int32_t hidden, int32_t n_out, int32_t max_batch, cmf_mlp_handle* out) {
    if (!out) return mfail(CMF_MLP_EINVAL, "NULL argument");
    *out = nullptr;
    if (n_in <= 0 || hidden <= 0 || n_out <= 0 || max_batch <= 0)
        return mfail(CMF_MLP_EINVAL, "sizes must be positive");
    cmf_mlp* h = new cmf_mlp();
    h->n_in = n_in; h->hid = hidden; h->n_out = n_out; h->max_batch = max_batch;
    const int din[4] = {n_in, hidden, hidden, hidden}, dout[4] = {hidden, hidden, hidden, n_out};
    long long o = 0;
    for (int l = 0; l < 4; ++l) {
        h->din[l] = din[l]; h->dout[l] = dout[l];
        h->off_w[l] = o; o += (long long)din[l] * dout[l];
        h->off_b[l] = o; o += dout[l];
    }
    h->np = o;
    int rc = 0;
    if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess) {
        delete h;
        return mfail(CMF_MLP_EHIP, "hipStreamCreate failed");
    }
    const size_t B = (size_t)max_batch, H = (size_t)hidden, wide = (size_t)(hidden > n_out ? hidden : n_out);
    h->fused = hidden == FH && n_in <= FKI && n_out <= FNO;
    rc = malloc_t(h, &h->p, h->np);
    if (!rc) rc = malloc_t(h, &h->g, h->np);
    if (!rc) rc = malloc_t(h, &h->m1, h->np);
    if (!rc) rc = malloc_t(h, &h->m2, h->np);
    if (!rc) rc = malloc_t(h, &h->wbf, h->np);
    if (!rc) rc = malloc_t(h, &h->y, B * n_out);
    if (!rc) rc = malloc_t(h, &h->t, B * n_out);
    if (!rc) rc = malloc_t(h, &h->part, (B * n_out + 255) / 256);
    if (!rc) rc = malloc_t(h, &h->xd, B * n_in);
    if (!rc && !h->fused) {                                         // batch buffers of the layer kernels
        if ((rc = malloc_t(h, &h->xb, B * n_in)) || (rc = malloc_t(h, &h->hb[0], B * H)) ||
            (rc = malloc_t(h, &h->hb[1], B * H)) || (rc = malloc_t(h, &h->hb[2], B * H)) ||
            (rc = malloc_t(h, &h->z, B * wide)) || (rc = malloc_t(h, &h->gy, B * n_out)) ||
            (rc = malloc_t(h, &h->gh[0], B * H)) || (rc = malloc_t(h, &h->gh[1], B * H)) ||
            (rc = malloc_t(h, &h->idx, B)) ||
            (rc = malloc_t(h, &h->colpart, ((B + COLSUM_CHUNK - 1) / COLSUM_CHUNK) * wide))) {}
    }
    if (!rc && h->fused) {                                          // weight layouts of the fused kernels
        int o[8];
        for (int l = 0; l < 4; ++l) { o[2 * l] = (int)h->off_w[l]; o[2 * l + 1] = (int)h->off_b[l]; }
        rc = malloc_t(h, &h->wt, (size_t)FH * FKI + 2 * FH * FH + FNO * FH);
        if (!rc) rc = malloc_t(h, &h->w3, (size_t)FH * FKI);
        if (!rc) rc = malloc_t(h, &h->off, 8);
        if (!rc && hipMemcpy(h->off, o, sizeof o, hipMemcpyHostToDevice) != hipSuccess)
            rc = mfail(CMF_MLP_EHIP, "hipMemcpy failed");
        if (!rc) rc = alloc_fused(h);
    }
    if (rc) {
        std::string keep = m_err;
        cmf_mlp_destroy(h);
        m_err = keep;
        return rc;
    }
    if (hipHostMalloc((void**)&h->h_scratch, 1024 * sizeof(float), hipHostMallocDefault) != hipSuccess) {
        cmf_mlp_destroy(h);
        return mfail(CMF_MLP_EHIP, "hipHostMalloc failed");
    }
    *out = h;
    return 0;
}

void cmf_mlp_destroy(cmf_mlp_handle h) {
    if (!h) return;
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    for (void* q : h->allocs) if (q) (void)hipFree(q);
    if (h->h_scratch) (void)hipHostFree(h->h_scratch);
    h->fwd_pin.release();
    for (hipStream_t st : h->fwd_stream)
        if (st) (void)hipStreamDestroy(st);
    if (h->stream) (void)hipStreamDestroy(h->stream);
    delete h;
}

int64_t cmf_mlp_param_count(cmf_mlp_handle h) { return h ? h->np : -1; }

int cmf_mlp_set_loss(cmf_mlp_handle h, float w_over) {
    if (!h || !(w_over > 0.f)) return mfail(CMF_MLP_EINVAL, "loss weight must be positive");
    h->w_over = w_over;
    return 0;
}

int cmf_mlp_set_params(cmf_mlp_handle h, const float* params) {
    if (!h || !params) return mfail(CMF_MLP_EINVAL, "NULL argument");
    MCHK(hipMemcpyAsync(h->p, params, h->np * sizeof(float), hipMemcpyHostToDevice, h->stream));
    MCHK(hipMemsetAsync(h->m1, 0, h->np * sizeof(float), h->stream));
    MCHK(hipMemsetAsync(h->m2, 0, h->np * sizeof(float), h->stream));
    refresh_bf16(h);
    MCHK(hipGetLastError());
    MCHK(hipStreamSynchronize(h->stream));
    return 0;
}

int cmf_mlp_get_params(cmf_mlp_handle h, float* params, float* grads) {
    if (!h) return mfail(CMF_MLP_EINVAL, "NULL handle");
    if (params) MCHK(hipMemcpyAsync(params, h->p, h->np * sizeof(float), hipMemcpyDeviceToHost, h->stream));
    if (grads) MCHK(hipMemcpyAsync(grads, h->g, h->np * sizeof(float), hipMemcpyDeviceToHost, h->stream));
    MCHK(hipStreamSynchronize(h->stream));
    return 0;
}

int cmf_mlp_forward(cmf_mlp_handle h, const float* x, int64_t n, float* y) {
    if (!h || !x || !y || n < 0) return mfail(CMF_MLP_EINVAL, "bad argument");
    if (h->fused) return n > 0 ? forward_fused(h, x, n, y) : 0;
    for (int64_t r0 = 0; r0 < n; r0 += h->max_batch) {
        const int rows = (int)((n - r0) < h->max_batch ? (n - r0) : h->max_batch);
        MCHK(hipMemcpyAsync(h->xd, x + (size_t)r0 * h->n_in, (size_t)rows * h->n_in * sizeof(float),
                            hipMemcpyHostToDevice, h->stream));
        hipLaunchKernelGGL(k_to_bf16, dim3(nblk((long long)rows * h->n_in)), dim3(256), 0, h->stream, h->xd, h->xb,
                           (long long)rows * h->n_in);
        forward(h, rows);
        MCHK(hipGetLastError());
        MCHK(hipMemcpyAsync(y + (size_t)r0 * h->n_out, h->y, (size_t)rows * h->n_out * sizeof(float),
                            hipMemcpyDeviceToHost, h->stream));
        MCHK(hipStreamSynchronize(h->stream));
    }
    return 0;
}

int cmf_mlp_grad(cmf_mlp_handle h, const float* x, const float* t, int32_t rows, float* loss) {
    if (!h || !x || !t || rows <= 0 || rows > h->max_batch) return mfail(CMF_MLP_EINVAL, "bad argument");
    MCHK(hipMemcpyAsync(h->xd, x, (size_t)rows * h->n_in * sizeof(float), hipMemcpyHostToDevice, h->stream));
    MCHK(hipMemcpyAsync(h->t, t, (size_t)rows * h->n_out * sizeof(float), hipMemcpyHostToDevice, h->stream));
    int rc = 0;
    if (h->fused) {
        MTRY(fused_grad(h, h->xd, h->t, nullptr, rows, h->part));
        if (loss) {
            const int nb = loss_parts(h, rows);
            std::vector<float> part((size_t)nb);
            MCHK(hipMemcpyAsync(part.data(), h->part, (size_t)nb * sizeof(float), hipMemcpyDeviceToHost, h->stream));
            MCHK(hipStreamSynchronize(h->stream));
            *loss = (float)(loss_of(part.data(), nb) / (rows * h->n_out));
        }
    } else {
        hipLaunchKernelGGL(k_to_bf16, dim3(nblk((long long)rows * h->n_in)), dim3(256), 0, h->stream, h->xd, h->xb,
                           (long long)rows * h->n_in);
        rc = grad_batch(h, rows, loss);
    }
    MCHK(hipStreamSynchronize(h->stream));
    return rc;
}

int cmf_mlp_set_data(cmf_mlp_handle h, const float* x, const float* t, int64_t n) {
    if (!h || !x || !t || n <= 0) return mfail(CMF_MLP_EINVAL, "bad argument");
    for (void*& q : h->allocs)
        if (q == (void*)h->tx || q == (void*)h->tt) { (void)hipFree(q); q = nullptr; }
    std::vector<void*> keep;
    for (void* q : h->allocs) if (q) keep.push_back(q);
    h->allocs = keep;
    h->tx = h->tt = nullptr;
    h->tn = 0;                                            // no data until both are there
    MTRY(malloc_t(h, &h->tx, (size_t)n * h->n_in));
    MTRY(malloc_t(h, &h->tt, (size_t)n * h->n_out));
    MCHK(hipMemcpyAsync(h->tx, x, (size_t)n * h->n_in * sizeof(float), hipMemcpyHostToDevice, h->stream));
    MCHK(hipMemcpyAsync(h->tt, t, (size_t)n * h->n_out * sizeof(float), hipMemcpyHostToDevice, h->stream));
    MCHK(hipStreamSynchronize(h->stream));
    h->tn = n;
    return 0;
}

int cmf_mlp_train(cmf_mlp_handle h, const int64_t* order, int64_t n_order, int32_t batch, float lr, float beta1,
                  float beta2, float eps, int32_t step0, float* loss_out) {
    if (!h || !order || n_order <= 0 || batch <= 0 || batch > h->max_batch)
        return mfail(CMF_MLP_EINVAL, "bad argument");
    if (h->tn == 0) return mfail(CMF_MLP_ESTATE, "cmf_mlp_set_data must come first");
    for (int64_t k = 0; k < n_order; ++k)
        if (order[k] < 0 || order[k] >= h->tn) return mfail(CMF_MLP_EINVAL, "order[%lld] outside the data", (long long)k);
    double lsum = 0.0;
    int32_t step = step0;
    int64_t nb = 0;
    if (h->fused) {
        // the whole order and the loss of every batch stay on the device, so the batches
        // follow each other without a word to the host: three launches each
        const int np = loss_parts(h, batch);
        const size_t nbatch = (size_t)(n_order / batch), need = nbatch * (size_t)np;
        MTRY(grow(h, &h->order, &h->order_cap, (size_t)n_order));
        MTRY(grow(h, &h->lossbuf, &h->loss_cap, need));
        MCHK(hipMemcpyAsync(h->order, order, (size_t)n_order * sizeof(int64_t), hipMemcpyHostToDevice, h->stream));
        for (int64_t r0 = 0; r0 + batch <= n_order; r0 += batch) {
            MTRY(fused_grad(h, h->tx, h->tt, h->order + r0, batch, h->lossbuf + (size_t)nb * np));
            ++step;
            const float c1 = 1.f - powf(beta1, (float)step), c2 = 1.f - powf(beta2, (float)step);
            hipLaunchKernelGGL(k_adam_fused, dim3(nblk(h->np)), dim3(256), 0, h->stream, h->p, h->g, h->m1, h->m2, h->np, lr,
                               beta1, beta2, eps, c1, c2, h->off, h->n_in, h->n_out, h->wbf, h->wt, h->w3);
            ++nb;
        }
        MCHK(hipGetLastError());
        std::vector<float> part(need);
        if (need) MCHK(hipMemcpyAsync(part.data(), h->lossbuf, need * sizeof(float), hipMemcpyDeviceToHost, h->stream));
        MCHK(hipStreamSynchronize(h->stream));
        for (size_t k = 0; k < nbatch; ++k) lsum += (float)(loss_of(&part[k * (size_t)np], np) / (batch * h->n_out));
        if (loss_out) *loss_out = nb ? (float)(lsum / nb) : 0.f;
        return (int)nb;
    }
    for (int64_t r0 = 0; r0 + batch <= n_order; r0 += batch) {
        MCHK(hipMemcpyAsync(h->idx, order + r0, (size_t)batch * sizeof(int64_t), hipMemcpyHostToDevice, h->stream));
        hipLaunchKernelGGL(k_gather_bf16, dim3(nblk((long long)batch * h->n_in)), dim3(256), 0, h->stream, h->tx,
                           h->idx, batch, h->n_in, h->xb);
        hipLaunchKernelGGL(k_gather_f32, dim3(nblk((long long)batch * h->n_out)), dim3(256), 0, h->stream, h->tt,
                           h->idx, batch, h->n_out, h->t);
        float l = 0.f;
        MTRY(grad_batch(h, batch, &l));
        ++step;
        const float c1 = 1.f - powf(beta1, (float)step), c2 = 1.f - powf(beta2, (float)step);
        hipLaunchKernelGGL(k_adam, dim3(nblk(h->np)), dim3(256), 0, h->stream, h->p, h->g, h->m1, h->m2, h->np, lr,
                           beta1, beta2, eps, c1, c2);
        refresh_bf16(h);
        lsum += l;
        ++nb;
    }
    MCHK(hipGetLastError());
    MCHK(hipStreamSynchronize(h->stream));
    if (loss_out) *loss_out = nb ? (float)(lsum / nb) : 0.f;
    return (int)nb;
}

int cmf_mlp_gemm_test(int32_t M, int32_t N, int32_t K, const uint16_t* A, int32_t lda, int32_t ta, const uint16_t* B,
                      int32_t ldb, int32_t tb, float* C) {
    if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0) return mfail(CMF_MLP_EINVAL, "bad argument");
    const size_t na = (size_t)(ta ? (size_t)K * lda : (size_t)M * lda);
    const size_t nbv = (size_t)(tb ? (size_t)N * ldb : (size_t)K * ldb);
    if ((ta ? lda < M : lda < K) || (tb ? ldb < K : ldb < N)) return mfail(CMF_MLP_EINVAL, "leading dimension too small");
    uint16_t *da = nullptr, *db = nullptr;
    float* dc = nullptr;
    MCHK(hipMalloc(&da, na * 2));
    MCHK(hipMalloc(&db, nbv * 2));
    MCHK(hipMalloc(&dc, (size_t)M * N * 4));
    MCHK(hipMemcpy(da, A, na * 2, hipMemcpyHostToDevice));
    MCHK(hipMemcpy(db, B, nbv * 2, hipMemcpyHostToDevice));
    dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM);
    hipLaunchKernelGGL(k_gemm_bf16, grid, dim3(256), 0, 0, M, N, K, da, lda, ta, db, ldb, tb, dc, N, 0);
    MCHK(hipGetLastError());
    MCHK(hipMemcpy(C, dc, (size_t)M * N * 4, hipMemcpyDeviceToHost));
    (void)hipFree(da); (void)hipFree(db); (void)hipFree(dc);
    return 0;
}

}  // extern "C"
