// lus_mlp.hip -- the per-particle warm-start network on gfx950 matrix cores.
//
// Network: 32 inputs -> 64 (SiLU) -> 64 (SiLU) -> 3.  BF16 weights and
// activations, FP32 accumulation (v_mfma_f32_16x16x32_bf16), FP32 bias and
// SiLU.  Parameter order (FP32 master copy): W1[32][64] b1[64] W2[64][64]
// b2[64] W3[64][3] b3[3]; W[k][n] maps input k to output n, so each (W, b)
// pair is one [fan_in + 1][fan_out] matrix whose last row is the bias.
//
// Operand layout of v_mfma_f32_16x16x32_bf16 (wave64, lane l):
//   A (16 x 32, rows m):   lane l holds A[l % 16][8 * (l / 16) + e], e = 0..7
//   B (32 x 16, cols n):   lane l holds B[8 * (l / 16) + e][l % 16], e = 0..7
//   C (16 x 16):           lane l holds C[4 * (l / 16) + i][l % 16], i = 0..3
// The GPU tests compare the forward pass and the gradients with a float64 CPU
// implementation that rounds to bf16 at the same points, which fixes these
// layouts.
#include <hip/hip_runtime.h>

#include "lus_device.hpp"
#include "lus_internal.hpp"
#include "lus_launch.hpp"

namespace lus {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }
__device__ __forceinline__ float silu_grad(float z) {
    const float s = 1.0f / (1.0f + __expf(-z));
    return s * (1.0f + z * (1.0f - s));
}

// ------------------------------------------------------------------ inference
// Inference runs each layer transposed, Y^T = W^T X^T: the weights are the A
// operand and the activations the B operand, so the C tile of a layer holds,
// in lane l, units 16j + 4(l/16) + i (i = 0..3) of sample l%16.  The next
// layer's reduction index is permuted to take those values as they lie:
// k-step s, lane group g = l/16, element e  <->  hidden unit
//   pi(s, g, e) = 16 (2s + e/4) + 4g + e%4,
// i.e. the B operand of k-step s is C tiles 2s and 2s+1 of the lane itself,
// and no activation leaves its lane.  A-operand images of the weights (one
// 16-byte load per lane and image):
//   [0, 4)    W1 m-tile j:            lane l: W1[8(l/16)+e][16j + l%16]
//   [4, 12)   W2 k-step s, m-tile j:  lane l: W2[pi(s, l/16, e)][16j + l%16]
//   [12, 14)  W3 k-step s (m < 3):    lane l: W3[pi(s, l/16, e)][l%16], 0 for l%16 >= 3
__device__ __forceinline__ int mlp_pi(int s, int g, int e) { return 16 * (2 * s + e / 4) + 4 * g + e % 4; }

__global__ void k_mlp_pack(const float* __restrict__ p, bf16x8* __restrict__ w) {
    const int t = threadIdx.x + blockIdx.x * blockDim.x;
    const int img = t / 64, l = t % 64;
    const int col = l % 16, grp = l / 16;
    if (img >= 14) return;
    bf16x8 v;
    if (img < 4) {
        for (int e = 0; e < 8; ++e) v[e] = (__bf16)p[kMlpW1 + (8 * grp + e) * 64 + 16 * img + col];
    } else if (img < 12) {
        const int s = (img - 4) / 4, j = (img - 4) % 4;
        for (int e = 0; e < 8; ++e) v[e] = (__bf16)p[kMlpW2 + mlp_pi(s, grp, e) * 64 + 16 * j + col];
    } else {
        const int s = img - 12;
        for (int e = 0; e < 8; ++e)
            v[e] = col < 3 ? (__bf16)p[kMlpW3 + mlp_pi(s, grp, e) * 3 + col] : (__bf16)0.0f;
    }
    w[t] = v;
}

hipError_t launch_mlp_pack(const float* params, void* packed, hipStream_t s) {
    launch_kernel(k_mlp_pack, dim3(4), dim3(256), 0, s, params, (bf16x8*)packed);
    return hipGetLastError();
}

// One wave per 16-sample tile (grid-stride over tiles).  X: bf16 [n][32]; a
// lane loads 8 features of one sample, which is the B operand of layer 1 as
// it lies.  The activations stay in registers (see the pack layout above) and
// the lanes of group 0 hold the three outputs of their sample at the end.  The
// next tile's features are requested before the current tile's layers run.
constexpr int kMlpWaves = 4;

// SiLU for inference with the hardware reciprocal (1 ulp): the activation is
// rounded to bf16 right after, far coarser than that error.
__device__ __forceinline__ float silu_fast(float z) {
    return z * __builtin_amdgcn_rcpf(1.0f + __expf(-z));
}

__global__ __launch_bounds__(64 * kMlpWaves) void k_mlp_forward(
    const bf16x8* __restrict__ X, int n, const float* __restrict__ params,
    const bf16x8* __restrict__ wpk, float out_scale, float* __restrict__ out,
    const float4* __restrict__ xp, float4* __restrict__ xa, PbfK k) {
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int col = lane % 16, grp = lane / 16;
    bf16x8 W1[4], W2[2][4], W3[2];
#pragma unroll
    for (int j = 0; j < 4; ++j) W1[j] = wpk[j * 64 + lane];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int j = 0; j < 4; ++j) W2[s][j] = wpk[(4 + s * 4 + j) * 64 + lane];
        W3[s] = wpk[(12 + s) * 64 + lane];
    }
    // biases of the units this lane's C values belong to: 16j + 4 grp + i
    f32x4 B1[4], B2[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            B1[j][i] = params[kMlpB1 + 16 * j + 4 * grp + i];
            B2[j][i] = params[kMlpB2 + 16 * j + 4 * grp + i];
        }
    float B3[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) B3[c] = params[kMlpB3 + c];
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const int ntiles = (n + 15) / 16;
    const int nwaves = gridDim.x * kMlpWaves;
    int tile = blockIdx.x * kMlpWaves + w;  // uniform per wave: the loop below never diverges
    bf16x8 a = {};
    if (tile < ntiles && tile * 16 + col < n) a = X[(size_t)(tile * 16 + col) * 4 + grp];
    for (; tile < ntiles; tile += nwaves) {
        const int nt = tile + nwaves;
        bf16x8 an = {};
        if (nt < ntiles && nt * 16 + col < n) an = X[(size_t)(nt * 16 + col) * 4 + grp];
        const int i = tile * 16 + col;
        const bool writer = grp == 0 && i < n;
        float4 p = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (xa && writer) p = xp[i];
        f32x4 z[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) z[j] = mfma(W1[j], a, zero);
        bf16x8 h[2];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                h[s][e] = (__bf16)silu_fast(z[2 * s + e / 4][e % 4] + B1[2 * s + e / 4][e % 4]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            z[j] = mfma(W2[0][j], h[0], zero);
            z[j] = mfma(W2[1][j], h[1], z[j]);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                h[s][e] = (__bf16)silu_fast(z[2 * s + e / 4][e % 4] + B2[2 * s + e / 4][e % 4]);
        f32x4 o = mfma(W3[0], h[0], zero);
        o = mfma(W3[1], h[1], o);
        if (writer) {
            const float dx = (o[0] + B3[0]) * out_scale;
            const float dy = (o[1] + B3[1]) * out_scale;
            const float dz = (o[2] + B3[2]) * out_scale;
            if (out) {
                out[(size_t)i * 3 + 0] = dx;
                out[(size_t)i * 3 + 1] = dy;
                out[(size_t)i * 3 + 2] = dz;
            }
            if (xa) {
                const float* lo = k.lo;
                const float* hi = k.hi;
                if (k.scenes) {
                    const SceneBox& sb = k.scenes[k.sid_out[i]];
                    lo = sb.lo;
                    hi = sb.hi;
                }
                xa[i] = make_float4(rclamp(p.x + dx, lo[0], hi[0]), rclamp(p.y + dy, lo[1], hi[1]),
                                    rclamp(p.z + dz, lo[2], hi[2]), 0.0f);
            }
        }
        a = an;
    }
}

hipError_t launch_mlp_forward(const void* X, int n, const float* params, const void* packed,
                              float out_scale, float* out, const float4* xp, float4* xa,
                              const PbfK& k, hipStream_t s) {
    const int ntiles = (n + 15) / 16;
    int blocks = (ntiles + kMlpWaves - 1) / kMlpWaves;
    if (blocks > 256 * 16) blocks = 256 * 16;
    if (blocks < 1) blocks = 1;
    launch_kernel(k_mlp_forward, dim3(blocks), dim3(64 * kMlpWaves), 0, s, (const bf16x8*)X, n,
                       params, (const bf16x8*)packed, out_scale, out, xp, xa, k);
    return hipGetLastError();
}

// ------------------------------------------------------------------ training
// A training step is two launches: k_mlp_train_rows takes a batch's rows
// forward and backward to the activations' gradients, k_mlp_train_weights
// contracts them over the rows to the weights' gradients and applies Adam.
// One launch per product and per elementwise pass (24 of 2 to 6 us each) took
// 97 us per step of 4,096 rows, all of it launches and their tails (a fit of
// 131,072 rows over 4 epochs: 11.7 -> 3.2 ms, the same bits).
//
// The weights are kept in bf16 twice, as stored ([fan_in][fan_out], w) and
// transposed ([fan_out][fan_in], wt), each layer at its fp32 offset, so that
// either product reads a lane's eight reduction elements as one 16-byte load.
// The activations the weight gradients need go out transposed ([unit][row],
// row stride ld) for the same reason.

// w and wt from the fp32 parameters
__global__ void k_mlp_train_pack(const float* __restrict__ p, __bf16* __restrict__ w, __bf16* __restrict__ wt) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= kMlpParams) return;
    const __bf16 v = (__bf16)p[t];
    w[t] = v;
    if (t < kMlpB1) {
        wt[(t % kMlpHid) * kMlpIn + t / kMlpHid] = v;
    } else if (t >= kMlpW2 && t < kMlpB2) {
        const int q = t - kMlpW2;
        wt[kMlpW2 + (q % kMlpHid) * kMlpHid + q / kMlpHid] = v;
    } else if (t >= kMlpW3 && t < kMlpB3) {
        const int q = t - kMlpW3;
        wt[kMlpW3 + (q % kMlpOut) * kMlpHid + q / kMlpOut] = v;
    }
}

hipError_t launch_mlp_train_pack(const float* params, void* w, void* wt, hipStream_t s) {
    launch_kernel(k_mlp_train_pack, dim3((kMlpParams + 255) / 256), dim3(256), 0, s, params, (__bf16*)w, (__bf16*)wt);
    return hipGetLastError();
}

// Sixteen rows per block, wave j computing units 16j..16j+15 of a layer (its
// z values stay in registers for the backward pass; the layers meet in LDS).
// Row r is row sel[r] (sel null: r) of feat and tgt; inputs are
// bf16((x - mu) inv_sigma), or bf16(x) without mu.
//   err[r] = sum_c (o_rc - y_rc inv_scale)^2, the loss is their mean
// kGrad: also the transposed activations and gradients t (rows past `rows` as
// zeros, up to the grid's end).  The latency of the chain from the row index to
// the last layer's gradient bounds it (one block per CU at 4,096 rows): every
// weight, bias and target is requested at the start, beside the inputs.
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

template <bool kGrad>
__global__ __launch_bounds__(256) void k_mlp_train_rows(const float* __restrict__ feat, const float* __restrict__ tgt,
                                                        const int* __restrict__ sel, int rows,
                                                        const float* __restrict__ mu,
                                                        const float* __restrict__ inv_sigma, float inv_scale,
                                                        const float* __restrict__ p, const __bf16* __restrict__ w,
                                                        const __bf16* __restrict__ wt, float* __restrict__ err,
                                                        MlpTrainAct t, long ld) {
    constexpr int kStride = kMlpHid + 8;  // LDS row stride (16-byte aligned rows, spread over the banks)
    __shared__ __attribute__((aligned(16))) __bf16 H1[16][kStride], H2[16][kStride], D[16][kStride];
    __shared__ __bf16 d3[16][4];
    __shared__ float sq[16][4];
    // the wave's number is made uniform for the compiler: matrix instructions
    // ignore the lane mask, so the conditions around them have to be branches
    const int lane = threadIdx.x & 63, j = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int col = lane % 16, grp = lane / 16;
    const int m0 = blockIdx.x * 16;
    const int n = 16 * j + col;       // this lane's unit (C columns, B columns)
    const int c0 = m0 + 4 * grp;      // and first row (C rows)
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    bool in[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) in[i] = c0 + i < rows;
    const bf16x8 W1 = *reinterpret_cast<const bf16x8*>(wt + kMlpW1 + n * kMlpIn + 8 * grp);
    const float bias1 = p[kMlpB1 + n], bias2 = p[kMlpB2 + n];
    bf16x8 W2[2], W3[2] = {}, V2[2] = {}, V3 = {};
    float bias3 = 0.0f, y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        W2[k] = *reinterpret_cast<const bf16x8*>(wt + kMlpW2 + n * kMlpHid + 32 * k + 8 * grp);
        if (kGrad) V2[k] = *reinterpret_cast<const bf16x8*>(w + kMlpW2 + n * kMlpHid + 32 * k + 8 * grp);
    }
    if (j == 0 && col < kMlpOut) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
            W3[k] = *reinterpret_cast<const bf16x8*>(wt + kMlpW3 + col * kMlpHid + 32 * k + 8 * grp);
        bias3 = p[kMlpB3 + col];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (in[i]) y[i] = tgt[(size_t)(sel ? sel[c0 + i] : c0 + i) * kMlpOut + col];
    }
    if (kGrad && grp == 0) {
#pragma unroll
        for (int c = 0; c < kMlpOut; ++c) V3[c] = w[kMlpW3 + n * kMlpOut + c];
    }
    // layer 1
    bf16x8 a = {};
    {
        const int r = m0 + col;
        if (r < rows) {
            const float4* x = reinterpret_cast<const float4*>(feat + (size_t)(sel ? sel[r] : r) * kMlpIn + 8 * grp);
            const float4 q0 = x[0], q1 = x[1];
            const float v[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
            for (int e = 0; e < 8; ++e)
                a[e] = mu ? (__bf16)((v[e] - mu[8 * grp + e]) * inv_sigma[8 * grp + e]) : (__bf16)v[e];
        }
        if (kGrad && j == 0) {
            __bf16* xt = (__bf16*)t.x;
#pragma unroll
            for (int e = 0; e < 8; ++e) xt[(8 * grp + e) * ld + r] = a[e];
        }
    }
    const f32x4 y1 = mfma(a, W1, zero);
    float z1[4], z2[4];
    bf16x4 h;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        z1[i] = y1[i] + bias1;
        h[i] = in[i] ? (__bf16)silu(z1[i]) : (__bf16)0.0f;
        H1[4 * grp + i][n] = h[i];
    }
    if (kGrad) *reinterpret_cast<bf16x4*>((__bf16*)t.h1 + n * ld + c0) = h;
    __syncthreads();
    // layer 2
    f32x4 y2 = zero;
#pragma unroll
    for (int k = 0; k < 2; ++k) y2 = mfma(*reinterpret_cast<const bf16x8*>(&H1[col][32 * k + 8 * grp]), W2[k], y2);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        z2[i] = y2[i] + bias2;
        h[i] = in[i] ? (__bf16)silu(z2[i]) : (__bf16)0.0f;
        H2[4 * grp + i][n] = h[i];
    }
    if (kGrad) *reinterpret_cast<bf16x4*>((__bf16*)t.h2 + n * ld + c0) = h;
    __syncthreads();
    // output and loss (wave 0)
    if (j == 0) {
        f32x4 o = zero;
#pragma unroll
        for (int k = 0; k < 2; ++k) o = mfma(*reinterpret_cast<const bf16x8*>(&H2[col][32 * k + 8 * grp]), W3[k], o);
        if (col < kMlpOut) {
            bf16x4 d;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float diff = in[i] ? (o[i] + bias3) - y[i] * inv_scale : 0.0f;
                d[i] = (__bf16)(2.0f * diff / (float)rows);
                d3[4 * grp + i][col] = d[i];
                sq[4 * grp + i][col] = diff * diff;
            }
            if (kGrad) *reinterpret_cast<bf16x4*>((__bf16*)t.d3 + col * ld + c0) = d;
        }
    }
    __syncthreads();
    if (threadIdx.x < 16 && m0 + (int)threadIdx.x < rows) {
        float e = 0.0f;
#pragma unroll
        for (int c = 0; c < kMlpOut; ++c) e += sq[threadIdx.x][c];
        err[m0 + threadIdx.x] = e;
    }
    if (!kGrad) return;
    // back through layer 3: dH2 = d3 W3^T
    bf16x8 d = {};
    if (grp == 0) {
#pragma unroll
        for (int c = 0; c < kMlpOut; ++c) d[c] = d3[col][c];
    }
    const f32x4 g2 = mfma(d, V3, zero);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        h[i] = in[i] ? (__bf16)(g2[i] * silu_grad(z2[i])) : (__bf16)0.0f;
        D[4 * grp + i][n] = h[i];
    }
    *reinterpret_cast<bf16x4*>((__bf16*)t.dz2 + n * ld + c0) = h;
    __syncthreads();
    // layer 2: dH1 = dZ2 W2^T
    f32x4 g1 = zero;
#pragma unroll
    for (int k = 0; k < 2; ++k) g1 = mfma(*reinterpret_cast<const bf16x8*>(&D[col][32 * k + 8 * grp]), V2[k], g1);
#pragma unroll
    for (int i = 0; i < 4; ++i) h[i] = in[i] ? (__bf16)(g1[i] * silu_grad(z1[i])) : (__bf16)0.0f;
    *reinterpret_cast<bf16x4*>((__bf16*)t.dz1 + n * ld + c0) = h;
}

hipError_t launch_mlp_train_rows(const float* feat, const float* tgt, const int* sel, int rows, const float* mu,
                                 const float* inv_sigma, float inv_scale, const float* params, const void* w,
                                 const void* wt, float* err, const MlpTrainAct* act, long ld, hipStream_t s) {
    if (act) {
        // rows up to the next multiple of 32 (a matrix step of the weight gradients) written, as zeros
        const int tiles = 2 * ((rows + 31) / 32);
        if ((long)tiles * 16 > ld || ld % 32) return hipErrorInvalidValue;
        launch_kernel((k_mlp_train_rows<true>), dim3(tiles), dim3(256), 0, s, feat, tgt, sel, rows, mu, inv_sigma,
                      inv_scale, params, (const __bf16*)w, (const __bf16*)wt, err, *act, ld);
    } else {
        launch_kernel((k_mlp_train_rows<false>), dim3((rows + 15) / 16), dim3(256), 0, s, feat, tgt, sel, rows, mu,
                      inv_sigma, inv_scale, params, (const __bf16*)w, (const __bf16*)wt, err, MlpTrainAct(), ld);
    }
    return hipGetLastError();
}

// Adam (Kingma & Ba, ICLR 2015) on the fp32 master parameters (p0, m0, v0:
// parameter t's state); returns the updated parameter
__device__ __forceinline__ float adam_step(const MlpAdam& a, int t, float g, float p0, float m0, float v0) {
    const float mt = a.b1 * m0 + (1.0f - a.b1) * g;
    const float vt = a.b2 * v0 + (1.0f - a.b2) * g * g;
    a.m[t] = mt;
    a.v[t] = vt;
    const float p = p0 - a.lr * (mt * a.c1) / (sqrtf(vt * a.c2) + a.eps);
    a.p[t] = p;
    return p;
}

__global__ void k_adam(MlpAdam a, const float* __restrict__ g) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < kMlpParams) adam_step(a, t, g[t], a.p[t], a.m[t], a.v[t]);
}

// *acc += the sum of v[0..n): 256 strided sums, then a tree (every thread of
// the block calls it)
__device__ __forceinline__ void block_sum_into(const float* __restrict__ v, int n, float* __restrict__ acc,
                                               float* part) {
    const int t = (int)threadIdx.x;
    if (t < 256) {
        float s = 0.0f;
#pragma unroll 8
        for (int i = t; i < n; i += 256) s += v[i];
        part[t] = s;
    }
    __syncthreads();
    for (int d = 128; d >= 1; d >>= 1) {
        if (t < d) part[t] += part[t + d];
        __syncthreads();
    }
    if (t == 0) acc[0] += part[0];
}

// *acc += sum of v[0..n), one block
__global__ __launch_bounds__(256) void k_sum_into(const float* __restrict__ v, int n, float* __restrict__ acc) {
    __shared__ float part[256];
    block_sum_into(v, n, acc, part);
}

hipError_t launch_sum_into(const float* v, int n, float* acc, hipStream_t s) {
    launch_kernel(k_sum_into, dim3(1), dim3(256), 0, s, v, n, acc);
    return hipGetLastError();
}

// out[t] = sum over chunks c (in order) of part[c * MN + t]
__global__ void k_sum_partials(const float* __restrict__ part, int chunks, int MN, float* __restrict__ out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= MN) return;
    float s = 0.0f;
    for (int c = 0; c < chunks; ++c) s += part[(size_t)c * MN + t];
    out[t] = s;
}

hipError_t launch_sum_partials(const float* part, int chunks, int MN, float* out, hipStream_t s) {
    launch_kernel(k_sum_partials, dim3((MN + 255) / 256), dim3(256), 0, s, part, chunks, MN, out);
    return hipGetLastError();
}

// Weight gradients: per layer [A^T; 1] dZ over the rows, the row of ones giving
// the bias gradient under the weight gradient.  One block per 16 x 16 tile of a layer's
// [fan_in + 1][fan_out] gradient; its waves take the row chunks of kMlpChunk
// in turn (sixteen at a time) and the chunks' sums are added in chunk order, so the
// result does not depend on scheduling.
//   adam      the tile's parameters are updated from their gradient (and w, wt)
//   otherwise the gradient goes to grad
//   part      (blockIdx.y > 0 too) every chunk's sum goes to part for
//             k_sum_partials: many chunks keep more than these blocks busy
// The block after the last tile adds the rows' err to *loss_acc.
constexpr int kTrainTiles1 = 3 * 4, kTrainTiles2 = 5 * 4, kTrainTiles3 = 5;
constexpr int kTrainTiles = kTrainTiles1 + kTrainTiles2 + kTrainTiles3;
constexpr int kTrainWaves = 16;

__global__ __launch_bounds__(64 * kTrainWaves) void k_mlp_train_weights(MlpTrainAct act, long ld, int rows, MlpAdam ad,
                                                                        float* __restrict__ grad,
                                                                        float* __restrict__ part,
                                                                        const float* __restrict__ err,
                                                                        float* __restrict__ loss_acc) {
    __shared__ float sum[kTrainWaves][256];
    int tile = blockIdx.x;
    if (tile == kTrainTiles) {
        block_sum_into(err, rows, loss_acc, sum[0]);
        return;
    }
    const __bf16 *A, *B;
    int M, N, off;
    if (tile < kTrainTiles1) {
        A = (const __bf16*)act.x, B = (const __bf16*)act.dz1, M = kMlpIn + 1, N = kMlpHid, off = kMlpW1;
    } else if (tile < kTrainTiles1 + kTrainTiles2) {
        tile -= kTrainTiles1;
        A = (const __bf16*)act.h1, B = (const __bf16*)act.dz2, M = kMlpHid + 1, N = kMlpHid, off = kMlpW2;
    } else {
        tile -= kTrainTiles1 + kTrainTiles2;
        A = (const __bf16*)act.h2, B = (const __bf16*)act.d3, M = kMlpHid + 1, N = kMlpOut, off = kMlpW3;
    }
    const int tiles_n = (N + 15) / 16;
    const int m0 = (tile / tiles_n) * 16, n0 = (tile % tiles_n) * 16;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int col = lane % 16, grp = lane / 16;
    const int m = m0 + col, nn = n0 + col;
    const int chunks = (rows + kMlpChunk - 1) / kMlpChunk;
    const int t = (int)threadIdx.x;
    const int mr = m0 + t / 16, nc = n0 + t % 16;  // thread t < 256: its element of the tile
    const bool mine = t < 256 && mr < M && nc < N;
    const int e = off + mr * N + nc;
    // the parameter's state, requested beside the activations
    float p0 = 0.0f, m0s = 0.0f, v0 = 0.0f;
    if (mine && ad.p) {
        p0 = ad.p[e];
        m0s = ad.m[e];
        v0 = ad.v[e];
    }
    float total = 0.0f;
    const int g1 = (chunks + kTrainWaves - 1) / kTrainWaves;
    for (int g = blockIdx.y; g < g1; g += gridDim.y) {
        const int c = g * kTrainWaves + wv;
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        if (c < chunks) {
            const int ke = rows < (c + 1) * kMlpChunk ? rows : (c + 1) * kMlpChunk;
            // a chunk's operands are all requested before the first product
            // (a step past `ke` repeats the first one's addresses, unused)
            constexpr int kSteps = kMlpChunk / 32;
            bf16x8 a[kSteps], b[kSteps];
            const long k0 = (long)c * kMlpChunk + 8 * grp;
#pragma unroll
            for (int q = 0; q < kSteps; ++q) {
                const long k = (long)c * kMlpChunk + 32 * q < ke ? k0 + 32 * q : k0;
                const bf16x8 fill = {};
                a[q] = fill;
                b[q] = fill;
                if (m < M - 1) a[q] = *reinterpret_cast<const bf16x8*>(A + m * ld + k);
                if (nn < N) b[q] = *reinterpret_cast<const bf16x8*>(B + nn * ld + k);
            }
            if (m == M - 1) {
#pragma unroll
                for (int q = 0; q < kSteps; ++q)
#pragma unroll
                    for (int u = 0; u < 8; ++u) a[q][u] = (__bf16)1.0f;
            }
#pragma unroll
            for (int q = 0; q < kSteps; ++q)
                if ((long)c * kMlpChunk + 32 * q < ke) acc = mfma(a[q], b[q], acc);
            if (part) {
                // partials of layer 1, then 2, then 3, each [chunk][M][N]
                const size_t base = (size_t)chunks * (off == kMlpW1 ? 0 : (off == kMlpW2 ? kMlpW2 : kMlpW3));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = m0 + 4 * grp + i;
                    if (r < M && nn < N) part[base + ((size_t)c * M + r) * N + nn] = acc[i];
                }
            }
        }
        if (part) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[wv][(4 * grp + i) * 16 + col] = acc[i];
        __syncthreads();
        if (mine) {
            const int left = chunks - g * kTrainWaves;
            for (int q = 0; q < kTrainWaves && q < left; ++q) total += sum[q][t];
        }
        __syncthreads();
    }
    if (part || !mine) return;
    if (grad) grad[e] = total;
    if (ad.p) {
        const float v = adam_step(ad, e, total, p0, m0s, v0);
        const __bf16 h = (__bf16)v;
        ((__bf16*)ad.w)[e] = h;
        if (mr < M - 1) ((__bf16*)ad.wt)[off + nc * (M - 1) + mr] = h;
    }
}

hipError_t launch_mlp_train_weights(const MlpTrainAct& act, long ld, int rows, const MlpAdam& adam, float* grad,
                                    float* part, const float* err, float* loss_acc, hipStream_t s) {
    const int chunks = (rows + kMlpChunk - 1) / kMlpChunk;
    if (rows < 1 || ld < (long)((rows + 31) / 32) * 32) return hipErrorInvalidValue;
    // up to kMlpFuseChunks chunks a block sums its tile alone
    const int gy = chunks <= kMlpFuseChunks ? 1 : (chunks + kTrainWaves - 1) / kTrainWaves;
    if (gy == 1) {
        launch_kernel(k_mlp_train_weights, dim3(kTrainTiles + 1), dim3(64 * kTrainWaves), 0, s, act, ld, rows, adam,
                      grad, (float*)nullptr, err, loss_acc);
        return hipGetLastError();
    }
    if (!part || !grad) return hipErrorInvalidValue;
    launch_kernel(k_mlp_train_weights, dim3(kTrainTiles, gy), dim3(64 * kTrainWaves), 0, s, act, ld, rows, MlpAdam(),
                  (float*)nullptr, part, err, loss_acc);
    const int off[4] = {kMlpW1, kMlpW2, kMlpW3, kMlpParams};
    for (int l = 0; l < 3; ++l)
        if (hipError_t e = launch_sum_partials(part + (size_t)chunks * off[l], chunks, off[l + 1] - off[l], grad + off[l], s))
            return e;
    if (hipError_t e = launch_sum_into(err, rows, loss_acc, s)) return e;
    if (!adam.p) return hipSuccess;
    launch_kernel(k_adam, dim3((kMlpParams + 255) / 256), dim3(256), 0, s, adam, (const float*)grad);
    if (hipError_t e = hipGetLastError()) return e;
    return launch_mlp_train_pack(adam.p, adam.w, adam.wt, s);
}

// xb[r][c] = bf16((x[src][c] - mu[c]) * inv_sigma[c]), src = rows ? rows[r] : r
__global__ void k_normalize_rows(const float* __restrict__ x, const int* __restrict__ rows, long nrows,
                                 const float* __restrict__ mu, const float* __restrict__ inv_sigma,
                                 __bf16* __restrict__ xb) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nrows * kFeat) return;
    const long r = t / kFeat;
    const int c = (int)(t % kFeat);
    const long src = rows ? rows[r] : r;
    xb[t] = (__bf16)((x[src * kFeat + c] - mu[c]) * inv_sigma[c]);
}

hipError_t launch_normalize_rows(const float* x, const int* rows, long nrows, const float* mu,
                                 const float* inv_sigma, void* xb, hipStream_t s) {
    const long tot = nrows * kFeat;
    launch_kernel(k_normalize_rows, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, x, rows, nrows,
                       mu, inv_sigma, (__bf16*)xb);
    return hipGetLastError();
}

// Column sums in float64: out[2c] = sum_r x[r][c], out[2c+1] = sum_r x[r][c]^2.
// Thread (q, c) sums the rows r with r % 256 = q in order (k_col_sums, whole rows
// per wave, so the loads are contiguous), then a block per column adds the 256
// sums by a tree: the order of one 256-thread block per column (155 us at
// 131,072 x 32, its loads 128 bytes apart), whose bits these are.
constexpr int kColSums = 256;

__global__ __launch_bounds__(256) void k_col_sums(const float* __restrict__ x, long rows, int w,
                                                  double* __restrict__ part) {
    const int t = blockIdx.x * 256 + (int)threadIdx.x;
    if (t >= kColSums * w) return;
    const int q = t / w;
    double a = 0.0, b = 0.0;
    const float* __restrict__ p = x + t;  // row q, column t % w
    long r = q;
    for (; r + 15 * kColSums < rows; r += 16 * kColSums, p += 16L * kColSums * w) {
        float f[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) f[u] = p[(long)u * kColSums * w];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const double v = f[u];
            a += v;
            b += v * v;
        }
    }
    for (; r < rows; r += kColSums, p += (long)kColSums * w) {
        const double v = *p;
        a += v;
        b += v * v;
    }
    part[2 * t] = a;
    part[2 * t + 1] = b;
}

__global__ __launch_bounds__(kColSums) void k_col_stats(const double* __restrict__ part, int w,
                                                        double* __restrict__ out) {
    __shared__ double s1[kColSums], s2[kColSums];
    const int c = blockIdx.x, t = (int)threadIdx.x;
    s1[t] = part[2 * (t * w + c)];
    s2[t] = part[2 * (t * w + c) + 1];
    __syncthreads();
    for (int d = kColSums / 2; d >= 1; d >>= 1) {
        if (t < d) {
            s1[t] += s1[t + d];
            s2[t] += s2[t + d];
        }
        __syncthreads();
    }
    if (t == 0) {
        out[2 * c] = s1[0];
        out[2 * c + 1] = s2[0];
    }
}

int col_stats_part(int w) { return 2 * kColSums * w; }

hipError_t launch_col_stats(const float* x, long rows, int w, double* part, double* out, hipStream_t s) {
    launch_kernel(k_col_sums, dim3((kColSums * w + 255) / 256), dim3(256), 0, s, x, rows, w, part);
    launch_kernel(k_col_stats, dim3(w), dim3(kColSums), 0, s, (const double*)part, w, out);
    return hipGetLastError();
}

}  // namespace lus
