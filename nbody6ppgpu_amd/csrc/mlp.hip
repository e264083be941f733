// mlp.hip -- the learned neighbour-radius predictor: a small MLP
// (8 -> 64 -> 64 -> 1, SiLU) that maps a particle's local state to log RS.
// Inference and training run on the GPU with these kernels; the plain
// Ahmad-Cohen radius update stays the fallback in the caller.
//
// Arithmetic: weights, activations and back-propagated deltas enter the
// products as BF16 (round to nearest even); products are accumulated in
// FP32 on the matrix cores (v_mfma_f32_16x16x16_bf16).  Bias additions, SiLU
// and the bias / output-layer gradients are FP32 vector work.  Training keeps
// FP32 master weights, FP32 gradients and an FP32 Adam state; the BF16
// weights are re-derived from the masters after every step.
//
// MFMA mapping.  A wavefront evaluates 16 samples.  Every layer is computed
// transposed, Z^T = W H^T: the weights are the A operand (16 output units x
// 16 inputs per instruction), the activations the B operand (16 inputs x 16
// samples).  The 16x16 FP32 result tile leaves lane l holding sample l%16 and
// units 4(l/16)..4(l/16)+3 of the tile, which is exactly the B-operand layout
// of the next layer's k-step, so activations never leave registers.  The
// backward delta d1^T = W2^T d2^T reuses the same layout with W2^T as A.
// Weight gradients (sums over samples) need the samples on the k dimension:
// the wave stages its deltas and activations through LDS and reads them back
// transposed.
//
// Kernels
//   k_mlp_forward   inference; 4 waves x 16 samples per workgroup, loop.
//   k_mlp_fwdbwd    forward + backward, a wavefront per 16 units, gradient
//                   sums accumulated in registers over a strided loop, one
//                   partial row per workgroup.
//   k_mlp_reduce    sums the partial rows in a fixed order (deterministic)
//                   and applies Adam (or only stores the sum).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#include <stdexcept>
#include <string>
#include <vector>

#include "gpunb.h"
#include "gpunb_internal.h"

namespace gpunb_mlp {

constexpr int NI = 8, NH = 64;
// Parameter layout (FP32 master, BF16 copy): W1[NH][NI] b1[NH] W2[NH][NH]
// b2[NH] W3[NH] b3.
constexpr int OW1 = 0, OB1 = OW1 + NH * NI, OW2 = OB1 + NH,
              OB2 = OW2 + NH * NH, OW3 = OB2 + NH, OB3 = OW3 + NH,
              NP = OB3 + 1;
// The BF16 copy also holds W2 transposed, WT[a][b] = W2[b][a], so that every
// MFMA operand is four consecutive values: one 8-byte load.
constexpr int OWT = (NP + 7) / 8 * 8, NWH = OWT + NH * NH;
static_assert(OB1 % 4 == 0 && OW2 % 4 == 0 && OB2 % 4 == 0 && OW3 % 4 == 0,
              "8-byte operand loads");
constexpr int kWaves = 4;               // waves per workgroup
constexpr int kGroup = 16 * kWaves;     // samples per workgroup iteration
constexpr int kMaxBlocks = 256;         // training workgroups (partial rows / 4)

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __host__ inline uint16_t bf16_bits(float x) {
    // Round to nearest even; upper 16 bits of the FP32 pattern.
    uint32_t u;
    memcpy(&u, &x, 4);
    u = u + 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ inline float bf16_val(uint16_t h) {
    return __uint_as_float((uint32_t)h << 16);
}

__device__ inline f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ inline float silu(float z) { return z / (1.0f + __expf(-z)); }
__device__ inline float dsilu(float z) {
    const float s = 1.0f / (1.0f + __expf(-z));
    return s * (1.0f + z * (1.0f - s));
}

struct Norm {
    float xm[NI], xs[NI], ym, ys;
};

// Per-lane weights of one wave.  Lane l (r = l%16, q = l/16):
//   w1[T]      A operand of layer 1, output tile T: W1[16T+r][4q..4q+3]
//              (inputs 8..15 are zero padding, q >= 2);
//   w2[T][t]   A operand of layer 2: W2[16T+r][16t+4q..+3];
//   b1/b2/w3   FP32 values for this lane's units u = 16T+4q+v (result layout).
struct FwdWeights {
    bf16x4 w1[4];
    bf16x4 w2[4][4];
    float b1[4][4], b2[4][4], w3[4][4], b3;
};

__device__ inline bf16x4 load4(const uint16_t *__restrict__ p) {
    return *reinterpret_cast<const bf16x4 *>(p);
}
__device__ inline void load4f(const uint16_t *__restrict__ p, float *v) {
    const bf16x4 h = load4(p);
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = bf16_val((uint16_t)h[k]);
}

__device__ inline void load_fwd(const uint16_t *__restrict__ wh, int l,
                                FwdWeights &W) {
    const int r = l & 15, q = l >> 4;
#pragma unroll
    for (int T = 0; T < 4; ++T) {
        const bf16x4 none = {0, 0, 0, 0};
        W.w1[T] = q < 2 ? load4(wh + OW1 + (16 * T + r) * NI + 4 * q) : none;
#pragma unroll
        for (int t = 0; t < 4; ++t)
            W.w2[T][t] = load4(wh + OW2 + (16 * T + r) * NH + 16 * t + 4 * q);
        const int u = 16 * T + 4 * q;
        load4f(wh + OB1 + u, W.b1[T]);
        load4f(wh + OB2 + u, W.b2[T]);
        load4f(wh + OW3 + u, W.w3[T]);
    }
    W.b3 = bf16_val(wh[OB3]);
}

// Layer-1 B operand of sample `sidx` (lanes q < 2 hold inputs 4q..4q+3).
__device__ inline bf16x4 input_operand(const Norm &nm, const float *__restrict__ x,
                                       int sidx, bool valid, int q, float *xh) {
    bf16x4 b = {0, 0, 0, 0};
#pragma unroll
    for (int v = 0; v < 4; ++v) xh[v] = 0.0f;
    if (valid && q < 2) {
        const float4 xv = *reinterpret_cast<const float4 *>(x + (size_t)NI * sidx + 4 * q);
        const float xx[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const uint16_t h = bf16_bits((xx[v] - nm.xm[4 * q + v]) / nm.xs[4 * q + v]);
            b[v] = (short)h;
            xh[v] = bf16_val(h);
        }
    }
    return b;
}

// Forward of the wave's 16 samples (result layout: lane = sample l%16, units
// 16T+4q+v): the network output for sample l%16, in every lane.
__device__ inline float forward16(const FwdWeights &W, bf16x4 xb) {
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    bf16x4 h1b[4];
#pragma unroll
    for (int T = 0; T < 4; ++T) {
        const f32x4 z = mfma16(W.w1[T], xb, zero);
#pragma unroll
        for (int v = 0; v < 4; ++v)
            h1b[T][v] = (short)bf16_bits(silu(z[v] + W.b1[T][v]));
    }
    float part = 0.0f;
#pragma unroll
    for (int T = 0; T < 4; ++T) {
        f32x4 z = zero;
#pragma unroll
        for (int t = 0; t < 4; ++t) z = mfma16(W.w2[T][t], h1b[t], z);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float h = bf16_val(bf16_bits(silu(z[v] + W.b2[T][v])));
            part = fmaf(W.w3[T][v], h, part);
        }
    }
    // Sum over the four lanes holding this sample (q = 0..3).
    part += __shfl_xor(part, 16);
    part += __shfl_xor(part, 32);
    return part + W.b3;
}

__global__ __launch_bounds__(256) void k_mlp_forward(
    int n, const float *__restrict__ x, const uint16_t *__restrict__ wh,
    Norm nm, float *__restrict__ y) {
    const int l = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = l & 15, q = l >> 4;
    FwdWeights W;
    load_fwd(wh, l, W);
    const int ngroups = (n + 15) / 16;
    for (int g = blockIdx.x * kWaves + wave; g < ngroups; g += gridDim.x * kWaves) {
        const int sidx = 16 * g + r;
        const bool valid = sidx < n;
        float xh[4];
        const bf16x4 xb = input_operand(nm, x, sidx, valid, q, xh);
        const float out = forward16(W, xb);
        if (valid && q == 0) y[sidx] = out * nm.ys + nm.ym;
    }
}

// Forward + backward of the samples idx[base .. base+count) (idx may be null:
// identity).  Loss = mean over the batch of (yhat - t_normalised)^2.  The
// derivative of the BF16 rounding is taken as 1 (straight-through).  Deltas
// d2 and d1 enter the MFMA products (d1 = W2^T d2, the weight gradients) as
// BF16; the bias and output-layer gradients use them in FP32.
//
// Workgroup b accumulates partial row b: the 16-sample groups b % 4 of the
// 64-sample blocks b / 4, b / 4 + gridDim / 4, ... in turn.  Its four
// wavefronts split a group by units: wavefront T evaluates units 16T..16T+15
// of every layer (an MFMA tile) and passes activations and deltas to the
// others through LDS.  A minibatch of 1024 has only 64 groups, and a
// wavefront alone on its SIMD issues an instruction every 7-8 cycles, so the
// length of a wavefront's instruction stream is the kernel's time: 16 us with
// a group per wavefront, 7 us so.
constexpr int LDS_ROW = NH + 8;   // bf16 per sample row (16-byte padding)
static_assert(NH == 16 * kWaves, "a wavefront per tile of units");
__global__ __launch_bounds__(256) void k_mlp_fwdbwd(
    int count, int base, const int *__restrict__ idx,
    const float *__restrict__ x, const float *__restrict__ t,
    const uint16_t *__restrict__ wh, Norm nm, float inv_batch,
    float *__restrict__ gpart, float *__restrict__ lpart) {
    __shared__ __align__(16) uint16_t h1s[16 * LDS_ROW], h2s[16 * LDS_ROW];
    __shared__ __align__(16) uint16_t d2s[16 * LDS_ROW], d1s[16 * LDS_ROW];
    __shared__ uint16_t xs[16 * 16];
    const int l = threadIdx.x & 63;
    const int T = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = l & 15, q = l >> 4;
    const int u0 = 16 * T + 4 * q;    // this lane's units of a result tile
    // Operands of this wavefront's tile (see FwdWeights), and of d1^T = W2^T
    // d2^T: lane holds W2[16t+4q+j][16T+r].
    const bf16x4 none = {0, 0, 0, 0};
    const bf16x4 w1 = q < 2 ? load4(wh + OW1 + (16 * T + r) * NI + 4 * q) : none;
    bf16x4 w2[4], w2t[4];
    float b1[4], b2[4], w3[4], w3all[4][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        w2[k] = load4(wh + OW2 + (16 * T + r) * NH + 16 * k + 4 * q);
        w2t[k] = load4(wh + OWT + (16 * T + r) * NH + 16 * k + 4 * q);
        load4f(wh + OW3 + 16 * k + 4 * q, w3all[k]);
    }
    load4f(wh + OB1 + u0, b1);
    load4f(wh + OB2 + u0, b2);
    load4f(wh + OW3 + u0, w3);
    const float b3 = bf16_val(wh[OB3]);
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 gw2[4], gw1 = zero;
    float gb1[4], gb2[4], gw3[4], gb3 = 0.0f, loss = 0.0f;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        gw2[v] = zero;
        gb1[v] = gb2[v] = gw3[v] = 0.0f;
    }
    const int row = r * LDS_ROW;      // this lane's sample
    const int nbg = (count + kGroup - 1) / kGroup;
    // Uniform trip count across the workgroup (barriers inside the loop).
    for (int bg = blockIdx.x / kWaves; bg < nbg; bg += gridDim.x / kWaves) {
        const int qi = bg * kGroup + 16 * (int)(blockIdx.x % kWaves) + r;
        const bool valid = qi < count;
        const int sidx = valid ? (idx ? idx[base + qi] : base + qi) : 0;
        float xh[4];
        const bf16x4 xb = input_operand(nm, x, sidx, valid, q, xh);
        const float tn = valid ? (t[sidx] - nm.ym) / nm.ys : 0.0f;
        bf16x4 hb;
        float ds1[4], ds2[4], h2[4];
        f32x4 z = mfma16(w1, xb, zero);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float zz = z[v] + b1[v];
            hb[v] = (short)bf16_bits(silu(zz));
            ds1[v] = dsilu(zz);
        }
        *reinterpret_cast<bf16x4 *>(h1s + row + u0) = hb;
        __syncthreads();
        z = zero;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            z = mfma16(w2[k], load4(h1s + row + 16 * k + 4 * q), z);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float zz = z[v] + b2[v];
            hb[v] = (short)bf16_bits(silu(zz));
            h2[v] = bf16_val((uint16_t)hb[v]);
            ds2[v] = dsilu(zz);
        }
        *reinterpret_cast<bf16x4 *>(h2s + row + u0) = hb;
        __syncthreads();
        // The output, in every wavefront: the lane's units of all tiles in
        // order, then the four lanes holding this sample (as in forward16).
        float part = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bf16x4 h = load4(h2s + row + 16 * k + 4 * q);
#pragma unroll
            for (int v = 0; v < 4; ++v)
                part = fmaf(w3all[k][v], bf16_val((uint16_t)h[v]), part);
        }
        part += __shfl_xor(part, 16);
        part += __shfl_xor(part, 32);
        const float out = part + b3;
        float d3 = 0.0f;
        if (valid) {
            const float e = out - tn;
            d3 = 2.0f * e * inv_batch;
            if (q == 0) loss += e * e;
        }
        if (q == 0) gb3 += d3;
        // d2 (result layout of layer 2 = B operand of the d1 product).
        bf16x4 db;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float d2 = d3 * w3[v] * ds2[v];
            db[v] = (short)bf16_bits(d2);
            gb2[v] += d2;
            gw3[v] = fmaf(d3, h2[v], gw3[v]);
        }
        *reinterpret_cast<bf16x4 *>(d2s + row + u0) = db;
        __syncthreads();
        // d1^T = W2^T d2^T, then times silu'(z1).
        z = zero;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            z = mfma16(w2t[k], load4(d2s + row + 16 * k + 4 * q), z);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float d1 = z[v] * ds1[v];
            gb1[v] += d1;
            db[v] = (short)bf16_bits(d1);
        }
        *reinterpret_cast<bf16x4 *>(d1s + row + u0) = db;
        if (T == 0) {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                xs[r * 16 + 4 * q + v] = q < 2 ? bf16_bits(xh[v]) : 0;
        }
        __syncthreads();
        // Weight gradients: samples on the k dimension.
        //   gW2[b][a] += sum_s d2[s][b] h1[s][a]:  A[b][s], B[s][a]
        //   gW1[a][k] += sum_s d1[s][a] xh[s][k]:  A[a][s], B[s][k]
        bf16x4 ad2, ad1, bh1[4], bx;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int at = (4 * q + j) * LDS_ROW;
            ad2[j] = (short)d2s[at + 16 * T + r];
            ad1[j] = (short)d1s[at + 16 * T + r];
#pragma unroll
            for (int k = 0; k < 4; ++k) bh1[k][j] = (short)h1s[at + 16 * k + r];
            bx[j] = (short)xs[(4 * q + j) * 16 + r];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) gw2[k] = mfma16(ad2, bh1[k], gw2[k]);
        gw1 = mfma16(ad1, bx, gw1);
        __syncthreads();
    }
    // This wavefront's units of the partial row.
    float *g = gpart + (size_t)blockIdx.x * NP;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int u = u0 + v;   // row unit of the result tiles
#pragma unroll
        for (int k = 0; k < 4; ++k) g[OW2 + u * NH + 16 * k + r] = gw2[k][v];
        if (r < NI) g[OW1 + u * NI + r] = gw1[v];
        // Bias / output-layer sums over the 16 samples of this lane group.
        float a1 = gb1[v], a2 = gb2[v], a3 = gw3[v];
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            a1 += __shfl_xor(a1, o);
            a2 += __shfl_xor(a2, o);
            a3 += __shfl_xor(a3, o);
        }
        if (r == 0) {
            g[OB1 + u] = a1;
            g[OB2 + u] = a2;
            g[OW3 + u] = a3;
        }
    }
    if (T != 0) return;
    for (int o = 32; o >= 1; o >>= 1) {
        gb3 += __shfl_xor(gb3, o);
        loss += __shfl_xor(loss, o);
    }
    if (l == 0) {
        g[OB3] = gb3;
        lpart[blockIdx.x] = loss;
    }
}

// BF16 copy of parameter k (and its place in WT).
__device__ inline void store_bf16(uint16_t *__restrict__ wh, int k, float w) {
    const uint16_t h = bf16_bits(w);
    wh[k] = h;
    if (k >= OW2 && k < OB2) {
        const int b = (k - OW2) / NH, a = (k - OW2) % NH;
        wh[OWT + a * NH + b] = h;
    }
}

// Sum the nrow partial rows in row order; with adam != 0 apply one Adam step
// to the FP32 masters and refresh the BF16 copy.  One wavefront per 64
// parameters; kRedU rows are loaded together and added in order (a row at a
// time, the kernel was one memory round trip per few rows: 64 rows 17 us,
// now 4 us).
constexpr int kRedU = 32;
__global__ __launch_bounds__(64) void k_mlp_reduce(
    int nrow, const float *__restrict__ gpart, float *__restrict__ gsum,
    int adam, float lr, float b1, float b2, float eps, float c1, float c2,
    float *__restrict__ w, uint16_t *__restrict__ wh, float *__restrict__ m,
    float *__restrict__ v) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= NP) return;
    float m0 = 0.0f, v0 = 0.0f, w0 = 0.0f;
    if (adam) {
        m0 = m[k];
        v0 = v[k];
        w0 = w[k];
    }
    float g = 0.0f;
    const float *__restrict__ p = gpart + k;
    int b = 0;
    for (; b + kRedU <= nrow; b += kRedU) {
        float r[kRedU];
#pragma unroll
        for (int u = 0; u < kRedU; ++u) r[u] = p[(size_t)(b + u) * NP];
#pragma unroll
        for (int u = 0; u < kRedU; ++u) g += r[u];
    }
    if (b < nrow) {
        float r[kRedU];
#pragma unroll
        for (int u = 0; u < kRedU; ++u)
            r[u] = b + u < nrow ? p[(size_t)(b + u) * NP] : 0.0f;
#pragma unroll
        for (int u = 0; u < kRedU; ++u)
            if (b + u < nrow) g += r[u];
    }
    gsum[k] = g;
    if (adam) {
        const float mk = b1 * m0 + (1.0f - b1) * g;
        const float vk = b2 * v0 + (1.0f - b2) * g * g;
        m[k] = mk;
        v[k] = vk;
        const float wk = w0 - lr * (mk / c1) / (sqrtf(vk / c2) + eps);
        w[k] = wk;
        store_bf16(wh, k, wk);
    }
}

__global__ void k_bf16_copy(const float *__restrict__ w, uint16_t *__restrict__ wh) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < NP) store_bf16(wh, k, w[k]);
}

// ---------------------------------------------------------------------------
// Host state and C-ABI
// ---------------------------------------------------------------------------

struct State {
    bool init = false;
    hipStream_t st = nullptr;
    float *w = nullptr, *m = nullptr, *v = nullptr;
    uint16_t *wh = nullptr;      // BF16 copy of the parameters
    float *gsum = nullptr;
    Norm nm{};
    long long adam_t = 0;
    // device copies of data
    float *dx = nullptr, *dt = nullptr, *dy = nullptr, *gpart = nullptr,
          *lpart = nullptr;
    int *didx = nullptr;
    size_t cap_n = 0, cap_rows = 0, cap_loss = 0;
};
State M;

#define MCHK(e)                                                               \
    do {                                                                      \
        hipError_t r_ = (e);                                                  \
        if (r_ != hipSuccess)                                                 \
            throw std::runtime_error(std::string(#e) + ": " +                 \
                                     hipGetErrorString(r_));                  \
    } while (0)

void ensure_init() {
    if (M.init) return;
    MCHK(hipStreamCreateWithFlags(&M.st, hipStreamNonBlocking));
    MCHK(hipMalloc((void **)&M.w, NP * sizeof(float)));
    MCHK(hipMalloc((void **)&M.wh, NWH * sizeof(uint16_t)));
    MCHK(hipMalloc((void **)&M.m, NP * sizeof(float)));
    MCHK(hipMalloc((void **)&M.v, NP * sizeof(float)));
    MCHK(hipMalloc((void **)&M.gsum, NP * sizeof(float)));
    for (int k = 0; k < NI; ++k) {
        M.nm.xm[k] = 0.0f;
        M.nm.xs[k] = 1.0f;
    }
    M.nm.ym = 0.0f;
    M.nm.ys = 1.0f;
    M.init = true;
}

// Samples, partial gradient rows and partial losses the buffers hold.
void ensure_data(size_t n, size_t nrows, size_t nloss) {
    if (n > M.cap_n) {
        if (M.dx) (void)hipFree(M.dx);
        if (M.dt) (void)hipFree(M.dt);
        if (M.dy) (void)hipFree(M.dy);
        if (M.didx) (void)hipFree(M.didx);
        MCHK(hipMalloc((void **)&M.dx, n * NI * sizeof(float)));
        MCHK(hipMalloc((void **)&M.dt, n * sizeof(float)));
        MCHK(hipMalloc((void **)&M.dy, n * sizeof(float)));
        MCHK(hipMalloc((void **)&M.didx, n * sizeof(int)));
        M.cap_n = n;
    }
    if (nrows > M.cap_rows) {
        if (M.gpart) (void)hipFree(M.gpart);
        M.gpart = nullptr;
        M.cap_rows = 0;
        MCHK(hipMalloc((void **)&M.gpart, nrows * NP * sizeof(float)));
        M.cap_rows = nrows;
    }
    if (nloss > M.cap_loss) {
        if (M.lpart) (void)hipFree(M.lpart);
        M.lpart = nullptr;
        M.cap_loss = 0;
        MCHK(hipMalloc((void **)&M.lpart, nloss * sizeof(float)));
        M.cap_loss = nloss;
    }
}

void set_params(const float *p) {
    ensure_init();
    MCHK(hipMemcpyAsync(M.w, p, NP * sizeof(float), hipMemcpyHostToDevice, M.st));
    hipLaunchKernelGGL(k_bf16_copy, dim3((NP + 255) / 256), dim3(256), 0, M.st,
                       M.w, M.wh);
    MCHK(hipMemsetAsync(M.m, 0, NP * sizeof(float), M.st));
    MCHK(hipMemsetAsync(M.v, 0, NP * sizeof(float), M.st));
    MCHK(hipStreamSynchronize(M.st));
    M.adam_t = 0;
}

// Partial rows (one per workgroup) of a pass over count samples.
int rows_of(int count) {
    return std::min((count + kGroup - 1) / kGroup, kMaxBlocks) * kWaves;
}

// Enqueue one pass of forward+backward over count samples starting at base
// (through idx if given): gradient (mean-square loss) summed into M.gsum,
// optionally followed by an Adam step, and the summed squared errors of its
// rows_of(count) rows in lpart.
void grad_step(int count, int base, const int *didx, float lr, int adam,
               float *lpart) {
    const int nrows = rows_of(count);
    hipLaunchKernelGGL(k_mlp_fwdbwd, dim3(nrows), dim3(64 * kWaves), 0,
                       M.st, count, base, didx, M.dx, M.dt, M.wh, M.nm,
                       1.0f / count, M.gpart, lpart);
    float c1 = 1.0f, c2 = 1.0f;
    const float b1 = 0.9f, b2 = 0.999f;
    if (adam) {
        M.adam_t++;
        c1 = 1.0f - std::pow(b1, (float)M.adam_t);
        c2 = 1.0f - std::pow(b2, (float)M.adam_t);
    }
    hipLaunchKernelGGL(k_mlp_reduce, dim3((NP + 63) / 64), dim3(64), 0,
                       M.st, nrows, M.gpart, M.gsum, adam, lr, b1, b2, 1e-8f,
                       c1, c2, M.w, M.wh, M.m, M.v);
    MCHK(hipGetLastError());
}

// The summed squared error of one pass from its rows' sums.
double loss_sum(const float *lp, int nrows) {
    double l = 0.0;
    for (int k = 0; k < nrows; ++k) l += lp[k];
    return l;
}

void upload_data(int n, const float *x, const float *t) {
    ensure_init();
    ensure_data((size_t)n, 0, 0);
    MCHK(hipMemcpyAsync(M.dx, x, (size_t)n * NI * sizeof(float),
                        hipMemcpyHostToDevice, M.st));
    if (t)
        MCHK(hipMemcpyAsync(M.dt, t, (size_t)n * sizeof(float),
                            hipMemcpyHostToDevice, M.st));
}

}  // namespace gpunb_mlp

using namespace gpunb_mlp;

#define MLP_EXPORT __attribute__((visibility("default")))

extern "C" {

MLP_EXPORT int gpunb_mlp_nparams(void) { return NP; }

MLP_EXPORT int gpunb_mlp_init(unsigned seed) {
    return gpunb::run_guarded("gpunb_mlp_init", [&] {
        std::mt19937 rng(seed);
        std::vector<float> p(NP, 0.0f);
        auto fill = [&](int off, int fan_in, int fan_out, int count) {
            const float a = std::sqrt(6.0f / (fan_in + fan_out));
            std::uniform_real_distribution<float> u(-a, a);
            for (int k = 0; k < count; ++k) p[off + k] = u(rng);
        };
        fill(OW1, NI, NH, NH * NI);
        fill(OW2, NH, NH, NH * NH);
        fill(OW3, NH, 1, NH);
        set_params(p.data());
    });
}

MLP_EXPORT int gpunb_mlp_set_norm(const float *xmean, const float *xstd,
                                  float ymean, float ystd) {
    return gpunb::run_guarded("gpunb_mlp_set_norm", [&] {
        ensure_init();
        for (int k = 0; k < NI; ++k) {
            if (!(xstd[k] > 0.0f)) throw std::runtime_error("xstd must be > 0");
            M.nm.xm[k] = xmean[k];
            M.nm.xs[k] = xstd[k];
        }
        if (!(ystd > 0.0f)) throw std::runtime_error("ystd must be > 0");
        M.nm.ym = ymean;
        M.nm.ys = ystd;
    });
}

MLP_EXPORT int gpunb_mlp_get_params(float *p) {
    return gpunb::run_guarded("gpunb_mlp_get_params", [&] {
        ensure_init();
        MCHK(hipMemcpyAsync(p, M.w, NP * sizeof(float), hipMemcpyDeviceToHost,
                            M.st));
        MCHK(hipStreamSynchronize(M.st));
    });
}

MLP_EXPORT int gpunb_mlp_set_params(const float *p) {
    return gpunb::run_guarded("gpunb_mlp_set_params", [&] { set_params(p); });
}

MLP_EXPORT int gpunb_mlp_predict(int n, const float *x, float *y) {
    return gpunb::run_guarded("gpunb_mlp_predict", [&] {
        if (n <= 0) return;
        upload_data(n, x, nullptr);
        const int ngroups = (n + 15) / 16;
        const int nblk = std::min((ngroups + kWaves - 1) / kWaves, 2048);
        hipLaunchKernelGGL(k_mlp_forward, dim3(nblk), dim3(64 * kWaves), 0,
                           M.st, n, M.dx, M.wh, M.nm, M.dy);
        MCHK(hipGetLastError());
        MCHK(hipMemcpyAsync(y, M.dy, (size_t)n * sizeof(float),
                            hipMemcpyDeviceToHost, M.st));
        MCHK(hipStreamSynchronize(M.st));
    });
}

MLP_EXPORT int gpunb_mlp_grad(int n, const float *x, const float *t,
                              float *grad, double *loss) {
    return gpunb::run_guarded("gpunb_mlp_grad", [&] {
        if (n <= 0) throw std::runtime_error("n must be > 0");
        upload_data(n, x, t);
        const int nrows = rows_of(n);
        ensure_data(0, (size_t)nrows, (size_t)nrows);
        grad_step(n, 0, nullptr, 0.0f, 0, M.lpart);
        std::vector<float> lp(nrows);
        MCHK(hipMemcpyAsync(lp.data(), M.lpart, nrows * sizeof(float),
                            hipMemcpyDeviceToHost, M.st));
        MCHK(hipMemcpyAsync(grad, M.gsum, NP * sizeof(float),
                            hipMemcpyDeviceToHost, M.st));
        MCHK(hipStreamSynchronize(M.st));
        if (loss) *loss = loss_sum(lp.data(), nrows) / n;
    });
}

MLP_EXPORT int gpunb_mlp_train(int n, const float *x, const float *t,
                               int epochs, int batch, float lr, unsigned seed,
                               double *loss_out) {
    return gpunb::run_guarded("gpunb_mlp_train", [&] {
        if (n <= 0 || epochs <= 0 || batch <= 0)
            throw std::runtime_error("n, epochs and batch must be > 0");
        // The whole epoch is enqueued at once: the minibatches' losses stay on
        // the device (row_max partial sums each) until the last epoch is done.
        const int nb = (n - 1) / batch + 1;
        const int row_max = rows_of(std::min(batch, n));
        upload_data(n, x, t);
        ensure_data(0, (size_t)row_max, (size_t)nb * row_max);
        std::vector<int> idx(n);
        for (int k = 0; k < n; ++k) idx[k] = k;
        std::mt19937 rng(seed);
        for (int e = 0; e < epochs; ++e) {
            std::shuffle(idx.begin(), idx.end(), rng);
            // Synchronous where idx is shuffled again, and in stream order
            // behind the previous epoch, which reads the old order.
            if (e + 1 < epochs)
                MCHK(hipMemcpyWithStream(M.didx, idx.data(), (size_t)n * sizeof(int),
                                         hipMemcpyHostToDevice, M.st));
            else
                MCHK(hipMemcpyAsync(M.didx, idx.data(), (size_t)n * sizeof(int),
                                    hipMemcpyHostToDevice, M.st));
            for (int b = 0; b < nb; ++b) {
                const int b0 = b * batch;
                grad_step(std::min(batch, n - b0), b0, M.didx, lr, 1,
                          M.lpart + (size_t)b * row_max);
            }
        }
        std::vector<float> lp((size_t)nb * row_max);
        MCHK(hipMemcpyAsync(lp.data(), M.lpart, lp.size() * sizeof(float),
                            hipMemcpyDeviceToHost, M.st));
        MCHK(hipStreamSynchronize(M.st));
        double sum = 0.0;
        for (int b = 0; b < nb; ++b)
            sum += loss_sum(lp.data() + (size_t)b * row_max,
                            rows_of(std::min(batch, n - b * batch)));
        if (loss_out) *loss_out = sum / n;
    });
}

}  // extern "C"
