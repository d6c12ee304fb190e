// dfsph_mlp.hip -- learned warm start of the two pressure solvers (no
// reference counterpart; the warm starts it replaces are the kappaV rescale of
// DFSPH_core_cuda.cu:240 and the kappa rescale of :3063-3068).
//
// A per-particle MLP 12 -> 64 -> 64 -> 64 -> 2 with SiLU activations predicts
// the converged (kappaV h, kappa h_f^2) of a step, the dt-invariant units of
// the reference CPU path (TimeStepDFSPH.cpp:458-459, 659-660), as a correction
// to the reference warm start formed from the previous step's totals
// (ws_base): the network's outputs are the totals less that warm start, and
// the solver's prediction adds it back.  Weights are
// BF16 on the matrix cores (v_mfma_f32_16x16x16_bf16, FP32 accumulate);
// biases, activations between layers and all reductions are FP32.
//
// MFMA 16x16x16 operand layout (lane l = 0..63, q = 0..3):
//   A[i][k]: lane l holds A[l % 16][4 (l / 16) + q]
//   B[k][n]: lane l holds B[4 (l / 16) + q][l % 16]
//   D[i][n]: lane l holds D[4 (l / 16) + q][l % 16]
// Layers are computed transposed, H_out^T = W H_in^T, with 16 samples as the N
// dimension: the output tile a lane holds is the B operand of the next layer's
// matching K block.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/dfsph_hip.h"
#include "dfsph_launch.hpp"
#include "dfsph_mlp_api.hpp"

namespace dfsph {

constexpr int kIn = 12, kH = 64, kOut = 2;
constexpr int kInPad = 16, kOutPad = 16;
// parameter offsets of the flat FP32 layout shared with the oracle:
// W1[64x12] b1[64] W2[64x64] b2[64] W3[64x64] b3[64] W4[2x64] b4[2]
constexpr int oW1 = 0, ob1 = oW1 + kH * kIn, oW2 = ob1 + kH, ob2 = oW2 + kH * kH, oW3 = ob2 + kH,
              ob3 = oW3 + kH * kH, oW4 = ob3 + kH, ob4 = oW4 + kOut * kH, kNParam = ob4 + kOut;
constexpr int kNNorm = 2 * kIn + 2 * kOut;   // in_mu, in_sig, out_mu, out_sig

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned short f2bf(float f)
{
    // round to nearest even (finite inputs)
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }

__device__ __forceinline__ float dsilu(float z)
{
    const float s = 1.0f / (1.0f + __expf(-z));
    return s * (1.0f + z * (1.0f - s));
}

__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Device copy of the model: padded BF16 weight matrices for the matrix cores
// and FP32 biases / normalisation.
struct DevModel {
    unsigned short W1[kH * kInPad];      // [64][16], columns 12..15 zero
    unsigned short W2[kH * kH];
    unsigned short W3[kH * kH];
    unsigned short W4[kOutPad * kH];     // [16][64], rows 2..15 zero
    unsigned short W2t[kH * kH];         // transposed (in x out): the backward pass's A operands
    unsigned short W3t[kH * kH];
    unsigned short W4t[kH * kOutPad];    // [64][16], columns 2..15 zero
    float b1[kH], b2[kH], b3[kH], b4[kOutPad];
    float norm[kNNorm];
};

// ---------------------------------------------------------------- inference
// x: [n][12] raw features (FP32); output o of row r goes to y[r * ystride + o * ocol]
// (denormalised when normalise is set: the solver's corrections).
//
// Register-resident form: each layer is computed transposed, H_out^T = W H_in^T,
// with W as the MFMA A operand and the particles as the N dimension.  The
// 16x16 output tile a lane holds (out features 4 (l/16) + q of 16 particles)
// is exactly the B operand layout of the next layer's matching K block, so
// activations never leave registers.  The weights' A fragments are loaded
// once into registers and each wave runs over 16-particle tiles; biases come
// from LDS as accumulator seeds.  Launch bounds ask for 3 waves per SIMD (168
// VGPRs, no spills; the default allocation held 2, and 4 spill).
constexpr int kInferBlock = 256;

__device__ __forceinline__ bf16x4 frag8(const unsigned short* p)     // 4 consecutive bf16 (8-byte aligned)
{
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    bf16x4 r;
    r[0] = (short)(u.x & 0xffffu); r[1] = (short)(u.x >> 16);
    r[2] = (short)(u.y & 0xffffu); r[3] = (short)(u.y >> 16);
    return r;
}

// Inference activation: SiLU with the hardware reciprocal (z / (1 + e^-z) to
// about 1 ulp; the IEEE division took three quarters of the kernel's vector
// instructions), rounded to bf16 two at a time by v_cvt_pk_bf16_f32 (round
// to nearest even, as f2bf).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float silu_fast(float z) { return z * __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }

__device__ __forceinline__ bf16x4 pack_bf16(float a, float b, float c, float d)
{
    struct {
        bf16x2 lo, hi;
    } p{__builtin_convertvector(f32x2{a, b}, bf16x2), __builtin_convertvector(f32x2{c, d}, bf16x2)};
    return __builtin_bit_cast(bf16x4, p);
}

__device__ __forceinline__ bf16x4 act_frag(const f32x4& z)
{
    return pack_bf16(silu_fast(z[0]), silu_fast(z[1]), silu_fast(z[2]), silu_fast(z[3]));
}

__global__ __launch_bounds__(kInferBlock, 3) void k_mlp_infer(const DevModel* __restrict__ Mg, const float* __restrict__ x,
                                                           uint32_t n, float* __restrict__ y, int normalise,
                                                           int ystride, int ocol)
{
    __shared__ __align__(16) float sb[3 * kH + kOutPad];
    const DevModel& M = *Mg;
    for (int k = threadIdx.x; k < 3 * kH + kOutPad; k += blockDim.x)
        sb[k] = k < kH ? M.b1[k] : k < 2 * kH ? M.b2[k - kH] : k < 3 * kH ? M.b3[k - 2 * kH] : M.b4[k - 3 * kH];
    __syncthreads();
    const int l = threadIdx.x & 63, r = l & 15, g = l >> 4;   // particle column, 4-row group
    bf16x4 w1[4], w2[4][4], w3[4][4], w4[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
        w1[mt] = frag8(M.W1 + (mt * 16 + r) * kInPad + 4 * g);
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            w2[mt][kt] = frag8(M.W2 + (mt * 16 + r) * kH + kt * 16 + 4 * g);
            w3[mt][kt] = frag8(M.W3 + (mt * 16 + r) * kH + kt * 16 + 4 * g);
        }
        w4[mt] = frag8(M.W4 + r * kH + mt * 16 + 4 * g);      // K block mt of the (padded) output layer
    }
    float mu[4], isg[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int f = 4 * g + j;
        mu[j] = (normalise && f < kIn) ? M.norm[f] : 0.0f;
        isg[j] = (normalise && f < kIn) ? 1.0f / M.norm[kIn + f] : 1.0f;
    }
    const uint32_t tiles = (n + 15) / 16;
    const uint32_t waves = gridDim.x * (blockDim.x / 64);
    for (uint32_t t = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6); t < tiles; t += waves) {
        const uint32_t p = t * 16 + r;
        // layer 1 input: features 4g..4g+3 of particle p (12..15 zero)
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (p < n && g < 3) v = *reinterpret_cast<const float4*>(x + (size_t)p * kIn + 4 * g);
        bf16x4 h[4];
        {
            bf16x4 xb = pack_bf16((v.x - mu[0]) * isg[0], (v.y - mu[1]) * isg[1], (v.z - mu[2]) * isg[2],
                                  (v.w - mu[3]) * isg[3]);
            if (g == 3) xb = bf16x4{0, 0, 0, 0};
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                const float4 b = *reinterpret_cast<const float4*>(sb + mt * 16 + 4 * g);
                h[mt] = act_frag(mfma(w1[mt], xb, f32x4{b.x, b.y, b.z, b.w}));
            }
        }
#pragma unroll
        for (int layer = 0; layer < 2; ++layer) {
            bf16x4 o[4];
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                const float4 b = *reinterpret_cast<const float4*>(sb + (layer + 1) * kH + mt * 16 + 4 * g);
                f32x4 acc{b.x, b.y, b.z, b.w};
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) acc = mfma(layer == 0 ? w2[mt][kt] : w3[mt][kt], h[kt], acc);
                o[mt] = act_frag(acc);
            }
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) h[mt] = o[mt];
        }
        const float4 b = *reinterpret_cast<const float4*>(sb + 3 * kH + 4 * g);
        f32x4 acc{b.x, b.y, b.z, b.w};
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) acc = mfma(w4[kt], h[kt], acc);
        if (g == 0 && p < n) {                  // outputs 0 and 1 of particle p
#pragma unroll
            for (int o = 0; o < kOut; ++o) {
                float val = acc[o];
                if (normalise) val = val * M.norm[2 * kIn + kOut + o] + M.norm[2 * kIn + o];
                y[(size_t)p * ystride + (size_t)o * ocol] = val;
            }
        }
    }
}

// Each wavefront loads all weights (20 KB) before its first tile, so small calls
// get two wavefronts per SIMD (150k particles: 41 us with 2048 blocks, 24 with
// 768, 22 with 512).  From 20 tiles a wavefront the third resident one joins
// (1 M: 88 us with 512, 83 with 768; 781 blocks start a second round: 106), and
// very large calls take more rounds, which even out the end (4.2 M: 322 us with
// 512, 295 with 768, 289 with 2048).
static uint32_t infer_grid(uint32_t n)
{
    const uint32_t tiles = (n + 15) / 16, per_block = kInferBlock / 64;
    const uint32_t need = (tiles + per_block - 1) / per_block;
    if (need >= 20u * 2048u) return 2048u;
    return std::max(1u, std::min(need, std::clamp(need / 20u, 512u, 768u)));
}

// ---------------------------------------------------------------- training

// row `row` of a mini-batch: a counter-based hash (splitmix64) of the training set
__device__ __forceinline__ uint32_t batch_sample(uint64_t seed, uint32_t row, uint32_t nsrc)
{
    uint64_t z = seed + 0x9e3779b97f4a7c15ull * (uint64_t)(row + 1);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    z ^= z >> 31;
    return (uint32_t)(z % nsrc);
}

// Forward, loss 0.5 |y - t|^2 inv_total, and backward of n samples (rows of x and
// t, or, with nsrc > 0, rows drawn from nsrc by batch_sample), 64 a block.  Its
// parameter gradient (flat FP32 layout) goes to partial[blockIdx.x][kNParam] and
// its loss to loss[blockIdx.x].
//
// A mini-batch of 4096 is 64 blocks, so a block's time is its chain of layers:
// 16 wavefronts share it, four per tile of 16 samples, each computing 16 of a
// layer's 64 features.  Activations and their gradients pass between a
// tile's wavefronts through LDS in the operand layout (ex), and once more with
// a feature's 16 samples together (tr_*), the operands of the weight
// gradients (K = samples), whose 16 x 16 tiles the wavefronts then share.
// The sums have the order of one wavefront taking the 64 samples in turn (as a
// mini-batch took 47 us; now 18): samples in K, then blocks, then wavefronts.
constexpr int kGradBlock = 1024, kGradSamples = 64;

__global__ __launch_bounds__(kGradBlock) void k_mlp_grad(const DevModel* __restrict__ Mg, const float* __restrict__ x,
                                                         const float* __restrict__ t, uint32_t n, uint32_t nsrc,
                                                         uint64_t seed, float inv_total, int normalise,
                                                         float* __restrict__ partial, float* __restrict__ loss)
{
    __shared__ bf16x4 ex[5][4][4][64];                  // h1, h2, h3, dz3, dz2 of each tile
    __shared__ __align__(8) unsigned short tr_h[3][4][kH][16], tr_d[3][4][kH][16], tr_x[4][kInPad][16],
        tr_y[4][kOutPad][16];
    __shared__ float s_e2[kOut][kGradSamples];          // e^2 / 2 of each output
    const DevModel& M = *Mg;
    const int l = threadIdx.x & 63, W = threadIdx.x >> 6, T = W >> 2, w = W & 3;
    const int r = l & 15, g = l >> 4;                   // sample column, 4-row group
    const int row0 = w * 16 + 4 * g;                    // the lane's first feature
    const uint32_t row = blockIdx.x * kGradSamples + T * 16u + (uint32_t)r;
    const bool valid = row < n;
    const uint32_t src = !valid ? 0u : nsrc ? batch_sample(seed, row, nsrc) : row;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (valid && g < 3) v = *reinterpret_cast<const float4*>(x + (size_t)src * kIn + 4 * g);
    float tv[kOut] = {0.0f, 0.0f};
    if (valid && g == 0) {
#pragma unroll
        for (int o = 0; o < kOut; ++o) tv[o] = t[(size_t)src * kOut + o];
    }
    const bf16x4 w1 = frag8(M.W1 + (w * 16 + r) * kInPad + 4 * g), w4t = frag8(M.W4t + (w * 16 + r) * kOutPad + 4 * g);
    bf16x4 w2[4], w3[4], w4[4], w3t[4], w2t[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
        w2[kt] = frag8(M.W2 + (w * 16 + r) * kH + kt * 16 + 4 * g);
        w3[kt] = frag8(M.W3 + (w * 16 + r) * kH + kt * 16 + 4 * g);
        w4[kt] = frag8(M.W4 + r * kH + kt * 16 + 4 * g);
        w3t[kt] = frag8(M.W3t + (w * 16 + r) * kH + kt * 16 + 4 * g);
        w2t[kt] = frag8(M.W2t + (w * 16 + r) * kH + kt * 16 + 4 * g);
    }
    const f32x4 zero{0.0f, 0.0f, 0.0f, 0.0f};
    auto put = [&](unsigned short (*tr)[16], int at, const bf16x4& b) {    // the lane's four rows of column r
#pragma unroll
        for (int q = 0; q < 4; ++q) tr[at + q][r] = (unsigned short)b[q];
    };
    auto samples = [&](const unsigned short (*tr)[16], int at) { return frag8(&tr[at][4 * g]); };
    auto product = [&](const bf16x4* wt, int k) {                          // rows of W H, H in ex[k]
        f32x4 a = zero;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) a = mfma(wt[kt], ex[k][T][kt][l], a);
        return a;
    };
    auto act = [&](f32x4& z, const float* b, int k) {                      // z += b, h = silu(z)
#pragma unroll
        for (int q = 0; q < 4; ++q) z[q] += b[row0 + q];
        const bf16x4 h = pack_bf16(silu(z[0]), silu(z[1]), silu(z[2]), silu(z[3]));
        ex[k][T][w][l] = h;
        put(tr_h[k][T], row0, h);
    };
    auto back = [&](const f32x4& d, const f32x4& z) {
        return pack_bf16(d[0] * dsilu(z[0]), d[1] * dsilu(z[1]), d[2] * dsilu(z[2]), d[3] * dsilu(z[3]));
    };
    if (valid && normalise && g < 3) {
        const float* mu = M.norm + 4 * g;
        const float* sg = M.norm + kIn + 4 * g;
        v = make_float4((v.x - mu[0]) / sg[0], (v.y - mu[1]) / sg[1], (v.z - mu[2]) / sg[2], (v.w - mu[3]) / sg[3]);
    }
    const bf16x4 xb = pack_bf16(v.x, v.y, v.z, v.w);
    if (w == 0) put(tr_x[T], 4 * g, xb);
    f32x4 z1 = mfma(w1, xb, zero);
    act(z1, M.b1, 0);
    __syncthreads();
    f32x4 z2 = product(w2, 0);
    act(z2, M.b2, 1);
    __syncthreads();
    f32x4 z3 = product(w3, 1);
    act(z3, M.b3, 2);
    __syncthreads();
    // every wavefront forms its tile's outputs (rows 0 and 1) and dY = (y - t) inv_total
    const f32x4 y = product(w4, 2);
    float d[kOut] = {0.0f, 0.0f}, e2[kOut] = {0.0f, 0.0f};
    if (valid && g == 0) {
#pragma unroll
        for (int o = 0; o < kOut; ++o) {
            if (normalise) tv[o] = (tv[o] - M.norm[2 * kIn + o]) / M.norm[2 * kIn + kOut + o];
            const float e = (y[o] + M.b4[o]) - tv[o];
            e2[o] = 0.5f * e * e;
            d[o] = e * inv_total;
        }
    }
    const bf16x4 dy = pack_bf16(d[0], d[1], 0.0f, 0.0f);
    if (w == 0) {
        put(tr_y[T], 4 * g, dy);
        if (g == 0) { s_e2[0][T * 16 + r] = e2[0]; s_e2[1][T * 16 + r] = e2[1]; }
    }
    const bf16x4 d3 = back(mfma(w4t, dy, zero), z3);
    ex[3][T][w][l] = d3;
    put(tr_d[2][T], row0, d3);
    __syncthreads();
    const bf16x4 d2 = back(product(w3t, 3), z2);
    ex[4][T][w][l] = d2;
    put(tr_d[1][T], row0, d2);
    __syncthreads();
    put(tr_d[0][T], row0, back(product(w2t, 4), z1));
    __syncthreads();
    // dW[o][k] = sum_s dZ[s][o] H[s][k], a 16 x 16 tile of W2 and of W3 a
    // wavefront; W1, W4 and the biases go to four each
    const int mt = W >> 2, nt = W & 3;
    float* out = partial + (size_t)blockIdx.x * kNParam;
    f32x4 g2 = zero, g3 = zero, gx = zero;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        g2 = mfma(samples(tr_d[1][k], mt * 16 + r), samples(tr_h[0][k], nt * 16 + r), g2);
        g3 = mfma(samples(tr_d[2][k], mt * 16 + r), samples(tr_h[1][k], nt * 16 + r), g3);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        out[oW2 + (mt * 16 + 4 * g + q) * kH + nt * 16 + r] = g2[q];
        out[oW3 + (mt * 16 + 4 * g + q) * kH + nt * 16 + r] = g3[q];
    }
    if (mt == 0) {                                      // W1, rows of tile nt
#pragma unroll
        for (int k = 0; k < 4; ++k) gx = mfma(samples(tr_d[0][k], nt * 16 + r), samples(tr_x[k], r), gx);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (r < kIn) out[oW1 + (nt * 16 + 4 * g + q) * kIn + r] = gx[q];
    } else if (mt == 1) {                               // W4, columns of tile nt
#pragma unroll
        for (int k = 0; k < 4; ++k) gx = mfma(samples(tr_y[k], r), samples(tr_h[2][k], nt * 16 + r), gx);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (4 * g + q < kOut) out[oW4 + (4 * g + q) * kH + nt * 16 + r] = gx[q];
    } else if (mt == 2) {                               // biases: a lane a feature, the samples in turn
        const int rows = nt < 3 ? kH : kOut;
        if (l < rows) {
            float sum = 0.0f;
            for (int k = 0; k < 4; ++k) {
                const unsigned short* p = nt < 3 ? tr_d[nt][k][l] : tr_y[k][l];
#pragma unroll
                for (int q = 0; q < 16; ++q) sum += __uint_as_float((uint32_t)p[q] << 16);
            }
            out[(nt == 0 ? ob1 : nt == 1 ? ob2 : nt == 2 ? ob3 : ob4) + l] = sum;
        }
    } else if (nt == 0 && l < 8) {                      // loss: output l & 1 of the samples 4 (l / 2) .. + 3 of each tile
        float sum = 0.0f;
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int q = 0; q < 4; ++q) sum = __builtin_fmaf(s_e2[l & 1][k * 16 + 4 * (l >> 1) + q], inv_total, sum);
        float all = __shfl(sum, 0, 64);
        for (int k = 1; k < 8; ++k) all += __shfl(sum, k, 64);
        if (l == 0) loss[blockIdx.x] = all;
    }
}

static uint32_t grad_grid(uint32_t n) { return (n + kGradSamples - 1) / kGradSamples; }

// One parameter of the flat layout into the model's copies.
__device__ __forceinline__ void pack_param(DevModel* M, uint32_t p, float w)
{
    const int q = (int)p;
    if (q < ob1) { M->W1[(q / kIn) * kInPad + q % kIn] = f2bf(w); }
    else if (q < oW2) { M->b1[q - ob1] = w; }
    else if (q < ob2) { const int e = q - oW2; M->W2[e] = f2bf(w); M->W2t[(e % kH) * kH + e / kH] = f2bf(w); }
    else if (q < oW3) { M->b2[q - ob2] = w; }
    else if (q < ob3) { const int e = q - oW3; M->W3[e] = f2bf(w); M->W3t[(e % kH) * kH + e / kH] = f2bf(w); }
    else if (q < oW4) { M->b3[q - ob3] = w; }
    else if (q < ob4) { const int e = q - oW4; M->W4[e] = f2bf(w); M->W4t[(e % kH) * kOutPad + e / kH] = f2bf(w); }
    else { M->b4[q - ob4] = w; }
}

// The blocks' partial gradients and losses summed in turn (many loads in flight),
// a thread a parameter, then either the gradient stored (grad) or one Adam
// step (Kingma & Ba 2015) on the FP32 master weights and their copies in the
// model.  The block after the last parameters sums the losses.
struct AdamArgs {
    float *w, *m, *v;
    float lr, b1, b2, eps, c1, c2;
};
constexpr uint32_t kUpdateBlock = 64, kUpdateGrid = (kNParam + kUpdateBlock - 1) / kUpdateBlock + 1;

__global__ __launch_bounds__(kUpdateBlock) void k_mlp_update(const float* __restrict__ partial,
                                                             const float* __restrict__ loss, uint32_t nparts,
                                                             float* __restrict__ grad, AdamArgs a,
                                                             DevModel* __restrict__ M, float* __restrict__ loss_out)
{
    const bool losses = blockIdx.x == kUpdateGrid - 1u;
    const uint32_t p = losses ? 0u : blockIdx.x * kUpdateBlock + threadIdx.x;
    if (p >= (uint32_t)kNParam || (losses && threadIdx.x != 0u)) return;
    const float* part = losses ? loss : partial + p;
    const size_t stride = losses ? 1u : (size_t)kNParam;
    float s = 0.0f;
    uint32_t b = 0;
    for (; b + 32u <= nparts; b += 32u) {
        float u[32];
#pragma unroll
        for (uint32_t k = 0; k < 32u; ++k) u[k] = part[(size_t)(b + k) * stride];
#pragma unroll
        for (uint32_t k = 0; k < 32u; ++k) s += u[k];
    }
    for (; b < nparts; ++b) s += part[(size_t)b * stride];
    if (losses) { *loss_out = s; return; }
    if (grad) { grad[p] = s; return; }
    const float mi = a.b1 * a.m[p] + (1.0f - a.b1) * s;
    const float vi = a.b2 * a.v[p] + (1.0f - a.b2) * s * s;
    a.m[p] = mi;
    a.v[p] = vi;
    const float wn = a.w[p] - a.lr * (mi * a.c1) / (sqrtf(vi * a.c2) + a.eps);
    a.w[p] = wn;
    pack_param(M, p, wn);
}

__global__ void k_mlp_pack(const float* __restrict__ w, const float* __restrict__ norm, DevModel* __restrict__ M)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < (uint32_t)(kH * kInPad)) {
        const int o = t / kInPad, k = t % kInPad;
        M->W1[t] = k < kIn ? f2bf(w[oW1 + o * kIn + k]) : 0;
    }
    if (t < (uint32_t)(kH * kH)) {
        const uint32_t tt = (t % kH) * kH + t / kH;
        M->W2[t] = M->W2t[tt] = f2bf(w[oW2 + t]);
        M->W3[t] = M->W3t[tt] = f2bf(w[oW3 + t]);
    }
    if (t < (uint32_t)(kOutPad * kH)) {
        const int o = t / kH;
        M->W4[t] = M->W4t[(t % kH) * kOutPad + o] = o < kOut ? f2bf(w[oW4 + t]) : 0;
    }
    if (t < (uint32_t)kH) {
        M->b1[t] = w[ob1 + t];
        M->b2[t] = w[ob2 + t];
        M->b3[t] = w[ob3 + t];
    }
    if (t < (uint32_t)kOutPad) M->b4[t] = t < (uint32_t)kOut ? w[ob4 + t] : 0.0f;
    if (t < (uint32_t)kNNorm) M->norm[t] = norm[t];
}

// ------------------------------------------------------------- model state

struct MlpState {
    DevModel* model = nullptr;
    float *w = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr, *norm = nullptr;
    float* partial = nullptr;
    float* lossp = nullptr;
    float* loss = nullptr;
    uint32_t partial_cap = 0;
    uint32_t adam_t = 0;
    bool loaded = false;
    // per-particle buffers of the solver integration
    float* feat = nullptr;      // [cap][12]
    float* pred = nullptr;      // [4][cap]: corrections (kappaV h, kappa h_f^2), then the last
                                // step's converged totals in the same units (the sweeps' bound)
    float* kvws = nullptr;      // predicted kappaV warm start (GPU units)
    uint32_t cap = 0;
    // training set
    float* ds_x = nullptr;
    float* ds_t = nullptr;
    uint32_t ds_cap = 0, ds_n = 0, ds_stride = 1;
    ~MlpState()
    {
        void* ps[] = {model, w, m, v, grad, norm, partial, lossp, loss, feat, pred, kvws, ds_x, ds_t};
        for (void* p : ps)
            if (p) (void)hipFree(p);
    }
};

void mlp_destroy(MlpState* m) { delete m; }

}  // namespace dfsph

// ------------------------------------------------------------- C ABI part
namespace {

using dfsph::MlpState;

int mfail(int code, const std::string& msg)
{
    dfsph::handle_set_error(msg.c_str());
    return code;
}

#define MHIP(x)                                                                                       \
    do {                                                                                              \
        hipError_t e_ = (x);                                                                          \
        if (e_ != hipSuccess) return mfail(DFSPH_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

template <class T>
int malloc_dev(T*& p, size_t n)
{
    if (p) (void)hipFree(p);
    p = nullptr;
    MHIP(hipMalloc((void**)&p, (n ? n : 1) * sizeof(T)));
    return DFSPH_OK;
}

int ensure_state(void* handle, MlpState** out)
{
    dfsph::MlpView v = dfsph::handle_view(handle);
    if (!*v.mlp) {
        MlpState* m = new MlpState();
        int rc = DFSPH_OK;
        if ((rc = malloc_dev(m->model, 1)) || (rc = malloc_dev(m->w, dfsph::kNParam)) ||
            (rc = malloc_dev(m->m, dfsph::kNParam)) || (rc = malloc_dev(m->v, dfsph::kNParam)) ||
            (rc = malloc_dev(m->grad, dfsph::kNParam)) || (rc = malloc_dev(m->norm, dfsph::kNNorm)) ||
            (rc = malloc_dev(m->loss, 1))) {
            delete m;
            return rc;
        }
        *v.mlp = m;
    }
    *out = *v.mlp;
    return DFSPH_OK;
}

int pack(MlpState* m, hipStream_t s)
{
    dfsph::k_mlp_pack<<<(dfsph::kH * dfsph::kH + 255) / 256, 256, 0, s>>>(m->w, m->norm, m->model);
    MHIP(hipGetLastError());
    return DFSPH_OK;
}

}  // namespace

// Staging of dfsph_mlp_forward_noalloc: features then outputs of up to
// DFSPH_MLP_NOALLOC_MAX samples, one copy per device for the life of the
// process.  Host code uses the device address that hipGetSymbolAddress
// returns for the current device, never the array's name.
static __device__ __align__(256) float scratch[(size_t)DFSPH_MLP_NOALLOC_MAX * (dfsph::kIn + dfsph::kOut)];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kMaxDevices] = {};

// the scratch address on the current device, looked up on its first use
int scratch_address(float** out)
{
    int dev = 0;
    MHIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return mfail(DFSPH_ERR_STATE, "device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        MHIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_ptr[dev] = static_cast<float*>(p);
    }
    *out = g_scratch_ptr[dev];
    return DFSPH_OK;
}
}  // namespace

extern "C" {

int dfsph_mlp_set_params(void* handle, const float* params, const float* norm)
{
    if (!params) return mfail(DFSPH_ERR_ARG, "null parameters");
    MlpState* m = nullptr;
    if (int rc = ensure_state(handle, &m)) return rc;
    hipStream_t s = dfsph::handle_view(handle).s;
    std::vector<float> nrm(dfsph::kNNorm);
    if (norm) std::memcpy(nrm.data(), norm, sizeof(float) * dfsph::kNNorm);
    else {
        for (int k = 0; k < dfsph::kIn; ++k) { nrm[k] = 0.0f; nrm[dfsph::kIn + k] = 1.0f; }
        for (int k = 0; k < dfsph::kOut; ++k) { nrm[2 * dfsph::kIn + k] = 0.0f; nrm[2 * dfsph::kIn + dfsph::kOut + k] = 1.0f; }
    }
    MHIP(hipMemcpyAsync(m->w, params, sizeof(float) * dfsph::kNParam, hipMemcpyHostToDevice, s));
    MHIP(hipMemcpyAsync(m->norm, nrm.data(), sizeof(float) * dfsph::kNNorm, hipMemcpyHostToDevice, s));
    MHIP(hipMemsetAsync(m->m, 0, sizeof(float) * dfsph::kNParam, s));
    MHIP(hipMemsetAsync(m->v, 0, sizeof(float) * dfsph::kNParam, s));
    m->adam_t = 0;
    if (int rc = pack(m, s)) return rc;
    MHIP(hipStreamSynchronize(s));
    m->loaded = true;
    return DFSPH_OK;
}

int dfsph_mlp_get_params(void* handle, float* params, float* norm)
{
    MlpState* m = nullptr;
    if (int rc = ensure_state(handle, &m)) return rc;
    if (!m->loaded) return mfail(DFSPH_ERR_NO_MODEL, "no model parameters set");
    hipStream_t s = dfsph::handle_view(handle).s;
    MHIP(hipStreamSynchronize(s));
    if (params) MHIP(hipMemcpy(params, m->w, sizeof(float) * dfsph::kNParam, hipMemcpyDeviceToHost));
    if (norm) MHIP(hipMemcpy(norm, m->norm, sizeof(float) * dfsph::kNNorm, hipMemcpyDeviceToHost));
    return DFSPH_OK;
}

int dfsph_mlp_forward(void* handle, const float* x, uint32_t n, float* y, int normalise)
{
    MlpState* m = nullptr;
    if (int rc = ensure_state(handle, &m)) return rc;
    if (!m->loaded) return mfail(DFSPH_ERR_NO_MODEL, "no model parameters set");
    if (n == 0) return DFSPH_OK;
    hipStream_t s = dfsph::handle_view(handle).s;
    float *dx = nullptr, *dy = nullptr;
    int rc = malloc_dev(dx, (size_t)n * dfsph::kIn);
    if (!rc) rc = malloc_dev(dy, (size_t)n * dfsph::kOut);
    if (!rc) {
        (void)hipMemcpyAsync(dx, x, sizeof(float) * n * dfsph::kIn, hipMemcpyHostToDevice, s);
        dfsph::k_mlp_infer<<<dfsph::infer_grid(n), dfsph::kInferBlock, 0, s>>>(m->model, dx, n, dy, normalise,
                                                                                  dfsph::kOut, 1);
        (void)hipMemcpyAsync(y, dy, sizeof(float) * n * dfsph::kOut, hipMemcpyDeviceToHost, s);
        if (hipStreamSynchronize(s) != hipSuccess) rc = mfail(DFSPH_ERR_HIP, "mlp forward");
    }
    if (dx) (void)hipFree(dx);
    if (dy) (void)hipFree(dy);
    return rc;
}

int dfsph_mlp_forward_noalloc(void* handle, const float* x, uint32_t n, float* y, int normalise)
{
    if (n > DFSPH_MLP_NOALLOC_MAX)
        return mfail(DFSPH_ERR_ARG, "dfsph_mlp_forward_noalloc: n exceeds DFSPH_MLP_NOALLOC_MAX (" +
                                        std::to_string(DFSPH_MLP_NOALLOC_MAX) + ")");
    if (n && (!x || !y)) return mfail(DFSPH_ERR_ARG, "null input or output");
    const dfsph::MlpView v = dfsph::handle_view(handle);
    MlpState* m = *v.mlp;            // never created here: that would allocate
    if (!m || !m->loaded) return mfail(DFSPH_ERR_NO_MODEL, "no model parameters set");
    if (n == 0) return DFSPH_OK;
    float* base = nullptr;
    if (int rc = scratch_address(&base)) return rc;
    float* dx = base;
    float* dy = base + (size_t)DFSPH_MLP_NOALLOC_MAX * dfsph::kIn;
    MHIP(hipMemcpyAsync(dx, x, sizeof(float) * n * dfsph::kIn, hipMemcpyHostToDevice, v.s));
    dfsph::k_mlp_infer<<<dfsph::infer_grid(n), dfsph::kInferBlock, 0, v.s>>>(m->model, dx, n, dy, normalise,
                                                                              dfsph::kOut, 1);
    MHIP(hipGetLastError());
    MHIP(hipMemcpyAsync(y, dy, sizeof(float) * n * dfsph::kOut, hipMemcpyDeviceToHost, v.s));
    MHIP(hipStreamSynchronize(v.s));
    return DFSPH_OK;
}

int dfsph_mlp_loss_grad(void* handle, const float* x, const float* t, uint32_t n, float* grad, double* loss,
                        int normalise)
{
    MlpState* m = nullptr;
    if (int rc = ensure_state(handle, &m)) return rc;
    if (!m->loaded) return mfail(DFSPH_ERR_NO_MODEL, "no model parameters set");
    if (n == 0) return mfail(DFSPH_ERR_ARG, "no samples");
    hipStream_t s = dfsph::handle_view(handle).s;
    const uint32_t nb = dfsph::grad_grid(n);
    float *dx = nullptr, *dt = nullptr, *part = nullptr, *lp = nullptr;
    int rc = malloc_dev(dx, (size_t)n * dfsph::kIn);
    if (!rc) rc = malloc_dev(dt, (size_t)n * dfsph::kOut);
    if (!rc) rc = malloc_dev(part, (size_t)nb * dfsph::kNParam);
    if (!rc) rc = malloc_dev(lp, nb);
    if (!rc) {
        (void)hipMemcpyAsync(dx, x, sizeof(float) * n * dfsph::kIn, hipMemcpyHostToDevice, s);
        (void)hipMemcpyAsync(dt, t, sizeof(float) * n * dfsph::kOut, hipMemcpyHostToDevice, s);
        dfsph::k_mlp_grad<<<nb, dfsph::kGradBlock, 0, s>>>(m->model, dx, dt, n, 0u, 0ull, 1.0f / (float)n, normalise, part,
                                                           lp);
        dfsph::k_mlp_update<<<dfsph::kUpdateGrid, dfsph::kUpdateBlock, 0, s>>>(part, lp, nb, m->grad,
                                                                                    dfsph::AdamArgs{}, nullptr, m->loss);
        float l = 0.0f;
        (void)hipMemcpyAsync(grad, m->grad, sizeof(float) * dfsph::kNParam, hipMemcpyDeviceToHost, s);
        (void)hipMemcpyAsync(&l, m->loss, sizeof(float), hipMemcpyDeviceToHost, s);
        if (hipStreamSynchronize(s) != hipSuccess) rc = mfail(DFSPH_ERR_HIP, "mlp grad");
        if (loss) *loss = l;
    }
    void* ps[] = {dx, dt, part, lp};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    return rc;
}

}  // extern "C"

namespace dfsph {

// ------------------------------------------------------- solver integration

bool mlp_loaded(const MlpState* m) { return m && m->loaded; }
bool mlp_harvesting(const MlpState* m) { return m && m->ds_cap > 0 && m->ds_n < m->ds_cap; }
float* mlp_feat(MlpState* m) { return m->feat; }
WsLearned mlp_ws_v(const MlpState* m, float diameter)
{
    return WsLearned{m->pred, m->pred + 2 * (size_t)m->cap, diameter};
}
WsLearned mlp_ws_p(const MlpState* m, float diameter)
{
    return WsLearned{m->pred + m->cap, m->pred + 3 * (size_t)m->cap, diameter * diameter};
}
float* mlp_prev_p(MlpState* m) { return m->pred + 3 * (size_t)m->cap; }
float* mlp_prev_v(MlpState* m) { return m->pred + 2 * (size_t)m->cap; }

int mlp_ensure_particles(MlpState* m, uint32_t cap)
{
    if (!m) return mfail(DFSPH_ERR_STATE, "no learned warm start state");
    if (cap <= m->cap && m->feat) return DFSPH_OK;
    if (int rc = malloc_dev(m->feat, (size_t)cap * kIn)) return rc;
    if (int rc = malloc_dev(m->pred, (size_t)cap * 4)) return rc;
    m->cap = cap;
    return DFSPH_OK;
}

int mlp_infer_particles(MlpState* m, hipStream_t s, uint32_t n)
{
    if (n == 0) return DFSPH_OK;
    k_mlp_infer<<<infer_grid(n), kInferBlock, 0, s>>>(m->model, m->feat, n, m->pred, 1, 1, (int)m->cap);
    MHIP(hipGetLastError());
    return DFSPH_OK;
}

int mlp_harvest_step(MlpState* m, hipStream_t s, const DevTime* t, uint32_t n, const float* kapv, const float* kap,
                     float diameter)
{
    if (!mlp_harvesting(m) || n == 0) return DFSPH_OK;
    const uint32_t stride = m->ds_stride ? m->ds_stride : 1;
    launch_harvest(s, t, n, stride, m->ds_n, m->ds_cap, m->feat, kapv, kap, diameter, m->ds_x, m->ds_t);
    MHIP(hipGetLastError());
    const uint32_t add = (n + stride - 1) / stride;
    m->ds_n = m->ds_n + add > m->ds_cap ? m->ds_cap : m->ds_n + add;
    return DFSPH_OK;
}

}  // namespace dfsph

extern "C" {

int dfsph_mlp_harvest(void* handle, uint32_t capacity, uint32_t stride)
{
    MlpState* m = nullptr;
    if (int rc = ensure_state(handle, &m)) return rc;
    if (capacity != m->ds_cap) {
        if (int rc = malloc_dev(m->ds_x, (size_t)capacity * dfsph::kIn)) return rc;
        if (int rc = malloc_dev(m->ds_t, (size_t)capacity * dfsph::kOut)) return rc;
    }
    m->ds_cap = capacity;
    m->ds_n = 0;
    m->ds_stride = stride ? stride : 1;
    return DFSPH_OK;
}

int dfsph_mlp_dataset_size(void* handle, uint32_t* n)
{
    MlpState* m = nullptr;
    if (int rc = ensure_state(handle, &m)) return rc;
    if (n) *n = m->ds_n;
    return DFSPH_OK;
}

int dfsph_mlp_dataset_download(void* handle, float* x, float* t, uint32_t n)
{
    MlpState* m = nullptr;
    if (int rc = ensure_state(handle, &m)) return rc;
    if (n > m->ds_n) return mfail(DFSPH_ERR_ARG, "more samples requested than harvested");
    MHIP(hipStreamSynchronize(dfsph::handle_view(handle).s));
    if (x && n) MHIP(hipMemcpy(x, m->ds_x, sizeof(float) * n * dfsph::kIn, hipMemcpyDeviceToHost));
    if (t && n) MHIP(hipMemcpy(t, m->ds_t, sizeof(float) * n * dfsph::kOut, hipMemcpyDeviceToHost));
    return DFSPH_OK;
}

int dfsph_mlp_dataset_upload(void* handle, const float* x, const float* t, uint32_t n)
{
    MlpState* m = nullptr;
    if (int rc = ensure_state(handle, &m)) return rc;
    if (int rc = dfsph_mlp_harvest(handle, n, 1)) return rc;
    hipStream_t s = dfsph::handle_view(handle).s;
    if (n) {
        MHIP(hipMemcpyAsync(m->ds_x, x, sizeof(float) * n * dfsph::kIn, hipMemcpyHostToDevice, s));
        MHIP(hipMemcpyAsync(m->ds_t, t, sizeof(float) * n * dfsph::kOut, hipMemcpyHostToDevice, s));
        MHIP(hipStreamSynchronize(s));
    }
    m->ds_n = n;
    m->ds_cap = n;   // full: no further harvesting into it
    return DFSPH_OK;
}

// Mean / standard deviation of the training set's features and targets (FP64
// on the host) become the model's normalisation.
int dfsph_mlp_fit_normalization(void* handle)
{
    MlpState* m = nullptr;
    if (int rc = ensure_state(handle, &m)) return rc;
    if (!m->loaded) return mfail(DFSPH_ERR_NO_MODEL, "set initial parameters first");
    const uint32_t n = m->ds_n;
    if (n < 2) return mfail(DFSPH_ERR_STATE, "training set is empty");
    std::vector<float> x((size_t)n * dfsph::kIn), t((size_t)n * dfsph::kOut);
    if (int rc = dfsph_mlp_dataset_download(handle, x.data(), t.data(), n)) return rc;
    std::vector<float> nrm(dfsph::kNNorm);
    auto stats = [&](const std::vector<float>& a, int w, int col, float* mu, float* sd) {
        double s = 0.0, s2 = 0.0;
        for (uint32_t i = 0; i < n; ++i) {
            const double v = a[(size_t)i * w + col];
            s += v;
            s2 += v * v;
        }
        // no absolute floor on the spread: the dt-invariant totals are O(1e-9)
        // in SI units; only a constant column falls back to its magnitude or 1
        const double mean = s / n, var = std::max(s2 / n - mean * mean, 0.0);
        double dev = std::sqrt(var);
        if (!(dev > 1e-7 * std::fabs(mean)) || !(dev > 1e-30)) dev = std::max(std::fabs(mean), 1.0);
        *mu = (float)mean;
        *sd = (float)dev;
    };
    for (int k = 0; k < dfsph::kIn; ++k) stats(x, dfsph::kIn, k, &nrm[k], &nrm[dfsph::kIn + k]);
    for (int k = 0; k < dfsph::kOut; ++k)
        stats(t, dfsph::kOut, k, &nrm[2 * dfsph::kIn + k], &nrm[2 * dfsph::kIn + dfsph::kOut + k]);
    hipStream_t s = dfsph::handle_view(handle).s;
    MHIP(hipMemcpyAsync(m->norm, nrm.data(), sizeof(float) * dfsph::kNNorm, hipMemcpyHostToDevice, s));
    if (int rc = pack(m, s)) return rc;
    MHIP(hipStreamSynchronize(s));
    return DFSPH_OK;
}

// Mini-batch Adam on the training set with the normalised loss; the learning
// rate decays linearly to 10 % over the run.  loss_first / loss_last: the
// batch losses of the first and last step.
int dfsph_mlp_train(void* handle, uint32_t steps, uint32_t batch, float lr, uint32_t seed, float* loss_first,
                    float* loss_last)
{
    MlpState* m = nullptr;
    if (int rc = ensure_state(handle, &m)) return rc;
    if (!m->loaded) return mfail(DFSPH_ERR_NO_MODEL, "set initial parameters first");
    if (m->ds_n == 0) return mfail(DFSPH_ERR_STATE, "training set is empty");
    if (batch == 0 || batch % 64) return mfail(DFSPH_ERR_ARG, "batch must be a positive multiple of 64");
    hipStream_t s = dfsph::handle_view(handle).s;
    const uint32_t nb = dfsph::grad_grid(batch);
    if (nb > m->partial_cap) {
        if (int rc = malloc_dev(m->partial, (size_t)nb * dfsph::kNParam)) return rc;
        if (int rc = malloc_dev(m->lossp, nb)) return rc;
        m->partial_cap = nb;
    }
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (uint32_t it = 0; it < steps; ++it) {
        dfsph::k_mlp_grad<<<nb, dfsph::kGradBlock, 0, s>>>(m->model, m->ds_x, m->ds_t, batch, m->ds_n,
                                                           ((uint64_t)seed << 32) ^ (uint64_t)it * 0x632be59bd9b4e019ull,
                                                           1.0f / (float)batch, 1, m->partial, m->lossp);
        m->adam_t++;
        const float c1 = 1.0f / (1.0f - std::pow(b1, (float)m->adam_t));
        const float c2 = 1.0f / (1.0f - std::pow(b2, (float)m->adam_t));
        const float lr_t = lr * (1.0f - 0.9f * (float)it / (float)(steps > 1 ? steps - 1 : 1));
        dfsph::k_mlp_update<<<dfsph::kUpdateGrid, dfsph::kUpdateBlock, 0, s>>>(
            m->partial, m->lossp, nb, nullptr, dfsph::AdamArgs{m->w, m->m, m->v, lr_t, b1, b2, eps, c1, c2}, m->model,
            m->loss);
        if (it == 0 && loss_first) MHIP(hipMemcpyAsync(loss_first, m->loss, sizeof(float), hipMemcpyDeviceToHost, s));
        if (it + 1 == steps && loss_last) MHIP(hipMemcpyAsync(loss_last, m->loss, sizeof(float), hipMemcpyDeviceToHost, s));
    }
    MHIP(hipGetLastError());
    MHIP(hipStreamSynchronize(s));
    return DFSPH_OK;
}

// features and predictions of the last learned / harvesting step (device order)
int dfsph_mlp_step_features(void* handle, float* feat, float* pred_v, float* pred_p, uint32_t n)
{
    MlpState* m = nullptr;
    if (int rc = ensure_state(handle, &m)) return rc;
    if (!m->feat || n > m->cap) return mfail(DFSPH_ERR_STATE, "no features computed");
    MHIP(hipStreamSynchronize(dfsph::handle_view(handle).s));
    if (feat) MHIP(hipMemcpy(feat, m->feat, sizeof(float) * n * dfsph::kIn, hipMemcpyDeviceToHost));
    if (pred_v) MHIP(hipMemcpy(pred_v, m->pred, sizeof(float) * n, hipMemcpyDeviceToHost));
    if (pred_p) MHIP(hipMemcpy(pred_p, m->pred + m->cap, sizeof(float) * n, hipMemcpyDeviceToHost));
    return DFSPH_OK;
}

}  // extern "C"
