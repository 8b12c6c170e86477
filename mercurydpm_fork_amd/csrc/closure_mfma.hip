// closure_mfma.hip -- the learned closure as configured for the rheology of
// dense chute flow: a multilayer perceptron 4 -> 128 -> 128 -> 128 -> 2
// (GELU hidden layers, linear output) with BF16 weights and FP32
// accumulation, trained by full-batch Adam on FP32 master weights.
//
// The two 128 x 128 layers run on the matrix cores (v_mfma_f32_16x16x32_bf16)
// in the forward pass (Z = H W^T), the data gradient (dH = dZ W) and the weight
// gradient (dW = dZ^T H).  One kernel takes a tile of samples through the whole
// network: inference keeps everything between the input and the output in
// registers and LDS, training also goes back through the network and adds the
// tile's gradient, and a second kernel sums the blocks' gradients in a fixed
// order (four runs of blocks, then the runs: the same bits every time) and
// applies Adam.  The 4-wide
// input layer and the 2-wide output layer are too narrow for a tile and run on
// the vector units with the same BF16 weights.  Activations fed to a matrix
// instruction are rounded to BF16 (round to nearest even); pre-activations,
// GELU and every sum stay FP32.
//
// Parameter layout (FP32, one flat array): W1[128][4], b1[128],
// W2[128][128], b2[128], W3[128][128], b3[128], W4[2][128], b4[2].
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

#include "../../include/mercurydpm_closure.h"

namespace {

constexpr int kH = DEM_CLOSURE_HIDDEN;  // 128
constexpr int kIn = 4, kOut = 2;
constexpr int oW1 = 0, oB1 = oW1 + kH * kIn, oW2 = oB1 + kH, oB2 = oW2 + kH * kH, oW3 = oB2 + kH,
              oB3 = oW3 + kH * kH, oW4 = oB3 + kH, oB4 = oW4 + kOut * kH, kP = oB4 + kOut;
static_assert(kP == DEM_CLOSURE_PARAMS, "parameter count");
constexpr int kBlock = 256;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint16_t ushort4_t __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (finite values)
__host__ __device__ inline uint16_t to_bf16(float f)
{
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__host__ __device__ inline float from_bf16(uint16_t h)
{
    const uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

// GELU, 0.5 z (1 + erf(z / sqrt 2)), and its derivative
__device__ inline float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ inline float gelu_grad(float z)
{
    return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// BF16 weights as the kernels read them: W1 and W4 row-major, then W2 and W3
// twice in operand order, for the forward pass (kF2, kF3: W as the second
// operand of H W^T) and for the data gradient (kT2, kT3: of dZ W).  In operand
// order the 8 values of lane l for tile t (16 columns of the product) and step
// k (32 deep) lie at ((t * 4 + k) * 64 + l) * 8: a wavefront loads an operand
// as one 1 KB run.
constexpr int kTile = kH * kH;
constexpr int kF2 = 1024, kF3 = kF2 + kTile, kT2 = kF3 + kTile, kT3 = kT2 + kTile, kPacked = kT3 + kTile;
constexpr int kPackW1 = 0, kPackW4 = 512;
static_assert(kH * kIn == 512 && kOut * kH == 256 && kH == 128, "packed layout");

// where weight (row, column of the product) = (col, depth) lies in operand order
__host__ __device__ inline int operand_at(int col, int depth)
{
    return (((col >> 4) * 4 + (depth >> 5)) * 64 + ((depth >> 3) & 3) * 16 + (col & 15)) * 8 + (depth & 7);
}

// parameter i, rounded, into the packed weights (biases are read as FP32)
__device__ inline void pack_param(uint16_t* __restrict__ wb, int i, float v)
{
    const uint16_t h = to_bf16(v);
    if (i < oB1) {
        wb[kPackW1 + i] = h;
    } else if (i >= oW2 && i < oB2) {
        const int o = (i - oW2) / kH, k = (i - oW2) % kH;
        wb[kF2 + operand_at(o, k)] = h;
        wb[kT2 + operand_at(k, o)] = h;
    } else if (i >= oW3 && i < oB3) {
        const int o = (i - oW3) / kH, k = (i - oW3) % kH;
        wb[kF3 + operand_at(o, k)] = h;
        wb[kT3 + operand_at(k, o)] = h;
    } else if (i >= oW4 && i < oB4) {
        wb[kPackW4 + i - oW4] = h;
    }
}

__global__ void k_pack(const float* __restrict__ p, uint16_t* __restrict__ wb)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kP) pack_param(wb, i, p[i]);
}

// orders the LDS accesses of a wavefront's lanes
__device__ inline void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A wavefront holds 16 samples: lane l = 16 q + r has, of an activation, the
// values of samples 4 q + i (i = 0..3) and columns 16 t + r (t = 0..7), which
// is how a matrix instruction leaves its result.  As the next first operand
// they go through LDS, 16 rows of kRow values (8 more than a row has, so that
// the 16 rows of a load start in different banks).
constexpr int kRow = kH + 8;
constexpr int kCols = kH / 16, kDeep = kH / 32;
typedef float Acts[kCols][4];

__device__ inline void load_operand(const uint16_t* rows, int r, int q, bf16x8 a[kDeep])
{
#pragma unroll
    for (int k = 0; k < kDeep; ++k) a[k] = *(const bf16x8*)(rows + r * kRow + 32 * k + 8 * q);
}

// columns 16 t .. 16 t + 15 of A times the packed second operand
__device__ inline float4_t tile_product(const bf16x8 a[kDeep], const uint16_t* __restrict__ w, int t, int lane)
{
    float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < kDeep; ++k)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[k], *(const bf16x8*)(w + ((t * kDeep + k) * 64 + lane) * 8), acc,
                                                      0, 0, 0);
    return acc;
}

// input layer: z = x W1^T + b1 for the lane's samples (zero past the last)
__device__ inline void layer_in(const float x[4][kIn], const bool live[4], const uint16_t* __restrict__ wb,
                                const float* __restrict__ p, int r, Acts z)
{
#pragma unroll
    for (int t = 0; t < kCols; ++t) {
        const int col = 16 * t + r;
        const ushort4_t w = *(const ushort4_t*)(wb + kPackW1 + col * kIn);
        const float bias = p[oB1 + col];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float v = bias;
#pragma unroll
            for (int k = 0; k < kIn; ++k) v += x[i][k] * from_bf16(w[k]);
            z[t][i] = live[i] ? v : 0.0f;
        }
    }
}

// Inference: 16 samples per wavefront and turn, the 128 x 128 weights of both
// layers in LDS (64 KB in operand order), nothing between x and y in memory.
// Bound by the GELUs (384 erf per sample; the matrix products take an eighth of
// the time).  1,000,003 samples: 0.31 ms; with a kernel per layer and the
// activations through memory 2.26 ms.  Non-finite inputs are reported in *bad.
constexpr int kInferWaves = 8;
__global__ void __launch_bounds__(64 * kInferWaves) k_infer(const float* __restrict__ x, int n,
                                                            const float* __restrict__ p,
                                                            const uint16_t* __restrict__ wb, float* __restrict__ y,
                                                            int* bad)
{
    __shared__ __align__(16) uint16_t w[2 * kTile];
    __shared__ __align__(16) uint16_t act[kInferWaves][16 * kRow];
    for (int i = threadIdx.x; i < 2 * kTile / 8; i += 64 * kInferWaves)
        ((uint4*)w)[i] = ((const uint4*)(wb + kF2))[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    uint16_t* rows = act[wave];
    const int tiles = (n + 15) / 16;
    for (int tile = blockIdx.x * kInferWaves + wave; tile < tiles; tile += gridDim.x * kInferWaves) {
        const int s0 = tile * 16;
        float xs[4][kIn];
        bool live[4];
        bool finite = true;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int s = s0 + 4 * q + i;
            live[i] = s < n;
            const float4 v = live[i] ? ((const float4*)x)[s] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            xs[i][0] = v.x;
            xs[i][1] = v.y;
            xs[i][2] = v.z;
            xs[i][3] = v.w;
            finite = finite && isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w);
        }
        if (!finite) *bad = 1;
        Acts z;
        layer_in(xs, live, wb, p, r, z);
#pragma unroll
        for (int layer = 0; layer < 2; ++layer) {
            wave_sync();
#pragma unroll
            for (int t = 0; t < kCols; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) rows[(4 * q + i) * kRow + 16 * t + r] = to_bf16(gelu(z[t][i]));
            wave_sync();
            bf16x8 a[kDeep];
            load_operand(rows, r, q, a);
#pragma unroll
            for (int t = 0; t < kCols; ++t) {
                const float bias = p[(layer ? oB3 : oB2) + 16 * t + r];
                const float4_t acc = tile_product(a, w + layer * kTile, t, lane);
#pragma unroll
                for (int i = 0; i < 4; ++i) z[t][i] = acc[i] + bias;
            }
        }
        float out[4][kOut] = {};
#pragma unroll
        for (int t = 0; t < kCols; ++t) {
            const float w0 = from_bf16(wb[kPackW4 + 16 * t + r]), w1 = from_bf16(wb[kPackW4 + kH + 16 * t + r]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float h = from_bf16(to_bf16(gelu(z[t][i])));
                out[i][0] += h * w0;
                out[i][1] += h * w1;
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int o = 0; o < kOut; ++o) {
                float v = out[i][o];
                for (int m = 1; m < 16; m <<= 1) v += __shfl_xor(v, m, 64);
                out[i][o] = v + p[oB4 + o];
            }
        if (r == 0)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (live[i]) ((float2*)y)[s0 + 4 * q + i] = make_float2(out[i][0], out[i][1]);
    }
}

// Forward and backward through the network for tiles of 64 samples, 16 per
// wavefront, and the block's share of the loss and of every gradient, written
// to row blockIdx.x of part (kP gradients, then the sum of squared errors).
//
// What crosses samples, the weight gradients dZ^T H, needs its operands sample
// by sample: activations and their gradients are therefore also kept in LDS
// column by column (kCol samples a column), where the four values that a lane
// holds of one column are neighbours.  After a tile the four wavefronts share
// the 64 tiles of each weight gradient, 16 apiece, which stay in registers over
// the block's tiles (one block per CU: 512 registers a lane).  The pre-
// activations stay in registers from the forward to the backward pass.
//
// Bound by the chain of GELUs and their derivatives that a wavefront evaluates
// (768 erf per sample), one wavefront per SIMD.  14,188 samples: 77 us, and 9 us
// for the sums and the Adam step; an epoch of the sixteen kernels this replaces
// took 4.6 ms, of which 3.9 ms were the sums over the samples by one thread per
// entry and 0.65 ms the loss by one thread.
constexpr int kTrainWaves = 4, kTrainTile = 16 * kTrainWaves;
constexpr int kCol = kTrainTile + 8;
constexpr int kPart = kP + 1;

// the lane's values of an activation, rounded, into rows and columns
__device__ inline void put_rows(uint16_t* rows, int r, int q, int t, const uint16_t h[4])
{
#pragma unroll
    for (int i = 0; i < 4; ++i) rows[(4 * q + i) * kRow + 16 * t + r] = h[i];
}
__device__ inline void put_column(uint16_t* cols, int wave, int r, int q, int t, const uint16_t h[4])
{
    *(ushort4_t*)(cols + (16 * t + r) * kCol + 16 * wave + 4 * q) = ushort4_t{h[0], h[1], h[2], h[3]};
}

// += the weight gradient dZ^T H of a block's tile, rows 32 wave .. 32 wave + 31
__device__ inline void add_weight_grad(const uint16_t* dz, const uint16_t* h, int wave, int r, int q,
                                       float4_t acc[2][kCols])
{
#pragma unroll
    for (int k = 0; k < kTrainTile / 32; ++k) {
        bf16x8 a[2];
#pragma unroll
        for (int o = 0; o < 2; ++o) a[o] = *(const bf16x8*)(dz + (32 * wave + 16 * o + r) * kCol + 32 * k + 8 * q);
#pragma unroll
        for (int t = 0; t < kCols; ++t) {
            const bf16x8 b = *(const bf16x8*)(h + (16 * t + r) * kCol + 32 * k + 8 * q);
#pragma unroll
            for (int o = 0; o < 2; ++o) acc[o][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[o], b, acc[o][t], 0, 0, 0);
        }
    }
}

__global__ void __launch_bounds__(64 * kTrainWaves, 1) k_train_tile(const float* __restrict__ x,
                                                                    const float* __restrict__ tgt, int n,
                                                                    const float* __restrict__ p,
                                                                    const uint16_t* __restrict__ packed,
                                                                    float* __restrict__ part)
{
    __shared__ __align__(16) uint16_t act[kTrainWaves][16 * kRow];
    __shared__ __align__(16) uint16_t h1[kH * kCol], h2[kH * kCol], e2[kH * kCol], e3[kH * kCol];
    // gradients that a wavefront sums over its own samples: W1, b1, b2, b3, W4,
    // b4, loss (a block's four rows of them are added in order at the end)
    constexpr int sW1 = 0, sB1 = sW1 + kH * kIn, sB2 = sB1 + kH, sB3 = sB2 + kH, sW4 = sB3 + kH, sB4 = sW4 + kOut * kH,
                  sLoss = sB4 + kOut, kSmall = sLoss + 1;
    __shared__ float small[kTrainWaves][kSmall];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    uint16_t* rows = act[wave];
    float4_t g2[2][kCols] = {}, g3[2][kCols] = {};
    float* mine = small[wave];
    for (int i = lane; i < kSmall; i += 64) mine[i] = 0.0f;
    // the sum of v over the four sample groups q, added to a small gradient
    auto add_small = [&](int at, float v) {
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        if (q == 0) mine[at] += v;
    };
    const float two_over_n = 2.0f / (float)n;
    const int tiles = (n + kTrainTile - 1) / kTrainTile;
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int s0 = tile * kTrainTile + 16 * wave;
        // (hidden from the compiler, which would load all the weights once, before
        // the loop, and spill them)
        const uint16_t* wb = packed;
        asm volatile("" : "+s"(wb));
        float xs[4][kIn];
        bool live[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int s = s0 + 4 * q + i;
            live[i] = s < n;
            const float4 v = live[i] ? ((const float4*)x)[s] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            xs[i][0] = v.x;
            xs[i][1] = v.y;
            xs[i][2] = v.z;
            xs[i][3] = v.w;
        }
        // forward
        Acts z1, z2, z3;
        uint16_t h[4];
        layer_in(xs, live, wb, p, r, z1);
        wave_sync();
#pragma unroll
        for (int t = 0; t < kCols; ++t) {
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = live[i] ? to_bf16(gelu(z1[t][i])) : (uint16_t)0;
            put_rows(rows, r, q, t, h);
            put_column(h1, wave, r, q, t, h);
        }
        wave_sync();
        bf16x8 a[kDeep];
        load_operand(rows, r, q, a);
        wave_sync();
#pragma unroll
        for (int t = 0; t < kCols; ++t) {
            const float bias = p[oB2 + 16 * t + r];
            const float4_t acc = tile_product(a, wb + kF2, t, lane);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                z2[t][i] = live[i] ? acc[i] + bias : 0.0f;
                h[i] = live[i] ? to_bf16(gelu(z2[t][i])) : (uint16_t)0;
            }
            put_rows(rows, r, q, t, h);
            put_column(h2, wave, r, q, t, h);
        }
        wave_sync();
        load_operand(rows, r, q, a);
        wave_sync();
        float out[4][kOut] = {};
        uint16_t h3[kCols][4];
#pragma unroll
        for (int t = 0; t < kCols; ++t) {
            const float bias = p[oB3 + 16 * t + r];
            const float4_t acc = tile_product(a, wb + kF3, t, lane);
            const float w0 = from_bf16(wb[kPackW4 + 16 * t + r]), w1 = from_bf16(wb[kPackW4 + kH + 16 * t + r]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                z3[t][i] = live[i] ? acc[i] + bias : 0.0f;
                h3[t][i] = live[i] ? to_bf16(gelu(z3[t][i])) : (uint16_t)0;
                out[i][0] += from_bf16(h3[t][i]) * w0;
                out[i][1] += from_bf16(h3[t][i]) * w1;
            }
        }
        // loss: dY = 2 (y - t) / n
        float dy[4][kOut], loss = 0.0f, gb4[kOut] = {};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int o = 0; o < kOut; ++o) {
                float v = out[i][o];
                for (int m = 1; m < 16; m <<= 1) v += __shfl_xor(v, m, 64);
                const float e = live[i] ? v + p[oB4 + o] - tgt[kOut * (s0 + 4 * q + i) + o] : 0.0f;
                dy[i][o] = e * two_over_n;
                gb4[o] += dy[i][o];
                loss += e * e;
            }
        // (the same in the 16 lanes of a group: lane 0 adds them)
        for (int m = 16; m < 64; m <<= 1) {
            gb4[0] += __shfl_xor(gb4[0], m, 64);
            gb4[1] += __shfl_xor(gb4[1], m, 64);
            loss += __shfl_xor(loss, m, 64);
        }
        if (lane == 0) {
            mine[sB4] += gb4[0];
            mine[sB4 + 1] += gb4[1];
            mine[sLoss] += loss;
        }
        // back through the output layer
#pragma unroll
        for (int t = 0; t < kCols; ++t) {
            const float w0 = from_bf16(wb[kPackW4 + 16 * t + r]), w1 = from_bf16(wb[kPackW4 + kH + 16 * t + r]);
            float gw0 = 0.0f, gw1 = 0.0f, gb = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float hv = from_bf16(h3[t][i]);
                gw0 += dy[i][0] * hv;
                gw1 += dy[i][1] * hv;
                const float dz = (dy[i][0] * w0 + dy[i][1] * w1) * gelu_grad(z3[t][i]);
                gb += dz;
                h[i] = to_bf16(dz);
            }
            add_small(sW4 + 16 * t + r, gw0);
            add_small(sW4 + kH + 16 * t + r, gw1);
            add_small(sB3 + 16 * t + r, gb);
            put_rows(rows, r, q, t, h);
            put_column(e3, wave, r, q, t, h);
        }
        // dZ2 = (dZ3 W3) * gelu'(Z2), dZ1 = (dZ2 W2) * gelu'(Z1)
        wave_sync();
        load_operand(rows, r, q, a);
        wave_sync();
#pragma unroll
        for (int t = 0; t < kCols; ++t) {
            const float4_t acc = tile_product(a, wb + kT3, t, lane);
            float gb = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float dz = acc[i] * gelu_grad(z2[t][i]);
                gb += dz;
                h[i] = to_bf16(dz);
            }
            add_small(sB2 + 16 * t + r, gb);
            put_rows(rows, r, q, t, h);
            put_column(e2, wave, r, q, t, h);
        }
        wave_sync();
        load_operand(rows, r, q, a);
#pragma unroll
        for (int t = 0; t < kCols; ++t) {
            const float4_t acc = tile_product(a, wb + kT2, t, lane);
            float gb = 0.0f, gw[kIn] = {};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float dz = acc[i] * gelu_grad(z1[t][i]);
                gb += dz;
#pragma unroll
                for (int k = 0; k < kIn; ++k) gw[k] += dz * xs[i][k];
            }
            add_small(sB1 + 16 * t + r, gb);
#pragma unroll
            for (int k = 0; k < kIn; ++k) add_small(sW1 + (16 * t + r) * kIn + k, gw[k]);
        }
        __syncthreads();
        add_weight_grad(e3, h2, wave, r, q, g3);
        add_weight_grad(e2, h1, wave, r, q, g2);
        __syncthreads();
    }
    float* row = part + (size_t)blockIdx.x * kPart;
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
        for (int t = 0; t < kCols; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int at = (32 * wave + 16 * o + 4 * q + i) * kH + 16 * t + r;
                row[oW2 + at] = g2[o][t][i];
                row[oW3 + at] = g3[o][t][i];
            }
    // the wavefronts' small gradients in order
    __syncthreads();
    for (int i = threadIdx.x; i < kSmall; i += 64 * kTrainWaves) {
        float v = small[0][i];
#pragma unroll
        for (int w = 1; w < kTrainWaves; ++w) v += small[w][i];
        const int at = i < sB1   ? oW1 + i - sW1
                       : i < sB2 ? oB1 + i - sB1
                       : i < sB3 ? oB2 + i - sB2
                       : i < sW4 ? oB3 + i - sB3
                       : i < sB4 ? oW4 + i - sW4
                                 : oB4 + i - sB4;
        row[at] = v;
    }
}

// The blocks' gradients summed (four quarters of the rows, each in order, then
// in order) into g and the mean squared error into loss; with lr > 0 the Adam
// step and the packed weights of the next pass as well.
constexpr int kSumWays = 4;
__global__ void __launch_bounds__(kBlock) k_sum_and_step(const float* __restrict__ part, int rows, int n,
                                                         float* __restrict__ g, float* __restrict__ loss,
                                                         float* __restrict__ p, float* __restrict__ m,
                                                         float* __restrict__ v, uint16_t* __restrict__ wb, float lr,
                                                         float c1, float c2)
{
    __shared__ float red[kSumWays][kBlock / kSumWays];
    const int way = threadIdx.x / (kBlock / kSumWays), at = threadIdx.x % (kBlock / kSumWays);
    const int i = blockIdx.x * (kBlock / kSumWays) + at;
    const int per = (rows + kSumWays - 1) / kSumWays;
    const int r0 = way * per, r1 = min(rows, r0 + per);
    float s = 0.0f;
    if (i < kPart)
#pragma unroll 8
        for (int r = r0; r < r1; ++r) s += part[(size_t)r * kPart + i];
    red[way][at] = s;
    __syncthreads();
    if (way != 0 || i >= kPart) return;
#pragma unroll
    for (int w = 1; w < kSumWays; ++w) s += red[w][at];
    if (i == kP) {
        loss[0] = s / (float)n;
        return;
    }
    g[i] = s;
    if (!(lr > 0.0f)) return;
    m[i] = 0.9f * m[i] + 0.1f * s;
    v[i] = 0.999f * v[i] + 0.001f * s * s;
    const float q = p[i] - lr * (m[i] / c1) / (sqrtf(v[i] / c2) + 1e-8f);
    p[i] = q;
    pack_param(wb, i, q);
}

inline unsigned blocks(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

}  // namespace

struct dem_closure {
    int device = 0;
    hipStream_t stream = nullptr;
    float *p = nullptr, *m = nullptr, *v = nullptr, *g = nullptr;
    uint16_t* wb = nullptr;
    int64_t step = 0;
    // sample buffers, grown on demand
    int64_t cap = 0;
    float *x = nullptr, *t = nullptr, *y = nullptr;
    // the training blocks' gradients, and the loss
    int64_t part_rows = 0;
    float *part = nullptr, *loss = nullptr;
    // pinned host memory that the kernels read and write directly: the inputs
    // and outputs of a small forward call, and the non-finite flag
    float *hx = nullptr, *hy = nullptr;
    int* bad = nullptr;
};

namespace {

#define CCHK(expr)                                  \
    do {                                            \
        if ((expr) != hipSuccess) return DEM_ERR_DEVICE; \
    } while (0)

// forward calls of up to this many samples go through pinned memory: two
// copies of a few KB each cost more than the kernel
constexpr int64_t kSmallCall = 2048;
constexpr int kMaxTrainBlocks = 256;  // one per CU

void free_samples(dem_closure* c)
{
    for (void* a : {(void*)c->x, (void*)c->t, (void*)c->y})
        if (a) (void)hipFree(a);
    c->x = c->t = c->y = nullptr;
    c->cap = 0;
}

int ensure(dem_closure* c, int64_t n)
{
    if (n <= c->cap) return DEM_OK;
    CCHK(hipStreamSynchronize(c->stream));
    free_samples(c);
    CCHK(hipMalloc(&c->x, sizeof(float) * kIn * n));
    CCHK(hipMalloc(&c->t, sizeof(float) * kOut * n));
    CCHK(hipMalloc(&c->y, sizeof(float) * kOut * n));
    c->cap = n;
    return DEM_OK;
}

int train_blocks(int64_t n)
{
    const int64_t tiles = (n + kTrainTile - 1) / kTrainTile;
    return (int)(tiles < kMaxTrainBlocks ? tiles : kMaxTrainBlocks);
}

int ensure_part(dem_closure* c, int64_t n)
{
    const int64_t rows = train_blocks(n);
    if (rows <= c->part_rows) return DEM_OK;
    CCHK(hipStreamSynchronize(c->stream));
    if (c->part) (void)hipFree(c->part);
    c->part = nullptr;
    c->part_rows = 0;
    CCHK(hipMalloc(&c->part, sizeof(float) * kPart * rows));
    c->part_rows = rows;
    return DEM_OK;
}

// the packed weights follow the parameters: after set_params here, after an
// Adam step in k_sum_and_step
void pack(dem_closure* c)
{
    hipLaunchKernelGGL(k_pack, dim3(blocks(kP)), dim3(kBlock), 0, c->stream, c->p, c->wb);
}

void forward(dem_closure* c, int n, const float* x, float* y)
{
    const int tiles = (n + 16 * kInferWaves - 1) / (16 * kInferWaves);
    hipLaunchKernelGGL(k_infer, dim3(tiles < 256 ? tiles : 256), dim3(64 * kInferWaves), 0, c->stream, x, n, c->p, c->wb,
                       y, c->bad);
}

// loss and gradient (into c->g) of the samples in c->x / c->t; lr > 0: and the
// Adam step
void backward(dem_closure* c, int n, float lr, float c1, float c2)
{
    const int rows = train_blocks(n);
    hipLaunchKernelGGL(k_train_tile, dim3(rows), dim3(64 * kTrainWaves), 0, c->stream, c->x, c->t, n, c->p, c->wb,
                       c->part);
    hipLaunchKernelGGL(k_sum_and_step, dim3((kPart + kBlock / kSumWays - 1) / (kBlock / kSumWays)), dim3(kBlock), 0,
                       c->stream, c->part, rows, n, c->g, c->loss, c->p, c->m, c->v, c->wb, lr, c1, c2);
}

int upload(dem_closure* c, int64_t n, const float* x, const float* t)
{
    if (ensure(c, n)) return DEM_ERR_DEVICE;
    CCHK(hipMemcpyAsync(c->x, x, sizeof(float) * kIn * n, hipMemcpyHostToDevice, c->stream));
    if (t) CCHK(hipMemcpyAsync(c->t, t, sizeof(float) * kOut * n, hipMemcpyHostToDevice, c->stream));
    return DEM_OK;
}

bool finite(const float* a, int64_t n)
{
    for (int64_t i = 0; i < n; ++i)
        if (!std::isfinite(a[i])) return false;
    return true;
}

}  // namespace

extern "C" {

int dem_closure_create(dem_closure** out, int32_t device)
{
    if (!out) return DEM_ERR_ARG;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) return DEM_ERR_ARG;
    dem_closure* c = new dem_closure();
    c->device = device;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
        hipMalloc(&c->p, sizeof(float) * kP) != hipSuccess || hipMalloc(&c->m, sizeof(float) * kP) != hipSuccess ||
        hipMalloc(&c->v, sizeof(float) * kP) != hipSuccess || hipMalloc(&c->g, sizeof(float) * kP) != hipSuccess ||
        hipMalloc(&c->wb, sizeof(uint16_t) * kPacked) != hipSuccess ||
        hipMemset(c->wb, 0, sizeof(uint16_t) * kPacked) != hipSuccess || hipMalloc(&c->loss, sizeof(float)) != hipSuccess ||
        hipHostMalloc((void**)&c->hx, sizeof(float) * (kIn + kOut) * kSmallCall + 64,
                      hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess || hipMemset(c->p, 0, sizeof(float) * kP) != hipSuccess ||
        hipMemset(c->m, 0, sizeof(float) * kP) != hipSuccess || hipMemset(c->v, 0, sizeof(float) * kP) != hipSuccess) {
        dem_closure_destroy(c);
        return DEM_ERR_DEVICE;
    }
    c->hy = c->hx + kIn * kSmallCall;
    c->bad = (int*)(c->hy + kOut * kSmallCall);
    *c->bad = 0;
    *out = c;
    return DEM_OK;
}

int dem_closure_destroy(dem_closure* c)
{
    if (!c) return DEM_OK;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    free_samples(c);
    for (void* a : {(void*)c->p, (void*)c->m, (void*)c->v, (void*)c->g, (void*)c->wb, (void*)c->part, (void*)c->loss})
        if (a) (void)hipFree(a);
    if (c->hx) (void)hipHostFree(c->hx);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return DEM_OK;
}

int dem_closure_set_params(dem_closure* c, const float* params)
{
    if (!c || !params || !finite(params, kP)) return DEM_ERR_ARG;
    CCHK(hipSetDevice(c->device));
    CCHK(hipMemcpyAsync(c->p, params, sizeof(float) * kP, hipMemcpyHostToDevice, c->stream));
    CCHK(hipMemsetAsync(c->m, 0, sizeof(float) * kP, c->stream));
    CCHK(hipMemsetAsync(c->v, 0, sizeof(float) * kP, c->stream));
    pack(c);
    CCHK(hipGetLastError());
    CCHK(hipStreamSynchronize(c->stream));
    c->step = 0;
    return DEM_OK;
}

int dem_closure_get_params(dem_closure* c, float* params)
{
    if (!c || !params) return DEM_ERR_ARG;
    CCHK(hipSetDevice(c->device));
    CCHK(hipMemcpyAsync(params, c->p, sizeof(float) * kP, hipMemcpyDeviceToHost, c->stream));
    CCHK(hipStreamSynchronize(c->stream));
    return DEM_OK;
}

int dem_closure_forward(dem_closure* c, int64_t n, const float* x, float* y)
{
    if (!c || n < 0 || n > (1 << 24) || (n > 0 && (!x || !y))) return DEM_ERR_ARG;
    if (n == 0) return DEM_OK;
    CCHK(hipSetDevice(c->device));
    const bool small = n <= kSmallCall;
    if (small) {
        std::memcpy(c->hx, x, sizeof(float) * kIn * n);
    } else {
        const int r = upload(c, n, x, nullptr);
        if (r) return r;
    }
    *c->bad = 0;
    forward(c, (int)n, small ? c->hx : c->x, small ? c->hy : c->y);
    CCHK(hipGetLastError());
    CCHK(hipStreamSynchronize(c->stream));
    if (__atomic_load_n(c->bad, __ATOMIC_ACQUIRE)) return DEM_ERR_ARG;  // an input is not finite
    if (small)
        std::memcpy(y, c->hy, sizeof(float) * kOut * n);
    else
        CCHK(hipMemcpy(y, c->y, sizeof(float) * kOut * n, hipMemcpyDeviceToHost));
    return DEM_OK;
}

int dem_closure_gradient(dem_closure* c, int64_t n, const float* x, const float* target, float* grad, float* loss)
{
    if (!c || n <= 0 || n > (1 << 24) || !x || !target) return DEM_ERR_ARG;
    if (!finite(x, kIn * n) || !finite(target, kOut * n)) return DEM_ERR_ARG;
    CCHK(hipSetDevice(c->device));
    int r = ensure_part(c, n);
    if (!r) r = upload(c, n, x, target);
    if (r) return r;
    backward(c, (int)n, 0.0f, 1.0f, 1.0f);
    CCHK(hipGetLastError());
    if (grad) CCHK(hipMemcpyAsync(grad, c->g, sizeof(float) * kP, hipMemcpyDeviceToHost, c->stream));
    if (loss) CCHK(hipMemcpyAsync(loss, c->loss, sizeof(float), hipMemcpyDeviceToHost, c->stream));
    CCHK(hipStreamSynchronize(c->stream));
    return DEM_OK;
}

int dem_closure_train(dem_closure* c, int64_t n, const float* x, const float* target, int32_t epochs, float lr,
                      float* loss)
{
    if (!c || n <= 0 || n > (1 << 24) || !x || !target || epochs < 0 || !(lr > 0) || !std::isfinite(lr))
        return DEM_ERR_ARG;
    if (!finite(x, kIn * n) || !finite(target, kOut * n)) return DEM_ERR_ARG;
    CCHK(hipSetDevice(c->device));
    int r = ensure_part(c, n);
    if (!r) r = upload(c, n, x, target);
    if (r) return r;
    for (int e = 0; e < epochs; ++e) {
        ++c->step;
        const float c1 = 1.0f - std::pow(0.9f, (float)c->step), c2 = 1.0f - std::pow(0.999f, (float)c->step);
        backward(c, (int)n, lr, c1, c2);
    }
    if (epochs == 0 && loss) backward(c, (int)n, 0.0f, 1.0f, 1.0f);
    CCHK(hipGetLastError());
    if (loss) CCHK(hipMemcpyAsync(loss, c->loss, sizeof(float), hipMemcpyDeviceToHost, c->stream));
    CCHK(hipStreamSynchronize(c->stream));
    return DEM_OK;
}

}  // extern "C"
