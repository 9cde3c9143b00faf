// Learned troubled-cell indicator (gfx950): a 4 -> 64 -> 64 -> 64 -> 1
// perceptron with GELU hidden layers and a sigmoid output that predicts the
// DG/FV blending factor alpha of an element from the log modal energy
// fractions of rho and p in the top one and top two mode shells.
//
// The reference has no learned indicator (its blending traces are in
// setups/mhd/3d/_common_/setup_checkpoint_mod.f90:395-450); this is the
// library's own network, trained on (features, alpha) pairs that the
// Persson-Peraire indicator produces during the method's own runs.
//
// Parameter vector (FP32, canonical layout, NPARAMS = 8705):
//   W1[64][4], b1[64], W2[64][64], b2[64], W3[64][64], b3[64], w4[64], b4
// with W[j][k] the weight from input k to unit j.  The inference layout
// used by the stage kernel stores W2 and W3 in blocks of four inputs,
// W[j][4b..4b+3] at 4 (64 b + j): lane j reads its unit's four weights as one
// 16-byte load and a wavefront reads 1 KB contiguous per block (16 loads per
// layer instead of 64).
//
// Inside the stage kernel one hidden unit is one lane of a 64-lane wavefront;
// an activation of another unit is read with v_readlane (uniform index).  The
// batch kernels (training, outputs of many samples) run on the matrix cores.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nemo {

constexpr int MLP_IN = 4, MLP_H = 64;
constexpr int MLP_W1 = 0, MLP_B1 = MLP_W1 + MLP_H * MLP_IN, MLP_W2 = MLP_B1 + MLP_H, MLP_B2 = MLP_W2 + MLP_H * MLP_H,
              MLP_W3 = MLP_B2 + MLP_H, MLP_B3 = MLP_W3 + MLP_H * MLP_H, MLP_W4 = MLP_B3 + MLP_H,
              MLP_B4 = MLP_W4 + MLP_H, MLP_NP = MLP_B4 + 1;
static_assert(MLP_NP == 8705, "parameter count");

// Feature of a modal energy fraction f in [0, 1]: 0.1 ln(f + 1e-12).
__device__ __forceinline__ float mlp_feature(float f) { return 0.1f * __logf(f + 1.0e-12f); }

// GELU in its tanh form, 0.5 x (1 + tanh(c (x + 0.044715 x^3))),
// c = sqrt(2/pi) (Hendrycks & Gimpel 2016).
// tanh(y) = 1 - 2/(exp(2y) + 1).
__device__ __forceinline__ float gelu_t(float x) {
    const float y = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    return 1.0f - 2.0f / (__expf(2.0f * y) + 1.0f);
}
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + gelu_t(x)); }
__device__ __forceinline__ float sigmoid(float z) { return 1.0f / (1.0f + __expf(-z)); }

__device__ __forceinline__ float lane_bcast(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Wave-wide sum (64 lanes) by butterfly shuffles.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// Forward pass for NB samples held uniformly by the wavefront (feat[s][k] is
// the same in every lane), with the inference-layout parameters P.  Lane j
// computes unit j of every hidden layer; y[s] (uniform) is the sigmoid output.
template <int NB>
__device__ __forceinline__ void mlp_forward_wave(const float* __restrict__ P, const float (&feat)[NB][MLP_IN],
                                                 float (&y)[NB]) {
    const int j = threadIdx.x & 63;
    float a1[NB], a2[NB], a3[NB];
    {
        const float w0 = P[MLP_W1 + j * 4 + 0], w1 = P[MLP_W1 + j * 4 + 1], w2 = P[MLP_W1 + j * 4 + 2],
                    w3 = P[MLP_W1 + j * 4 + 3], b = P[MLP_B1 + j];
#pragma unroll
        for (int s = 0; s < NB; ++s)
            a1[s] = gelu(b + w0 * feat[s][0] + w1 * feat[s][1] + w2 * feat[s][2] + w3 * feat[s][3]);
    }
    {
        float z[NB];
        const float b = P[MLP_B2 + j];
#pragma unroll
        for (int s = 0; s < NB; ++s) z[s] = b;
        for (int kb = 0; kb < MLP_H / 4; ++kb) {
            const float4 w = *reinterpret_cast<const float4*>(P + MLP_W2 + kb * 4 * MLP_H + j * 4);
#pragma unroll
            for (int s = 0; s < NB; ++s) {
                z[s] += w.x * lane_bcast(a1[s], 4 * kb);
                z[s] += w.y * lane_bcast(a1[s], 4 * kb + 1);
                z[s] += w.z * lane_bcast(a1[s], 4 * kb + 2);
                z[s] += w.w * lane_bcast(a1[s], 4 * kb + 3);
            }
        }
#pragma unroll
        for (int s = 0; s < NB; ++s) a2[s] = gelu(z[s]);
    }
    {
        float z[NB];
        const float b = P[MLP_B3 + j];
#pragma unroll
        for (int s = 0; s < NB; ++s) z[s] = b;
        for (int kb = 0; kb < MLP_H / 4; ++kb) {
            const float4 w = *reinterpret_cast<const float4*>(P + MLP_W3 + kb * 4 * MLP_H + j * 4);
#pragma unroll
            for (int s = 0; s < NB; ++s) {
                z[s] += w.x * lane_bcast(a2[s], 4 * kb);
                z[s] += w.y * lane_bcast(a2[s], 4 * kb + 1);
                z[s] += w.z * lane_bcast(a2[s], 4 * kb + 2);
                z[s] += w.w * lane_bcast(a2[s], 4 * kb + 3);
            }
        }
#pragma unroll
        for (int s = 0; s < NB; ++s) a3[s] = gelu(z[s]);
    }
    const float w4 = P[MLP_W4 + j], b4 = P[MLP_B4];
#pragma unroll
    for (int s = 0; s < NB; ++s) y[s] = sigmoid(b4 + wave_sum(w4 * a3[s]));
}

// ---------------------------------------------------------------------------
// Batch kernels (canonical layout): the layers as matrix products over tiles
// of 16 samples, on the FP32 matrix cores
// ---------------------------------------------------------------------------
//
// A workgroup of four wavefronts takes a tile of 16 samples; wavefront w owns
// units 16w .. 16w+15 of every hidden layer.  v_mfma_f32_16x16x4_f32 forms a
// 16 x 16 block from four terms of the sum: lane l gives A[l % 16][l / 16] and
// B[l / 16][l % 16] and holds D[4 (l / 16) + r][l % 16], r = 0..3 (samples by
// units, so the activations stay in the lane that computed them).  The order
// of the terms is free as long as A and B agree: step b takes term
// 16 (l / 16) + b, so that a lane's sixteen activations (or weights of a
// unit) are consecutive.  The weights stay in registers over all tiles of a
// workgroup; activations and deltas change hands through LDS.
//
// What bounds them: the chain of layers of one tile (gradient: about 100 matrix
// instructions a wavefront and seven barriers; outputs: 33 and four); the
// arithmetic of 4096 samples is 2 us at the FP32 matrix rate.  One sample at a
// time per wavefront, with the other units' activations by v_readlane, took
// 98 us for the gradient of 4096 samples and 74 us for the outputs of 100 000.
constexpr int MLP_TILE = 16;   // samples of a tile
constexpr int MLP_NT = 256;    // four wavefronts
constexpr int MLP_LD = 68;     // row of an LDS tile: 16-byte aligned, rows four banks apart
constexpr int MLP_PARTS = 256; // most gradient partials: one workgroup per CU

using mlp_f4 = float __attribute__((ext_vector_type(4)));

// Sixteen consecutive floats (16-byte aligned) of LDS or of a weight row.
__device__ __forceinline__ void load16(const float* p, float (&v)[16]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const mlp_f4 x = *reinterpret_cast<const mlp_f4*>(p + 4 * q);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[4 * q + r] = x[r];
    }
}

// c += the product of a 16 x 64 tile held in LDS with the lane's weights.
__device__ __forceinline__ mlp_f4 tile_mfma(const float* row, const float (&w)[16], mlp_f4 c) {
    float a[16];
    load16(row, a);
#pragma unroll
    for (int b = 0; b < 16; ++b) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[b], w[b], c, 0, 0, 0);
    return c;
}

// Sum over the 16 lanes of a row group (l % 16).
__device__ __forceinline__ float row_sum(float v) {
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// LDS tiles of a workgroup.
struct MlpTile {
    float (*act)[MLP_TILE * MLP_LD];  // activations of the first two layers, samples by units
    float* feat;                      // [16][4]
    float (*zsum)[MLP_TILE];          // [4 wavefronts][16 samples] parts of the output sum
};

// Forward weights of a lane.
struct MlpLane {
    float w1, b1, b2, b3, w4, b4;  // of unit 16 w + l % 16; w1 from input l / 16
    float w2[16], w3[16];          // inputs 16 (l / 16) .. + 15
};

__device__ __forceinline__ void mlp_lane_load(const float* __restrict__ P, MlpLane& n) {
    const int l = threadIdx.x & 63, unit = 16 * (threadIdx.x >> 6) + (l & 15), kg = l >> 4;
    n.w1 = P[MLP_W1 + unit * MLP_IN + kg];
    n.b1 = P[MLP_B1 + unit];
    n.b2 = P[MLP_B2 + unit];
    n.b3 = P[MLP_B3 + unit];
    n.w4 = P[MLP_W4 + unit];
    n.b4 = P[MLP_B4];
    load16(P + MLP_W2 + unit * MLP_H + 16 * kg, n.w2);
    load16(P + MLP_W3 + unit * MLP_H + 16 * kg, n.w3);
}

// Forward pass of the tile in feat; z the arguments and t the tanh of the
// GELUs of the three layers (for the backward pass), a3 the last activations,
// z4 the output's argument of the lane's samples.  Three barriers: feat must
// be complete before; feat and act[0] may be written again once the last one
// is passed, act[1] and zsum after a further one.
__device__ __forceinline__ void mlp_tile_forward(const MlpLane& n, const MlpTile& T, mlp_f4 (&z)[3], mlp_f4 (&t)[3],
                                                 mlp_f4& a3, float (&z4)[4]) {
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, unit = 16 * w + (l & 15), g = l >> 4;
    auto bias = [](float b) { return mlp_f4{b, b, b, b}; };
    auto activate = [&](int layer, float* out) {
        mlp_f4 a;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            t[layer][r] = gelu_t(z[layer][r]);
            a[r] = 0.5f * z[layer][r] * (1.0f + t[layer][r]);
            if (out) out[(4 * g + r) * MLP_LD + unit] = a[r];
        }
        return a;
    };
    z[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(T.feat[(l & 15) * MLP_IN + g], n.w1, bias(n.b1), 0, 0, 0);
    activate(0, T.act[0]);
    __syncthreads();
    const int row = (l & 15) * MLP_LD + 16 * g;
    z[1] = tile_mfma(T.act[0] + row, n.w2, bias(n.b2));
    activate(1, T.act[1]);
    __syncthreads();
    z[2] = tile_mfma(T.act[1] + row, n.w3, bias(n.b3));
    a3 = activate(2, nullptr);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float s = row_sum(n.w4 * a3[r]);
        if ((l & 15) == 0) T.zsum[w][4 * g + r] = s;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int s = 4 * g + r;
        z4[r] = n.b4 + ((T.zsum[0][s] + T.zsum[1][s]) + (T.zsum[2][s] + T.zsum[3][s]));
    }
}

// Outputs of n samples for the host API.
static __global__ __launch_bounds__(MLP_NT) void mlp_forward_kernel(const float* __restrict__ P, long long n,
                                                                    const float* __restrict__ feat,
                                                                    float* __restrict__ out) {
    __shared__ __align__(16) float act[2][MLP_TILE * MLP_LD];
    __shared__ float sfeat[MLP_TILE * MLP_IN], zsum[4][MLP_TILE];
    const MlpTile T{act, sfeat, zsum};
    const int tid = threadIdx.x, l = tid & 63;
    MlpLane net;
    mlp_lane_load(P, net);
    const long long tiles = (n + MLP_TILE - 1) / MLP_TILE;
    for (long long k = blockIdx.x; k < tiles; k += gridDim.x) {
        const long long i0 = k * MLP_TILE;
        if (tid < MLP_TILE * MLP_IN) sfeat[tid] = i0 * MLP_IN + tid < n * MLP_IN ? feat[i0 * MLP_IN + tid] : 0.0f;
        __syncthreads();
        mlp_f4 z[3], t[3], a3;
        float z4[4];
        mlp_tile_forward(net, T, z, t, a3, z4);
        if (tid < 64 && (l & 15) == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const long long i = i0 + 4 * (l >> 4) + r;
                if (i < n) out[i] = sigmoid(z4[r]);
            }
        }
        // the next tile's first writes (feat, act[0]) come before its first
        // barrier; every wavefront has read both before the pass's last one
    }
}

// Loss and gradient of L = 1/(2B) sum_s (y_s - t_s)^2 over one minibatch
// (sample ids idx[off .. off+B), or off .. off+B when idx is null).  Block b
// takes the tiles b, b + gridDim.x, ... and writes its partial gradient
// (canonical layout) to part[b][NP] and its partial loss to part_loss[b];
// mlp_reduce_kernel sums the partials in a fixed order (deterministic).
static __global__ __launch_bounds__(MLP_NT) void mlp_grad_kernel(const float* __restrict__ P,
                                                                 const float* __restrict__ feat,
                                                                 const float* __restrict__ target,
                                                                 const long long* __restrict__ idx, long long off,
                                                                 int B, float* __restrict__ part,
                                                                 float* __restrict__ part_loss) {
    __shared__ __align__(16) float act[2][MLP_TILE * MLP_LD], del[2][MLP_TILE * MLP_LD];
    __shared__ float sfeat[MLP_TILE * MLP_IN], starget[MLP_TILE], zsum[4][MLP_TILE];
    const MlpTile T{act, sfeat, zsum};
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, c = l & 15, g = l >> 4, unit = 16 * w + c;
    MlpLane net;
    mlp_lane_load(P, net);
    // weights of the backward products: column `unit`, rows 16 g + b
    float w2t[16], w3t[16];
#pragma unroll
    for (int b = 0; b < 16; ++b) {
        w2t[b] = P[MLP_W2 + (16 * g + b) * MLP_H + unit];
        w3t[b] = P[MLP_W3 + (16 * g + b) * MLP_H + unit];
    }
    mlp_f4 gW2[4] = {}, gW3[4] = {};  // rows 16 w + 4 g + r, columns 16 q + c
    float gW1[4] = {0, 0, 0, 0}, gb1 = 0, gb2 = 0, gb3 = 0, gw4 = 0, gb4 = 0, loss = 0;
    const float invB = 1.0f / float(B);
    auto gelu_slope = [](float x, float t) {
        const float dy = 0.7978845608028654f * (1.0f + 3.0f * 0.044715f * x * x);
        return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * dy;
    };
    // g += sum_s d[s][16 w + i] a[s][16 q + j] over the tile's samples
    auto outer = [&](const float* d, const float* a, mlp_f4 (&acc)[4]) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int s = (4 * g + b) * MLP_LD;
            const float dv = d[s + unit];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                acc[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(dv, a[s + 16 * q + c], acc[q], 0, 0, 0);
        }
    };
    const int row = c * MLP_LD + 16 * g;
    const int tiles = (B + MLP_TILE - 1) / MLP_TILE;
    for (int k = blockIdx.x; k < tiles; k += gridDim.x) {
        const int s0 = k * MLP_TILE;
        __syncthreads();  // the last tile's gradients have read the LDS tiles
        if (tid < MLP_TILE * MLP_IN) {
            const int s = s0 + tid / MLP_IN;
            float x = 0.0f;
            if (s < B) {
                const long long i = idx ? idx[off + s] : off + s;
                x = feat[i * MLP_IN + tid % MLP_IN];
                if (tid % MLP_IN == 0) starget[tid / MLP_IN] = target[i];
            }
            sfeat[tid] = x;
        }
        __syncthreads();
        mlp_f4 z[3], t[3], a3, d;
        float z4[4];
        mlp_tile_forward(net, T, z, t, a3, z4);
        // output layer and third layer
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int s = 4 * g + r;
            const float y = sigmoid(z4[r]);
            const float res = s0 + s < B ? y - starget[s] : 0.0f;  // no share beyond the batch
            loss += 0.5f * res * res * invB;
            const float d4 = res * y * (1.0f - y) * invB;
            gb4 += d4;
            gw4 += d4 * a3[r];
            d[r] = d4 * net.w4 * gelu_slope(z[2][r], t[2][r]);
            gb3 += d[r];
            del[0][s * MLP_LD + unit] = d[r];
        }
        __syncthreads();
        d = tile_mfma(del[0] + row, w3t, mlp_f4{0, 0, 0, 0});
        outer(del[0], act[1], gW3);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            d[r] *= gelu_slope(z[1][r], t[1][r]);
            gb2 += d[r];
            del[1][(4 * g + r) * MLP_LD + unit] = d[r];
        }
        __syncthreads();
        d = tile_mfma(del[1] + row, w2t, mlp_f4{0, 0, 0, 0});
        outer(del[1], act[0], gW2);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            d[r] *= gelu_slope(z[0][r], t[0][r]);
            gb1 += d[r];
#pragma unroll
            for (int q = 0; q < MLP_IN; ++q) gW1[q] += d[r] * sfeat[(4 * g + r) * MLP_IN + q];
        }
    }
    // sums over the four sample groups (lanes of equal c)
    auto groups = [](float v) {
        v += __shfl_xor(v, 16);
        return v + __shfl_xor(v, 32);
    };
    float* out = part + (long long)blockIdx.x * MLP_NP;
#pragma unroll
    for (int q = 0; q < MLP_IN; ++q) {
        const float v = groups(gW1[q]);
        if (g == 0) out[MLP_W1 + unit * MLP_IN + q] = v;
    }
    const float v1 = groups(gb1), v2 = groups(gb2), v3 = groups(gb3), v4 = groups(gw4), vb = groups(gb4),
                vl = groups(loss);
    if (g == 0) {
        out[MLP_B1 + unit] = v1;
        out[MLP_B2 + unit] = v2;
        out[MLP_B3 + unit] = v3;
        out[MLP_W4 + unit] = v4;
    }
    if (tid == 0) {
        out[MLP_B4] = vb;
        part_loss[blockIdx.x] = vl;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int at = (16 * w + 4 * g + r) * MLP_H + 16 * q + c;
            out[MLP_W2 + at] = gW2[q][r];
            out[MLP_W3 + at] = gW3[q][r];
        }
}

// Sum of the per-block partial gradients in a fixed order (deterministic), in
// FP64; with adam != 0 also one Adam step (Kingma & Ba 2015) on P (canonical)
// with moments m, v and bias corrections c1 = 1 - beta1^t, c2 = 1 - beta2^t.
// A workgroup owns 64 parameters; its 16 wavefronts sum every sixteenth
// partial each (256 consecutive bytes per load, all independent), then one
// adds the 16 sums.  Bound by the latency of those loads: one thread per
// parameter that walked 128 partials in turn took 37 us.
constexpr int MLP_RW = 16;
static __global__ __launch_bounds__(64 * MLP_RW) void mlp_reduce_kernel(
    const float* __restrict__ part, int nparts, const float* __restrict__ part_loss, float* __restrict__ grad,
    float* __restrict__ loss, float* __restrict__ P, float* __restrict__ m, float* __restrict__ v, int adam, float lr,
    float c1, float c2) {
    __shared__ double sum[MLP_RW][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane;
    double s = 0.0;
    if (p < MLP_NP) {
#pragma unroll 8
        for (int b = w; b < nparts; b += MLP_RW) s += double(part[(long long)b * MLP_NP + p]);
    }
    sum[w][lane] = s;
    __syncthreads();
    if (w == 1 && blockIdx.x == 0 && loss) {
        double x = 0.0;
        for (int b = lane; b < nparts; b += 64) x += double(part_loss[b]);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
        if (lane == 0) *loss += float(x);
    }
    if (w != 0 || p >= MLP_NP) return;
    s = 0.0;
#pragma unroll
    for (int b = 0; b < MLP_RW; ++b) s += sum[b][lane];
    const float gsum = float(s);
    if (grad) grad[p] = gsum;
    if (adam) {
        const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
        const float mm = beta1 * m[p] + (1.0f - beta1) * gsum;
        const float vv = beta2 * v[p] + (1.0f - beta2) * gsum * gsum;
        m[p] = mm;
        v[p] = vv;
        P[p] -= lr * (mm / c1) / (sqrtf(vv / c2) + eps);
    }
}

// Canonical -> inference layout (W2 and W3 in blocks of four inputs).
static __global__ void mlp_inference_layout_kernel(const float* __restrict__ P, float* __restrict__ Q) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= MLP_NP) return;
    if (p >= MLP_W2 && p < MLP_B2) {
        const int r = (p - MLP_W2) / MLP_H, c = (p - MLP_W2) % MLP_H;
        Q[MLP_W2 + (c >> 2) * 4 * MLP_H + r * 4 + (c & 3)] = P[p];
    } else if (p >= MLP_W3 && p < MLP_B3) {
        const int r = (p - MLP_W3) / MLP_H, c = (p - MLP_W3) % MLP_H;
        Q[MLP_W3 + (c >> 2) * 4 * MLP_H + r * 4 + (c & 3)] = P[p];
    } else {
        Q[p] = P[p];
    }
}

}  // namespace nemo
