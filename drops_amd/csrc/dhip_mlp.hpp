// dhip_mlp.hpp -- the learned warm start: a per-DOF network 12 -> 64 -> 64 -> 64 -> 2 (tanh
// hidden layers) that predicts the next time level's change of [mu; c] from the last four time
// levels, the step's right-hand side and the preconditioner diagonal.  No reference
// counterpart: GMRES still runs to the same tolerance from the predicted start.
//
//   k_mlp_features  one lane per DOF: 12 features in float64 (differences of the history first),
//                   normalised, stored float32 [S][12].
//   k_mlp_infer     matrix cores: one wave per 16 DOFs, v_mfma_f32_16x16x32_bf16 for every layer
//                   (bf16 weights and layer inputs, float32 accumulation); weights staged in LDS.
//   k_mlp_train     matrix cores: 16 samples per wave, forward with k_mlp_infer's rounding points,
//                   backward in float32, gradients of at most 32 samples in float32 and their sums in
//                   float64; a block's gradient goes to its own slot (no atomics).
//   k_mlp_reduce    gradient = sum of the block slots in slot order; k_mlp_adam the update.
#pragma once

#include "dhip_assembly.hpp"
#include "dhip_common.hpp"

namespace dhip {

constexpr int MLP_NF = 12, MLP_H = 64, MLP_NO = 2;
constexpr int MLP_W1 = 0, MLP_B1 = MLP_W1 + MLP_H * MLP_NF, MLP_W2 = MLP_B1 + MLP_H, MLP_B2 = MLP_W2 + MLP_H * MLP_H,
              MLP_W3 = MLP_B2 + MLP_H, MLP_B3 = MLP_W3 + MLP_H * MLP_H, MLP_W4 = MLP_B3 + MLP_H,
              MLP_B4 = MLP_W4 + MLP_NO * MLP_H, MLP_NPARAM = MLP_B4 + MLP_NO;
static_assert(MLP_NPARAM == 9282, "parameter layout");

// packed bf16 weights for the matrix cores: [out][in] rows, layer 1 inputs padded to 32,
// layer 4 outputs padded to 16
constexpr int MLP_P1 = 0, MLP_P2 = MLP_P1 + MLP_H * 32, MLP_P3 = MLP_P2 + MLP_H * MLP_H,
              MLP_P4 = MLP_P3 + MLP_H * MLP_H, MLP_NPACK = MLP_P4 + 16 * MLP_H;

// float -> bfloat16 bits, round to nearest even
__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bfround(float f) { return __uint_as_float((uint32_t)f2bf(f) << 16); }

struct MlpNorm {
    double in_mean[MLP_NF], in_scale[MLP_NF];   // feature -> (feature - mean) * scale
    double out_mean[MLP_NO], out_scale[MLP_NO]; // correction = y * scale + mean
};

// Step scale: s_mu, s_c = RMS over the DOFs of the last change of mu and c (1 where it is 0).
// Two passes: per-block partial sums of squares, then one block adds them in block order.
constexpr int SCALE_B = 256;

__global__ void __launch_bounds__(SCALE_B) k_mlp_scale_part(const double *x0, const double *x1, int64_t n,
                                                            double *part) {
    double sm = 0.0, sc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * SCALE_B + threadIdx.x; i < n; i += (int64_t)gridDim.x * SCALE_B) {
        const double dm = x0[i] - x1[i], dc = x0[n + i] - x1[n + i];
        sm += dm * dm;
        sc += dc * dc;
    }
    sm = block_sum<SCALE_B>(sm);
    sc = block_sum<SCALE_B>(sc);
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = sm;
        part[2 * blockIdx.x + 1] = sc;
    }
}

// one wave: lane-strided partials, then the wave's butterfly sum (the same order in every call)
__global__ void k_mlp_scale_final(const double *part, int nb, int64_t n, double *scale) {
    double sm = 0.0, sc = 0.0;
    for (int b = threadIdx.x & 63; b < nb; b += 64) {
        sm += part[2 * b];
        sc += part[2 * b + 1];
    }
    sm = wave_sum(sm);
    sc = wave_sum(sc);
    if (threadIdx.x != 0) return;
    const double rm = sqrt(sm / (double)n), rc = sqrt(sc / (double)n);
    scale[0] = rm > 0.0 ? rm : 1.0;
    scale[1] = rc > 0.0 ? rc : 1.0;
}

// ---------------------------------------------------------------------------------------------
// Features of DOF i for the step n -> n+1 (h0 = x_n, newest first; s = step scale):
//   c_n, dc_n/s_c, dc_{n-1}/s_c, dc_{n-2}/s_c, mu_n, dmu_n/s_mu, dmu_{n-1}/s_mu, dmu_{n-2}/s_mu,
//   (r_i/d_i)/s_mu, (r_{n+i}/d_{n+i})/s_c, d_i, d_{n+i}
// with dv_k = v_k - v_{k-1}, r = b - K x_n the residual of the new system at the current state
// (the local right-hand side of the correction), d the preconditioner diagonal.
struct FeatArgs {
    const double *h0, *h1, *h2, *h3;
    const double *res, *pcdiag;
    const double *scale;
    int64_t n;
    MlpNorm norm;
    float *X;  // [n][12]
};

__global__ void k_mlp_features(FeatArgs a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const int64_t n = a.n;
    const double sm = a.scale[0], sc = a.scale[1];
    double f[MLP_NF];
    const double c0 = a.h0[n + i], c1 = a.h1[n + i], c2 = a.h2[n + i], c3 = a.h3[n + i];
    const double m0 = a.h0[i], m1 = a.h1[i], m2 = a.h2[i], m3 = a.h3[i];
    f[0] = c0;
    f[1] = (c0 - c1) / sc;
    f[2] = (c1 - c2) / sc;
    f[3] = (c2 - c3) / sc;
    f[4] = m0;
    f[5] = (m0 - m1) / sm;
    f[6] = (m1 - m2) / sm;
    f[7] = (m2 - m3) / sm;
    f[8] = (a.res[i] / a.pcdiag[i]) / sm;
    f[9] = (a.res[n + i] / a.pcdiag[n + i]) / sc;
    f[10] = a.pcdiag[i];
    f[11] = a.pcdiag[n + i];
#pragma unroll
    for (int k = 0; k < MLP_NF; ++k) a.X[i * MLP_NF + k] = (float)((f[k] - a.norm.in_mean[k]) * a.norm.in_scale[k]);
}

// The prediction is a correction of linear extrapolation in scaled units:
//   x_{n+1} = x_n + s * (dx_n/s + y * out_scale + out_mean).
// (Linear, not quadratic: extrapolating the solver's own tolerance-level errors with weights
// 3, -3, 1 lets them grow from step to step in the slowly converging modes of GMRES.)
__device__ __forceinline__ double extrap_scaled(double v0, double v1, double, double s) { return (v0 - v1) / s; }

// targets: ((x_next - x_n)/s - extrapolation - mean) / out_scale, per DOF [mu, c]
struct TargetArgs {
    const double *xn1, *h0, *h1, *h2;
    const double *scale;
    int64_t n;
    MlpNorm norm;
    float *T;  // [n][2]
};

__global__ void k_mlp_targets(TargetArgs a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const int64_t n = a.n;
#pragma unroll
    for (int o = 0; o < MLP_NO; ++o) {
        const int64_t j = o == 0 ? i : n + i;  // o = 0: mu, o = 1: c
        const double s = a.scale[o];
        const double corr = (a.xn1[j] - a.h0[j]) / s - extrap_scaled(a.h0[j], a.h1[j], a.h2[j], s);
        a.T[2 * i + o] = (float)((corr - a.norm.out_mean[o]) / a.norm.out_scale[o]);
    }
}

// candidate starts: x0 = x_n + s * (extrapolation + y * out_scale + out_mean) (the network's) and
// xq = x_n + s * extrapolation (linear extrapolation alone)
struct CombineArgs {
    const double *h0, *h1, *h2;
    const float *Y;
    const double *scale;
    int64_t n;
    MlpNorm norm;
    double *x0, *xq;
};

__global__ void k_mlp_combine(CombineArgs a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const int64_t n = a.n;
#pragma unroll
    for (int o = 0; o < MLP_NO; ++o) {
        const int64_t j = o == 0 ? i : n + i;
        const double s = a.scale[o];
        const double ex = extrap_scaled(a.h0[j], a.h1[j], a.h2[j], s);
        const double corr = (double)a.Y[2 * i + o] * a.norm.out_scale[o] + a.norm.out_mean[o];
        a.x0[j] = a.h0[j] + s * (ex + corr);
        a.xq[j] = a.h0[j] + s * ex;
    }
}

// ---------------------------------------------------------------------------------------------
// packed bf16 weights from the float32 master parameters
__global__ void k_mlp_pack(const float *theta, uint16_t *pk) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= MLP_NPACK) return;
    float v = 0.f;
    if (t < MLP_P2) {
        const int o = t / 32, k = t % 32;
        v = k < MLP_NF ? theta[MLP_W1 + o * MLP_NF + k] : 0.f;
    } else if (t < MLP_P3) {
        v = theta[MLP_W2 + (t - MLP_P2)];
    } else if (t < MLP_P4) {
        v = theta[MLP_W3 + (t - MLP_P3)];
    } else {
        const int o = (t - MLP_P4) / MLP_H, k = (t - MLP_P4) % MLP_H;
        v = o < MLP_NO ? theta[MLP_W4 + o * MLP_H + k] : 0.f;
    }
    pk[t] = f2bf(v);
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

constexpr int INFER_WAVES = 4;  // 64 DOFs per block

// Matrix-core inference.  v_mfma_f32_16x16x32_bf16 lane layout: lane l holds A[l%16][8(l/16)+j],
// B[8(l/16)+j][l%16] (j < 8) and D[4(l/16)+i][l%16] (i < 4).  A = layer input (16 DOFs x 32),
// B = W^T (32 inputs x 16 outputs), read as 8 consecutive bf16 of a packed [out][in] row.
__global__ void __launch_bounds__(64 * INFER_WAVES) k_mlp_infer(const float *X, int64_t S, const uint16_t *packed,
                                                               const float *theta, float *Y) {
    __shared__ __align__(16) uint16_t W[MLP_NPACK];
    __shared__ float bias[3 * MLP_H + MLP_NO];
    __shared__ __align__(16) uint16_t act[INFER_WAVES][16][MLP_H];
    for (int t = threadIdx.x; t < MLP_NPACK; t += blockDim.x) W[t] = packed[t];
    for (int t = threadIdx.x; t < MLP_H; t += blockDim.x) {
        bias[t] = theta[MLP_B1 + t];
        bias[MLP_H + t] = theta[MLP_B2 + t];
        bias[2 * MLP_H + t] = theta[MLP_B3 + t];
    }
    if (threadIdx.x < MLP_NO) bias[3 * MLP_H + threadIdx.x] = theta[MLP_B4 + threadIdx.x];
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int row = lane & 15, kq = lane >> 4;
    // each block stages the weights once and walks its share of 64-DOF tiles
    const int64_t ntiles = (S + 16 * INFER_WAVES - 1) / (16 * INFER_WAVES);
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t m0 = (tile * INFER_WAVES + wv) * 16;
    // layer 1 input: features 8kq .. 8kq+7 of DOF m0+row (12 real features, zero padding)
    bf16x8_t a1;
    {
        const int64_t s = m0 + row;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = 8 * kq + j;
            const float v = (s < S && k < MLP_NF) ? X[s * MLP_NF + k] : 0.f;
            a1[j] = __builtin_bit_cast(__bf16, f2bf(v));
        }
    }
    auto bfrag = [&](int base, int ld, int n0, int k0) {
        return *reinterpret_cast<const bf16x8_t *>(&W[base + (n0 + row) * ld + k0 + 8 * kq]);
    };
    auto store_act = [&](const floatx4_t &d, int n0, const float *b) {
#pragma unroll
        for (int i = 0; i < 4; ++i) act[wv][4 * kq + i][n0 + row] = f2bf(tanhf(d[i] + b[n0 + row]));
    };
    // layer 1 (K = 32)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
        floatx4_t d = {0.f, 0.f, 0.f, 0.f};
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, bfrag(MLP_P1, 32, 16 * nt, 0), d, 0, 0, 0);
        store_act(d, 16 * nt, bias);
    }
    __syncthreads();
    // layers 2 and 3 (K = 64)
#pragma unroll
    for (int layer = 0; layer < 2; ++layer) {
        const int base = layer == 0 ? MLP_P2 : MLP_P3;
        bf16x8_t a[2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) a[kk] = *reinterpret_cast<const bf16x8_t *>(&act[wv][row][32 * kk + 8 * kq]);
        floatx4_t d[4];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
            d[nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
                d[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kk], bfrag(base, MLP_H, 16 * nt, 32 * kk), d[nt], 0, 0, 0);
        }
        __syncthreads();  // every lane has read its layer input
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) store_act(d[nt], 16 * nt, bias + (layer + 1) * MLP_H);
        __syncthreads();
    }
    // output layer (16 padded outputs, 2 real)
    {
        bf16x8_t a[2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) a[kk] = *reinterpret_cast<const bf16x8_t *>(&act[wv][row][32 * kk + 8 * kq]);
        floatx4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kk], bfrag(MLP_P4, MLP_H, 0, 32 * kk), d, 0, 0, 0);
        if (row < MLP_NO) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t s = m0 + 4 * kq + i;
                if (s < S) Y[s * MLP_NO + row] = d[i] + bias[3 * MLP_H + row];
            }
        }
    }
    __syncthreads();  // the next tile overwrites this wave's activations
    }
}

// ---------------------------------------------------------------------------------------------
// training
//
// One wave owns 16 samples at a time, a block 64, and keeps them in registers from the forward pass to the last
// weight gradient.
//   * Products are taken with the units as the matrix rows and the samples as the columns, so a lane
//     holds units 16 t + 4 q + i (q = lane / 16, i = 0..3) of sample lane % 16, and that register file is
//     the B operand of the next product when its contraction index is enumerated in the same order: the
//     forward weights are staged in that order, the backward ones are read through it.
//   * Forward: bf16 weights and layer inputs, v_mfma_f32_16x16x32_bf16 (as k_mlp_infer).  Backward: the
//     float32 deltas meet float32 copies of the rounded weights and inputs in v_mfma_f32_16x16x4_f32, so
//     no operand is rounded further.
//   * Weight gradients contract over the block's samples: delta and layer input go through LDS once per layer
//     (rows of 68 floats: the lanes' four sample rows 4 q + kk lie 16 banks apart) and each wave takes
//     one tile row of every gradient over all 64 samples, so that its sums are few enough to be kept
//     in float64.  The matrix cores add 32 samples in float32, which then go into the float64 sums: the error does
//     not grow with the minibatch.  Two sets of tiles in turn, one barrier a layer: a set is written again only
//     after the barrier behind its readers.
// A block's sums go to one float64 slot; k_mlp_reduce adds the slots.
// Bound by the float32 matrix rate and the tanh evaluations, about 9,500 matrix cycles per 16 samples.
// At 65,536 samples on 256 CUs 90 us (81 with every product of a wave's own samples and its sums over all its tiles
// in float32: an entry's error was 1e-6 there and 1.5e-5 for 2^20 equal samples, now 5e-7 for any number);
// 32 samples a block with every product on the vector units and one slot per 32 samples took 350 us.
constexpr int TW = 4;               // waves per block
constexpr int TRAIN_T = 64 * TW;    // threads per block
constexpr int TSW = 16;             // samples per wave and pass
constexpr int TLD = 68;             // row length of the LDS tiles and of the float32 weights

struct TrainArgs {
    const float *X, *T;       // [S][12], [S][2]
    const int32_t *idx;       // minibatch sample ids
    int64_t B;                // minibatch size
    const float *theta;
    double *part;             // [blocks][MLP_NPARAM + 1] (last: loss)
};

// bf16 forward weights as A fragments of v_mfma_f32_16x16x32_bf16: [fragment][lane][8].
constexpr int TF_1 = 0, TF_2 = 4, TF_3 = 12, TF_4 = 20, TF_N = 22;

struct TrainShared {
    __align__(16) uint16_t frag[TF_N * 64 * 8];
    float w2[MLP_H * TLD], w3[MLP_H * TLD];   // rounded weights [out][in] for the backward products
    float w4[MLP_NO * MLP_H];
    float bias[3 * MLP_H + MLP_NO];
    float dy[MLP_NO][TW * TSW];
    struct Tiles {
        __align__(16) float dz[TW][TSW * TLD], in[TW][TSW * TLD];
    };
    Tiles tiles0;
    union {
        Tiles tiles1;
        __align__(16) float theta[MLP_NPARAM];   // until the weights are staged
        double sums[TW][2 * MLP_H + MLP_NO + 1]; // the waves' bias gradients and losses at the end
    };
};
constexpr size_t TRAIN_LDS = sizeof(TrainShared);
static_assert(TRAIN_LDS <= 160 * 1024, "k_mlp_train's LDS");

// weight of out unit n at in unit k (layer 1: k >= 12 is padding; layer 4: n >= 2)
__device__ inline float train_weight(const float *th, int layer, int n, int k) {
    if (layer == 1) return k < MLP_NF ? th[MLP_W1 + n * MLP_NF + k] : 0.f;
    if (layer == 4) return n < MLP_NO ? th[MLP_W4 + n * MLP_H + k] : 0.f;
    return th[(layer == 2 ? MLP_W2 : MLP_W3) + n * MLP_H + k];
}

__global__ void __launch_bounds__(TRAIN_T) k_mlp_train(TrainArgs a) {
    extern __shared__ __align__(16) unsigned char train_lds[];
    TrainShared &sh = *reinterpret_cast<TrainShared *>(train_lds);
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, col = lane & 15, q = lane >> 4;
    // the parameters once into LDS, every load in flight before the first use
    {
        constexpr int NV = (MLP_NPARAM / 2 + TRAIN_T - 1) / TRAIN_T;
        float2 v[NV];
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int e = t + u * TRAIN_T;
            if (e < MLP_NPARAM / 2) v[u] = reinterpret_cast<const float2 *>(a.theta)[e];
        }
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int e = t + u * TRAIN_T;
            if (e < MLP_NPARAM / 2) reinterpret_cast<float2 *>(sh.theta)[e] = v[u];
        }
    }
    __syncthreads();
    const float *theta = sh.theta;
    for (int e = t; e < TF_N * 512; e += TRAIN_T) {
        const int f = e >> 9, ln = (e >> 3) & 63, x = e & 7, row = ln & 15, j = ln >> 4;
        int layer, n, k;
        if (f < TF_2) {
            layer = 1;
            n = 16 * f + row;
            k = 8 * j + x;
        } else {
            layer = f < TF_3 ? 2 : f < TF_4 ? 3 : 4;
            const int g = f - (layer == 2 ? TF_2 : layer == 3 ? TF_3 : TF_4);
            n = 16 * (g >> 1) + row;
            k = 16 * (2 * (g & 1) + (x >> 2)) + 4 * j + (x & 3);
        }
        sh.frag[e] = f2bf(train_weight(theta, layer, n, k));
    }
    for (int e = t; e < MLP_H * MLP_H; e += TRAIN_T) {
        const int n = e / MLP_H, k = e % MLP_H;
        sh.w2[n * TLD + k] = bfround(theta[MLP_W2 + e]);
        sh.w3[n * TLD + k] = bfround(theta[MLP_W3 + e]);
    }
    for (int e = t; e < MLP_NO * MLP_H; e += TRAIN_T) sh.w4[e] = bfround(theta[MLP_W4 + e]);
    for (int e = t; e < MLP_H; e += TRAIN_T) {
        sh.bias[e] = theta[MLP_B1 + e];
        sh.bias[MLP_H + e] = theta[MLP_B2 + e];
        sh.bias[2 * MLP_H + e] = theta[MLP_B3 + e];
    }
    if (t < MLP_NO) sh.bias[3 * MLP_H + t] = theta[MLP_B4 + t];
    __syncthreads();

    // the wave's dW tiles: out tile wv of layers 1 (its column 12 is the bias), 2 and 3, in tile wv of layer 4
    double g1[1][4] = {}, g2[4][4] = {}, g3[4][4] = {}, g4[1][4] = {};
    double gb2[16] = {}, gb3[16] = {}, gb4[2] = {}, loss = 0.0;   // over the lane's samples

    auto frag = [&](int f) { return *reinterpret_cast<const bf16x8_t *>(&sh.frag[(f * 64 + lane) * 8]); };
    // tanh of a layer's products, in place
    auto activate = [&](float (&h)[4][4], const float *b) {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) h[nt][i] = tanhf(h[nt][i] + b[16 * nt + 4 * q + i]);
    };
    // the rounded layer inputs of contraction step ks
    auto act_frag = [&](const float (&h)[4][4], int ks) {
        bf16x8_t v;
#pragma unroll
        for (int x = 0; x < 8; ++x) v[x] = __builtin_bit_cast(__bf16, f2bf(h[2 * ks + (x >> 2)][x & 3]));
        return v;
    };
    auto forward = [&](const float (&hin)[4][4], int f0, float (&hout)[4][4]) {
        const bf16x8_t b0 = act_frag(hin, 0), b1 = act_frag(hin, 1);
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
            floatx4_t d = {0.f, 0.f, 0.f, 0.f};
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(f0 + 2 * nt), b0, d, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(f0 + 2 * nt + 1), b1, d, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) hout[nt][i] = d[i];
        }
    };
    auto store = [&](float *buf, const float (&v)[4][4], bool round) {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
            floatx4_t x;
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = round ? bfround(v[nt][i]) : v[nt][i];
            *reinterpret_cast<floatx4_t *>(&buf[col * TLD + 16 * nt + 4 * q]) = x;
        }
    };
    // g[kt] += A^T B over the block's samples, A(k) the lane's entry of sample row k of the wave's out tile, B(k, kt) of
    // the layer input's tile kt; 32 samples in float32
    auto weight_grad = [&](auto &g, auto &&A, auto &&B) {
        constexpr int NK = sizeof(g) / sizeof(g[0]);
#pragma unroll
        for (int w0 = 0; w0 < TW; w0 += 2) {
            floatx4_t acc[NK];
#pragma unroll
            for (int kt = 0; kt < NK; ++kt) acc[kt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = w0; w < w0 + 2; ++w)
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    const float av = A(w, 4 * q + kk);
#pragma unroll
                    for (int kt = 0; kt < NK; ++kt)
                        acc[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, B(w, 4 * q + kk, kt), acc[kt], 0, 0, 0);
                }
#pragma unroll
            for (int kt = 0; kt < NK; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) g[kt][i] += (double)acc[kt][i];
        }
    };
    // delta of the layer below: (W^T d) (1 - h^2), the contraction index n = 16 nt + 4 q + i from d's registers
    auto backward = [&](const float *w, const float (&d)[4][4], const float (&h)[4][4], float (&out)[4][4]) {
        floatx4_t acc[4];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) acc[kt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
                    acc[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[(16 * nt + 4 * q + i) * TLD + 16 * kt + col],
                                                                   d[nt][i], acc[kt], 0, 0, 0);
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) out[kt][i] = acc[kt][i] * (1.f - h[kt][i] * h[kt][i]);
    };

    const int64_t ntile = (a.B + TSW * TW - 1) / (TSW * TW);
    for (int64_t tile = blockIdx.x; tile < ntile; tile += gridDim.x) {   // the same for every wave of the block
        const int64_t g = tile * (TSW * TW) + TSW * wv + col;
        const int64_t sid = g < a.B ? (int64_t)a.idx[g] : -1;
        // features 8 q .. 8 q + 7 of the lane's sample (12 real ones, zero padding)
        float x0[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            const int k = 8 * q + x;
            x0[x] = sid >= 0 && k < MLP_NF ? bfround(a.X[sid * MLP_NF + k]) : 0.f;
        }
        float tv[2] = {0.f, 0.f};
        if (sid >= 0) {
            tv[0] = a.T[sid * MLP_NO];
            tv[1] = a.T[sid * MLP_NO + 1];
        }
        float h1[4][4], h2[4][4], h3[4][4];
        {
            bf16x8_t b;
#pragma unroll
            for (int x = 0; x < 8; ++x) b[x] = __builtin_bit_cast(__bf16, f2bf(x0[x]));
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                floatx4_t d = {0.f, 0.f, 0.f, 0.f};
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(TF_1 + nt), b, d, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) h1[nt][i] = d[i];
            }
        }
        activate(h1, sh.bias);
        forward(h1, TF_2, h2);
        activate(h2, sh.bias + MLP_H);
        forward(h2, TF_3, h3);
        activate(h3, sh.bias + 2 * MLP_H);
        // output (units 0 and 1 in lanes q = 0), residual, loss, dY = (y - t) / B
        float dy[2];
        {
            floatx4_t d = {0.f, 0.f, 0.f, 0.f};
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(TF_4), act_frag(h3, 0), d, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(TF_4 + 1), act_frag(h3, 1), d, 0, 0, 0);
#pragma unroll
            for (int o = 0; o < MLP_NO; ++o) {
                const float y = __shfl(d[o], col, 64) + sh.bias[3 * MLP_H + o];
                const float r = sid >= 0 ? y - tv[o] : 0.f;
                dy[o] = r / (float)a.B;
                if (q == 0) {
                    loss += (double)(0.5f * r * r);
                    gb4[o] += (double)dy[o];
                    sh.dy[o][TSW * wv + col] = dy[o];
                }
            }
        }
        // layer 4: weights and the delta of layer 3
        TrainShared::Tiles &t0 = sh.tiles0, &t1 = sh.tiles1;
        store(t0.in[wv], h3, true);
        float d3[4][4], d2[4][4], d1[4][4];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = 16 * nt + 4 * q + i;
                const float v = __fmaf_rn(dy[1], sh.w4[MLP_H + n], dy[0] * sh.w4[n]);
                d3[nt][i] = v * (1.f - h3[nt][i] * h3[nt][i]);
                gb3[4 * nt + i] += (double)d3[nt][i];
            }
        __syncthreads();
        weight_grad(g4, [&](int w, int k) { return col < MLP_NO ? sh.dy[col < MLP_NO ? col : 0][TSW * w + k] : 0.f; },
                    [&](int w, int k, int) { return t0.in[w][k * TLD + 16 * wv + col]; });
        // layer 3
        store(t1.in[wv], h2, true);
        store(t1.dz[wv], d3, false);
        backward(sh.w3, d3, h2, d2);
#pragma unroll
        for (int e = 0; e < 16; ++e) gb2[e] += (double)d2[e >> 2][e & 3];
        __syncthreads();
        weight_grad(g3, [&](int w, int k) { return t1.dz[w][k * TLD + 16 * wv + col]; },
                    [&](int w, int k, int kt) { return t1.in[w][k * TLD + 16 * kt + col]; });
        // layer 2
        store(t0.in[wv], h1, true);
        store(t0.dz[wv], d2, false);
        backward(sh.w2, d2, h1, d1);
        __syncthreads();
        weight_grad(g2, [&](int w, int k) { return t0.dz[w][k * TLD + 16 * wv + col]; },
                    [&](int w, int k, int kt) { return t0.in[w][k * TLD + 16 * kt + col]; });
        // layer 1: inputs 0..11, a one in column 12 for the bias
        store(t1.dz[wv], d1, false);
        if (q < 2) {
#pragma unroll
            for (int x = 0; x < 8; ++x) t1.in[wv][col * TLD + 8 * q + x] = 8 * q + x == MLP_NF ? 1.f : x0[x];
        }
        __syncthreads();
        weight_grad(g1, [&](int w, int k) { return t1.dz[w][k * TLD + 16 * wv + col]; },
                    [&](int w, int k, int) { return t1.in[w][k * TLD + col]; });
    }

    // sums over the 16 lanes that share units, then over the waves in their order
    auto over_samples = [&](double v) {
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        return v;
    };
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        gb2[e] = over_samples(gb2[e]);
        gb3[e] = over_samples(gb3[e]);
    }
    gb4[0] = over_samples(gb4[0]);
    gb4[1] = over_samples(gb4[1]);
    loss = over_samples(loss);
    __syncthreads();
    if (col == 0) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int n = 16 * (e >> 2) + 4 * q + (e & 3);
            sh.sums[wv][n] = gb2[e];
            sh.sums[wv][MLP_H + n] = gb3[e];
        }
    }
    if (lane == 0) {
        sh.sums[wv][2 * MLP_H] = gb4[0];
        sh.sums[wv][2 * MLP_H + 1] = gb4[1];
        sh.sums[wv][2 * MLP_H + 2] = loss;
    }
    double *P = a.part + (size_t)blockIdx.x * (MLP_NPARAM + 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = 16 * wv + 4 * q + i;
        if (col < MLP_NF) P[MLP_W1 + n * MLP_NF + col] = g1[0][i];
        else if (col == MLP_NF) P[MLP_B1 + n] = g1[0][i];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            P[MLP_W2 + n * MLP_H + 16 * kt + col] = g2[kt][i];
            P[MLP_W3 + n * MLP_H + 16 * kt + col] = g3[kt][i];
        }
        if (q == 0 && i < MLP_NO) P[MLP_W4 + i * MLP_H + 16 * wv + col] = g4[0][i];
    }
    __syncthreads();
    if (t < 2 * MLP_H + MLP_NO + 1) {
        double v = sh.sums[0][t];
#pragma unroll
        for (int w = 1; w < TW; ++w) v += sh.sums[w][t];
        P[t < MLP_H ? MLP_B2 + t : t < 2 * MLP_H ? MLP_B3 + t - MLP_H : t < 2 * MLP_H + MLP_NO ? MLP_B4 + t - 2 * MLP_H
                                                                                             : MLP_NPARAM] = v;
    }
}

// grad[p] = sum over the block slots of part[slot][p]; p = MLP_NPARAM is the loss.  64 columns
// per block, 16 threads a column that take every 16th slot, added in order: 6.6 us for 256 slots (one thread a
// column over the 2,048 slots that 32 samples a block left: 500 us).
constexpr int MLP_RED_G = 16;
__global__ void __launch_bounds__(64 * MLP_RED_G) k_mlp_reduce(const double *part, int nslot, double *grad) {
    __shared__ double s[MLP_RED_G][64];
    const int c = threadIdx.x & 63, g = threadIdx.x >> 6, p = blockIdx.x * 64 + c;
    double v = 0.0;
    if (p <= MLP_NPARAM)
        for (int b = g; b < nslot; b += MLP_RED_G) v += part[(size_t)b * (MLP_NPARAM + 1) + p];
    s[g][c] = v;
    __syncthreads();
    if (g == 0 && p <= MLP_NPARAM) {
        for (int k = 1; k < MLP_RED_G; ++k) v += s[k][c];
        grad[p] = v;
    }
}

struct AdamArgs {
    float *theta, *m, *v;
    const double *grad;
    float lr, beta1, beta2, eps;
    int step;  // 1-based
};

__global__ void k_mlp_adam(AdamArgs a) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= MLP_NPARAM) return;
    const float g = (float)a.grad[p];
    const float m = a.beta1 * a.m[p] + (1.f - a.beta1) * g;
    const float v = a.beta2 * a.v[p] + (1.f - a.beta2) * g * g;
    a.m[p] = m;
    a.v[p] = v;
    const float mh = m / (1.f - powf(a.beta1, (float)a.step));
    const float vh = v / (1.f - powf(a.beta2, (float)a.step));
    a.theta[p] -= a.lr * mh / (sqrtf(vh) + a.eps);
}

}  // namespace dhip
