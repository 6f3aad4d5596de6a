// rp_mlp.hip -- forward, backward and AdamW kernels of the Krylov-schedule
// proposer network, a 12 -> 64 -> 64 -> 2 perceptron with tanh hidden
// layers, in FP32.
//
// Parameter layout (RP_MLP_NPARAMS = 5122 floats):
//   W1[64][12] @ 0, b1[64] @ 768, W2[64][64] @ 832, b2[64] @ 4928,
//   W3[2][64] @ 4992, b3[2] @ 5120.
//
// Forward: one 64-wide wavefront evaluates one sample: lane j owns hidden unit
// j of both layers, so the 64x64 layer is one LDS-broadcast dot product per
// lane (W2 is staged transposed so that the 64 lanes read 64 consecutive
// words) and the 2 outputs are wavefront reductions.
//
// Gradient: a workgroup takes tiles of 64 samples and forms every product of
// the two passes with the FP32 matrix instructions; it writes one partial row
// of gradients, and a second kernel adds the rows in a fixed order, so
// gradients are bitwise deterministic for a given sample count.
#include "rp_internal.h"

#include <math.h>
#include <string.h>

#include <algorithm>

namespace rp {
namespace {

constexpr int kIn = RP_MLP_IN, kHid = RP_MLP_HIDDEN, kOut = RP_MLP_OUT;
constexpr int oW1 = 0, oB1 = oW1 + kHid * kIn, oW2 = oB1 + kHid, oB2 = oW2 + kHid * kHid,
              oW3 = oB2 + kHid, oB3 = oW3 + kOut * kHid, kNP = oB3 + kOut;
static_assert(kNP == RP_MLP_NPARAMS, "parameter layout");
static_assert(kHid == 64, "one lane per hidden unit of a 64-wide wavefront");

constexpr int kWaves = 4, kThreads = 64 * kWaves;
constexpr int kMaxGradBlocks = kMlpRows;

struct Shared {
    float w1t[kIn * kHid];     // w1t[i*64 + j] = W1[j][i]
    float w2t[kHid * kHid];    // w2t[k*64 + j] = W2[j][k]
    float h1[kWaves][kHid];
    float x[kWaves][kIn];
};

__device__ inline float wave_sum(float v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ inline void stage_weights(Shared &sh, const float *__restrict__ p)
{
    for (int e = threadIdx.x; e < kHid * kIn; e += kThreads) {
        int j = e / kIn, i = e % kIn;
        sh.w1t[i * kHid + j] = p[oW1 + e];
    }
    for (int e = threadIdx.x; e < kHid * kHid; e += kThreads) {
        int j = e / kHid, k = e % kHid;
        sh.w2t[k * kHid + j] = p[oW2 + e];
    }
}

// forward of one sample by one wave; returns h1, h2 of this lane and y[2]
__device__ inline void wave_forward(Shared &sh, int wv, int lane, const float *__restrict__ p,
                                    const float *__restrict__ xs, float &h1, float &h2,
                                    float y[kOut])
{
    if (lane < kIn) sh.x[wv][lane] = xs[lane];
    __builtin_amdgcn_wave_barrier();
    float z = p[oB1 + lane];
    for (int i = 0; i < kIn; i++) z += sh.w1t[i * kHid + lane] * sh.x[wv][i];
    h1 = tanhf(z);
    sh.h1[wv][lane] = h1;
    __builtin_amdgcn_wave_barrier();
    z = p[oB2 + lane];
    for (int k = 0; k < kHid; k++) z += sh.w2t[k * kHid + lane] * sh.h1[wv][k];
    h2 = tanhf(z);
    for (int o = 0; o < kOut; o++) y[o] = wave_sum(p[oW3 + o * kHid + lane] * h2) + p[oB3 + o];
}

__global__ __launch_bounds__(kThreads) void k_mlp_forward(const float *__restrict__ p,
                                                          const float *__restrict__ X, long n,
                                                          float *__restrict__ Y)
{
    __shared__ Shared sh;
    stage_weights(sh, p);
    __syncthreads();
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (long s = (long)blockIdx.x * kWaves + wv; s < n; s += (long)gridDim.x * kWaves) {
        float h1, h2, y[kOut];
        wave_forward(sh, wv, lane, p, X + s * kIn, h1, h2, y);
        if (lane < kOut) Y[s * kOut + lane] = y[lane];
        __builtin_amdgcn_wave_barrier();
    }
}

// Loss and gradient of tiles of 64 samples: loss = sum_s sum_o w[s,o]
// (y[s,o] - t[s,o])^2 / n.  The layers' products are 16x16x4 FP32 matrix
// instructions (operand A: lane l holds row l mod 16 at k = l / 16; B: column
// l mod 16 at k = l / 16; result register r: row 4 (l / 16) + r, column l mod
// 16), all operands from LDS, whose rows are padded by one word against bank
// conflicts.  Wavefront w takes the samples 16 w .. 16 w + 15 in the passes
// and the rows 16 w .. of dW1, dW2 in the sums over samples, which stay in
// registers over the workgroup's tiles.
//
// Bound by latency: 2792 samples are 44 workgroups.  One wavefront per sample
// with LDS dot products, on 32 workgroups, took 61 us there (22 samples in
// series, 2.8 us each).
constexpr int kTile = 64, kPad = kHid + 1, kXPad = 17;
using f4 = __attribute__((ext_vector_type(4))) float;

// c += A B over K (a multiple of 4); a(row, k), b(k, column) for rows and
// columns 0..15 of this tile
template <int K, typename FA, typename FB>
__device__ __forceinline__ f4 tile_mma(f4 c, int lane, FA &&a, FB &&b)
{
#pragma unroll
    for (int k = 0; k < K; k += 4)
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(a(lane & 15, k + (lane >> 4)),
                                                 b(k + (lane >> 4), lane & 15), c, 0, 0, 0);
    return c;
}

__global__ __launch_bounds__(kThreads) void k_mlp_grad(const float *__restrict__ p,
                                                       const float *__restrict__ X,
                                                       const float *__restrict__ T,
                                                       const float *__restrict__ W, long n,
                                                       float *__restrict__ part)
{
    __shared__ float w1[kHid][kXPad], w2[kHid][kPad];     // W1 with zero columns 12..15
    __shared__ float x[kTile][kXPad], h1[kTile][kPad], dz2[kTile][kPad], dz1[kTile][kPad];
    __shared__ float red[kWaves][5 * kHid + 4];           // gb1, gb2, gw3[2], loss and gb3
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
    for (int e = threadIdx.x; e < kHid * 16; e += kThreads) {
        const int j = e >> 4, i = e & 15;
        w1[j][i] = i < kIn ? p[oW1 + j * kIn + i] : 0.f;
    }
    for (int e = threadIdx.x; e < kHid * kHid; e += kThreads) w2[e >> 6][e & 63] = p[oW2 + e];
    float b1[4], b2[4], w3[kOut][4], b3[kOut];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        b1[t] = p[oB1 + 16 * t + col];
        b2[t] = p[oB2 + 16 * t + col];
        for (int o = 0; o < kOut; o++) w3[o][t] = p[oW3 + o * kHid + 16 * t + col];
    }
    for (int o = 0; o < kOut; o++) b3[o] = p[oB3 + o];
    const float inv_n = 1.0f / (float)n;
    f4 gw2[4], gw1 = {0, 0, 0, 0};
    float gb1[4], gb2[4], gw3[kOut][4], gb3[kOut] = {0, 0}, loss = 0;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        gw2[t] = f4{0, 0, 0, 0};
        gb1[t] = gb2[t] = gw3[0][t] = gw3[1][t] = 0;
    }
    const long tiles = (n + kTile - 1) / kTile;
    const int row0 = 16 * wv;
    for (long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const long s0 = tile * kTile;
        __syncthreads();     // the last tile's reads are done (first: w1, w2 follow)
        for (int e = threadIdx.x; e < kTile * 16; e += kThreads) {
            const int r = e >> 4, i = e & 15;
            x[r][i] = i < kIn && s0 + r < n ? X[(s0 + r) * kIn + i] : 0.f;
        }
        __syncthreads();
        // forward, layer 1
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const f4 z = tile_mma<16>(f4{b1[t], b1[t], b1[t], b1[t]}, lane,
                                      [&](int r, int k) { return x[row0 + r][k]; },
                                      [&](int k, int c) { return w1[16 * t + c][k]; });
#pragma unroll
            for (int r = 0; r < 4; r++) h1[row0 + 4 * grp + r][16 * t + col] = tanhf(z[r]);
        }
        // (a wavefront reads only its own rows of h1 until the sums below)
        __builtin_amdgcn_wave_barrier();
        // layer 2 and the outputs; the 16 lanes of a group hold 4 samples
        float h2[4][4], y[kOut][4];
#pragma unroll
        for (int r = 0; r < 4; r++) y[0][r] = y[1][r] = 0;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const f4 z = tile_mma<kHid>(f4{b2[t], b2[t], b2[t], b2[t]}, lane,
                                        [&](int r, int k) { return h1[row0 + r][k]; },
                                        [&](int k, int c) { return w2[16 * t + c][k]; });
#pragma unroll
            for (int r = 0; r < 4; r++) {
                h2[t][r] = tanhf(z[r]);
                y[0][r] += w3[0][t] * h2[t][r];
                y[1][r] += w3[1][t] * h2[t][r];
            }
        }
        float dy[kOut][4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const long smp = s0 + row0 + 4 * grp + r;
#pragma unroll
            for (int o = 0; o < kOut; o++) {
                float v = y[o][r];
                for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
                float d = 0;
                if (smp < n) {
                    const float w = W ? W[smp * kOut + o] : 1.0f;
                    const float e = v + b3[o] - T[smp * kOut + o];
                    d = 2.0f * w * e * inv_n;
                    if (col == 0) {
                        loss += w * e * e;
                        gb3[o] += d;
                    }
                }
                dy[o][r] = d;
            }
        }
        // backward, layer 2
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float h = h2[t][r];
                const float d = (w3[0][t] * dy[0][r] + w3[1][t] * dy[1][r]) * (1.0f - h * h);
                gw3[0][t] += dy[0][r] * h;
                gw3[1][t] += dy[1][r] * h;
                gb2[t] += d;
                dz2[row0 + 4 * grp + r][16 * t + col] = d;
            }
        __builtin_amdgcn_wave_barrier();
        // layer 1
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const f4 d = tile_mma<kHid>(f4{0, 0, 0, 0}, lane,
                                        [&](int r, int k) { return dz2[row0 + r][k]; },
                                        [&](int k, int c) { return w2[k][16 * t + c]; });
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float h = h1[row0 + 4 * grp + r][16 * t + col];
                const float v = d[r] * (1.0f - h * h);
                gb1[t] += v;
                dz1[row0 + 4 * grp + r][16 * t + col] = v;
            }
        }
        __syncthreads();
        // the sums over the tile's samples
#pragma unroll
        for (int t = 0; t < 4; t++)
            gw2[t] = tile_mma<kTile>(gw2[t], lane, [&](int r, int k) { return dz2[k][row0 + r]; },
                                     [&](int k, int c) { return h1[k][16 * t + c]; });
        gw1 = tile_mma<kTile>(gw1, lane, [&](int r, int k) { return dz1[k][row0 + r]; },
                              [&](int k, int c) { return x[k][c]; });
    }
    float *row = part + (size_t)blockIdx.x * (kNP + 1);
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 4; r++)
            row[oW2 + (row0 + 4 * grp + r) * kHid + 16 * t + col] = gw2[t][r];
    if (col < kIn)
#pragma unroll
        for (int r = 0; r < 4; r++) row[oW1 + (row0 + 4 * grp + r) * kIn + col] = gw1[r];
    // per-unit sums: over the four groups of lanes, then the wavefronts
    auto groups = [](float v) {
        v += __shfl_xor(v, 16, 64);
        return v + __shfl_xor(v, 32, 64);
    };
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const float a = groups(gb1[t]), b = groups(gb2[t]), c = groups(gw3[0][t]),
                    d = groups(gw3[1][t]);
        if (grp == 0) {
            float *q = red[wv] + 16 * t + col;
            q[0] = a;
            q[kHid] = b;
            q[2 * kHid] = c;
            q[3 * kHid] = d;
        }
    }
    const float l = groups(loss), g0 = groups(gb3[0]), g1 = groups(gb3[1]);
    if (lane == 0) {
        red[wv][4 * kHid] = g0;
        red[wv][4 * kHid + 1] = g1;
        red[wv][4 * kHid + 2] = l;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 4 * kHid + 3; e += kThreads) {
        float a = red[0][e];
        for (int q = 1; q < kWaves; q++) a += red[q][e];
        row[e < kHid ? oB1 + e : e < 2 * kHid ? oB2 + e - kHid : e < 4 * kHid ? oW3 + e - 2 * kHid
            : e < 4 * kHid + 2 ? oB3 + e - 4 * kHid : kNP] = a;
    }
}

// out[e] = sum over blocks b of part[b][e], each of a workgroup's kRedRows
// groups of threads every kRedRows-th row, then the groups in order; the loss
// sums, at index kNP of each row, go to loss_out divided by n
constexpr int kRedRows = 8, kRedCols = 32;
__global__ __launch_bounds__(kRedRows *kRedCols) void k_mlp_reduce(
    const float *__restrict__ part, int nb, float *__restrict__ out, double *__restrict__ loss_out,
    long n)
{
    __shared__ float sh[kRedRows][kRedCols];
    const int c = threadIdx.x % kRedCols, g = threadIdx.x / kRedCols;
    const int e = blockIdx.x * kRedCols + c;
    float a = 0;
    if (e <= kNP)
#pragma unroll 8
        for (int b = g; b < nb; b += kRedRows) a += part[(size_t)b * (kNP + 1) + e];
    sh[g][c] = a;
    __syncthreads();
    if (g || e > kNP) return;
    for (int q = 1; q < kRedRows; q++) a += sh[q][c];
    if (e < kNP)
        out[e] = a;
    else
        loss_out[0] = (double)a / (double)n;
}

__global__ void k_mlp_adam(float *__restrict__ p, const float *__restrict__ g,
                           float *__restrict__ m, float *__restrict__ v, long np, float lr,
                           float b1, float b2, float eps, float wd, float c1, float c2)
{
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < np;
         e += (long)gridDim.x * blockDim.x) {
        float ge = g[e];
        float me = b1 * m[e] + (1.0f - b1) * ge;
        float ve = b2 * v[e] + (1.0f - b2) * ge * ge;
        m[e] = me;
        v[e] = ve;
        float mh = me / c1, vh = ve / c2;
        p[e] = p[e] - lr * (mh / (sqrtf(vh) + eps) + wd * p[e]);
    }
}

int grad_blocks(long n) { return (int)std::min<long>(kMaxGradBlocks, (n + kTile - 1) / kTile); }

}  // namespace
}  // namespace rp

using namespace rp;

extern "C" {

int rp_mlp_forward(const float *params, const float *X, int64_t n, float *Y)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(n >= 0, "n must be non-negative");
    if (n == 0) return RP_OK;
    RP_REQUIRE(params && X && Y, "null argument");
    int g = (int)std::min<int64_t>(1024, (n + kWaves - 1) / kWaves);
    RP_LAUNCH(RP_KERNEL_OTHER, k_mlp_forward, dim3(g), dim3(kThreads), 0, params, X, (long)n, Y);
    return RP_OK;
}

int rp_mlp_loss_grad(const float *params, const float *X, const float *T, const float *W,
                     int64_t n, float *grad, double *loss)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(n > 0, "n must be positive");
    RP_REQUIRE(params && X && T && grad, "null argument");
    Context &c = ctx();
    const int nb = grad_blocks((long)n);
    float *part = (float *)((char *)c.work + kMlpOffset);
    static_assert(kMlpRowFloats == kNP + 1, "gradient partial rows");
    RP_LAUNCH(RP_KERNEL_OTHER, k_mlp_grad, dim3(nb), dim3(kThreads), 0, params, X, T, W,
              (long)n, part);
    // the loss straight to pinned memory, in a place of its own: without a
    // wait (loss null) it may still be written while others use the buffer
    double *host_loss = c.pinned + kHostLoss;
    RP_LAUNCH(RP_KERNEL_OTHER, k_mlp_reduce, dim3(kNP / kRedCols + 1), dim3(kRedRows * kRedCols), 0,
              (const float *)part, nb, grad, host_loss, (long)n);
    if (loss) {
        RP_CHECK_HIP(hipStreamSynchronize(c.stream));
        if (c.prof) {
            st = prof_collect();
            if (st) return st;
        }
        *loss = *host_loss;
    }
    return RP_OK;
}

int rp_mlp_adam(float *params, const float *grad, float *m, float *v, int64_t np, double lr,
                double beta1, double beta2, double eps, double weight_decay, int64_t step)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(np > 0 && step >= 1, "np and step must be positive");
    RP_REQUIRE(params && grad && m && v, "null argument");
    RP_REQUIRE(beta1 >= 0 && beta1 < 1 && beta2 >= 0 && beta2 < 1, "betas must be in [0, 1)");
    const double c1 = 1.0 - pow(beta1, (double)step), c2 = 1.0 - pow(beta2, (double)step);
    int g = (int)std::min<int64_t>(1024, (np + 255) / 256);
    RP_LAUNCH(RP_KERNEL_OTHER, k_mlp_adam, dim3(g), dim3(256), 0, params, grad, m, v, (long)np,
              (float)lr, (float)beta1, (float)beta2, (float)eps, (float)weight_decay, (float)c1,
              (float)c2);
    return RP_OK;
}

int rp_mlp_infer(const float *params, const float *x_host, int n, float *y_host)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(n >= 1 && n <= RP_MLP_MAX_INFER, "n must be in [1, RP_MLP_MAX_INFER]");
    RP_REQUIRE(params && x_host && y_host, "null argument");
    Context &c = ctx();
    // staging: inputs and outputs in the pinned buffer and in the tail of the
    // workspace (stream order keeps them apart from reduction partials)
    float *hin = (float *)c.pinned, *hout = hin + RP_MLP_MAX_INFER * kIn;
    float *din = (float *)((char *)c.work + kMlpOffset - 32 * 1024);
    float *dout = din + RP_MLP_MAX_INFER * kIn;
    // the previous user of the pinned buffer has completed: every entry point
    // that fills it synchronizes before returning
    memcpy(hin, x_host, sizeof(float) * n * kIn);
    RP_CHECK_HIP(hipMemcpyAsync(din, hin, sizeof(float) * n * kIn, hipMemcpyHostToDevice,
                                c.stream));
    RP_LAUNCH(RP_KERNEL_OTHER, k_mlp_forward, dim3((n + kWaves - 1) / kWaves), dim3(kThreads), 0,
              params, (const float *)din, (long)n, dout);
    RP_CHECK_HIP(hipMemcpyAsync(hout, dout, sizeof(float) * n * kOut, hipMemcpyDeviceToHost,
                                c.stream));
    RP_CHECK_HIP(hipStreamSynchronize(c.stream));
    if (c.prof) {
        st = prof_collect();
        if (st) return st;
    }
    memcpy(y_host, hout, sizeof(float) * n * kOut);
    return RP_OK;
}

}  // extern "C"
