// rp_vec.hip -- vector kernels of libreapers_hip.so: the BLAS-1 operations
// of the reference's GPUImpl (inc/gpuimpl.h:806-1062, src/krnl.cu:25-58),
// reductions accumulated in FP64 for both element precisions, and the fused
// Gram-Schmidt / linear-combination sweeps the Krylov driver uses in place of
// one cuBLAS call per vector (inc/algo.h:86-101, inc/algo.h:342-345).
//
// All kernels are memory-bound streams with grid-stride loops.  Reductions
// keep FP64 partial sums per thread, reduce them within a wavefront with
// cross-lane shuffles, across the workgroup in LDS, and across workgroups in
// the last workgroup to arrive, in an order of its own, so every reduction is
// deterministic for a given n.
#include "rp_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace rp {

template <typename R> struct Cx;
template <> struct Cx<float> { using T = float2; };
template <> struct Cx<double> { using T = double2; };

static inline int grid_for(uint64_t units, int threads, int cap)
{
    uint64_t g = (units + threads - 1) / threads;
    if (g < 1) g = 1;
    if (g > (uint64_t)cap) g = cap;
    return (int)g;
}

constexpr int kEwThreads = 256;
constexpr int kEwMaxBlocks = 65536;
constexpr int kMaxVecs = RP_MAX_SWEEP_VECS;   // vectors per fused sweep (API limit)
constexpr int kDotChunk = 8;      // most vectors whose dots one workgroup accumulates
constexpr int kUpdChunk = 16;     // vectors an update / lincomb thread loads at once
constexpr int kWaves = kRedThreads / 64;

// basis pointers and coefficients as kernel arguments (read by scalar loads)
struct VecPtrs { const void *p[kMaxVecs]; };
struct Coefs { double c[2 * kMaxVecs]; };

// Workspace of the reductions (doubles): the partials, kDotCols for each of up
// to kDotBlocks workgroups of each row of vectors (kRedBlocks x 2 kMaxVecs + 1
// are reserved), then the results of the pass in flight:
//   [0, 2k) coefficients h; kResNorm (host only) the norm after the pass when
//   it was not fused; kResIn ||w||^2 before it; kResBeta the fused norm (0: not
//   fused); kResStop (an int) set by an Arnoldi step that needs the host, to
//   the step's number;
//   kResCount arrival counters of the dot workgroups, zero between launches
//   (for each row of workgroups one, and 16 below it, 64 bytes apart).
// The pinned host copy that the kernels write has the layout up to kResStop.
constexpr int kResNorm = 2 * kMaxVecs, kResIn = kResNorm + 1, kResBeta = kResNorm + 2,
              kResStop = kResNorm + 4, kResCount = kResNorm + 8;
constexpr int kDotRows = 16, kCountStep = 8;      // counters: doubles apart
constexpr int kResDoubles = kResCount + kDotRows * 17 * kCountStep;
static_assert(kResBeta < kHostSlot && (size_t)kResDoubles * sizeof(double) < 32 * 1024,
              "result slots");

// ---------------------------------------------------------------------------
// elementwise kernels
// ---------------------------------------------------------------------------
#define GRID_STRIDE(i, m)                                                        \
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < (m); \
         i += (uint64_t)gridDim.x * blockDim.x)

template <typename R>
__global__ void k_add(R *__restrict__ a, const R *__restrict__ b, uint64_t m)
{
    GRID_STRIDE(i, m) a[i] += b[i];
}

template <typename R>
__global__ void k_add3(R *__restrict__ r, const R *__restrict__ a, const R *__restrict__ b,
                       uint64_t m)
{
    GRID_STRIDE(i, m) r[i] = a[i] + b[i];
}

template <typename R>
__global__ void k_axpy(typename Cx<R>::T *__restrict__ y, R sr, R si,
                       const typename Cx<R>::T *__restrict__ x, uint64_t n)
{
    GRID_STRIDE(i, n) {
        auto v = x[i];
        auto o = y[i];
        o.x += sr * v.x - si * v.y;
        o.y += sr * v.y + si * v.x;
        y[i] = o;
    }
}

template <typename R>
__global__ void k_scale(typename Cx<R>::T *__restrict__ y, R sr, R si, uint64_t n)
{
    GRID_STRIDE(i, n) {
        auto v = y[i];
        typename Cx<R>::T o;
        o.x = sr * v.x - si * v.y;
        o.y = sr * v.y + si * v.x;
        y[i] = o;
    }
}

__global__ void k_f2d(double *__restrict__ d, const float *__restrict__ s, uint64_t m)
{
    GRID_STRIDE(i, m) d[i] = (double)s[i];
}

// double -> float, round to nearest or toward zero.  Toward zero is derived
// from the round-to-nearest result, which either is the truncation already or
// lies one ulp further from zero.
__global__ void k_d2f(float *__restrict__ d, const double *__restrict__ s, uint64_t m, int rz)
{
    GRID_STRIDE(i, m) {
        double v = s[i];
        float f = (float)v;
        if (rz && fabs((double)f) > fabs(v)) f = nextafterf(f, 0.0f);
        d[i] = f;
    }
}

// ---------------------------------------------------------------------------
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) + Box-Muller
// ---------------------------------------------------------------------------
__device__ inline void philox_round(uint32_t (&c)[4], uint32_t k0, uint32_t k1)
{
    const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u;
    uint64_t p0 = (uint64_t)M0 * c[0];
    uint64_t p1 = (uint64_t)M1 * c[2];
    uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
    uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
    c[0] = hi1 ^ c[1] ^ k0;
    c[1] = lo1;
    c[2] = hi0 ^ c[3] ^ k1;
    c[3] = lo0;
}

__device__ inline void philox4x32_10(uint32_t (&c)[4], uint32_t k0, uint32_t k1)
{
#pragma unroll
    for (int r = 0; r < 10; r++) {
        philox_round(c, k0, k1);
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

template <typename R>
__global__ void k_fill_normal(typename Cx<R>::T *__restrict__ v, uint64_t n, uint32_t k0,
                              uint32_t k1)
{
    GRID_STRIDE(i, n) {
        uint32_t c[4] = {(uint32_t)i, (uint32_t)(i >> 32), 0x52454150u, 0x45525321u};
        philox4x32_10(c, k0, k1);
        // two uniforms with 53 random bits each, u1 in (0, 1]
        uint64_t a = ((uint64_t)c[0] << 21) ^ (uint64_t)(c[1] >> 11);
        uint64_t b = ((uint64_t)c[2] << 21) ^ (uint64_t)(c[3] >> 11);
        double u1 = ((double)(a & ((1ull << 53) - 1)) + 1.0) * (1.0 / 9007199254740992.0);
        double u2 = (double)(b & ((1ull << 53) - 1)) * (1.0 / 9007199254740992.0);
        double r = sqrt(-2.0 * log(u1));
        double s, co;
        sincospi(2.0 * u2, &s, &co);
        typename Cx<R>::T o;
        o.x = (R)(r * co);
        o.y = (R)(r * s);
        v[i] = o;
    }
}

// ---------------------------------------------------------------------------
// reductions
// ---------------------------------------------------------------------------
__device__ inline double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Reduce NV per-thread doubles over the workgroup; the NV sums end up in
// sh[kWaves*NV + q].  sh must hold (kWaves + 1) * NV doubles.
template <int NV>
__device__ inline void block_reduce(double (&v)[NV], double *sh)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < NV; q++) v[q] = wave_sum(v[q]);
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < NV; q++) sh[wid * NV + q] = v[q];
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        double s = 0;
#pragma unroll
        for (int w = 0; w < kWaves; w++) s += sh[w * NV + threadIdx.x];
        sh[kWaves * NV + threadIdx.x] = s;
    }
    __syncthreads();
}

// sum of `nparts` rows: out[j] = sum_p partial[p*width + j], one block per j
__global__ void __launch_bounds__(kRedThreads)
k_reduce_cols(const double *__restrict__ partial, int nparts, int width, double *__restrict__ out)
{
    __shared__ double sh[(kWaves + 1) * 1];
    const int j = blockIdx.x;
    double v[1] = {0.0};
    for (int p = threadIdx.x; p < nparts; p += blockDim.x) v[0] += partial[(size_t)p * width + j];
    block_reduce<1>(v, sh);
    if (threadIdx.x == 0) out[j] = sh[kWaves];
}

// Sums of NV (a power of two up to 64) per-lane values over the wavefront by
// recursive halving: each exchange halves the values a lane carries, so NV
// sums take about 2 NV + 6 - 2 log2 NV shuffles instead of 6 NV.  On return
// v[0] of every lane l holds the sum of value l >> (6 - log2 NV).
template <int NV>
__device__ __forceinline__ void wave_multi_sum(double (&v)[NV])
{
    int off = 32;
#pragma unroll
    for (int h = NV / 2; h > 0; h >>= 1, off >>= 1) {
        const bool hi = (threadIdx.x & off) != 0;
#pragma unroll
        for (int i = 0; i < h; i++) {
            const double keep = hi ? v[i + h] : v[i], send = hi ? v[i] : v[i + h];
            v[i] = keep + __shfl_xor(send, off, 64);
        }
    }
    for (; off > 0; off >>= 1) v[0] += __shfl_xor(v[0], off, 64);
}

constexpr int pow2_at_least(int v) { return v <= 1 ? 1 : 2 * pow2_at_least((v + 1) / 2); }

// Dots of one Gram-Schmidt pass: workgroup (x, y) forms the FP64 partials of
// <V[q]|w> over its share of the elements for the KC vectors q0 = y KC ..
// (the last row of workgroups repeats the last vector past k), and row y = 0
// also ||w||^2.  The last workgroup of a row y to arrive adds the row's
// partials in an order of their own, so the result does not depend on which
// one that was, and writes res (and host, pinned memory, when given).  real:
// the imaginary parts are written as zero (Lanczos).
//
// HBM bound for vectors beyond the caches; for the short vectors of small
// chains bound by latency: the reduction by the last workgroup saves the
// separate reduction launches (4.5 us each with their gap, two to three a
// pass), the recursive halving the shuffles of the workgroup's reduction.
// At most kDotBlocks workgroups a row, so that every thread of the last one
// has all its partials in flight at once (past the caches each read takes
// about 1 us); from 2^19 elements they have 1024 threads.
constexpr int kDotBlocks = 256, kDotCols = 24;
static_assert(2 * kDotChunk + 1 <= kDotCols &&
                  kDotRows * kDotBlocks * kDotCols <= kRedBlocks * (2 * kMaxVecs + 1),
              "dot partials");
template <typename R, int KC, int NT>
__global__ void __launch_bounds__(NT)
k_gs_dots(VecPtrs V, int k, const typename Cx<R>::T *__restrict__ w, uint64_t n,
          double *__restrict__ part, double *__restrict__ res, int real,
          double *__restrict__ host, const int *__restrict__ stop)
{
    using T = typename Cx<R>::T;
    constexpr int NV = pow2_at_least(KC ? 2 * KC : 1), W = NT / 64;
    constexpr int SH = 6 - (NV == 1 ? 0 : NV == 2 ? 1 : NV == 4 ? 2 : NV == 8 ? 3 : 4);
    __shared__ double sh[W][NV + 1];
    __shared__ int last;
    if (stop && *stop) return;
    const int y = blockIdx.y, q0 = y * KC, nb = gridDim.x;
    double acc[NV], wn = 0.0;
#pragma unroll
    for (int q = 0; q < NV; q++) acc[q] = 0.0;
    const T *vp[KC ? KC : 1];
#pragma unroll
    for (int q = 0; q < KC; q++) vp[q] = (const T *)V.p[min(q0 + q, k - 1)];
    GRID_STRIDE(i, n) {
        const T e = w[i];
        T x[KC ? KC : 1];
#pragma unroll
        for (int q = 0; q < KC; q++) x[q] = vp[q][i];
        const double yr = e.x, yi = e.y;
#pragma unroll
        for (int q = 0; q < KC; q++) {
            const double xr = x[q].x, xi = x[q].y;
            acc[2 * q] += xr * yr + xi * yi;
            acc[2 * q + 1] += xr * yi - xi * yr;
        }
        wn += yr * yr + yi * yi;
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if constexpr (KC > 0) {
        wave_multi_sum<NV>(acc);
        if ((lane & ((1 << SH) - 1)) == 0) sh[wid][lane >> SH] = acc[0];
    }
    if (y == 0) {
        wn = wave_sum(wn);
        if (lane == 0) sh[wid][NV] = wn;
    }
    __syncthreads();
    // columns of this row: 2 per vector, and ||w||^2
    const int nv = KC ? 2 * min(KC, k - q0) : 0, ncol = nv + (y == 0 ? 1 : 0);
    double *rows = part + (size_t)y * kDotBlocks * kDotCols;
    auto store = [&](int c, double v) {
        const int at = c < nv ? 2 * q0 + c : kResIn;
        if (real && c < nv && (c & 1)) v = 0.0;
        res[at] = v;
        if (host) host[at] = v;
    };
    if (threadIdx.x < 64) {
        if (lane < ncol) {
            const int c = lane < nv ? lane : NV;
            double v = 0;
#pragma unroll
            for (int q = 0; q < W; q++) v += sh[q][c];
            if (nb == 1) store(lane, v);
            else put_shared(rows + blockIdx.x * kDotCols + lane, v);
        }
        if (nb > 1) {
            // Arrivals at one counter are served one after the other (256 of
            // them took 15 us): 16 counters, whose last arrivals meet at one
            double *cnt = res + kResCount + (size_t)y * 17 * kCountStep;
            const unsigned sub = blockIdx.x & 15u, subs = min(nb, 16);
            unsigned *leaf = (unsigned *)(cnt + (1 + sub) * kCountStep);
            bool l = arrive_last(leaf, ((unsigned)nb - sub + 15u) / 16u);
            if (l) {
                if (lane == 0) *leaf = 0;
                l = arrive_last((unsigned *)cnt, subs);
            }
            if (lane == 0) last = l;
        }
    }
    if (nb == 1) return;
    __syncthreads();
    if (!last) return;
    // thread (g, c): column c of every (NT / 32)-th workgroup's partials
    constexpr int G = NT / 32, PER = kDotBlocks / G;
    __shared__ double sums[G][kDotCols];
    const int c = threadIdx.x & 31, g = threadIdx.x >> 5;
    if (c < ncol) {
        double p[PER], v = 0;
#pragma unroll
        for (int i = 0; i < PER; i++)
            p[i] = g + i * G < nb ? get_shared(rows + (g + i * G) * kDotCols + c) : 0.0;
#pragma unroll
        for (int i = 0; i < PER; i++) v += p[i];
        sums[g][c] = v;
    }
    __syncthreads();
    if ((int)threadIdx.x < ncol) {
        double v = 0;
#pragma unroll
        for (int i = 0; i < G; i++) v += sums[i][threadIdx.x];
        store(threadIdx.x, v);
    }
    if (threadIdx.x == 0) *(unsigned *)(res + kResCount + (size_t)y * 17 * kCountStep) = 0;
}

// sum over q of h_q x_q for the KC vectors from p on, added to (yr, yi) or
// (SIGN < 0) subtracted from it; h uniform, read by scalar loads
template <typename R, int KC, int SIGN>
__device__ __forceinline__ void add_vectors(const VecPtrs &V, int p, const double *__restrict__ h,
                                            uint64_t i, double &yr, double &yi)
{
    using T = typename Cx<R>::T;
    T x[KC];
#pragma unroll
    for (int q = 0; q < KC; q++) x[q] = ((const T *)V.p[p + q])[i];
#pragma unroll
    for (int q = 0; q < KC; q++) {
        const double xr = x[q].x, xi = x[q].y, hr = h[2 * (p + q)], hi = h[2 * (p + q) + 1];
        if (SIGN < 0) {
            yr -= hr * xr - hi * xi;
            yi -= hr * xi + hi * xr;
        } else {
            yr += hr * xr - hi * xi;
            yi += hr * xi + hi * xr;
        }
    }
}

// w -= sum_q h_q V[q] over all k vectors (FP64 arithmetic, one rounding; KR =
// k mod 16, 16 for 0: the vectors after the full chunks of 16, LONG where
// there are any), h = res[0..2k).
// Fused normalization (fuse_min > 0): beta^2 = ||w||^2 - sum |h_q|^2 is the
// norm of the result when the basis is orthonormal; if beta^2 >= ||w||^2 / 2
// (no cancellation to speak of) and beta >= fuse_min, the result is written
// scaled by 1/beta and beta stored (else 0); otherwise the workgroups leave
// partials of the result's norm.  Block 0 copies h and beta to host.
//
// Bound by HBM; the elements are walked from the end, where the dot sweep
// just finished, so that what is left of the basis in the 256 MB Infinity
// Cache is read from there.
template <typename R, int KR, bool LONG>
__global__ void __launch_bounds__(kRedThreads)
k_gs_update(VecPtrs V, int k, typename Cx<R>::T *__restrict__ w, uint64_t n,
            double *__restrict__ part, const double *__restrict__ hc, double *res, double fuse_min,
            double *__restrict__ host, const int *__restrict__ stop)
{
    using T = typename Cx<R>::T;
    __shared__ double sh[(kWaves + 1) * 1];
    __shared__ double fbeta;
    if (stop && *stop) return;
    if (threadIdx.x < 64) {
        const int q = threadIdx.x;
        const double hr = q < k ? hc[2 * q] : 0.0, hi = q < k ? hc[2 * q + 1] : 0.0;
        if (blockIdx.x == 0 && q < k) {
            host[2 * q] = hr;
            host[2 * q + 1] = hi;
        }
        double beta = 0.0;
        if (fuse_min > 0) {
            const double s2 = wave_sum(hr * hr + hi * hi), wn2 = hc[kResIn], b2 = wn2 - s2;
            if (b2 > 0 && b2 >= 0.5 * wn2 && sqrt(b2) >= fuse_min) beta = sqrt(b2);
        }
        if (q == 0) {
            fbeta = beta;
            if (blockIdx.x == 0) {
                res[kResBeta] = beta;
                host[kResBeta] = beta;
            }
        }
    }
    __syncthreads();
    const double beta = fbeta, f = beta > 0 ? 1.0 / beta : 1.0;
    double nacc[1] = {0.0};
    const uint64_t rows = (n + kRedThreads - 1) / kRedThreads;
    for (uint64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const uint64_t i = (rows - 1 - r) * kRedThreads + threadIdx.x;
        if (i >= n) continue;
        const T e = w[i];
        double yr = e.x, yi = e.y;
        int p = 0;
        if constexpr (LONG)
            for (; p + kUpdChunk < k; p += kUpdChunk)
                add_vectors<R, kUpdChunk, -1>(V, p, hc, i, yr, yi);
        add_vectors<R, KR, -1>(V, p, hc, i, yr, yi);
        T o;
        o.x = (R)(yr * f);
        o.y = (R)(yi * f);
        w[i] = o;
        const double orr = o.x, oi = o.y;
        nacc[0] += orr * orr + oi * oi;
    }
    if (beta == 0) {
        block_reduce<1>(nacc, sh);
        if (threadIdx.x == 0) part[blockIdx.x] = sh[kWaves];
    }
}

// The end of a pass that was not fused (nothing to do after one that was):
// every workgroup adds the nb norm partials in the same order; block 0 gives
// the norm to res (and as the second coefficient of a Lanczos step behind)
// and to host.  With scale, w is divided by the norm unless it is below
// min_norm or not a number: then stop is set for the Arnoldi steps queued
// behind, and w left as the pass made it.
template <typename R>
__global__ void __launch_bounds__(kRedThreads)
k_gs_finish(typename Cx<R>::T *__restrict__ w, uint64_t n, const double *__restrict__ part, int nb,
            double *res, int scale, double min_norm, double *__restrict__ host, int *stop, int step)
{
    __shared__ double sh[(kWaves + 1) * 1];
    if (res[kResBeta] > 0) return;
    if (stop) {
        const int s = *(volatile int *)stop;
        if (s && s != step) return;
    }
    double v[1] = {0.0};
    for (int p = threadIdx.x; p < nb; p += kRedThreads) v[0] += part[p];
    block_reduce<1>(v, sh);
    const double norm = sqrt(sh[kWaves]);
    const bool ok = norm >= min_norm;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        res[2] = norm;
        res[3] = 0.0;
        host[kResNorm] = norm;
        if (scale && !ok && stop) *(volatile int *)stop = step;
    }
    if (!scale || !ok) return;
    const R f = (R)(1.0 / norm);
    GRID_STRIDE(i, n) {
        auto e = w[i];
        e.x *= f;
        e.y *= f;
        w[i] = e;
    }
}

// y += sum_q c[q] V[q] over k vectors (FP64 arithmetic, one rounding; KR as
// in k_gs_update)
template <typename R, int KR, bool LONG>
__global__ void __launch_bounds__(kRedThreads)
k_lincomb(VecPtrs V, Coefs c, int k, typename Cx<R>::T *__restrict__ y, uint64_t n)
{
    using T = typename Cx<R>::T;
    GRID_STRIDE(i, n) {
        T o = y[i];
        double yr = o.x, yi = o.y;
        int p = 0;
        if constexpr (LONG)
            for (; p + kUpdChunk < k; p += kUpdChunk)
                add_vectors<R, kUpdChunk, 1>(V, p, c.c, i, yr, yi);
        add_vectors<R, KR, 1>(V, p, c.c, i, yr, yi);
        o.x = (R)yr;
        o.y = (R)yi;
        y[i] = o;
    }
}

// ---------------------------------------------------------------------------
// host helpers
// ---------------------------------------------------------------------------
constexpr size_t kPartDoubles = (size_t)kRedBlocks * (2 * kMaxVecs + 1);
static inline double *ws_partial() { return (double *)ctx().work; }
static inline double *ws_result() { return ws_partial() + kPartDoubles; }

// The Gram-Schmidt pass's workspace in a file-scope device array, for
// rp_gs_pass_fused_noalloc: the partials and results of the library
// workspace layout above, 1.08 MB.  Each device holds its own copy; the
// host reaches it only through the address hipGetSymbolAddress returns for
// the current device (taken once per device at rp_init).
static __device__ __align__(256) double scratch[kPartDoubles + kResDoubles];
static std::vector<double *> g_scratch_ptr;     // per device, null until set up

int vec_scratch_setup(int device)
{
    if (device < 0) return set_error(RP_ERR_INVALID_ARGUMENT, "bad device %d", device);
    // the arrival counters and the stop flag start at zero
    RP_CHECK_HIP(hipMemsetAsync(ws_result(), 0, kResDoubles * sizeof(double), ctx().stream));
    RP_CHECK_HIP(hipStreamSynchronize(ctx().stream));
    if ((size_t)device >= g_scratch_ptr.size()) g_scratch_ptr.resize(device + 1, nullptr);
    if (g_scratch_ptr[device]) return RP_OK;
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        return set_error(RP_ERR_RUNTIME, "hipGetSymbolAddress(scratch) failed: %s",
                         hipGetErrorString(e));
    g_scratch_ptr[device] = (double *)p;
    return RP_OK;
}

static double *vec_scratch(int device)
{
    if (device < 0 || (size_t)device >= g_scratch_ptr.size()) return nullptr;
    return g_scratch_ptr[device];
}

// wait for the queued kernels: their results are then in pinned host memory
static int wait_results()
{
    RP_CHECK_HIP(hipStreamSynchronize(ctx().stream));
    prof_collect();
    return RP_OK;
}

// launch kernel K<R, KC> for a runtime chunk width kc in [1, 16]
#define RP_KC_SWITCH(kc, LAUNCH)                                                  \
    switch (kc) {                                                                 \
    case 1: LAUNCH(1); break;   case 2: LAUNCH(2); break;                         \
    case 3: LAUNCH(3); break;   case 4: LAUNCH(4); break;                         \
    case 5: LAUNCH(5); break;   case 6: LAUNCH(6); break;                         \
    case 7: LAUNCH(7); break;   case 8: LAUNCH(8); break;                         \
    case 9: LAUNCH(9); break;   case 10: LAUNCH(10); break;                       \
    case 11: LAUNCH(11); break; case 12: LAUNCH(12); break;                       \
    case 13: LAUNCH(13); break; case 14: LAUNCH(14); break;                       \
    case 15: LAUNCH(15); break; default: LAUNCH(16); break;                       \
    }

// queue the dots of w against V[0..k) and ||w||^2 (k = 0: only that).  Each
// workgroup takes up to 8 vectors (w is read once for all of them), 4 where
// the vectors are so short that more workgroups matter more.  At most
// kDotBlocks of them, of 1024 threads where 256 would each walk too many
// elements in series: from 2^19, with one or two vectors from 2^17 (2^19
// complex<double> elements: a dot product 19.2 -> 18.5 us with its wait).
template <typename R>
static int dots_launch(int cls, const VecPtrs &P, int k, const void *w, uint64_t n, double *work,
                       int real, double *host, const int *stop)
{
    using T = typename Cx<R>::T;
    const int most = n <= (1u << 15) ? kDotChunk / 2 : kDotChunk;
    const int rows = k > 0 ? (k + most - 1) / most : 1;
    const int kc = (k + rows - 1) / rows;
    const int nt = n <= (kc <= 2 ? 1u << 17 : 1u << 19) ? 256 : 1024;
    const dim3 grid((unsigned)std::min<uint64_t>((n + nt - 1) / nt, kDotBlocks), rows);
    double *res = work + kPartDoubles;
#define RP_DOTS(KC)                                                               \
    if (nt == 256)                                                                \
        RP_LAUNCH(cls, (k_gs_dots<R, KC, 256>), grid, dim3(256), 0, P, k, (const T *)w, n, work,   \
                  res, real, host, stop);                                         \
    else                                                                          \
        RP_LAUNCH(cls, (k_gs_dots<R, KC, 1024>), grid, dim3(1024), 0, P, k, (const T *)w, n, work, \
                  res, real, host, stop);                                         \
    break
    switch (kc) {
    case 0: RP_DOTS(0);
    case 1: RP_DOTS(1);
    case 2: RP_DOTS(2);
    case 3: RP_DOTS(3);
    case 4: RP_DOTS(4);
    case 5: RP_DOTS(5);
    case 6: RP_DOTS(6);
    case 7: RP_DOTS(7);
    default: RP_DOTS(8);
    }
#undef RP_DOTS
    return RP_OK;
}

// queue the update of w by V[0..k) and the end of the pass
template <typename R>
static int update_launch(const VecPtrs &P, int k, void *w, uint64_t n, double *work, double *host,
                         double fuse_min, int scale, double min_norm, int *stop, int step)
{
    using T = typename Cx<R>::T;
    const int nb = grid_for(n, kRedThreads, kRedBlocks), kr = (k - 1) % kUpdChunk + 1;
    double *res = work + kPartDoubles;
#define RP_UPD(KR)                                                                \
    RP_LAUNCH(RP_KERNEL_GS, (k_gs_update<R, KR, false>), dim3(nb), dim3(kRedThreads), 0, P, k,     \
              (T *)w, n, work, (const double *)res, res, fuse_min, host, (const int *)stop)
#define RP_UPD_LONG(KR)                                                           \
    RP_LAUNCH(RP_KERNEL_GS, (k_gs_update<R, KR, true>), dim3(nb), dim3(kRedThreads), 0, P, k,      \
              (T *)w, n, work, (const double *)res, res, fuse_min, host, (const int *)stop)
    if (k <= kUpdChunk) {
        RP_KC_SWITCH(kr, RP_UPD)
    } else {
        RP_KC_SWITCH(kr, RP_UPD_LONG)
    }
#undef RP_UPD
#undef RP_UPD_LONG
    RP_LAUNCH(RP_KERNEL_GS, k_gs_finish<R>, dim3(scale ? nb : 1), dim3(kRedThreads), 0, (T *)w, n,
              (const double *)work, nb, res, scale, min_norm, host, stop, step);
    return RP_OK;
}

// One Gram-Schmidt pass.  pre / pre_rows: the dot partials of w already
// formed by the apply's epilogue (rows of 2 kMaxVecs + 1 doubles, ||w||^2 in
// the last column); the pass then starts from their reduction
template <typename R>
static int gs_pass_impl(const void *const *V, int k, void *w, uint64_t n, double *h,
                        double *norm, double fuse_min, int *normalized, double *work = nullptr,
                        const double *pre = nullptr, uint64_t pre_rows = 0)
{
    double *host = ctx().pinned;
    if (!work) work = ws_partial();
    double *res = work + kPartDoubles;
    VecPtrs P{};
    for (int q = 0; q < k; q++) P.p[q] = V[q];
    int st;
    if (pre) {
        const int width = 2 * kMaxVecs + 1;
        if (k > 0)
            RP_LAUNCH(RP_KERNEL_GS, k_reduce_cols, dim3(2 * k), dim3(kRedThreads), 0, pre,
                      (int)pre_rows, width, res);
        RP_LAUNCH(RP_KERNEL_GS, k_reduce_cols, dim3(1), dim3(kRedThreads), 0, pre + 2 * kMaxVecs,
                  (int)pre_rows, width, k > 0 ? res + kResIn : host + kResIn);
    } else if ((st = dots_launch<R>(RP_KERNEL_GS, P, k, w, n, work, 0,
                                    k > 0 ? nullptr : host, nullptr))) {
        return st;
    }
    if (k > 0 &&
        (st = update_launch<R>(P, k, w, n, work, host, fuse_min, 0, 0.0, (int *)nullptr, 0)))
        return st;
    if ((st = wait_results())) return st;
    for (int q = 0; q < 2 * k; q++) h[q] = host[q];
    const double beta = k > 0 ? host[kResBeta] : 0.0;
    if (normalized) *normalized = beta > 0 ? 1 : 0;
    *norm = k == 0 ? sqrt(host[kResIn]) : beta > 0 ? beta : host[kResNorm];
    return RP_OK;
}

template <typename R>
static int dot_impl(const void *a, const void *b, uint64_t n, double *out2)
{
    double *host = ctx().pinned;
    VecPtrs P{};
    P.p[0] = a;
    int st = dots_launch<R>(RP_KERNEL_OTHER, P, 1, b, n, ws_partial(), 0, host, nullptr);
    if (st || (st = wait_results())) return st;
    out2[0] = host[0];
    out2[1] = host[1];
    return RP_OK;
}

template <typename R>
static int nrm2_impl(const void *a, uint64_t n, double *nrm)
{
    double *host = ctx().pinned;
    int st = dots_launch<R>(RP_KERNEL_OTHER, VecPtrs{}, 0, a, n, ws_partial(), 0, host, nullptr);
    if (st || (st = wait_results())) return st;
    *nrm = sqrt(host[kResIn]);
    return RP_OK;
}

// Steps j0 .. m-1 of an Arnoldi (or Lanczos) recurrence queued without a wait
// between them: every step applies, forms its coefficients, updates and
// normalizes on the device and leaves its results in a pinned slot of its
// own; one wait ends them all.  A step whose norm is below min_norm raises
// the stop flag, which every kernel queued behind it reads first.
template <typename R>
static int steps_impl(rp_terms_t hd, void *const *V, int j0, int m, uint64_t n, double min_norm,
                      int lanczos)
{
    Context &c = ctx();
    double *work = ws_partial(), *res = ws_result();
    int *stop = lanczos ? nullptr : (int *)(res + kResStop);
    int st = RP_OK;
    VecPtrs P{};
    if (!lanczos)
        for (int j = 0; j < j0; j++) P.p[j] = V[j];
    for (int j = j0; j < m; j++) {
        double *host = c.pinned + kHostSteps + (size_t)(j - j0) * kHostSlot;
        // not reached before the stop: neither normalized nor a norm
        host[kResBeta] = 0;
        host[kResNorm] = 0;
    }
    for (int j = j0; j < m; j++) {
        double *host = c.pinned + kHostSteps + (size_t)(j - j0) * kHostSlot;
        if ((st = apply_queued(hd, V[j + 1], V[j], stop))) break;
        if (lanczos) {
            P.p[0] = V[j];
            P.p[1] = j > j0 ? V[j - 1] : nullptr;
            if ((st = dots_launch<R>(RP_KERNEL_GS, P, 1, V[j + 1], n, work, 1, host, stop))) break;
            if (j == m - 1) break;
            st = update_launch<R>(P, j > j0 ? 2 : 1, V[j + 1], n, work, host, 0.0, 1, 0.0, stop, 0);
        } else {
            P.p[j] = V[j];
            if ((st = dots_launch<R>(RP_KERNEL_GS, P, j + 1, V[j + 1], n, work, 0, nullptr,
                                     stop))) break;
            st = update_launch<R>(P, j + 1, V[j + 1], n, work, host, min_norm, 1, min_norm, stop,
                                  j + 1);
        }
        if (st) break;
    }
    const int wst = wait_results();
    if (st || wst) return st ? st : wst;
    return RP_OK;
}

template <typename R>
static int lincomb_impl(void *y, const void *const *V, int k, const double *c, uint64_t n)
{
    using T = typename Cx<R>::T;
    const int nb = grid_for(n, kRedThreads, kRedBlocks);
    for (int q0 = 0; q0 < k; q0 += kMaxVecs) {
        const int kc = k - q0 < kMaxVecs ? k - q0 : kMaxVecs, kr = (kc - 1) % kUpdChunk + 1;
        VecPtrs P{};
        Coefs C{};
        for (int q = 0; q < kc; q++) {
            P.p[q] = V[q0 + q];
            C.c[2 * q] = c[2 * (q0 + q)];
            C.c[2 * q + 1] = c[2 * (q0 + q) + 1];
        }
#define RP_LC(KR)                                                                 \
    RP_LAUNCH(RP_KERNEL_OTHER, (k_lincomb<R, KR, false>), dim3(nb), dim3(kRedThreads), 0, P, C, kc,\
              (T *)y, n)
#define RP_LC_LONG(KR)                                                            \
    RP_LAUNCH(RP_KERNEL_OTHER, (k_lincomb<R, KR, true>), dim3(nb), dim3(kRedThreads), 0, P, C, kc, \
              (T *)y, n)
        if (kc <= kUpdChunk) {
            RP_KC_SWITCH(kr, RP_LC)
        } else {
            RP_KC_SWITCH(kr, RP_LC_LONG)
        }
#undef RP_LC
#undef RP_LC_LONG
    }
    return RP_OK;
}

}  // namespace rp

using namespace rp;

extern "C" {

int rp_zero_vec(int prec, void *v, uint64_t n)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    if (n == 0) return RP_OK;
    RP_REQUIRE(v, "null vector");
    RP_CHECK_HIP(hipMemsetAsync(v, 0, n * elem_bytes(prec), ctx().stream));
    return RP_OK;
}

int rp_copy_vec(int dst_prec, void *dst, int src_prec, const void *src, uint64_t n, int rounding)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(dst_prec) && valid_prec(src_prec), "bad precision");
    if (n == 0) return RP_OK;
    RP_REQUIRE(dst && src, "null vector");
    uint64_t m = 2 * n;
    int g = grid_for(m, kEwThreads, kEwMaxBlocks);
    if (dst_prec == src_prec) {
        RP_CHECK_HIP(hipMemcpyAsync(dst, src, n * elem_bytes(dst_prec), hipMemcpyDeviceToDevice,
                                    ctx().stream));
    } else if (dst_prec == RP_C128) {
        RP_LAUNCH(RP_KERNEL_OTHER, k_f2d, dim3(g), dim3(kEwThreads), 0, (double *)dst,
                  (const float *)src, m);
    } else {
        RP_REQUIRE(rounding == RP_ROUND_NEAREST || rounding == RP_ROUND_TOWARD_ZERO,
                   "bad rounding mode");
        RP_LAUNCH(RP_KERNEL_OTHER, k_d2f, dim3(g), dim3(kEwThreads), 0, (float *)dst,
                  (const double *)src, m, rounding == RP_ROUND_TOWARD_ZERO ? 1 : 0);
    }
    return RP_OK;
}

int rp_add_vec(int prec, void *v0, const void *v1, uint64_t n)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    if (n == 0) return RP_OK;
    RP_REQUIRE(v0 && v1, "null vector");
    uint64_t m = 2 * n;
    int g = grid_for(m, kEwThreads, kEwMaxBlocks);
    if (prec == RP_C64)
        RP_LAUNCH(RP_KERNEL_OTHER, k_add<float>, dim3(g), dim3(kEwThreads), 0, (float *)v0,
                  (const float *)v1, m);
    else
        RP_LAUNCH(RP_KERNEL_OTHER, k_add<double>, dim3(g), dim3(kEwThreads), 0, (double *)v0,
                  (const double *)v1, m);
    return RP_OK;
}

int rp_add_vec3(int prec, void *res, const void *v0, const void *v1, uint64_t n)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    if (n == 0) return RP_OK;
    RP_REQUIRE(res && v0 && v1, "null vector");
    uint64_t m = 2 * n;
    int g = grid_for(m, kEwThreads, kEwMaxBlocks);
    if (prec == RP_C64)
        RP_LAUNCH(RP_KERNEL_OTHER, k_add3<float>, dim3(g), dim3(kEwThreads), 0, (float *)res,
                  (const float *)v0, (const float *)v1, m);
    else
        RP_LAUNCH(RP_KERNEL_OTHER, k_add3<double>, dim3(g), dim3(kEwThreads), 0, (double *)res,
                  (const double *)v0, (const double *)v1, m);
    return RP_OK;
}

int rp_axpy(int prec, void *v0, double s_re, double s_im, const void *v1, uint64_t n)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    if (n == 0) return RP_OK;
    RP_REQUIRE(v0 && v1, "null vector");
    int g = grid_for(n, kEwThreads, kEwMaxBlocks);
    if (prec == RP_C64)
        RP_LAUNCH(RP_KERNEL_OTHER, k_axpy<float>, dim3(g), dim3(kEwThreads), 0, (float2 *)v0,
                  (float)s_re, (float)s_im, (const float2 *)v1, n);
    else
        RP_LAUNCH(RP_KERNEL_OTHER, k_axpy<double>, dim3(g), dim3(kEwThreads), 0, (double2 *)v0,
                  s_re, s_im, (const double2 *)v1, n);
    return RP_OK;
}

int rp_scale_vec(int prec, void *v, double s_re, double s_im, uint64_t n)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    if (n == 0) return RP_OK;
    RP_REQUIRE(v, "null vector");
    int g = grid_for(n, kEwThreads, kEwMaxBlocks);
    if (prec == RP_C64)
        RP_LAUNCH(RP_KERNEL_OTHER, k_scale<float>, dim3(g), dim3(kEwThreads), 0, (float2 *)v,
                  (float)s_re, (float)s_im, n);
    else
        RP_LAUNCH(RP_KERNEL_OTHER, k_scale<double>, dim3(g), dim3(kEwThreads), 0, (double2 *)v,
                  s_re, s_im, n);
    return RP_OK;
}

int rp_vec_prod(int prec, const void *v0, const void *v1, uint64_t n, double *re, double *im)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    RP_REQUIRE(re && im, "null output");
    if (n == 0) { *re = 0; *im = 0; return RP_OK; }
    RP_REQUIRE(v0 && v1, "null vector");
    double out[2];
    st = prec == RP_C64 ? dot_impl<float>(v0, v1, n, out) : dot_impl<double>(v0, v1, n, out);
    if (st) return st;
    *re = out[0];
    *im = out[1];
    return RP_OK;
}

int rp_vec_norm(int prec, const void *v, uint64_t n, double *nrm)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    RP_REQUIRE(nrm, "null output");
    if (n == 0) { *nrm = 0; return RP_OK; }
    RP_REQUIRE(v, "null vector");
    return prec == RP_C64 ? nrm2_impl<float>(v, n, nrm) : nrm2_impl<double>(v, n, nrm);
}

int rp_init_random(int prec, void *v, uint64_t n, uint64_t seed)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    if (n == 0) return RP_OK;
    RP_REQUIRE(v, "null vector");
    int g = grid_for(n, kEwThreads, kEwMaxBlocks);
    if (prec == RP_C64)
        RP_LAUNCH(RP_KERNEL_OTHER, k_fill_normal<float>, dim3(g), dim3(kEwThreads), 0,
                  (float2 *)v, n, (uint32_t)seed, (uint32_t)(seed >> 32));
    else
        RP_LAUNCH(RP_KERNEL_OTHER, k_fill_normal<double>, dim3(g), dim3(kEwThreads), 0,
                  (double2 *)v, n, (uint32_t)seed, (uint32_t)(seed >> 32));
    double nrm;
    st = rp_vec_norm(prec, v, n, &nrm);
    if (st) return st;
    return rp_scale_vec(prec, v, 1.0 / nrm, 0.0, n);
}

int rp_gs_pass(int prec, const void *const *V, int k, void *w, uint64_t n, double *h,
               double *norm)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    RP_REQUIRE(k >= 0 && k <= kMaxVecs, "k must be in [0, 64]");
    RP_REQUIRE(norm && (k == 0 || (h && V)), "null argument");
    RP_REQUIRE(w || n == 0, "null vector");
    for (int q = 0; q < k; q++) RP_REQUIRE(V[q], "null basis vector");
    if (n == 0) {
        for (int q = 0; q < 2 * k; q++) h[q] = 0;
        *norm = 0;
        return RP_OK;
    }
    return prec == RP_C64 ? gs_pass_impl<float>(V, k, w, n, h, norm, 0.0, nullptr)
                          : gs_pass_impl<double>(V, k, w, n, h, norm, 0.0, nullptr);
}

int rp_gs_pass_fused(int prec, const void *const *V, int k, void *w, uint64_t n, double *h,
                     double *norm, double fuse_min, int *normalized)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    RP_REQUIRE(k >= 0 && k <= kMaxVecs, "k must be in [0, 64]");
    RP_REQUIRE(norm && normalized && (k == 0 || (h && V)), "null argument");
    RP_REQUIRE(w || n == 0, "null vector");
    for (int q = 0; q < k; q++) RP_REQUIRE(V[q], "null basis vector");
    *normalized = 0;
    if (n == 0) {
        for (int q = 0; q < 2 * k; q++) h[q] = 0;
        *norm = 0;
        return RP_OK;
    }
    return prec == RP_C64 ? gs_pass_impl<float>(V, k, w, n, h, norm, fuse_min, normalized)
                          : gs_pass_impl<double>(V, k, w, n, h, norm, fuse_min, normalized);
}

int rp_gs_pass_fused_noalloc(int prec, const void *const *V, int k, void *w, uint64_t n,
                             double *h, double *norm, double fuse_min, int *normalized)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    RP_REQUIRE(k >= 0 && k <= kMaxVecs,
               "k must be in [0, 64]: the fixed scratch holds partials of 64 basis vectors");
    RP_REQUIRE(norm && normalized && (k == 0 || (h && V)), "null argument");
    RP_REQUIRE(w || n == 0, "null vector");
    for (int q = 0; q < k; q++) RP_REQUIRE(V[q], "null basis vector");
    double *work = vec_scratch(ctx().device);
    if (!work)
        return set_error(RP_ERR_RUNTIME, "rp_gs_pass_fused_noalloc: no scratch on device %d",
                         ctx().device);
    *normalized = 0;
    if (n == 0) {
        for (int q = 0; q < 2 * k; q++) h[q] = 0;
        *norm = 0;
        return RP_OK;
    }
    return prec == RP_C64 ? gs_pass_impl<float>(V, k, w, n, h, norm, fuse_min, normalized, work)
                          : gs_pass_impl<double>(V, k, w, n, h, norm, fuse_min, normalized, work);
}

int rp_apply_gs(rp_terms_t hd, void *res, const void *vec, const void *const *V, int k,
                double *h, double *norm, double fuse_min, int *normalized)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(hd, "null term handle");
    RP_REQUIRE(res && vec && res != vec, "res and vec must be different non-null buffers");
    RP_REQUIRE(k >= 0 && k <= kMaxVecs, "k must be in [0, 64]");
    RP_REQUIRE(norm && normalized && (k == 0 || (h && V)), "null argument");
    for (int q = 0; q < k; q++) {
        RP_REQUIRE(V[q], "null basis vector");
        RP_REQUIRE(V[q] != res, "res must not be one of the basis vectors");
    }
    rp_terms_info_t info;
    if ((st = rp_terms_info(hd, &info))) return st;
    const uint64_t n = 1ull << info.len;
    *normalized = 0;
    Context &c = ctx();
    const int width = 2 * kMaxVecs + 1;
    // partial rows for up to 2^16 workgroups (2^28 amplitudes at 2^12 per tile)
    const uint64_t max_rows = 1ull << 16;
    const uint64_t want = (n >> 12) < max_rows ? (n >> 12) : max_rows;
    const size_t need = (size_t)want * width * sizeof(double);
    if (want && c.epi_bytes < need) {
        if (c.epi_work) {
            RP_CHECK_HIP(hipStreamSynchronize(c.stream));
            (void)hipFree(c.epi_work);
        }
        c.epi_work = nullptr;
        c.epi_bytes = 0;
        if (dev_malloc(&c.epi_work, need) != hipSuccess) {
            (void)hipGetLastError();
            c.epi_work = nullptr;
        } else {
            c.epi_bytes = need;
        }
    }
    uint64_t rows = 0;
    if (c.epi_work) {
        st = apply_dots_launch(hd, res, vec, V, k, (double *)c.epi_work, width,
                               c.epi_bytes / (width * sizeof(double)), &rows);
        if (st) return st;
    }
    if (rows == 0) {
        if ((st = rp_apply_ops(hd, res, vec, 0))) return st;
        return rp_gs_pass_fused(info.prec, V, k, res, n, h, norm, fuse_min, normalized);
    }
    return info.prec == RP_C64
               ? gs_pass_impl<float>(V, k, res, n, h, norm, fuse_min, normalized, nullptr,
                                     (const double *)c.epi_work, rows)
               : gs_pass_impl<double>(V, k, res, n, h, norm, fuse_min, normalized, nullptr,
                                      (const double *)c.epi_work, rows);
}

static int steps_check(rp_terms_t hd, void *const *V, int j0, int m, const double *out,
                       rp_terms_info_t *info)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(hd, "null term handle");
    RP_REQUIRE(V && out, "null argument");
    RP_REQUIRE(j0 >= 0 && j0 < m && m <= kMaxVecs, "need 0 <= j0 < m <= 64");
    for (int j = 0; j <= m; j++) {
        RP_REQUIRE(V[j], "null basis vector");
        RP_REQUIRE(j == 0 || V[j] != V[j - 1], "consecutive vectors must be different buffers");
    }
    return rp_terms_info(hd, info);
}

int rp_arnoldi_steps(rp_terms_t hd, void *const *V, int j0, int m, double min_norm, double *out,
                     int *done)
{
    rp_terms_info_t info;
    int st = steps_check(hd, V, j0, m, out, &info);
    if (st) return st;
    RP_REQUIRE(done, "null argument");
    RP_REQUIRE(min_norm > 0, "min_norm must be positive");
    for (int j = 0; j <= m; j++)
        for (int i = 0; i < j; i++) RP_REQUIRE(V[i] != V[j], "vectors must be different buffers");
    const uint64_t n = 1ull << info.len;
    st = info.prec == RP_C64 ? steps_impl<float>(hd, V, j0, m, n, min_norm, 0)
                             : steps_impl<double>(hd, V, j0, m, n, min_norm, 0);
    const double *slots = ctx().pinned + kHostSteps;
    *done = 0;
    bool raised = st != RP_OK;
    for (int j = j0; j < m && !raised; j++) {
        const double *s = slots + (size_t)(j - j0) * kHostSlot, beta = s[kResBeta];
        double *o = out + (size_t)(j - j0) * RP_STEP_DOUBLES;
        for (int q = 0; q < 2 * (j + 1); q++) o[q] = s[q];
        o[2 * kMaxVecs] = beta > 0 ? beta : s[kResNorm];
        o[2 * kMaxVecs + 1] = beta > 0 ? 1.0 : 0.0;
        (*done)++;
        raised = !(beta > 0 || s[kResNorm] >= min_norm);
    }
    // the stop flag is taken down for the next call
    if (raised)
        RP_CHECK_HIP(hipMemsetAsync(ws_result() + kResStop, 0, sizeof(double), ctx().stream));
    return st;
}

int rp_lanczos_steps(rp_terms_t hd, void *const *V, int m, double *alpha, double *beta)
{
    rp_terms_info_t info;
    int st = steps_check(hd, V, 0, m, alpha, &info);
    if (st) return st;
    RP_REQUIRE(m == 1 || beta, "null argument");
    for (int j = 2; j <= m; j++) RP_REQUIRE(V[j] != V[j - 2], "vectors must be different buffers");
    const uint64_t n = 1ull << info.len;
    st = info.prec == RP_C64 ? steps_impl<float>(hd, V, 0, m, n, 0.0, 1)
                             : steps_impl<double>(hd, V, 0, m, n, 0.0, 1);
    if (st) return st;
    for (int j = 0; j < m; j++) {
        const double *s = ctx().pinned + kHostSteps + (size_t)j * kHostSlot;
        alpha[j] = s[0];
        if (j < m - 1) beta[j] = s[kResNorm];
    }
    return RP_OK;
}

int rp_lincomb(int prec, void *y, const void *const *V, int k, const double *c, uint64_t n)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    RP_REQUIRE(k >= 0, "k must not be negative");
    if (n == 0 || k == 0) return RP_OK;
    RP_REQUIRE(y && V && c, "null argument");
    for (int q = 0; q < k; q++) RP_REQUIRE(V[q], "null basis vector");
    return prec == RP_C64 ? lincomb_impl<float>(y, V, k, c, n)
                          : lincomb_impl<double>(y, V, k, c, n);
}

}  // extern "C"
