// rp_apply.hip -- the matrix-free Pauli-sum apply of libreapers_hip.so.
//
// Reference: DevSumOps::upload (inc/gpuimpl.h:1064-1085) copies the raw
// SpinOp array to the device and krnl_apply_ops (src/krnl.cu:80-94) runs one
// thread per output amplitude that walks every term's 2-bit-per-site string
// (SpinOp::apply, inc/ops.h:421-440):
//
//     res[m] += coeff * (-1)^popcount((m ^ x) & z) * vec[m ^ x]
//
// Here the upload does the per-term bit work once on the host:
//   x = flip mask (X bits, even positions of SpinOp::bits),
//   z = phase mask (Z bits, odd positions),
//   c = coeff * (-1)^popcount(x & z), so that
//     res[m] += c * (-1)^popcount(m & z) * vec[m ^ x],
// and sorts the terms by x.  Terms with equal x ("subs") share one gather of
// vec; subs whose x agree above the tile bits b ("groups") share one staged
// input tile.  A Hermitian term has c purely real or purely imaginary, so
// single-term subs are classified real / imaginary / complex on the host and
// the kernel spends 2 FMAs (not 4) per term and amplitude on the first two.
//
// Tiled kernel: one workgroup of NT threads owns the output tile
// [t0, t0 + 2^b); thread tid holds amplitudes t0 + r*NT + tid, r < RP (in
// k_apply_stream pairs of neighbours, see stream_row).  For each group it stages
// the input tile t0 ^ (xh << b) in LDS with coalesced loads (an XOR with the
// high part maps an aligned tile onto an aligned tile), then applies every sub of the group from LDS: the low bits of x
// permute lanes (tid ^ (x mod NT)) and rows (r ^ (x / NT)).  The sign
// (-1)^popcount(m & z) splits into a per-workgroup part (t0 & z), a per-lane
// part (tid & z) computed once per sub, and a per-row part (r*NT & z) that is
// uniform across the wavefront.  The output accumulates in registers (FP64
// for both state precisions by default) and is written once, with the
// caller's zero_vec fused in when accumulate == 0.
// Workgroups are numbered so that each XCD walks a contiguous range of
// output tiles, whose input tiles overlap in that XCD's L2.
// HBM traffic per apply: (G_b + 1) * 2^len * S bytes, G_b = number of groups.
#include "rp_internal.h"
#include "rp_tables.h"

#include <algorithm>
#include <type_traits>
#include <cstring>
#include <vector>

namespace rp {

constexpr int kSmallThreads = 256;

}  // namespace rp

struct rp_terms {
    int prec = RP_C64;
    int len = 0;
    int tile_bits = 0;       // 0: no tiles (k_apply_wave)
    int threads = 0;         // workgroup size of the tiled kernel
    int depth = 2;           // LDS tiles in the tiled kernel's pipeline; without
                             // tiles the number of term slices (1: none)
    int acc64 = 1;           // accumulate in FP64
    int group_acc = 0;       // FP32 within a group, FP64 across groups (complex<float>)
    uint64_t nterms = 0, nflips = 0, ngroups = 0, nsubs = 0;
    rp::TileMap tmap{};               // output-tile order of the tiled kernels
    void *d_groups = nullptr, *d_subs = nullptr, *d_terms = nullptr;
    void *d_wflips = nullptr, *d_wsubs = nullptr, *d_wterms = nullptr, *d_wcut = nullptr;
                                      // k_apply_wave
    void *d_cgroups = nullptr, *d_csubs = nullptr, *d_cterms = nullptr;   // compact stream
    void *d_split = nullptr;          // per-slice partial sums of k_apply_wave and
                                      // the arrival counters behind them
    int rows = 1;                     // its amplitudes per lane
    double apply_passes = 0;          // measured apply cost in state passes (autotune)
    std::vector<uint64_t> raw_bits;   // the uploaded term list, for re-tiling
    std::vector<double> raw_coeff;
};

namespace rp {

// XCD-aware numbering: consecutive workgroup ids go to different XCDs, so
// give each XCD a contiguous range of tiles
__device__ __forceinline__ uint32_t xcd_tile_index()
{
    const uint32_t nb = gridDim.x, b = blockIdx.x;
    return (nb & 7u) == 0 ? (b & 7u) * (nb >> 3) + (b >> 3) : b;
}

// ---------------------------------------------------------------------------
// The apply without tiles: a wavefront owns 64 ROWS consecutive amplitudes
// (lane l the amplitudes r 64 + l of them) and gathers the input amplitudes of
// one flip mask after the other straight from memory; the XOR keeps each
// gather inside an aligned block of 64, so it is coalesced.  The terms that
// share a flip mask are first summed to the coefficient they have at each
// amplitude, d(m) = sum c (-1)^popcount(m & z), so that the amplitude is read
// and multiplied once for all of them: 2 to 3 VALU instructions per term, the
// lane part of its sign a 64-bit mask made at upload (a scalar operand of a
// select), the part of the wavefront's own index bits scalar.  Terms with no
// phase bit among the row bits are summed once for all rows.
//
// For chains of up to kWaveMaxLen sites, whose tiles are too few to fill the
// 256 CUs, the flip masks are cut into `depth` slices of about equal work,
// one per wavefront, so that all CUs have several wavefronts; the 8 or 16 of
// a workgroup add their sums in LDS, workgroups through memory, the last one
// to arrive in slice order.  Bound by latency there: dense SYK N=24 FP64 (10626
// terms, 4096 amplitudes) took 33 us in one chain of loads per term and slice
// and 14 us in a second launch that added the slices.
// ---------------------------------------------------------------------------
// One flip mask, or a piece of one.  One or two terms of one kind (real, or kWaveImag imaginary
// coefficients) stand in the record itself (kWaveTwo: two); kWaveRow: one of
// them has phase bits among the row bits.  Otherwise (kWaveMulti) the terms
// from `term` on: real ones without and with such bits, then imaginary ones
// likewise, their counts z0, z1 and the halves of l0.
template <typename A> struct alignas(16) SubW { uint64_t l0, l1; A c0, c1; uint32_t z0, z1, kind, term; };
enum : uint32_t { kWaveImag = 1, kWaveRow = 2, kWaveTwo = 4, kWaveMulti = 8 };
template <typename A> struct TermW { uint64_t lanes; A c; uint32_t z, pad; };

constexpr int kWaveMaxLen = 19, kWaveMaxFlips = 40;
constexpr int kWavePad = 16;       // flip masks read past the end of the list
// Where the list is cut into slices, a flip mask of more terms than this is
// cut into records of its own, each with its gather (worth about six terms),
// so that few masks of many terms fill the slices too: one mask of 300 terms
// at 14 sites takes 15.0 us in one slice, 6.1 in 8.
constexpr uint32_t kWavePiece = 32;

__device__ __forceinline__ float flip_bit31(float c, uint32_t b)
{
    return __uint_as_float(__float_as_uint(c) ^ b);
}
__device__ __forceinline__ double flip_bit31(double c, uint32_t b)
{
    return __hiloint2double(__double2hiint(c) ^ (int)b, __double2loint(c));
}
// c with the sign of (-1)^popcount(m & z), uniform, for the first amplitude
// m = m0 of each row r of 64 (index bits 6 and 7 number four rows)
template <typename A, int ROWS>
__device__ __forceinline__ void row_signs(A c, uint32_t m0, uint32_t z, A (&s)[ROWS])
{
    static_assert(ROWS == 1 || ROWS == 4, "rows");
    s[0] = flip_bit31(c, (uint32_t)__popc(m0 & z) << 31);
    if constexpr (ROWS == 4) {
        const uint32_t b0 = (z << 25) & 0x80000000u, b1 = (z << 24) & 0x80000000u;
        s[1] = flip_bit31(s[0], b0);
        s[2] = flip_bit31(s[0], b1);
        s[3] = flip_bit31(s[1], b1);
    }
}
// +-1 by the lane's bit of `neg`
__device__ __forceinline__ float lane_sign(uint64_t neg, float)
{
    return __builtin_amdgcn_inverse_ballot_w64(neg) ? -1.f : 1.f;
}
__device__ __forceinline__ double lane_sign(uint64_t neg, double)
{
    return __hiloint2double(__builtin_amdgcn_inverse_ballot_w64(neg) ? 0xbff00000 : 0x3ff00000, 0);
}

// d[r] += one term (BYROW: it has phase bits among the row bits; otherwise
// only d[0], which the caller copies); m0: the wavefront's first amplitude
template <typename A, int ROWS, bool BYROW>
__device__ __forceinline__ void add_term(const TermW<A> &C, uint32_t m0, A (&d)[ROWS])
{
    const A sg = lane_sign(C.lanes, A(0));
    A c[BYROW ? ROWS : 1];
    row_signs<A, BYROW ? ROWS : 1>(C.c, m0, C.z, c);
#pragma unroll
    for (int r = 0; r < (BYROW ? ROWS : 1); r++) d[r] = fma(sg, c[r], d[r]);
}

template <typename A, int ROWS, bool BYROW>
__device__ __forceinline__ void sum_terms(const TermW<A> *__restrict__ p, uint32_t n, uint32_t m0,
                                          A (&d)[ROWS])
{
    uint32_t t = 0;
    for (; t + 4 <= n; t += 4) {     // four records in flight
        const TermW<A> C[4] = {p[t], p[t + 1], p[t + 2], p[t + 3]};
#pragma unroll
        for (int i = 0; i < 4; i++) add_term<A, ROWS, BYROW>(C[i], m0, d);
    }
    for (; t < n; t++) add_term<A, ROWS, BYROW>(p[t], m0, d);
}

// the coefficient of one flip mask at the wavefront's amplitudes: na terms
// shared by all rows, nb by row
template <typename A, int ROWS>
__device__ __forceinline__ void sum_coef(const TermW<A> *__restrict__ p, uint32_t na, uint32_t nb,
                                         uint32_t m0, A (&d)[ROWS])
{
    A one[1] = {0};
    sum_terms<A, 1, false>(p, na, m0, one);
#pragma unroll
    for (int r = 0; r < ROWS; r++) d[r] = one[0];
    if (ROWS > 1 && nb) sum_terms<A, ROWS, true>(p + na, nb, m0, d);
}

// acc += d v, or i d v
template <typename T, typename A, int ROWS>
__device__ __forceinline__ void add_rows(const A (&d)[ROWS], const T (&v)[ROWS], bool imag,
                                         A (&ar)[ROWS], A (&ai)[ROWS])
{
    if constexpr (ROWS == 1 && sizeof(A) == 4) {
        // the components as values first: sunk below the branch, their loads
        // from v became one load at a chosen address, and v an array in scratch
        // memory.  (With more rows or FP64 sums it costs registers instead:
        // 79 against 68, and the occupancy that hides the gathers.)
        A x = v[0].x, y = v[0].y;
        asm volatile("" : "+v"(x), "+v"(y));
        ar[0] = fma(imag ? -d[0] : d[0], imag ? y : x, ar[0]);
        ai[0] = fma(d[0], imag ? x : y, ai[0]);
        return;
    }
    if (!imag) {
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            ar[r] = fma(d[r], (A)v[r].x, ar[r]);
            ai[r] = fma(d[r], (A)v[r].y, ai[r]);
        }
    } else {
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            ar[r] = fma(-d[r], (A)v[r].y, ar[r]);
            ai[r] = fma(d[r], (A)v[r].x, ai[r]);
        }
    }
}

// W wavefronts per workgroup: with one slice each its own amplitudes, else
// slices of the same ones
// BIG: states of 4 GiB and more, whose gathers need 64-bit offsets
template <typename R, typename A, int ROWS, int W, bool BIG>
__global__ void __launch_bounds__(64 * W)
k_apply_wave(const typename CxA<R>::T *__restrict__ in, typename CxA<R>::T *__restrict__ out,
             uint64_t dim, const uint32_t *__restrict__ flips, const SubW<A> *__restrict__ subs,
             const TermW<A> *__restrict__ terms, const uint32_t *__restrict__ cut, int depth,
             int accumulate, double *__restrict__ part, unsigned *__restrict__ count,
             const int *__restrict__ stop)
{
    using T = typename CxA<R>::T;
    constexpr int U = ROWS == 1 ? 4 : 2;       // flip masks whose gathers go out together
    constexpr bool SLICED = W > 4;
    __shared__ A sh[SLICED ? 2 * ROWS : 1][W][64];
    if (stop && *stop) return;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // one slice: each XCD a contiguous range of amplitudes
    const uint32_t chunk = SLICED ? blockIdx.x : xcd_tile_index() * W + wid;
    const uint32_t slice = SLICED ? blockIdx.y * W + wid : 0;
    const uint32_t m0 = chunk * (64 * ROWS);
    if (!SLICED && m0 >= dim) return;          // the grid is whole workgroups
    // fewer than 64 amplitudes: the upper lanes repeat the lower ones
    const uint32_t ll = dim < 64 ? lane & ((uint32_t)dim - 1) : lane;
    A ar[ROWS], ai[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; r++) { ar[r] = 0; ai[r] = 0; }
    const uint32_t s0 = cut[slice], s1 = cut[slice + 1];

    // byte offset of the lane's amplitude in row 0; a flip mask and a row
    // change bits of it: one scalar and one vector instruction per gather
    const uint32_t own = (m0 | ll) * (uint32_t)sizeof(T);
    auto gather = [&](const uint32_t (&x)[U], T (&v)[U][ROWS]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int r = 0; r < ROWS; r++) {
                const uint32_t f = x[u] ^ (uint32_t)(r * 64);
                if constexpr (BIG) v[u][r] = in[(uint64_t)((m0 | ll) ^ f)];
                else v[u][r] = *(const T *)((const char *)in + (own ^ f * (uint32_t)sizeof(T)));
            }
    };
    auto load_flips = [&](uint32_t s, uint32_t (&x)[U]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; u++) x[u] = flips[s + u];
    };
    auto apply = [&](const SubW<A> &S, const T (&v)[ROWS]) __attribute__((always_inline)) {
        A d[ROWS];
        if (S.kind & kWaveMulti) {
            const uint32_t n2 = (uint32_t)S.l0, n3 = (uint32_t)(S.l0 >> 32);
            const TermW<A> *p = terms + S.term;
            if (S.z0 + S.z1) {
                sum_coef<A, ROWS>(p, S.z0, S.z1, m0, d);
                add_rows<T, A, ROWS>(d, v, false, ar, ai);
            }
            if (n2 + n3) {
                sum_coef<A, ROWS>(p + S.z0 + S.z1, n2, n3, m0, d);
                add_rows<T, A, ROWS>(d, v, true, ar, ai);
            }
            return;
        }
        const A g0 = lane_sign(S.l0, A(0));
        if (ROWS > 1 && (S.kind & kWaveRow)) {
            A c[ROWS];
            row_signs<A, ROWS>(S.c0, m0, S.z0, c);
#pragma unroll
            for (int r = 0; r < ROWS; r++) d[r] = g0 * c[r];
            if (S.kind & kWaveTwo) {
                const A g1 = lane_sign(S.l1, A(0));
                row_signs<A, ROWS>(S.c1, m0, S.z1, c);
#pragma unroll
                for (int r = 0; r < ROWS; r++) d[r] = fma(g1, c[r], d[r]);
            }
        } else {
            A c[1];
            row_signs<A, 1>(S.c0, m0, S.z0, c);
            d[0] = g0 * c[0];
            if (S.kind & kWaveTwo) {
                row_signs<A, 1>(S.c1, m0, S.z1, c);
                d[0] = fma(lane_sign(S.l1, A(0)), c[0], d[0]);
            }
#pragma unroll
            for (int r = 1; r < ROWS; r++) d[r] = d[0];
        }
        add_rows<T, A, ROWS>(d, v, S.kind & kWaveImag, ar, ai);
    };
    // the gathers of the next U flip masks are in flight while the current
    // ones are used, their masks loaded one step earlier
    uint32_t xn[U];
    T va[U][ROWS], vb[U][ROWS];
    load_flips(s0, xn);
    gather(xn, va);
    load_flips(s0 + U, xn);
    auto step = [&](uint32_t s, T (&cur)[U][ROWS], T (&nxt)[U][ROWS]) __attribute__((always_inline)) {
        // the records as words: an array of the struct itself goes to scratch
        constexpr int NW = sizeof(SubW<A>) / 4;
        uint32_t S[U][NW];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int i = 0; i < NW; i++) S[u][i] = ((const uint32_t *)(subs + s + u))[i];
        if (s + U < s1) gather(xn, nxt);
        load_flips(s + 2 * U, xn);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (s + u < s1) apply(__builtin_bit_cast(SubW<A>, S[u]), cur[u]);
    };
    for (uint32_t s = s0; s < s1; s += 2 * U) {
        step(s, va, vb);
        if (s + U < s1) step(s + U, vb, va);
    }

    if constexpr (SLICED) {
        // the slices of this workgroup, then those of the others
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            sh[2 * r][wid][lane] = ar[r];
            sh[2 * r + 1][wid][lane] = ai[r];
        }
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < 128 * ROWS; i += 64 * W) {
            A *q = &sh[i >> 6][0][i & 63], a = q[0];
#pragma unroll
            for (int w = 1; w < W; w++) a += q[w * 64];
            q[0] = a;
        }
        __syncthreads();
        if (wid) return;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            ar[r] = sh[2 * r][0][lane];
            ai[r] = sh[2 * r + 1][0][lane];
        }
        const uint32_t nw = gridDim.y;
        if constexpr (W == 16) {
            double *row = part + (size_t)chunk * nw * (128 * ROWS) + lane;
#pragma unroll
            for (int r = 0; r < ROWS; r++) {
                double *q = row + (size_t)blockIdx.y * (128 * ROWS) + r * 128;
                put_shared(q, (double)ar[r]);
                put_shared(q + 64, (double)ai[r]);
            }
            if (!arrive_last(count + chunk, nw)) return;
            // at most 8 workgroups, the sums of 8 / ROWS of them in flight
            constexpr int PER = 8 / ROWS;
            double sum[2 * ROWS] = {};
            for (uint32_t i0 = 0; i0 < nw; i0 += PER) {
                double p[PER][2 * ROWS];
#pragma unroll
                for (int i = 0; i < PER; i++)
#pragma unroll
                    for (int r = 0; r < 2 * ROWS; r++)
                        p[i][r] = i0 + i < nw
                                      ? get_shared(row + (size_t)(i0 + i) * (128 * ROWS) + r * 64)
                                      : 0.0;
#pragma unroll
                for (int i = 0; i < PER; i++)
#pragma unroll
                    for (int r = 0; r < 2 * ROWS; r++) sum[r] += p[i][r];
            }
            if (lane == 0) count[chunk] = 0;
#pragma unroll
            for (int r = 0; r < ROWS; r++) {
                ar[r] = (A)sum[2 * r];
                ai[r] = (A)sum[2 * r + 1];
            }
        }
    }
    if (lane >= dim) return;
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        T *o = out + (size_t)m0 + r * 64 + lane;
        A xr = ar[r], xi = ai[r];
        if (accumulate) {
            const T b = *o;
            xr += (A)b.x;
            xi += (A)b.y;
        }
        T e;
        e.x = (R)xr;
        e.y = (R)xi;
        *o = e;
    }
}

// wavefronts per workgroup of k_apply_wave: for 8 slices one workgroup, for
// 32 and 128 two and eight of 16 wavefronts
static int wave_width(int depth) { return depth == 1 ? 4 : depth == 8 ? 8 : 16; }

template <typename R, int TB, int NT, int D = 2>
constexpr int apply_waves_per_eu()
{
    constexpr int lds = D * (1 << TB) * 2 * (int)sizeof(R);
    constexpr int wg_by_lds = (160 * 1024) / lds;
    // 1024-thread workgroups: two per CU (32 waves) when their LDS fits
    constexpr int wg_by_waves = (NT == 1024 ? 2048 : 1024) / NT;
    constexpr int wg = wg_by_lds < wg_by_waves ? wg_by_lds : wg_by_waves;
    constexpr int w = (wg < 1 ? 1 : wg) * (NT / 64) / 4;
    return w < 1 ? 1 : w;
}

// Copy the input tile starting at element `src` into LDS buffer `dst` with
// gfx950's asynchronous global->LDS loads: every lane moves 16 bytes, a
// wavefront fills a contiguous 1 KiB run starting at the wave-uniform LDS
// address.  Completion is tracked by the vector memory counter.
template <typename T, int TB, int NT>
__device__ inline void tile_dma(const T *__restrict__ in, uint64_t src, T *dst)
{
    constexpr int TILE_BYTES = (1 << TB) * (int)sizeof(T);
    constexpr int PER_THREAD = TILE_BYTES / (16 * NT);
    static_assert(PER_THREAD >= 1 && TILE_BYTES % (16 * NT) == 0, "tile too small for DMA");
    // uniform tile base plus a 32-bit lane offset (below 64 KiB)
    const char *g = (const char *)(in + src);
    char *l = (char *)dst;
    // wave-uniform: kept in a scalar register, so that the LDS address
    // (M0) of every DMA is scalar arithmetic
    const uint32_t tid = threadIdx.x,
                   wave_base = __builtin_amdgcn_readfirstlane(tid & ~63u);
#pragma unroll
    for (int c = 0; c < PER_THREAD; c++) {
        const uint32_t chunk = c * NT;
        __builtin_amdgcn_global_load_lds(
            (const void *)(g + (uint32_t)((chunk + tid) * 16)),
            (__attribute__((address_space(3))) void *)(l + (size_t)(chunk + wave_base) * 16),
            16, 0, 0);
    }
}

// a sub's coefficient in the partial-sum type P (float copies for FP32
// partial sums of FP64-coefficient layouts: no conversion in the loop)
template <typename P, typename A>
__device__ __forceinline__ P sub_re(const SubRec<A> &S)
{
    if constexpr (std::is_same_v<P, float> && !std::is_same_v<A, float>) return S.fr;
    else return (P)S.cr;
}
template <typename P, typename A>
__device__ __forceinline__ P sub_im(const SubRec<A> &S)
{
    if constexpr (std::is_same_v<P, float> && !std::is_same_v<A, float>) return S.fi;
    else return (P)S.ci;
}

// Sign bit (bit 31) of (-1)^popcount(v), and a coefficient with that sign
// applied by flipping its sign bit
__device__ __forceinline__ uint32_t parity_sign(uint32_t v) { return (uint32_t)__popc(v) << 31; }
// (adding bit 31 flips it like an xor: one shift-add instruction with the
// shift of the sign bit)
__device__ __forceinline__ float flip_sign(float c, uint32_t sb)
{
    return __uint_as_float(__float_as_uint(c) + sb);
}
__device__ __forceinline__ double flip_sign(double c, uint32_t sb)
{
    return __longlong_as_double(__double_as_longlong(c) ^ ((long long)sb << 32));
}
// a * b + c with one rounding
__device__ __forceinline__ float fmadd(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmadd(double a, double b, double c) { return __builtin_fma(a, b, c); }

// the lane-signed coefficient of a sub whose rows flip it again: kept in a
// register, so that each row's flip is one xor with a scalar sign instead
// of the whole popcount per row
template <typename P> __device__ __forceinline__ P opaque(P c)
{
    asm volatile("" : "+v"(c));
    return c;
}

// The LDS address of this lane's input element in tile row 0 for flip mask
// xl: the lane offset is formed once per sub (one xor) and kept opaque, so
// that each row's address is that offset plus a scalar row offset
template <typename T, int NT>
__device__ __forceinline__ const T *sub_lane_base(const T *buf, uint32_t lane8, uint32_t xl)
{
    uint32_t la = lane8 ^ ((xl & (NT - 1)) * (uint32_t)sizeof(T));
    asm volatile("" : "+v"(la));
    return (const T *)((const char *)buf + la);
}

// Apply every sub of group G from the staged input tile `buf` (LDS) to the
// RP accumulated rows of this thread.  Amplitude t0 + r NT + tid of the
// output tile reads the input at (t0 + r NT + tid) ^ x: lane tid ^ (x mod NT)
// of tile row r ^ (x / NT mod RP); lanebits = t0 | tid (the index bits
// outside the row bits) gives the lane's share of the phase sign.
template <typename R, typename A, int TB, int NT, typename P = A>
__device__ __forceinline__ void apply_group(const GroupRuns &G, const typename CxA<R>::T *buf,
                                            const SubRec<A> *__restrict__ subs,
                                            const TermRec<A> *__restrict__ terms,
                                            uint32_t lanebits, uint32_t tid,
                                            P (&accr)[(1 << TB) / NT], P (&acci)[(1 << TB) / NT])
{
    using T = typename CxA<R>::T;
    constexpr int RP = (1 << TB) / NT;
    constexpr int LB = NT == 1024 ? 10 : NT == 512 ? 9 : NT == 256 ? 8 : 7;

    // this lane's byte offset in a tile row
    const uint32_t lane8 = tid * (uint32_t)sizeof(T);
#define RP_SUB_PROLOGUE                                                            \
    const SubRec<A> S = subs[s];                                               \
    const T *row = sub_lane_base<T, NT>(buf, lane8, S.xl);                     \
    const uint32_t xr = S.xl >> LB;                                            \
    const uint32_t lsb = parity_sign(lanebits & S.z);                          \
    const uint32_t zr = (S.z >> LB) & (RP - 1);                                \
    (void)zr;
    // real c, no phase bit among the row bits
    for (uint32_t s = G.b[kRunReal0]; s < G.b[kRunReal0 + 1]; s++) {
        RP_SUB_PROLOGUE
        const P c = flip_sign(sub_re<P>(S), lsb);
#pragma unroll
        for (int r = 0; r < RP; r++) {
            const T v = row[(r ^ xr) * NT];
            accr[r] += c * (P)v.x;
            acci[r] += c * (P)v.y;
        }
    }
    for (uint32_t s = G.b[kRunReal1]; s < G.b[kRunReal1 + 1]; s++) {
        RP_SUB_PROLOGUE
        const P c = opaque(flip_sign(sub_re<P>(S), lsb));
#pragma unroll
        for (int r = 0; r < RP; r++) {
            const T v = row[(r ^ xr) * NT];
            const P cc = flip_sign(c, parity_sign(r & zr));
            accr[r] += cc * (P)v.x;
            acci[r] += cc * (P)v.y;
        }
    }
    // imaginary c = i ci: (i ci)(vr + i vi) = -ci vi + i ci vr
    for (uint32_t s = G.b[kRunImag0]; s < G.b[kRunImag0 + 1]; s++) {
        RP_SUB_PROLOGUE
        const P c = flip_sign(sub_im<P>(S), lsb);
#pragma unroll
        for (int r = 0; r < RP; r++) {
            const T v = row[(r ^ xr) * NT];
            accr[r] -= c * (P)v.y;
            acci[r] += c * (P)v.x;
        }
    }
    for (uint32_t s = G.b[kRunImag1]; s < G.b[kRunImag1 + 1]; s++) {
        RP_SUB_PROLOGUE
        const P c = opaque(flip_sign(sub_im<P>(S), lsb));
#pragma unroll
        for (int r = 0; r < RP; r++) {
            const T v = row[(r ^ xr) * NT];
            const P cc = flip_sign(c, parity_sign(r & zr));
            accr[r] -= cc * (P)v.y;
            acci[r] += cc * (P)v.x;
        }
    }
    for (uint32_t s = G.b[kRunCplx]; s < G.b[kRunCplx + 1]; s++) {
        RP_SUB_PROLOGUE
        const P cr = opaque(flip_sign(sub_re<P>(S), lsb)), ci = opaque(flip_sign(sub_im<P>(S), lsb));
#pragma unroll
        for (int r = 0; r < RP; r++) {
            const T v = row[(r ^ xr) * NT];
            const uint32_t rsb = parity_sign(r & zr);
            const P a = flip_sign(cr, rsb), c = flip_sign(ci, rsb);
            // two nested fused multiply-adds per component (the rounding
            // order of the compact-record kernel)
            accr[r] = fmadd(a, (P)v.x, fmadd(-c, (P)v.y, accr[r]));
            acci[r] = fmadd(a, (P)v.y, fmadd(c, (P)v.x, acci[r]));
        }
    }
#undef RP_SUB_PROLOGUE
    // several terms share x: d(m) = sum_t c_t (-1)^popcount(m & z_t),
    // formed for four rows at a time to bound register use
    for (uint32_t s = G.b[kRunMulti]; s < G.b[kRunMulti + 1]; s++) {
        const SubRec<A> S = subs[s];
        const T *row = sub_lane_base<T, NT>(buf, lane8, S.xl);
        const uint32_t xr = S.xl >> LB;
        constexpr int RC = RP < 4 ? RP : 4;
#pragma unroll
        for (int r0 = 0; r0 < RP; r0 += RC) {
            P dr[RC], di[RC];
#pragma unroll
            for (int q = 0; q < RC; q++) { dr[q] = 0; di[q] = 0; }
            for (uint32_t t = S.term_begin; t < S.term_end; t++) {
                const TermRec<A> C = terms[t];
                const uint32_t lsb = parity_sign(lanebits & C.z);
                const P cr = (P)flip_sign(C.cr, lsb);
                const P ci = (P)flip_sign(C.ci, lsb);
                const uint32_t zr = (C.z >> LB) & (RP - 1);
#pragma unroll
                for (int q = 0; q < RC; q++) {
                    const uint32_t rsb = parity_sign((r0 + q) & zr);
                    dr[q] += flip_sign(cr, rsb);
                    di[q] += flip_sign(ci, rsb);
                }
            }
#pragma unroll
            for (int q = 0; q < RC; q++) {
                const T v = row[((r0 + q) ^ xr) * NT];
                accr[r0 + q] = fmadd(dr[q], (P)v.x, fmadd(-di[q], (P)v.y, accr[r0 + q]));
                acci[r0 + q] = fmadd(dr[q], (P)v.y, fmadd(di[q], (P)v.x, acci[r0 + q]));
            }
        }
    }
}

// s_waitcnt immediate that waits until at most N vector memory operations
// of this wave are outstanding and all of its LDS operations have completed
// (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt 6:4 left at its
// maximum, lgkmcnt 11:8 = 0)
template <int N>
__device__ inline void wait_vmcnt_lds()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}

// Workgroup barrier without the release/acquire fences of __syncthreads(),
// whose release would drain every outstanding global->LDS load.  The caller
// has waited for its own loads into the tile about to be read (vmcnt) and
// for its own LDS reads of the tile about to be overwritten (lgkmcnt 0); the
// compiler barriers keep memory operations on their side.
__device__ inline void tile_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Pipeline of D LDS tiles: the input tiles of the next D-1 groups are in
// flight while a group is applied.  Phase K of an unrolled round uses the
// statically named buffer K, so the compiler sees which DMA writes which
// array and does not drain every load before each LDS read.
template <typename R, typename A, int TB, int NT, int D, int K, bool GA>
__device__ __forceinline__ void pipe_phase(
    int g, int ngroups, const typename CxA<R>::T *__restrict__ in,
    const GroupRuns *__restrict__ groups, const SubRec<A> *__restrict__ subs,
    const TermRec<A> *__restrict__ terms, uint32_t t0, uint32_t tid,
    typename CxA<R>::T *b0, typename CxA<R>::T *b1, typename CxA<R>::T *b2,
    typename CxA<R>::T *b3, A (&accr)[(1 << TB) / NT], A (&acci)[(1 << TB) / NT],
    float (&gr)[(1 << TB) / NT], float (&gi)[(1 << TB) / NT])
{
    using T = typename CxA<R>::T;
    constexpr int PT = ((1 << TB) * (int)sizeof(T)) / (16 * NT);   // DMA ops per thread per tile
    T *const bufs[4] = {b0, b1, b2, b3};
    // this thread's share of group g's tile has landed once at most the
    // DMAs issued after it (groups g+1 .. g+D-2) are outstanding; after the
    // barrier every share is visible and group g-1's buffer is no longer read
    if constexpr (D == 2) {
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
    } else {
        if (g + D - 2 < ngroups) wait_vmcnt_lds<(D - 2) * PT>();
        else __builtin_amdgcn_s_waitcnt(0);
        tile_barrier();
    }
    if (g + D - 1 < ngroups)
        tile_dma<T, TB, NT>(in, t0 ^ (groups[g + D - 1].xh << TB), bufs[(K + D - 1) % D]);
    if constexpr (GA) {
        // the terms of four consecutive groups summed in FP32 (gr, gi), those
        // sums added to the FP64 accumulators by the caller
        apply_group<R, A, TB, NT, float>(groups[g], bufs[K], subs, terms, t0 | tid, tid, gr, gi);
    } else {
        apply_group<R, A, TB, NT>(groups[g], bufs[K], subs, terms, t0 | tid, tid, accr, acci);
    }
}

// add the FP32 partial sums to the FP64 accumulators and clear them
template <typename A, int RP>
__device__ __forceinline__ void flush_partials(A (&accr)[RP], A (&acci)[RP], float (&gr)[RP],
                                               float (&gi)[RP])
{
#pragma unroll
    for (int r = 0; r < RP; r++) {
        accr[r] += (A)gr[r];
        acci[r] += (A)gi[r];
        gr[r] = 0;
        gi[r] = 0;
        // opaque zeros: the compiler would otherwise propagate the constant
        // into the next round and zero the registers again on every path
        asm volatile("" : "+v"(gr[r]), "+v"(gi[r]));
    }
}

// The body of the tiled apply for the output tile of this workgroup: every
// group's input tile through the LDS pipeline, then the tile written once.
// wv receives the values written (the rounded outputs), for an epilogue.
template <typename R, typename A, int TB, int NT, int D, bool GA>
__device__ __forceinline__ void apply_tile(const typename CxA<R>::T *__restrict__ in,
                                           typename CxA<R>::T *__restrict__ out,
                                           const GroupRuns *__restrict__ groups, int ngroups,
                                           const SubRec<A> *__restrict__ subs,
                                           const TermRec<A> *__restrict__ terms, int accumulate,
                                           typename CxA<R>::T *tile0, typename CxA<R>::T *tile1,
                                           typename CxA<R>::T *tile2, typename CxA<R>::T *tile3,
                                           uint32_t t0, typename CxA<R>::T (&wv)[(1 << TB) / NT])
{
    using T = typename CxA<R>::T;
    constexpr int TILE = 1 << TB;
    constexpr int RP = TILE / NT;          // amplitudes per thread
    const uint32_t tid = threadIdx.x;

    A accr[RP], acci[RP];
    float gr[RP], gi[RP];      // FP32 partial sums (group accumulation)
#pragma unroll
    for (int r = 0; r < RP; r++) {
        accr[r] = 0;
        acci[r] = 0;
        gr[r] = 0;
        gi[r] = 0;
        if constexpr (GA) asm volatile("" : "+v"(gr[r]), "+v"(gi[r]));
    }

    T *const ring[4] = {tile0, tile1, tile2, tile3};
#pragma unroll
    for (int q = 0; q < D - 1; q++)
        if (q < ngroups) tile_dma<T, TB, NT>(in, t0 ^ (groups[q].xh << TB), ring[q]);
    for (int g = 0; g < ngroups; g += D) {
        pipe_phase<R, A, TB, NT, D, 0, GA>(g, ngroups, in, groups, subs, terms, t0, tid, tile0, tile1,
                                       tile2, tile3, accr, acci, gr, gi);
        if (g + 1 >= ngroups) break;
        pipe_phase<R, A, TB, NT, D, 1, GA>(g + 1, ngroups, in, groups, subs, terms, t0, tid, tile0,
                                       tile1, tile2, tile3, accr, acci, gr, gi);
        if constexpr (D > 2) {
            if (g + 2 >= ngroups) break;
            pipe_phase<R, A, TB, NT, D, 2, GA>(g + 2, ngroups, in, groups, subs, terms, t0, tid, tile0,
                                           tile1, tile2, tile3, accr, acci, gr, gi);
        }
        if constexpr (D > 3) {
            if (g + 3 >= ngroups) break;
            pipe_phase<R, A, TB, NT, D, 3, GA>(g + 3, ngroups, in, groups, subs, terms, t0, tid, tile0,
                                           tile1, tile2, tile3, accr, acci, gr, gi);
        }
        // FP32 partial sums of every other round (four groups at D = 2) into
        // the FP64 accumulators
        if constexpr (GA) {
            if ((g / D) & 1) flush_partials(accr, acci, gr, gi);
        }
    }
    if constexpr (GA) flush_partials(accr, acci, gr, gi);
#pragma unroll
    for (int r = 0; r < RP; r++) {
        const uint64_t m = (uint64_t)t0 + r * NT + tid;
        T o;
        if (accumulate) {
            const T p = out[m];
            o.x = (R)(accr[r] + (A)p.x);
            o.y = (R)(acci[r] + (A)p.y);
        } else {
            o.x = (R)accr[r];
            o.y = (R)acci[r];
        }
        out[m] = o;
        wv[r] = o;
    }
}

// the workgroup's output tile under the map tm (rp_tables.h): index bits
// 0..p-1 = position within the XCD's resident workgroups, p..p+2 = XCD,
// above = batch; the grid has 2^n >= 2^(p+3) workgroups
__device__ __forceinline__ uint32_t tile_index(const TileMap &tm)
{
    if (!tm.n) return xcd_tile_index();
    const uint32_t b = blockIdx.x, p = (uint32_t)tm.p, j = b >> 3;
    const uint32_t idx = ((j >> p) << (p + 3)) | ((b & 7u) << p) | (j & ((1u << p) - 1));
    uint32_t t = 0;
    for (int i = 0; i < tm.n; i++)
        if (idx >> i & 1u) t ^= tm.col[i];
    return t;
}

// The first amplitude of that tile, formed before the kernel looks at its stop
// flag.  The tiled kernels take the flag's address before the map, so that
// their arguments still fill three 64-byte lines: with the address behind the
// map, and the flag looked at first, every workgroup waited for a fourth line,
// 3 to 6 percent of an apply with few groups.
template <int TB> __device__ __forceinline__ uint32_t first_amplitude(const TileMap &tm)
{
    uint32_t t0 = tile_index(tm) << TB;
    asm volatile("" : "+s"(t0));
    return t0;
}

template <typename R, typename A, int TB, int NT, int D, bool GA>
__global__ void __launch_bounds__(NT, (apply_waves_per_eu<R, TB, NT, D>()))
k_apply_tiled(const typename CxA<R>::T *__restrict__ in, typename CxA<R>::T *__restrict__ out,
              const GroupRuns *__restrict__ groups, int ngroups, int accumulate,
              const SubRec<A> *__restrict__ subs, const TermRec<A> *__restrict__ terms,
              const int *__restrict__ stop, TileMap tm)
{
    const uint32_t t0 = first_amplitude<TB>(tm);
    if (stop && *stop) return;
    using T = typename CxA<R>::T;
    constexpr int TILE = 1 << TB;
    static_assert(NT == 1024 || NT == 512 || NT == 256 || NT == 128,
                  "NT must be a power of two in [128, 1024]");
    static_assert(D >= 2 && D <= 4, "2 to 4 LDS tiles");
    // D separate LDS tiles (the unused ones have one element)
    __shared__ T tile0[TILE];
    __shared__ T tile1[TILE];
    __shared__ T tile2[D > 2 ? TILE : 1];
    __shared__ T tile3[D > 3 ? TILE : 1];
    T wv[TILE / NT];
    apply_tile<R, A, TB, NT, D, GA>(in, out, groups, ngroups, subs, terms, accumulate, tile0, tile1,
                                    tile2, tile3, t0, wv);
}

// ---------------------------------------------------------------------------
// The complex<float> group-accumulating apply over compact sub records.
// The 48-byte SubRec list of a sparse SYK Hamiltonian at 24-30 qubits
// (370-480 subs, 18-23 KiB) does not fit the 16 KiB scalar data cache, so
// every sub record of the kernel above is a dependent load from L2.  Here
// each sub is 16 bytes and each group header 16 bytes (8-12 KiB together);
// the subs of all groups form one list in group order, and the record of
// the next sub, and the header of the group after next, are loaded while
// the current ones are in use.  Each single-term sub branches once on its
// row flip (uniform) to a code path whose LDS row reads are immediate
// offsets from one lane address.
// ---------------------------------------------------------------------------
// xl: bytes that the flip moves the lane by (bits 0..15), the row flip (16..)
// and the phase bits among the row bits (24..)
struct SubC { uint32_t xl, z; float c0, c1; };
struct TermC { uint32_t z; float cr, ci; uint32_t zr; };
// group header: tile index above the tile bits, first sub, subs per class
// run (kRunReal0 .. kRunMulti)
struct GroupC { uint32_t xh, begin; uint8_t n[kRuns]; uint8_t pad[8 - kRuns]; };
static_assert(sizeof(GroupC) == 16, "16-byte group header");

template <int V> struct IC { static constexpr int value = V; };

// f(IC<xr>) for the run-time row flip xr < RP: one code path per value, so
// that the row offsets are immediates
template <int RP, typename F>
__device__ __forceinline__ void with_row_flip(uint32_t xr, F &&f)
{
    if constexpr (RP == 8) {
        switch (xr) {
        case 0: f(IC<0>{}); break;
        case 1: f(IC<1>{}); break;
        case 2: f(IC<2>{}); break;
        case 3: f(IC<3>{}); break;
        case 4: f(IC<4>{}); break;
        case 5: f(IC<5>{}); break;
        case 6: f(IC<6>{}); break;
        default: f(IC<7>{}); break;
        }
    } else if constexpr (RP == 4) {
        switch (xr) {
        case 0: f(IC<0>{}); break;
        case 1: f(IC<1>{}); break;
        case 2: f(IC<2>{}); break;
        default: f(IC<3>{}); break;
        }
    } else if constexpr (RP == 2) {
        if (xr) f(IC<1>{});
        else f(IC<0>{});
    } else {
        f(IC<0>{});
    }
}

// all RP row values of a sub loaded before any is used: the reads go out
// back to back and one wait covers them
template <int PR> __device__ __forceinline__ void pin_rows(float4 (&v)[PR])
{
#pragma unroll
    for (int i = 0; i + 1 < PR; i += 2)
        asm volatile("" : "+v"(v[i].x), "+v"(v[i].y), "+v"(v[i].z), "+v"(v[i].w), "+v"(v[i + 1].x),
                     "+v"(v[i + 1].y), "+v"(v[i + 1].z), "+v"(v[i + 1].w));
    if constexpr (PR & 1)
        asm volatile("" : "+v"(v[PR - 1].x), "+v"(v[PR - 1].y), "+v"(v[PR - 1].z), "+v"(v[PR - 1].w));
}

// The rows of a thread in the streamed kernel: amplitude r = 2 p + h of
// thread tid is element p 2 NT + 2 tid + h of the tile.  Neighbouring pairs
// make every LDS read 16 bytes wide: ds_read_b128 delivers 212 bytes per
// clock and CU, ds_read2st64_b64 120.  Flip masks and phase masks in these
// terms: bits 1 .. log2 NT move the lane, bit 0 and the top log2 (RP / 2)
// bits the row.
static inline uint32_t stream_row(uint32_t v, int tb, int nt)
{
    return (v & 1u) | (((v & ((1u << tb) - 1)) / (2u * (unsigned)nt)) << 1);
}

// One single-term sub with the row flip XR fixed: input amplitude j of the
// lane feeds output amplitude j ^ XR.  c (and ci for the complex class) carry
// the lane's phase sign; zr = the phase bits among the row bits (classes 1
// and complex).
template <int RP, int NT, uint32_t CLS, int XR>
__device__ __forceinline__ void sub_rows(float4 (&vv)[RP / 2], float c, float ci, uint32_t zr,
                                         float (&gr)[RP], float (&gi)[RP])
{
    pin_rows<RP / 2>(vv);
#pragma unroll
    for (int j = 0; j < RP; j++) {
        const int r = j ^ XR;
        const float4 q = vv[j / 2];
        const float2 v = (j & 1) ? float2{q.z, q.w} : float2{q.x, q.y};
        // explicit fused multiply-adds: one rounding each, and no product
        // that the compiler could share between the row-flip paths
        if constexpr (CLS == kRunReal0) {
            gr[r] = __builtin_fmaf(c, v.x, gr[r]);
            gi[r] = __builtin_fmaf(c, v.y, gi[r]);
        } else if constexpr (CLS == kRunImag0) {
            gr[r] = __builtin_fmaf(-c, v.y, gr[r]);
            gi[r] = __builtin_fmaf(c, v.x, gi[r]);
        } else if constexpr (CLS == kRunReal1) {
            const float cc = flip_sign(c, parity_sign((uint32_t)r & zr));
            gr[r] = __builtin_fmaf(cc, v.x, gr[r]);
            gi[r] = __builtin_fmaf(cc, v.y, gi[r]);
        } else if constexpr (CLS == kRunImag1) {
            const float cc = flip_sign(c, parity_sign((uint32_t)r & zr));
            gr[r] = __builtin_fmaf(-cc, v.y, gr[r]);
            gi[r] = __builtin_fmaf(cc, v.x, gi[r]);
        } else {
            const uint32_t rsb = parity_sign((uint32_t)r & zr);
            const float a = flip_sign(c, rsb), b = flip_sign(ci, rsb);
            gr[r] = __builtin_fmaf(a, v.x, __builtin_fmaf(-b, v.y, gr[r]));
            gi[r] = __builtin_fmaf(a, v.y, __builtin_fmaf(b, v.x, gi[r]));
        }
    }
}

// The subs of one class run [s, end) of a group from the staged tile buf.
// c0 holds the real coefficient (real classes), the imaginary one
// (imaginary classes) or the real part with c1 the imaginary part
// (complex); a multi sub holds its term range [z, bits of c0) in the FP32
// term list.  S is the record at s on entry and at end on exit.
template <int TB, int NT, uint32_t CLS>
__device__ __forceinline__ void stream_run(uint32_t &s, uint32_t end, SubC &S,
                                           const SubC *__restrict__ subs, const float4 *buf,
                                           uint32_t lane16, uint32_t lanebits,
                                           const TermC *__restrict__ terms,
                                           float (&gr)[(1 << TB) / NT], float (&gi)[(1 << TB) / NT])
{
    constexpr int RP = (1 << TB) / NT;
    for (; s < end; s++) {
        const SubC Sn = subs[s + 1];     // the list has one sentinel record
        // the lane's address: one xor, kept opaque, so that each row is an
        // immediate offset from it
        uint32_t la = lane16 ^ (S.xl & 0xffffu);
        asm volatile("" : "+v"(la));
        const float4 *row = (const float4 *)((const char *)buf + la);
        const uint32_t xr = (S.xl >> 16) & (RP - 1);
        if constexpr (CLS != kRunMulti) {
            // the reads go out first: the sign and the branch on the row flip
            // run while they are under way
            float4 vv[RP / 2];
#pragma unroll
            for (int p = 0; p < RP / 2; p++) vv[p] = row[p * NT];
            asm volatile("" ::: "memory");
            const uint32_t lsb = parity_sign(lanebits & S.z);
            const uint32_t zr = S.xl >> 24;
            float c = flip_sign(S.c0, lsb), ci = 0.f;
            // a lane-signed coefficient that each row flips again stays in a
            // register (one xor per row instead of the popcount per row)
            if constexpr (CLS == kRunReal1 || CLS == kRunImag1 || CLS == kRunCplx) c = opaque(c);
            if constexpr (CLS == kRunCplx) ci = opaque(flip_sign(S.c1, lsb));
            with_row_flip<RP>(xr, [&](auto X) {
                sub_rows<RP, NT, CLS, decltype(X)::value>(vv, c, ci, zr, gr, gi);
            });
        } else {
            const uint32_t tb = S.z, te = __float_as_uint(S.c0);
            // d(m) = sum_t c_t (-1)^popcount(m & z_t), two pairs at a time
            constexpr int RC = RP < 4 ? RP : 4;
#pragma unroll
            for (int r0 = 0; r0 < RP; r0 += RC) {
                float dr[RC], di[RC];
#pragma unroll
                for (int q = 0; q < RC; q++) { dr[q] = 0; di[q] = 0; }
                for (uint32_t t = tb; t < te; t++) {
                    const TermC C = terms[t];
                    const uint32_t lsb = parity_sign(lanebits & C.z);
                    const float cr = flip_sign(C.cr, lsb), ci = flip_sign(C.ci, lsb);
#pragma unroll
                    for (int q = 0; q < RC; q++) {
                        const uint32_t rsb = parity_sign((r0 + q) & C.zr);
                        dr[q] += flip_sign(cr, rsb);
                        di[q] += flip_sign(ci, rsb);
                    }
                }
                // input pair ((r0 + q) ^ xr) / 2, its halves exchanged where xr is
                // odd: 16-byte reads (8 bytes of every 16 took the LDS twice)
                float4 v[RC / 2];
#pragma unroll
                for (int a = 0; a < RC / 2; a++) v[a] = row[((r0 / 2 + a) ^ (xr >> 1)) * NT];
                auto pairs = [&](auto X) __attribute__((always_inline)) {
#pragma unroll
                    for (int q = 0; q < RC; q++) {
                        const float4 w = v[q / 2];
                        const bool hi = (q ^ decltype(X)::value) & 1;
                        const float x = hi ? w.z : w.x, y = hi ? w.w : w.y;
                        gr[r0 + q] = __builtin_fmaf(dr[q], x, __builtin_fmaf(-di[q], y, gr[r0 + q]));
                        gi[r0 + q] = __builtin_fmaf(dr[q], y, __builtin_fmaf(di[q], x, gi[r0 + q]));
                    }
                };
                if (xr & 1) pairs(IC<1>{});
                else pairs(IC<0>{});
            }
        }
        S = Sn;
    }
}

// one group of the streamed kernel: wait for its tile (buffer `cur`),
// start the next group's tile into `nxt`, apply the group's subs run by
// run.  Gc / Gn: this and the next group's headers (the header list has two
// sentinel entries); S the record of the group's first sub on entry and of
// the next group's first sub on exit.
template <int TB, int NT>
__device__ __forceinline__ void stream_phase(int g, int ngroups, const float2 *__restrict__ in,
                                             const GroupC *__restrict__ groups,
                                             const SubC *__restrict__ subs,
                                             const TermC *__restrict__ terms, uint32_t t0,
                                             uint32_t tid, const float4 *cur, float4 *nxt,
                                             SubC &S, uint32_t &s, GroupC &Gc, GroupC &Gn,
                                             float (&gr)[(1 << TB) / NT],
                                             float (&gi)[(1 << TB) / NT])
{
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (g + 1 < ngroups) tile_dma<float2, TB, NT>(in, t0 ^ (Gn.xh << TB), (float2 *)nxt);
    const GroupC Gnn = groups[g + 2];
    const uint32_t lane16 = tid * (uint32_t)sizeof(float4), lb = t0 | (tid << 1);
    uint32_t e = Gc.begin;
#define RP_STREAM_RUN(CLS)                                                                  \
    e += Gc.n[CLS];                                                                         \
    stream_run<TB, NT, CLS>(s, e, S, subs, cur, lane16, lb, terms, gr, gi);
    RP_STREAM_RUN(kRunReal0)
    RP_STREAM_RUN(kRunReal1)
    RP_STREAM_RUN(kRunImag0)
    RP_STREAM_RUN(kRunImag1)
    RP_STREAM_RUN(kRunCplx)
    RP_STREAM_RUN(kRunMulti)
#undef RP_STREAM_RUN
    Gc = Gn;
    Gn = Gnn;
}

// the whole output tile t0 of the streamed kernel: every group's input tile
// through the two LDS tiles, then the tile written once
template <int TB, int NT>
__device__ __forceinline__ void stream_tile(const float2 *__restrict__ in, float2 *__restrict__ out,
                                            const GroupC *__restrict__ groups, int ngroups,
                                            const SubC *__restrict__ subs,
                                            const TermC *__restrict__ terms, int accumulate,
                                            uint32_t t0, float4 *tile0, float4 *tile1)
{
    using T = float2;
    constexpr int RP = (1 << TB) / NT;
    const uint32_t tid = threadIdx.x;
    double accr[RP], acci[RP];
    float gr[RP], gi[RP];
#pragma unroll
    for (int r = 0; r < RP; r++) {
        accr[r] = 0;
        acci[r] = 0;
        gr[r] = 0;
        gi[r] = 0;
        asm volatile("" : "+v"(gr[r]), "+v"(gi[r]));
    }
    GroupC Gc = groups[0], Gn = groups[1];
    uint32_t s = 0;
    SubC S = subs[0];
    tile_dma<T, TB, NT>(in, t0 ^ (Gc.xh << TB), (float2 *)tile0);
    for (int g = 0; g < ngroups; g += 2) {
        stream_phase<TB, NT>(g, ngroups, in, groups, subs, terms, t0, tid, tile0, tile1, S, s, Gc,
                             Gn, gr, gi);
        if (g + 1 >= ngroups) break;
        stream_phase<TB, NT>(g + 1, ngroups, in, groups, subs, terms, t0, tid, tile1, tile0, S, s,
                             Gc, Gn, gr, gi);
        // FP32 partial sums of every four groups into the FP64 accumulators
        if ((g / 2) & 1) flush_partials(accr, acci, gr, gi);
    }
    flush_partials(accr, acci, gr, gi);
    // vectors are aligned to their elements, 8 bytes
    typedef float Pair __attribute__((ext_vector_type(4), aligned(8)));
#pragma unroll
    for (int p = 0; p < RP / 2; p++) {
        Pair *at = (Pair *)(out + (uint64_t)t0 + p * (2 * NT) + 2 * tid), o;
        if (accumulate) {
            const Pair b = *at;
            o.x = (float)(accr[2 * p] + (double)b.x);
            o.y = (float)(acci[2 * p] + (double)b.y);
            o.z = (float)(accr[2 * p + 1] + (double)b.z);
            o.w = (float)(acci[2 * p + 1] + (double)b.w);
        } else {
            o.x = (float)accr[2 * p];
            o.y = (float)acci[2 * p];
            o.z = (float)accr[2 * p + 1];
            o.w = (float)acci[2 * p + 1];
        }
        *at = o;
    }
}

template <int TB, int NT>
__global__ void __launch_bounds__(NT, (apply_waves_per_eu<float, TB, NT, 2>()))
k_apply_stream(const float2 *__restrict__ in, float2 *__restrict__ out,
               const GroupC *__restrict__ groups, int ngroups, int accumulate,
               const SubC *__restrict__ subs, const TermC *__restrict__ terms,
               const int *__restrict__ stop, TileMap tm)
{
    const uint32_t t0 = first_amplitude<TB>(tm);
    if (stop && *stop) return;
    __shared__ float4 tile0[1 << (TB - 1)];
    __shared__ float4 tile1[1 << (TB - 1)];
    stream_tile<TB, NT>(in, out, groups, ngroups, subs, terms, accumulate, t0, tile0, tile1);
}

// ---------------------------------------------------------------------------
// The same with FP64 sums throughout (complex<double>, and complex<float>
// without group accumulation): 16-byte records {flip, phase, coefficient} of
// the real and imaginary single-term subs, one list in group order, the next
// one loaded while the current one is in use; complex coefficients and flip
// masks with several terms go through the term list.  The rows are the SubRec
// kernel's; each sub branches once on its row flip, so that its row reads are
// immediate offsets, and the reads go out before its sign is formed.  The
// SubRec kernel's 48-byte records (17 KiB for sparse SYK at 23 qubits) do not
// fit the 16 KiB scalar cache and its rows need an address each.
// ---------------------------------------------------------------------------
struct SubD { uint32_t xl, z; double c; };
static_assert(sizeof(SubD) == 16, "16-byte record");

template <typename T, int RP, int NT, uint32_t CLS, int XR>
__device__ __forceinline__ void wide_rows(const T (&v)[RP], double c, uint32_t zr,
                                          double (&ar)[RP], double (&ai)[RP])
{
#pragma unroll
    for (int j = 0; j < RP; j++) {
        const int r = j ^ XR;
        const double x = (double)v[j].x, y = (double)v[j].y;
        double cc = c;
        if constexpr (CLS == kRunReal1 || CLS == kRunImag1)
            cc = flip_sign(c, parity_sign((uint32_t)r & zr));
        if constexpr (CLS == kRunReal0 || CLS == kRunReal1) {
            ar[r] = fmadd(cc, x, ar[r]);
            ai[r] = fmadd(cc, y, ai[r]);
        } else {
            ar[r] = fmadd(-cc, y, ar[r]);
            ai[r] = fmadd(cc, x, ai[r]);
        }
    }
}

template <typename T, int TB, int NT, uint32_t CLS>
__device__ __forceinline__ void wide_run(uint32_t &s, uint32_t end, SubD &S,
                                         const SubD *__restrict__ subs, const T *buf, uint32_t lane,
                                         uint32_t lanebits, const TermRec<double> *__restrict__ terms,
                                         double (&ar)[(1 << TB) / NT], double (&ai)[(1 << TB) / NT])
{
    constexpr int RP = (1 << TB) / NT;
    constexpr int LB = NT == 1024 ? 10 : NT == 512 ? 9 : NT == 256 ? 8 : 7;
    for (; s < end; s++) {
        const T *row = sub_lane_base<T, NT>(buf, lane, S.xl);
        const uint32_t xr = S.xl >> LB;
        if constexpr (CLS != kRunMulti) {
            T v[RP];
#pragma unroll
            for (int j = 0; j < RP; j++) v[j] = row[j * NT];
            asm volatile("" ::: "memory");
            const SubD Sn = subs[s + 1];     // the list has one sentinel record
            const uint32_t zr = (S.z >> LB) & (RP - 1);
            double c = flip_sign(S.c, parity_sign(lanebits & S.z));
            if constexpr (CLS == kRunReal1 || CLS == kRunImag1) c = opaque(c);
            with_row_flip<RP>(xr, [&](auto X) {
                wide_rows<T, RP, NT, CLS, decltype(X)::value>(v, c, zr, ar, ai);
            });
            S = Sn;
        } else {
            const SubD Sn = subs[s + 1];
            const uint32_t tb = S.z, te = (uint32_t)__double2loint(S.c);
            constexpr int RC = RP < 4 ? RP : 4;
#pragma unroll
            for (int r0 = 0; r0 < RP; r0 += RC) {
                double dr[RC], di[RC];
#pragma unroll
                for (int q = 0; q < RC; q++) { dr[q] = 0; di[q] = 0; }
                for (uint32_t t = tb; t < te; t++) {
                    const TermRec<double> C = terms[t];
                    const uint32_t lsb = parity_sign(lanebits & C.z);
                    const double cr = flip_sign(C.cr, lsb), ci = flip_sign(C.ci, lsb);
                    const uint32_t zr = (C.z >> LB) & (RP - 1);
#pragma unroll
                    for (int q = 0; q < RC; q++) {
                        const uint32_t rsb = parity_sign((r0 + q) & zr);
                        dr[q] += flip_sign(cr, rsb);
                        di[q] += flip_sign(ci, rsb);
                    }
                }
#pragma unroll
                for (int q = 0; q < RC; q++) {
                    const T v = row[((r0 + q) ^ xr) * NT];
                    const double x = (double)v.x, y = (double)v.y;
                    ar[r0 + q] = fmadd(dr[q], x, fmadd(-di[q], y, ar[r0 + q]));
                    ai[r0 + q] = fmadd(dr[q], y, fmadd(di[q], x, ai[r0 + q]));
                }
            }
            S = Sn;
        }
    }
}

template <typename R, int TB, int NT>
__global__ void __launch_bounds__(NT, (apply_waves_per_eu<R, TB, NT, 2>()))
k_apply_wide(const typename CxA<R>::T *__restrict__ in, typename CxA<R>::T *__restrict__ out,
             const GroupC *__restrict__ groups, int ngroups, int accumulate,
             const SubD *__restrict__ subs, const TermRec<double> *__restrict__ terms,
             const int *__restrict__ stop, TileMap tm)
{
    using T = typename CxA<R>::T;
    constexpr int RP = (1 << TB) / NT;
    const uint32_t t0 = first_amplitude<TB>(tm);
    if (stop && *stop) return;
    __shared__ T tile0[1 << TB];
    __shared__ T tile1[1 << TB];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid * (uint32_t)sizeof(T), lb = t0 | tid;
    double ar[RP], ai[RP];
#pragma unroll
    for (int r = 0; r < RP; r++) { ar[r] = 0; ai[r] = 0; }
    GroupC Gc = groups[0], Gn = groups[1];
    uint32_t s = 0;
    SubD S = subs[0];
    tile_dma<T, TB, NT>(in, t0 ^ (Gc.xh << TB), tile0);
    auto stage = [&](int g, const T *cur, T *nxt) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (g + 1 < ngroups) tile_dma<T, TB, NT>(in, t0 ^ (Gn.xh << TB), nxt);
        const GroupC Gnn = groups[g + 2];
        uint32_t e = Gc.begin;
#define RP_WIDE_RUN(CLS)                                                                    \
    e += Gc.n[CLS];                                                                         \
    wide_run<T, TB, NT, CLS>(s, e, S, subs, cur, lane, lb, terms, ar, ai);
        RP_WIDE_RUN(kRunReal0)
        RP_WIDE_RUN(kRunReal1)
        RP_WIDE_RUN(kRunImag0)
        RP_WIDE_RUN(kRunImag1)
        RP_WIDE_RUN(kRunMulti)
#undef RP_WIDE_RUN
        Gc = Gn;
        Gn = Gnn;
    };
    for (int g = 0; g < ngroups; g += 2) {
        stage(g, tile0, tile1);
        if (g + 1 >= ngroups) break;
        stage(g + 1, tile1, tile0);
    }
#pragma unroll
    for (int r = 0; r < RP; r++) {
        T *at = out + (uint64_t)t0 + r * NT + tid;
        double x = ar[r], y = ai[r];
        if (accumulate) {
            const T b = *at;
            x += (double)b.x;
            y += (double)b.y;
        }
        T o;
        o.x = (R)x;
        o.y = (R)y;
        *at = o;
    }
}

// ---------------------------------------------------------------------------
// The apply with the first Gram-Schmidt pass's coefficients formed in its
// epilogue: after writing its output tile w, the workgroup reads the same
// rows of V_0..V_{k-1} and writes its FP64 partials of <V_q|w> (columns
// 2q, 2q+1) and of ||w||^2 (column 2 kMaxSweep) to row blockIdx.x of part.
// The w values are the rounded ones just written, so the coefficients are
// those of the stored vector.
// ---------------------------------------------------------------------------
constexpr int kMaxSweep = RP_MAX_SWEEP_VECS;
constexpr int kEpiChunk = 8;                        // vectors per block reduction
struct VecPtrs64 { const void *p[kMaxSweep]; };

// sum NV per-thread doubles over the NT-thread workgroup into sh[(NT/64)*NV + q]
template <int NT, int NV>
__device__ __forceinline__ void wg_reduce(double (&v)[NV], double *sh)
{
    constexpr int W = NT / 64;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < NV; q++) {
        double x = v[q];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        v[q] = x;
    }
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < NV; q++) sh[wid * NV + q] = v[q];
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        double s = 0;
        for (int w = 0; w < W; w++) s += sh[w * NV + threadIdx.x];
        sh[W * NV + threadIdx.x] = s;
    }
    __syncthreads();
}

template <typename R, typename A, int TB, int NT, int D, bool GA>
__global__ void __launch_bounds__(NT, (apply_waves_per_eu<R, TB, NT, D>()))
k_apply_tiled_gs(const typename CxA<R>::T *__restrict__ in, typename CxA<R>::T *__restrict__ out,
                 const GroupRuns *__restrict__ groups, int ngroups,
                 const SubRec<A> *__restrict__ subs, const TermRec<A> *__restrict__ terms,
                 VecPtrs64 V, int k, double *__restrict__ part, int width, TileMap tm)
{
    using T = typename CxA<R>::T;
    constexpr int TILE = 1 << TB;
    constexpr int RP = TILE / NT;
    constexpr int NV = 2 * kEpiChunk + 1;
    __shared__ T tile0[TILE];
    __shared__ T tile1[TILE];
    __shared__ T tile2[D > 2 ? TILE : 1];
    __shared__ T tile3[D > 3 ? TILE : 1];
    __shared__ double sh[(NT / 64 + 1) * NV];
    T wv[RP];
    const uint32_t t0 = tile_index(tm) << TB;
    apply_tile<R, A, TB, NT, D, GA>(in, out, groups, ngroups, subs, terms, 0, tile0, tile1, tile2,
                                    tile3, t0, wv);
    const uint32_t tid = threadIdx.x;
    double wn2 = 0;
#pragma unroll
    for (int r = 0; r < RP; r++) wn2 += (double)wv[r].x * wv[r].x + (double)wv[r].y * wv[r].y;
    double *row = part + (size_t)blockIdx.x * width;
    for (int q0 = 0; q0 == 0 || q0 < k; q0 += kEpiChunk) {
        double acc[NV];
#pragma unroll
        for (int q = 0; q < NV; q++) acc[q] = 0;
#pragma unroll
        for (int q = 0; q < kEpiChunk; q++) {
            if (q0 + q < k) {
                const T *vq = (const T *)V.p[q0 + q];
#pragma unroll
                for (int r = 0; r < RP; r++) {
                    const T x = vq[(uint64_t)t0 + r * NT + tid];
                    const double xr = x.x, xi = x.y, yr = wv[r].x, yi = wv[r].y;
                    acc[2 * q] += xr * yr + xi * yi;
                    acc[2 * q + 1] += xr * yi - xi * yr;
                }
            }
        }
        if (q0 == 0) acc[2 * kEpiChunk] = wn2;
        wg_reduce<NT, NV>(acc, sh);
        constexpr int W = NT / 64;
        if ((int)tid < 2 * kEpiChunk && q0 + (int)tid / 2 < k) row[2 * q0 + tid] = sh[W * NV + tid];
        if (q0 == 0 && tid == 2 * kEpiChunk) row[2 * kMaxSweep] = sh[W * NV + tid];
    }
}

constexpr int tiling_key(int tb, int nt, int d) { return tb * 100000 + nt * 10 + d; }

// the tilings the tiled kernel is instantiated for: {tile bits, threads,
// pipeline depth, element bytes (0: both precisions)}
struct TilingDesc { int tb, nt, depth, esz; };
// Tile bits 0 is the kernel without tiles, its depth the number of term slices.
constexpr int kSplitMaxLen = 16;       // with any slice count up to here
constexpr TilingDesc kTilings[] = {
    {0, kSmallThreads, 1, 0}, {0, kSmallThreads, 8, 0}, {0, kSmallThreads, 32, 0},
    {0, kSmallThreads, 128, 0},
    {8, 128, 2, 0}, {10, 128, 2, 0}, {11, 256, 4, 16}, {12, 512, 2, 0},
    {12, 512, 3, 8}, {12, 512, 4, 8}, {12, 1024, 2, 8}, {13, 1024, 2, 8}};

// Where the kernel without tiles may be set: up to kSplitMaxLen sites with any
// slice count, and beyond in the shapes an upload chooses itself, which keep no
// partial sums in memory (8 slices are added in LDS)
static bool wave_allowed(int len, uint64_t flips, int depth)
{
    if (len <= kSplitMaxLen) return true;
    return depth == 1 ? len <= kWaveMaxLen || flips <= (uint64_t)kWaveMaxFlips
                      : depth == 8 && len <= kWaveMaxLen;
}

static bool tiling_instantiated(int prec, int tb, int nt, int d)
{
    for (const TilingDesc &t : kTilings)
        if (t.tb == tb && t.nt == nt && t.depth == d &&
            (t.esz == 0 || t.esz == (int)elem_bytes(prec)))
            return true;
    return false;
}

// what the choice of a layout looks at in a term list (zero coefficients
// included)
struct ListShape {
    uint64_t terms = 0, flips = 0;    // terms, distinct flip masks
    uint64_t pieces = 0;              // flip masks in pieces of kWavePiece terms
    uint64_t groups = 0;              // distinct flip masks above 2^12 tiles
    uint64_t shared = 0;              // terms of flip masks that have several
    uint64_t by_row = 0;              // those with a phase bit among the row bits of
                                      // k_apply_wave
};
// ascending order of v by bits [1, bits); long lists by a radix sort (10626
// terms at 12 sites 0.05 ms, std::sort 0.5)
static void sort_masks(std::vector<uint64_t> &v, int bits)
{
    if (v.size() < 512) {
        std::sort(v.begin(), v.end());
        return;
    }
    constexpr int kDigit = 11;
    std::vector<uint64_t> w(v.size());
    for (int s = 1; s < bits; s += kDigit) {
        uint64_t at[(1 << kDigit) + 1] = {0};
        for (uint64_t e : v) at[(e >> s & ((1 << kDigit) - 1)) + 1]++;
        for (int d = 0; d < 1 << kDigit; d++) at[d + 1] += at[d];
        for (uint64_t e : v) w[at[e >> s & ((1 << kDigit) - 1)]++] = e;
        v.swap(w);
    }
}
static ListShape list_shape(const uint64_t *bits, uint64_t n)
{
    // flip mask, and whether the phase mask has a row bit (sites 6 and 7)
    std::vector<uint64_t> v(n);
    uint64_t any = 0;
    for (uint64_t t = 0; t < n; t++) {
        v[t] = (uint64_t)pext_even(bits[t]) << 1 | ((bits[t] >> 13 & 5) != 0);
        any |= v[t];
    }
    sort_masks(v, any ? 64 - __builtin_clzll(any) : 1);
    ListShape L;
    L.terms = n;
    for (uint64_t i = 0, j; i < n; i = j) {
        uint64_t rows = 0;
        for (j = i; j < n && v[j] >> 1 == v[i] >> 1; j++) rows += v[j] & 1;
        L.flips++;
        L.pieces += (j - i + kWavePiece - 1) / kWavePiece;
        if (!i || v[i] >> 13 != v[i - 1] >> 13) L.groups++;
        if (j - i == 1) continue;
        L.shared += j - i;
        L.by_row += rows;
    }
    return L;
}

// Whether a list is long enough for the 16-byte records of k_apply_wide.  The
// 48-byte ones of a short list stay in the 16 KiB scalar cache, and reading
// them costs less than the branch on the row flip that k_apply_wide makes for
// every record.  us per apply, single-term masks, 48-byte / 16-byte records:
//   complex<float> 12/1024:   20 sites, 150 masks 76 / 63; 22 sites, 150 222 / 219;
//     24 sites, 150 895 / 936, 200 1095 / 1119, 240 1421 / 1355; 25 sites, 200
//     2213 / 2364, 240 2804 / 2767
//   complex<double> 12/512:   20 sites, 150 masks 94 / 80; 22 sites, 60 158 / 163;
//     24 sites, 200 2082 / 2202, 240 3032 / 2635; 26 sites, 200 9923 / 10613,
//     240 14464 / 12210, and 60 masks of 3 terms 6577 / 7640, 200 of 3 24734 / 22615
static bool long_list(int len, uint64_t flips, uint64_t shared)
{
    return flips + shared / 4 >= (len <= 20 ? 0u : len <= 22 ? 110u : 234u);
}

// Amplitudes per lane of the kernel without tiles: four where that leaves
// enough wavefronts.  Every term's sign and record is then shared by four
// amplitudes, and the scalar instructions of a flip mask (about 35), which
// bound the lists of many masks, by 256 instead of 64.  At 12 sites one
// amplitude a lane has 8192 wavefronts in 128 slices, four have 2048: 1000
// masks 9.1 / 10.2 us, 600 masks of 4 terms 14.1 / 13.4.
static int wave_rows(int len, int depth, uint64_t pieces, uint64_t nterms)
{
    if (len > kSplitMaxLen || depth == 1)
        return depth <= 8 && ((uint64_t)depth << len) >= (1ull << 20) ? 4 : 1;
    return len > 8 && ((uint64_t)depth << (len - 8)) >= 2048 &&
                   pieces + nterms >= (uint64_t)((len == 12 ? 20 : 10) * depth)
               ? 4 : 1;
}

// Slices of the flip masks for the kernel without tiles.  With one amplitude
// per lane the most that keep about 8192 wavefronts (the GPU holds that many;
// with 8 slices each lane has four amplitudes from 17 sites on) and the work
// of 22 terms a slice.  From 13 to 16 sites longer lists take four amplitudes
// per lane and the slices that give at least 2048 wavefronts; more of them
// only where the list is long enough to pay for adding the sums of 8 to 16
// times as many workgroups.  us per apply, one amplitude a lane (8 slices at
// 15 and 16 sites, 32 below) / four, masks x terms a mask, complex<float>:
//   13 sites: 300 x 1  6.3 / 7.8 (not taken), 300 x 4  12.4 / 10.1, 1000 x 4  30.5 / 17.8
//   14 sites: 100 x 4  10.4 / 9.6 (32 slices), 1000 x 1  18.8 / 15.7, 4000 x 4  216 / 99
//   15 sites: 300 x 1  11.5 / 9.6, 1000 x 1  31.8 / 20.4, 1000 x 4  108 / 48.8
//   16 sites: 300 x 1  18.4 / 12.9 (8 slices), 1000 x 1  53 / 37, 4000 x 4  765 / 357
// and FP32 sums, whose wavefronts need half the registers, 128 slices at 15
// sites: 4000 x 1  64.4 (32) / 61.8, 4000 x 4  155 / 129, 1000 x 1  19.3 / 20.2.
static int wave_depth(int len, uint64_t pieces, uint64_t nterms, int acc64)
{
    const uint64_t chunks = len > 6 ? 1ull << (len - 6) : 1;
    int d = 1;
    for (int s : {8, 32, 128})
        if (chunks * s <= (s == 8 ? 65536 : 8192) && pieces >= (uint64_t)s &&
            6 * pieces + nterms >= (uint64_t)(22 * s))
            d = s;
    if (len < 13 || len > kSplitMaxLen) return d;
    uint64_t more = 0;             // list length from which more slices pay
    for (int s : {8, 32, 128}) {
        const uint64_t waves = (uint64_t)s << (len - 8);
        if (waves < 2048 || pieces < (uint64_t)s) continue;
        if (waves > (acc64 ? 8192u : 16384u)) break;
        if (waves > 8192) more = 4096;
        if (pieces + nterms >= std::max<uint64_t>(10 * s, more)) d = s;
        more = 1280;
    }
    return d;
}

// Whether the apply takes no tiles by default.  Without tiles every flip mask
// reads the state once, with tiles every group of masks that agree above the
// tile; a term of a shared mask costs the tiled kernel a product for every
// row, the other only a sum, and that once for four rows unless the term has
// a phase bit among the row bits.
//
// Short chains have too few tiles for the 256 CUs.  us per apply without
// tiles / with (12, 512, 2), FP64 sums:
//   sparse SYK, k = 8, complex<float>:  16 sites 17 / 93, 18 sites 41 / 110,
//     19 sites 80 / 136 (group accumulation 80 / 87), 20 sites 154 / 153,
//     21 sites 321 / 210; complex<double> 19 sites 92 / 137, 20 191 / 160
//   random masks of single terms at 19 sites: 1000 248 / 309, 4000 964 / 1107;
//     but group accumulation 300 76 / 79, 1000 239 / 194 (12/1024), 4000 937 /
//     649; from 12000 masks on its tiled kernel's records overflow, 2810 / 3119
//
// From 20 sites on few flip masks (up to 40) that share terms:
//   XXZ with fields (4 terms a mask), FP64 sums:  20 sites 17 / 40, 24 sites
//     201 / 431, 26 sites 1050 / 1814, complex<double> 24 sites 385 / 728
//   with group accumulation / its best tiling:  24 sites 195 / 310, 26 sites
//     1052 / 1329
//   random masks, whose terms mostly have row bits: FP64 sums, 24 sites, 20
//     masks x 4 terms  375 / 381, 40 x 20  1911 / 2264; group accumulation
//     375 / 313 and 1916 / 1586; FP32 sums 312 / 290 and 1531 / 1687
// Two terms a mask is the narrow case, decided by how many groups the masks
// make; us, masks / groups:
//   complex<float>, FP64 sums: 26 sites 10/10 802 / 582, 40/33 1947 / 2071, 27
//     sites 20/15 2516 / 2034, XY chain 26/15 2223 / 2454
//   group accumulation: 22 sites 20/18 58 / 71, 40/20 116 / 106, XY chain
//     21/11 46 / 62; 24 sites 10/9 158 / 141, XY chain 23/13 186 / 235
//   FP32 sums: 20 sites 40/21 34 / 48, 23 sites 40/20 175 / 196, 24 sites 10/9
//     154 / 132, 25 sites 40/32 972 / 840, XY chain 24/14 448 / 472
//   complex<double>: 22 sites 40/28 194 / 243, 23 sites 40/28 465 / 449, 26
//     sites 40/30 4252 / 3666, 20/14 1518 / 1877, XY chain 25/15 1885 / 2640
static bool without_tiles(int prec, int len, const ListShape &L, int group_acc, int acc64)
{
    const bool single = 2 * L.terms < 3 * L.flips;
    if (len <= kWaveMaxLen)
        return !(len == kWaveMaxLen && group_acc && single && L.flips >= 600 && L.flips <= 8192);
    if (L.flips > kWaveMaxFlips || L.terms < 2 * L.flips) return false;
    const bool fp32 = prec == RP_C64 && (group_acc || !acc64), rows = 4 * L.by_row > L.terms;
    const double per = (double)L.flips / (double)L.groups;      // masks a group
    if (2 * L.terms < 5 * L.flips) {      // two terms a mask
        if (group_acc && rows) return len < 24 && per < 1.5;
        if (fp32) return len < 24 || (len == 24 && per >= 7. / 6) ||
                         (len == 25 && !group_acc && per >= 5. / 3);
        if (prec == RP_C128) return len < 23 || per >= 1.4;
        return len < 26 || per >= (len == 26 ? 7. / 6 : 1.4);
    }
    return !fp32 || !rows ||
           (!group_acc && (len < 22 || L.terms >= 6 * L.flips || per < 1.5));
}

// default tiling (RP_TERMS_AUTOTUNE measures the alternatives)
static void choose_tiling(int prec, int len, const ListShape &L, int group_acc, int acc64, int *tb,
                          int *nt, int *depth)
{
    *depth = 2;
    if (without_tiles(prec, len, L, group_acc, acc64)) {
        *tb = 0;
        *nt = kSmallThreads;
        *depth = wave_depth(len, L.pieces, L.terms, acc64);
        return;
    }
    // Tiles of 2^12 amplitudes by 512 threads; for complex<double> the largest
    // in two 64 KiB buffers.  us per apply with 12/512, 12/1024, 13/1024:
    //   group accumulation, sparse SYK: 20 sites 101, 89, 118; 21 sites 140,
    //     161, 139; 25 sites 3283, 3635, 3325; 26 sites (beyond the Infinity
    //     Cache, where the workgroups of a CU drift apart and the larger tile has
    //     fewer passes) 10579, 8946, 7899; 28 sites 59465, 51047, 40086
    //   but masks that share terms, 60 x 3: 24 sites 777, 720, 884; 26 sites
    //     2953, 2725, 3484; 28 sites 12773, 11840, 15067; and few single ones:
    //     26 sites, 20 masks 869, 863, 983, 60 masks 1702, 1726, 1825 in one
    //     list and 2225, 2092, 2098 in another
    //   FP64 sums, sparse SYK: 20 sites 137, 116, 178; 24 sites 1896, 1842, 1984;
    //     26 sites 9655, 9546, 10130; 27 sites 20634, 20351, 20351; 28 sites
    //     44428, 49490, 44979
    //   200 single masks: 24 sites 1133, 1119, -; 27 sites 11994, 11067, 12870;
    //     28 sites 23980, 24228, 26742; 60 x 3: 26 sites 3853, 3517, 4777; 28
    //     sites 14982, 13698, 18917
    *tb = 12;
    *nt = 512;
    if (prec != RP_C64 || (!group_acc && !acc64)) return;
    const bool single = 2 * L.terms < 3 * L.flips;
    if (group_acc) {
        if (single && (len >= 28 || (len >= 26 && L.flips > 64))) *tb = 13;
        if (!single || len >= 26 || len <= 20) *nt = 1024;
    } else if (!single || (len < 28 && long_list(len, L.flips, L.shared))) {
        *nt = 1024;
    }
}

// the compact lists of the tiled tables (complex<float> states, FP64 term
// coefficients): one 16-byte record per sub in the SubRec order,
// coefficients rounded to float, one sentinel record; one 16-byte header
// per group, two sentinel headers; the multi-sub terms in FP32.  False when
// a class run of some group has more than 255 subs (the header's count
// width): the handle then keeps the SubRec kernel.
static bool compact_stream(const Tables<double> &tab, int tb, int nt, std::vector<GroupC> &cg,
                           std::vector<SubC> &cs, std::vector<TermC> &ct)
{
    for (const TermRec<double> &t : tab.terms)
        ct.push_back({t.z, (float)t.cr, (float)t.ci, stream_row(t.z, tb, nt)});
    for (const GroupRuns &G : tab.groups) {
        GroupC h{};
        h.xh = G.xh;
        h.begin = G.b[0];
        // this kernel's row bits are not the SubRec kernel's: the single-term
        // real and imaginary subs are classed again
        std::vector<SubC> run[kRuns];
        for (uint32_t k = 0; k < kRuns; k++) {
            for (uint32_t i = G.b[k]; i < G.b[k + 1]; i++) {
                const SubRec<double> &S = tab.subs[i];
                const uint32_t zr = k == kRunMulti ? 0 : stream_row(S.z, tb, nt);
                SubC c{(S.xl & (2u * nt - 2u)) * 8u | stream_row(S.xl, tb, nt) << 16 | zr << 24, S.z,
                       0.f, 0.f};
                const uint32_t cls = k >= kRunCplx ? k : (k & ~1u) | (zr ? 1u : 0u);
                if (k == kRunMulti) {
                    c.z = S.term_begin;
                    memcpy(&c.c0, &S.term_end, sizeof(float));
                } else if (k == kRunImag0 || k == kRunImag1) {
                    c.c0 = S.fi;
                } else {
                    c.c0 = S.fr;
                    c.c1 = S.fi;
                }
                run[cls].push_back(c);
            }
        }
        for (uint32_t k = 0; k < kRuns; k++) {
            if (run[k].size() > 255) return false;
            h.n[k] = (uint8_t)run[k].size();
            cs.insert(cs.end(), run[k].begin(), run[k].end());
        }
        cg.push_back(h);
    }
    GroupC end{};
    end.begin = (uint32_t)cs.size();
    cg.push_back(end);
    cg.push_back(end);
    cs.push_back({0, 0, 0.f, 0.f});
    if (ct.empty()) ct.push_back(TermC{});
    return true;
}

// Where k_apply_wide takes the place of the SubRec kernel, the list being
// long enough: for complex<float> in every pipeline of two tiles (sparse SYK,
// 24 qubits: 12/512 1.96 -> 1.90 ms, 12/1024 1.97 -> 1.84, 13/1024 2.19 -> 1.98),
// for complex<double> with 2^12 tiles (24 qubits 4.01 -> 3.39 ms); with 2^10
// tiles of 128 threads its workgroups drift apart in group order and lose
// each other's tiles in L2 (24 qubits 3.79 -> 5.78 ms), and so do those of
// complex<float> 2^12 tiles beyond the Infinity Cache (12/512 at 26 qubits
// 9.65 -> 10.01 ms, at 25 320 masks 3.81 -> 4.13 ms; 12/1024 there 3.79 -> 3.82).
static bool wide_table(int prec, int acc64, int len, int tb, int nt, int depth, uint64_t flips,
                       uint64_t shared)
{
    if (!acc64 || depth != 2) return false;
    if (prec == RP_C64 ? tb <= 12 && len > (nt == 1024 ? 25 : 24) : tb != 12) return false;
    return long_list(len, flips, shared);
}
template <typename R, typename A, int TB, int D> constexpr bool wide_tiling()
{
    return sizeof(A) == 8 && D == 2 && (sizeof(R) == 4 || TB == 12);
}

// the lists of k_apply_wide, in the SubRec order; a complex single term is
// appended to the term list.  False as for compact_stream.
static bool compact_wide(Tables<double> &tab, std::vector<GroupC> &cg, std::vector<SubD> &cs)
{
    for (const GroupRuns &G : tab.groups) {
        GroupC h{};
        h.xh = G.xh;
        h.begin = G.b[0];
        for (uint32_t k = 0; k < kRuns; k++) {
            const uint32_t cls = k == kRunCplx ? (uint32_t)kRunMulti : k;
            if (h.n[cls] + (G.b[k + 1] - G.b[k]) > 255) return false;
            h.n[cls] += (uint8_t)(G.b[k + 1] - G.b[k]);
            for (uint32_t i = G.b[k]; i < G.b[k + 1]; i++) {
                const SubRec<double> &S = tab.subs[i];
                SubD c{S.xl, S.z, k == kRunImag0 || k == kRunImag1 ? S.ci : S.cr};
                if (cls == kRunMulti) {
                    uint64_t end = S.term_end;
                    c.z = S.term_begin;
                    if (k == kRunCplx) {
                        c.z = (uint32_t)tab.terms.size();
                        tab.terms.push_back({S.z, 0, S.cr, S.ci});
                        end = tab.terms.size();
                    }
                    memcpy(&c.c, &end, sizeof(double));
                }
                cs.push_back(c);
            }
        }
        cg.push_back(h);
    }
    GroupC end{};
    end.begin = (uint32_t)cs.size();
    cg.push_back(end);
    cg.push_back(end);
    cs.push_back({0, 0, 0.0});
    return true;
}

// bytes of the partial sums of k_apply_wave: (re, im) of every amplitude from
// each workgroup of its slices, where there are several
static size_t wave_part_bytes(const rp_terms *h)
{
    const int wgs = h->depth / wave_width(h->depth);
    const uint64_t dim = std::max<uint64_t>(64ull * h->rows, 1ull << h->len);
    return wgs > 1 ? (size_t)dim * 2 * sizeof(double) * wgs : 0;
}

// log2 of the tiled kernel's resident workgroups per XCD (32 CUs) at the
// occupancy apply_waves_per_eu gives it: the p of its output-tile map
static int xcd_resident_bits(int prec, int tb, int nt, int depth)
{
    if (!tb) return 0;
    const int lds = depth * (1 << tb) * (int)elem_bytes(prec);
    int wg = std::min((160 * 1024) / lds, (nt == 1024 ? 2048 : 1024) / nt);
    wg = std::max(wg, 1);
    int p = 5;
    while ((2 << p) <= 32 * wg) p++;
    return p;
}

// The tables of k_apply_wave from the x-sorted terms: one record per flip
// mask (or piece of it), its terms by class, and the cuts of the flip masks into h->depth
// slices of about equal work (a flip mask costs about as much as six terms:
// the gather, its address and the products).
template <typename A, typename UP>
static int upload_wave(rp_terms *h, const std::vector<FlatTerm<A>> &flat, UP &&up)
{
    const uint64_t dim = 1ull << h->len;
    const size_t piece = h->depth > 1 ? kWavePiece : flat.size();
    auto run_end = [&](size_t i) {
        size_t j = i;
        while (j < flat.size() && flat[j].x == flat[i].x && j - i < piece) j++;
        return j;
    };
    uint64_t pieces = 0;
    for (size_t i = 0; i < flat.size(); i = run_end(i)) pieces++;
    h->rows = wave_rows(h->len, h->depth, pieces, flat.size());
    std::vector<SubW<A>> subs;
    std::vector<TermW<A>> terms;
    std::vector<uint32_t> flips;
    std::vector<uint64_t> cost(1, 0);
    terms.reserve(flat.size());
    // bit l: parity of l & z, the sum of the patterns of z's bits
    auto lanes = [](uint32_t z) {
        constexpr uint64_t bit[6] = {0xaaaaaaaaaaaaaaaaull, 0xccccccccccccccccull,
                                     0xf0f0f0f0f0f0f0f0ull, 0xff00ff00ff00ff00ull,
                                     0xffff0000ffff0000ull, 0xffffffff00000000ull};
        uint64_t m = 0;
        for (int b = 0; b < 6; b++) m ^= bit[b] & -(uint64_t)(z >> b & 1);
        return m;
    };
    const uint32_t rowbits = 64u * (h->rows - 1);
    for (size_t i = 0; i < flat.size();) {
        const size_t j = run_end(i);
        bool re = true, im = true;
        for (size_t q = i; q < j; q++) {
            re = re && flat[q].ci == 0;
            im = im && flat[q].cr == 0;
        }
        SubW<A> S{};
        uint64_t work = 6;
        if (j - i <= 2 && (re || im)) {
            const FlatTerm<A> &a = flat[i], &b = flat[j - 1];
            S.kind = (re ? 0 : kWaveImag) | (((a.z | b.z) & rowbits) ? kWaveRow : 0);
            S.c0 = re ? a.cr : a.ci;
            S.z0 = a.z;
            S.l0 = lanes(a.z);
            if (j - i == 2) {
                S.kind |= kWaveTwo;
                S.c1 = re ? b.cr : b.ci;
                S.z1 = b.z;
                S.l1 = lanes(b.z);
            }
            work += j - i;
        } else {
            // counted, then placed: real parts without and with phase bits
            // among the row bits, then imaginary ones
            uint32_t n[4] = {0, 0, 0, 0}, at[4];
            for (size_t q = i; q < j; q++) {
                const int byrow = (flat[q].z & rowbits) != 0;
                n[byrow] += flat[q].cr != 0;
                n[2 + byrow] += flat[q].ci != 0;
            }
            S.kind = kWaveMulti;
            S.term = (uint32_t)terms.size();
            at[0] = S.term;
            for (int k = 1; k < 4; k++) at[k] = at[k - 1] + n[k - 1];
            terms.resize(at[3] + n[3]);
            for (size_t q = i; q < j; q++) {
                const int byrow = (flat[q].z & rowbits) != 0;
                const uint64_t l = lanes(flat[q].z);
                if (flat[q].cr != 0) terms[at[byrow]++] = {l, flat[q].cr, flat[q].z, 0};
                if (flat[q].ci != 0) terms[at[2 + byrow]++] = {l, flat[q].ci, flat[q].z, 0};
            }
            S.z0 = n[0];
            S.z1 = n[1];
            S.l0 = (uint64_t)n[3] << 32 | n[2];
            work += n[0] + n[2] + (uint64_t)h->rows * (n[1] + n[3]);
        }
        cost.push_back(cost.back() + work);
        subs.push_back(S);
        flips.push_back(flat[i].x);
        i = j;
    }
    const size_t nsubs = subs.size();
    flips.resize(nsubs + kWavePad, 0);
    subs.resize(nsubs + kWavePad);
    std::vector<uint32_t> cut;
    for (int s = 0; s <= h->depth; s++) {
        const uint64_t want = cost.back() * (uint64_t)s / (uint64_t)h->depth;
        cut.push_back((uint32_t)(std::lower_bound(cost.begin(), cost.end(), want) - cost.begin()));
    }
    int st;
    if ((st = up(&h->d_wflips, flips.data(), flips.size() * sizeof(uint32_t)))) return st;
    if ((st = up(&h->d_wsubs, subs.data(), subs.size() * sizeof(SubW<A>)))) return st;
    if ((st = up(&h->d_wterms, terms.data(), terms.size() * sizeof(TermW<A>)))) return st;
    if ((st = up(&h->d_wcut, cut.data(), cut.size() * sizeof(uint32_t)))) return st;
    if (wave_part_bytes(h)) {
        const size_t chunks = std::max<uint64_t>(1, dim / (64 * h->rows));
        // the partial sums are written before they are read: only the arrival
        // counters behind them start at zero
        const std::vector<unsigned> zero(chunks, 0u);
        const size_t at = wave_part_bytes(h), bytes = at + chunks * sizeof(unsigned);
        if (dev_malloc(&h->d_split, bytes) != hipSuccess) {
            (void)hipGetLastError();
            return set_error(RP_ERR_OUT_OF_MEMORY, "Failed to allocate %zu bytes on GPU device.",
                             bytes);
        }
        RP_CHECK_HIP(hipMemcpyAsync((char *)h->d_split + at, zero.data(), bytes - at,
                                    hipMemcpyHostToDevice, ctx().stream));
        RP_CHECK_HIP(hipStreamSynchronize(ctx().stream));     // zero is a host temporary
    }
    // the tables are host temporaries
    RP_CHECK_HIP(hipStreamSynchronize(ctx().stream));
    return RP_OK;
}

template <typename R, typename A>
static int upload_impl(rp_terms *h, const uint64_t *bits, const double *coeff, uint64_t n)
{
    Tables<A> tab;
    int st = build_tables<R, A>(h->len, h->tile_bits, h->threads, bits, coeff, n, tab,
                                xcd_resident_bits(h->prec, h->tile_bits, h->threads, h->depth));
    if (st) return st;
    h->tmap = tab.tilemap;
    auto &groups = tab.groups;
    auto &subs = tab.subs;
    auto &terms = tab.terms;
    auto &flat = tab.flat;
    const int tb = h->tile_bits;
    const uint64_t nflips = tab.nflips;
    h->nterms = tab.nterms;
    h->nflips = nflips;
    h->ngroups = tb ? groups.size() : 1;
    h->nsubs = subs.size();
    Context &c = ctx();
    auto up = [&](void **dst, const void *src, size_t bytes) -> int {
        if (!bytes) return RP_OK;
        hipError_t e = dev_malloc((void **)dst, bytes);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            return set_error(RP_ERR_OUT_OF_MEMORY, "Failed to allocate %zu bytes on GPU device.",
                             bytes);
        }
        RP_CHECK_HIP(hipMemcpyAsync(*dst, src, bytes, hipMemcpyHostToDevice, c.stream));
        return RP_OK;
    };
    if (!tb && (st = upload_wave<A>(h, flat, up))) return st;
    if constexpr (sizeof(A) == 8) {
        std::vector<GroupC> cg;
        std::vector<SubD> cs;
        if (tb && !h->group_acc &&
            wide_table(h->prec, h->acc64, h->len, tb, h->threads, h->depth, nflips,
                       terms.size()) &&
            compact_wide(tab, cg, cs)) {
            if ((st = up(&h->d_cgroups, cg.data(), cg.size() * sizeof(GroupC)))) return st;
            if ((st = up(&h->d_csubs, cs.data(), cs.size() * sizeof(SubD)))) return st;
            RP_CHECK_HIP(hipStreamSynchronize(c.stream));     // host temporaries
        }
    }
    if (tb) {
        if ((st = up(&h->d_groups, groups.data(), groups.size() * sizeof(GroupRuns)))) return st;
        if ((st = up(&h->d_subs, subs.data(), subs.size() * sizeof(SubRec<A>)))) return st;
        if ((st = up(&h->d_terms, terms.data(), terms.size() * sizeof(TermRec<A>)))) return st;
    }
    if constexpr (sizeof(R) == 4 && sizeof(A) == 8) {
        std::vector<GroupC> cg;
        std::vector<SubC> cs;
        std::vector<TermC> ct;
        if (tb && h->group_acc && compact_stream(tab, tb, h->threads, cg, cs, ct)) {
            if ((st = up(&h->d_cgroups, cg.data(), cg.size() * sizeof(GroupC)))) return st;
            if ((st = up(&h->d_csubs, cs.data(), cs.size() * sizeof(SubC)))) return st;
            if ((st = up(&h->d_cterms, ct.data(), ct.size() * sizeof(TermC)))) return st;
        }
    }
    RP_CHECK_HIP(hipStreamSynchronize(c.stream));
    return RP_OK;
}

static void free_handle(rp_terms *h)
{
    if (!h) return;
    if (h->d_groups) (void)hipFree(h->d_groups);
    if (h->d_subs) (void)hipFree(h->d_subs);
    if (h->d_terms) (void)hipFree(h->d_terms);
    for (void *p : {h->d_cgroups, h->d_csubs, h->d_cterms, h->d_wflips, h->d_wsubs,
                    h->d_wterms, h->d_wcut, h->d_split})
        if (p) (void)hipFree(p);
    delete h;
}

template <typename R, typename A, int TB, int NT, int D = 2>
static int launch_tiled(rp_terms *h, void *res, const void *vec, int accumulate, const int *stop)
{
    using T = typename CxA<R>::T;
    const uint64_t grid = (1ull << h->len) >> TB;
    if constexpr (sizeof(R) == 4 && sizeof(A) == 8 && D == 2) {
        if (h->group_acc && h->d_csubs) {
            RP_LAUNCH(RP_KERNEL_APPLY, (k_apply_stream<TB, NT>), dim3((unsigned)grid), dim3(NT), 0,
                      (const T *)vec, (T *)res, (const GroupC *)h->d_cgroups, (int)h->ngroups,
                      accumulate, (const SubC *)h->d_csubs, (const TermC *)h->d_cterms, stop,
                      h->tmap);
            return RP_OK;
        }
        if (h->group_acc) {
            RP_LAUNCH(RP_KERNEL_APPLY, (k_apply_tiled<R, A, TB, NT, D, true>), dim3((unsigned)grid),
                      dim3(NT), 0, (const T *)vec, (T *)res, (const GroupRuns *)h->d_groups,
                      (int)h->ngroups, accumulate, (const SubRec<A> *)h->d_subs,
                      (const TermRec<A> *)h->d_terms, stop, h->tmap);
            return RP_OK;
        }
    }
    if constexpr (wide_tiling<R, A, TB, D>()) {
        if (h->d_csubs) {
            RP_LAUNCH(RP_KERNEL_APPLY, (k_apply_wide<R, TB, NT>), dim3((unsigned)grid), dim3(NT), 0,
                      (const T *)vec, (T *)res, (const GroupC *)h->d_cgroups, (int)h->ngroups,
                      accumulate, (const SubD *)h->d_csubs, (const TermRec<double> *)h->d_terms,
                      stop, h->tmap);
            return RP_OK;
        }
    }
    RP_LAUNCH(RP_KERNEL_APPLY, (k_apply_tiled<R, A, TB, NT, D, false>), dim3((unsigned)grid),
              dim3(NT), 0, (const T *)vec, (T *)res, (const GroupRuns *)h->d_groups,
              (int)h->ngroups, accumulate, (const SubRec<A> *)h->d_subs,
              (const TermRec<A> *)h->d_terms, stop, h->tmap);
    return RP_OK;
}

// res = 0: the apply of an operator without terms
template <typename T>
__global__ void __launch_bounds__(kSmallThreads)
k_apply_none(T *__restrict__ out, uint64_t dim, const int *__restrict__ stop)
{
    if (stop && *stop) return;
    for (uint64_t i = blockIdx.x * (uint64_t)kSmallThreads + threadIdx.x; i < dim;
         i += (uint64_t)gridDim.x * kSmallThreads) {
        T e;
        e.x = 0;
        e.y = 0;
        out[i] = e;
    }
}

template <typename R, typename A>
static int apply_impl(rp_terms *h, void *res, const void *vec, int accumulate, const int *stop)
{
    using T = typename CxA<R>::T;
    const uint64_t dim = 1ull << h->len;
    if (h->nterms == 0) {
        if (accumulate) return RP_OK;
        const uint64_t wgs = (dim + kSmallThreads - 1) / kSmallThreads;
        RP_LAUNCH(RP_KERNEL_APPLY, k_apply_none<T>, dim3((unsigned)std::min<uint64_t>(wgs, 8192)),
                  dim3(kSmallThreads), 0, (T *)res, dim, stop);
        return RP_OK;
    }
    if (h->tile_bits == 0) {
        const uint64_t chunks = std::max<uint64_t>(1, dim / (64 * h->rows));
        const int w = wave_width(h->depth);
        const dim3 grid = h->depth == 1 ? dim3((unsigned)((chunks + w - 1) / w))
                                        : dim3((unsigned)chunks, h->depth / w);
        unsigned *count = (unsigned *)((char *)h->d_split + wave_part_bytes(h));
        const bool big = dim * sizeof(T) >= (1ull << 32);
#define RP_WAVE(ROWS, W, BIG)                                                     \
    RP_LAUNCH(RP_KERNEL_APPLY, (k_apply_wave<R, A, ROWS, W, BIG>), grid, dim3(64 * W), 0,         \
              (const T *)vec, (T *)res, dim, (const uint32_t *)h->d_wflips,                      \
              (const SubW<A> *)h->d_wsubs, (const TermW<A> *)h->d_wterms,                        \
              (const uint32_t *)h->d_wcut, h->depth, accumulate, (double *)h->d_split, count, stop)
        if (w == 16 && h->rows == 1) RP_WAVE(1, 16, false);
        else if (w == 16) RP_WAVE(4, 16, false);
        else if (w == 8 && h->rows == 1) RP_WAVE(1, 8, false);
        else if (w == 8) RP_WAVE(4, 8, false);
        else if (h->rows == 1) RP_WAVE(1, 4, false);
        else if (!big) RP_WAVE(4, 4, false);
        else RP_WAVE(4, 4, true);
#undef RP_WAVE
        return RP_OK;
    }
    switch (tiling_key(h->tile_bits, h->threads, h->depth)) {
    case tiling_key(8, 128, 2): return launch_tiled<R, A, 8, 128>(h, res, vec, accumulate, stop);
    case tiling_key(10, 128, 2): return launch_tiled<R, A, 10, 128>(h, res, vec, accumulate, stop);
    case tiling_key(12, 512, 2): return launch_tiled<R, A, 12, 512>(h, res, vec, accumulate, stop);
    case tiling_key(11, 256, 4):
        if constexpr (sizeof(R) == 8) return launch_tiled<R, A, 11, 256, 4>(h, res, vec, accumulate, stop);
        break;
    case tiling_key(12, 512, 3):
        if constexpr (sizeof(R) == 4) return launch_tiled<R, A, 12, 512, 3>(h, res, vec, accumulate, stop);
        break;
    case tiling_key(12, 512, 4):
        if constexpr (sizeof(R) == 4) return launch_tiled<R, A, 12, 512, 4>(h, res, vec, accumulate, stop);
        break;
    case tiling_key(12, 1024, 2):
        if constexpr (sizeof(R) == 4) return launch_tiled<R, A, 12, 1024>(h, res, vec, accumulate, stop);
        break;
    case tiling_key(13, 1024, 2):
        if constexpr (sizeof(R) == 4) return launch_tiled<R, A, 13, 1024>(h, res, vec, accumulate, stop);
        break;
    default: break;
    }
    return set_error(RP_ERR_RUNTIME, "rp_apply_ops: unsupported tiling b=%d threads=%d depth=%d",
                     h->tile_bits, h->threads, h->depth);
}

// rp_apply_gs's kernel: the tiled apply with the Gram-Schmidt dots in its
// epilogue, for the tilings it is instantiated for (complex<float> states,
// 2^12 tiles, 512 threads, 2 LDS tiles, FP64 or group accumulation) and at
// most max_rows workgroups; *rows = the partial rows written, 0 when the
// handle's layout has no such kernel (the caller then applies and sweeps
// separately)
int apply_dots_launch(rp_terms *h, void *res, const void *vec, const void *const *V, int k,
                      double *part, int width, uint64_t max_rows, uint64_t *rows)
{
    using T = float2;
    *rows = 0;
    if (h->prec != RP_C64 || !h->acc64 || h->nterms == 0 || h->tile_bits != 12 ||
        h->threads != 512 || h->depth != 2 || k < 0 || k > kMaxSweep)
        return RP_OK;
    const uint64_t grid = (1ull << h->len) >> 12;
    if (grid > max_rows) return RP_OK;
    VecPtrs64 P{};
    for (int q = 0; q < k; q++) P.p[q] = V[q];
    if (h->group_acc)
        RP_LAUNCH(RP_KERNEL_APPLY, (k_apply_tiled_gs<float, double, 12, 512, 2, true>),
                  dim3((unsigned)grid), dim3(512), 0, (const T *)vec, (T *)res,
                  (const GroupRuns *)h->d_groups, (int)h->ngroups, (const SubRec<double> *)h->d_subs,
                  (const TermRec<double> *)h->d_terms, P, k, part, width, h->tmap);
    else
        RP_LAUNCH(RP_KERNEL_APPLY, (k_apply_tiled_gs<float, double, 12, 512, 2, false>),
                  dim3((unsigned)grid), dim3(512), 0, (const T *)vec, (T *)res,
                  (const GroupRuns *)h->d_groups, (int)h->ngroups, (const SubRec<double> *)h->d_subs,
                  (const TermRec<double> *)h->d_terms, P, k, part, width, h->tmap);
    *rows = grid;
    return RP_OK;
}

}  // namespace rp

using namespace rp;

static int upload_any(rp_terms *h, const uint64_t *bits, const double *coeff, uint64_t n)
{
    if (h->prec == RP_C128) return upload_impl<double, double>(h, bits, coeff, n);
    if (h->acc64) return upload_impl<float, double>(h, bits, coeff, n);
    return upload_impl<float, float>(h, bits, coeff, n);
}

static void free_tables(rp_terms *h)
{
    for (void **p : {&h->d_groups, &h->d_subs, &h->d_terms, &h->d_cgroups, &h->d_csubs,
                     &h->d_cterms, &h->d_wflips, &h->d_wsubs, &h->d_wterms, &h->d_wcut, &h->d_split})
        if (*p) { (void)hipFree(*p); *p = nullptr; }
}

static int apply_dispatch(rp_terms *h, void *res, const void *vec, int accumulate,
                          const int *stop = nullptr)
{
    if (h->prec == RP_C128) return apply_impl<double, double>(h, res, vec, accumulate, stop);
    if (h->acc64) return apply_impl<float, double>(h, res, vec, accumulate, stop);
    return apply_impl<float, float>(h, res, vec, accumulate, stop);
}

namespace rp {
int apply_queued(rp_terms_t h, void *res, const void *vec, const int *stop)
{
    return apply_dispatch(h, res, vec, 0, stop);
}
}  // namespace rp

// rebuild the device tables for another tiling (from the stored term list)
static int retile(rp_terms *h, int tb, int nt, int d)
{
    free_tables(h);
    h->tile_bits = tb;
    h->threads = nt;
    h->depth = d;
    return upload_any(h, h->raw_bits.data(), h->raw_coeff.data(), h->raw_bits.size());
}

// Time every instantiated tiling that fits len on scratch vectors (3
// applies each after a warm-up) and keep the fastest.
static int autotune(rp_terms *h)
{
    Context &c = ctx();
    const size_t bytes = (size_t)elem_bytes(h->prec) << h->len;
    void *x = nullptr, *y = nullptr;
    if (dev_malloc(&x, bytes) != hipSuccess || dev_malloc(&y, bytes) != hipSuccess) {
        (void)hipGetLastError();
        if (x) (void)hipFree(x);
        return set_error(RP_ERR_OUT_OF_MEMORY, "rp_terms_upload_ex: no memory for autotuning");
    }
    int st = RP_OK;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    float best = 1e30f;
    TilingDesc pick{h->tile_bits, h->threads, h->depth, 0};
    if (hipMemsetAsync(x, 0, bytes, c.stream) != hipSuccess ||
        hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)
        st = set_error(RP_ERR_RUNTIME, "rp_terms_upload_ex: autotuning set-up failed");
    // Without tiles, 32 and 128 slices only up to 16 sites: beyond, they are
    // at least eight times the wavefronts the GPU holds, and their partial sums
    // (67 MB at 19 sites) cost the upload more than the rest of it.
    for (const TilingDesc &cd : kTilings) {
        if (st) break;
        if (cd.tb > h->len || !tiling_instantiated(h->prec, cd.tb, cd.nt, cd.depth)) continue;
        if (cd.tb == 0 && (!wave_allowed(h->len, h->nflips, cd.depth) ||
                           (cd.depth > 1 && h->nterms < (uint64_t)(2 * cd.depth))))
            continue;
        if ((st = retile(h, cd.tb, cd.nt, cd.depth))) break;
        if ((st = apply_dispatch(h, y, x, 0))) break;
        if (hipEventRecord(e0, c.stream) != hipSuccess) { st = RP_ERR_RUNTIME; break; }
        for (int r = 0; r < 3 && !st; r++) st = apply_dispatch(h, y, x, 0);
        float ms = 0;
        if (st || hipEventRecord(e1, c.stream) != hipSuccess ||
            hipEventSynchronize(e1) != hipSuccess || hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
            if (!st) st = set_error(RP_ERR_RUNTIME, "rp_terms_upload_ex: autotuning timing failed");
            break;
        }
        if (ms < best) { best = ms; pick = cd; }
    }
    // the kept tiling's apply against one streaming pass of the same vector
    // (3 scalings of x, each reading and writing it: 6 passes); a failure
    // here leaves the figure at 0 and the upload as it is
    if (!st && best < 1e30f) {
        float ms = 0;
        int sst = hipEventRecord(e0, c.stream) == hipSuccess ? RP_OK : RP_ERR_RUNTIME;
        for (int r = 0; r < 3 && !sst; r++)
            sst = rp_scale_vec(h->prec, x, 1.0, 0.0, 1ull << h->len);
        if (!sst && hipEventRecord(e1, c.stream) == hipSuccess &&
            hipEventSynchronize(e1) == hipSuccess && hipEventElapsedTime(&ms, e0, e1) == hipSuccess &&
            ms > 0)
            h->apply_passes = std::max(1.0, (double)best / 3.0 / ((double)ms / 6.0));
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipStreamSynchronize(c.stream);
    (void)hipFree(x);
    (void)hipFree(y);
    if (st) return st;
    if (pick.tb != h->tile_bits || pick.nt != h->threads || pick.depth != h->depth)
        st = retile(h, pick.tb, pick.nt, pick.depth);
    return st;
}

extern "C" {

int rp_terms_upload_ex(rp_terms_t *out, int prec, int len, const uint64_t *bits,
                       const double *coeff, uint64_t nterms, int flags)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(out, "null output handle");
    *out = nullptr;
    RP_REQUIRE(valid_prec(prec), "bad precision");
    RP_REQUIRE(len >= 1 && len <= 32, "len must be in [1, 32]");
    RP_REQUIRE(nterms == 0 || (bits && coeff), "null term arrays");
    RP_REQUIRE((flags & ~(RP_TERMS_ACC_NATIVE | RP_TERMS_AUTOTUNE | RP_TERMS_ACC_GROUP)) == 0,
               "unknown flags");
    RP_REQUIRE(!((flags & RP_TERMS_ACC_NATIVE) && (flags & RP_TERMS_ACC_GROUP)),
               "RP_TERMS_ACC_NATIVE and RP_TERMS_ACC_GROUP exclude each other");
    rp_terms *h = new rp_terms;
    h->prec = prec;
    h->len = len;
    h->acc64 = (prec == RP_C128 || !(flags & RP_TERMS_ACC_NATIVE)) ? 1 : 0;
    h->group_acc = (prec == RP_C64 && (flags & RP_TERMS_ACC_GROUP)) ? 1 : 0;
    choose_tiling(prec, len, list_shape(bits, nterms), h->group_acc, h->acc64, &h->tile_bits,
                  &h->threads, &h->depth);
    h->raw_bits.assign(bits, bits + nterms);
    h->raw_coeff.assign(coeff, coeff + 2 * nterms);
    st = upload_any(h, bits, coeff, nterms);
    if (!st && (flags & RP_TERMS_AUTOTUNE) && h->nterms && len <= 31)
        st = autotune(h);
    if (st) {
        free_handle(h);
        return st;
    }
    *out = h;
    return RP_OK;
}

int rp_terms_upload(rp_terms_t *out, int prec, int len, const uint64_t *bits,
                    const double *coeff, uint64_t nterms)
{
    return rp_terms_upload_ex(out, prec, len, bits, coeff, nterms, 0);
}

int rp_terms_free(rp_terms_t h)
{
    int st = check_init();
    if (st) return st;
    if (!h) return RP_OK;
    RP_CHECK_HIP(hipStreamSynchronize(ctx().stream));
    free_handle(h);
    return RP_OK;
}

int rp_terms_set_tiling(rp_terms_t h, int tile_bits, int threads, int depth)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(h, "null term handle");
    RP_REQUIRE(tile_bits <= h->len, "tile bits exceed the chain length");
    RP_REQUIRE(tile_bits != 0 || wave_allowed(h->len, h->nflips, depth),
               "tile bits 0 only up to len 16, and where an upload may choose it");
    RP_REQUIRE(tiling_instantiated(h->prec, tile_bits, threads, depth),
               "tiling not instantiated for this precision");
    RP_CHECK_HIP(hipStreamSynchronize(ctx().stream));
    return retile(h, tile_bits, threads, depth);
}

int rp_terms_info(rp_terms_t h, rp_terms_info_t *info)
{
    RP_REQUIRE(h && info, "null argument");
    info->prec = h->prec;
    info->len = h->len;
    info->tile_bits = h->tile_bits;
    info->threads = h->threads;
    info->depth = h->depth;
    info->nterms = h->nterms;
    info->nflips = h->nflips;
    info->ngroups = h->tile_bits ? h->ngroups : h->nflips;
    info->apply_passes = h->apply_passes;
    info->kernel = h->tile_bits == 0 ? RP_APPLY_SMALL
                   : (h->prec == RP_C64 && h->acc64 && h->group_acc && h->depth == 2 && h->d_csubs)
                       ? RP_APPLY_STREAM
                       : RP_APPLY_TILED;
    info->bytes_per_apply = (info->ngroups + 1) * (1ull << h->len) * elem_bytes(h->prec);
    info->tile_map = h->tmap.n;
    return RP_OK;
}

int rp_apply_ops(rp_terms_t h, void *res, const void *vec, int accumulate)
{
    int st = check_init();
    if (st) return st;
    RP_REQUIRE(h, "null term handle");
    RP_REQUIRE(res && vec, "null vector");
    RP_REQUIRE(res != vec, "res and vec must be different buffers");
    return apply_dispatch(h, res, vec, accumulate);
}

}  // extern "C"
