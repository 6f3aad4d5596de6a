// expm.h -- small dense complex matrices on the host in FP64 and their
// exponential, for the Krylov driver's Hessenberg matrix.
//
// The reference evaluates exp((-beta - i t) Hfull) with Eigen's
// MatrixFunctions in the run's FpType (inc/algo.h:331-332).  This build keeps
// the small matrices in FP64 for both state precisions and uses the scaling
// and squaring Pade method of N. J. Higham, SIAM J. Matrix Anal. Appl. 26
// (2005) 1179-1193: Pade degree m in {3,5,7,9,13} chosen from the 1-norm
// against Higham's theta_m bounds for double precision, 2^-s scaling so that
// ||A||_1 <= theta_13, and s squarings.
#pragma once

#ifndef _REAPERS_H_
#error "Do not include this file directly. Include the master header file reapers.h"
#endif

namespace dense {

using cd = std::complex<double>;

// column-major n x n complex matrix
struct CMat {
    int n = 0;
    std::vector<cd> a;
    CMat() = default;
    explicit CMat(int n_) : n(n_), a((size_t)n_ * n_) {}
    cd &operator()(int i, int j) { return a[(size_t)j * n + i]; }
    const cd &operator()(int i, int j) const { return a[(size_t)j * n + i]; }
    static CMat identity(int n) {
        CMat m(n);
        for (int i = 0; i < n; i++) m(i, i) = 1.0;
        return m;
    }
    // resize keeping the top-left block, new entries zero
    void grow(int nn) {
        CMat m(nn);
        for (int j = 0; j < std::min(n, nn); j++)
            for (int i = 0; i < std::min(n, nn); i++) m(i, j) = (*this)(i, j);
        *this = std::move(m);
    }
};

inline CMat matmul(const CMat &A, const CMat &B)
{
    const int n = A.n;
    CMat C(n);
    for (int j = 0; j < n; j++)
        for (int k = 0; k < n; k++) {
            const cd b = B(k, j);
            if (b == cd(0)) continue;
            const cd *ak = &A.a[(size_t)k * n];
            cd *cj = &C.a[(size_t)j * n];
            for (int i = 0; i < n; i++) cj[i] += ak[i] * b;
        }
    return C;
}

inline double norm1(const CMat &A)
{
    double best = 0;
    for (int j = 0; j < A.n; j++) {
        double s = 0;
        for (int i = 0; i < A.n; i++) s += std::abs(A(i, j));
        best = std::max(best, s);
    }
    return best;
}

// solve D X = B with partial pivoting; B is overwritten by X
inline void lu_solve(CMat D, CMat &B)
{
    const int n = D.n;
    for (int k = 0; k < n; k++) {
        int p = k;
        double best = -1;
        for (int i = k; i < n; i++) {
            double v = std::abs(D(i, k));
            if (v > best) { best = v; p = i; }
        }
        if (p != k)
            for (int j = 0; j < n; j++) {
                std::swap(D(k, j), D(p, j));
                std::swap(B(k, j), B(p, j));
            }
        const cd inv = 1.0 / D(k, k);
        for (int i = k + 1; i < n; i++) {
            const cd l = D(i, k) * inv;
            if (l == cd(0)) continue;
            for (int j = k + 1; j < n; j++) D(i, j) -= l * D(k, j);
            for (int j = 0; j < n; j++) B(i, j) -= l * B(k, j);
        }
    }
    for (int j = 0; j < n; j++)
        for (int i = n - 1; i >= 0; i--) {
            cd s = B(i, j);
            for (int k = i + 1; k < n; k++) s -= D(i, k) * B(k, j);
            B(i, j) = s / D(i, i);
        }
}

// sum_k w[k] M[k] + w0 I
inline CMat combo(const std::vector<const CMat *> &M, const std::vector<double> &w, double w0, int n)
{
    CMat R(n);
    for (size_t k = 0; k < M.size(); k++)
        for (size_t q = 0; q < R.a.size(); q++) R.a[q] += w[k] * M[k]->a[q];
    for (int i = 0; i < n; i++) R(i, i) += w0;
    return R;
}

inline CMat expm(const CMat &A0)
{
    const int n = A0.n;
    if (n == 0) return CMat();
    static const double theta[] = {1.495585217958292e-2, 2.539398330063230e-1,
                                   9.504178996162932e-1, 2.097847961257068e0,
                                   5.371920351148152e0};
    double nrm = norm1(A0);
    CMat A = A0;
    int s = 0, deg;
    if (nrm <= theta[0]) deg = 3;
    else if (nrm <= theta[1]) deg = 5;
    else if (nrm <= theta[2]) deg = 7;
    else if (nrm <= theta[3]) deg = 9;
    else {
        deg = 13;
        s = std::max(0, (int)std::ceil(std::log2(nrm / theta[4])));
        const double sc = std::ldexp(1.0, -s);
        for (auto &v : A.a) v *= sc;
    }
    CMat U, V;
    CMat A2 = matmul(A, A);
    if (deg == 3) {
        U = matmul(A, combo({&A2}, {1.}, 60., n));
        V = combo({&A2}, {12.}, 120., n);
    } else if (deg == 5) {
        CMat A4 = matmul(A2, A2);
        U = matmul(A, combo({&A4, &A2}, {1., 420.}, 15120., n));
        V = combo({&A4, &A2}, {30., 3360.}, 30240., n);
    } else if (deg == 7) {
        CMat A4 = matmul(A2, A2), A6 = matmul(A4, A2);
        U = matmul(A, combo({&A6, &A4, &A2}, {1., 1512., 277200.}, 8648640., n));
        V = combo({&A6, &A4, &A2}, {56., 25200., 1995840.}, 17297280., n);
    } else if (deg == 9) {
        CMat A4 = matmul(A2, A2), A6 = matmul(A4, A2), A8 = matmul(A6, A2);
        U = matmul(A, combo({&A8, &A6, &A4, &A2}, {1., 3960., 2162160., 302702400.},
                            8821612800., n));
        V = combo({&A8, &A6, &A4, &A2}, {90., 110880., 30270240., 2075673600.}, 17643225600., n);
    } else {
        const double b[] = {64764752532480000., 32382376266240000., 7771770303897600.,
                            1187353796428800., 129060195264000., 10559470521600.,
                            670442572800., 33522128640., 1323241920., 40840800.,
                            960960., 16380., 182., 1.};
        CMat A4 = matmul(A2, A2), A6 = matmul(A4, A2);
        CMat Ui = matmul(A6, combo({&A6, &A4, &A2}, {b[13], b[11], b[9]}, 0., n));
        CMat Ul = combo({&A6, &A4, &A2}, {b[7], b[5], b[3]}, b[1], n);
        for (size_t q = 0; q < Ui.a.size(); q++) Ui.a[q] += Ul.a[q];
        U = matmul(A, Ui);
        V = matmul(A6, combo({&A6, &A4, &A2}, {b[12], b[10], b[8]}, 0., n));
        CMat Vl = combo({&A6, &A4, &A2}, {b[6], b[4], b[2]}, b[0], n);
        for (size_t q = 0; q < V.a.size(); q++) V.a[q] += Vl.a[q];
    }
    CMat P(n), Q(n);
    for (size_t q = 0; q < P.a.size(); q++) {
        P.a[q] = V.a[q] + U.a[q];
        Q.a[q] = V.a[q] - U.a[q];
    }
    lu_solve(Q, P);
    for (int k = 0; k < s; k++) P = matmul(P, P);
    return P;
}

// ---------------------------------------------------------------------------
// The first column of exp(A).  The Krylov drivers need only that column, and
// their A, the Hessenberg blocks of all restarts so far, has one diagonal
// below the main one.  Products of matrices with few lower diagonals are
// nearly triangular (a sixth of the work), so are the numerator and the
// denominator of the Pade approximant r, and exp(A) e_1 = r(A / 2^s)^(2^s) e_1
// is 2^s triangular products and solves with one factorization instead of a
// full solve and s squarings.  On one core: 60 x 60 with ||A||_1 = 30, 4.8 ms
// by expm() above, 0.3 ms here.
// ---------------------------------------------------------------------------
// column-major n x n, real and imaginary parts apart, rows padded to whole
// vectors of four; entries more than `low` below the diagonal are zero
struct BandMat {
    int n = 0, ld = 0, low = 0;
    std::vector<double> re, im;
    BandMat(int n_, int low_)
        : n(n_), ld((n_ + 3) / 4 * 4), low(std::min(low_, std::max(0, n_ - 1))),
          re((size_t)ld * n_), im((size_t)ld * n_) {}
    // rows of column j that may be nonzero
    int rows(int j) const { return std::min(n, j + low + 1); }
};

typedef double vec4 __attribute__((vector_size(32), aligned(8), may_alias));

// one version with 256-bit vectors beside the baseline one, chosen at load
// time (no fused multiply-adds in either: the same bits)
#if defined(__GNUC__) && !defined(__clang__) && defined(__x86_64__) && !defined(__AVX2__)
#define REAPERS_VEC_CLONES __attribute__((target_clones("avx2", "default")))
#else
#define REAPERS_VEC_CLONES
#endif

// y += A[:, k0..k1) b over the rows those columns reach (whole vectors: the
// rows past a column's band are zero), four columns at a time
REAPERS_VEC_CLONES
static void band_gemv(const BandMat &A, int k0, int k1, const double *br, const double *bi,
                      double *yr, double *yi)
{
    const size_t ld = A.ld;
    for (int k = k0; k < k1; k += 4) {
        const int c = std::min(4, k1 - k), m = A.rows(k + c - 1);
        const double *ar = &A.re[k * ld], *ai = &A.im[k * ld];
        if (c == 4) {
            const double r0 = br[k], r1 = br[k + 1], r2 = br[k + 2], r3 = br[k + 3];
            const double i0 = bi[k], i1 = bi[k + 1], i2 = bi[k + 2], i3 = bi[k + 3];
            for (int i = 0; i < m; i += 4) {
                vec4 sr = *(vec4 *)(yr + i), si = *(vec4 *)(yi + i);
                vec4 xr = *(const vec4 *)(ar + i), xi = *(const vec4 *)(ai + i);
                sr += xr * r0 - xi * i0;
                si += xr * i0 + xi * r0;
                xr = *(const vec4 *)(ar + ld + i), xi = *(const vec4 *)(ai + ld + i);
                sr += xr * r1 - xi * i1;
                si += xr * i1 + xi * r1;
                xr = *(const vec4 *)(ar + 2 * ld + i), xi = *(const vec4 *)(ai + 2 * ld + i);
                sr += xr * r2 - xi * i2;
                si += xr * i2 + xi * r2;
                xr = *(const vec4 *)(ar + 3 * ld + i), xi = *(const vec4 *)(ai + 3 * ld + i);
                sr += xr * r3 - xi * i3;
                si += xr * i3 + xi * r3;
                *(vec4 *)(yr + i) = sr;
                *(vec4 *)(yi + i) = si;
            }
        } else {
            for (int q = 0; q < c; q++)
                for (int i = 0; i < m; i += 4) {
                    const vec4 xr = *(const vec4 *)(ar + q * ld + i);
                    const vec4 xi = *(const vec4 *)(ai + q * ld + i);
                    *(vec4 *)(yr + i) += xr * br[k + q] - xi * bi[k + q];
                    *(vec4 *)(yi + i) += xr * bi[k + q] + xi * br[k + q];
                }
        }
    }
}

inline BandMat band_mul(const BandMat &A, const BandMat &B)
{
    const int n = A.n;
    BandMat C(n, A.low + B.low);
    for (int j = 0; j < n; j++) {
        const size_t b = (size_t)j * B.ld, c = (size_t)j * C.ld;
        band_gemv(A, 0, B.rows(j), &B.re[b], &B.im[b], &C.re[c], &C.im[c]);
    }
    return C;
}

// sum_k w[k] M[k] + w0 I
inline BandMat band_combo(std::initializer_list<const BandMat *> M, std::initializer_list<double> w,
                          double w0)
{
    const BandMat &F = **M.begin();
    int low = 0;
    for (auto *m : M) low = std::max(low, m->low);
    BandMat R(F.n, low);
    auto f = w.begin();
    for (auto *m : M) {
        for (size_t q = 0; q < R.re.size(); q++) {
            R.re[q] += *f * m->re[q];
            R.im[q] += *f * m->im[q];
        }
        ++f;
    }
    for (int i = 0; i < F.n; i++) R.re[(size_t)i * R.ld + i] += w0;
    return R;
}

inline void band_add(BandMat &A, const BandMat &B, double f)
{
    A.low = std::max(A.low, B.low);
    for (size_t q = 0; q < A.re.size(); q++) {
        A.re[q] += f * B.re[q];
        A.im[q] += f * B.im[q];
    }
}

inline std::vector<cd> expm_col0(const CMat &A0)
{
    const int n = A0.n;
    if (n == 0) return {};
    static const double theta[] = {1.495585217958292e-2, 2.539398330063230e-1,
                                   9.504178996162932e-1, 2.097847961257068e0,
                                   5.371920351148152e0};
    const double nrm = norm1(A0);
    const int deg = nrm <= theta[0] ? 3 : nrm <= theta[1] ? 5 : nrm <= theta[2] ? 7
                    : nrm <= theta[3] ? 9 : 13;
    int s = 0;
    if (deg == 13) s = std::max(0, (int)std::ceil(std::log2(nrm / theta[4])));
    int low = 0;
    for (int j = 0; j < n; j++)
        for (int i = n - 1; i > j + low; i--)
            if (A0(i, j) != cd(0)) low = i - j;
    // not finite, or so many applications of r that squaring is less work
    if (!std::isfinite(nrm) || s > 30 || std::ldexp(1.0, s) > (double)(s + 1) * n) {
        const CMat E = expm(A0);
        return std::vector<cd>(E.a.begin(), E.a.begin() + n);
    }
    BandMat A(n, low);
    const double sc = std::ldexp(1.0, -s);
    for (int j = 0; j < n; j++)
        for (int i = 0; i < A.rows(j); i++) {
            A.re[(size_t)j * A.ld + i] = A0(i, j).real() * sc;
            A.im[(size_t)j * A.ld + i] = A0(i, j).imag() * sc;
        }
    // numerator V + U and denominator V - U of the diagonal Pade approximant
    // (coefficients as in expm)
    const BandMat A2 = band_mul(A, A);
    BandMat U(n, 0), V(n, 0);
    if (deg == 3) {
        U = band_mul(A, band_combo({&A2}, {1.}, 60.));
        V = band_combo({&A2}, {12.}, 120.);
    } else if (deg == 5) {
        const BandMat A4 = band_mul(A2, A2);
        U = band_mul(A, band_combo({&A4, &A2}, {1., 420.}, 15120.));
        V = band_combo({&A4, &A2}, {30., 3360.}, 30240.);
    } else if (deg == 7) {
        const BandMat A4 = band_mul(A2, A2), A6 = band_mul(A4, A2);
        U = band_mul(A, band_combo({&A6, &A4, &A2}, {1., 1512., 277200.}, 8648640.));
        V = band_combo({&A6, &A4, &A2}, {56., 25200., 1995840.}, 17297280.);
    } else if (deg == 9) {
        const BandMat A4 = band_mul(A2, A2), A6 = band_mul(A4, A2), A8 = band_mul(A6, A2);
        U = band_mul(A, band_combo({&A8, &A6, &A4, &A2}, {1., 3960., 2162160., 302702400.},
                                   8821612800.));
        V = band_combo({&A8, &A6, &A4, &A2}, {90., 110880., 30270240., 2075673600.}, 17643225600.);
    } else {
        const double b[] = {64764752532480000., 32382376266240000., 7771770303897600.,
                            1187353796428800., 129060195264000., 10559470521600.,
                            670442572800., 33522128640., 1323241920., 40840800.,
                            960960., 16380., 182., 1.};
        const BandMat A4 = band_mul(A2, A2), A6 = band_mul(A4, A2);
        BandMat Ui = band_mul(A6, band_combo({&A6, &A4, &A2}, {b[13], b[11], b[9]}, 0.));
        band_add(Ui, band_combo({&A6, &A4, &A2}, {b[7], b[5], b[3]}, b[1]), 1.0);
        U = band_mul(A, Ui);
        V = band_mul(A6, band_combo({&A6, &A4, &A2}, {b[12], b[10], b[8]}, 0.));
        band_add(V, band_combo({&A6, &A4, &A2}, {b[6], b[4], b[2]}, b[0]), 1.0);
    }
    BandMat P = V, Q = std::move(V);
    band_add(P, U, 1.0);
    band_add(Q, U, -1.0);
    // Q = L U with partial pivoting; a column has at most Q.low multipliers
    const int ql = Q.low;
    std::vector<int> piv(n);
    std::vector<cd> dinv(n), mult((size_t)n * std::max(1, ql));
    auto at = [&](int i, int j) { return (size_t)j * Q.ld + i; };
    for (int k = 0; k < n; k++) {
        const int end = std::min(n, k + ql + 1);
        int best = k;
        double mag = -1;
        for (int i = k; i < end; i++) {
            const double v = std::hypot(Q.re[at(i, k)], Q.im[at(i, k)]);
            if (v > mag) { mag = v; best = i; }
        }
        piv[k] = best;
        if (best != k)
            for (int j = k; j < n; j++) {
                std::swap(Q.re[at(k, j)], Q.re[at(best, j)]);
                std::swap(Q.im[at(k, j)], Q.im[at(best, j)]);
            }
        dinv[k] = 1.0 / cd(Q.re[at(k, k)], Q.im[at(k, k)]);
        cd *l = &mult[(size_t)k * std::max(1, ql)];
        for (int i = k + 1; i < end; i++) l[i - k - 1] = cd(Q.re[at(i, k)], Q.im[at(i, k)]) * dinv[k];
        for (int j = k + 1; j < n; j++) {
            const double br = Q.re[at(k, j)], bi = Q.im[at(k, j)];
            for (int i = k + 1; i < end; i++) {
                const double lr = l[i - k - 1].real(), li = l[i - k - 1].imag();
                Q.re[at(i, j)] -= lr * br - li * bi;
                Q.im[at(i, j)] -= lr * bi + li * br;
            }
        }
    }
    std::vector<double> xr(Q.ld), xi(Q.ld), yr(Q.ld), yi(Q.ld);
    xr[0] = 1.0;
    int top = 1;                              // rows of x from `top` on are zero
    for (long q = 0; q < 1L << s; q++) {
        std::fill(yr.begin(), yr.end(), 0.0);
        std::fill(yi.begin(), yi.end(), 0.0);
        band_gemv(P, 0, top, xr.data(), xi.data(), yr.data(), yi.data());
        for (int k = 0; k < n; k++) {
            std::swap(yr[k], yr[piv[k]]);
            std::swap(yi[k], yi[piv[k]]);
            const cd *l = &mult[(size_t)k * std::max(1, ql)];
            const int end = std::min(n, k + ql + 1);
            for (int i = k + 1; i < end; i++) {
                const double lr = l[i - k - 1].real(), li = l[i - k - 1].imag();
                yr[i] -= lr * yr[k] - li * yi[k];
                yi[i] -= lr * yi[k] + li * yr[k];
            }
        }
        for (int j = n - 1; j >= 0; j--) {
            const double dr = dinv[j].real(), di = dinv[j].imag();
            const double vr = yr[j] * dr - yi[j] * di, vi = yr[j] * di + yi[j] * dr;
            for (int i = 0; i < j; i++) {
                yr[i] -= Q.re[at(i, j)] * vr - Q.im[at(i, j)] * vi;
                yi[i] -= Q.re[at(i, j)] * vi + Q.im[at(i, j)] * vr;
            }
            xr[j] = vr;
            xi[j] = vi;
        }
        top = n;
    }
    std::vector<cd> out(n);
    for (int i = 0; i < n; i++) out[i] = cd(xr[i], xi[i]);
    return out;
}

// eigen-decomposition of the symmetric tridiagonal matrix with diagonal a
// and off-diagonal b, by cyclic Jacobi rotations (the Lanczos matrices are
// small); eigenvector k is column k of Q (column-major)
inline void tridiag_eigen(const std::vector<double> &a, const std::vector<double> &b,
                          std::vector<double> &w, std::vector<double> &Q)
{
    const int n = (int)a.size();
    std::vector<double> A((size_t)n * n, 0.0);
    for (int i = 0; i < n; i++) A[(size_t)i * n + i] = a[i];
    for (int i = 0; i + 1 < n; i++) {
        A[(size_t)i * n + i + 1] = b[i];
        A[(size_t)(i + 1) * n + i] = b[i];
    }
    Q.assign((size_t)n * n, 0.0);
    for (int i = 0; i < n; i++) Q[(size_t)i * n + i] = 1.0;
    auto at = [&](int i, int j) -> double & { return A[(size_t)j * n + i]; };
    for (int sweep = 0; sweep < 100; sweep++) {
        double off = 0;
        for (int p = 0; p < n; p++)
            for (int q = p + 1; q < n; q++) off += at(p, q) * at(p, q);
        if (off < 1e-300) break;
        for (int p = 0; p < n; p++)
            for (int q = p + 1; q < n; q++) {
                double apq = at(p, q);
                if (apq == 0) continue;
                double th = (at(q, q) - at(p, p)) / (2 * apq);
                double t = (th >= 0 ? 1.0 : -1.0) / (std::abs(th) + std::sqrt(th * th + 1));
                double c = 1 / std::sqrt(t * t + 1), s = t * c;
                for (int k = 0; k < n; k++) {
                    double akp = at(k, p), akq = at(k, q);
                    at(k, p) = c * akp - s * akq;
                    at(k, q) = s * akp + c * akq;
                }
                for (int k = 0; k < n; k++) {
                    double apk = at(p, k), aqk = at(q, k);
                    at(p, k) = c * apk - s * aqk;
                    at(q, k) = s * apk + c * aqk;
                }
                for (int k = 0; k < n; k++) {
                    double qkp = Q[(size_t)p * n + k], qkq = Q[(size_t)q * n + k];
                    Q[(size_t)p * n + k] = c * qkp - s * qkq;
                    Q[(size_t)q * n + k] = s * qkp + c * qkq;
                }
            }
    }
    w.resize(n);
    for (int i = 0; i < n; i++) w[i] = at(i, i);
}

}  // namespace dense
