// Compares expm_col0 with the first column of expm on Hessenberg, full and
// special matrices; prints the largest relative difference of each kind.
#define _REAPERS_H_
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdio>
#include <limits>
#include <random>
#include <vector>
#include "expm.h"

using namespace dense;

static std::mt19937_64 rng(7);
static double gauss() { static std::normal_distribution<double> d; return d(rng); }

static CMat make(int n, int low, double nrm, bool skew)
{
    CMat A(n);
    for (int j = 0; j < n; j++)
        for (int i = 0; i < std::min(n, j + low + 1); i++)
            if (skew) {     // -i times a Hermitian tridiagonal matrix: a Krylov block
                if (i == j) A(i, j) = cd(0, gauss());
                else if (i == j + 1) A(i, j) = cd(0, -std::abs(gauss()));
            } else {
                A(i, j) = cd(gauss(), gauss());
            }
    if (skew)
        for (int j = 1; j < n; j++) A(j - 1, j) = A(j, j - 1);
    const double f = nrm / std::max(norm1(A), 1e-300);
    for (auto &v : A.a) v *= f;
    return A;
}

static double diff(const CMat &A)
{
    const CMat E = expm(A);
    const auto c = expm_col0(A);
    double d = 0, s = 0;
    for (int i = 0; i < A.n; i++) {
        d += std::norm(c[i] - E(i, 0));
        s += std::norm(E(i, 0));
    }
    return std::sqrt(d / s);
}

int main()
{
    for (double nrm : {1e-3, 0.1, 0.7, 2.0, 5.0, 30.0, 200.0, 3000.0}) {
        double skew = 0, hess = 0, full = 0;
        for (int n : {1, 2, 3, 5, 12, 13, 14, 15, 20, 33, 60}) {
            skew = std::max(skew, diff(make(n, 1, nrm, true)));
            if (nrm <= 30) {
                hess = std::max(hess, diff(make(n, 1, nrm, false)));
                full = std::max(full, diff(make(n, n, nrm, false)));
            }
        }
        std::printf("norm %g skew %.3e hess %.3e full %.3e\n", nrm, skew, hess, full);
    }
    CMat Z(5);
    std::printf("zero %.3e\n", std::abs(expm_col0(Z)[0] - 1.0) + std::abs(expm_col0(Z)[4]));
    CMat N(4);                                       // nilpotent: exp = sum of 4 terms
    for (int i = 0; i < 3; i++) N(i + 1, i) = 1.0;
    std::printf("nilpotent %.3e\n", std::abs(expm_col0(N)[3] - 1.0 / 6));
    CMat B(3);
    B(1, 1) = std::numeric_limits<double>::quiet_NaN();
    std::printf("empty %d nan %d\n", (int)expm_col0(CMat()).size(), (int)std::isnan(std::abs(expm_col0(B)[1])));
    return 0;
}
