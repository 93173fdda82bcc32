// Small symmetric eigenproblems on the host (the Davidson driver's subspace matrices and the P space
// of its guess).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <numeric>
#include <vector>

namespace hipotf {

// Eigen-decomposition of a symmetric m x m matrix (row-major a), ascending eigenvalues,
// eigenvectors in the columns of v (row-major): Householder reduction to tridiagonal form, implicit
// QR steps with Wilkinson's shift (Golub and Van Loan, Matrix Computations, 8.3), reflectors applied
// to the eigenvectors.  The eigenvectors are kept as rows while they are rotated, so every inner
// loop runs over contiguous values.  (Cyclic Jacobi took 0.73 s for the 256 x 256 P space of a solve
// and 1.3 ms per iteration at 64 x 64: 1.1 s of a 12-orbital ground state.)  The matrix, and each
// column before it is squared, is scaled by a power of two (exact), so that entries of any size
// neither vanish nor overflow there.  False if the matrix holds infinities or NaN, or the QR steps do not converge.
inline bool sym_eigh(int m, std::vector<double> a, std::vector<double> &w, std::vector<double> &v) {
    double amax = 0.0;
    for (double x : a) {
        if (!std::isfinite(x)) return false;
        amax = std::max(amax, std::fabs(x));
    }
    const int ea = amax > 0.0 ? std::ilogb(amax) : 0;
    for (double &x : a) x = std::ldexp(x, -ea);
    std::vector<double> d(m), e(m, 0.0), p(m), refl, beta(m, 0.0);
    refl.assign((size_t)m * m, 0.0);  // reflector k in row k, entries k + 1 ..
    for (int k = 0; k + 2 < m; ++k) {
        // reflect column k below the diagonal onto its first entry
        double *x = &refl[(size_t)k * m];
        double top = 0.0, nrm = 0.0, tail = 0.0;
        for (int i = k + 1; i < m; ++i) top = std::max(top, std::fabs(a[(size_t)i * m + k]));
        if (top == 0.0) continue;
        const int ex = std::ilogb(top);
        for (int i = k + 1; i < m; ++i) {
            x[i] = std::ldexp(a[(size_t)i * m + k], -ex);
            nrm += x[i] * x[i];
            if (i > k + 1) tail += x[i] * x[i];
        }
        if (tail == 0.0) continue;  // already tridiagonal here
        const double alpha = x[k + 1] > 0.0 ? -std::sqrt(nrm) : std::sqrt(nrm);
        x[k + 1] -= alpha;
        const double bt = 2.0 / (tail + x[k + 1] * x[k + 1]);
        beta[k] = bt;
        // trailing block: A - x y^T - y x^T with y = bt A x - (bt / 2) (x . bt A x) x
        double xp = 0.0;
        for (int i = k + 1; i < m; ++i) {
            const double *r = &a[(size_t)i * m];
            double t = 0.0;
            for (int j = k + 1; j < m; ++j) t += r[j] * x[j];
            p[i] = bt * t;
            xp += p[i] * x[i];
        }
        for (int i = k + 1; i < m; ++i) p[i] -= 0.5 * bt * xp * x[i];
        for (int i = k + 1; i < m; ++i) {
            double *r = &a[(size_t)i * m];
            const double xi = x[i], yi = p[i];
            for (int j = k + 1; j < m; ++j) r[j] -= xi * p[j] + yi * x[j];
        }
        a[(size_t)(k + 1) * m + k] = std::ldexp(alpha, ex);
    }
    for (int i = 0; i < m; ++i) {
        d[i] = a[(size_t)i * m + i];
        if (i + 1 < m) e[i] = a[(size_t)(i + 1) * m + i];
    }
    std::vector<double> z((size_t)m * m, 0.0);  // row i: eigenvector i of the tridiagonal matrix
    for (int i = 0; i < m; ++i) z[(size_t)i * m + i] = 1.0;
    const double eps = 2.220446049250313e-16, least = eps * eps;  // (the largest entry is in [1, 2))
    auto negligible = [&](int i) {
        return std::fabs(e[i]) <= std::max(eps * (std::fabs(d[i]) + std::fabs(d[i + 1])), least);
    };
    int hi = m - 1;
    for (int it = 0; hi > 0 && it < 60 * m; ++it) {
        if (negligible(hi - 1)) {
            e[hi - 1] = 0.0;
            --hi;
            continue;
        }
        int lo = hi - 1;  // the unreduced block that ends at hi
        while (lo > 0 && !negligible(lo - 1)) --lo;
        const double g = 0.5 * (d[hi - 1] - d[hi]), t = e[hi - 1];
        const double mu = d[hi] - t * (t / (g + (g >= 0.0 ? 1.0 : -1.0) * std::hypot(g, t)));
        double x = d[lo] - mu, bulge = e[lo];
        for (int k = lo; k < hi; ++k) {
            const double r = std::hypot(x, bulge);
            const double c = r > 0.0 ? x / r : 1.0, s = r > 0.0 ? bulge / r : 0.0;
            if (k > lo) e[k - 1] = r;
            const double dk = d[k], ek = e[k], dn = d[k + 1];
            d[k] = c * c * dk + 2.0 * c * s * ek + s * s * dn;
            d[k + 1] = s * s * dk - 2.0 * c * s * ek + c * c * dn;
            e[k] = (c * c - s * s) * ek + c * s * (dn - dk);
            if (k + 1 < hi) {
                bulge = s * e[k + 1];
                e[k + 1] *= c;
            }
            x = e[k];
            double *zk = &z[(size_t)k * m], *zn = zk + m;
            for (int j = 0; j < m; ++j) {
                const double u = zk[j], q = zn[j];
                zk[j] = c * u + s * q;
                zn[j] = c * q - s * u;
            }
        }
    }
    if (hi > 0) return false;
    std::vector<int> order(m);
    std::iota(order.begin(), order.end(), 0);
    std::sort(order.begin(), order.end(), [&](int i, int j) { return d[i] < d[j]; });
    w.resize(m);
    v.assign((size_t)m * m, 0.0);
    for (int c = 0; c < m; ++c) {
        double *y = &z[(size_t)order[c] * m];
        for (int k = m - 3; k >= 0; --k) {
            if (beta[k] == 0.0) continue;
            const double *x = &refl[(size_t)k * m];
            double t = 0.0;
            for (int i = k + 1; i < m; ++i) t += x[i] * y[i];
            t *= beta[k];
            for (int i = k + 1; i < m; ++i) y[i] -= t * x[i];
        }
        w[c] = std::ldexp(d[order[c]], ea);
        for (int r = 0; r < m; ++r) v[(size_t)r * m + c] = y[r];
    }
    return true;
}

}  // namespace hipotf
