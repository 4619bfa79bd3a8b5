// Host-side symmetric tridiagonal eigensolver of the duct's z-wall operator
// (plain C++, no HIP: also compiled on its own by the CPU tests).
#pragma once

#include <algorithm>
#include <cmath>
#include <limits>
#include <vector>

namespace dfp {

// Eigenvalues and orthonormal eigenvectors of the symmetric tridiagonal
// matrix with diagonal d[0..n) and off-diagonal e[i] (coupling rows i and
// i+1) by implicit QL sweeps with Wilkinson shifts (Golub & Van Loan,
// Matrix Computations sec. 8.3, in the QL orientation of EISPACK's tql2):
// on return d holds the eigenvalues in ascending order and column m of v
// (n x n, column-major) the eigenvector of d[m].  false if an eigenvalue
// takes more than 60 sweeps.
inline bool symtri_eigen(int n, std::vector<double>& d, std::vector<double> e, std::vector<double>& v) {
    v.assign((size_t)n * n, 0.0);
    for (int i = 0; i < n; ++i) v[(size_t)i * n + i] = 1.0;
    e.resize(n, 0.0);
    e[n - 1] = 0.0;
    const double eps = std::numeric_limits<double>::epsilon();
    for (int l = 0; l < n; ++l) {
        for (int sweep = 0;; ++sweep) {
            // the first negligible off-diagonal at or below row l closes the block
            int m = l;
            while (m < n - 1 && std::fabs(e[m]) > eps * (std::fabs(d[m]) + std::fabs(d[m + 1]))) ++m;
            if (m == l) break;
            if (sweep == 60) return false;
            // shift: the eigenvalue of the leading 2x2 block nearer d[l]
            double g = (d[l + 1] - d[l]) / (2.0 * e[l]);
            double r = std::hypot(g, 1.0);
            g = d[m] - d[l] + e[l] / (g + std::copysign(r, g));
            double s = 1.0, c = 1.0, p = 0.0;
            bool split = false;
            // chase the bulge from the bottom of the block up to row l
            for (int i = m - 1; i >= l; --i) {
                const double f = s * e[i], b = c * e[i];
                r = std::hypot(f, g);
                e[i + 1] = r;
                if (r == 0.0) {  // the block splits: restart on the smaller one
                    d[i + 1] -= p;
                    e[m] = 0.0;
                    split = true;
                    break;
                }
                s = f / r;
                c = g / r;
                g = d[i + 1] - p;
                r = (d[i] - g) * s + 2.0 * c * b;
                p = s * r;
                d[i + 1] = g + p;
                g = c * r - b;
                double* vi = v.data() + (size_t)i * n;
                double* vj = v.data() + (size_t)(i + 1) * n;
                for (int k = 0; k < n; ++k) {
                    const double a1 = vi[k], a2 = vj[k];
                    vj[k] = s * a1 + c * a2;
                    vi[k] = c * a1 - s * a2;
                }
            }
            if (split) continue;
            d[l] -= p;
            e[l] = g;
            e[m] = 0.0;
        }
    }
    // ascending order, eigenvectors along
    for (int i = 0; i < n - 1; ++i) {
        int k = i;
        for (int j = i + 1; j < n; ++j)
            if (d[j] < d[k]) k = j;
        if (k != i) {
            std::swap(d[i], d[k]);
            for (int q = 0; q < n; ++q) std::swap(v[(size_t)i * n + q], v[(size_t)k * n + q]);
        }
    }
    return true;
}

// One step of inverse iteration in long double on the eigenpair (lam, x) of the
// symmetric tridiagonal matrix d, e (n rows; x normalised, already accurate to
// double): lam is its Rayleigh quotient, x the normalised solution y of
// (T - lam I) y = x (tridiagonal elimination with row interchanges), lam the
// Rayleigh quotient of that.
inline void symtri_refine(int n, const long double* d, const long double* e, long double& lam, std::vector<long double>& x) {
    using T = long double;
    if (n == 1) {
        lam = d[0];
        return;
    }
    auto rayleigh = [&]() {
        T s = 0, q = 0;
        for (int i = 0; i < n; ++i) {
            s += d[i] * x[i] * x[i] + (i + 1 < n ? T(2) * e[i] * x[i] * x[i + 1] : T(0));
            q += x[i] * x[i];
        }
        return s / q;
    };
    lam = rayleigh();
    std::vector<T> a(n), u(n, T(0)), w(n, T(0)), y = x;  // diagonal, first and second superdiagonal
    T big = 0;
    for (int i = 0; i < n; ++i) {
        a[i] = d[i] - lam;
        if (i + 1 < n) u[i] = e[i];
        big = std::max(big, std::fabs(d[i]));
    }
    const T tiny = std::numeric_limits<T>::epsilon() * std::max(big, std::numeric_limits<T>::min());
    for (int i = 0; i + 1 < n; ++i) {
        T sub = e[i];
        if (std::fabs(sub) > std::fabs(a[i])) {  // interchange rows i and i+1
            std::swap(a[i], sub);
            std::swap(u[i], a[i + 1]);
            w[i] = u[i + 1];
            u[i + 1] = T(0);
            std::swap(y[i], y[i + 1]);
        }
        if (std::fabs(a[i]) < tiny) a[i] = std::copysign(tiny, a[i]);
        const T m = sub / a[i];
        a[i + 1] -= m * u[i];
        u[i + 1] -= m * w[i];
        y[i + 1] -= m * y[i];
    }
    if (std::fabs(a[n - 1]) < tiny) a[n - 1] = std::copysign(tiny, a[n - 1]);
    T norm = 0, dot = 0;
    for (int i = n - 1; i >= 0; --i) {
        T s = y[i];
        if (i + 1 < n) s -= u[i] * y[i + 1];
        if (i + 2 < n) s -= w[i] * y[i + 2];
        y[i] = s / a[i];
    }
    for (int i = 0; i < n; ++i) {
        norm += y[i] * y[i];
        dot += y[i] * x[i];
    }
    norm = std::copysign(std::sqrt(norm), dot);
    for (int i = 0; i < n; ++i) x[i] = y[i] / norm;
    lam = rayleigh();
}

// The same for a matrix that is symmetric about its middle as well
// (persymmetric: d[i] = d[n-1-i], e[i] = e[n-2-i], up to rounding, which is
// averaged away): the eigenvectors are even or odd, and each kind is the
// eigenproblem of a half.  Even n folds the middle coupling c = e[n/2-1] into
// the half's last diagonal element, +c for the even and -c for the odd vectors;
// odd n keeps the middle row with the even ones, coupled by sqrt(2) e.  The QL
// sweeps' error is absolute, a few units of the largest eigenvalue, which
// leaves the smallest ones of a stretched grid with the leading error of the
// whole solve; one step of inverse iteration in long double on the matrix as
// given removes it.  On return columns m < ceil(n/2) of v are the even vectors
// and the rest the odd ones, each kind in ascending order of d, exactly
// symmetric.
inline bool symtri_eigen_sym(int n, const std::vector<long double>& dl, const std::vector<long double>& el,
                             std::vector<double>& d, std::vector<double>& v) {
    using T = long double;
    const int h = (n + 1) / 2, ho = n / 2;
    d.assign(n, 0.0);
    v.assign((size_t)n * n, 0.0);
    for (int par = 0; par < 2; ++par) {
        const int len = par ? ho : h;
        if (len == 0) continue;
        std::vector<T> dh(len), eh(std::max(len - 1, 1), T(0)), x(len);
        for (int i = 0; i < len; ++i) dh[i] = T(0.5) * (dl[i] + dl[n - 1 - i]);
        for (int i = 0; i + 1 < len; ++i) eh[i] = T(0.5) * (el[i] + el[n - 2 - i]);
        if (n % 2 == 0) dh[len - 1] += (par ? T(-1) : T(1)) * el[n / 2 - 1];
        else if (!par && len > 1) eh[len - 2] *= std::sqrt(T(2));
        std::vector<double> dd(dh.begin(), dh.end()), ee(eh.begin(), eh.end()), q;
        if (!symtri_eigen(len, dd, ee, q)) return false;
        for (int m = 0; m < len; ++m) {
            T lam = dd[m];
            std::copy(q.begin() + (size_t)m * len, q.begin() + (size_t)(m + 1) * len, x.begin());
            symtri_refine(len, dh.data(), eh.data(), lam, x);
            const int col = par ? h + m : m;
            d[col] = (double)lam;
            double* c = v.data() + (size_t)col * n;
            for (int k = 0; k < len; ++k) {
                if (k == n - 1 - k) {
                    c[k] = (double)x[k];
                } else {
                    c[k] = (double)(x[k] * std::sqrt(T(0.5)));
                    c[n - 1 - k] = par ? -c[k] : c[k];
                }
            }
        }
    }
    return true;
}

}  // namespace dfp
