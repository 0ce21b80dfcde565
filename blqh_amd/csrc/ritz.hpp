// ritz.hpp -- host routines for low Ritz vectors of a Lanczos tridiagonal,
// shared by the batched solver and its CPU tests.
#pragma once
#include <algorithm>
#include <cmath>
#include <vector>

namespace blqh {

// Number of eigenvalues below x of the tridiagonal (a, b) (Sturm sequence).
inline int sturm_below(int m, const double* a, const double* b, double x) {
    int c = 0;
    double q = 1.0;
    for (int i = 0; i < m; ++i) {
        q = a[i] - x - (i ? b[i - 1] * b[i - 1] / q : 0.0);
        if (q == 0.0) q = -1e-300;
        if (q < 0) ++c;
    }
    return c;
}

// Eight Sturm sequences at once: bit k of the result says whether (a, b) has an
// eigenvalue below x[k].  A sequence is a chain of divisions, about 20 clocks a row;
// the eight fill the divider between them, so they cost what one costs.
inline unsigned sturm_any8(int m, const double* a, const double* b, const double* x) {
    typedef double d2 __attribute__((vector_size(16)));
    typedef long long l2 __attribute__((vector_size(16)));
    d2 q[4], xs[4];
    l2 neg[4];
    const d2 zero = {0.0, 0.0}, tiny = {-1e-300, -1e-300};
    for (int k = 0; k < 4; ++k) {
        xs[k] = d2{x[2 * k], x[2 * k + 1]};
        q[k] = d2{1.0, 1.0};
        neg[k] = l2{0, 0};
    }
    for (int i = 0; i < m; ++i) {
        const double bb = i ? b[i - 1] * b[i - 1] : 0.0;
        const d2 av = {a[i], a[i]}, bv = {bb, bb};
        for (int k = 0; k < 4; ++k) {
            d2 v = av - xs[k] - bv / q[k];
            const l2 z = (l2)(v == zero);
            v = (d2)(((l2)v & ~z) | ((l2)tiny & z));
            neg[k] |= (l2)(v < zero);
            q[k] = v;
        }
    }
    unsigned r = 0;
    for (int k = 0; k < 8; ++k) r |= neg[k >> 1][k & 1] ? 1u << k : 0u;
    return r;
}

// The lowest eigenvalue of (a, b), lo <= it <= hi: the bracket is cut in nine by
// eight sequences at a time until no number lies between its ends, where bisection ends
// too (17 passes instead of 52 from a bracket of the matrix's norm).
inline double lowest_in(int m, const double* a, const double* b, double lo, double hi) {
    for (int it = 0; it < 200; ++it) {
        const double mid = 0.5 * (lo + hi);
        if (mid <= lo || mid >= hi) break;
        double x[8];
        for (int k = 0; k < 8; ++k) x[k] = lo + (hi - lo) * ((k + 1) / 9.0);
        x[4] = mid;  // close to the fifth point, and always between the ends
        const unsigned r = sturm_any8(m, a, b, x);
        double nlo = lo, nhi = hi;
        for (int k = 0; k < 8; ++k) {
            if (r >> k & 1) nhi = x[k] < nhi ? x[k] : nhi;
            else nlo = x[k] > nlo ? x[k] : nlo;
        }
        if (nlo >= nhi) {  // rounding at the last ulps: bisect
            nlo = r >> 4 & 1 ? lo : mid;
            nhi = r >> 4 & 1 ? mid : hi;
        }
        lo = nlo;
        hi = nhi;
    }
    return 0.5 * (lo + hi);
}

// True if the residual beta_m |s_m| / |s| of the Ritz pair of theta, an eigenvalue of
// (a, b) to rounding, certainly exceeds ten times res_tol: s by the three-term
// recurrence from its last component, s_m = 1, which is the stable direction while the
// components fall towards the end.  Its defect, all in the first row, bounds the error;
// if that is not small the answer is false and the pair is left to inverse iteration,
// whose four eliminations and bisection cost a hundred times as much.
inline bool residual_exceeds(int m, const double* a, const double* b, double theta, double beta_m, double res_tol) {
    double z1 = 1.0, z2 = 0.0, s2 = 1.0;  // components i and i + 1
    for (int i = m - 1; i > 0; --i) {
        const double z0 = ((theta - a[i]) * z1 - (i + 1 < m ? b[i] * z2 : 0.0)) / b[i - 1];
        s2 += z0 * z0;
        z2 = z1;
        z1 = z0;
        if (!(s2 < 1e200)) return false;
    }
    const double defect = std::fabs((a[0] - theta) * z1 + (m > 1 ? b[0] * z2 : 0.0));
    const double nrm = std::sqrt(s2);
    return defect <= 1e-11 * nrm && beta_m > 10.0 * res_tol * nrm;
}

// Eigenvector k (ascending) of the m x m tridiagonal (a, b): the eigenvalue
// by bisection on Sturm counts, the vector by three steps of inverse
// iteration, each solve by Gaussian elimination with partial pivoting on the
// band (the steps of LAPACK's dgttrf / dgttrs).  x gets a unit vector.
inline void tridiag_vector_k(int m, const double* a, const double* b, int k, double* x) {
    double lo = a[0], hi = a[0];
    for (int i = 0; i < m; ++i) {
        const double r = (i ? std::fabs(b[i - 1]) : 0.0) + (i + 1 < m ? std::fabs(b[i]) : 0.0);
        lo = std::min(lo, a[i] - r);
        hi = std::max(hi, a[i] + r);
    }
    for (int it = 0; it < 200; ++it) {
        const double mid = 0.5 * (lo + hi);
        if (mid <= lo || mid >= hi) break;
        if (sturm_below(m, a, b, mid) >= k + 1) hi = mid; else lo = mid;
    }
    const double e = 0.5 * (lo + hi);
    const double sh = e - 1e-13 * std::max(1.0, std::fabs(e));
    std::vector<double> dl(m), dd(m), du(m), du2(m), y(m);
    std::vector<char> sw(m, 0);
    for (int i = 0; i < m; ++i) {
        dd[i] = a[i] - sh;
        du[i] = i + 1 < m ? b[i] : 0.0;
        dl[i] = i + 1 < m ? b[i] : 0.0;
        du2[i] = 0.0;
    }
    for (int i = 0; i + 1 < m; ++i) {
        if (std::fabs(dd[i]) >= std::fabs(dl[i])) {
            if (dd[i] == 0.0) dd[i] = 1e-300;
            const double l = dl[i] / dd[i];
            dl[i] = l;
            dd[i + 1] -= l * du[i];
        } else {  // rows i and i + 1 swap
            const double l = dd[i] / dl[i];
            dd[i] = dl[i];
            dl[i] = l;
            const double t = du[i];
            du[i] = dd[i + 1];
            dd[i + 1] = t - l * dd[i + 1];
            if (i + 2 < m) {
                du2[i] = du[i + 1];
                du[i + 1] = -l * du[i + 1];
            }
            sw[i] = 1;
        }
    }
    if (dd[m - 1] == 0.0) dd[m - 1] = 1e-300;
    for (int i = 0; i < m; ++i) x[i] = 1.0 / std::sqrt((double)m);
    for (int iter = 0; iter < 3; ++iter) {
        for (int i = 0; i < m; ++i) y[i] = x[i];
        for (int i = 0; i + 1 < m; ++i) {
            if (sw[i]) {
                const double t = y[i];
                y[i] = y[i + 1];
                y[i + 1] = t - dl[i] * y[i];
            } else {
                y[i + 1] -= dl[i] * y[i];
            }
        }
        for (int i = m - 1; i >= 0; --i) {
            double v = y[i];
            if (i + 1 < m) v -= du[i] * x[i + 1];
            if (i + 2 < m) v -= du2[i] * x[i + 2];
            x[i] = v / dd[i];
        }
        double s = 0;
        for (int i = 0; i < m; ++i) s += x[i] * x[i];
        s = 1.0 / std::sqrt(s);
        for (int i = 0; i < m; ++i) x[i] *= s;
    }
}

// Excited mix of a finished Lanczos run: the normalised sum of the second
// and third lowest Ritz vectors (those that exist), orthogonalised against
// the ground Ritz vector c0; zero when m = 1.  The start of a continuation
// solve adds it so that a state that was excited at the previous parameter
// point and is the ground state at the next one starts with a large weight.
inline void excited_mix(int m, const double* a, const double* b, const double* c0, double* out) {
    for (int l = 0; l < m; ++l) out[l] = 0.0;
    if (m < 2) return;
    std::vector<double> v(m);
    for (int k = 1; k <= std::min(2, m - 1); ++k) {
        tridiag_vector_k(m, a, b, k, v.data());
        for (int l = 0; l < m; ++l) out[l] += v[l];
    }
    double d = 0, s = 0;
    for (int l = 0; l < m; ++l) d += out[l] * c0[l];
    for (int l = 0; l < m; ++l) {
        out[l] -= d * c0[l];
        s += out[l] * out[l];
    }
    if (!(s > 0) || !std::isfinite(s)) {
        for (int l = 0; l < m; ++l) out[l] = 0.0;
        return;
    }
    s = 1.0 / std::sqrt(s);
    for (int l = 0; l < m; ++l) out[l] *= s;
}

}  // namespace blqh
