// Build-time generator of the Rys quadrature tables (printed as a C++ initialiser list).
//
// For n = 1..kRysMaxN the nodes u_i = t_i^2 and weights w_i with
//   int_0^1 exp(-T t^2) f(t^2) dt = sum_i w_i f(u_i)   for polynomials f of degree <= 2n - 1.
// The recursion coefficients of the polynomials orthogonal under exp(-T t^2) dt in u = t^2 come
// from the discretised Stieltjes procedure (W. Gautschi, Orthogonal Polynomials: Computation and
// Approximation, 2.2.3) on 96 Gauss-Legendre points, the nodes and weights from the eigenvalues
// and first eigenvector components of their Jacobi matrix (Golub and Welsch), in long double. Per
// interval of T both are Chebyshev-interpolated to degree kRysDeg and stored as powers of the
// interval's variable in [-1, 1]: 1.2e-17 of the largest node, 2.2e-17 of F_0 for the weights.
#include <cmath>
#include <cstdio>
#include <utility>
#include <vector>

#include "rys_layout.hpp"

using ld = long double;
using namespace hfg;

static constexpr int kPoints = 96;
static ld gx[kPoints], gw[kPoints];  // Gauss-Legendre on (0, 1)

static void legendre() {
    for (int i = 0; i < kPoints; ++i) {
        ld x = cosl(M_PIl * (i + 0.75L) / (kPoints + 0.5L)), dp = 0;
        for (int it = 0; it < 100; ++it) {
            ld p0 = 1, p1 = x;
            for (int k = 2; k <= kPoints; ++k) {
                const ld p2 = ((2 * k - 1) * x * p1 - (k - 1) * p0) / k;
                p0 = p1;
                p1 = p2;
            }
            dp = kPoints * (x * p1 - p0) / (x * x - 1);
            const ld dx = p1 / dp;
            x -= dx;
            if (fabsl(dx) < 1e-19L) break;
        }
        gx[i] = 0.5L * (1 + x);
        gw[i] = 1 / ((1 - x * x) * dp * dp);
    }
}

// Recursion coefficients a_k, b_k (b_0 = F_0(T)), k < kRysMaxN.
static void stieltjes(ld T, ld* a, ld* b) {
    std::vector<ld> u(kPoints), w(kPoints), p0(kPoints, 0), p1(kPoints, 1);
    for (int i = 0; i < kPoints; ++i) {
        u[i] = gx[i] * gx[i];
        w[i] = gw[i] * expl(-T * u[i]);
    }
    ld prev = 1;
    for (int k = 0; k < kRysMaxN; ++k) {
        ld nn = 0, un = 0;
        for (int i = 0; i < kPoints; ++i) {
            nn += w[i] * p1[i] * p1[i];
            un += w[i] * u[i] * p1[i] * p1[i];
        }
        a[k] = un / nn;
        b[k] = k ? nn / prev : nn;
        prev = nn;
        for (int i = 0; i < kPoints; ++i) {
            const ld t = (u[i] - a[k]) * p1[i] - (k ? b[k] : 0) * p0[i];
            p0[i] = p1[i];
            p1[i] = t;
        }
    }
}

// Nodes (ascending) and weights of the n-point rule: implicit QL on the Jacobi matrix.
static void rule(int n, const ld* a, const ld* b, ld* r, ld* w) {
    ld d[kRysMaxN], e[kRysMaxN + 1], z[kRysMaxN];
    for (int i = 0; i < n; ++i) {
        d[i] = a[i];
        e[i] = i + 1 < n ? sqrtl(b[i + 1]) : 0;
        z[i] = i == 0;
    }
    for (int l = 0; l < n; ++l)
        for (;;) {
            int m = l;
            while (m < n - 1 && fabsl(e[m]) > 1e-20L * (fabsl(d[m]) + fabsl(d[m + 1]))) ++m;
            if (m == l) break;
            ld g = (d[l + 1] - d[l]) / (2 * e[l]), h = hypotl(g, 1);
            g = d[m] - d[l] + e[l] / (g + (g >= 0 ? h : -h));
            ld s = 1, c = 1, p = 0;
            int i = m - 1;
            for (; i >= l; --i) {
                const ld f = s * e[i], q = c * e[i];
                h = hypotl(f, g);
                e[i + 1] = h;
                if (h == 0) {
                    d[i + 1] -= p;
                    e[m] = 0;
                    break;
                }
                s = f / h;
                c = g / h;
                g = d[i + 1] - p;
                h = (d[i] - g) * s + 2 * c * q;
                p = s * h;
                d[i + 1] = g + p;
                g = c * h - q;
                const ld t = z[i + 1];
                z[i + 1] = s * z[i] + c * t;
                z[i] = c * z[i] - s * t;
            }
            if (h == 0 && i >= l) continue;
            d[l] -= p;
            e[l] = g;
            e[m] = 0;
        }
    for (int i = 0; i < n; ++i) {
        r[i] = d[i];
        w[i] = b[0] * z[i] * z[i];
    }
    for (int i = 0; i < n; ++i)
        for (int j = i + 1; j < n; ++j)
            if (r[j] < r[i]) {
                std::swap(r[i], r[j]);
                std::swap(w[i], w[j]);
            }
}

// Values at the K Chebyshev points of [-1, 1] -> coefficients of powers of x.
static void powers(const ld* f, int K, ld* out) {
    std::vector<ld> t0(K, 0), t1(K, 0), t2(K, 0);
    for (int j = 0; j < K; ++j) out[j] = 0;
    t0[0] = 1;
    if (K > 1) t1[1] = 1;
    for (int j = 0; j < K; ++j) {
        ld c = 0;
        for (int k = 0; k < K; ++k) c += f[k] * cosl(j * M_PIl * (k + 0.5L) / K);
        c *= (j ? 2.0L : 1.0L) / K;
        const std::vector<ld>& t = j == 0 ? t0 : t1;
        for (int i = 0; i < K; ++i) out[i] += c * t[i];
        if (j == 0) continue;
        for (int i = 0; i < K; ++i) t2[i] = (i ? 2 * t1[i - 1] : 0) - t0[i];
        t0 = t1;
        t1 = t2;
    }
}

int main() {
    constexpr int K = kRysDeg + 1;
    legendre();
    std::vector<ld> r(kRysIntervals * K * kRysMaxN * kRysMaxN), w(r.size());
    ld a[kRysMaxN], b[kRysMaxN];
    auto at = [&](int k, int c, int n) { return (((size_t)k * K + c) * kRysMaxN + n - 1) * kRysMaxN; };
    for (int k = 0; k < kRysIntervals; ++k)
        for (int c = 0; c < K; ++c) {
            const ld x = cosl(M_PIl * (c + 0.5L) / K);
            stieltjes((k + 0.5L * (1 + x)) / kRysPerUnit, a, b);
            for (int n = 1; n <= kRysMaxN; ++n) rule(n, a, b, &r[at(k, c, n)], &w[at(k, c, n)]);
        }
    ld f[K], p[K];
    for (int n = 1; n <= kRysMaxN; ++n)
        for (int k = 0; k < kRysIntervals; ++k)
            for (int i = 0; i < n; ++i)
                for (int q = 0; q < 2; ++q) {
                    for (int c = 0; c < K; ++c) f[c] = (q ? w : r)[at(k, c, n) + i];
                    powers(f, K, p);
                    for (int j = 0; j < K; ++j) std::printf("%.17Lg,%c", p[j], j + 1 < K ? ' ' : '\n');
                }
    // beyond the table the upper limit is infinity to rounding: u_i T and w_i sqrt(T) are the
    // constants of the half-range Hermite rule, taken at T = 200
    const ld Tl = 200;
    stieltjes(Tl, a, b);
    for (int n = 1; n <= kRysMaxN; ++n) {
        rule(n, a, b, f, p);
        for (int i = 0; i < n; ++i) std::printf("%.17Lg, %.17Lg,\n", f[i] * Tl, p[i] * sqrtl(Tl));
    }
    return 0;
}
