// Rys quadrature on the device: nodes and weights from the generated tables (rys_layout.hpp) and
// the 1-D recursion of one direction at one node (J. Rys, M. Dupuis, H. F. King, J. Comput. Chem.
// 4, 154 (1983)).
#pragma once
#include <hip/hip_runtime.h>

#include "cart.hpp"
#include "rys_layout.hpp"

namespace hfg {

// exponent of direction d of component k of a shell (hfscf's order, as cart.hpp's)
HFG_HD int cart_exp(int L, int k, int d) {
    int i = 0;
    while ((i + 1) * (i + 2) / 2 <= k) ++i;
    const int lz = k - i * (i + 1) / 2;
    return d == 0 ? L - i : (d == 1 ? i - lz : lz);
}

// Device address of the tables on `device` (looked up once per device).
hipError_t rys_table(int device, const double** out);

// Node u in (0, 1) and weight w of point r of the N-point rule at T >= 0.
template <int N>
HFG_INLINE void rys_point(const double* __restrict__ tab, double T, int r, double& u, double& w) {
    if (T < (double)kRysTmax) {
        const int k = (int)(T * kRysPerUnit);
        const double x = 2.0 * kRysPerUnit * T - (2.0 * k + 1.0);
        const double* c = tab + rys_offset(N) + (k * N + r) * kRysRow;
        u = c[kRysDeg];
        w = c[2 * kRysDeg + 1];
#pragma unroll
        for (int j = kRysDeg - 1; j >= 0; --j) {
            u = u * x + c[j];
            w = w * x + c[kRysDeg + 1 + j];
        }
    } else {
        const double* c = tab + rys_far(N) + 2 * r;
        const double rs = rsqrt(T);
        u = c[0] * (rs * rs);
        w = c[1] * rs;
    }
}

// G(n, m) of one direction at one node, n < NN, m < NM, stored at g[m * NN + n]: g00 on (0, 0), c0 =
// PA - u q/(p+q) PQ, d0 = QC + u p/(p+q) PQ, b10, b01, b00 the usual coefficients of the node.
template <int NN, int NM>
HFG_INLINE void rys_2d(double g00, double c0, double d0, double b10, double b01, double b00, double* g) {
    double p0[NN], p1[NN];  // columns m - 1 and m
    p1[0] = g00;
    if constexpr (NN > 1) p1[1] = c0 * g00;
    sfor<(NN > 2 ? NN - 2 : 0)>([&](auto k) { p1[k + 2] = c0 * p1[k + 1] + (double)(k + 1) * b10 * p1[k]; });
    sfor<NN>([&](auto n) { g[n] = p1[n]; });
    sfor<NM - 1>([&](auto m) {
        double t[NN];
        sfor<NN>([&](auto n) {
            double v = d0 * p1[n];
            if constexpr (m > 0) v += (double)(int)m * b01 * p0[n];
            if constexpr (n > 0) v += (double)(int)n * b00 * p1[n - 1];
            t[n] = v;
        });
        sfor<NN>([&](auto n) {
            p0[n] = p1[n];
            p1[n] = t[n];
            g[(m + 1) * NN + n] = t[n];
        });
    });
}

}  // namespace hfg
