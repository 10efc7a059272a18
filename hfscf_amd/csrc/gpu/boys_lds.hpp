// Boys functions F_0..F_M in FP64 from a table in LDS, for the kernels whose primitive quartets they
// dominate.
//
// The rows of the device table at T = k/8 (every fourth of boys.hpp), cut to the M + 9 columns that the
// Taylor sums of F_0..F_M about the nearest row need: 9 terms each (|T - k/8| <= 1/16, truncation below
// 5e-17 relative), no e^-T and no recursion. From T = 36 F_0 = sqrt(pi/T)/2 and the upward recursion, with
// e^-T only where it reaches the last bit of F_M.
//
// Against erf and exp from the library (boys_low) the group kernels of jk_gc.hip and jk_gc_impl.hpp lost
// about half of their instructions per primitive quartet; alone on (H2O)16 / cc-pVDZ (ss|ss) 4.8 -> 3.3 ms,
// (ps|ss) 7.2 -> 5.9. The table in L2 instead stalls on the lanes' scattered rows.
#pragma once
#include "boys.hpp"

namespace hfg {

constexpr int kBoysLdsMaxM = 4;  // e^-T is dropped by orders up to 4
constexpr int kBoysLdsRows = 36 * 8 + 1;
__host__ __device__ constexpr int boys_lds_cols(int M) { return (M + 10) & ~1; }  // rows of whole 16-byte reads
__host__ __device__ constexpr int boys_lds_size(int M) { return kBoysLdsRows * boys_lds_cols(M); }

// Fills the workgroup's table (the caller synchronises before the first evaluation).
template <int M>
__device__ __forceinline__ void boys_lds_load(const double* __restrict__ tab, double* lds) {
    constexpr int cols = boys_lds_cols(M);
    for (int k = threadIdx.x; k < boys_lds_size(M); k += blockDim.x)
        lds[k] = tab[(k / cols) * (4 * kBoysCols) + k % cols];
}

// F_0..F_M scaled by `scale`; lds from boys_lds_load<M>, 16-byte aligned.
template <int M>
__device__ __forceinline__ void boys_lds(double T, const double* lds, double scale, double* F) {
    static_assert(M <= kBoysLdsMaxM, "e^-T is dropped by orders up to 4");
    if (T < kBoysTmax) {
        const int k = __double2int_rn(T * 8.0);
        const double dt = (double)k * 0.125 - T;
        const double2* row = reinterpret_cast<const double2*>(lds + k * boys_lds_cols(M));
        double r[boys_lds_cols(M)], d[9];
#pragma unroll
        for (int n = 0; n < boys_lds_cols(M) / 2; ++n) {
            const double2 v = row[n];
            r[2 * n] = v.x;
            r[2 * n + 1] = v.y;
        }
#pragma unroll
        for (int n = 1; n <= 8; ++n) d[n] = dt * (1.0 / n);
#pragma unroll
        for (int m = 0; m <= M; ++m) {
            double s = r[m + 8];
#pragma unroll
            for (int n = 8; n >= 1; --n) s = r[m + n - 1] + s * d[n];
            F[m] = scale * s;
        }
    } else {
        const double y = rsqrt(T), h = 0.5 * y * y;
        double f = 0.88622692545275801365 * y;  // sqrt(pi)/2
        F[0] = scale * f;
        if constexpr (M > 0) {
            double eT = 0.0;
            if (T < 39.0 + 3.0 * M) eT = exp(-T);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                f = ((2 * m + 1) * f - eT) * h;
                F[m + 1] = scale * f;
            }
        }
    }
}

}  // namespace hfg
