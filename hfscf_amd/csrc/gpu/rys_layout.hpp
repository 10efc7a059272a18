// Layout of the Rys quadrature tables, shared by their build-time generator and the kernels.
#pragma once

namespace hfg {

constexpr int kRysGradMinL = 4;    // FP64 gradient classes from this L run the Rys kernel
// FP64 J/K classes from kRysJkMinL run the Rys kernel, from kRysJkSmallL those with few shell quartets.
constexpr int kRysJkMinL = 6, kRysJkSmallL = 4;
// Mixed builds and gradients run the same FP64 kernels from kRysMixedL.
constexpr int kRysMixedL = 7;
constexpr bool jk_has_rys(int la, int lb, int lc, int ld) { return la + lb + lc + ld >= kRysJkSmallL; }
// Gradient classes that keep their FP64 register kernel for many shell quartets.
constexpr bool grad_keeps_register(int la, int lb, int lc, int ld) {
    return la + lb + lc + ld < kRysGradMinL || (la + lb + lc + ld == 4 && la == 2);
}
constexpr int kRysMaxN = 6;        // rules of 1..6 points (degree 11: total order up to 11)
constexpr int kRysDeg = 9;         // polynomial degree per interval
constexpr int kRysPerUnit = 2;     // intervals per unit of T
constexpr int kRysTmax = 72;       // from here on the half-range Hermite constants hold to 1e-18
constexpr int kRysIntervals = kRysTmax * kRysPerUnit;
constexpr int kRysRow = 2 * (kRysDeg + 1);  // node and weight polynomials of one point

// Doubles before the n-point rule's rows ([interval][point][node, weight polynomial]), and before
// its constants beyond kRysTmax ([point][node, weight]).
constexpr int rys_offset(int n) { return kRysIntervals * kRysRow * (n * (n - 1) / 2); }
constexpr int kRysFarBase = kRysIntervals * kRysRow * (kRysMaxN * (kRysMaxN + 1) / 2);
constexpr int rys_far(int n) { return kRysFarBase + n * (n - 1); }
constexpr int kRysTableSize = kRysFarBase + kRysMaxN * (kRysMaxN + 1);

// A molecule's slice of the concatenated Cartesian densities.
struct MolCart {
    long long off;
    int n;     // Cartesian functions
    int row0;  // first row of the concatenated CartTerms
};

// A Cartesian function as a sum of at most two output functions (indices in its molecule).
struct CartTerms {
    int n, f[2];
    double w[2];
};

}  // namespace hfg
