// Run-time dispatch of the Rys gradient and J/K kernels and the Cartesian densities that they read.
#include "rys_grad.hpp"
#include "rys_jk.hpp"

namespace hfg {

#define HFG_RYS_CASE(A, B, C, D)                                                                  \
    if constexpr (A + B + C + D >= kRysGradMinL)                                                  \
        if (la == A && lb == B && lc == C && ld == D) return launch_rys_grad_class<A, B, C, D>(b, sh, s);

#define HFG_DECL(A, B, C, D) \
    template <>              \
    hipError_t launch_rys_grad_class<A, B, C, D>(const RysGradArgs&, LaunchShape, hipStream_t);
HFG_FOR_CLASSES(HFG_DECL)
#undef HFG_DECL

hipError_t launch_rys_grad(int la, int lb, int lc, int ld, const RysGradArgs& a, int nitems, LaunchShape sh,
                           hipStream_t s) {
    if (nitems == 0) return hipSuccess;
    RysGradArgs b = a;
    b.g.nitems = nitems;
    HFG_FOR_CLASSES(HFG_RYS_CASE)
    return hipErrorInvalidValue;
}

#define HFG_DECL(A, B, C, D) \
    template <>              \
    hipError_t launch_rys_jk_class<A, B, C, D>(const RysJkArgs&, LaunchShape, hipStream_t);
HFG_FOR_CLASSES(HFG_DECL)
#undef HFG_DECL

#define HFG_RYS_JK_CASE(A, B, C, D)   \
    if constexpr (jk_has_rys(A, B, C, D)) \
        if (la == A && lb == B && lc == C && ld == D) return launch_rys_jk_class<A, B, C, D>(b, sh, s);

hipError_t launch_rys_jk(int la, int lb, int lc, int ld, const RysJkArgs& a, int nitems, LaunchShape sh, hipStream_t s) {
    if (nitems == 0) return hipSuccess;
    RysJkArgs b = a;
    b.j.nitems = nitems;
    HFG_FOR_CLASSES(HFG_RYS_JK_CASE)
    return hipErrorInvalidValue;
}

// One thread per Cartesian element; 2 x 2 terms at most, so it moves little more than D and Dc. Molecules on
// blockIdx.x: a batch may hold more than the 65,536 workgroups of the other dimensions.
__global__ __launch_bounds__(256) void to_cart_kernel(const double* __restrict__ D, const MolDev* __restrict__ mols,
                                                      const MolCart* __restrict__ mc, const CartTerms* __restrict__ terms,
                                                      double* __restrict__ Dc) {
    const MolCart m = mc[blockIdx.x];
    const MolDev md = mols[blockIdx.x];
    const double* Dm = D + md.moff;
    for (int e = blockIdx.y * 256 + threadIdx.x; e < m.n * m.n; e += gridDim.y * 256) {
        const int i = e / m.n, j = e - i * m.n;
        const CartTerms ti = terms[m.row0 + i], tj = terms[m.row0 + j];
        double v = 0.0;
        for (int x = 0; x < ti.n; ++x)
            for (int y = 0; y < tj.n; ++y) v += ti.w[x] * tj.w[y] * Dm[(size_t)ti.f[x] * md.n + tj.f[y]];
        Dc[m.off + e] = v;
    }
}

hipError_t launch_to_cart(const double* D, const MolDev* mols, const MolCart* mc, int nmol, int max_ncart,
                          const CartTerms* terms, double* Dc, hipStream_t s) {
    const int grid = std::max(1, std::min(1024, (max_ncart * max_ncart + 255) / 256));
    hipLaunchKernelGGL(to_cart_kernel, dim3(nmol, grid), dim3(256), 0, s, D, mols, mc, terms, Dc);
    return hipGetLastError();
}

}  // namespace hfg
