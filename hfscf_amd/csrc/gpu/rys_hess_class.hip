// One angular-momentum class of the Hessian kernel; built once per class with -DHFG_LA=.. -DHFG_LB=..
// -DHFG_LC=.. -DHFG_LD=.. (the Cartesian density serves both basis types).
#include "rys_hess.hpp"

namespace hfg {

template <>
hipError_t launch_rys_hess_class<HFG_LA, HFG_LB, HFG_LC, HFG_LD>(const HessArgs& g, hipStream_t s) {
    // persistent workgroups: 3 per CU by their LDS; the queue drains whatever their number
    const long long grid = std::min<long long>(g.nitems, 256 * 3);
    hipLaunchKernelGGL((rys_hess_kernel<HFG_LA, HFG_LB, HFG_LC, HFG_LD>), dim3((unsigned)grid), dim3(kHessBlock), 0, s, g);
    return hipGetLastError();
}

}  // namespace hfg
