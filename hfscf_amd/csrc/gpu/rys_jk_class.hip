// One angular-momentum class of the Rys J/K kernel; built once per class with -DHFG_LA=.. -DHFG_LB=..
// -DHFG_LC=.. -DHFG_LD=.. (the Cartesian density serves both basis types).
#include "rys_jk.hpp"

namespace hfg {

template <>
hipError_t launch_rys_jk_class<HFG_LA, HFG_LB, HFG_LC, HFG_LD>(const RysJkArgs& a, LaunchShape sh, hipStream_t s) {
    // persistent workgroups: by default as many as items (the queue drains either way)
    const int grid = sh.grid > 0 ? std::min(sh.grid, a.j.nitems) : a.j.nitems;
    hipLaunchKernelGGL((rys_jk_kernel<HFG_LA, HFG_LB, HFG_LC, HFG_LD>), dim3(grid), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace hfg
