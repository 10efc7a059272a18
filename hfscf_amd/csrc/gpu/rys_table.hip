// The Rys quadrature tables as device data (0.48 MB, L2-resident), generated at build time.
#include <mutex>
#include <vector>

#include "rys.hpp"

namespace hfg {

// not const: a const table that no kernel of this file reads would not be emitted for the device
static __device__ __align__(256) double rys_data[kRysTableSize] = {
#include "rys_table.inc"
};

hipError_t rys_table(int device, const double** out) {
    static std::mutex mu;
    static std::vector<const double*> addr;
    std::lock_guard<std::mutex> lock(mu);
    if ((int)addr.size() <= device) addr.resize(device + 1, nullptr);
    if (!addr[device]) {
        int cur = 0;
        hipError_t e = hipGetDevice(&cur);
        if (e != hipSuccess) return e;
        if (cur != device && (e = hipSetDevice(device)) != hipSuccess) return e;
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(rys_data));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess) return e;
        addr[device] = static_cast<const double*>(p);
    }
    *out = addr[device];
    return hipSuccess;
}

}  // namespace hfg
