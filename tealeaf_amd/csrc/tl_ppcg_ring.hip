// The LDS-ring PPCG and Chebyshev loops (tl_ppcg_ring.h): choice of the mode.
#include "tl_fused.h"
#include "tealeaf_hip.h"

namespace tl {
namespace fused {

double g_ring_fill = -1.0;   // tlhip_set_ring_fill

// instantiated in tl_ppcg_ring_{f64,f32}_{0,1,2,3}.hip
template <class T, int MODE>
int dispatch_ring(int count, const FusedArgs<T>& a);

template <class T>
int launch_ppcg_ring(int count, int mode, const FusedArgs<T>& a)
{
    switch (mode) {
    case 0: return dispatch_ring<T, 0>(count, a);
    case 1: return dispatch_ring<T, 1>(count, a);
    case 2: return dispatch_ring<T, 2>(count, a);
    default: return dispatch_ring<T, 3>(count, a);
    }
}

template int launch_ppcg_ring<double>(int, int, const FusedArgs<double>&);
template int launch_ppcg_ring<float>(int, int, const FusedArgs<float>&);

}  // namespace fused
}  // namespace tl

extern "C" int tlhip_set_ring_fill(double fill)
{
    if (!(fill <= 1.5)) return tl_fail(TLHIP_ERR_ARG, "tlhip_set_ring_fill: %g", fill);
    tl::fused::g_ring_fill = fill;
    return 0;
}
