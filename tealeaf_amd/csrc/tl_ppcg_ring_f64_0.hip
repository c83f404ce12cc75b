// tl_ppcg_ring.h for double, mode 0.
#include "tl_ppcg_ring.h"

template int tl::fused::dispatch_ring<double, 0>(int, const FusedArgs<double>&);
