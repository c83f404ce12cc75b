// tl_ppcg_ring.h for double, mode 2.
#include "tl_ppcg_ring.h"

template int tl::fused::dispatch_ring<double, 2>(int, const FusedArgs<double>&);
