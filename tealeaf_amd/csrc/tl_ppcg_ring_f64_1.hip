// tl_ppcg_ring.h for double, mode 1.
#include "tl_ppcg_ring.h"

template int tl::fused::dispatch_ring<double, 1>(int, const FusedArgs<double>&);
