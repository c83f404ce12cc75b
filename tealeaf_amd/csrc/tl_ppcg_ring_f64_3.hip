// tl_ppcg_ring.h for double, mode 3.
#include "tl_ppcg_ring.h"

template int tl::fused::dispatch_ring<double, 3>(int, const FusedArgs<double>&);
