// tl_ppcg_ring.h for float, mode 2.
#include "tl_ppcg_ring.h"

template int tl::fused::dispatch_ring<float, 2>(int, const FusedArgs<float>&);
