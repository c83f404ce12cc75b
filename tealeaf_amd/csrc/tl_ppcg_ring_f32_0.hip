// tl_ppcg_ring.h for float, mode 0.
#include "tl_ppcg_ring.h"

template int tl::fused::dispatch_ring<float, 0>(int, const FusedArgs<float>&);
