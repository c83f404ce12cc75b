// tl_ppcg_ring.h for float, mode 3.
#include "tl_ppcg_ring.h"

template int tl::fused::dispatch_ring<float, 3>(int, const FusedArgs<float>&);
