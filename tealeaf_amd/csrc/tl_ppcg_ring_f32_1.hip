// tl_ppcg_ring.h for float, mode 1.
#include "tl_ppcg_ring.h"

template int tl::fused::dispatch_ring<float, 1>(int, const FusedArgs<float>&);
