// Kernel specialisations built with the occupancy machine scheduler, the
// compiler's default (-amdgpu-sched-strategy=max-occupancy, set for this file
// in build.py), instead of the max-ILP one of the other fit kernels: XYNBS
// 16 px sCMOS on 4 lanes, which max-ILP takes past 256 VGPRs (1M ROIs: 2.93
// against 4.19 ms).  Its finder declares it extern.
#include "gmle_instances.hpp"
GMLE_INSTANTIATE_FIT(XYNBS, SCMOS, PREC_FP32, 16, 4)
