// Kernel specialisations built with the occupancy machine scheduler, the
// compiler's default (-amdgpu-sched-strategy=max-occupancy, set for this file
// in build.py), instead of the max-ILP one of the other fit kernels.  Their
// finders declare them extern.  Both schedulers keep these within the same waves
// per SIMD; max-ILP spends more moves on them.  us per launch of 300,000 ROIs,
// max-ILP and here: XYNBS 8 px on one lane 287.7 and 275.5, XYNBS 11 px on 2 lanes
// 498.7 and 486.5, astigmatic 14 px on 2 lanes 726.7 and 699.6.
#include "gmle_instances.hpp"
GMLE_INSTANTIATE_FIT(XYNBS, IDEAL, PREC_FP32, 8, 1)
GMLE_INSTANTIATE_FIT(XYNBS, IDEAL, PREC_FP32, 11, 2)
GMLE_INSTANTIATE_FIT(ASTIG, IDEAL, PREC_FP32, 14, 2)
