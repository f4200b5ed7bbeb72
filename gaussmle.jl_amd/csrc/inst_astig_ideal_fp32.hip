// Kernel specialisations for model ASTIG, camera IDEAL, precision FP32.
#include "gmle_instances.hpp"
// 14 px on 2 lanes is built in inst_sched_occ.hip.
GMLE_EXTERN_FIT(ASTIG, IDEAL, PREC_FP32, 14, 2)
GMLE_DEFINE_FINDER(ASTIG, IDEAL, PREC_FP32)
