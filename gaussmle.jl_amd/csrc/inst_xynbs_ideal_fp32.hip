// Kernel specialisations for model XYNBS, camera IDEAL, precision FP32.
#include "gmle_instances.hpp"
// 8 px on one lane and 11 px on 2 are built in inst_sched_occ.hip.
GMLE_EXTERN_FIT(XYNBS, IDEAL, PREC_FP32, 8, 1)
GMLE_EXTERN_FIT(XYNBS, IDEAL, PREC_FP32, 11, 2)
GMLE_DEFINE_FINDER(XYNBS, IDEAL, PREC_FP32)
