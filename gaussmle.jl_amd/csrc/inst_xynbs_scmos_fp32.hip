// Kernel specialisations for model XYNBS, camera SCMOS, precision FP32.
#include "gmle_instances.hpp"
// 16 px on 4 lanes is built in inst_sched_occ.hip.
GMLE_EXTERN_FIT(XYNBS, SCMOS, PREC_FP32, 16, 4)
GMLE_DEFINE_FINDER(XYNBS, SCMOS, PREC_FP32)
