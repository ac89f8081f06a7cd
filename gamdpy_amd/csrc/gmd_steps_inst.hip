// gmd_steps_inst.hip -- one group of step kernels, compiled apart from
// gmd_core.hip (which declares them extern) so the groups build in parallel:
//   GMD_INST_BASE=b GMD_INST_CUT=c   pair-function base b with cutoff wrapper c,
//                                    every integrator but NPT_Atomic
//   GMD_INST_BASE=b GMD_INST_NPT     base b with every wrapper, NPT_Atomic
// Bases: 0 LJ sigma/epsilon, 1 LJ 12-6, 2 the inline family (IPL_n, LJ_m_n,
// harmonic_repulsion, hertzian), 3 functions read from parameter rows (SAAP
// and sums of two terms).
#include <hip/hip_runtime.h>

#include "gamdpy_amd.h"
#include "gmd_steps.h"

#ifdef GMD_INST_NPT
GMD_STEP_KERNELS_NPT(, GMD_INST_BASE)
#else
GMD_STEP_KERNELS_CUT(, GMD_INST_BASE, GMD_INST_CUT)
#endif
