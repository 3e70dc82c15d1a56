// The matrix kernels with freely shaped tiles, of operands contiguous along one index.
#include "pam_gemm_kernel.h"

void pamgemm::launch_free(int lk, int rk, unsigned groups, hipStream_t st, const GemmArgs& g)
{
#define PAM_GEMM_CASE(LK, RK) \
    if (lk == LK && rk == RK) { hipLaunchKernelGGL((gemm_kernel<4 * kFreeFoursM, 4 * kFreeFoursN, 4, 4, 16, MODE_PAM, LK, RK, false, true>), dim3(groups), dim3(256), 0, st, g); return; }
    PAM_GEMM_CASE(LOAD_KODD, LOAD_KODD) PAM_GEMM_CASE(LOAD_KODD, LOAD_RODD) PAM_GEMM_CASE(LOAD_RODD, LOAD_KODD) PAM_GEMM_CASE(LOAD_RODD, LOAD_RODD)
#undef PAM_GEMM_CASE
}
