// The fp16 kernels of wol_linear_wide.hip, compiled as a translation unit of their own.
#define WOL_GEMM_F16_UNIT
#define WOL_GEMM_DTYPE WOL_DTYPE_F16
#include "wol_linear_wide.hip"
