// The fp16 kernels of wol_linear_gemm.hip, compiled as a translation unit of
// their own (the bf16 and fp16 instantiations take about the same time, and
// together they were the longest step of the build).
#define WOL_GEMM_F16_UNIT
#define WOL_GEMM_DTYPE WOL_DTYPE_F16
#include "wol_linear_gemm.hip"
