// The fp16 instantiations of the kernels of grouped_gemm.hip, beside the bf16 ones instead of behind them: either takes the compiler minutes.
#define XMA_GROUPED_GEMM_F16
#include "grouped_gemm.hip"
