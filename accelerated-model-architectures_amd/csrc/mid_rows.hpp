// Grouped GEMMs of 128 x 256 tiles (mid_rows.hip): argument checks are the callers'.
#pragma once

#include "gemm_common.hpp"

// Rows per expert on average beyond which the few-row entry point takes the forward-type kernels (measured in few_rows.hip).
constexpr int MID_ROWS_FWD_FROM = 24;

namespace xma_rocm {

// whether the kernels have the variant, and whether they can address the operands as well
bool mid_fwd_has(int64_t M, int32_t E, int w_is_kn, int epilogue);
bool mid_fwd_takes(const FwdArgs &a, int w_is_kn, int epilogue);
bool mid_dw_takes(const DwArgs &a, int64_t M);
// whether dW is shorter with 128 x 256 tiles than with the small ones of the few-row entry point
bool mid_dw_leads(const DwArgs &a, int64_t M);
// whether a forward-type launch beyond the few-row regime is shorter with 128 x 256 than with 256 x 256 tiles, as far as its sizes tell
bool mid_fwd_leads(int64_t M, int32_t N, int32_t K, int32_t E, int epilogue);
// fp32 sums of the K ranges of a launch with few tiles; 0: not cut
size_t mid_fwd_workspace_bytes(int64_t M, int32_t N, int32_t K, int32_t E);
int mid_fwd(const FwdArgs &a, int w_is_kn, int epilogue, int dtype, float *part, hipStream_t st);
int mid_dw(const DwArgs &a, int dtype, hipStream_t st);

} // namespace xma_rocm

// few_rows.hip: adds the S parts part[S][M][N] in order and applies bias, scale and the epilogue of `a`
int split_sums_epilogue(const FwdArgs &a, const float *part, int S, int epilogue, int dtype, hipStream_t st);
