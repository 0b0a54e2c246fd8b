// Weight gradients of batch-size-first fp16 blocks of 48 and more (ksmm_wgrad_wide.hip)
#pragma once
#include "ksmm_common.h"

namespace ksmm {

// fp32 elements of partial sums (0: one slice, written as it is; < 0: not taken)
int64_t wgrad_wide_partial_floats(int64_t batch, int a, int b, int c, int d, int dtype);
// As wgrad_bf_run; KSMM_ERR_BAD_ALGO: not taken (sizes, or tensors off the 16-byte vector)
int wgrad_wide_run(const void *dy, const void *x, void *dw, float *acc, int64_t batch, int a, int b, int c, int d, int dtype, float scale,
                   hipStream_t stream, int *splits);

}  // namespace ksmm
