// Two factors in one launch (ksmm_pair.hip)
#pragma once
#include "ksmm_common.h"

namespace ksmm {

struct PairShape {
    int nt, mg;  // a workgroup's batch columns / 16 and outputs of a block of the second factor / 64
};
// (of a chain that check_chain() has passed)
float pair_us(const ksmm_factor_desc *f, int n, int64_t batch, int x_dtype, int y_dtype, int bs_last, PairShape *best);
int pair_run(const ksmm_factor_desc *f, int n, const void *x, void *y, int64_t batch, int x_dtype, int y_dtype, int bs_last,
             const PairShape &shape, hipStream_t stream, const ksmm_epilogue *ep, const float *x_scale = nullptr);

}  // namespace ksmm
