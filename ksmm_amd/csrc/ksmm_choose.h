// Price of a kernel instance on a problem, and the cheapest one (ksmm_choose.hip).  Host only.
#pragma once
#include "ksmm_common.h"

namespace ksmm {

struct Choice {
    int algo, variant;  // KSMM_ALGO_AUTO: none
    float us;           // predicted microseconds
};

// predicted time of the instance `t` describes (as a family reported it), < 0 when it has no price
float predicted_us(const Problem &p, const ksmm_tile &t);
// the cheapest instance that takes the problem as it is; any_alignment: of the split-K kernel and the whole-d tiles, which
// need no aligned pointers
Choice cheapest_instance(const Problem &p, bool any_alignment);
// predicted time of one transposing or re-pitching copy of `rows` rows
float copy_us(int64_t rows, int64_t cols_in, int64_t cols_out, int elem_bytes, bool transpose);

}  // namespace ksmm
