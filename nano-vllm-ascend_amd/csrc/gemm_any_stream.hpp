// Which products over fp32 activations and bf16 weights gemm_any_stream_kernel takes (gemm_any.hip), where x and w lie on 16 bytes;
// gemm_any_tile.hip asks it.  n_groups: 0, or the groups that `rows` rows lie in;
// dual: two weights (without groups).
#pragma once
#include "mi_common.hpp"

namespace mi {
bool any_stream_takes(int rows, int N, int K, int n_groups, bool dual);
}  // namespace mi
