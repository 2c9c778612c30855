// SPDX-License-Identifier: Apache-2.0
// Few-row prefill kernels of the 3INST codebook.
#include "exl3_prefill_rows_body.h"

namespace exl3 {

void rows_launch_cb0(int K, int rt, const dim3& grid, const RowsArgs& a, hipStream_t st) {
  launch_rows_k<0>(K, rt, grid, a, st);
}

}  // namespace exl3
