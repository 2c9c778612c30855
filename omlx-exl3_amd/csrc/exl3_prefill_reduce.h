// SPDX-License-Identifier: Apache-2.0
// Second launch of the prefill forms that split k over workgroups (exl3_prefill_mm.hip, exl3_prefill_rows.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace exl3 {

// Most bytes of split sums an automatic plan asks a caller for: well below one window of reconstructed weights, so that a
// prefill call's transient memory keeps the bound the windows set.
constexpr size_t kPrefillWorkspaceLimit = (size_t)128 << 20;

// y[r, c] = (H128 of the sum over s of partials[s, r, c], in split order) / sqrt(128) * svh (+ bias) per 128-column
// block, into rows x n of out_dtype with row stride ldy (defined in exl3_prefill_mm.hip).
void launch_prefill_reduce(const float* partials, int S, int rows, int n, const uint16_t* svh, const void* bias,
                           void* y, int ldy, int out_dtype, hipStream_t st);

}  // namespace exl3
