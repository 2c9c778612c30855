// SPDX-License-Identifier: Apache-2.0
// Arguments and per-codebook launchers of the few-row prefill (exl3_prefill_rows.hip). Each codebook's kernels compile
// in a file of their own, side by side.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace exl3 {

struct RowsArgs {
  const uint16_t* xh;      // (rows, k) fp16
  const uint32_t* tr;
  float* partials;         // (S, rows, n) fp32
  int k, KT, NT, rows, n, kt_per_split;
  // one split: the epilogue runs in this launch (partials unused)
  const uint16_t* svh;
  const void* bias;
  void* y;
  int out_dtype;
};

// The kernel of rt 16-row tiles (1, 2, 3, 4, 6, 8, 12, 16) at K bits per weight, codebook 0, 1, 2.
void rows_launch_cb0(int K, int rt, const dim3& grid, const RowsArgs& a, hipStream_t st);
void rows_launch_cb1(int K, int rt, const dim3& grid, const RowsArgs& a, hipStream_t st);
void rows_launch_cb2(int K, int rt, const dim3& grid, const RowsArgs& a, hipStream_t st);

}  // namespace exl3
