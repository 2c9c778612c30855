// SPDX-License-Identifier: Apache-2.0
// Entry point and launch plan of the few-row prefill; the kernels and what bounds them: exl3_prefill_rows_body.h.
#include "exl3_prefill_rows.h"

#include <algorithm>

#include "exl3_capi_common.h"
#include "exl3_device.h"
#include "exl3_prefill_reduce.h"

namespace exl3 {

// Launch plan, from rows, k, n and K only: row blocks of up to 256 rows (16 RT), and S splits of k. The time of a plan is
// estimated from what was measured at 7 shapes (k 1,024-17,408, n 1,024-17,408) x 15 row counts x up to 13 splits: a
// 64-k step of a workgroup costs 0.195 + 0.0355 RT us when others share its CU, at least 0.21 + 0.055 RT alone (latency),
// two to four workgroups fit a CU, ~6.3 us are fixed, and the splits' sums are written and read once at ~6.4 TB/s
// plus a second launch. Over 500 other shapes (150-1,100 rows, 2-8 bits) the pick's S is 0.7% behind the best measured one
// on average, 49 of them more than 3% (14% at most). Automatic plans split while the sums stay within
// kPrefillWorkspaceLimit (a wide head has column blocks enough: 92 rows of 17408 -> 151936 took 160 MiB of sums, 246 rows
// 428 MiB).
struct RowsPlan {
  int rt, row_blocks, splits, kt_per_split;
};

static int rows_rt(int rows) {   // the smallest built tile count that holds the rows
  const int tiles = (rows + 15) / 16;
  return tiles <= 4 ? tiles : tiles <= 6 ? 6 : tiles <= 8 ? 8 : tiles <= 12 ? 12 : 16;
}

static double rows_cost(int K, int rt, long groups, int steps_per_split, int splits, double out_bytes) {
  const int resident = rt <= 6 ? 4 : rt <= 8 || (rt <= 12 && K < 8) ? 3 : 2;   // workgroups a CU holds (registers)
  const long per_cu = (groups * splits + 255) / 256;
  const double shared = 0.195 + 0.0355 * rt, alone = 0.21 + 0.055 * rt;
  auto round_us = [&](long g) { return g * shared > alone ? g * shared : alone; };
  double us = 6.3 + (double)(per_cu / resident) * steps_per_split * round_us(resident);
  if (per_cu % resident) us += steps_per_split * round_us(per_cu % resident);
  return us + (splits > 1 ? 1.9 + 0.1 * splits + (2 * splits + 0.5) * out_bytes / 6.4e6 : 0.13 * rt);
}

static RowsPlan rows_plan(int rows, int k, int n, int K, int splits) {
  constexpr int kMaxSplits = 16, kMaxRowsPerBlock = 256;
  const int steps = k / 64, z0 = (rows + kMaxRowsPerBlock - 1) / kMaxRowsPerBlock;
  RowsPlan best{};
  double best_us = -1.0;
  for (int z = z0; z < z0 + 3; ++z) {
    const int rt = rows_rt((rows + z - 1) / z);
    if (z > z0 && rt < 4) break;   // (smaller tiles decode more often than they spread the work)
    if ((rows + 16 * rt - 1) / (16 * rt) != z) continue;   // the same row blocks as a smaller z
    // (a step per split at most; steps + S - 1 below stays in range for any `splits`)
    const int s_lo = splits > 0 ? std::min(splits, steps) : 1, s_hi = splits > 0 ? s_lo : kMaxSplits;
    for (int S = s_lo; S <= s_hi; ++S) {
      const int per = (steps + S - 1) / S;
      if (splits <= 0 && S > 1 &&
          (per < 3 || (size_t)S * (size_t)rows * (size_t)n * sizeof(float) > kPrefillWorkspaceLimit))
        break;
      const int real = (steps + per - 1) / per;   // no empty split
      const double us = rows_cost(K, rt, (long)(n / 128) * z, per, real, (double)rows * n * 4.0);
      if (best_us < 0 || us < best_us) {
        best = RowsPlan{rt, z, real, 4 * per};
        best_us = us;
      }
    }
  }
  return best;
}

static size_t rows_workspace(const RowsPlan& p, int rows, int n) {
  return p.splits > 1 ? (size_t)p.splits * (size_t)rows * (size_t)n * sizeof(float) : 0;
}

}  // namespace exl3

using namespace exl3;

// 32-bit byte offsets: activations, one split's sums, and a split's trellis with the two look-ahead steps
static bool rows_fits(int rows, int k, int n, int K) {
  return (uint64_t)rows * (uint64_t)k * 2u < (1ull << 31) && (uint64_t)rows * (uint64_t)n * 4u < (1ull << 31) &&
         (uint64_t)(k + 128) * (uint64_t)n * (uint64_t)K / 8u < (1ull << 31) && n / 128 < (1 << 24);
}

static bool rows_shape_ok(int rows, int k, int n, int K) {
  return rows >= 1 && k >= 64 && k % 64 == 0 && n >= 128 && n % 128 == 0 && K >= 1 && K <= 8;
}

extern "C" size_t exl3_prefill_rows_workspace_bytes(int rows, int k, int n, int K, int splits) {
  if (!rows_shape_ok(rows, k, n, K) || !rows_fits(rows, k, n, K) || rows > 65535) return 0;
  return rows_workspace(rows_plan(rows, k, n, K, splits), rows, n);
}

extern "C" int exl3_prefill_rows(const uint16_t* xh, const uint32_t* trellis, int k, int n, int K, int cb,
                                 const uint16_t* svh, const void* bias, void* y, int out_dtype, int rows, int splits,
                                 void* workspace, size_t workspace_bytes, void* stream) {
  EXL3_REQUIRE(xh && trellis && svh && y, EXL3_ERR_ARG, "exl3_prefill_rows: NULL pointer argument");
  EXL3_REQUIRE(k > 0 && k % 64 == 0, EXL3_ERR_ARG, "exl3_prefill_rows: k must be a positive multiple of 64 (got %d)", k);
  EXL3_REQUIRE(n > 0 && n % 128 == 0, EXL3_ERR_ARG, "exl3_prefill_rows: n must be a positive multiple of 128 (got %d)",
               n);
  EXL3_REQUIRE(K >= 1 && K <= 8, EXL3_ERR_ARG, "exl3_prefill_rows: K must be 1..8 (got %d)", K);
  EXL3_REQUIRE(cb >= 0 && cb <= 2, EXL3_ERR_ARG, "exl3_prefill_rows: codebook must be 0, 1 or 2 (got %d)", cb);
  EXL3_REQUIRE(rows >= 1 && rows <= 65535, EXL3_ERR_ARG, "exl3_prefill_rows: rows must be 1..65535 (got %d)", rows);
  EXL3_REQUIRE(out_dtype >= 0 && out_dtype <= 2, EXL3_ERR_ARG, "exl3_prefill_rows: bad out_dtype %d", out_dtype);
  EXL3_REQUIRE(aligned(xh, 16) && aligned(trellis, 4) && aligned(y, 16), EXL3_ERR_ARG,
               "exl3_prefill_rows: xh and y must be 16-byte and trellis 4-byte aligned");
  EXL3_REQUIRE(rows_fits(rows, k, n, K), EXL3_ERR_ARG,
               "exl3_prefill_rows: activations, a split's sums or the trellis exceed 2 GiB");
  const RowsPlan p = rows_plan(rows, k, n, K, splits);
  EXL3_REQUIRE(p.splits >= 1 && (p.splits - 1) * p.kt_per_split < k / 16, EXL3_ERR_ARG,
               "exl3_prefill_rows: %d splits leave an empty split", p.splits);
  const size_t need = rows_workspace(p, rows, n);
  EXL3_REQUIRE(need == 0 || (workspace && workspace_bytes >= need && aligned(workspace, 16)), EXL3_ERR_WORKSPACE,
               "exl3_prefill_rows: this shape splits k over %d workgroups and needs a 16-byte aligned workspace of %zu "
               "bytes (exl3_prefill_rows_workspace_bytes), got %zu", p.splits, need, workspace_bytes);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const RowsArgs a{xh, trellis, static_cast<float*>(workspace), k, k / 16, n / 16, rows, n, p.kt_per_split, svh, bias,
                   y, out_dtype};
  const dim3 grid((unsigned)(n / 128), (unsigned)p.splits, (unsigned)p.row_blocks);
  if (cb == 0) rows_launch_cb0(K, p.rt, grid, a, st);
  else if (cb == 1) rows_launch_cb1(K, p.rt, grid, a, st);
  else rows_launch_cb2(K, p.rt, grid, a, st);
  if (p.splits > 1) launch_prefill_reduce(a.partials, p.splits, rows, n, svh, bias, y, n, out_dtype, st);
  EXL3_LAUNCH_CHECK("exl3_prefill_rows");
  return EXL3_OK;
}
