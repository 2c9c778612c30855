// SPDX-License-Identifier: Apache-2.0
// Prefill contraction for short prompts, prompt chunks and decode batches: y = had128(xh @ W_inner) * svh (+ bias)
// for a few to several hundred rows, each weight decoded from the trellis straight into the MFMA operand registers
// that multiply it (replaces decode_wt + matmul + hadamard_transform + svh, reference src/omlx/exl3/linear.py:97-105,
// where the reconstruction of the weights would cost more than the product).
//
// What bounds it: per 32 x 64 weights a wavefront spends ~140 VALU instructions on the decode (as the GEMV does) and
// 4 MFMAs per 16 rows, and the two add up rather than overlap (measured with the MFMAs interleaved into the decode
// instruction by instruction, and with the two wavefronts of a SIMD held in opposite phases: both slower). So one
// decode serves as many rows as the accumulators hold: 16 RT rows, RT up to 16, 8 RT accumulator registers.
//
// Workgroup = 4 wavefronts, a 128-column block x 16 RT rows x a k-range (split). Wavefront w owns n-tiles 2w, 2w + 1
// of the block; k advances 64 per step. Lane 16q + c decodes run c % 8 of n-tile 2w + c / 8 for k-tile 4 it + q, which
// leaves the B operands of v_mfma_f32_16x16x32_f16 in its registers (the GEMV's layout, exl3_gemv.hip). The step's
// activations (16 RT rows x 64 k) are shared by the four wavefronts through LDS: two stages, filled by buffer loads
// with an LDS destination one step ahead, one barrier per step; two trellis sets are in flight per lane.
// Several splits: raw fp32 sums to a caller workspace and a second launch that adds them in split order and applies
// the epilogue (exl3_prefill_reduce.h). One split: the epilogue in this launch.
//
// Measured (MI355X, K = 6, whole calls without the input rotation) against reconstruction + GEMM: 5120 -> 17408 at
// 9 / 33 / 96 / 256 / 512 rows 21 / 26 / 36 / 68 / 115 us against 75 / 77 / 78 / 99 / 136; 17408 -> 5120 22 / 26 /
// 34 / 65 / 111 against 75 / 76 / 81 / 110 / 151; 4096 -> 4096 at K = 4 10 / 13 / 18 / 25 / 36 against 28 / 25 / 26 /
// 38 / 41. Not kept: 32x32x16 MFMAs on 64 columns per wavefront with two or four k-groups added in LDS (half the
// LDS reads; level up to 64 rows, 5-15% slower above).
#pragma once

#include "exl3_device.h"
#include "exl3_gemv_common.h"
#include "exl3_prefill_rows.h"

namespace exl3 {

constexpr int kRowsWaves = 4;          // wavefronts per workgroup, 32 columns each
// s_waitcnt immediate of gfx9: vmcnt in bits 3:0 and 15:14, expcnt 6:4 (not waited for), lgkmcnt 11:8
constexpr int rows_waitcnt(int vm, int lgkm) {
  return (vm & 15) | ((vm >> 4) & 3) << 14 | 7 << 4 | (lgkm & 15) << 8;
}

// 16-byte slots of one activation stage: 16 RT rows x 64 k, and room for a 16 x 128 fp32 tile of the epilogue
constexpr int rows_stage_slots(int rt) { return rt < 4 ? 512 : rt * 128; }

template <int OT>
__device__ __forceinline__ void rows_store(const RowsArgs& a, const float (&e)[8], const float (&sv)[8],
                                           const float (&bs)[8], int gr, int c0) {
  float o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    o[i] = round_through<OT>(e[i] * kHadScale * sv[i]);
    if (a.bias) o[i] = round_through<OT>(o[i] + bs[i]);
  }
  store8<OT>(a.y, (size_t)gr * a.n + c0, o);
}

// Output rotation, svh, bias and rounding of the workgroup's 16 RT x 128 sums (one split): the tiles go through
// LDS, as many at a time as the stages hold, to rows of 16 lanes with 8 consecutive columns each, where the
// arithmetic is the reduction launch's. Column chunks of 4 are placed at chunk ^ (2 (R >> 2 & 1) + 8 (R >> 3)) in row R,
// so that the four rows a wavefront writes at once sit on different banks.
template <int RT>
__device__ __forceinline__ void rows_epilogue(const RowsArgs& a, u32x4* sA0, u32x4* sA1, const f32x4 (&lo)[RT],
                                              const f32x4 (&hi)[RT], int row0) {
  constexpr int kPer = rows_stage_slots(RT) / 512, kTiles = 2 * kPer;   // tiles per stage, per round
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int q = lane >> 4, c = lane & 15;
  const int col = wave * 32 + (c >> 3) * 16 + (c & 7);
  auto place = [](int R) { return 2 * (R >> 2 & 1) + 8 * (R >> 3); };
  auto tile = [&](int t) { return reinterpret_cast<float*>(t < kPer ? sA0 + 512 * t : sA1 + 512 * (t - kPer)); };
  const int wlo = ((col >> 2) ^ place(4 * q)) * 4 + (col & 3), whi = (((col + 8) >> 2) ^ place(4 * q)) * 4 + (col & 3);
  const int R = wave * 4 + q, c0 = blockIdx.x * 128 + 8 * c;
  float sv[8], bs[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 8; ++i) sv[i] = f16_to_f32(a.svh[c0 + i]);
  if (a.bias) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      bs[i] = a.out_dtype == kF16    ? load_as_f32<kF16>(a.bias, c0 + i)
              : a.out_dtype == kBF16 ? load_as_f32<kBF16>(a.bias, c0 + i)
                                     : load_as_f32<kF32>(a.bias, c0 + i);
  }
  static_for<0, (RT + kTiles - 1) / kTiles>([&](auto G) {
    constexpr int g0 = decltype(G)::value * kTiles;
    constexpr int nt = RT - g0 < kTiles ? RT - g0 : kTiles;
    __syncthreads();
    static_for<0, nt>([&](auto T) {
      constexpr int t = decltype(T)::value;
      float* d = tile(t);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        d[(4 * q + r) * 128 + wlo] = lo[g0 + t][r];
        d[(4 * q + r) * 128 + whi] = hi[g0 + t][r];
      }
    });
    __syncthreads();
#pragma unroll 2
    for (int t = 0; t < nt; ++t) {
      const f32x4* d = reinterpret_cast<const f32x4*>(tile(t)) + R * 32;
      const f32x4 u = d[(2 * c) ^ place(R)], v = d[(2 * c + 1) ^ place(R)];
      float e[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
      fwht128_lane8(e, lane);
      const int gr = row0 + 16 * (g0 + t) + R;
      if (gr < a.rows) {
        if (a.out_dtype == kF16) rows_store<kF16>(a, e, sv, bs, gr, c0);
        else if (a.out_dtype == kBF16) rows_store<kBF16>(a, e, sv, bs, gr, c0);
        else rows_store<kF32>(a, e, sv, bs, gr, c0);
      }
    }
  });
}

template <int K, int CB, int RT>
__device__ __forceinline__ void rows_body(const RowsArgs& a, u32x4* sA0, u32x4* sA1) {
  constexpr int TW = 8 * K;
  constexpr int kTrLoads = K / 4 + (K % 4 != 0) + 1;   // buffer loads of one trellis set (load_run)
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int blk = blockIdx.x, s = blockIdx.y, row0 = blockIdx.z * (16 * RT);
  const int kt0 = s * a.kt_per_split;
  const int nkt = min(a.KT - kt0, a.kt_per_split);   // a multiple of 4
  const int iters = nkt >> 2;

  // ---- trellis: lane (q, c) of iteration it decodes run c % 8 of n-tile 2 wave + c / 8, k-tile kt0 + 4 it + q ----
  const int q = lane >> 4, c = lane & 15, g = c & 7;
  const uint32_t kstride = (uint32_t)a.NT * TW;
  const int nt = blk * 8 + wave * 2 + (c >> 3);
  const uint32_t split_bytes = (uint32_t)nkt * kstride * 4u;
  char* const tr_split = reinterpret_cast<char*>(const_cast<uint32_t*>(a.tr + (size_t)kt0 * kstride));
  const uint32_t vo_t = ((uint32_t)q * kstride + (uint32_t)nt * TW + K * g) * 4u;
  const uint32_t vo_wp = ((uint32_t)q * kstride + (uint32_t)nt * TW + (K * g + TW - 1) % TW) * 4u;
  const uint32_t step_t = 16u * kstride;
  auto issue_T = [&](Stage<K>& st, int it) {
    const uint32_t adv = (uint32_t)it * step_t;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        tr_split + adv, (short)0, max((int)split_bytes - (int)adv, 0), kBufferFlags);
    load_run<K>(rs, vo_t, vo_wp, 0u, st.w, st.wp);
  };

  // ---- activations: a stage holds 16 RT rows of eight 16-byte pieces (piece p: k 8p .. 8p + 7 of the step) ----
  // Piece 2q + h is what lane (q, c) multiplies first (h = 0) or second (h = 1); it sits at position (4h + q) ^ (row & 7)
  // of its row, which makes the fragment reads (16 rows x one h, four q) free of bank conflicts. Lane L of load i fills
  // slot 64 i + L: row 8 i + L / 8, position L % 8. Rows past the batch get offset 2^31, past any descriptor: zeros. The
  // step is the loads' scalar offset; a step past the split loads its last one again, into a stage that nothing reads.
  const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.xh), (short)0, (int)((uint32_t)a.rows * (uint32_t)a.k * 2u), kBufferFlags);
  constexpr int kLoads = (2 * RT + kRowsWaves - 1) / kRowsWaves;
  const int lr = lane >> 3, lpos = (lane & 7) ^ lr;
  const int piece = 2 * (lpos & 3) + (lpos >> 2);
  uint32_t oa[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const int r = row0 + (wave + kRowsWaves * j) * 8 + lr;
    oa[j] = r < a.rows ? ((uint32_t)r * (uint32_t)a.k + (uint32_t)(kt0 * 16 + piece * 8)) * 2u : 0x80000000u;
  }
  auto issue_A = [&](int it, u32x4* st) {
    const uint32_t so = (uint32_t)it * 128u;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      if (2 * RT % kRowsWaves == 0 || wave + kRowsWaves * j < 2 * RT) {
        u32x4* dst = st + (wave + kRowsWaves * j) * 64;
        uint32_t vo = oa[j];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_x, dst, 16, vo, so, 0, 0);
      }
    }
  };
  auto frag = [&](const u32x4* st, int i, int h) { return st[(16 * i + c) * 8 + ((4 * h + q) ^ (c & 7))]; };

  f32x4 lo[RT], hi[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) lo[i] = hi[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Step it: wait until its activations are in LDS (every load but the newest trellis set, which is younger) and every
  // wavefront is done with the other stage, refill that one, decode this step's trellis set and reload it for step
  // it + 2, multiply. The activation fragments are read two row tiles ahead of their MFMAs. (Scheduling barriers every
  // four decoded registers: without them the scheduler interleaves all sixteen chains and spills at RT = 8.)
  auto step = [&](int it, Stage<K>& st, const u32x4* cur, u32x4* next) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(rows_waitcnt(kTrLoads, 0));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    __builtin_amdgcn_sched_barrier(0);
    issue_A(min(it + 1, iters - 1), next);
    constexpr int kRing = RT < 3 ? RT : 3;
    u32x4 X[kRing][2];
    static_for<0, kRing - (RT >= 3)>([&](auto I) {
      constexpr int i = decltype(I)::value;
      X[i][0] = frag(cur, i, 0);
      X[i][1] = frag(cur, i, 1);
    });
    uint32_t b[16];
    static_for<0, 16>([&](auto P) {
      constexpr int p = decltype(P)::value;
      b[p] = decode_pair<K, CB, p>(st.w, st.wp, kXor3);
      if constexpr (p % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    });
    const u32x4 l0 = mfma_src(b[0], b[4], b[8], b[12]), h0 = mfma_src(b[2], b[6], b[10], b[14]);
    const u32x4 l1 = mfma_src(b[1], b[5], b[9], b[13]), h1 = mfma_src(b[3], b[7], b[11], b[15]);
    issue_T(st, it + 2);
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, RT>([&](auto I) {
      constexpr int i = decltype(I)::value;
      if constexpr (RT >= 3 && i + 2 < RT) {
        X[(i + 2) % 3][0] = frag(cur, i + 2, 0);
        X[(i + 2) % 3][1] = frag(cur, i + 2, 1);
      }
      const f16x8 x0 = as_f16x8(X[i % kRing][0]), x1 = as_f16x8(X[i % kRing][1]);
      lo[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x0, as_f16x8(l0), lo[i], 0, 0, 0);
      hi[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x0, as_f16x8(h0), hi[i], 0, 0, 0);
      lo[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x1, as_f16x8(l1), lo[i], 0, 0, 0);
      hi[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x1, as_f16x8(h1), hi[i], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  Stage<K> t0, t1;
  issue_A(0, sA0);
  __builtin_amdgcn_sched_barrier(0);
  issue_T(t0, 0);
  __builtin_amdgcn_sched_barrier(0);
  issue_T(t1, 1);
  __builtin_amdgcn_sched_barrier(0);
  int it = 0;
  for (; it + 2 <= iters; it += 2) {
    step(it, t0, sA0, sA1);
    step(it + 1, t1, sA1, sA0);
  }
  if (it < iters) step(it, t0, sA0, sA1);
  // no load is left in flight (the builtin: the compiler then knows it, and the stores below wait for nothing)
  __builtin_amdgcn_s_waitcnt(rows_waitcnt(0, 15));

  if (gridDim.y == 1) {
    rows_epilogue<RT>(a, sA0, sA1, lo, hi, row0);
    return;
  }
  // rows past the batch lie past the descriptor: their stores are dropped
  const uint32_t pbytes = (uint32_t)a.rows * (uint32_t)a.n * 4u;
  const __amdgpu_buffer_rsrc_t rs_p = __builtin_amdgcn_make_buffer_rsrc(
      a.partials + (size_t)s * a.rows * a.n, (short)0, (int)pbytes, kBufferFlags);
  const uint32_t col = (uint32_t)(blk * 128 + wave * 32 + (c >> 3) * 16 + g);
  static_for<0, RT>([&](auto I) {
    constexpr int i = decltype(I)::value;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t off = ((uint32_t)(row0 + 16 * i + 4 * q + r) * (uint32_t)a.n + col) * 4u;
      const float vl = lo[i][r], vh = hi[i][r];
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, vl), rs_p, off, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, vh), rs_p, off + 32u, 0, 0);
    }
  });
}

// one kernel per number of 16-row tiles, compiled for as many wavefronts per SIMD as its registers allow (RT = 12 at K = 8
// needs 178, 10 more than three leave: spilled, it took 15-20% longer than reconstruction + GEMM): the LDS stages' size is spelled out (an LDS array whose size depends on a
// template parameter makes hipcc drop the kernel's host stub when the buffer-to-LDS load builtin writes into it)
#define EXL3_ROWS_KERNEL(RT, WPE, SLOTS)                                                                         \
  template <int K, int CB>                                                                                       \
  __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE))) void prefill_rows##RT##_kernel(    \
      RowsArgs a) {                                                                                              \
    __shared__ u32x4 sA0[SLOTS], sA1[SLOTS];                                                                     \
    static_assert(SLOTS == rows_stage_slots(RT), "LDS stage");                                                   \
    rows_body<K, CB, RT>(a, sA0, sA1);                                                                           \
  }
EXL3_ROWS_KERNEL(1, 4, 512)
EXL3_ROWS_KERNEL(2, 4, 512)
EXL3_ROWS_KERNEL(3, 4, 512)
EXL3_ROWS_KERNEL(4, 4, 512)
EXL3_ROWS_KERNEL(6, 4, 768)
EXL3_ROWS_KERNEL(8, 3, 1024)
EXL3_ROWS_KERNEL(12, (K == 8 ? 2 : 3), 1536)
EXL3_ROWS_KERNEL(16, 2, 2048)
#undef EXL3_ROWS_KERNEL

template <int K, int CB>
static void launch_rows(int rt, const dim3& grid, const RowsArgs& a, hipStream_t st) {
  switch (rt) {
    case 1: prefill_rows1_kernel<K, CB><<<grid, 256, 0, st>>>(a); break;
    case 2: prefill_rows2_kernel<K, CB><<<grid, 256, 0, st>>>(a); break;
    case 3: prefill_rows3_kernel<K, CB><<<grid, 256, 0, st>>>(a); break;
    case 4: prefill_rows4_kernel<K, CB><<<grid, 256, 0, st>>>(a); break;
    case 6: prefill_rows6_kernel<K, CB><<<grid, 256, 0, st>>>(a); break;
    case 8: prefill_rows8_kernel<K, CB><<<grid, 256, 0, st>>>(a); break;
    case 12: prefill_rows12_kernel<K, CB><<<grid, 256, 0, st>>>(a); break;
    default: prefill_rows16_kernel<K, CB><<<grid, 256, 0, st>>>(a); break;
  }
}

template <int CB>
static void launch_rows_k(int K, int rt, const dim3& grid, const RowsArgs& a, hipStream_t st) {
  switch (K) {
    case 1: launch_rows<1, CB>(rt, grid, a, st); break;
    case 2: launch_rows<2, CB>(rt, grid, a, st); break;
    case 3: launch_rows<3, CB>(rt, grid, a, st); break;
    case 4: launch_rows<4, CB>(rt, grid, a, st); break;
    case 5: launch_rows<5, CB>(rt, grid, a, st); break;
    case 6: launch_rows<6, CB>(rt, grid, a, st); break;
    case 7: launch_rows<7, CB>(rt, grid, a, st); break;
    default: launch_rows<8, CB>(rt, grid, a, st); break;
  }
}

}  // namespace exl3
