// SPDX-License-Identifier: Apache-2.0
// Decode attention that produces o_proj's rotated input, for batch-1 decode with a static KV cache.
//
// The reference fuses each EXL3 linear's input rotation into the kernel that produces that input (RMSNorm ->
// q/k/v and gate/up, SwiGLU -> down_proj; src/omlx/exl3/fusion.py:4-18) and leaves o_proj to rotate on its
// own. This kernel applies the same fusion to the attention output: one launch per layer does rotary
// position embedding of the new q and k, appends k and v to the caches, attends over positions 0..pos, and
// writes xh = fp16(H128(o * suh) / sqrt(128)) for o_proj (plus o itself when asked). A head's 128 output
// values are exactly one Hadamard block, so each workgroup rotates its own head.
//
// grid = n_heads workgroups of 1024 threads; workgroup h serves query head h of key/value head
// h / (n_heads / n_kv_heads). Thread t works on dimensions 8 (t % 16) .. 8 (t % 16) + 7 of position slot
// t / 16 (64 slots): scores and the weighted sum each read one 16-byte segment of a cache row per thread and
// position, with eight positions' loads in flight. Every workgroup of a kv head writes the new position's
// k and v rows itself (identical bytes) before reading the caches, so no workgroup depends on another's
// writes. The position is read from device memory, so a captured graph advances it without host work; a
// position outside [0, max_len) writes nothing and yields zeros.
#include <algorithm>

#include "exl3_capi_common.h"
#include "exl3_device.h"

namespace exl3 {

constexpr int kAttnHD = 128;
constexpr int kAttnMaxLen = 8192;
constexpr int kAttnThreads = 1024;
constexpr int kAttnSlots = kAttnThreads / 16;   // position slots
constexpr int kAttnUnroll = 8;

typedef _Float16 h2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float round_f16(float v) { return f16_to_f32(f32_to_f16(v)); }

__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }

// reduce over the 16 lanes of a dimension group (lanes 16a .. 16a + 15 of a wavefront)
__device__ __forceinline__ float sum16(float v) {
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o);
  return v;
}

__device__ __forceinline__ float block_reduce(float v, float* red, bool is_max) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float u = __shfl_xor(v, o);
    v = is_max ? fmaxf(v, u) : v + u;
  }
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int w = 1; w < kAttnThreads / 64; ++w) r = is_max ? fmaxf(r, red[w]) : r + red[w];
  return r;
}

// o (fp16) of a head and its rotation by one wavefront: 16 lanes x 8 consecutive values
__device__ __forceinline__ void write_head(const float* sfin, int h, int lane, const uint16_t* __restrict__ suh,
                                           uint16_t* __restrict__ o_out, uint16_t* __restrict__ xh) {
  const int e0 = 8 * (lane & 15);
  float e[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) e[i] = sfin[e0 + i];
  if (o_out && lane < 16) {
#pragma unroll
    for (int i = 0; i < 8; ++i) o_out[(size_t)h * kAttnHD + e0 + i] = f32_to_f16(e[i]);
  }
  if (xh) {
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = e[i] * f16_to_f32(suh[(size_t)h * kAttnHD + e0 + i]);
    fwht128_lane8(e, lane);
    if (lane < 16) {
#pragma unroll
      for (int i = 0; i < 8; ++i) xh[(size_t)h * kAttnHD + e0 + i] = f32_to_f16(e[i] * kHadScale);
    }
  }
}

__global__ __launch_bounds__(kAttnThreads) void attn_decode_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, uint16_t* kc,
    uint16_t* vc, const int64_t* __restrict__ pos_p, const float* __restrict__ rcos, const float* __restrict__ rsin,
    int n_heads, int n_kv, int max_len, float scale, const uint16_t* __restrict__ suh, uint16_t* __restrict__ o_out,
    uint16_t* __restrict__ xh) {
  extern __shared__ float sp[];                  // scores, then probabilities, positions 0..pos
  __shared__ float sq[kAttnHD], sk[kAttnHD], sv[kAttnHD], sfin[kAttnHD];
  __shared__ float so[kAttnSlots][kAttnHD];
  __shared__ float red[kAttnThreads / 64];
  const int h = blockIdx.x, grp = n_heads / n_kv, kh = h / grp;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int dg = tid & 15, slot = tid >> 4;
  const int64_t pos64 = *pos_p;
  const bool ok = pos64 >= 0 && pos64 < (int64_t)max_len;
  const int pos = ok ? (int)pos64 : 0;
  const int L = ok ? pos + 1 : 0;
  const size_t kv_row0 = (size_t)kh * max_len;

  // ---- rope of q (threads 0..63) and k (64..127), copy of v (128..255) ----
  if (tid < 128) {
    const int i = tid & 63;
    const uint16_t* src = tid < 64 ? q + (size_t)h * kAttnHD : k + (size_t)kh * kAttnHD;
    float* dst = tid < 64 ? sq : sk;
    const float c = rcos[(size_t)pos * (kAttnHD / 2) + i], s = rsin[(size_t)pos * (kAttnHD / 2) + i];
    const float a = f16_to_f32(src[i]), b = f16_to_f32(src[i + 64]);
    const float ac = a * c, bs = b * s, bc = b * c, as = a * s;
    dst[i] = round_f16(ac - bs);
    dst[i + 64] = round_f16(bc + as);
  } else if (tid < 256) {
    sv[tid - 128] = f16_to_f32(v[(size_t)kh * kAttnHD + (tid - 128)]);
  }
  __syncthreads();
  if (ok && tid < 256) {      // every workgroup of the kv head writes the same new rows
    if (tid < 128) kc[(kv_row0 + pos) * kAttnHD + tid] = f32_to_f16(sk[tid]);
    else vc[(kv_row0 + pos) * kAttnHD + (tid - 128)] = f32_to_f16(sv[tid - 128]);
  }
  // this thread's 8 query values as fp16 pairs
  uint32_t qp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    qp[i] = (uint32_t)f32_to_f16(sq[8 * dg + 2 * i]) | ((uint32_t)f32_to_f16(sq[8 * dg + 2 * i + 1]) << 16);
  __syncthreads();           // the new cache rows are visible to the whole workgroup

  // ---- scores ----
  const u32x4* krow = reinterpret_cast<const u32x4*>(kc + kv_row0 * kAttnHD) + dg;   // + 16 * j
  auto score = [&](const u32x4 w) {
    float d = __builtin_amdgcn_fdot2(as_h2(w.x), as_h2(qp[0]), 0.f, false);
    d = __builtin_amdgcn_fdot2(as_h2(w.y), as_h2(qp[1]), d, false);
    d = __builtin_amdgcn_fdot2(as_h2(w.z), as_h2(qp[2]), d, false);
    d = __builtin_amdgcn_fdot2(as_h2(w.w), as_h2(qp[3]), d, false);
    return sum16(d) * scale;
  };
  // batches of kAttnUnroll positions per slot, every batch's loads issued together (the last one predicated)
  constexpr int kBatch = kAttnUnroll * kAttnSlots;
  float lmax = -INFINITY;
  for (int j = slot; j < L; j += kBatch) {
    u32x4 w[kAttnUnroll];
#pragma unroll
    for (int u = 0; u < kAttnUnroll; ++u)
      if (j + u * kAttnSlots < L) w[u] = krow[(size_t)(j + u * kAttnSlots) * 16];
#pragma unroll
    for (int u = 0; u < kAttnUnroll; ++u) {
      if (j + u * kAttnSlots < L) {
        const float d = score(w[u]);
        if (dg == 0) sp[j + u * kAttnSlots] = d;
        lmax = fmaxf(lmax, d);
      }
    }
  }
  // the first batch of V rows, in flight during the softmax reductions
  const u32x4* vrow = reinterpret_cast<const u32x4*>(vc + kv_row0 * kAttnHD) + dg;
  u32x4 vw[kAttnUnroll];
#pragma unroll
  for (int u = 0; u < kAttnUnroll; ++u)
    if (slot + u * kAttnSlots < L) vw[u] = vrow[(size_t)(slot + u * kAttnSlots) * 16];
  const float gmax = block_reduce(lmax, red, true);
  float lsum = 0.f;
  for (int jj = tid; jj < L; jj += kAttnThreads) {
    const float e = expf(sp[jj] - gmax);
    sp[jj] = e;
    lsum += e;
  }
  const float gsum = block_reduce(lsum, red, false);     // (its barriers also publish sp)
  const float inv = L > 0 ? 1.0f / gsum : 0.f;

  // ---- o = sum_j p_j v_j over this slot's positions, dimensions 8 dg .. 8 dg + 7 ----
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto accum = [&](const u32x4 w, float p) {
    const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      acc[2 * t] += p * f16_to_f32((uint16_t)(ww[t] & 0xFFFFu));
      acc[2 * t + 1] += p * f16_to_f32((uint16_t)(ww[t] >> 16));
    }
  };
  for (int j = slot; j < L; j += kBatch) {
    if (j != slot) {
#pragma unroll
      for (int u = 0; u < kAttnUnroll; ++u)
        if (j + u * kAttnSlots < L) vw[u] = vrow[(size_t)(j + u * kAttnSlots) * 16];
    }
#pragma unroll
    for (int u = 0; u < kAttnUnroll; ++u)
      if (j + u * kAttnSlots < L) accum(vw[u], sp[j + u * kAttnSlots] * inv);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) so[slot][8 * dg + i] = acc[i];
  __syncthreads();
  if (tid < kAttnHD) {
    float o = 0.f;
    for (int sl = 0; sl < kAttnSlots; ++sl) o += so[sl][tid];
    sfin[tid] = round_f16(o);
  }
  __syncthreads();

  if (wave == 0) write_head(sfin, h, lane, suh, o_out, xh);
}

// ------------------------------------------------------------------------------------------------
// Split form for longer caches (a workspace given). The form above walks a head's positions on one CU (~8 ns each) and
// reads each key/value row once per query head; here a workgroup takes passes of 64 positions (pass j of workgroup s:
// positions 64 (j S + s) ..) of one key/value head for a group of its query heads, so a long context spreads over the
// chip, and the workgroups' results are merged: by the last one to arrive when arrival counters are given, else by a
// second launch. The launch is sized by max_len (known to the host), the position is read on the device: workgroups past
// it end at once, and while there are few positions (AttnSplitArgs::direct) the first workgroups of a head group take a
// head each with all its passes, write the outputs themselves, and nothing is merged. Bound by latency: the chain
// position -> rows and rotary operands -> scores -> softmax -> P V -> merge (4.8 us for one pass of one head), plus
// 0.85 us per further pass of one head, ~1.1 of three; issue-bound by then: rows loaded two passes ahead instead of one
// were level or slower (8,192 positions: 16.0 -> 16.5 us).
//   scores: v_mfma_f32_16x16x32_f16, A = the query heads (rows past them are never used), B = 16 cached rows as their
//     lanes load them from memory (lane 16q + c: row c, dimensions 32 s + 8 q ..), so keys pass through no LDS
//   softmax of the workgroup's positions in fp32, probabilities in LDS, P V on the VALU in fp32 (lane 16 q + c:
//     dimensions 8 c .. of row 4 i + q), added over slots and wavefronts
// A wavefront's key and value loads of a pass (8 x 16 bytes per lane) are issued together, the next pass's ahead.
// ------------------------------------------------------------------------------------------------
constexpr int kAsThreads = 256, kAsWaves = kAsThreads / 64;
constexpr int kAsMaxHeads = 8;     // query heads of one workgroup
constexpr int kAsPitch = kAttnHD + 8;
constexpr int kAsPass = 16 * kAsWaves;   // positions of a workgroup per pass: 16 per wavefront
constexpr int kAsMaxPasses = 8;

__device__ __forceinline__ float max16(float v) {
  static_for<0, 4>([&](auto I) { v = fmaxf(v, lane_xor<(1 << decltype(I)::value)>(v)); });
  return v;
}
__device__ __forceinline__ float add16(float v) {
  static_for<0, 4>([&](auto I) { v += lane_xor<(1 << decltype(I)::value)>(v); });
  return v;
}

struct AttnSplitArgs {
  const uint16_t *q, *k, *v;
  uint16_t *kc, *vc;
  const int64_t* pos;
  const float *rcos, *rsin;
  int grp, max_len, splits, passes;   // passes: the most 64-position passes of a workgroup
  int direct;                         // positions below it are held by one workgroup per head
  float scale;
  float* part_o;    // (n_heads, splits, 128): the range's sum of exp(s - m) v
  float2* part_ml;  // (n_heads, splits): its m and sum of exp(s - m)
  uint32_t* counters;   // arrivals, one per 256-byte line and (key/value head, head group), or null: a second launch merges
  const uint16_t* suh;
  uint16_t *o, *xh;
};
constexpr int kAsCounterStride = 64;

// What a workgroup of the split form does: nh query heads from h0 on of key/value head kh, the passes at base, base +
// stride, ... . n: workgroups that hold positions of these heads (1: this one writes their outputs). part: its place among
// them; group: the arrival counter; adds_row: it writes the new key/value rows if it holds their position.
struct AttnWork {
  int kh, h0, nh, base, stride, n, part, group;
  bool adds_row;
};

template <int GH>
__device__ __forceinline__ void attn_split_body(const AttnSplitArgs& a, const AttnWork& wk, int pos) {
  extern __shared__ float sp[];   // [GH][64 x passes]: scores, then exp(s - m), of this workgroup's positions
  __shared__ __align__(16) uint16_t sq[16 * kAsPitch];
  __shared__ __align__(16) uint16_t sk[kAttnHD], sv[kAttnHD];
  __shared__ __align__(16) float so[kAsWaves][GH][kAttnHD];
  __shared__ float sm[kAsWaves][16], sl[kAsWaves][16];
  __shared__ float sw[GH][128], sf[GH][kAttnHD];   // the merge's weights; the heads' outputs
  __shared__ uint32_t arrived_last;
  const int base = wk.base, stride = wk.stride, kh = wk.kh, h0 = wk.h0, nh = wk.nh, n = wk.n;
  const int L = pos + 1, passes = (pos - base) / stride + 1, pitch = a.passes * kAsPass;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int q = lane >> 4, c = lane & 15;
  const size_t kv0 = (size_t)kh * a.max_len * kAttnHD;
  const int last = max(pos - 1, 0);   // (rows from pos on are replaced or masked below)

  auto load_k = [&](int j, u32x4 (&w)[4]) {
    const int p = min(base + j * stride + wave * 16 + c, last);
    const u32x4* kr = reinterpret_cast<const u32x4*>(a.kc + kv0 + (size_t)p * kAttnHD) + q;
#pragma unroll
    for (int s = 0; s < 4; ++s) w[s] = kr[4 * s];
  };
  auto load_v = [&](int j, u32x4 (&w)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = min(base + j * stride + wave * 16 + 4 * i + q, last);
      w[i] = *(reinterpret_cast<const u32x4*>(a.vc + kv0 + (size_t)p * kAttnHD) + c);
    }
  };
  u32x4 kw[4], vw[4];
  load_k(0, kw);
  load_v(0, vw);

  // ---- rotary embedding of the query heads, and of the new key where this workgroup holds its position ----
  const bool has_new = pos - base - (passes - 1) * stride < kAsPass;
  // (thread: pair tid % 64 of heads tid / 64, + 4, ...; the new key counts as head nh; every load before any use)
  {
    const int i = tid & 63, n_rot = nh + (has_new ? 1 : 0);
    const float cs = a.rcos[(size_t)pos * (kAttnHD / 2) + i], sn = a.rsin[(size_t)pos * (kAttnHD / 2) + i];
    constexpr int kSlots = (GH + 1 + 3) / 4;
    uint16_t x[kSlots], y[kSlots];
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
      const int hh = (tid >> 6) + 4 * u;
      const uint16_t* src = hh < nh ? a.q + (size_t)(h0 + hh) * kAttnHD : a.k + (size_t)kh * kAttnHD;
      x[u] = src[i];
      y[u] = src[i + 64];
    }
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
      const int hh = (tid >> 6) + 4 * u;
      if (hh < n_rot) {
        uint16_t* dst = hh < nh ? sq + hh * kAsPitch : sk;
        const float xf = f16_to_f32(x[u]), yf = f16_to_f32(y[u]);
        const float xc = xf * cs, ys = yf * sn, yc = yf * cs, xs = xf * sn;
        dst[i] = f32_to_f16(xc - ys);
        dst[i + 64] = f32_to_f16(yc + xs);
      }
    }
  }
  if (has_new && tid < kAttnHD) sv[tid] = a.v[(size_t)kh * kAttnHD + tid];
  __syncthreads();
  if (has_new && wk.adds_row && tid < 32) {   // the new rows, once per key/value head
    const int e = tid & 15;
    uint16_t* dst = (tid < 16 ? a.kc : a.vc) + kv0 + (size_t)pos * kAttnHD;
    reinterpret_cast<u32x4*>(dst)[e] = reinterpret_cast<const u32x4*>(tid < 16 ? sk : sv)[e];
  }

  // ---- scores: sc[r] = head 4q + r, this lane's position of the pass ----
  float m[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  u32x4 A[4], kn[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    A[s] = *reinterpret_cast<const u32x4*>(sq + c * kAsPitch + 32 * s + 8 * q);
    kn[s] = *reinterpret_cast<const u32x4*>(sk + 32 * s + 8 * q);
  }
  for (int j = 0; j < passes; ++j) {
    u32x4 next[4];
    load_k(min(j + 1, passes - 1), next);
    const int at = j * kAsPass + wave * 16 + c, p = base + j * stride + wave * 16 + c;
    f32x4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s)
      sc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, A[s]),
                                                  __builtin_bit_cast(f16x8, p == pos ? kn[s] : kw[s]), sc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float x = p < L ? sc[r] * a.scale : -INFINITY;
      m[r] = fmaxf(m[r], x);
      if (4 * q + r < GH) sp[(4 * q + r) * pitch + at] = x;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) kw[s] = next[s];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    m[r] = max16(m[r]);
    if (c == 0) sm[wave][4 * q + r] = m[r];
  }
  __syncthreads();
  // exp(s - m) in place and its sum; a wavefront's own positions, so no further barrier
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    m[r] = fmaxf(fmaxf(sm[0][4 * q + r], sm[1][4 * q + r]), fmaxf(sm[2][4 * q + r], sm[3][4 * q + r]));
    // (a range of scores that are all -inf adds nothing: exp(-inf - 0), not exp(-inf + inf))
    const float mr = m[r] == -INFINITY ? 0.f : m[r];
    float l = 0.f;
    if (4 * q + r < GH) {
      for (int j = 0; j < passes; ++j) {
        float& x = sp[(4 * q + r) * pitch + j * kAsPass + wave * 16 + c];
        const float e = expf(x - mr);
        x = e;
        l += e;
      }
    }
    l = add16(l);
    if (c == 0) sl[wave][4 * q + r] = l;
  }

  // ---- P V: slot q's rows 4 i + q of each pass, dimensions 8 c .. 8 c + 7 ----
  float acc[GH][8];
#pragma unroll
  for (int h = 0; h < GH; ++h)
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[h][d] = 0.f;
  const u32x4 vn = reinterpret_cast<const u32x4*>(sv)[c];
  for (int j = 0; j < passes; ++j) {
    u32x4 next[4];
    load_v(min(j + 1, passes - 1), next);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = base + j * stride + wave * 16 + 4 * i + q;
      // (rows past the position hold anything: zeros, not probability zero times what is there)
      const u32x4 w = p == pos ? vn : p < pos ? vw[i] : u32x4{0u, 0u, 0u, 0u};
      const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
      float vf[8];
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        vf[2 * d] = f16_to_f32((uint16_t)(ww[d] & 0xFFFFu));
        vf[2 * d + 1] = f16_to_f32((uint16_t)(ww[d] >> 16));
      }
#pragma unroll
      for (int h = 0; h < GH; ++h) {
        const float pr = sp[h * pitch + j * kAsPass + wave * 16 + 4 * i + q];
#pragma unroll
        for (int d = 0; d < 8; ++d) acc[h][d] = __builtin_fmaf(pr, vf[d], acc[h][d]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) vw[i] = next[i];
  }
  // added over the four slots (lanes 16 and 32 apart), two registers into one per exchange: slot q is left with dimensions
  // 8 c + 4 (q >> 1) + 2 (q & 1) + {0, 1}
#pragma unroll
  for (int h = 0; h < GH; ++h) {
    float r4[4], r2[2];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const auto x = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, acc[h][d]),
                                                      __builtin_bit_cast(uint32_t, acc[h][d + 4]), false, false);
      r4[d] = __builtin_bit_cast(float, (uint32_t)x[0]) + __builtin_bit_cast(float, (uint32_t)x[1]);
    }
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const auto x = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, r4[d]),
                                                      __builtin_bit_cast(uint32_t, r4[d + 2]), false, false);
      r2[d] = __builtin_bit_cast(float, (uint32_t)x[0]) + __builtin_bit_cast(float, (uint32_t)x[1]);
    }
    *reinterpret_cast<float2*>(&so[wave][h][8 * c + 4 * (q >> 1) + 2 * (q & 1)]) = float2{r2[0], r2[1]};
  }
  __syncthreads();
  if (n == 1) {   // this one holds them all
    for (int idx = tid; idx < nh * kAttnHD; idx += kAsThreads) {
      const int h = idx >> 7, d = idx & 127;
      const float l = ((sl[0][h] + sl[1][h]) + sl[2][h]) + sl[3][h];
      sf[h][d] = round_f16((((so[0][h][d] + so[1][h][d]) + so[2][h][d]) + so[3][h][d]) / l);
    }
    __syncthreads();
    for (int h = wave; h < nh; h += kAsWaves) write_head(sf[h], h0 + h, lane, a.suh, a.o, a.xh);
    return;
  }
  // device-scope stores: with counters, the last workgroup to arrive reads them in this launch
  for (int idx = tid; idx < nh * kAttnHD; idx += kAsThreads) {
    const int h = idx >> 7, d = idx & 127;
    __hip_atomic_store(a.part_o + ((size_t)(h0 + h) * a.splits + wk.part) * kAttnHD + d,
                       ((so[0][h][d] + so[1][h][d]) + so[2][h][d]) + so[3][h][d], __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
  if (tid < nh) {
    float* ml = reinterpret_cast<float*>(a.part_ml + (size_t)(h0 + tid) * a.splits + wk.part);
    __hip_atomic_store(ml, fmaxf(fmaxf(sm[0][tid], sm[1][tid]), fmaxf(sm[2][tid], sm[3][tid])), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(ml + 1, ((sl[0][tid] + sl[1][tid]) + sl[2][tid]) + sl[3][tid], __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
  if (!a.counters) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this thread's stores are acknowledged
  __syncthreads();
  if (tid == 0) {
    uint32_t* ctr = a.counters + (size_t)wk.group * kAsCounterStride;
    const uint32_t prev = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    arrived_last = prev == (uint32_t)(n - 1);
    if (arrived_last) __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // zero again at rest
  }
  __syncthreads();
  if (!arrived_last) return;
  // ---- the last arriver merges: weights exp(m - max m) of the n <= 128 workgroups, head h by wavefront h % 4 ----
  const __amdgpu_buffer_rsrc_t rs_o = __builtin_amdgcn_make_buffer_rsrc(
      a.part_o + (size_t)h0 * a.splits * kAttnHD, (short)0, nh * a.splits * kAttnHD * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_ml = __builtin_amdgcn_make_buffer_rsrc(
      a.part_ml + (size_t)h0 * a.splits, (short)0, nh * a.splits * 8, 0x00020000);
  constexpr int kDeviceScope = 16;   // sc1: coherent at device scope
  constexpr int kPerWave = (GH + kAsWaves - 1) / kAsWaves;
  u32x2 ml[kPerWave][2];
#pragma unroll
  for (int u = 0; u < kPerWave; ++u)
#pragma unroll
    for (int e = 0; e < 2; ++e)   // (past the heads: past the descriptor; past the workgroups in use: not added below)
      ml[u][e] = __builtin_amdgcn_raw_buffer_load_b64(rs_ml, (uint32_t)((wave + kAsWaves * u) * a.splits + lane + 64 * e) * 8u, 0, kDeviceScope);
  // thread (g, e): workgroups g, g + 8, ... of dimensions 4 e .. 4 e + 3 of each head
  const int e4 = tid & 31, g = tid >> 5;
  auto load_o = [&](int h, int s) {
    return __builtin_amdgcn_raw_buffer_load_b128(rs_o, (uint32_t)((h * a.splits + s) * kAttnHD + 4 * e4) * 4u, 0, kDeviceScope);
  };
  u32x4 first[GH][2];   // workgroups g and g + 8 of every head, in flight during the reductions
#pragma unroll
  for (int h = 0; h < GH; ++h)
#pragma unroll
    for (int u = 0; u < 2; ++u) first[h][u] = load_o(h, g + 8 * u);
  __syncthreads();   // (sp is free)
#pragma unroll
  for (int u = 0; u < kPerWave; ++u) {
    const int h = wave + kAsWaves * u;
    if (h < nh) {
      const uint32_t m0b = ml[u][0].x, l0b = ml[u][0].y, m1b = ml[u][1].x, l1b = ml[u][1].y;
      const float m0 = lane < n ? __builtin_bit_cast(float, m0b) : -INFINITY;
      const float m1 = lane + 64 < n ? __builtin_bit_cast(float, m1b) : -INFINITY;
      float mx = fmaxf(m0, m1);
      static_for<0, 6>([&](auto I) { mx = fmaxf(mx, xor_partner<(1 << decltype(I)::value)>(mx, lane)); });
      const float w0 = lane < n ? expf(m0 - mx) : 0.f, w1 = lane + 64 < n ? expf(m1 - mx) : 0.f;
      sw[h][lane] = w0;
      sw[h][lane + 64] = w1;
      float l = (lane < n ? __builtin_bit_cast(float, l0b) * w0 : 0.f) +
                (lane + 64 < n ? __builtin_bit_cast(float, l1b) * w1 : 0.f);
      static_for<0, 6>([&](auto I) { l += xor_partner<(1 << decltype(I)::value)>(l, lane); });
      if (lane == 0) sl[0][h] = l;
    }
  }
  __syncthreads();
  auto add = [&](f32x4& t, int h, int s, const u32x4& v) {
    if (s < n) {
      const float ws = sw[h][s];
      const uint32_t b[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int d = 0; d < 4; ++d) t[d] = __builtin_fmaf(ws, __builtin_bit_cast(float, b[d]), t[d]);
    }
  };
#pragma unroll
  for (int h = 0; h < GH; ++h) {
    f32x4 t = {0.f, 0.f, 0.f, 0.f};
    add(t, h, g, first[h][0]);
    add(t, h, g + 8, first[h][1]);
    for (int s0 = 16 + g; s0 < n; s0 += 32) {
      u32x4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = load_o(h, s0 + 8 * u);
#pragma unroll
      for (int u = 0; u < 4; ++u) add(t, h, s0 + 8 * u, v[u]);
    }
    float r[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      float x0, x1;
      pair_values<32>(t[d], x0, x1);
      r[d] = x0 + x1;
    }
    if (lane < 32) *reinterpret_cast<f32x4*>(&so[wave][h][4 * e4]) = f32x4{r[0], r[1], r[2], r[3]};
  }
  __syncthreads();
  for (int idx = tid; idx < nh * kAttnHD; idx += kAsThreads) {
    const int h = idx >> 7, d = idx & 127;
    sf[h][d] = round_f16((((so[0][h][d] + so[1][h][d]) + so[2][h][d]) + so[3][h][d]) / sl[0][h]);
  }
  __syncthreads();
  for (int h = wave; h < nh; h += kAsWaves) write_head(sf[h], h0 + h, lane, a.suh, a.o, a.xh);
}

template <int GH>
__global__ __launch_bounds__(kAsThreads) void attn_split_kernel(AttnSplitArgs a) {
  const int64_t pos64 = *a.pos;
  // the arguments used past the first branch, loaded with the position's address instead of where they are used
  asm volatile("" ::"s"(a.q), "s"(a.kc), "s"(a.rcos), "s"(a.direct), "s"(a.scale), "s"(a.part_o), "s"(a.counters), "s"(a.o));
  const int x = blockIdx.x, kh = blockIdx.y, hz = blockIdx.z * GH;
  const int h0 = kh * a.grp + hz, nh = min(GH, a.grp - hz);
  if (pos64 < 0 || pos64 >= (int64_t)a.max_len) {   // an invalid position yields zeros
    if (x == 0)
      for (int idx = threadIdx.x; idx < nh * kAttnHD; idx += kAsThreads) {
        const size_t at = (size_t)h0 * kAttnHD + idx;
        if (a.o) a.o[at] = 0;
        if (a.xh) a.xh[at] = 0;
      }
    return;
  }
  const int pos = (int)pos64, group = kh * gridDim.z + blockIdx.z;
  AttnWork wk{kh, h0, nh, x * kAsPass, a.splits * kAsPass, min(pos / kAsPass + 1, a.splits), x, group, blockIdx.z == 0};
  if (pos < a.direct) {   // few positions: a workgroup per head holds them all
    if (x >= nh) return;
    wk = AttnWork{kh, h0 + x, 1, 0, kAsPass, 1, 0, group, blockIdx.z == 0 && x == 0};
    if constexpr (GH > 1) {
      attn_split_body<1>(a, wk, pos);
      return;
    }
  }
  if (wk.base > pos || nh <= 0) return;
  attn_split_body<GH>(a, wk, pos);
}

// Adds a head's workgroups (at most 128) and writes o and its rotation, as the one-launch form does. Thread (g, e) adds
// workgroups g, g + 16, ... of dimensions 4 e .. 4 e + 3, all loads of a thread in flight together (two threads per
// dimension with eight loads each, in batches: 2.6 us more at 64 workgroups; loads only of the slots there are, a branch
// each: 0.25 us more, the first is waited for alone). Every slot is loaded before the position is known; the slots past
// the workgroups in use hold anything and are not added.
constexpr int kAmThreads = 512, kAmGroups = kAmThreads / 32, kAmLoads = 8;

__global__ __launch_bounds__(kAmThreads) void attn_merge_kernel(const float* __restrict__ part_o,
                                                                const float2* __restrict__ part_ml,
                                                                const int64_t* __restrict__ pos_p, int max_len,
                                                                int direct, int splits, const uint16_t* __restrict__ suh,
                                                                uint16_t* __restrict__ o_out, uint16_t* __restrict__ xh) {
  __shared__ float sw[128], red[4], sfin[kAttnHD];
  __shared__ f32x4 so[kAmGroups][32];
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int e = tid & 31, g = tid >> 5;
  const int64_t pos64 = *pos_p;
  const f32x4* po = reinterpret_cast<const f32x4*>(part_o + (size_t)h * splits * kAttnHD) + e;
  f32x4 t[kAmLoads];
#pragma unroll
  for (int u = 0; u < kAmLoads; ++u)
    t[u] = po[(size_t)min(g + u * kAmGroups, splits - 1) * 32];
  const float2 ml = part_ml[(size_t)h * splits + min(tid, splits - 1)];
  asm volatile("" ::"v"(ml.x), "v"(ml.y));   // (every load ahead of the branch)
  // (the first launch wrote the outputs: of few positions, and the zeros of an invalid one)
  if (pos64 < (int64_t)direct || pos64 < kAsPass || pos64 >= (int64_t)max_len || splits == 1) return;
  const int n = min((int)(pos64 / kAsPass) + 1, splits);
  float mx = 0.f, w = 0.f;
  if (wave < 2) {   // the weights exp(m - max m) of up to 128 workgroups, by two wavefronts
    mx = tid < n ? ml.x : -INFINITY;
    static_for<0, 6>([&](auto I) { mx = fmaxf(mx, xor_partner<(1 << decltype(I)::value)>(mx, lane)); });
    if (lane == 0) red[wave] = mx;
  }
  __syncthreads();
  if (wave < 2) {
    mx = fmaxf(red[0], red[1]);
    w = tid < n ? expf(ml.x - mx) : 0.f;
    sw[tid] = w;
    float ls = tid < n ? ml.y * w : 0.f;
    static_for<0, 6>([&](auto I) { ls += xor_partner<(1 << decltype(I)::value)>(ls, lane); });
    if (lane == 0) red[2 + wave] = ls;
  }
  __syncthreads();
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < kAmLoads; ++u) {
    if (g + u * kAmGroups < n) {
      const float ws = sw[g + u * kAmGroups];
#pragma unroll
      for (int d = 0; d < 4; ++d) acc[d] = __builtin_fmaf(ws, t[u][d], acc[d]);
    }
  }
  so[g][e] = acc;
  __syncthreads();
  if (tid < kAttnHD) {
    float o = 0.f;
#pragma unroll
    for (int u = 0; u < kAmGroups; ++u) o += reinterpret_cast<const float*>(so[u])[tid];
    sfin[tid] = round_f16(o / (red[2] + red[3]));
  }
  __syncthreads();
  if (wave == 0) write_head(sfin, h, lane, suh, o_out, xh);
}

template <int GH>
static void launch_attn_split(const dim3& grid, const AttnSplitArgs& a, hipStream_t st) {
  attn_split_kernel<GH><<<grid, kAsThreads, (size_t)GH * a.passes * kAsPass * sizeof(float), st>>>(a);
}

// Head groups of a key/value head and workgroups (S) per head group, from the shape alone: one workgroup per CU in all. A
// workgroup's latency grows with its heads (~0.5 us each) and its passes (at most kAsMaxPasses at full capacity: their
// scores stay in LDS), so the smallest head groups are taken that leave S that many workgroups; more groups than CUs, or
// more splits, cost more in dispatch and merge than they save. Measured at 48 / 8 heads, us, graph replays of one call
// (rows in the caches from the replay before; in a decode step, among the layers' weights, 9.8-10.4 at position 700 of
// 1,024), position 15 / 100 / 200 / 300 / 700 / 2,000 / 4,000 / 8,100:
//   one launch, capacity 1,024    4.8 / 5.9 / 7.0 / 7.3 / 8.4
//               capacity 4,096    4.7 / 5.7 / 7.2 / 7.4 / 8.1 / 10.1 / 13.3
//               capacity 8,192    4.6 / 5.6 / 7.2 / 8.1 / 8.6 /  9.9 / 12.0 / 16.2
//   two launches, 1,024           6.3 / 7.2 / 8.1 / 8.4 / 9.6
//                 8,192           6.1 / 7.1 / 8.7 / 8.8 / 9.1 / 10.4 / 12.4 / 16.5
//   one workgroup per head        5.9 / 6.7 / 7.3 / 8.0 / 11.3 / 21.4 / 36.4 / 66
// Two launches lose to one workgroup per head below ~350 positions (the second launch is 1.4 us that nothing can take
// back once it is enqueued); only a captured call that holds no workspace takes them. Plans of 512 and 768 workgroups with
// smaller head groups: up to 0.6 us less at position 100, 3-6 us more at 8,100; groups of up to 8 heads: 2.5 us more at 100.
constexpr int kAsWorkgroups = 256;

static int attn_least_splits(int max_len) {
  return (max_len + kAsMaxPasses * kAsPass - 1) / (kAsMaxPasses * kAsPass);
}

static int attn_head_groups(int n_kv, int grp, int max_len) {
  const int least = attn_least_splits(max_len);
  int gh = 1;
  while (gh < grp && gh < kAsMaxHeads && (int64_t)n_kv * ((grp + gh - 1) / gh) * least > kAsWorkgroups) ++gh;
  return (grp + gh - 1) / gh;
}

// Passes up to which a workgroup per head holds all positions (no merge) in a plan of GH heads per workgroup: a pass costs
// 0.85 us, spreading the passes costs the merge and GH heads' work per workgroup. Without counters the merge is a launch
// that is there in any case, so less is saved.
static int attn_direct_passes(int slots, bool counters) {
  return slots <= 2 ? 3 : std::min(slots + 1, counters ? 6 : 4);
}

// (at least a pass of 64 positions each)
static int attn_splits(int n_kv, int z, int max_len) {
  const int most = (max_len + kAsPass - 1) / kAsPass, least = attn_least_splits(max_len);
  const int want = kAsWorkgroups / (n_kv * z);
  return want > most ? most : want < least ? least : want;
}

}  // namespace exl3

using namespace exl3;

extern "C" size_t exl3_attn_decode_workspace_bytes(int n_heads, int n_kv_heads, int max_len) {
  if (n_heads < 1 || n_kv_heads < 1 || n_heads % n_kv_heads != 0 || max_len < 1 || max_len > kAttnMaxLen) return 0;
  const int z = attn_head_groups(n_kv_heads, n_heads / n_kv_heads, max_len);
  return (size_t)n_heads * attn_splits(n_kv_heads, z, max_len) * (kAttnHD * sizeof(float) + sizeof(float2));
}

extern "C" int exl3_attn_decode_rotate(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* k_cache,
                                       uint16_t* v_cache, const int64_t* pos, const float* rope_cos,
                                       const float* rope_sin, int n_heads, int n_kv_heads, int head_dim,
                                       int max_len, const uint16_t* suh, uint16_t* o, uint16_t* xh, void* stream) {
  return exl3_attn_decode_rotate_ws(q, k, v, k_cache, v_cache, pos, rope_cos, rope_sin, n_heads, n_kv_heads, head_dim,
                                    max_len, suh, o, xh, nullptr, 0, nullptr, stream);
}

extern "C" int exl3_attn_decode_rotate_ws(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* k_cache,
                                          uint16_t* v_cache, const int64_t* pos, const float* rope_cos,
                                          const float* rope_sin, int n_heads, int n_kv_heads, int head_dim,
                                          int max_len, const uint16_t* suh, uint16_t* o, uint16_t* xh, void* workspace,
                                          size_t workspace_bytes, uint32_t* counters, void* stream) {
  EXL3_REQUIRE(q && k && v && k_cache && v_cache && pos && rope_cos && rope_sin, EXL3_ERR_ARG,
               "exl3_attn_decode_rotate: NULL input, cache, position or rope table");
  EXL3_REQUIRE(o || xh, EXL3_ERR_ARG, "exl3_attn_decode_rotate: neither o nor xh requested");
  EXL3_REQUIRE(!xh || suh, EXL3_ERR_ARG, "exl3_attn_decode_rotate: xh needs suh");
  EXL3_REQUIRE(head_dim == kAttnHD, EXL3_ERR_ARG, "exl3_attn_decode_rotate: head_dim must be 128 (got %d)",
               head_dim);
  EXL3_REQUIRE(n_heads >= 1 && n_kv_heads >= 1 && n_heads % n_kv_heads == 0, EXL3_ERR_ARG,
               "exl3_attn_decode_rotate: n_heads must be a positive multiple of n_kv_heads");
  EXL3_REQUIRE(max_len >= 1 && max_len <= kAttnMaxLen, EXL3_ERR_ARG,
               "exl3_attn_decode_rotate: max_len must be 1..%d (got %d)", kAttnMaxLen, max_len);
  EXL3_REQUIRE(aligned(k_cache, 16) && aligned(v_cache, 16) && aligned(pos, 8) && aligned(rope_cos, 4) &&
                   aligned(rope_sin, 4),
               EXL3_ERR_ARG, "exl3_attn_decode_rotate: caches must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const float scale = 1.0f / sqrtf((float)head_dim);
  if (workspace && n_heads <= 65535) {   // (grid dimensions of the split form)
    const size_t need = exl3_attn_decode_workspace_bytes(n_heads, n_kv_heads, max_len);
    EXL3_REQUIRE(workspace_bytes >= need && aligned(workspace, 16), EXL3_ERR_WORKSPACE,
                 "exl3_attn_decode_rotate_ws: a 16-byte aligned workspace of %zu bytes is needed (got %zu)", need,
                 workspace_bytes);
    const int grp = n_heads / n_kv_heads, z = attn_head_groups(n_kv_heads, grp, max_len), gh = (grp + z - 1) / z;
    const int splits = attn_splits(n_kv_heads, z, max_len);
    const int slots = gh <= 4 ? gh : gh <= 6 ? 6 : 8;   // heads the kernel is built for
    // (a workgroup of the head group for each of its heads)
    const int direct_passes = std::min(slots, grp) <= splits ? attn_direct_passes(slots, counters != nullptr) : 0;
    const int passes = std::max((max_len + splits * kAsPass - 1) / (splits * kAsPass), direct_passes);
    float* part_o = static_cast<float*>(workspace);
    const AttnSplitArgs a{q, k, v, k_cache, v_cache, pos, rope_cos, rope_sin, grp, max_len, splits, passes,
                          direct_passes * kAsPass, scale, part_o,
                          reinterpret_cast<float2*>(part_o + (size_t)n_heads * splits * kAttnHD), counters, suh, o, xh};
    const dim3 grid((unsigned)splits, (unsigned)n_kv_heads, (unsigned)z);
    if (slots == 1) launch_attn_split<1>(grid, a, st);
    else if (slots == 2) launch_attn_split<2>(grid, a, st);
    else if (slots == 3) launch_attn_split<3>(grid, a, st);
    else if (slots == 4) launch_attn_split<4>(grid, a, st);
    else if (slots == 6) launch_attn_split<6>(grid, a, st);
    else launch_attn_split<8>(grid, a, st);
    if (!counters)
      attn_merge_kernel<<<n_heads, kAmThreads, 0, st>>>(a.part_o, a.part_ml, pos, max_len, a.direct, splits, suh, o, xh);
    EXL3_LAUNCH_CHECK("exl3_attn_decode_rotate_ws");
    return EXL3_OK;
  }
  attn_decode_kernel<<<n_heads, kAttnThreads, (size_t)max_len * sizeof(float), st>>>(
      q, k, v, k_cache, v_cache, pos, rope_cos, rope_sin, n_heads, n_kv_heads, max_len, scale, suh, o, xh);
  EXL3_LAUNCH_CHECK("exl3_attn_decode_rotate");
  return EXL3_OK;
}
