// Device side of the router shared by the kernels that route rows of E experts with E a power of
// two up to 256 (topk_softmax_pow2_kernel, the gate-fused kernel, the single-workgroup routing +
// alignment kernel): lane geometry, lane exchanges and the softmax + top-k of one row.
#pragma once

#include "common.h"

namespace {

template <int E>
struct Pow2Geom {
  static constexpr int kEpl = (E < 4) ? E : 4;  // floats per vector load
  static constexpr int kVecs = (E / (kEpl * 32)) < 1 ? 1 : (E / (kEpl * 32));
  static constexpr int kVpt = kVecs * kEpl;     // values per lane
  static constexpr int kTpr = E / kVpt;         // lanes per row
  static constexpr int kRowsPerWave = kWave / kTpr;
};

constexpr int kWavesPerBlock = 4;

// Lane exchanges of a row of TPR lanes, by DPP moves and v_permlane16_swap: a few clocks each, where the LDS-crossbar
// shuffle behind __shfl_xor costs ~100 and was most of a round.
// max over the row: any order will do, so distances 4 and 8 use the mirror patterns, which pair every lane with a lane of
// the other half of its 8- or 16-lane group: the same thing once the lanes of each half already agree.
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
// The values of the lane's row of 16 and of the row beside it (lane ^ 16), as an unordered pair.  (In assembly: given the
// same value twice, the compiler takes the builtin's two results for one.  The wait states are those that it puts in
// front of the instruction.)
__device__ __forceinline__ void rows_of_16(float v, float& a, float& b) {
  a = b = v;
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
template <int TPR>
__device__ __forceinline__ float row_max(float v) {
  static_assert(TPR <= 32, "a row of lanes");
  if constexpr (TPR > 1) v = fmaxf(v, dpp_move<0xB1>(v));   // quad_perm [1,0,3,2]
  if constexpr (TPR > 2) v = fmaxf(v, dpp_move<0x4E>(v));   // quad_perm [2,3,0,1]
  if constexpr (TPR > 4) v = fmaxf(v, dpp_move<0x141>(v));  // row_half_mirror
  if constexpr (TPR > 8) v = fmaxf(v, dpp_move<0x140>(v));  // row_mirror
  if constexpr (TPR > 16) {
    float a, b;
    rows_of_16(v, a, b);
    v = fmaxf(a, b);
  }
  return v;
}
// The sum with the association of the xor butterfly from distance TPR / 2 down to 1.
template <int TPR>
__device__ __forceinline__ float row_sum(float v) {
  static_assert(TPR <= 32, "a row of lanes");
  if constexpr (TPR > 16) {
    float a, b;
    rows_of_16(v, a, b);
    v = a + b;
  }
  if constexpr (TPR > 8) v += dpp_move<0x128>(v);  // row_ror:8 is lane ^ 8
  if constexpr (TPR > 8) {
    v += dpp_move<0x124>(v);                       // row_ror:4 is lane ^ 4 where lanes eight apart agree
  } else if constexpr (TPR > 4) {
    // lane ^ 4: row_shl:4 into the first and third four lanes of a row of 16, row_shr:4 into the others
    const int b = __builtin_bit_cast(int, v), up = __builtin_amdgcn_update_dpp(0, b, 0x104, 0xf, 0x5, false);
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(up, b, 0x114, 0xf, 0xa, false));
  }
  if constexpr (TPR > 2) v += dpp_move<0x4E>(v);   // quad_perm [2,3,0,1]
  if constexpr (TPR > 1) v += dpp_move<0xB1>(v);   // quad_perm [1,0,3,2]
  return v;
}

// The logits of row `row` as route_row wants them, widened to fp32: lane t of the row loads columns
// (i / EPL) * EPL * TPR + t * EPL + i % EPL into v[i], EPL at a time.  A caller's rows need no more than the
// alignment of an element, and the type says so; the load is one instruction all the same (a global load takes
// any address).
template <typename S, int N>
struct __attribute__((packed, aligned(sizeof(S)))) RowVec {
  S v[N];
};
template <int E, typename El = ElemF32>
__device__ __forceinline__ void load_row(const typename El::S* __restrict__ gating, int row, int t,
                                         float (&v)[Pow2Geom<E>::kVpt]) {
  using G = Pow2Geom<E>;
  constexpr int EPL = G::kEpl, VECS = G::kVecs, TPR = G::kTpr;
  using V = RowVec<typename El::S, EPL>;
  const typename El::S* src = gating + static_cast<size_t>(row) * E + t * EPL;
#pragma unroll
  for (int j = 0; j < VECS; ++j) {
    const V q = *reinterpret_cast<const V*>(src + j * EPL * TPR);
#pragma unroll
    for (int i = 0; i < EPL; ++i) v[j * EPL + i] = El::ld(q.v[i]);
  }
}

// Softmax and K argmax rounds of one row spread over TPR lanes: lane t of the
// row holds columns (i / EPL) * EPL * TPR + t * EPL + i % EPL in v[i].
template <int E>
__device__ __forceinline__ void route_row(float (&v)[Pow2Geom<E>::kVpt], int t, int row, bool live,
                                          float* __restrict__ topk_w, int32_t* __restrict__ topk_ids,
                                          int32_t* __restrict__ tok_exp_idx, int T, int K,
                                          int renormalize) {
  using G = Pow2Geom<E>;
  constexpr int EPL = G::kEpl, VPT = G::kVpt, TPR = G::kTpr;
  float mx = v[0];
#pragma unroll
  for (int i = 1; i < VPT; ++i) mx = fmaxf(mx, v[i]);
  mx = row_max<TPR>(mx);

  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    v[i] = moe_expf(v[i] - mx);
    sum += v[i];
  }
  sum = row_sum<TPR>(sum);
  const float rinv = 1.f / sum;
#pragma unroll
  for (int i = 0; i < VPT; ++i) v[i] = v[i] * rinv;  // subnormal probabilities are kept, as the reference keeps them

  // Up to kRegK winners stay in registers until the row is done (after the
  // all-reduce every lane of the row knows them): the renormalised weights are
  // then written once, and when the row has at least K lanes, lane k writes
  // winner k, so a row's results leave as three short coalesced stores instead
  // of three single-lane stores per round.
  constexpr int kRegK = 16;
  float wsum = 0.f;
  float bw[kRegK];
  int bi[kRegK];
#pragma unroll
  for (int k = 0; k < kRegK; ++k) { bw[k] = 0.f; bi[k] = 0; }
  // One round: the row's largest value, then the lowest of the columns that hold it, from one ballot per value of a
  // lane.  (Column 0 where none does: all values NaN.  A row of one lane looks for itself.)  Carrying value and column
  // through every exchange, two of them through the LDS crossbar, was most of the kernel: 128 experts top-8, 1 token
  // 5.4 -> 3.7 us, 256 tokens 5.9 -> 4.2, 16896 13.4 -> 12.0.
  const int lane = threadIdx.x % kWave, row0 = lane & 31 & ~(TPR - 1);
  auto round = [&](float& best_out, int& bidx_out) {
    float best = v[0];
    uint32_t col = TPR == 1 ? 0u : ~0u;
#pragma unroll
    for (int i = 1; i < VPT; ++i) {
      if constexpr (TPR == 1) {
        if (v[i] > best) best = v[i], col = i;
      } else {
        best = fmaxf(best, v[i]);
      }
    }
    best = row_max<TPR>(best);
#pragma unroll
    for (int i = 0; TPR > 1 && i < VPT; ++i) {
      const uint64_t bal = __ballot(v[i] == best);
      const uint32_t half = lane & 32 ? static_cast<uint32_t>(bal >> 32) : static_cast<uint32_t>(bal);
      const uint32_t mine = TPR == 32 ? half : __builtin_amdgcn_ubfe(half, row0, TPR);
      const uint32_t c = (i / EPL) * (EPL * TPR) + static_cast<uint32_t>(__builtin_ctz(mine)) * EPL + i % EPL;
      col = min(col, mine ? c : ~0u);
    }
    const int bidx = col == ~0u ? 0 : static_cast<int>(col);
    wsum += best;
    best_out = best;
    bidx_out = bidx;
    // blank the winner in the lane that holds it
#pragma unroll
    for (int i = 0; i < VPT; ++i)
      if (bidx == (i / EPL) * (EPL * TPR) + t * EPL + i % EPL) v[i] = -10000.f;
  };
  if (K <= kRegK) {
#pragma unroll
    for (int k = 0; k < kRegK; ++k)
      if (k < K) round(bw[k], bi[k]);
    if (K <= TPR) {
      float my_w = 0.f;
      int my_i = 0;
#pragma unroll
      for (int k = 0; k < kRegK; ++k)
        if (t == k) { my_w = bw[k]; my_i = bi[k]; }
      if (live && t < K) {
        const size_t o = static_cast<size_t>(row) * K + t;
        topk_w[o] = renormalize ? my_w / wsum : my_w;
        topk_ids[o] = my_i;
        if (tok_exp_idx) tok_exp_idx[o] = t * T + row;
      }
    } else if (live && t == 0) {
#pragma unroll
      for (int k = 0; k < kRegK; ++k)
        if (k < K) {
          const size_t o = static_cast<size_t>(row) * K + k;
          topk_w[o] = renormalize ? bw[k] / wsum : bw[k];
          topk_ids[o] = bi[k];
          if (tok_exp_idx) tok_exp_idx[o] = k * T + row;
        }
    }
  } else {
    for (int k = 0; k < K; ++k) {
      float best;
      int bidx;
      round(best, bidx);
      if (live && t == 0) {
        const size_t o = static_cast<size_t>(row) * K + k;
        topk_w[o] = best;
        topk_ids[o] = bidx;
        if (tok_exp_idx) tok_exp_idx[o] = k * T + row;
      }
    }
    if (renormalize && live && t == 0) {
      for (int k = 0; k < K; ++k) {
        const size_t o = static_cast<size_t>(row) * K + k;
        topk_w[o] = topk_w[o] / wsum;
      }
    }
  }
}

}  // namespace
