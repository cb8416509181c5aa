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
    v[i] = moe_expf<true>(v[i] - mx);
    sum += v[i];
  }
  sum = row_sum<TPR>(sum);
  const float rinv = 1.f / sum;
#pragma unroll
  for (int i = 0; i < VPT; ++i) v[i] = v[i] * rinv;  // subnormal probabilities are kept, as the reference keeps them

  float wsum = 0.f;
  const int lane = threadIdx.x % kWave, row0 = lane & 31 & ~(TPR - 1);
  // The rounds are one rolled loop: a kernel that runs through its code once waits for its instructions, too, and sixteen
  // rounds in a row were three quarters of the router's code (128 experts: 10.6 KB and, rolled, 2.6; few_gate_kernel 18.8
  // and 10.2 then).  Router alone, 128 experts top-8, us, with them unrolled and as all of this function is now: 1 token 3.5
  // and 2.6, 128 3.8 and 2.8, 16896 11.7 and 8.6; norm and layer 1 token 23.4 and 22.3, 9 49.9 and 48.7, 64 88.4 and 87.5,
  // 128 114.6 and 113.7.
  // Winner k stays in lane k % TPR of the row (every lane knows it after the round), the TPR latest in a lane's first pair of
  // registers and those before them one pair on: a lane has as many pairs as columns, so that all K of a row find a place,
  // nothing is stored before the sum is known and the renormalised weights leave as short coalesced stores.  With K beyond
  // the lanes stored round by round, read back, divided and stored again by one lane, and this way, router alone, us: 16
  // experts top-6, 1 token 3.8 and 2.8, 135 4.3 and 3.0, 16896 5.0 and 3.7; top-8, 135 5.0 and 3.2; 8 top-8, 135 4.8 and 3.7;
  // 32 top-16, 135 7.6 and 4.0; 64 top-24, 4096 11.7 and 5.1.  The loop without those stores is the shorter one for fewer
  // winners, too: 128 top-8, 1 token 3.3 and 2.9, 16896 10.2 and 9.3.  Layer, 16 experts, H 1024, I 384, top-6, 16 tokens
  // 19.9 and 19.0; 128, H 2048, I 768, top-8, 128 tokens 117.3 and 116.3.
  float my_w[VPT];
  int my_i[VPT];
#pragma unroll
  for (int j = 0; j < VPT; ++j) my_w[j] = 0.f, my_i[j] = 0;
  // K rounds; a round says its winner to `keep`.
  auto rounds = [&](auto&& round) {
#pragma unroll 1
    for (int base = 0; base < K; base += TPR) {
#pragma unroll
      for (int j = VPT - 1; j > 0; --j) my_w[j] = my_w[j - 1], my_i[j] = my_i[j - 1];
      const int n = K - base < TPR ? K - base : TPR;
#pragma unroll 1
      for (int k = 0; k < n; ++k)
        round([&](float best, int bidx) {
          wsum += best;
          my_w[0] = t == k ? best : my_w[0];
          my_i[0] = t == k ? bidx : my_i[0];
        });
    }
  };
  // The bits that a ballot has for this lane's row of lanes.
  auto row_bits = [&](uint64_t bal) {
    const uint32_t half = lane & 32 ? static_cast<uint32_t>(bal >> 32) : static_cast<uint32_t>(bal);
    return TPR == 32 ? half : __builtin_amdgcn_ubfe(half, row0, TPR);
  };
  constexpr bool kHeads = VPT == 4 && TPR > 1;   // a lane's columns are four in a row, so that lanes are in their order
  if (kHeads && !__ballot(v[0] != v[0])) {
    // Probabilities are not negative, so that their bits compare as they do.  A lane sorts its four, the lower column first
    // where two are equal, and a round looks at the lanes' largest only: one exchange, the first lane that holds the row's
    // largest wins and goes on to its next.  A round is a chain of dependent instructions, 0.28 us of it when each looked at
    // all four values of a lane, and stands in front of everything in a call of few tokens.  Router alone, 128 experts top-8,
    // us, that way and this: 1 token 3.1 and 2.6, 128 3.4 and 2.8, 16896 11.3 and 8.6; 16 top-6, 135 2.9 and 2.6.
    int h[4], which[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) h[i] = __builtin_bit_cast(int, v[kHeads ? i : 0]), which[i] = i;
#pragma unroll
    for (int pass = 0; pass < 4; ++pass)
#pragma unroll
      for (int i = pass & 1; i + 1 < 4; i += 2) {   // (neighbours only, and never equal ones: the order of equals stays)
        const bool swap = h[i] < h[i + 1];
        const int hi = swap ? h[i + 1] : h[i], lo = swap ? h[i] : h[i + 1];
        const int wi = swap ? which[i + 1] : which[i], wl = swap ? which[i] : which[i + 1];
        h[i] = hi, h[i + 1] = lo, which[i] = wi, which[i + 1] = wl;
      }
    uint32_t order = which[0] | which[1] << 2 | which[2] << 4 | which[3] << 6;
    rounds([&](auto&& keep) {
      const int best = row_max_bits<TPR>(h[0]);
      const uint32_t at = __builtin_ctz(row_bits(__ballot(h[0] == best)));
      const uint32_t low = __builtin_amdgcn_ubfe(row_bits(__ballot((order & 1) != 0)), at, 1);
      const uint32_t high = __builtin_amdgcn_ubfe(row_bits(__ballot((order & 2) != 0)), at, 1);
      keep(__builtin_bit_cast(float, best), static_cast<int>(4 * at + 2 * high + low));
      const bool won = t == static_cast<int>(at);
      h[0] = won ? h[1] : h[0];
      h[1] = won ? h[2] : h[1];
      h[2] = won ? h[3] : h[2];
      h[3] = won ? -1 : h[3];
      order = won ? order >> 2 : order;
    });
  } else {
    // One round: the row's largest value, then the lowest of the columns that hold it, from one ballot per value of a
    // lane.  (Column 0 where none does: all values NaN.  A row of one lane looks for itself.)
    rounds([&](auto&& keep) {
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
        const uint32_t mine = row_bits(__ballot(v[i] == best));
        const uint32_t c = (i / EPL) * (EPL * TPR) + static_cast<uint32_t>(__builtin_ctz(mine)) * EPL + i % EPL;
        col = min(col, mine ? c : ~0u);
      }
      const int bidx = col == ~0u ? 0 : static_cast<int>(col);
      keep(best, bidx);
      // blank the winner in the lane that holds it
#pragma unroll
      for (int i = 0; i < VPT; ++i)
        if (bidx == (i / EPL) * (EPL * TPR) + t * EPL + i % EPL) v[i] = -10000.f;
    });
  }
  const int last = (K - 1) / TPR;   // pair j of a lane holds winner (last - j) * TPR + t
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (j > last) break;
    const int k = (last - j) * TPR + t;
    if (live && k < K) {
      const size_t o = static_cast<size_t>(row) * K + k;
      topk_w[o] = renormalize ? my_w[j] / wsum : my_w[j];
      topk_ids[o] = my_i[j];
      if (tok_exp_idx) tok_exp_idx[o] = k * T + row;
    }
  }
}

}  // namespace
