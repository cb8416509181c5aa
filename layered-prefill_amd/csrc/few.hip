// The expert MLP of a handful of tokens in two launches: routing with the gate-up pass, and the down pass with the
// top-k combine.
//
// Replaces, for calls of up to 16 tokens of the 16-bit dtypes, the chain of nanovllm/layers/fused_moe.py:163-216 and
// nanovllm/layers/for_moe/fused_moe.py:547-631 of the reference (select_experts, moe_align_block_size, two grouped GEMMs,
// moe_sum), with the bits of the kernels that run those steps here.
#include "common.h"
#include "gemm_device.h"
#include "routing_device.h"

#include <type_traits>

namespace {

constexpr int kFewTokens = 16;     // columns of a 16x16 product
constexpr int kFewFlats = 128;     // most (token, k)
constexpr int kFewCus = 256;
constexpr int kFewRow = 128;       // bytes of a row that a step takes: 64 elements
// Steps that a wavefront has in flight; a unit has more of them, so that its requests are at most one unit ahead.  Eight
// wavefronts of four steps: 1, 2 and 9 tokens of the layer below 21.0, 27.0 and 48.3 us; four of eight: 20.8, 28.7 and 50.6.
// A gate-up workgroup has twelve of them where its rings leave room for the hidden states, else eight: a CU's 8 to 12 units
// then go side by side instead of in two rounds.  Layer with the norm, three sets of weights, eight and twelve, us: 4
// tokens 40.1 and 40.3, 8 52.6 and 51.7, 9 57 and 56, 10 56.5 and 55.9; 32 experts, H 2048, I 1024, 12 tokens 74.0 and 72.9;
// H 4096, 4 tokens 101.8 and 98.1.
constexpr int kFewGateRing = 4, kFewDownRing = 4;
constexpr int kFewGateStep = 16 * kFewRow;                // 16 weight rows
constexpr int kFewDownStep = 2 * 16 * kFewRow;            // 16 weight rows and 16 token rows
constexpr int kFewXBytes = 64 * 1024;                     // most bytes of hidden states
constexpr int kFewXMost12 = 56 * 1024;                    // the same beside the rings of twelve wavefronts
constexpr int kFewLeastLds = 84 * 1024;                   // of which no two fit a CU

struct FewParams {
  const void *x, *w13, *w2, *b13, *b2;
  void *inter, *out;
  float* topk_w;
  int32_t* topk_ids;
  int32_t* experts;   // their number, then the experts that have a token, ascending
  int64_t w13_stride_e, w13_stride_n, w2_stride_e, w2_stride_n;
  int T, H, I, K;
  uint32_t cols8_rcp; // 2^32 / (I / 8) + 1
  int activation, interleaved, weight_on_input, w_tiled;
  float alpha, limit;
};

// The rank-th set bit of a mask of W words (there is one).
template <int W>
__device__ __forceinline__ int nth_set(const uint64_t (&m)[W], int rank) {
  int at = -1, before = 0;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    const int r = before + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m[i] >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m[i]), 0));
    const int lane = threadIdx.x & 63;
    const uint64_t hit = __ballot((m[i] >> lane & 1) != 0 && r == rank);
    if (hit) at = 64 * i + __builtin_ctzll(hit);
    before += __popcll(m[i]);
  }
  return at;
}

// A call of a few tokens is a chain of short kernels around the time that its experts' weights take to arrive.  Two of
// them go here: every workgroup of the gate-up pass routes the few rows by itself, so that neither a launch nor a trip of
// ids through memory stands in front of the weights, and nothing is aligned; and a workgroup of the down pass has all terms
// of its columns' sums.  The weights are cut evenly: a CU's share of a pass is within one wavefront's unit of every other's.
// Whole layer, us, replayed from a graph, against routing with alignment, two streaming passes and the combine (all of them
// with the weights asked for once, lds_dma16<true>); one set of weights again and again, and four in rotation:
//   E 128, H 2048, I 768, top-8, tiled: 1 token 26.3 -> 19.1 and 27.6 -> 21.5; 2 33.2 -> 25.7 and 34.3 -> 28.0; 9 50.7 ->
//   45.4 and 53.4 -> 48.5; 12 57.8 -> 55.1 and 57.6 -> 56.0
//   E 64, H 1024, I 384, top-4, tiled: 1 token 18.3 -> 10.9 and 18.6 -> 12.4, 16 21.8 -> 17.8 and 20.6 -> 17.5
//   E 32, H 4096, I 1024, top-8: 1 token 46.1 -> 41.5 and 47.4 -> 44.1; 4 83.4 -> 77.4 and 85.9 -> 79.6; 12 108.5 -> 106.4
//   and 114.5 -> 112.8
// (Weights that stay in the memory-side cache would come faster without the hint: that layer at 1 token 40.2 with one set,
// 54.1 with six in rotation, where it takes 42.7 and 45.2 here.)
// The line (moe_layer_few) is T * K <= 96: beyond, experts with more than eight tokens become common, whose weights the
// down pass goes through twice.
//
// Routing and gate-up pass.  One workgroup to a CU takes an equal share of the (expert, eight columns) units of the experts
// that have a token.  A wavefront streams the 16 weight rows of its unit on its own, without a barrier, and multiplies them
// with all tokens' hidden states, which stay in LDS; the tokens that the expert has are picked at the end.  UN: steps of 64
// elements an iteration (one where H is an odd number of them): two keep the chain of a wait, LDS reads, requests and
// dependent products short (H 1536, I 512, top-2: 12.9 -> 11.1 us at 1 token).  The products, their order and every
// rounding are the streaming kernel's.
template <int E, typename Mma, int UN, int NW>
__global__ __launch_bounds__(NW * kWave, 1) void few_gate_kernel(const void* __restrict__ logits, int logits_dtype, int renormalize,
                                                               const FewParams p) {
  using El = typename Mma::El;
  using G = Pow2Geom<E>;
  constexpr int RING = NW * kFewGateRing * kFewGateStep;
  constexpr int TPR = G::kTpr, RPW = G::kRowsPerWave, W = (E + 63) / 64;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  __shared__ int s_ids[kFewFlats], s_flag[E];
  __shared__ float s_w[kFewFlats];
  __shared__ uint32_t s_kmap[kFewTokens * E / 4];   // which of a token's k an expert is (ids that repeat: any of them), a byte each
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, lq = lane >> 4;
  const int T = p.T, K = p.K, numel = T * K, nu = p.H / 64;
  const uint32_t lds0 = lds_offset_of(smem);
  // hidden states: row t of step s at 128 * (s * T + t), eight rows a request
  {
    const int cells = T * nu;
    const uint32_t rcp = 65536u / T + 1;
    for (int j = wave; j * 8 < cells; j += NW) {
      int i = j * 8 + (lane >> 3);
      i = i < cells ? i : cells - 1;
      const int s = static_cast<int>((static_cast<uint32_t>(i) * rcp) >> 16), t = i - s * T;
      const uint32_t off = static_cast<uint32_t>(t) * (p.H * 2) + s * kFewRow + (((lane & 7) ^ ((t >> 1) & 7)) << 4);
      lds_dma16(static_cast<const char*>(p.x), off, __builtin_amdgcn_readfirstlane(lds0 + RING + j * 1024));
    }
  }
  for (int i = tid; i < kFewTokens * E / 4; i += (NW * kWave)) s_kmap[i] = ~0u;
  for (int i = tid; i < E; i += (NW * kWave)) s_flag[i] = 0;
  for (int r0 = wave * RPW; r0 < T; r0 += NW * RPW) {  // (whole wavefronts take part in a row's exchanges)
    const int row = r0 + lane / TPR, from = row < T ? row : T - 1;
    float v[G::kVpt];
    if (logits_dtype == MOE_BF16) load_row<E, ElemBF16>(static_cast<const uint16_t*>(logits), from, lane % TPR, v);
    else if (logits_dtype == MOE_F16) load_row<E, ElemF16>(static_cast<const uint16_t*>(logits), from, lane % TPR, v);
    else load_row<E, ElemF32>(static_cast<const float*>(logits), from, lane % TPR, v);
    route_row<E>(v, lane % TPR, row, row < T, s_w, s_ids, nullptr, T, K, renormalize);
  }
  wait_vmcnt<0>();  // the hidden states
  __syncthreads();
  if (tid < numel) {
    const int id = s_ids[tid], t = tid / K;
    reinterpret_cast<uint8_t*>(s_kmap)[t * E + id] = static_cast<uint8_t>(tid - t * K);
    s_flag[id] = 1;
    if (blockIdx.x == 0) {
      p.topk_ids[tid] = id;
      p.topk_w[tid] = s_w[tid];
    }
  }
  __syncthreads();
  uint64_t mask[W];
  int experts = 0;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    mask[i] = __ballot(64 * i + lane < E && s_flag[64 * i + lane < E ? 64 * i + lane : 0] != 0);
    if (blockIdx.x == 0 && wave == 0 && (mask[i] >> lane & 1))
      p.experts[1 + experts + __popcll(mask[i] & ((1ull << lane) - 1))] = 64 * i + lane;
    experts += __popcll(mask[i]);
  }
  if (blockIdx.x == 0 && tid == 0) p.experts[0] = experts;

  const int cols8 = p.I / 8;
  const uint32_t units = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(experts)) * cols8;
  const int begin_u = __builtin_amdgcn_readfirstlane(static_cast<int>(units * blockIdx.x / kFewCus));
  const int last = __builtin_amdgcn_readfirstlane(static_cast<int>(units * (blockIdx.x + 1) / kFewCus));  // (one behind)
  // no more wavefronts than share the units in as many rounds
  const int first = begin_u + wave;
  const int rounds = (last - begin_u + NW - 1) / NW;
  int stride = NW;
  while (rounds > 1 && (stride - 1) * rounds >= last - begin_u) --stride;
  if (wave >= stride || first >= last) return;
  // the side of a unit that asks for weights
  const char* w_at = nullptr;
  uint32_t w_off[2] = {0, 0};
  const int w_step = p.w_tiled ? 32768 : kFewRow;
  int e_ask = 0, c_ask = 0;
  auto begin = [&](int u) {
    int j = __umulhi(u, p.cols8_rcp);  // u / cols8, or one more
    c_ask = u - j * cols8;
    if (c_ask < 0) { j -= 1; c_ask += cols8; }
    e_ask = __builtin_amdgcn_readfirstlane(nth_set<W>(mask, j));
    w_at = static_cast<const char*>(p.w13) + static_cast<int64_t>(e_ask) * p.w13_stride_e * 2;
    if (p.w_tiled) w_at += static_cast<int64_t>(8 * c_ask / 128) * nu * 32768;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      // rows of a unit in the order g, g + 1, u, u + 1: a lane ends with gate and up of two columns
      const int r = 8 * q + (lane >> 3), col = 2 * (r >> 2) + (r & 1), half = (r >> 1) & 1;
      const int chunk = (lane & 7) ^ ((r >> 1) & 7);
      if (p.w_tiled) {
        const int R = half * 128 + 8 * c_ask % 128 + col;
        w_off[q] = static_cast<uint32_t>(R * kFewRow + ((chunk ^ ((R >> 1) & 7)) << 4));
      } else {
        const int n = 8 * c_ask + col;
        w_off[q] = static_cast<uint32_t>(p.interleaved ? 2 * n + half : half * p.I + n) * (static_cast<uint32_t>(p.w13_stride_n) * 2) + (chunk << 4);
      }
    }
  };
  constexpr int kRing = kFewGateRing / UN;
  const uint32_t ring = __builtin_amdgcn_readfirstlane(lds0 + wave * kRing * UN * kFewGateStep);
  const char* const ring_p = smem + wave * kRing * UN * kFewGateStep;
  int u_ask = first, k_ask = 0, at_ask = 0;
  auto ask = [&] {
#pragma unroll
    for (int q = 0; q < UN; ++q) {
      lds_dma16<true>(w_at, w_off[0], ring + at_ask + q * kFewGateStep);
      lds_dma16<true>(w_at, w_off[1], ring + at_ask + q * kFewGateStep + 1024);
      w_at += w_step;
    }
    at_ask = at_ask + UN * kFewGateStep == kRing * UN * kFewGateStep ? 0 : at_ask + UN * kFewGateStep;
    if ((k_ask += UN) == nu) {
      k_ask = 0;
      u_ask += stride;
      if (u_ask < last) begin(u_ask);
    }
  };
  begin(first);
  int e = e_ask, c = c_ask;
  for (int i = 0; i < kRing; ++i) ask();
  const int t = l15 < T ? l15 : T - 1;
  // a row of logits without a largest one has expert 0 at every k, and its first weight is no number (without
  // renormalisation only that one)
  const bool repeats = s_w[t * K] != s_w[t * K];
  int rd_w[2], rd_x[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    rd_w[kk] = l15 * kFewRow + (((4 * kk + lq) ^ ((l15 >> 1) & 7)) << 4);
    rd_x[kk] = RING + t * kFewRow + (((4 * kk + lq) ^ ((t >> 1) & 7)) << 4);
  }
  int at = 0;
  for (int u = first; u < last; u += stride) {
    // what the unit's end needs
    const int k_of = reinterpret_cast<const uint8_t*>(s_kmap)[t * E + e];
    const bool mine = l15 < T && k_of != 0xff;
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.b13) {
      const int32_t* b = reinterpret_cast<const int32_t*>(static_cast<const char*>(p.b13) + static_cast<int64_t>(e) * (2 * p.I) * 2) + (p.interleaved ? 8 * c : 4 * c);
      const int32_t* b2 = p.interleaved ? b + 4 : b + p.I / 2;
      int lo[4], hi[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) lo[i] = uniform_load(b + i), hi[i] = uniform_load(b2 + i);
      uint32_t g, v;
      if (p.interleaved) {   // words 2 lq and 2 lq + 1 of the eight: gate and up of a column each
        const uint32_t a0 = lq == 0 ? lo[0] : lq == 1 ? lo[2] : lq == 2 ? hi[0] : hi[2];
        const uint32_t a1 = lq == 0 ? lo[1] : lq == 1 ? lo[3] : lq == 2 ? hi[1] : hi[3];
        g = (a0 & 0xffffu) | (a1 << 16);
        v = (a0 >> 16) | (a1 & 0xffff0000u);
      } else {
        g = lq == 0 ? lo[0] : lq == 1 ? lo[1] : lq == 2 ? lo[2] : lo[3];
        v = lq == 0 ? hi[0] : lq == 1 ? hi[1] : lq == 2 ? hi[2] : hi[3];
      }
      bias[0] = unpack_lo<El>(g); bias[1] = unpack_hi<El>(g);
      bias[2] = unpack_lo<El>(v); bias[3] = unpack_hi<El>(v);
    }
    f32x4 acc;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = 0.f;
    int x_at = 0;
    for (int k = 0; k < nu; k += UN) {
      if (u_ask < last) wait_vmcnt<2 * UN * (kRing - 1)>();
      else wait_vmcnt<0>();
      uint4 w[UN][2], x[UN][2];
#pragma unroll
      for (int q = 0; q < UN; ++q)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          w[q][kk] = *reinterpret_cast<const uint4*>(ring_p + at + q * kFewGateStep + rd_w[kk]);
          x[q][kk] = *reinterpret_cast<const uint4*>(smem + x_at + q * T * kFewRow + rd_x[kk]);
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the place is read, the next request may land there
      if (u_ask < last) ask();
#pragma unroll
      for (int q = 0; q < UN; ++q)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) acc = Mma::mma16(w[q][kk], x[q][kk], acc);
      at = at + UN * kFewGateStep == kRing * UN * kFewGateStep ? 0 : at + UN * kFewGateStep;
      x_at += UN * T * kFewRow;
    }
    if (mine) {
      // (every k of a row whose ids repeat: the down pass reads all of them)
      for (int k = repeats ? 0 : k_of; k < (repeats ? K : k_of + 1); ++k) {
        const float rw = p.weight_on_input ? s_w[t * K + k] : 1.f;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = acc[i];
          if (p.b13) v[i] += bias[i];
          v[i] *= rw;
        }
        const uint32_t g = pack2<El>(v[0], v[1]), up = pack2<El>(v[2], v[3]);
        uint32_t o;
        if (p.activation == MOE_ACT_SILU) o = gated_pair<El, MOE_ACT_SILU>(p.alpha, p.limit, g, up);
        else if (p.activation == MOE_ACT_SWIGLUOAI) o = gated_pair<El, MOE_ACT_SWIGLUOAI>(p.alpha, p.limit, g, up);
        else o = gated_pair<El, MOE_ACT_GELU>(p.alpha, p.limit, g, up);
        *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(p.inter) + static_cast<int64_t>(t * K + k) * p.I + 8 * c + 2 * lq) = o;
      }
    }
    e = e_ask;
    c = c_ask;
  }
}

// Down pass and combine.  A workgroup owns eight output columns: their weight rows of every expert that has a token, and
// so every term of their sums, which meet in LDS.  A wavefront streams the rows of two experts beside their tokens' rows:
// the first eight columns of a product are the first expert's tokens, the others the second's (more than eight of one
// expert: a second time).  NW wavefronts: eight where a CU has one workgroup, four and two workgroups a CU where H has more
// than 256 times eight columns (H 4096, I 384, top-4: 19.9 -> 17.5 us at 1 token).
template <typename Mma, int UN, int NW>
__global__ __launch_bounds__(NW * kWave, NW == 4 ? 2 : 1) void few_down_kernel(const int32_t* __restrict__ experts, const int32_t* __restrict__ topk_ids,
                                                               const float* __restrict__ topk_w, const FewParams p) {
  using El = typename Mma::El;
  constexpr int HALVES = 2, COLS = 8, REQ = HALVES + 2;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  __shared__ uint16_t s_res[kFewFlats * 8];
  __shared__ float s_w[kFewFlats];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, lq = lane >> 4;
  const int T = p.T, K = p.K, numel = T * K, nu = p.I / 64;
  const int n0 = blockIdx.x * 8;
  const int count = uniform_load(experts);
  const int list[2] = {experts[1 + lane], experts[1 + 64 + lane]};      // (behind the last expert: not looked at)
  const int id[2] = {lane < numel ? topk_ids[lane] : -1, 64 + lane < numel ? topk_ids[64 + lane] : -1};
  if (tid < numel) s_w[tid] = topk_w[tid];
  __syncthreads();
  const int units = (count + HALVES - 1) / HALVES;
  const char* w_at[HALVES];
  uint32_t a_off[2] = {0, 0};
  bool a_live[2] = {false, false};
  const int w_step = p.w_tiled ? 32768 : kFewRow;
  int e_ask[HALVES], flat_ask = 0;   // flat (token, k) of this lane's column, plus one
  bool again = false;                // the unit has more tokens than columns (ids that repeat: rows of NaN)
#pragma unroll
  for (int h = 0; h < HALVES; ++h) w_at[h] = nullptr, e_ask[h] = 0;
  auto begin = [&](int u, int group) {
    int push = 0;
    again = false;
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
      const int j = HALVES * u + h, have = j < count ? j : count - 1;
      e_ask[h] = have < 64 ? __builtin_amdgcn_readlane(list[0], have) : __builtin_amdgcn_readlane(list[1], have & 63);
      w_at[h] = static_cast<const char*>(p.w2) + static_cast<int64_t>(e_ask[h]) * p.w2_stride_e * 2;
      if (p.w_tiled) w_at[h] += static_cast<int64_t>(n0 / 256) * nu * 32768;
      int before = 0;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint64_t m = j < count ? __ballot(id[i] == e_ask[h]) : 0;
        const int rank = before + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0)) - group * COLS;
        const bool in = (m >> lane & 1) != 0 && rank >= 0 && rank < COLS;
        push |= __builtin_amdgcn_ds_permute(4 * (in ? 8 * h + rank : 63), 64 * i + lane + 1);
        before += __popcll(m);
      }
      again |= before > (group + 1) * COLS;
    }
    flat_ask = __builtin_amdgcn_ds_bpermute(4 * l15, push);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int col = 8 * q + (lane >> 3);
      const int f = __builtin_amdgcn_ds_bpermute(4 * col, push);
      a_live[q] = f != 0 || lane == 0;   // lane 0 always: a request with no lane at all would not count
      a_off[q] = static_cast<uint32_t>(f ? f - 1 : 0) * (p.I * 2) + (((lane & 7) ^ ((col >> 1) & 7)) << 4);
    }
  };
  uint32_t w_lane[HALVES];
#pragma unroll
  for (int h = 0; h < HALVES; ++h) {
    const int i = lane >> 3, r = 8 * h + i, chunk = (lane & 7) ^ ((r >> 1) & 7);
    if (p.w_tiled) {
      const int R = n0 % 256 + i;
      w_lane[h] = static_cast<uint32_t>(R * kFewRow + ((chunk ^ ((R >> 1) & 7)) << 4));
    } else {
      w_lane[h] = static_cast<uint32_t>(n0 + i) * (static_cast<uint32_t>(p.w2_stride_n) * 2) + (chunk << 4);
    }
  }
  constexpr int kRing = kFewDownRing / UN;
  const uint32_t ring = __builtin_amdgcn_readfirstlane(lds_offset_of(smem) + wave * kRing * UN * kFewDownStep);
  const char* const ring_p = smem + wave * kRing * UN * kFewDownStep;
  int u_ask = wave, g_ask = 0, k_ask = 0, at_ask = 0;
  auto ask = [&] {
#pragma unroll
    for (int s = 0; s < UN; ++s) {
#pragma unroll
      for (int h = 0; h < HALVES; ++h) {
        lds_dma16<true>(w_at[h], w_lane[h], ring + at_ask + s * kFewDownStep + h * 1024);
        w_at[h] += w_step;
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (a_live[q]) lds_dma16(static_cast<const char*>(p.inter), a_off[q], ring + at_ask + s * kFewDownStep + 2048 + q * 1024);
        a_off[q] += kFewRow;
      }
    }
    at_ask = at_ask + UN * kFewDownStep == kRing * UN * kFewDownStep ? 0 : at_ask + UN * kFewDownStep;
    if ((k_ask += UN) == nu) {
      k_ask = 0;
      g_ask = again ? g_ask + 1 : 0;
      u_ask = again ? u_ask : u_ask + NW;
      if (u_ask < units) begin(u_ask, g_ask);
    }
  };
  if (u_ask < units) {
    begin(u_ask, 0);
    int e[HALVES], flat = flat_ask, at = 0;
#pragma unroll
    for (int h = 0; h < HALVES; ++h) e[h] = e_ask[h];
    int rd[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) rd[kk] = l15 * kFewRow + (((4 * kk + lq) ^ ((l15 >> 1) & 7)) << 4);
    for (int i = 0; i < kRing; ++i) ask();
    for (bool more = true; more;) {
      const int half = lq >> 1;
      float bias[4] = {0.f, 0.f, 0.f, 0.f};
      if (p.b2) {
        uint32_t b[2] = {0, 0};
#pragma unroll
        for (int h = 0; h < HALVES; ++h) {
          const int32_t* src = reinterpret_cast<const int32_t*>(static_cast<const char*>(p.b2) + (static_cast<int64_t>(e[h]) * p.H + n0) * 2);
          int q[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) q[i] = uniform_load(src + i);
          if (half == h) {
            b[0] = lq & 1 ? q[2] : q[0];
            b[1] = lq & 1 ? q[3] : q[1];
          }
        }
        bias[0] = unpack_lo<El>(b[0]); bias[1] = unpack_hi<El>(b[0]);
        bias[2] = unpack_lo<El>(b[1]); bias[3] = unpack_hi<El>(b[1]);
      }
      f32x4 acc;
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = 0.f;
      for (int k = 0; k < nu; k += UN) {
        if (u_ask < units) wait_vmcnt<REQ * UN * (kRing - 1)>();
        else wait_vmcnt<0>();
        uint4 w[UN][2], x[UN][2];
#pragma unroll
        for (int q = 0; q < UN; ++q)
#pragma unroll
          for (int kk = 0; kk < 2; ++kk) {
            w[q][kk] = *reinterpret_cast<const uint4*>(ring_p + at + q * kFewDownStep + rd[kk]);
            x[q][kk] = *reinterpret_cast<const uint4*>(ring_p + at + q * kFewDownStep + 2048 + rd[kk]);
          }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the place is read, the next request may land there
        if (u_ask < units) ask();
#pragma unroll
        for (int q = 0; q < UN; ++q)
#pragma unroll
          for (int kk = 0; kk < 2; ++kk) acc = Mma::mma16(w[q][kk], x[q][kk], acc);
        at = at + UN * kFewDownStep == kRing * UN * kFewDownStep ? 0 : at + UN * kFewDownStep;
      }
      if (flat && (l15 >> 3) == half) {
        const float rw = p.weight_on_input ? 1.f : s_w[flat - 1];
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = acc[i];
          if (p.b2) v[i] += bias[i];
          v[i] *= rw;
        }
        *reinterpret_cast<uint2*>(s_res + (flat - 1) * 8 + 4 * (lq & 1)) = uint2{pack2<El>(v[0], v[1]), pack2<El>(v[2], v[3])};
      }
      more = u_ask < units;   // the requests are inside the next unit, if there is one
      flat = flat_ask;
#pragma unroll
      for (int h = 0; h < HALVES; ++h) e[h] = e_ask[h];
    }
  }
  __syncthreads();
  if (tid < T * 8) {
    const int t = tid >> 3, col = tid & 7;
    float sum = 0.f;
    for (int k = 0; k < K; ++k) sum += El::ld(s_res[(t * K + k) * 8 + col]);
    static_cast<uint16_t*>(p.out)[static_cast<int64_t>(t) * p.H + n0 + col] = El::st(sum);
  }
}

template <int E, typename Mma>
int launch_few(const void* logits, int logits_dtype, int renormalize, const FewParams& p, hipStream_t s) {
  const int x_bytes = (p.T * (p.H / 64) + 7) / 8 * 1024;
  auto gate = [&](auto un, auto nw) {
    constexpr int NW = decltype(nw)::value, ring = NW * kFewGateRing * kFewGateStep;
    static MoeLdsOptIn flags;
    auto kernel = few_gate_kernel<E, Mma, decltype(un)::value, NW>;
    const int lds = ring + x_bytes > kFewLeastLds ? ring + x_bytes : kFewLeastLds;
    if (int rc = moe_opt_in_lds(flags, reinterpret_cast<const void*>(kernel), ring + (NW > 8 ? kFewXMost12 : kFewXBytes), "layer"))
      return rc;
    hipLaunchKernelGGL(kernel, dim3(kFewCus), dim3(NW * kWave), lds, s, logits, logits_dtype, renormalize, p);
    return moe_check_launch("layer (routing and gate-up pass)");
  };
  auto down = [&](auto un, auto nw) {
    constexpr int UN = decltype(un)::value, NW = decltype(nw)::value, bytes = NW * kFewDownRing * kFewDownStep;
    static MoeLdsOptIn flags;
    auto kernel = few_down_kernel<Mma, UN, NW>;
    if (int rc = moe_opt_in_lds(flags, reinterpret_cast<const void*>(kernel), bytes, "layer")) return rc;
    hipLaunchKernelGGL(kernel, dim3(p.H / 8), dim3(NW * kWave), bytes, s, p.experts, p.topk_ids, p.topk_w, p);
    return moe_check_launch("layer (down pass and combine)");
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  using Four = std::integral_constant<int, 4>;
  using Eight = std::integral_constant<int, 8>;
  using Twelve = std::integral_constant<int, 12>;
  const bool wide = x_bytes <= kFewXMost12;
  const int rc = p.H % 128 ? (wide ? gate(One{}, Twelve{}) : gate(One{}, Eight{})) : wide ? gate(Two{}, Twelve{}) : gate(Two{}, Eight{});
  if (rc) return rc;
  const bool many = p.H / 8 > kFewCus;
  if (p.I % 128) return many ? down(One{}, Four{}) : down(One{}, Eight{});
  return many ? down(Two{}, Four{}) : down(Two{}, Eight{});
}

}  // namespace

bool moe_layer_few(const MoeLayerArgs* a, float* topk_w, int32_t* topk_ids, int32_t* experts, void* inter, int* rc) {
  const int64_t numel = static_cast<int64_t>(a->T) * a->K;
  // (a block size of the caller's own names the kernel that is meant)
  if (!a->router_logits || a->block_size || a->T > kFewTokens || numel > 96 || a->K > 16 || a->K > a->E || a->K < 1) return false;
  if ((a->act_dtype != MOE_BF16 && a->act_dtype != MOE_F16) || a->weight_dtype != a->act_dtype) return false;
  if (a->logits_dtype != MOE_BF16 && a->logits_dtype != MOE_F16 && a->logits_dtype != MOE_F32) return false;
  if (a->activation < MOE_ACT_SILU || a->activation > MOE_ACT_GELU) return false;
  if (a->H % 64 || a->I % 64 || a->H <= 64 * kFewGateRing || a->I <= 64 * kFewDownRing) return false;
  if (static_cast<int64_t>(a->T) * a->H * 2 > kFewXBytes || a->I > (1 << 18)) return false;
  if (a->w13_stride_n % 8 || a->w2_stride_n % 8 || (a->E > 1 && (a->w13_stride_e % 8 || a->w2_stride_e % 8))) return false;
  const int64_t span = (1LL << 32) - 16384;  // of the lanes' 32-bit offsets
  if (a->w13_stride_n < a->H || a->w2_stride_n < a->I || 2LL * a->I * a->w13_stride_n * 2 >= span || static_cast<int64_t>(a->H) * a->w2_stride_n * 2 >= span) return false;
  if ((reinterpret_cast<uintptr_t>(a->x) | reinterpret_cast<uintptr_t>(a->w13) | reinterpret_cast<uintptr_t>(a->w2) |
       reinterpret_cast<uintptr_t>(a->out)) & 15u)
    return false;
  if ((reinterpret_cast<uintptr_t>(a->w13_bias) | reinterpret_cast<uintptr_t>(a->w2_bias)) & 3u) return false;
  const bool tiled = a->weight_layout == MOE_WEIGHTS_TILED;
  if (a->weight_layout != MOE_WEIGHTS_PLAIN && !tiled) return false;
  if (tiled && (a->I % 128 || a->H % 256 || a->w13_stride_n != a->H || a->w13_stride_e != 2LL * a->I * a->H ||
                a->w2_stride_n != a->I || a->w2_stride_e != static_cast<int64_t>(a->H) * a->I))
    return false;   // (named as an error by moe_fused_experts)
  FewParams p{};
  p.x = a->x; p.w13 = a->w13; p.w2 = a->w2; p.b13 = a->w13_bias; p.b2 = a->w2_bias;
  p.inter = inter; p.out = a->out; p.topk_w = topk_w; p.topk_ids = topk_ids; p.experts = experts;
  p.w13_stride_e = a->w13_stride_e; p.w13_stride_n = a->w13_stride_n;
  p.w2_stride_e = a->w2_stride_e; p.w2_stride_n = a->w2_stride_n;
  p.T = a->T; p.H = a->H; p.I = a->I; p.K = a->K;
  p.cols8_rcp = static_cast<uint32_t>((1LL << 32) / (a->I / 8) + 1);
  p.activation = a->activation; p.interleaved = a->activation == MOE_ACT_SWIGLUOAI;
  p.weight_on_input = a->apply_router_weight_on_input; p.w_tiled = tiled;
  p.alpha = a->swiglu_alpha; p.limit = a->swiglu_limit;
  hipStream_t s = static_cast<hipStream_t>(a->stream);
  auto go = [&](auto tag) {
    constexpr int E = decltype(tag)::value;
    *rc = a->act_dtype == MOE_BF16 ? launch_few<E, MmaBF16>(a->router_logits, a->logits_dtype, a->renormalize, p, s)
                                   : launch_few<E, MmaF16>(a->router_logits, a->logits_dtype, a->renormalize, p, s);
    return true;
  };
  switch (a->E) {
    case 32: return go(std::integral_constant<int, 32>{});
    case 64: return go(std::integral_constant<int, 64>{});
    case 128: return go(std::integral_constant<int, 128>{});
    case 256: return go(std::integral_constant<int, 256>{});
    default: return false;
  }
}
