// Router: row softmax over E experts + K rounds of argmax, one launch.
//
// Replaces topkGatingSoftmax / moeSoftmax + moeTopK of the reference
// (csrc/moe_topk_softmax_kernels.cu:50-166,182-380, dispatch :421-471).
// For power-of-two E <= 256 a row is shared by the same number of lanes, with
// the same column-to-lane assignment and the same butterfly order, as in the
// reference's fused kernel, so the fp32 sum has the same association; the
// 64-lane wavefront simply carries twice as many rows as a 32-lane warp.
// Any other E takes one wavefront per row: in registers up to 1024 columns, in LDS up to 16384.
#include <stdarg.h>

#include <type_traits>

#include "common.h"
#include "quant_device.h"
#include "routing_device.h"

namespace {

template <int E, typename El>
__global__ __launch_bounds__(kWave* kWavesPerBlock) void topk_softmax_pow2_kernel(
    const typename El::S* __restrict__ gating, float* __restrict__ topk_w, int32_t* __restrict__ topk_ids,
    int32_t* __restrict__ tok_exp_idx, int T, int K, int renormalize) {
  using G = Pow2Geom<E>;
  constexpr int VPT = G::kVpt, TPR = G::kTpr;
  const int lane = threadIdx.x % kWave;
  const int wave = threadIdx.x / kWave;
  const int row = (blockIdx.x * kWavesPerBlock + wave) * G::kRowsPerWave + lane / TPR;
  const int t = lane % TPR;
  const bool live = row < T;
  const int ld_row = live ? row : (T - 1);

  float v[VPT];
  load_row<E, El>(gating, ld_row, t, v);
  route_row<E>(v, t, row, live, topk_w, topk_ids, tok_exp_idx, T, K, renormalize);
}

// The same with the e4m3 codes of x beside it, which wait for nothing either: the first `route_blocks` workgroups route,
// the others quantise a row per wavefront.  One launch less, and the router, a chain of latencies, hides behind a copy's
// traffic.  Whole layer, us, 128 experts, H 2048, I 768, top-8, with the codes in a launch of their own and here: 1 token
// 24.6 and 22.7, 16 40.3 and 38.2, 100 69.7 and 67.5, 741 155.5 and 152.4, 8448 539 and 528.
template <int E, typename El, int NV>
__global__ __launch_bounds__(kWave* kWavesPerBlock) void topk_softmax_quant_kernel(
    const typename El::S* __restrict__ gating, float* __restrict__ topk_w, int32_t* __restrict__ topk_ids, int T, int K,
    int renormalize, int route_blocks, const typename El::S* __restrict__ x, int H, uint8_t* __restrict__ codes,
    float* __restrict__ scales) {
  using G = Pow2Geom<E>;
  constexpr int VPT = G::kVpt, TPR = G::kTpr;
  const int lane = threadIdx.x % kWave;
  const int wave = threadIdx.x / kWave;
  if (static_cast<int>(blockIdx.x) >= route_blocks) {
    const int64_t row = static_cast<int64_t>(blockIdx.x - route_blocks) * kWavesPerBlock + wave;
    if (row < T) quant_row<El, NV, kWave>(x + row * H, lane, H, codes + row * H, scales + row);
    return;
  }
  const int row = (blockIdx.x * kWavesPerBlock + wave) * G::kRowsPerWave + lane / TPR;
  float v[VPT];
  load_row<E, El>(gating, row < T ? row : T - 1, lane % TPR, v);
  route_row<E>(v, lane % TPR, row, row < T, topk_w, topk_ids, nullptr, T, K, renormalize);
}

// ---------------------------------------------------------------------------
// Router gate fused in front: logits = x . Wg^T (the reference's ReplicatedLinear,
// nanovllm/models/qwen3_moe.py:93-104, whose output has the activation dtype),
// rounded to that dtype, then the same softmax / top-k as above, without the
// logits ever leaving the CU.  A workgroup takes 32 tokens and all E experts
// and walks K in units of 64 elements: the unit's 32 token rows and E gate rows
// (128 bytes each) go global->LDS by DMA into a ring of four units, full
// 128-byte lines per request (operands fetched straight into MFMA register
// layout touch 64 different lines per wavefront load and ran 3x slower than the
// separate GEMM + routing kernels).  Wavefront f multiplies expert fragment f
// (MFMA 32x32x16, experts as the A operand, tokens as B); the rounded logits
// are laid out in LDS as [token][expert] and routed from there with the lane
// layout of the stand-alone kernel.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(8))) __bf16 gate_bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 gate_f16x8;
typedef __attribute__((ext_vector_type(16))) float gate_f32x16;
typedef __attribute__((address_space(3))) char gate_lds_char;

template <typename El>
__device__ __forceinline__ gate_f32x16 gate_mma(const uint4& a, const uint4& b, gate_f32x16 c);
template <>
__device__ __forceinline__ gate_f32x16 gate_mma<ElemBF16>(const uint4& a, const uint4& b, gate_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(gate_bf16x8, a),
                                                 __builtin_bit_cast(gate_bf16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ gate_f32x16 gate_mma<ElemF16>(const uint4& a, const uint4& b, gate_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(gate_f16x8, a),
                                                __builtin_bit_cast(gate_f16x8, b), c, 0, 0, 0);
}

// 16 bytes per lane from global memory straight into LDS at lds_wave_base + 16 * lane
// (issued from assembly: the compiler would order every later LDS read behind it with vmcnt(0))
__device__ __forceinline__ void gate_dma16(const char* base, uint32_t lane_byte_offset, uint32_t lds_wave_base) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2"
      :
      : "s"(lds_wave_base), "v"(lane_byte_offset), "s"(base)
      : "memory");
}

constexpr int kGateTokens = 32, kGateRowBytes = 128;

constexpr int kGateWaves = 16;  // wavefronts 0..3 stream and multiply; all sixteen route (two rows each)

template <typename El, int E, int kGateRing>
__global__ __launch_bounds__(kWave* kGateWaves) void gate_topk_softmax_kernel(
    const typename El::S* __restrict__ x, const typename El::S* __restrict__ wg,
    float* __restrict__ logits_out, float* __restrict__ topk_w, int32_t* __restrict__ topk_ids,
    int32_t* __restrict__ tok_exp_idx, int T, int H, int K, int renormalize) {
  using G = Pow2Geom<E>;
  constexpr int NF = E / 32;                         // expert fragments = computing wavefronts
  constexpr int WJ = E / 32;                         // gate-row requests per wavefront and unit
  constexpr int kWBytes = E * kGateRowBytes;
  constexpr int kUnitBytes = kWBytes + kGateTokens * kGateRowBytes;
  constexpr int kDma = WJ + 1;                       // requests per wavefront and unit
  static_assert(NF >= 1 && NF <= kWavesPerBlock, "one expert fragment per wavefront");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int l32 = lane & 31, lhi = lane >> 5;
  const int t0 = blockIdx.x * kGateTokens;

  // DMA: a request covers 8 rows x 128 bytes; lane / 8 is the row, lane % 8 the 16-byte chunk
  // it lands in; chunk c of row r holds logical chunk c ^ ((r >> 1) & 7) (bank spreading)
  const int q = lane >> 3;
  uint32_t a_off, w_off[WJ];
  {
    const int rr = 8 * wave + q;
    const int row = t0 + rr < T ? t0 + rr : T - 1;
    a_off = static_cast<uint32_t>(static_cast<size_t>(row) * H * 2 + (((lane & 7) ^ ((rr >> 1) & 7)) << 4));
  }
#pragma unroll
  for (int j = 0; j < WJ; ++j) {
    const int rr = (E / 4) * wave + 8 * j + q;
    w_off[j] = static_cast<uint32_t>(static_cast<size_t>(rr) * H * 2 + (((lane & 7) ^ ((rr >> 1) & 7)) << 4));
  }
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const gate_lds_char*)smem));
  const uint32_t dma_w = __builtin_amdgcn_readfirstlane(lds0 + (E / 4) * wave * kGateRowBytes);
  const uint32_t dma_a = __builtin_amdgcn_readfirstlane(lds0 + kWBytes + 8 * wave * kGateRowBytes);
  const char* xb = reinterpret_cast<const char*>(x);
  const char* wb = reinterpret_cast<const char*>(wg);
  const bool worker = wave < kWavesPerBlock;  // the other wavefronts only keep the barriers company
  auto issue = [&](int u) {
    if (!worker) return;
    const uint32_t ring = (u % kGateRing) * kUnitBytes;
    gate_dma16(xb + u * kGateRowBytes, a_off, dma_a + ring);
#pragma unroll
    for (int j = 0; j < WJ; ++j) gate_dma16(wb + u * kGateRowBytes, w_off[j], dma_w + ring + j * 1024);
  };
  int rd_k[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) rd_k[kk] = l32 * kGateRowBytes + (((2 * kk + lhi) ^ ((l32 >> 1) & 7)) << 4);

  gate_f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  const int nu = H / 64;
  constexpr int AHEAD = kGateRing - 1;  // units in flight
#pragma unroll
  for (int u = 0; u < AHEAD; ++u)
    if (u < nu) issue(u);
  for (int u = 0; u < nu; ++u) {
    // unit u has landed (only the AHEAD-1 younger units may be outstanding; near the end
    // fewer are, and waiting for all of them is as good); everybody has left unit u-1
    if (u + AHEAD - 1 < nu) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((AHEAD - 1) * kDma) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    if (u + AHEAD < nu) issue(u + AHEAD);
    if (worker && wave < NF) {
      const char* st = smem + (u % kGateRing) * kUnitBytes;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const uint4 xf = *reinterpret_cast<const uint4*>(st + kWBytes + rd_k[kk]);
        const uint4 wf = *reinterpret_cast<const uint4*>(st + wave * 32 * kGateRowBytes + rd_k[kk]);
        acc = gate_mma<El>(wf, xf, acc);
      }
    }
  }
  __syncthreads();  // the ring is free: it now holds the logits, [token][expert] fp32
  float* lg = reinterpret_cast<float*>(smem);
  if (worker && wave < NF) {
    // acc[r]: expert 32 wave + 8 (r / 4) + 4 lhi + r % 4, token l32; one rounding to the activation dtype
#pragma unroll
    for (int r = 0; r < 16; ++r)
      lg[l32 * E + wave * 32 + 8 * (r / 4) + 4 * lhi + (r % 4)] = El::ld(El::st(acc[r]));
  }
  __syncthreads();
  if (logits_out) {
    for (int i = threadIdx.x; i < kGateTokens * E; i += kWave * kGateWaves) {
      const int row = t0 + i / E;
      if (row < T) logits_out[static_cast<size_t>(row) * E + i % E] = lg[i];
    }
  }
  // routing, rows in the stand-alone kernel's lane layout
  constexpr int EPL = G::kEpl, VECS = G::kVecs, VPT = G::kVpt, TPR = G::kTpr, RPW = G::kRowsPerWave;
  const int t = lane % TPR;
  for (int r0 = wave * RPW; r0 < kGateTokens; r0 += kGateWaves * RPW) {
    const int lrow = r0 + lane / TPR;
    const int row = t0 + lrow;
    float v[VPT];
#pragma unroll
    for (int j = 0; j < VECS; ++j)
#pragma unroll
      for (int i = 0; i < EPL; ++i) v[j * EPL + i] = lg[lrow * E + j * EPL * TPR + t * EPL + i];
    route_row<E>(v, t, row, row < T, topk_w, topk_ids, tok_exp_idx, T, K, renormalize);
  }
}

template <typename El, int E>
int launch_gate(const void* x, const void* wg, float* logits_out, float* w, int32_t* ids,
                 int32_t* tei, int T, int H, int K, int renorm, hipStream_t s) {
  using S = typename El::S;
  const int blocks = (T + kGateTokens - 1) / kGateTokens;
  // few workgroups (decode): one per CU with a deep ring, 140 KB at E = 128; many: two per CU, 80 KB
  if (blocks <= 256) {
    constexpr int lds = 7 * (E + kGateTokens) * kGateRowBytes;
    auto kern = gate_topk_softmax_kernel<El, E, 7>;
    static MoeLdsOptIn opted;
    if (int rc = moe_opt_in_lds(opted, reinterpret_cast<const void*>(kern), lds, "gate_topk_softmax")) return rc;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(kWave * kGateWaves), lds, s,
                       static_cast<const S*>(x), static_cast<const S*>(wg), logits_out, w, ids, tei, T, H, K, renorm);
  } else {
    constexpr int lds = 4 * (E + kGateTokens) * kGateRowBytes;
    auto kern = gate_topk_softmax_kernel<El, E, 4>;
    static MoeLdsOptIn opted;
    if (int rc = moe_opt_in_lds(opted, reinterpret_cast<const void*>(kern), lds, "gate_topk_softmax")) return rc;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(kWave * kGateWaves), lds, s,
                       static_cast<const S*>(x), static_cast<const S*>(wg), logits_out, w, ids, tei, T, H, K, renorm);
  }
  return MOE_OK;
}

template <typename El>
int launch_gate_e(const void* x, const void* wg, float* logits_out, float* w, int32_t* ids,
                  int32_t* tei, int T, int H, int E, int K, int renorm, hipStream_t s) {
  switch (E) {
    case 32: if (int rc = launch_gate<El, 32>(x, wg, logits_out, w, ids, tei, T, H, K, renorm, s)) return rc; break;
    case 64: if (int rc = launch_gate<El, 64>(x, wg, logits_out, w, ids, tei, T, H, K, renorm, s)) return rc; break;
    case 128: if (int rc = launch_gate<El, 128>(x, wg, logits_out, w, ids, tei, T, H, K, renorm, s)) return rc; break;
    default: return moe_fail(MOE_ERR_UNSUPPORTED, "gate_topk_softmax: num_experts %d (32, 64 or 128)", E);
  }
  return moe_check_launch("gate_topk_softmax");
}

// ---------------------------------------------------------------------------
// The same for up to a few hundred tokens, as two short kernels.  A workgroup of the kernel above pulls all E gate rows
// through one CU, which a CU does at 37 bytes a nanosecond (E 128, H 2048: 512 KB, 17 us, whatever T).  Here the gate
// linear is cut in tokens, experts and K: a workgroup takes 16 (32) tokens by 16 (32) experts by 512 elements of K,
// everything it reads (32 or 64 KB) is on its way at once, its four wavefronts multiply straight out of registers (MFMA 16x16x32, gate rows as
// the A operand; a wavefront's two units of 64 elements fill whole lines) and add up in LDS.  The sums of the K pieces
// leave in fp32; the kernel that routes adds them, rounds the logit once, to the activation dtype, as the output of a
// gate linear is, and goes on with the lane layout of the stand-alone router.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(4))) float gate_f32x4;
template <typename El>
__device__ __forceinline__ gate_f32x4 gate_mma16(const uint4& a, const uint4& b, gate_f32x4 c) {
  if constexpr (std::is_same_v<El, ElemBF16>)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gate_bf16x8, a), __builtin_bit_cast(gate_bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(gate_f16x8, a), __builtin_bit_cast(gate_f16x8, b), c, 0, 0, 0);
}
constexpr int kPieceUnits = 8;                     // units of 64 elements in a piece of K
constexpr int kPieceWaves = 4, kPieceThreads = kWave * kPieceWaves;
static int gate_pieces(int H) { return (H / 64 + kPieceUnits - 1) / kPieceUnits; }
static int64_t gate_small_tiles(int T, int H, int E) {
  return (static_cast<int64_t>(T) + 15) / 16 * (E / 16) * gate_pieces(H);
}

// grid: token tiles x (pieces x expert tiles), the latter fastest, so that a gate piece stays with one XCD's L2.  Tiles of
// 16 M tokens by 16 N experts.
template <typename El, int M, int N>
__global__ __launch_bounds__(kPieceThreads) void gate_piece_kernel(
    const typename El::S* __restrict__ x, const typename El::S* __restrict__ wg, float* __restrict__ sums, int T, int H, int E,
    int pieces) {
  constexpr int ROW = 16 * N + 4;  // floats of a token in LDS, padded: the sixteen tokens of a store spread over the banks
  __shared__ __attribute__((aligned(16))) float part[kPieceWaves][16 * M][ROW];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int l15 = lane & 15, lq = lane >> 4;
  const int et = E / (16 * N), per_token_tile = pieces * et;
  const int t0 = blockIdx.x / per_token_tile * (16 * M), rest = blockIdx.x % per_token_tile;
  const int piece = rest / et, e0 = rest % et * (16 * N);
  const int nu = H / 64;
  const typename El::S *xr[M], *wr[N];
#pragma unroll
  for (int m = 0; m < M; ++m) xr[m] = x + static_cast<size_t>(min(t0 + 16 * m + l15, T - 1)) * H + lq * 8;
#pragma unroll
  for (int n = 0; n < N; ++n) wr[n] = wg + static_cast<size_t>(e0 + 16 * n + l15) * H + lq * 8;
  gate_f32x4 acc[M][N];
  uint4 xf[4][M], wf[4][N];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const int u = piece * kPieceUnits + 2 * wave + (kk >> 1);  // a unit behind the end of K: zeros
    const size_t k = static_cast<size_t>(u) * 64 + (kk & 1) * 32;
#pragma unroll
    for (int n = 0; n < N; ++n) wf[kk][n] = u < nu ? *reinterpret_cast<const uint4*>(wr[n] + k) : uint4{0, 0, 0, 0};
#pragma unroll
    for (int m = 0; m < M; ++m) xf[kk][m] = u < nu ? *reinterpret_cast<const uint4*>(xr[m] + k) : uint4{0, 0, 0, 0};
  }
  __builtin_amdgcn_sched_barrier(0);  // all requests first
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int n = 0; n < N; ++n) {
      acc[m][n] = gate_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) acc[m][n] = gate_mma16<El>(wf[kk][n], xf[kk][m], acc[m][n]);
      // element i: token 16 m + l15, expert 16 n + 4 lq + i
      *reinterpret_cast<gate_f32x4*>(&part[wave][16 * m + l15][16 * n + 4 * lq]) = acc[m][n];
    }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < M * N; ++r) {
    const int at = r * kPieceThreads + threadIdx.x, tok = at / (16 * N), col = at % (16 * N);
    if (t0 + tok < T)
      sums[(static_cast<size_t>(piece) * T + t0 + tok) * E + e0 + col] =
          (part[0][tok][col] + part[1][tok][col]) + (part[2][tok][col] + part[3][tok][col]);
  }
}

template <int E, typename El>
__global__ __launch_bounds__(kWave* kWavesPerBlock) void topk_softmax_sums_kernel(
    const float* __restrict__ sums, float* __restrict__ topk_w, int32_t* __restrict__ topk_ids,
    int32_t* __restrict__ tok_exp_idx, int T, int K, int renormalize, int pieces) {
  using G = Pow2Geom<E>;
  constexpr int VPT = G::kVpt, TPR = G::kTpr;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int row = (blockIdx.x * kWavesPerBlock + wave) * G::kRowsPerWave + lane / TPR;
  const bool live = row < T;
  const int ld_row = live ? row : (T - 1);
  float v[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) v[i] = 0.f;
  for (int p0 = 0; p0 < pieces; p0 += 4) {
    float q[4][VPT];
#pragma unroll
    for (int j = 0; j < 4; ++j) load_row<E>(sums + static_cast<size_t>(min(p0 + j, pieces - 1)) * T * E, ld_row, lane % TPR, q[j]);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (p0 + j < pieces)
#pragma unroll
        for (int i = 0; i < VPT; ++i) v[i] += q[j][i];
  }
#pragma unroll
  for (int i = 0; i < VPT; ++i) v[i] = El::ld(El::st(v[i]));
  route_row<E>(v, lane % TPR, row, live, topk_w, topk_ids, tok_exp_idx, T, K, renormalize);
}

template <int E, typename El>
int launch_gate_pieces(const void* x, const void* wg, float* sums, float* w, int32_t* ids, int32_t* tei, int T, int H, int K,
                       int renorm, hipStream_t s) {
  using S = typename El::S;
  const int pieces = gate_pieces(H);
  auto go = [&](auto kernel, int tokens, int experts) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((T + tokens - 1) / tokens) * pieces * (E / experts)), dim3(kPieceThreads),
                       0, s, static_cast<const S*>(x), static_cast<const S*>(wg), sums, T, H, E, pieces);
  };
  // Up to 512 small tiles, two a CU, are done sooner than an eighth as many large ones; beyond, what they read twice as
  // often counts.  us, gate and router, tiles of 16 and of 32: E 128, H 2048: 7.8 and 8.4 at 135 tokens, 8.1 and 8.4 at 256
  // (512 tiles of 16), 9.1 and 8.5 at 384, 10.0 and 8.7 at 512; E 32: 7.3 and 7.6 at 1024 tokens (512); E 64, H 4096: 8.3
  // and 8.6 at 256 (512), 10.2 and 8.9 at 512.
  if (gate_small_tiles(T, H, E) > 512) go(gate_piece_kernel<El, 2, 2>, 32, 32);
  else go(gate_piece_kernel<El, 1, 1>, 16, 16);
  constexpr int rows = kWavesPerBlock * Pow2Geom<E>::kRowsPerWave;
  hipLaunchKernelGGL((topk_softmax_sums_kernel<E, El>), dim3((T + rows - 1) / rows), dim3(kWave * kWavesPerBlock), 0, s, sums, w,
                     ids, tei, T, K, renorm, pieces);
  return moe_check_launch("gate_topk_softmax (pieces of K)");
}

// One wavefront per row; lane l holds columns l, l+64, ... (up to 16 of them).
constexpr int kGenericMaxPerLane = 16;

template <typename El>
__global__ __launch_bounds__(kWave* kWavesPerBlock) void topk_softmax_generic_kernel(
    const typename El::S* __restrict__ gating, float* __restrict__ topk_w, int32_t* __restrict__ topk_ids,
    int32_t* __restrict__ tok_exp_idx, int T, int E, int K, int renormalize) {
  const int lane = threadIdx.x % kWave;
  const int row = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
  const bool live = row < T;
  const typename El::S* src = gating + static_cast<size_t>(live ? row : T - 1) * E;
  const float ninf = -__builtin_inff();

  float v[kGenericMaxPerLane];
  float mx = ninf;
#pragma unroll
  for (int j = 0; j < kGenericMaxPerLane; ++j) {
    const int c = lane + j * kWave;
    v[j] = c < E ? El::ld(src[c]) : ninf;
    mx = fmaxf(mx, v[j]);
  }
#pragma unroll
  for (int m = 32; m > 0; m /= 2) mx = fmaxf(mx, __shfl_xor(mx, m, kWave));
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < kGenericMaxPerLane; ++j) {
    const int c = lane + j * kWave;
    if (c < E) {
      v[j] = moe_expf<true>(v[j] - mx);
      sum += v[j];
    }
  }
#pragma unroll
  for (int m = 32; m > 0; m /= 2) sum += __shfl_xor(sum, m, kWave);
  const float rinv = 1.f / sum;
#pragma unroll
  for (int j = 0; j < kGenericMaxPerLane; ++j) {
    const int c = lane + j * kWave;
    const float p = v[j] * rinv;
    v[j] = c < E ? p : -20000.f;  // columns past E can never win
  }

  float wsum = 0.f;
  for (int k = 0; k < K; ++k) {
    float best = v[0];
    int bidx = lane;
#pragma unroll
    for (int j = 1; j < kGenericMaxPerLane; ++j)
      if (v[j] > best) { best = v[j]; bidx = lane + j * kWave; }
#pragma unroll
    for (int m = 32; m > 0; m /= 2) {
      float ov = __shfl_xor(best, m, kWave);
      int oi = __shfl_xor(bidx, m, kWave);
      if (ov > best || (ov == best && oi < bidx)) { best = ov; bidx = oi; }
    }
    if (live && lane == 0) {
      const size_t o = static_cast<size_t>(row) * K + k;
      topk_w[o] = best;
      topk_ids[o] = bidx;
      if (tok_exp_idx) tok_exp_idx[o] = k * T + row;
    }
    wsum += best;
#pragma unroll
    for (int j = 0; j < kGenericMaxPerLane; ++j)
      if (lane == bidx % kWave && j == bidx / kWave) v[j] = -10000.f;
  }
  if (renormalize && live && lane == 0) {
    for (int k = 0; k < K; ++k) {
      const size_t o = static_cast<size_t>(row) * K + k;
      topk_w[o] = topk_w[o] / wsum;
    }
  }
}

// Wider rows (more columns than 64 lanes x 16 registers): one wavefront per row,
// the row's probabilities in LDS.  Lane l owns columns l, l+64, ... exactly as in
// the register kernel above, so the order of every max, sum and comparison is the
// same; every LDS word is read and written by its owning lane only, which is why
// no barrier appears.
constexpr int kWideMaxExperts = 16384;  // 64 KiB of LDS per row

template <typename El>
__global__ __launch_bounds__(kWave) void topk_softmax_wide_kernel(
    const typename El::S* __restrict__ gating, float* __restrict__ topk_w, int32_t* __restrict__ topk_ids,
    int32_t* __restrict__ tok_exp_idx, int T, int E, int K, int renormalize) {
  extern __shared__ float prob[];
  const int lane = threadIdx.x;
  const int row = blockIdx.x;
  const typename El::S* src = gating + static_cast<size_t>(row) * E;
  const float ninf = -__builtin_inff();

  float mx = ninf;
  for (int c = lane; c < E; c += kWave) mx = fmaxf(mx, El::ld(src[c]));
#pragma unroll
  for (int m = 32; m > 0; m /= 2) mx = fmaxf(mx, __shfl_xor(mx, m, kWave));
  float sum = 0.f;
  for (int c = lane; c < E; c += kWave) {
    const float e = moe_expf<true>(El::ld(src[c]) - mx);
    prob[c] = e;
    sum += e;
  }
#pragma unroll
  for (int m = 32; m > 0; m /= 2) sum += __shfl_xor(sum, m, kWave);
  const float rinv = 1.f / sum;
  for (int c = lane; c < E; c += kWave) prob[c] = prob[c] * rinv;

  float wsum = 0.f;
  for (int k = 0; k < K; ++k) {
    // below the marker of a taken column.  (A row with fewer than K comparable probabilities, i.e.
    // NaN logits, lets a taken column win again: the reference's fallback kernel behaves the same,
    // csrc/moe_topk_softmax_kernels.cu:117-150, and such rows carry no meaning.)
    float best = -20000.f;
    int bidx = lane;
    for (int c = lane; c < E; c += kWave) {
      const float v = prob[c];
      if (v > best) { best = v; bidx = c; }
    }
#pragma unroll
    for (int m = 32; m > 0; m /= 2) {
      float ov = __shfl_xor(best, m, kWave);
      int oi = __shfl_xor(bidx, m, kWave);
      if (ov > best || (ov == best && oi < bidx)) { best = ov; bidx = oi; }
    }
    if (lane == 0) {
      const size_t o = static_cast<size_t>(row) * K + k;
      topk_w[o] = best;
      topk_ids[o] = bidx;
      if (tok_exp_idx) tok_exp_idx[o] = k * T + row;
    }
    wsum += best;
    if (lane == bidx % kWave) prob[bidx] = -10000.f;
  }
  if (renormalize && lane == 0) {
    for (int k = 0; k < K; ++k) {
      const size_t o = static_cast<size_t>(row) * K + k;
      topk_w[o] = topk_w[o] / wsum;
    }
  }
}

template <int E, typename El>
void launch_pow2(const typename El::S* g, float* w, int32_t* ids, int32_t* tei, int T, int K, int renorm,
                 hipStream_t s) {
  constexpr int rows_per_block = Pow2Geom<E>::kRowsPerWave * kWavesPerBlock;
  const int blocks = (T + rows_per_block - 1) / rows_per_block;
  hipLaunchKernelGGL((topk_softmax_pow2_kernel<E, El>), dim3(blocks), dim3(kWave * kWavesPerBlock), 0, s,
                     g, w, ids, tei, T, K, renorm);
}

template <int E, typename El>
int launch_topk_quant(const void* logits, float* w, int32_t* ids, int T, int K, int renorm, const MoeXCodes& xc, hipStream_t s) {
  constexpr int rows_per_block = Pow2Geom<E>::kRowsPerWave * kWavesPerBlock;
  const int route_blocks = (T + rows_per_block - 1) / rows_per_block, quant_blocks = (T + kWavesPerBlock - 1) / kWavesPerBlock;
  auto kern = xc.H <= 2048 ? topk_softmax_quant_kernel<E, El, 4> : topk_softmax_quant_kernel<E, El, 8>;
  using S = typename El::S;
  hipLaunchKernelGGL(kern, dim3(route_blocks + quant_blocks), dim3(kWave * kWavesPerBlock), 0, s, static_cast<const S*>(logits), w,
                     ids, T, K, renorm, route_blocks, static_cast<const S*>(xc.x), xc.H, xc.codes, xc.scales);
  return moe_check_launch("layer (routing and quantisation)");
}

template <typename El>
int launch_topk(const void* logits, float* w, int32_t* ids, int32_t* tei, int T, int E, int K, int renorm, hipStream_t s) {
  const typename El::S* g = static_cast<const typename El::S*>(logits);
  switch (E) {
    case 1: launch_pow2<1, El>(g, w, ids, tei, T, K, renorm, s); break;
    case 2: launch_pow2<2, El>(g, w, ids, tei, T, K, renorm, s); break;
    case 4: launch_pow2<4, El>(g, w, ids, tei, T, K, renorm, s); break;
    case 8: launch_pow2<8, El>(g, w, ids, tei, T, K, renorm, s); break;
    case 16: launch_pow2<16, El>(g, w, ids, tei, T, K, renorm, s); break;
    case 32: launch_pow2<32, El>(g, w, ids, tei, T, K, renorm, s); break;
    case 64: launch_pow2<64, El>(g, w, ids, tei, T, K, renorm, s); break;
    case 128: launch_pow2<128, El>(g, w, ids, tei, T, K, renorm, s); break;
    case 256: launch_pow2<256, El>(g, w, ids, tei, T, K, renorm, s); break;
    default: {
      if (E > kWave * kGenericMaxPerLane) {
        hipLaunchKernelGGL(topk_softmax_wide_kernel<El>, dim3(T), dim3(kWave), sizeof(float) * E, s, g, w, ids, tei, T, E,
                           K, renorm);
        break;
      }
      const int blocks = (T + kWavesPerBlock - 1) / kWavesPerBlock;
      hipLaunchKernelGGL(topk_softmax_generic_kernel<El>, dim3(blocks), dim3(kWave * kWavesPerBlock), 0, s, g, w, ids,
                         tei, T, E, K, renorm);
    }
  }
  return moe_check_launch("topk_softmax");
}

}  // namespace

MOE_EXPORT int moe_topk_softmax_typed(const void* gating_output, int dtype, float* topk_weights, int32_t* topk_ids,
                                      int32_t* token_expert_indices, int T, int E, int K, int renormalize, void* stream) {
  if (T < 0 || E < 1 || K < 1) return moe_fail(MOE_ERR_ARG, "topk_softmax: bad sizes T=%d E=%d K=%d", T, E, K);
  if (K > E) return moe_fail(MOE_ERR_ARG, "topk_softmax: topk %d exceeds num_experts %d", K, E);
  if (E > kWideMaxExperts)
    return moe_fail(MOE_ERR_UNSUPPORTED, "topk_softmax: num_experts %d > %d", E, kWideMaxExperts);
  if (static_cast<int64_t>(T) * K > INT32_MAX)
    return moe_fail(MOE_ERR_ARG, "topk_softmax: T*K overflows int32 token_expert_indices");
  // one 64-lane workgroup per row beyond 1024 experts: the grid's thread count has to fit 32 bits
  if (E > kWave * kGenericMaxPerLane && static_cast<int64_t>(T) > (static_cast<int64_t>(UINT32_MAX) / kWave))
    return moe_fail(MOE_ERR_UNSUPPORTED, "topk_softmax: %d rows of %d experts exceed the launch limit of %lld rows", T, E,
                    static_cast<long long>(UINT32_MAX / kWave));
  if (T == 0) return MOE_OK;
  if (!gating_output || !topk_weights || !topk_ids) return moe_fail(MOE_ERR_ARG, "topk_softmax: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case MOE_F32: return launch_topk<ElemF32>(gating_output, topk_weights, topk_ids, token_expert_indices, T, E, K, renormalize, s);
    case MOE_F16: return launch_topk<ElemF16>(gating_output, topk_weights, topk_ids, token_expert_indices, T, E, K, renormalize, s);
    case MOE_BF16: return launch_topk<ElemBF16>(gating_output, topk_weights, topk_ids, token_expert_indices, T, E, K, renormalize, s);
    default: return moe_fail(MOE_ERR_ARG, "topk_softmax: dtype code %d", dtype);
  }
}

bool moe_layer_route_quant(const void* logits, int dtype, float* topk_w, int32_t* topk_ids, int T, int E, int K, int renormalize,
                           const MoeXCodes& xc, hipStream_t s, int* rc) {
  if (!logits || (dtype != MOE_BF16 && dtype != MOE_F16) || T < 1 || K < 1 || K > E || static_cast<int64_t>(T) * K > INT32_MAX) return false;
  auto go = [&](auto tag) {
    constexpr int N = decltype(tag)::value;
    *rc = dtype == MOE_BF16 ? launch_topk_quant<N, ElemBF16>(logits, topk_w, topk_ids, T, K, renormalize, xc, s)
                            : launch_topk_quant<N, ElemF16>(logits, topk_w, topk_ids, T, K, renormalize, xc, s);
    return true;
  };
  switch (E) {
    case 16: return go(std::integral_constant<int, 16>{});
    case 32: return go(std::integral_constant<int, 32>{});
    case 64: return go(std::integral_constant<int, 64>{});
    case 128: return go(std::integral_constant<int, 128>{});
    case 256: return go(std::integral_constant<int, 256>{});
    default: return false;
  }
}

MOE_EXPORT int moe_topk_softmax(const float* gating_output, float* topk_weights, int32_t* topk_ids,
                                int32_t* token_expert_indices, int T, int E, int K,
                                int renormalize, void* stream) {
  if (T > 0 && !token_expert_indices && E >= 1 && K >= 1 && K <= E && E <= kWideMaxExperts)
    return moe_fail(MOE_ERR_ARG, "topk_softmax: null pointer");
  return moe_topk_softmax_typed(gating_output, MOE_F32, topk_weights, topk_ids, token_expert_indices, T, E, K, renormalize, stream);
}

MOE_EXPORT int moe_gate_topk_softmax(const void* x, const void* gate_weight, int dtype,
                                     float* logits_out, float* topk_weights, int32_t* topk_ids,
                                     int32_t* token_expert_indices, int T, int H, int E, int K,
                                     int renormalize, void* stream) {
  if (T < 0 || H < 1 || E < 1 || K < 1) return moe_fail(MOE_ERR_ARG, "gate_topk_softmax: bad sizes T=%d H=%d E=%d K=%d", T, H, E, K);
  if (K > E) return moe_fail(MOE_ERR_ARG, "gate_topk_softmax: topk %d exceeds num_experts %d", K, E);
  if (static_cast<int64_t>(T) * K > INT32_MAX)
    return moe_fail(MOE_ERR_ARG, "gate_topk_softmax: T*K overflows int32 token_expert_indices");
  if (H % 64 != 0)
    return moe_fail(MOE_ERR_UNSUPPORTED, "gate_topk_softmax: hidden size %d is not a multiple of 64", H);
  if (static_cast<int64_t>(T) * H * 2 >= (1LL << 32))
    return moe_fail(MOE_ERR_UNSUPPORTED, "gate_topk_softmax: x larger than 4 GiB (32-bit row offsets)");
  if (T == 0) return MOE_OK;
  if (!x || !gate_weight || !topk_weights || !topk_ids || !token_expert_indices)
    return moe_fail(MOE_ERR_ARG, "gate_topk_softmax: null pointer");
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(gate_weight)) & 15u)
    return moe_fail(MOE_ERR_ARG, "gate_topk_softmax: x and the gate weight must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case MOE_BF16: return launch_gate_e<ElemBF16>(x, gate_weight, logits_out, topk_weights, topk_ids, token_expert_indices, T, H, E, K, renormalize, s);
    case MOE_F16: return launch_gate_e<ElemF16>(x, gate_weight, logits_out, topk_weights, topk_ids, token_expert_indices, T, H, E, K, renormalize, s);
    default: return moe_fail(MOE_ERR_UNSUPPORTED, "gate_topk_softmax: dtype code %d (bf16 or fp16)", dtype);
  }
}

// Sizes for which the kernels that cut K serve a call: up to 1024 tiles of 16 tokens by 16 experts by 512 of K (256 of the
// large ones); then what all token tiles read of the gate outgrows what a product with fewer, larger tiles reads.  us, gate
// linear and router, against the library's GEMM and the router: E 128, H 2048, top-8: 6.5 and 9.2 at 1 token, 7.8 and 9.4
// at 135, 8.5 and 9.4 at 384, 8.7 and 9.4 at 512 (1024 tiles), 10.5 and 10.2 at 640, 10.9 and 10.4 at 1024; E 32, H 2048:
// 7.3 and 9.1 at 1024, 7.9 and 9.2 at 2047 (1024); E 64, H 4096: 8.0 and 11.6 at 135, 8.9 and 11.5 at 512 (1024), 11.0 and
// 11.9 at 1024; E 256, H 7168: 12.3 and 12.8 at 64 (896), 15.4 and 13.5 at 135 (2016).  The line follows the GPU's time, as
// a replayed graph sees it.  Called from Python these sizes are bound by the host, for which this way is one entry into
// native code and the other two and an operator: norm and router, us, E 128: 15.5 and 30.9 at 640 tokens, 17.9 and 30.8 at
// 1024, 23.9 and 30.7 at 2047; E 256, H 7168, 135 tokens: 23.2 and 30.9.  16 experts (33 us from Python) have no instance.
MOE_EXPORT int64_t moe_gate_topk_few_bytes(int T, int H, int E, int dtype) {
  if (T < 1 || H < 64 || H % 64 || (E != 32 && E != 64 && E != 128 && E != 256) || (dtype != MOE_BF16 && dtype != MOE_F16)) return 0;
  if (gate_small_tiles(T, H, E) > 1024) return 0;
  return static_cast<int64_t>(gate_pieces(H)) * T * E * static_cast<int64_t>(sizeof(float));
}

template <typename El>
static int launch_gate_pieces_e(const void* x, const void* wg, float* sums, float* w, int32_t* ids, int32_t* tei, int T, int H,
                                int E, int K, int renorm, hipStream_t s) {
  switch (E) {
    case 32: return launch_gate_pieces<32, El>(x, wg, sums, w, ids, tei, T, H, K, renorm, s);
    case 64: return launch_gate_pieces<64, El>(x, wg, sums, w, ids, tei, T, H, K, renorm, s);
    case 128: return launch_gate_pieces<128, El>(x, wg, sums, w, ids, tei, T, H, K, renorm, s);
    default: return launch_gate_pieces<256, El>(x, wg, sums, w, ids, tei, T, H, K, renorm, s);
  }
}

MOE_EXPORT int moe_gate_topk_few(const void* x, const void* gate_weight, int dtype, float* topk_weights, int32_t* topk_ids,
                                 int32_t* token_expert_indices, int T, int H, int E, int K, int renormalize, void* workspace,
                                 int64_t workspace_bytes, void* stream) {
  const int64_t need = moe_gate_topk_few_bytes(T, H, E, dtype);
  if (need == 0) return moe_fail(MOE_ERR_UNSUPPORTED, "gate_topk_few: T=%d H=%d E=%d dtype code %d", T, H, E, dtype);
  if (K < 1 || K > E) return moe_fail(MOE_ERR_ARG, "gate_topk_few: topk %d of %d experts", K, E);
  if (!x || !gate_weight || !topk_weights || !topk_ids) return moe_fail(MOE_ERR_ARG, "gate_topk_few: null pointer");
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(gate_weight)) & 15u)
    return moe_fail(MOE_ERR_ARG, "gate_topk_few: x and the gate weight must be 16-byte aligned");
  if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15u))
    return moe_fail(MOE_ERR_WORKSPACE, "gate_topk_few: workspace %lld B, needs %lld B, 16-byte aligned",
                    static_cast<long long>(workspace_bytes), static_cast<long long>(need));
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* sums = static_cast<float*>(workspace);
  return dtype == MOE_BF16
             ? launch_gate_pieces_e<ElemBF16>(x, gate_weight, sums, topk_weights, topk_ids, token_expert_indices, T, H, E, K, renormalize, s)
             : launch_gate_pieces_e<ElemF16>(x, gate_weight, sums, topk_weights, topk_ids, token_expert_indices, T, H, E, K, renormalize, s);
}
