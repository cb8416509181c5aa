// Shared host/device helpers for libmoe_gfx950.so (gfx950 / CDNA4 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "../../include/moe_gfx950.h"

#define MOE_EXPORT extern "C" __attribute__((visibility("default")))

// Records a thread-local message and returns `code`.
int moe_fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
// Checks hipGetLastError() after a launch; 0 or MOE_ERR_LAUNCH.
int moe_check_launch(const char* what);

// moe_quant_rows_e4m3 restricted to the live slots of an expert-sorted matrix (library-internal).
int moe_quant_slot_rows_e4m3(const void* w, int src_dtype, int64_t rows, int cols, uint8_t* q,
                             float* scales, const int32_t* row_ids, int64_t id_count, int numel,
                             void* stream);

// Dynamic LDS above 64 KB must be opted into once per kernel and device.  One MoeLdsOptIn
// per kernel instantiation (a zero-initialised static); moe_opt_in_lds sets the attribute on
// the current device when it has not been set there yet.  Safe from several host threads.
constexpr int kMoeMaxDevices = 64;
struct MoeLdsOptIn {
  std::atomic<bool> done[kMoeMaxDevices];
};
int moe_opt_in_lds(MoeLdsOptIn& flags, const void* kernel, int lds_bytes, const char* what);

// The e4m3 codes of a layer call's x, which wait for nothing and so may be made beside the routing: where x is and where
// they and their row scales go.  moe_x_codes_ok: rows that the routing kernels quantise.
struct MoeXCodes {
  const void* x;
  int H;
  uint8_t* codes;
  float* scales;
};
static inline bool moe_x_codes_ok(const MoeXCodes& c) {
  return c.H % 8 == 0 && c.H <= 4096 && (reinterpret_cast<uintptr_t>(c.x) & 15u) == 0 && (reinterpret_cast<uintptr_t>(c.codes) & 7u) == 0;
}

// Router and alignment of a layer call in one launch, for the batches and layers where that is the faster way (align.hip);
// false, and nothing enqueued, elsewhere.  With `xc` it makes those codes, too.  `rc` is the launch's status.
bool moe_layer_route_align(const void* logits, int dtype, float* topk_w, int T, int E, int K, int renormalize, int block_size,
                           int32_t* sorted_ids, int64_t sorted_cap, int32_t* expert_ids, int64_t expert_cap, int32_t* npp,
                           const MoeXCodes* xc, hipStream_t s, int* rc);

// Router and e4m3 codes of x, which wait for nothing of each other, in one launch; false, and nothing enqueued, where no
// instance serves the call.
bool moe_layer_route_quant(const void* logits, int dtype, float* topk_w, int32_t* topk_ids, int T, int E, int K, int renormalize,
                           const MoeXCodes& xc, hipStream_t s, int* rc);

// Where a moe_fused_experts call of e4m3 weights keeps the codes and scales of x in its workspace, and that call with them
// there already.
void moe_experts_x_codes(const MoeFusedExpertsArgs* a, uint8_t** codes, float** scales);
// `ids`: the call's [T, K] ids, whose alignment (sorted_token_ids, expert_ids and num_tokens_post_pad, all of them) the gate-up
// pass makes and leaves; only where moe_experts_align says so.  Null: they are aligned already.
int moe_fused_experts_of_codes(const MoeFusedExpertsArgs* a, bool x_coded, const int32_t* ids);
bool moe_experts_align(const MoeFusedExpertsArgs* a);

// moe_sum of terms that a layer's down pass has just written (`in_layer`) or of a caller's own.
int moe_sum_terms(void* out, const void* in, int64_t T, int K, int H, int dtype, bool in_layer, void* stream);

// A layer call of a few tokens in two launches, where it is one that they serve (few.hip); false, and nothing enqueued,
// elsewhere.  `experts` holds E + 1 ids, `inter` T * K rows.  `rc` is the launches' status.
bool moe_layer_few(const MoeLayerArgs* a, float* topk_w, int32_t* topk_ids, int32_t* experts, void* inter, int* rc);

// int32 index, inside the 256-byte table of per-XCD ranges at the end of a moe_fused_experts
// workspace, of the count of expired waits of the one-launch form (cleared with the plan).
constexpr int kMoeStatusWord = 16;

static inline int64_t moe_align_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

constexpr int kWave = 64;

// Inclusive prefix sum over a wavefront, by lane exchanges inside the vector unit: shifts inside rows of 16 lanes, then the
// last lane of a row to the row behind it and of the first half to the second (a shuffle through the LDS crossbar costs
// about a hundred clocks, six of them more than a short kernel's whole scan).
__device__ __forceinline__ int wave_inclusive_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

// 16 bytes that nothing reads again: not kept in the caches on the way.  A large buffer that a kernel has just written lies
// partly unwritten-back in the 256 MB memory-side cache, and every line taken in on the way to it has one of those evicted.
__device__ __forceinline__ uint4 load_once(const void* p) {
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  return __builtin_bit_cast(uint4, __builtin_nontemporal_load(static_cast<const u32x4*>(p)));
}

// ---------------------------------------------------------------------------
// Lane exchanges of a row of TPR lanes (a power of two, up to the wavefront), by DPP moves and the swaps of 16 and 32 lanes: a few clocks each, where the LDS-crossbar
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
// The same of the two halves of the wavefront (lane ^ 32).
__device__ __forceinline__ void halves_of_wave(float v, float& a, float& b) {
  a = b = v;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
template <int TPR>
__device__ __forceinline__ float row_max(float v) {
  if constexpr (TPR > 1) v = fmaxf(v, dpp_move<0xB1>(v));   // quad_perm [1,0,3,2]
  if constexpr (TPR > 2) v = fmaxf(v, dpp_move<0x4E>(v));   // quad_perm [2,3,0,1]
  if constexpr (TPR > 4) v = fmaxf(v, dpp_move<0x141>(v));  // row_half_mirror
  if constexpr (TPR > 8) v = fmaxf(v, dpp_move<0x140>(v));  // row_mirror
  if constexpr (TPR > 16) {
    float a, b;
    rows_of_16(v, a, b);
    v = fmaxf(a, b);
  }
  if constexpr (TPR > 32) {
    float a, b;
    halves_of_wave(v, a, b);
    v = fmaxf(a, b);
  }
  return v;
}
// The same of integers: an exchange and the comparison are one instruction, as a float's cannot be, whose NaN has to be
// made quiet in between.
template <int CTRL>
__device__ __forceinline__ int dpp_move_bits(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int TPR>
__device__ __forceinline__ int row_max_bits(int v) {
  if constexpr (TPR > 1) v = max(v, dpp_move_bits<0xB1>(v));
  if constexpr (TPR > 2) v = max(v, dpp_move_bits<0x4E>(v));
  if constexpr (TPR > 4) v = max(v, dpp_move_bits<0x141>(v));
  if constexpr (TPR > 8) v = max(v, dpp_move_bits<0x140>(v));
  if constexpr (TPR > 16) {
    float a, b;
    rows_of_16(__builtin_bit_cast(float, v), a, b);
    v = max(__builtin_bit_cast(int, a), __builtin_bit_cast(int, b));
  }
  static_assert(TPR <= 32, "rows of half a wavefront at most");
  return v;
}
// The sum with the association of the xor butterfly from distance TPR / 2 down to 1.
template <int TPR>
__device__ __forceinline__ float row_sum(float v) {
  if constexpr (TPR > 32) {
    float a, b;
    halves_of_wave(v, a, b);
    v = a + b;
  }
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

// ---------------------------------------------------------------------------
// bf16 / f16 scalar conversions with explicit rounding (round to nearest even)
// ---------------------------------------------------------------------------
__device__ __forceinline__ float bf16_bits_to_f32(uint16_t h) {
  return __uint_as_float(static_cast<uint32_t>(h) << 16);
}
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return static_cast<uint16_t>(u >> 16);
}
__device__ __forceinline__ float f16_bits_to_f32(uint16_t h) {
  _Float16 v;
  __builtin_memcpy(&v, &h, 2);
  return static_cast<float>(v);
}
__device__ __forceinline__ uint16_t f32_to_f16_bits(float f) {
  _Float16 v = static_cast<_Float16>(f);  // v_cvt_f16_f32, round to nearest even
  uint16_t h;
  __builtin_memcpy(&h, &v, 2);
  return h;
}

// Element traits used by the elementwise kernels: storage type, load, store.
struct ElemF32 {
  using S = float;
  static __device__ __forceinline__ float ld(S v) { return v; }
  static __device__ __forceinline__ S st(float v) { return v; }
};
struct ElemBF16 {
  using S = uint16_t;
  static __device__ __forceinline__ float ld(S v) { return bf16_bits_to_f32(v); }
  static __device__ __forceinline__ S st(float v) { return f32_to_bf16_bits(v); }
};
struct ElemF16 {
  using S = uint16_t;
  static __device__ __forceinline__ float ld(S v) { return f16_bits_to_f32(v); }
  static __device__ __forceinline__ S st(float v) { return f32_to_f16_bits(v); }
};

// ---------------------------------------------------------------------------
// exp in fp32 as a fixed sequence of IEEE operations: Cody-Waite reduction by
// ln2 (two constants), degree-6 polynomial evaluated with fused multiply-adds,
// scaling through the exponent field.  <= 2 ulp.  Inputs above 88 give +inf,
// inputs below -104 give 0; between about -87.3 and -104 the result is
// subnormal, as CUDA's expf returns it when built without flush-to-zero (the
// reference's build, setup.py:46-47): such results are scaled in two steps, by
// 2^(n+64) through the exponent field (exact) and by one multiplication with
// 2^-64, which rounds once.  gfx950 code objects keep fp32 subnormals (denormal
// mode 3).  Translation units that use it are compiled with -ffp-contract=off
// so that no other operation is fused.
// The ends of the range leave by branches, which a wavefront whose values are all inside passes by at once; with ENDS_SELECTED
// they are put in by selects.  Kernels of many values are bound by how many instructions a value takes: silu_and_mul, bf16, us,
// with selects, with a branch for each end only, and this way: 67584 x 768 82, 76.4 and 71.1, 16896 x 4096 105, 98.5 and 91,
// 8 x 768 3.1, 3.3 and 2.9 (gates of standard deviation 50, an end in nearly every wavefront, 83, 77 and 78).  A router of few
// rows waits for one chain of instructions and is better without a branch: 128 experts, 1 token 2.5, 2.9 and 2.6.
// ---------------------------------------------------------------------------
template <bool ENDS_SELECTED = false>
__device__ __forceinline__ float moe_expf(float x) {
  auto mantissa = [](float in, float& n) {
    n = __builtin_rintf(in * 1.44269504088896341f);
    float r = __builtin_fmaf(n, -0.693359375f, in);
    r = __builtin_fmaf(n, 2.12194440e-4f, r);
    float p = 1.9875691500e-4f;
    p = __builtin_fmaf(p, r, 1.3981999507e-3f);
    p = __builtin_fmaf(p, r, 8.3334519073e-3f);
    p = __builtin_fmaf(p, r, 4.1665795894e-2f);
    p = __builtin_fmaf(p, r, 1.6666665459e-1f);
    p = __builtin_fmaf(p, r, 5.0000001201e-1f);
    float r2 = r * r;
    p = __builtin_fmaf(p, r2, r);
    return p + 1.0f;
  };
  float n;
  if constexpr (!ENDS_SELECTED) {
    if (__builtin_expect(!__ballot(!(__builtin_fabsf(x) <= 86.0f)), 1)) {   // (n from -124 to 124; NaN is outside)
      const float p = mantissa(x, n);
      return __uint_as_float(__float_as_uint(p) + (static_cast<uint32_t>(static_cast<int32_t>(n)) << 23));
    }
    if (x != x) return x;
    if (x > 88.0f) return __builtin_inff();
    if (x < -104.0f) return 0.0f;
    const float p = mantissa(x, n);
    const int32_t ni = static_cast<int32_t>(n);
    if (ni < -125) return __uint_as_float(__float_as_uint(p) + (static_cast<uint32_t>(ni + 64) << 23)) * 5.42101086242752217e-20f;
    return __uint_as_float(__float_as_uint(p) + (static_cast<uint32_t>(ni) << 23));
  }
  const float p = mantissa(__builtin_fminf(__builtin_fmaxf(x, -104.0f), 88.0f), n);
  const int32_t ni = static_cast<int32_t>(n);
  const bool small = ni < -125;
  const float y = __uint_as_float(__float_as_uint(p) + (static_cast<uint32_t>(small ? ni + 64 : ni) << 23));
  float e = small ? y * 5.42101086242752217e-20f : y;  // 2^-64
  e = x < -104.0f ? 0.0f : e;
  e = x > 88.0f ? __builtin_inff() : e;
  return x != x ? x : e;
}

__device__ __forceinline__ float moe_silu(float x) { return x / (1.0f + moe_expf(-x)); }

__device__ __forceinline__ float moe_swigluoai(float g, float u, float alpha, float limit) {
  float cg = g > limit ? limit : g;
  float cu = u > limit ? limit : (u < -limit ? -limit : u);
  float sig = 1.0f / (1.0f + moe_expf(-cg * alpha));
  float glu = cg * sig;
  float r = (cu + 1.0f) * glu;
  // The product is an fp32 value before it is narrowed, as in the reference's kernel.  Without
  // this the compiler may fold the multiplication into the conversion to fp16 (one rounding
  // of the exact product instead of two), which differs in one element in ten thousand.
  asm volatile("" : "+v"(r));
  return r;
}
