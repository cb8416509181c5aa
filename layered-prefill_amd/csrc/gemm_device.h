// Device side shared by the kernels that multiply expert weights: matrix products, direct global-to-LDS loads, waits,
// conversions and the gated activations.
#pragma once

#include "common.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;

struct MmaBF16 {
  using El = ElemBF16;
  static constexpr int kEs = 2;  // bytes per input element
  static constexpr int kBigChunks = 1;  // large-tile kernel: 16-byte chunks per lane and MFMA step
  static __device__ __forceinline__ f32x16 mma(const uint4& a, const uint4& b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x16 mma_big(const uint4 (&a)[1], const uint4 (&b)[1], f32x16 c) {
    return mma(a[0], b[0], c);
  }
  // 16 x 16, four 16-byte chunks of a row (lane / 16 says which of them a lane holds)
  static __device__ __forceinline__ f32x4 mma16(const uint4& a, const uint4& b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
struct MmaF16 {
  using El = ElemF16;
  static constexpr int kEs = 2;
  static constexpr int kBigChunks = 1;
  static __device__ __forceinline__ f32x16 mma(const uint4& a, const uint4& b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x16 mma_big(const uint4 (&a)[1], const uint4 (&b)[1], f32x16 c) {
    return mma(a[0], b[0], c);
  }
  static __device__ __forceinline__ f32x4 mma16(const uint4& a, const uint4& b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

constexpr int kThreads = 256;
constexpr int kXcds = 8;

typedef __attribute__((address_space(3))) char lds_char;

__device__ __forceinline__ uint32_t lds_offset_of(const char* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const lds_char*)p));
}

// 16 bytes per lane from global memory straight into LDS at
// lds_wave_base + 16 * lane.  `base` and `lds_wave_base` are wavefront-uniform.
// ONCE: nobody reads these bytes again soon, so they are not kept in the caches (the non-temporal hint).  Weights that one
// workgroup reads arrive up to a tenth faster that way, which is most of a decode call (whole calls: stream_gemm_kernel).
template <bool ONCE = false>
__device__ __forceinline__ void lds_dma16(const char* base, uint32_t lane_byte_offset,
                                          uint32_t lds_wave_base) {
  if constexpr (ONCE) {
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %2 nt"
        :
        : "s"(lds_wave_base), "v"(lane_byte_offset), "s"(base)
        : "memory");
  } else {
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %2"
        :
        : "s"(lds_wave_base), "v"(lane_byte_offset), "s"(base)
        : "memory");
  }
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ void bare_barrier() {
  asm volatile("s_barrier" ::: "memory");
}

// x * sigmoid(x) with the hardware exp2 and reciprocal (about 1e-6 relative
// error); the result is rounded to 16 bits right after, so it differs from the
// exact-sequence moe_silu in well under one rounding in a thousand.
__device__ __forceinline__ float silu_fast(float x) {
  const float e = __builtin_amdgcn_exp2f(x * -1.44269504088896341f);
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

template <typename El>
__device__ __forceinline__ uint32_t pack2(float a, float b);
template <>
__device__ __forceinline__ uint32_t pack2<ElemBF16>(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
template <>
__device__ __forceinline__ uint32_t pack2<ElemF16>(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2));
}

// A word that no workgroup of the launch writes, at an address that is the same for the whole wavefront: as a scalar
// load, so that it does not stand in the queue of the vector requests.
__device__ __forceinline__ int uniform_load(const int32_t* at) {
  return *reinterpret_cast<const __attribute__((address_space(4))) int32_t*>(reinterpret_cast<uintptr_t>(at));
}

template <typename El>
__device__ __forceinline__ float unpack_lo(uint32_t w);
template <typename El>
__device__ __forceinline__ float unpack_hi(uint32_t w);
template <>
__device__ __forceinline__ float unpack_lo<ElemBF16>(uint32_t w) { return __uint_as_float(w << 16); }
template <>
__device__ __forceinline__ float unpack_hi<ElemBF16>(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
template <>
__device__ __forceinline__ float unpack_lo<ElemF16>(uint32_t w) { return f16_bits_to_f32(static_cast<uint16_t>(w)); }
template <>
__device__ __forceinline__ float unpack_hi<ElemF16>(uint32_t w) { return f16_bits_to_f32(static_cast<uint16_t>(w >> 16)); }

template <typename El, int ACT>
__device__ __forceinline__ uint32_t gated_pair(float alpha, float limit, uint32_t gw, uint32_t uw) {
  const float g0 = unpack_lo<El>(gw), g1 = unpack_hi<El>(gw);
  const float u0 = unpack_lo<El>(uw), u1 = unpack_hi<El>(uw);
  if constexpr (ACT == MOE_ACT_SWIGLUOAI) {
    return pack2<El>(moe_swigluoai(g0, u0, alpha, limit), moe_swigluoai(g1, u1, alpha, limit));
  } else {
    float a0, a1;
    if constexpr (ACT == MOE_ACT_SILU) {
      a0 = silu_fast(g0);
      a1 = silu_fast(g1);
    } else {
      a0 = 0.5f * g0 * (1.f + erff(g0 * 0.70710678118654752f));
      a1 = 0.5f * g1 * (1.f + erff(g1 * 0.70710678118654752f));
    }
    const uint32_t aw = pack2<El>(a0, a1);  // the activation is stored in T before the product
    return pack2<El>(unpack_lo<El>(aw) * u0, unpack_hi<El>(aw) * u1);
  }
}

}  // namespace
