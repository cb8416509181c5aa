// RMSNorm with the residual add in front of it: the step that feeds the MoE block
// (post_attention_layernorm in nanovllm/models/qwen3_moe.py, kernels
// csrc/layernorm_kernels.cu:10-35 and :77-108 of the reference).
//
//   s        = float(x) + float(residual)        (residual absent: s = float(x))
//   residual = T(s)
//   r        = rsqrt(mean(s^2) + eps)            (s before it is rounded, fp32)
//   out      = T( T(float(residual) * r) * weight )
//
// Bandwidth-bound: each element is read once and written once per tensor.  One
// wavefront owns one row; a lane holds its share of the row in registers (16-byte
// loads), so the rounded sums are never read back from memory, the reduction is
// a butterfly of lane moves inside the wavefront and no LDS or barrier is needed.  (With
// shuffles through the LDS crossbar 64 rows of 2048 took 3.2 us, 3.0 this way.)
#include "common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kRowsPerBlock = kThreads / kWave;

// The product as an fp32 value, as the definition above has it: without this the compiler may fold the
// multiplication into the conversion to fp16 (v_fma_mixlo_f16: one rounding of the exact product instead of two), and
// it did so in one kernel here and not in the other, which then differed in one element in ten thousand.
template <typename El>
__device__ __forceinline__ float product(float a, float b) {
  float v = a * b;
  if constexpr (__is_same(El, ElemF16)) asm("" : "+v"(v));
  return v;
}

// Two values rounded to the 16-bit dtype in one conversion instruction (written out with integers, the rounding of
// an element took five operations and every element is rounded three times).
template <typename El>
__device__ __forceinline__ uint32_t round_pair(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  if constexpr (__is_same(El, ElemBF16)) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
  } else {
    typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2));
  }
}

// 16-bit dtypes, H a multiple of 8 and at most 512 * NV, all rows 16-byte aligned.
template <typename El, int NV, bool ADD>
__global__ __launch_bounds__(kThreads) void rms_norm_vec_kernel(uint16_t* out, int64_t out_stride,
                                                                uint16_t* residual, int64_t res_stride,
                                                                const uint16_t* x, int64_t x_stride,
                                                                const uint16_t* __restrict__ weight, float eps,
                                                                int64_t T, int H) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = blockIdx.x * static_cast<int64_t>(kRowsPerBlock) + (threadIdx.x >> 6);
  if (row >= T) return;
  // Every load of the row goes out before the first store: x, the residual and the result may be one buffer, so
  // the compiler keeps a load behind any store that stands in front of it in the source, and with the residual
  // stored chunk by chunk a row took NV round trips to memory one after the other.  Rows stay packed, two
  // elements a register, so that several wavefronts of a SIMD still hold a row each (unpacked, 116 registers, the
  // same loads made it slower: 72 us at 16896 rows).  bf16 rows of 2048: 8.6 -> 4.8 us for 64 of them, 32.6 ->
  // 25.5 us (5.4 TB/s) for 8448, 49.6 -> 44.8 us (6.2 TB/s) for 16896.  Longer rows gain more, although NV = 8 and
  // 16 take 138 and 284 registers, one wavefront a SIMD: the round trips of a row were its time (8448 rows of 4096
  // 65.0 -> 57.0 us, of 8192 133.6 -> 107.1; 64 rows 11.9 -> 4.5 and 22.8 -> 6.8; fp16 59.0 -> 57.1, 113.7 -> 105.0).
  uint4 xv[NV], rv[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = (j * kWave + lane) * 8;
    xv[j] = rv[j] = uint4{0, 0, 0, 0};
    if (c < H) {
      xv[j] = *reinterpret_cast<const uint4*>(x + row * x_stride + c);
      if constexpr (ADD) rv[j] = *reinterpret_cast<const uint4*>(residual + row * res_stride + c);
    }
  }
  auto lo = [](uint32_t v) { return El::ld(static_cast<uint16_t>(v)); };
  auto hi = [](uint32_t v) { return El::ld(static_cast<uint16_t>(v >> 16)); };
  auto pack = [](float a, float b) { return round_pair<El>(a, b); };
  float sq = 0.f;
  auto add = [&](uint32_t a, uint32_t b) {   // the rounded sum of a pair; sq takes it before it is rounded
    const float v0 = lo(a) + lo(b), v1 = hi(a) + hi(b);
    sq += v0 * v0;
    sq += v1 * v1;
    return pack(v0, v1);
  };
  auto square = [&](uint32_t a) {
    sq += lo(a) * lo(a);
    sq += hi(a) * hi(a);
  };
#pragma unroll
  for (int j = 0; j < NV; ++j) {   // (chunks behind H are zero and add nothing)
    if constexpr (ADD) {
      xv[j] = uint4{add(xv[j].x, rv[j].x), add(xv[j].y, rv[j].y), add(xv[j].z, rv[j].z), add(xv[j].w, rv[j].w)};
    } else {
      square(xv[j].x); square(xv[j].y); square(xv[j].z); square(xv[j].w);
    }
  }
  uint4 wv[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = (j * kWave + lane) * 8;
    if (c < H) {
      wv[j] = *reinterpret_cast<const uint4*>(weight + c);
      if constexpr (ADD) *reinterpret_cast<uint4*>(residual + row * res_stride + c) = xv[j];
    }
  }
  const float r = rsqrtf(row_sum<kWave>(sq) / static_cast<float>(H) + eps);
  auto scale = [&](uint32_t v, uint32_t w) {
    const uint32_t n = pack(product<El>(lo(v), r), product<El>(hi(v), r));
    return pack(lo(n) * lo(w), hi(n) * hi(w));
  };
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = (j * kWave + lane) * 8;
    if (c < H)
      *reinterpret_cast<uint4*>(out + row * out_stride + c) =
          uint4{scale(xv[j].x, wv[j].x), scale(xv[j].y, wv[j].y), scale(xv[j].z, wv[j].z), scale(xv[j].w, wv[j].w)};
  }
}

// Any dtype, size and alignment: two passes over the row, the second one reads
// back what this lane itself stored.
template <typename El, bool ADD>
__global__ __launch_bounds__(kThreads) void rms_norm_any_kernel(typename El::S* out, int64_t out_stride,
                                                                typename El::S* residual, int64_t res_stride,
                                                                const typename El::S* x, int64_t x_stride,
                                                                const typename El::S* __restrict__ weight, float eps,
                                                                int64_t T, int H) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = blockIdx.x * static_cast<int64_t>(kRowsPerBlock) + (threadIdx.x >> 6);
  if (row >= T) return;
  float sq = 0.f;
  for (int c = lane; c < H; c += kWave) {
    float v = El::ld(x[row * x_stride + c]);
    if constexpr (ADD) {
      v += El::ld(residual[row * res_stride + c]);
      residual[row * res_stride + c] = El::st(v);
    }
    sq += v * v;
  }
  const float r = rsqrtf(row_sum<kWave>(sq) / static_cast<float>(H) + eps);
  for (int c = lane; c < H; c += kWave) {
    const float v = ADD ? El::ld(residual[row * res_stride + c]) : El::ld(x[row * x_stride + c]);
    out[row * out_stride + c] = El::st(El::ld(El::st(product<El>(v, r))) * El::ld(weight[c]));
  }
}

template <typename El, bool ADD>
int launch_norm(void* out, int64_t out_stride, void* residual, int64_t res_stride, const void* x,
                int64_t x_stride, const void* weight, float eps, int64_t T, int H, hipStream_t s) {
  using S = typename El::S;
  const int64_t blocks = (T + kRowsPerBlock - 1) / kRowsPerBlock;
  if (blocks > INT32_MAX) return moe_fail(MOE_ERR_ARG, "rms_norm: %lld rows", static_cast<long long>(T));
  const dim3 grid(static_cast<unsigned>(blocks)), block(kThreads);
  if constexpr (sizeof(S) == 2) {
    auto aligned = [](const void* p, int64_t stride) {
      return (reinterpret_cast<uintptr_t>(p) & 15u) == 0 && (stride & 7) == 0;
    };
    const bool vec = (H & 7) == 0 && H <= 512 * 16 && aligned(out, out_stride) && aligned(x, x_stride) &&
                     (!ADD || aligned(residual, res_stride)) && (reinterpret_cast<uintptr_t>(weight) & 15u) == 0;
    if (vec) {
      uint16_t* o = static_cast<uint16_t*>(out);
      uint16_t* r = static_cast<uint16_t*>(residual);
      const uint16_t* xi = static_cast<const uint16_t*>(x);
      const uint16_t* w = static_cast<const uint16_t*>(weight);
#define MOE_NORM_CASE(NV)                                                                                   \
  hipLaunchKernelGGL((rms_norm_vec_kernel<El, NV, ADD>), grid, block, 0, s, o, out_stride, r, res_stride, xi, \
                     x_stride, w, eps, T, H)
      if (H <= 512) MOE_NORM_CASE(1);
      else if (H <= 1024) MOE_NORM_CASE(2);
      else if (H <= 2048) MOE_NORM_CASE(4);
      else if (H <= 4096) MOE_NORM_CASE(8);
      else MOE_NORM_CASE(16);
#undef MOE_NORM_CASE
      return moe_check_launch(ADD ? "add_rms_norm" : "rms_norm");
    }
  }
  hipLaunchKernelGGL((rms_norm_any_kernel<El, ADD>), grid, block, 0, s, static_cast<S*>(out), out_stride,
                     static_cast<S*>(residual), res_stride, static_cast<const S*>(x), x_stride,
                     static_cast<const S*>(weight), eps, T, H);
  return moe_check_launch(ADD ? "add_rms_norm" : "rms_norm");
}

}  // namespace

MOE_EXPORT int moe_add_rms_norm(void* out, int64_t out_stride, void* residual, int64_t residual_stride,
                                const void* x, int64_t x_stride, const void* weight, int dtype, int64_t T,
                                int H, float eps, void* stream) {
  if (T < 0 || H < 1) return moe_fail(MOE_ERR_ARG, "rms_norm: bad sizes T=%lld H=%d", static_cast<long long>(T), H);
  if (T == 0) return MOE_OK;
  if (!out || !x || !weight) return moe_fail(MOE_ERR_ARG, "rms_norm: null tensor pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
#define MOE_NORM_DTYPE(El)                                                                                        \
  return residual ? launch_norm<El, true>(out, out_stride, residual, residual_stride, x, x_stride, weight, eps, T, H, s) \
                  : launch_norm<El, false>(out, out_stride, nullptr, 0, x, x_stride, weight, eps, T, H, s)
  switch (dtype) {
    case MOE_BF16: MOE_NORM_DTYPE(ElemBF16);
    case MOE_F16: MOE_NORM_DTYPE(ElemF16);
    case MOE_F32: MOE_NORM_DTYPE(ElemF32);
    default: return moe_fail(MOE_ERR_UNSUPPORTED, "rms_norm: dtype code %d", dtype);
  }
#undef MOE_NORM_DTYPE
}
