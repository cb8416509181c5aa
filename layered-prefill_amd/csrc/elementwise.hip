// Bandwidth-bound helpers of the expert path: the stand-alone gated
// activations (csrc/activation_kernels.cu:14-64 of the reference), the top-k
// combine (nanovllm/layers/for_moe/moe_easy_kernel.py:26-31) and fp8 row
// quantisation.  16-byte vector accesses, grid-stride loops.
#include "common.h"
#include "quant_device.h"

namespace {

constexpr int kThreads = 256;

template <typename S, int N>
struct alignas(sizeof(S) * N) Vec {
  S v[N];
};

template <bool ONCE, typename S, int N>
__device__ __forceinline__ Vec<S, N> load_terms(const S* p) {
  if constexpr (ONCE && sizeof(Vec<S, N>) == 16) return __builtin_bit_cast(Vec<S, N>, load_once(p));
  else return *reinterpret_cast<const Vec<S, N>*>(p);
}

// out[r, i] = T(silu(in[r, i])) * in[r, d + i]; the product is taken in T.
template <typename El, int VEC>
__global__ __launch_bounds__(kThreads) void silu_and_mul_kernel(typename El::S* __restrict__ out,
                                                                const typename El::S* __restrict__ in,
                                                                int64_t rows, int d) {
  using S = typename El::S;
  const int per_row = d / VEC;
  const int64_t total = rows * per_row;
  for (int64_t idx = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x; idx < total;
       idx += static_cast<int64_t>(gridDim.x) * kThreads) {
    const int64_t r = idx / per_row;
    const int c = static_cast<int>(idx - r * per_row) * VEC;
    const Vec<S, VEC> g = *reinterpret_cast<const Vec<S, VEC>*>(in + r * 2 * d + c);
    const Vec<S, VEC> u = *reinterpret_cast<const Vec<S, VEC>*>(in + r * 2 * d + d + c);
    Vec<S, VEC> o;
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      const float s = El::ld(El::st(moe_silu(El::ld(g.v[i]))));
      o.v[i] = El::st(s * El::ld(u.v[i]));
    }
    *reinterpret_cast<Vec<S, VEC>*>(out + r * d + c) = o;
  }
}

// out[r, i] = T(swigluoai(in[r, 2i], in[r, 2i+1]))
template <typename El, int VEC>
__global__ __launch_bounds__(kThreads) void swigluoai_and_mul_kernel(
    typename El::S* __restrict__ out, const typename El::S* __restrict__ in, int64_t rows, int d,
    float alpha, float limit) {
  using S = typename El::S;
  const int per_row = d / VEC;
  const int64_t total = rows * per_row;
  for (int64_t idx = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x; idx < total;
       idx += static_cast<int64_t>(gridDim.x) * kThreads) {
    const int64_t r = idx / per_row;
    const int c = static_cast<int>(idx - r * per_row) * VEC;
    const Vec<S, 2 * VEC> x = *reinterpret_cast<const Vec<S, 2 * VEC>*>(in + r * 2 * d + 2 * c);
    Vec<S, VEC> o;
#pragma unroll
    for (int i = 0; i < VEC; ++i)
      o.v[i] = El::st(moe_swigluoai(El::ld(x.v[2 * i]), El::ld(x.v[2 * i + 1]), alpha, limit));
    *reinterpret_cast<Vec<S, VEC>*>(out + r * d + c) = o;
  }
}

// out[t, h] = sum_k in[t, k, h], ascending k, fp32 accumulation.  KK: K, where it is known here and all of a
// result's terms are asked for at once; else 0.  Bound by memory.  ONCE: the terms are read past the caches (load_once).
template <typename El, int VEC, int KK, bool ONCE>
__global__ __launch_bounds__(kThreads) void moe_sum_kernel(typename El::S* __restrict__ out,
                                                           const typename El::S* __restrict__ in,
                                                           int64_t T, int K, int H) {
  using S = typename El::S;
  const int per_row = H / VEC;
  const int64_t total = T * per_row;
  for (int64_t idx = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x; idx < total;
       idx += static_cast<int64_t>(gridDim.x) * kThreads) {
    const int64_t t = total <= INT32_MAX ? static_cast<int>(idx) / per_row : idx / per_row;
    const int c = static_cast<int>(idx - t * per_row) * VEC;
    float acc[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
    if constexpr (KK > 0) {
      const S* src = in + t * KK * static_cast<int64_t>(H) + c;
      Vec<S, VEC> x[KK];
#pragma unroll
      for (int k = 0; k < KK; ++k) x[k] = load_terms<ONCE, S, VEC>(src + k * static_cast<int64_t>(H));
#pragma unroll
      for (int k = 0; k < KK; ++k)
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[i] += El::ld(x[k].v[i]);
    } else {
      for (int k = 0; k < K; ++k) {
        const Vec<S, VEC> x = load_terms<ONCE, S, VEC>(in + (t * K + k) * static_cast<int64_t>(H) + c);
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[i] += El::ld(x.v[i]);
      }
    }
    Vec<S, VEC> o;
#pragma unroll
    for (int i = 0; i < VEC; ++i) o.v[i] = El::st(acc[i]);
    *reinterpret_cast<Vec<S, VEC>*>(out + t * static_cast<int64_t>(H) + c) = o;
  }
}


// fp32 -> OCP e4m3fn code, saturating at +-448, round to nearest even
// (v_cvt_pk_fp8_f32 on gfx950 produces the OCP encoding).
__device__ __forceinline__ uint8_t f32_to_e4m3(float v) {
  v = fminf(fmaxf(v, -448.f), 448.f);
  return static_cast<uint8_t>(__builtin_amdgcn_cvt_pk_fp8_f32(v, v, 0, false) & 0xff);
}

// One wavefront per row: s = max(amax|row| / 448, 2^-100) (1 for an all-zero row),
// q = e4m3(row * (1 / s)): one correctly rounded division per row, then one
// multiplication per element (a division per element made the kernel
// VALU-bound: 48 us for 67584 x 768 against 28 us of memory time).
template <typename El>
__global__ __launch_bounds__(kThreads) void quant_rows_e4m3_kernel(
    const typename El::S* __restrict__ w, int64_t rows, int cols, uint8_t* __restrict__ q,
    float* __restrict__ scales, const int32_t* __restrict__ row_ids, int64_t id_count, int numel) {
  const int lane = threadIdx.x % kWave;
  const int64_t row = blockIdx.x * static_cast<int64_t>(kThreads / kWave) + threadIdx.x / kWave;
  if (row >= rows) return;
  if (row_ids && (row >= id_count || row_ids[row] >= numel)) return;  // a padding slot: nobody reads it
  const typename El::S* src = w + row * cols;
  float amax = 0.f;
  for (int c = lane; c < cols; c += kWave) amax = fmaxf(amax, fabsf(El::ld(src[c])));
  amax = row_max<kWave>(amax);
  const float s = amax > 0.f ? fmaxf(amax / 448.f, kMinScale) : 1.f;
  if (lane == 0) scales[row] = s;
  const float inv = 1.0f / s;
  for (int c = lane; c < cols; c += kWave) q[row * cols + c] = f32_to_e4m3(El::ld(src[c]) * inv);
}

// 16-bit sources with up to NV * LPR * 8 columns: the row stays in registers between
// the amax pass and the conversion, 16 bytes in and 8 bytes out per lane and
// step.  Same arithmetic as the kernel above, element by element.  LPR lanes own a row: rows of at most 1024
// columns go two to a wavefront, so that 768 of them are three whole steps instead of one and a half
// (67584 rows of 768 among their padding: 35.7 -> 29.4 us, 5.3 TB/s).
template <typename El, int NV, int LPR>
__global__ __launch_bounds__(kThreads) void quant_rows_e4m3_vec_kernel(
    const typename El::S* __restrict__ w, int64_t rows, int cols, uint8_t* __restrict__ q,
    float* __restrict__ scales, const int32_t* __restrict__ row_ids, int64_t id_count, int numel) {
  const int lane = threadIdx.x % LPR;
  const int64_t row = blockIdx.x * static_cast<int64_t>(kThreads / LPR) + threadIdx.x / LPR;
  if (row >= rows) return;
  if (row_ids && (row >= id_count || row_ids[row] >= numel)) return;  // a padding slot: nobody reads it
  quant_row<El, NV, LPR>(w + row * cols, lane, cols, q + row * cols, scales + row);
}

template <typename El>
bool launch_quant_vec(const void* w, int64_t rows, int cols, uint8_t* q, float* scales,
                      const int32_t* row_ids, int64_t id_count, int numel, hipStream_t s) {
  using S = typename El::S;
  if (cols % 8 != 0 || cols > 4096 || (reinterpret_cast<uintptr_t>(w) & 15u) || (reinterpret_cast<uintptr_t>(q) & 7u))
    return false;
  const S* src = static_cast<const S*>(w);
#define MOE_QUANT_CASE(NV, LPR)                                                                                       \
  hipLaunchKernelGGL((quant_rows_e4m3_vec_kernel<El, NV, LPR>),                                                       \
                     dim3(static_cast<unsigned>((rows + kThreads / LPR - 1) / (kThreads / LPR))), dim3(kThreads), 0, s, src, \
                     rows, cols, q, scales, row_ids, id_count, numel)
  if (cols <= 512) MOE_QUANT_CASE(2, 32);
  else if (cols <= 768) MOE_QUANT_CASE(3, 32);
  else if (cols <= 1024) MOE_QUANT_CASE(4, 32);
  else if (cols <= 2048) MOE_QUANT_CASE(4, 64);
  else MOE_QUANT_CASE(8, 64);
#undef MOE_QUANT_CASE
  return true;
}

int grid_for(int64_t work_items) {
  int64_t b = (work_items + kThreads - 1) / kThreads;
  const int64_t cap = 256 * 16;  // 256 CUs, 16 workgroups each; the loops stride past this
  if (b > cap) b = cap;
  if (b < 1) b = 1;
  return static_cast<int>(b);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <typename El>
int launch_silu(void* out, const void* in, int64_t rows, int d, hipStream_t s) {
  using S = typename El::S;
  constexpr int V = 16 / sizeof(S);
  if (d % V == 0 && aligned16(out) && aligned16(in))
    hipLaunchKernelGGL((silu_and_mul_kernel<El, V>), dim3(grid_for(rows * (d / V))), dim3(kThreads),
                       0, s, static_cast<S*>(out), static_cast<const S*>(in), rows, d);
  else
    hipLaunchKernelGGL((silu_and_mul_kernel<El, 1>), dim3(grid_for(rows * d)), dim3(kThreads), 0, s,
                       static_cast<S*>(out), static_cast<const S*>(in), rows, d);
  return moe_check_launch("silu_and_mul");
}

template <typename El>
int launch_swiglu(void* out, const void* in, int64_t rows, int d, float alpha, float limit,
                  hipStream_t s) {
  using S = typename El::S;
  constexpr int V = 8 / sizeof(S);  // the input vector is twice as wide
  if (d % V == 0 && aligned16(in) && (reinterpret_cast<uintptr_t>(out) & 7u) == 0)
    hipLaunchKernelGGL((swigluoai_and_mul_kernel<El, V>), dim3(grid_for(rows * (d / V))),
                       dim3(kThreads), 0, s, static_cast<S*>(out), static_cast<const S*>(in), rows,
                       d, alpha, limit);
  else
    hipLaunchKernelGGL((swigluoai_and_mul_kernel<El, 1>), dim3(grid_for(rows * d)), dim3(kThreads),
                       0, s, static_cast<S*>(out), static_cast<const S*>(in), rows, d, alpha, limit);
  return moe_check_launch("swigluoai_and_mul");
}

template <typename El>
int launch_sum(void* out, const void* in, int64_t T, int K, int H, bool in_layer, hipStream_t s) {
  using S = typename El::S;
  constexpr int V = 16 / sizeof(S);
  if (H % V == 0 && aligned16(out) && aligned16(in)) {
    // All terms at once: 8 terms of 2048 elements, bf16, us, this way and term by term: 1 row 2.3 and 3.0, 64 rows 2.5
    // and 3.4, 741 rows 3.5 and 3.8, 8448 rows (277 MB) 47.9 and 48.7, 16896 rows 93.1 and 94.8.  4 and 8 terms have an
    // instance.  2 would gain next to nothing by one (64 rows 2.13 and 2.24, 8448 rows 16.5 and 16.4); 6 would gain half a
    // microsecond where rows are few (64 rows 2.23 and 2.80, 741 rows 3.01 and 3.36, 8448 rows 36.2 and 36.0).
    //
    // Past the caches, and a workgroup for every 256 vectors instead of 4096 that stride on, where the terms are more than
    // the memory-side cache still holds of what has just been written.  Behind a kernel that writes them, us, through the
    // caches and past them: 8 terms of 2048, 1024 rows (34 MB) 7.4 and 7.8, 4096 (134 MB) 26.3 and 23.4, 8448 (277 MB)
    // 52.8 and 33.4, 16896 (554 MB) 116 and 94; 4 of 2048 (68 to 277 MB) 13.1 and 13.9, 26.8 and 24.0, 56.9 and 40.0; 6 of
    // 4096, 101 MB 18.2 and 18.3.  A row that is no whole number of 128-byte lines has its ends fetched twice that way:
    // 6 of 1000, 101 MB 19.5 and 23.2, 203 MB 32.7 and 31.0, 8 of 1000, 135 MB 24.0 and 26.6, 270 MB 51.3 and 34.3.
    // In a layer's call the terms otherwise take the place of weights in that cache, so that whole lines go past it at every
    // size: 32 experts, H 4096, I 1024, 301 tokens, one set of weights again and again 193 and 184, e4m3 2000 tokens of 128
    // experts 219 and 215; sets in rotation, 1 to 8448 tokens, within 0.7 % of each other.
    const bool lines = H * static_cast<int64_t>(sizeof(S)) % 128 == 0;
    const int64_t bytes = T * K * static_cast<int64_t>(H) * static_cast<int64_t>(sizeof(S));
    const bool once = lines ? in_layer || bytes > int64_t{120} << 20 : bytes > int64_t{190} << 20;
    const int64_t want = (T * (H / V) + kThreads - 1) / kThreads;
    const unsigned grid = once ? static_cast<unsigned>(want < (1 << 22) ? want : 1 << 22) : grid_for(T * (H / V));
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(grid), dim3(kThreads), 0, s, static_cast<S*>(out), static_cast<const S*>(in), T, K, H);
    };
    if (once) go(K == 8 ? moe_sum_kernel<El, V, 8, true> : K == 4 ? moe_sum_kernel<El, V, 4, true> : moe_sum_kernel<El, V, 0, true>);
    else go(K == 8 ? moe_sum_kernel<El, V, 8, false> : K == 4 ? moe_sum_kernel<El, V, 4, false> : moe_sum_kernel<El, V, 0, false>);
  } else {
    hipLaunchKernelGGL((moe_sum_kernel<El, 1, 0, false>), dim3(grid_for(T * H)), dim3(kThreads), 0, s,
                       static_cast<S*>(out), static_cast<const S*>(in), T, K, H);
  }
  return moe_check_launch("moe_sum");
}

}  // namespace

MOE_EXPORT int moe_silu_and_mul(void* out, const void* in, int64_t rows, int d, int dtype,
                                void* stream) {
  if (rows < 0 || d < 1) return moe_fail(MOE_ERR_ARG, "silu_and_mul: bad sizes rows=%lld d=%d", static_cast<long long>(rows), d);
  if (rows == 0) return MOE_OK;
  if (!out || !in) return moe_fail(MOE_ERR_ARG, "silu_and_mul: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case MOE_F32: return launch_silu<ElemF32>(out, in, rows, d, s);
    case MOE_F16: return launch_silu<ElemF16>(out, in, rows, d, s);
    case MOE_BF16: return launch_silu<ElemBF16>(out, in, rows, d, s);
    default: return moe_fail(MOE_ERR_ARG, "silu_and_mul: unsupported dtype code %d", dtype);
  }
}

MOE_EXPORT int moe_swigluoai_and_mul(void* out, const void* in, int64_t rows, int d, int dtype,
                                     float alpha, float limit, void* stream) {
  if (rows < 0 || d < 1) return moe_fail(MOE_ERR_ARG, "swigluoai_and_mul: bad sizes rows=%lld d=%d", static_cast<long long>(rows), d);
  if (rows == 0) return MOE_OK;
  if (!out || !in) return moe_fail(MOE_ERR_ARG, "swigluoai_and_mul: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case MOE_F32: return launch_swiglu<ElemF32>(out, in, rows, d, alpha, limit, s);
    case MOE_F16: return launch_swiglu<ElemF16>(out, in, rows, d, alpha, limit, s);
    case MOE_BF16: return launch_swiglu<ElemBF16>(out, in, rows, d, alpha, limit, s);
    default: return moe_fail(MOE_ERR_ARG, "swigluoai_and_mul: unsupported dtype code %d", dtype);
  }
}

MOE_EXPORT int moe_sum(void* out, const void* in, int64_t T, int K, int H, int dtype, void* stream) {
  return moe_sum_terms(out, in, T, K, H, dtype, false, stream);
}

int moe_sum_terms(void* out, const void* in, int64_t T, int K, int H, int dtype, bool in_layer, void* stream) {
  if (T < 0 || K < 1 || H < 1) return moe_fail(MOE_ERR_ARG, "moe_sum: bad sizes T=%lld K=%d H=%d", static_cast<long long>(T), K, H);
  if (T == 0) return MOE_OK;
  if (!out || !in) return moe_fail(MOE_ERR_ARG, "moe_sum: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case MOE_F32: return launch_sum<ElemF32>(out, in, T, K, H, in_layer, s);
    case MOE_F16: return launch_sum<ElemF16>(out, in, T, K, H, in_layer, s);
    case MOE_BF16: return launch_sum<ElemBF16>(out, in, T, K, H, in_layer, s);
    default: return moe_fail(MOE_ERR_ARG, "moe_sum: unsupported dtype code %d", dtype);
  }
}

MOE_EXPORT int moe_quant_rows_e4m3(const void* w, int src_dtype, int64_t rows, int cols,
                                   uint8_t* q, float* scales, void* stream) {
  return moe_quant_slot_rows_e4m3(w, src_dtype, rows, cols, q, scales, nullptr, 0, 0, stream);
}

// Row r is skipped (q and scales left untouched) when row_ids is given and r >= id_count or
// row_ids[r] >= numel: the padding slots of an expert-sorted intermediate.
int moe_quant_slot_rows_e4m3(const void* w, int src_dtype, int64_t rows, int cols, uint8_t* q,
                             float* scales, const int32_t* row_ids, int64_t id_count, int numel,
                             void* stream) {
  if (rows < 0 || cols < 1) return moe_fail(MOE_ERR_ARG, "quant_rows_e4m3: bad sizes rows=%lld cols=%d", static_cast<long long>(rows), cols);
  if (rows == 0) return MOE_OK;
  if (!w || !q || !scales) return moe_fail(MOE_ERR_ARG, "quant_rows_e4m3: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t blocks = (rows + kThreads / kWave - 1) / (kThreads / kWave);
  if (blocks > INT32_MAX) return moe_fail(MOE_ERR_ARG, "quant_rows_e4m3: too many rows");
  const dim3 grid(static_cast<unsigned>(blocks)), block(kThreads);
  switch (src_dtype) {
    case MOE_F32:
      hipLaunchKernelGGL(quant_rows_e4m3_kernel<ElemF32>, grid, block, 0, s, static_cast<const float*>(w), rows, cols, q, scales, row_ids, id_count, numel);
      break;
    case MOE_F16:
      if (!launch_quant_vec<ElemF16>(w, rows, cols, q, scales, row_ids, id_count, numel, s))
        hipLaunchKernelGGL(quant_rows_e4m3_kernel<ElemF16>, grid, block, 0, s, static_cast<const uint16_t*>(w), rows, cols, q, scales, row_ids, id_count, numel);
      break;
    case MOE_BF16:
      if (!launch_quant_vec<ElemBF16>(w, rows, cols, q, scales, row_ids, id_count, numel, s))
        hipLaunchKernelGGL(quant_rows_e4m3_kernel<ElemBF16>, grid, block, 0, s, static_cast<const uint16_t*>(w), rows, cols, q, scales, row_ids, id_count, numel);
      break;
    default:
      return moe_fail(MOE_ERR_ARG, "quant_rows_e4m3: unsupported source dtype code %d", src_dtype);
  }
  return moe_check_launch("quant_rows_e4m3");
}
