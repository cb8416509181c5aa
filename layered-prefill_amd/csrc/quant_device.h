// Device side of the e4m3 row quantiser: codes and scale of one row of 16-bit values that is a whole number of 16-byte
// vectors.
#pragma once

#include "common.h"

namespace {

// Two values at once: bits 0-7 the code of a, bits 8-15 the code of b.
__device__ __forceinline__ uint32_t f32x2_to_e4m3(float a, float b) {
  a = __builtin_amdgcn_fmed3f(a, -448.f, 448.f);
  b = __builtin_amdgcn_fmed3f(b, -448.f, 448.f);
  return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false)) & 0xffffu;
}

// Smallest row scale: a row whose largest magnitude is tiny but not zero would get
// a scale whose reciprocal overflows (amax below about 1.3e-36); from 2^-100 down
// the scale stays 2^-100 and the row's codes are simply small.
constexpr float kMinScale = 7.888609052210118e-31f;  // 2^-100

// The codes of a row that LPR lanes of a wavefront hold, NV vectors of eight values each (zeros behind its end), and its
// scale.
template <typename El, int NV, int LPR>
__device__ __forceinline__ float quant_vecs(const uint4 (&v)[NV], uint2 (&codes)[NV]) {
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const uint32_t wds[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      amax = fmaxf(amax, fabsf(El::ld(static_cast<uint16_t>(wds[j]))));
      amax = fmaxf(amax, fabsf(El::ld(static_cast<uint16_t>(wds[j] >> 16))));
    }
  }
  amax = row_max<LPR>(amax);
  const float s = amax > 0.f ? fmaxf(amax / 448.f, kMinScale) : 1.f;
  const float inv = 1.0f / s;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const uint32_t wds[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
    uint32_t o[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o[j >> 1] |= f32x2_to_e4m3(El::ld(static_cast<uint16_t>(wds[j])) * inv,
                                 El::ld(static_cast<uint16_t>(wds[j] >> 16)) * inv)
                   << (16 * (j & 1));
    codes[i] = uint2{o[0], o[1]};
  }
  return s;
}

// A row of up to NV * LPR * 8 columns by LPR lanes of a wavefront: it stays in registers between the amax pass and the
// conversion, 16 bytes in and 8 bytes out per lane and step.
template <typename El, int NV, int LPR>
__device__ __forceinline__ void quant_row(const typename El::S* __restrict__ row, int lane, int cols, uint8_t* __restrict__ q,
                                          float* __restrict__ scale) {
  const uint4* src = reinterpret_cast<const uint4*>(row);
  const int nvec = cols / 8;
  uint4 v[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = lane + i * LPR;
    v[i] = c < nvec ? src[c] : uint4{0, 0, 0, 0};
  }
  uint2 codes[NV];
  const float s = quant_vecs<El, NV, LPR>(v, codes);
  if (lane == 0) *scale = s;
  uint2* dst = reinterpret_cast<uint2*>(q);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = lane + i * LPR;
    if (c < nvec) dst[c] = codes[i];
  }
}

}  // namespace
