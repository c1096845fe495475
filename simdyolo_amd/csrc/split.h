// Device pieces of the f16-split matrix kernels (split_gemm.hip states the
// arithmetic and its scales).
#pragma once

#include "igemm.h"

namespace sy {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2v __attribute__((ext_vector_type(2)));

// hi and lo of four floats times the power of two s, packed.
__device__ __forceinline__ void split4(const f32x4 v, float s, u32x2& hi, u32x2& lo) {
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const float a = v[2 * p], b = v[2 * p + 1];
    const f16x2 h = __builtin_convertvector((f32x2v{a * s, b * s}), f16x2);
    const float ra = __builtin_fmaf(a, s, -(float)h[0]), rb = __builtin_fmaf(b, s, -(float)h[1]);
    const f16x2 l = __builtin_convertvector((f32x2v{ra * 2048.f, rb * 2048.f}), f16x2);
    hi[p] = __builtin_bit_cast(unsigned, h);
    lo[p] = __builtin_bit_cast(unsigned, l);
  }
}

// A workgroup that reads kSplitHuge or more (or infinity) multiplies in plain
// float32: below it an element's error is at most 2^-32, however large its
// neighbours are (networks that also run in f16 stay below 65,504 anyway).
constexpr float kSplitHuge = 0x1p16f;
// Exponent fields of the activations' power-of-two scale: its first guess
// (largest values from 2^-2 to below 2^11 need no other) and its cap (every
// normal float is 2^-13 or more under it).
constexpr int kSplitExpGuess = 127 + 4, kSplitExpMax = 127 + 113;
// Set in one of the bits of the top four exponent bits of an f16 (two packed)
// of 2^-13 or more: its pair is within 2^-23 of the value.
constexpr unsigned kSplitFull = 0x78007800u;
__device__ __forceinline__ float exp_float(int e) { return __builtin_bit_cast(float, (unsigned)e << 23); }

// v or'ed over aligned groups of W lanes.
template <int W>
__device__ __forceinline__ unsigned or_lanes(unsigned v) {
  static_assert(W == 4 || W == 8 || W == 16 || W == 32, "quads to half waves");
  v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf, false);               // lane ^ 1
  v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf, false);               // lane ^ 2
  if (W > 4) v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, false);  // 7 - lane
  if (W > 8) v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, false);  // 15 - lane
  if (W > 16) v |= (unsigned)__shfl_xor((int)v, 16);
  return v;
}

// Four elements' bits, without their signs.
__device__ __forceinline__ unsigned magnitude_bits(const f32x4 v) {
  const u32x4 b = __builtin_bit_cast(u32x4, v);
  return (b[0] | b[1] | b[2] | b[3]) & 0x7fffffffu;
}

// Largest magnitude of four.
__device__ __forceinline__ float max4(const f32x4 v) {
  return fmaxf(fmaxf(__builtin_fabsf(v[0]), __builtin_fabsf(v[1])), fmaxf(__builtin_fabsf(v[2]), __builtin_fabsf(v[3])));
}

// Four weights from their pair (hi at w, lo 512 halves on) and inverse scale.
__device__ __forceinline__ f32x4 join4(const _Float16* w, float ws) {
  typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
  const f16x4 hi = *(const f16x4*)w, lo = *(const f16x4*)(w + 512);
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf((float)lo[e], 1.f / 2048, (float)hi[e]) * ws;
  return v;
}

// One step of a wave reduction: m and the m that DPP control ctrl moves here.
template <int ctrl, int rows>
__device__ __forceinline__ float dpp_max(float m) {
  const int o = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, m), ctrl, rows, 0xf, false);
  return fmaxf(m, __builtin_bit_cast(float, o));
}
// Largest of the wave's non-negative values, in lane 63: shifts within rows of
// 16, then the last lane of row 0 / 2 into row 1 / 3, and of row 1 into 2, 3.
__device__ __forceinline__ float wave_max63(float m) {
  m = dpp_max<0x111, 0xf>(m);
  m = dpp_max<0x112, 0xf>(m);
  m = dpp_max<0x114, 0xf>(m);
  m = dpp_max<0x118, 0xf>(m);
  m = dpp_max<0x142, 0xa>(m);
  return dpp_max<0x143, 0xc>(m);
}

__device__ __forceinline__ float readlane63(float m) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), 63));
}

// Exponent field of the scale that takes a largest magnitude m into
// [2^11, 2^12).
__device__ __forceinline__ int scale_exp(float m) {
  return min(265 - (int)(__builtin_bit_cast(unsigned, m) >> 23), kSplitExpMax);
}

// Whether the scale 2^(se - 127) suits operands whose largest magnitude so far
// is m: the scaled maximum lies in [2^2, 2^15) (a zero maximum suits any).
// Otherwise *ne is the one that takes m into [2^11, 2^12).
__device__ __forceinline__ bool scale_fits(float m, int se, int* ne) {
  const int me = __builtin_amdgcn_readfirstlane((int)(__builtin_bit_cast(unsigned, m) >> 23));
  *ne = __builtin_amdgcn_readfirstlane(scale_exp(m));
  const int top = me + se - 127;
  return top < 127 + 15 && (top >= 127 + 2 || *ne == se || __builtin_amdgcn_readfirstlane(m == 0.f ? 1 : 0));
}

// The sums so far from one scale to another: times the exact ratio.
template <int TM, int TN>
__device__ __forceinline__ void rescale(int se, int ne, f32x16 (&acc)[TM][TN], f32x16 (&crs)[TM][TN]) {
  const float f = exp_float(min(max(127 + ne - se, 1), 254));
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[i][j][r] *= f;
        crs[i][j][r] *= f;
      }
}

// acc = the sums in true scale.  ws: the lane's columns' inverse weight scales.
template <int TM, int TN>
__device__ __forceinline__ void unscale(const float (&ws)[TN], int se, f32x16 (&acc)[TM][TN],
                                        const f32x16 (&crs)[TM][TN]) {
  const float xs = exp_float(254 - se);
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = __builtin_fmaf(crs[i][j][r], 1.f / 2048, acc[i][j][r]) * xs * ws[j];
}

}  // namespace sy
