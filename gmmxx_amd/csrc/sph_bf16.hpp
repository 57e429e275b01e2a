// Device helpers of the single-pass spherical bf16 kernels (em_coop.hip, em_one.hip).
#pragma once

#include "common.hpp"

namespace gx {
namespace sphb {

constexpr int kAug = 32;           // augmented k-chunk width (bf16 columns)
constexpr float kHuge = 1e30f;     // "minus infinity" that stays finite through MFMA
constexpr int kCW = 32;            // components per wave
constexpr int kRS = 48;            // r row stride (bf16): 32 components + padding

// Padded row width DP -> staged row stride (bf16): XS / 2 dwords ≡ 8 or 24 (mod 32),
// as in em_sph_bf16.hip; and the lanes (16-byte chunks) that load a row.
constexpr int row_stride(int dp) { return dp <= 32 ? 80 : (dp <= 64 ? 112 : (dp <= 96 ? 144 : 176)); }
constexpr int row_lanes(int dp) { return dp <= 32 ? 4 : (dp <= 64 ? 8 : 16); }

typedef short v4s __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

template <typename T>
__device__ __forceinline__ T ld16(const void* p) { return *reinterpret_cast<const T*>(p); }

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

// Sum over groups of G consecutive lanes (G <= 16), result in every lane.
template <int G>
__device__ __forceinline__ float group_sum(float v) {
  if constexpr (G >= 2) v += dpp<0xB1>(v);    // lane ^ 1
  if constexpr (G >= 4) v += dpp<0x4E>(v);    // lane ^ 2
  if constexpr (G >= 8) v += dpp<0x141>(v);   // row_half_mirror
  if constexpr (G >= 16) v += dpp<0x140>(v);  // row_mirror
  return v;
}
template <int G>
__device__ __forceinline__ float group_max(float v) {
  if constexpr (G >= 2) v = fmaxf(v, dpp<0xB1>(v));
  if constexpr (G >= 4) v = fmaxf(v, dpp<0x4E>(v));
  if constexpr (G >= 8) v = fmaxf(v, dpp<0x141>(v));
  return v;
}

// v shifted down by s elements of 16 bits (0 <= s; 8 or more: all zero).
__device__ __forceinline__ uint4 shift_elems(uint4 v, int s) {
  if (s & 4) { v.x = v.z; v.y = v.w; v.z = 0u; v.w = 0u; }
  if (s & 2) { v.x = v.y; v.y = v.z; v.z = v.w; v.w = 0u; }
  const unsigned b = (s & 1) * 16;
  v = make_uint4(__builtin_amdgcn_alignbit(v.y, v.x, b), __builtin_amdgcn_alignbit(v.z, v.y, b),
                 __builtin_amdgcn_alignbit(v.w, v.z, b), v.w >> b);
  return s >= 8 ? make_uint4(0, 0, 0, 0) : v;
}

// v combined with lane l ^ 16 (OFF = 16) or l ^ 32 (OFF = 32).
template <int OFF, bool MAX>
__device__ __forceinline__ float lanes_op(float v) {
  const auto t = (OFF == 16) ? __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false)
                             : __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  const float a = __uint_as_float(t[0]), b = __uint_as_float(t[1]);
  return MAX ? fmaxf(a, b) : a + b;
}

__device__ __forceinline__ void split3(float v, __bf16& h, __bf16& m, __bf16& l) {
  h = (__bf16)v;
  const float r = v - (float)h;
  m = (__bf16)r;
  l = (__bf16)(r - (float)m);
}

__device__ __forceinline__ uint32_t pack2(__bf16 a, __bf16 b) {
  return (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
}

// Two floats rounded to bf16 (nearest even) in one dword, a in the low half.
__device__ __forceinline__ uint32_t cvt2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// Transposing LDS read: in each 16-lane group, lane L supplies the address of
// an 8-byte chunk; lane i receives word (i % 4) of the chunks of lanes 4j + i/4.
__device__ __forceinline__ v4s tr16(const __bf16* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)p);
}

__device__ __forceinline__ bf16x8 cat(v4s lo, v4s hi) {
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// r rows: the 4-element column chunk is XOR-swizzled by (row / 4) % 4, so that
// 16 lanes writing one chunk of consecutive rows, and the transposing reads of
// 4 rows x 4 chunks, touch distinct bank pairs.
__device__ __forceinline__ int rswz(int row, int col) { return col ^ (((row >> 2) & 3) << 2); }

// Chunk cc (8 columns from cc) of a row of D columns, zeros past its end.  EXACT:
// D == DP and aligned rows; vec (uniform): whole aligned chunks, D % 8 == 0;
// otherwise the row's last 16 bytes, shifted down, where the chunk passes its
// end (an element-aligned 16-byte load: four times fewer than by element), or
// by element for rows under 8 columns.
template <bool EXACT>
__device__ __forceinline__ uint4 load_row_chunk(const __bf16* row, int cc, int D, bool vec, bool valid) {
  const uint4 zero = make_uint4(0, 0, 0, 0);
  if constexpr (EXACT) {
    const uint4 v = *reinterpret_cast<const uint4*>(row + cc);
    return valid ? v : zero;
  } else if (vec) {
    const uint4 v = *reinterpret_cast<const uint4*>(row + (cc < D ? cc : 0));
    return valid && cc < D ? v : zero;
  } else if (D >= 8) {
    const int base = cc < D - 8 ? cc : D - 8;
    const uint4 v = shift_elems(ld16_any(row + base), cc - base);
    return valid ? v : zero;
  } else {
    union { uint4 u; __bf16 e[8]; } t;
#pragma unroll
    for (int j = 0; j < 8; ++j) t.e[j] = (valid && cc + j < D) ? row[cc + j] : (__bf16)0.f;
    return t.u;
  }
}

}  // namespace sphb
}  // namespace gx
