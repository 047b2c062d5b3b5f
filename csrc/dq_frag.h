// Packed weights as matrix-core operands: eight codes of one weight row as
// the exact bf16 numbers 128 + c (int4, one dword) or c (int8, two dwords).
// With a group's scale s and zero z,
//   sum s (c - z) x = s (sum code x) - s zb sum x,  zb = z + 128 or z.
#pragma once
#include <type_traits>

#include "common.h"

template <int BITS>
__device__ __forceinline__ s16x8 codes8(const u32* w) {
  if constexpr (BITS == 4) {
    const DequantPairs4 d = dequant4_pairs(w[0]);
    return __builtin_bit_cast(s16x8, u32x4{d.p01, d.p23, d.p45, d.p67});
  } else {
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // at most 8 significant bits: the upper half of the float is exact
      const u32 p = w[i >> 1] >> (16 * (i & 1));
      const float lo = (float)(p & 0xFFu), hi = (float)((p >> 8) & 0xFFu);
      o[i] = __builtin_amdgcn_perm(__builtin_bit_cast(u32, hi),
                                   __builtin_bit_cast(u32, lo), 0x07060302u);
    }
    return __builtin_bit_cast(s16x8, o);
  }
}

// The same eight codes of a dword in the order 0 2 4 6 1 3 5 7, which takes
// seven instructions instead of eleven, and eight numbers of x in that order.
__device__ __forceinline__ s16x8 codes8_dealt(u32 w) {
  const u32 even = w & 0x0F0F0F0Fu, odd = (w >> 4) & 0x0F0F0F0Fu;
  return __builtin_bit_cast(
      s16x8, u32x4{__builtin_amdgcn_perm(0x43434343u, even, 0x04010400u),
                   __builtin_amdgcn_perm(0x43434343u, even, 0x04030402u),
                   __builtin_amdgcn_perm(0x43434343u, odd, 0x04010400u),
                   __builtin_amdgcn_perm(0x43434343u, odd, 0x04030402u)});
}
__device__ __forceinline__ s16x8 deal8(s16x8 x) {
  const u32x4 a = __builtin_bit_cast(u32x4, x);
  return __builtin_bit_cast(
      s16x8, u32x4{__builtin_amdgcn_perm(a[1], a[0], 0x05040100u),
                   __builtin_amdgcn_perm(a[3], a[2], 0x05040100u),
                   __builtin_amdgcn_perm(a[1], a[0], 0x07060302u),
                   __builtin_amdgcn_perm(a[3], a[2], 0x07060302u)});
}

// Eight codes as bf16, exact.  int4: a nibble c is the fp8 (e4m3) number
// c 2^-9, denormal or not, which an instruction turns into bf16 two at a time.
template <int BITS>
__device__ __forceinline__ s16x8 codes8_exact(const u32* w) {
  if constexpr (BITS == 8) {
    return codes8<8>(w);
  } else {
    const u32 even = w[0] & 0x0F0F0F0Fu, odd = (w[0] >> 4) & 0x0F0F0F0Fu;
    const u32 lo = __builtin_amdgcn_perm(odd, even, 0x05010400u);
    const u32 hi = __builtin_amdgcn_perm(odd, even, 0x07030602u);
    auto two = [](u32 v, auto up) {
      return __builtin_bit_cast(
          u32, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                   v, 512.f, decltype(up)::value));
    };
    constexpr std::false_type l{};
    constexpr std::true_type h{};
    return __builtin_bit_cast(
        s16x8, u32x4{two(lo, l), two(lo, h), two(hi, l), two(hi, h)});
  }
}

// zb of group gi from its word of packed zeros
template <int BITS>
__device__ __forceinline__ float zero_bias(u32 word, int gi) {
  return BITS == 4 ? (float)(unpack4(word, gi & 7) + 128u)
                   : (float)unpack8(word, gi & 3);
}

__device__ __forceinline__ s16x8 bf16_ones() {
  return __builtin_bit_cast(
      s16x8, u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
}

// The sum of `parts` results, `stride` floats apart, in order; up to eight of
// them on their way at once.
template <int B>
__device__ __forceinline__ f32x4 sum_in(const float* p, u64 stride, int parts) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < parts; s0 += B) {
    f32x4 t[B];
#pragma unroll
    for (int i = 0; i < B; ++i)
      t[i] = *(const f32x4*)(p + (u64)min(s0 + i, parts - 1) * stride);
#pragma unroll
    for (int i = 0; i < B; ++i)
      if (s0 + i < parts) v += t[i];
  }
  return v;
}
__device__ __forceinline__ f32x4 sum_of_parts(const float* p, u64 stride,
                                              int parts) {
  return parts <= 2 ? sum_in<2>(p, stride, parts)
                    : (parts <= 4 ? sum_in<4>(p, stride, parts)
                                  : sum_in<8>(p, stride, parts));
}

// What follows a whole row of the result, r = sum + bias (+ residual) in bf16.
// normed: y = r + to in bf16, normed = (r + to) w over its root mean square;
// else scale: y = r, scale = 1 / its root mean square (mean square + eps).
struct DqRowEnd {
  float* scale;                  // [m]
  unsigned short* normed;        // [m, n]
  const unsigned short *to, *w;  // [m, n], [n]
  float eps;
};

// what the packed-product kernels (dq_rows, dq_tile) take
struct DqArgs {
  const char* w;                 // [n, k * BITS / 8] bytes
  const unsigned short* scales;  // [n, G]
  const u32* zeros;              // [n, zw]
  const unsigned short* x;       // [m, k]
  unsigned short* y;             // [m, n]
  const unsigned short *bias, *resid;
  float* part;                   // [splits, m, n], splits > 1
  int m, n, k, g, splits;
  // experts: w, scales and zeros have one [n, ..] each; a row tile is {expert
  // (-1: none), first slot, slots}
  const i32* tiles;
  const i32* src;                // row of x for a slot, or null: the slot
  float* y32;                    // [slots, n]
  float rms_eps = -1.f;          // >= 0: rows of x over their root mean square
  const float* row_scale = nullptr;  // [m] x's rows times this
  DqRowEnd end{};
};

// DENSE: y = x W^T (+ bias) (+ residual).  Of an expert's rows, GLU: W is
// [gate | up], y [slots, n / 2] = silu(gate) * up; SLOTS: y32 in fp32.
enum DqMode { DENSE, GLU, SLOTS };

__device__ __forceinline__ float silu_mul_f(float g, float u) {
  return g / (1.f + __expf(-g)) * u;
}

// The rows of the result that a workgroup of the sum of parts can hold whole.
bool lfmq_dq_row_end_ok(int n);

// y = sum of part [splits, m, n] (row_scale: times that of its row) (+ bias)
// (+ residual), or the gate of it; end: without a gate, n that row_end_ok takes,
// vectors on 8 bytes
hipError_t lfmq_dq_rows_sum(const void* part, void* y, const void* bias,
                            const void* resid, int m, int n, int splits,
                            bool glu, hipStream_t stream,
                            const float* row_scale = nullptr,
                            const DqRowEnd* end = nullptr);
