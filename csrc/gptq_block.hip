// K13 — GPTQ's inner loop: quantize one block of columns, column by column,
// each column's rounding error pushed onto the block's later ones.
//
//   per group start:  scale, zero from the block's unquantized columns
//   q_j = clamp(round(w_j / s) + z),  e_j = (w_j - (q_j - z) s) / u_jj
//   w_c -= e_j u_jc  for the block's c > j
//
// Rows do not meet, so a row runs in 16 lanes (four rows a wave), its block
// in their registers, and the block of U in LDS for all 32 rows of a
// workgroup.  Lane c of a row holds columns 64 i + 4 c + 0..3: a row of U is
// read in 16-byte pieces side by side, the same address for all four rows.
// Bound by the chain broadcast -> quotients -> update, 128 times 0.25 us:
// 2048 rows take 34.7 us a block of 128 (56 with divisions and a search for
// the groups' starts in the chain), where one launch per elementwise
// operation took 7.2 ms (with the gaps between them).  Four rows that meet
// numbers whose quotients need a division are done again with divisions: 65
// us (tested column by column: 37 for all).
//
// Every operation rounds on its own, in the order of the tensor expressions
// above, so that results are those of a GPU tensor loop, bit by bit: no
// contraction, and a division by a constant is a product with its
// reciprocal.
#include <type_traits>

#include "common.h"

namespace {

#pragma clang fp contract(off)

constexpr int TPB = 512, RPW = 4;            // rows a wave
constexpr int ROWS = TPB / LFMQ_WAVE * RPW;  // rows a workgroup

// NaN wins, as in tensor reductions and clamps
__device__ __forceinline__ float nmin(float a, float b) {
  return b < a || b != b ? b : a;
}
__device__ __forceinline__ float nmax(float a, float b) {
  return b > a || b != b ? b : a;
}
__device__ __forceinline__ float nclamp(float x, float hi) {
  return x < 0.f ? 0.f : (x > hi ? hi : x);
}

// 1 / d, or NaN where quotient() is not x / d to the last bit: its remainders
// leave the normal range, or there is no reciprocal
__device__ __forceinline__ float inverse(float d) {
  const float r = 1.f / d;
  return fabsf(r) > 0x1p-40f && fabsf(r) < 0x1p100f ? r : NAN;
}

// x / d given r = 1 / d, both rounded to nearest: the product corrected twice
// by its remainder is the rounded quotient (Markstein), in half the steps of a
// division that starts from d alone.  NaN where the product is not finite; x
// from 2^-80 on (below, the last bit of a quotient below it may differ).
__device__ __forceinline__ float quotient(float x, float d, float r) {
  const float q0 = x * r;
  const float q1 = fmaf(fmaf(-q0, d, x), r, q0);
  return fmaf(fmaf(-q1, d, x), r, q1);
}

template <int NC>  // chunks of 64 columns
__global__ __launch_bounds__(TPB) void gptq_block_kernel(
    const float* __restrict__ w, const float* __restrict__ ub, int ldu,
    i32* __restrict__ codes, float* __restrict__ scales,
    i32* __restrict__ zeros, float* __restrict__ err, int n, int k, int G,
    int i1, int nb, int g, float qmax, float inv_range, int sym) {
  constexpr int BS = NC * 64;
  // U [nb][BS], then 1 / u_jj
  extern __shared__ __attribute__((aligned(16))) float us[];
  float* ru = us + nb * BS;
  constexpr int IN = 16;                   // loads in flight
  for (int t0 = threadIdx.x; t0 < nb * BS; t0 += IN * TPB) {
    float v[IN];
#pragma unroll
    for (int i = 0; i < IN; ++i) {
      const int t = t0 + i * TPB, r = t / BS, c = t % BS;
      v[i] = c < nb && r < nb ? ub[(size_t)r * ldu + c] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < IN; ++i)
      if (t0 + i * TPB < nb * BS) us[t0 + i * TPB] = v[i];
  }
  __syncthreads();
  for (int j = threadIdx.x; j < nb; j += TPB) ru[j] = inverse(us[j * BS + j]);
  __syncthreads();
  const int lane = threadIdx.x & 63, c16 = lane & 15;
  const int row = blockIdx.x * ROWS + (threadIdx.x >> 6) * RPW + (lane >> 4);
  const bool live = row < n;
  const float* wr = w + (u64)(live ? row : n - 1) * k;

  // the block's columns; EXACT: with divisions.  Whether the quotients were
  // those of divisions.
  auto columns = [&](auto exact) {
    constexpr bool EXACT = decltype(exact)::value;
    float v[NC * 4];
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = i * 64 + c16 * 4 + r;
        v[i * 4 + r] = c < nb ? wr[i1 + c] : 0.f;
      }
    float s = 1.f, z = 0.f, rs;
    int start = (g - i1 % g) % g;          // column where the next group starts
    if (i1 % g != 0) {                     // inside a group begun earlier
      s = scales[(u64)(live ? row : n - 1) * G + i1 / g];
      z = (float)zeros[(u64)(live ? row : n - 1) * G + i1 / g];
    }
    rs = inverse(s);
    u32 least = ~0u;                       // dividend but 0, as bits
    float finite = 0.f;                    // NaN if an error was not

#pragma unroll
    for (int i = 0; i < NC; ++i)
      for (int c = 0; c < 16; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = i * 64 + c * 4 + r;
          if (j >= nb) break;
          if (j == start) {
            start += g;
            float lo = INFINITY, hi = -INFINITY;
            for (int t = c16; t < g; t += 16) {
              const float x = wr[i1 + j + t];
              lo = nmin(lo, x);
              hi = nmax(hi, x);
            }
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) {
              lo = nmin(lo, __shfl_xor(lo, o, 64));
              hi = nmax(hi, __shfl_xor(hi, o, 64));
            }
            if (sym) {
              s = nmax(fabsf(lo), fabsf(hi)) * inv_range;
              s = s == 0.f ? 1.f : s;
              z = (qmax + 1.f) * 0.5f;
            } else {
              s = (hi - lo) * inv_range;
              s = s == 0.f ? 1.f : s;
              z = (float)(i32)nclamp(rintf(-lo / s), qmax);
            }
            rs = inverse(s);
            if (live && c16 == 0) {
              scales[(u64)row * G + (i1 + j) / g] = s;
              zeros[(u64)row * G + (i1 + j) / g] = (i32)z;
            }
          }
          const float x = __shfl(v[i * 4 + r], (lane & 48) + c, 64);
          const float u_jj = us[j * BS + j];
          const float q = nclamp(
              rintf(EXACT ? x / s : quotient(x, s, rs)) + z, qmax);
          const float y = x - (q - z) * s;
          const float e = EXACT ? y / u_jj : quotient(y, u_jj, ru[j]);
          least = min(least, (__builtin_bit_cast(u32, y) << 1) - 1u);
          finite = fmaf(e, 0.f, finite);
          if (live && c16 == 0) {
            codes[(u64)row * k + i1 + j] = (i32)q;
            err[(u64)row * nb + j] = e;
          }
#pragma unroll
          for (int i2 = i; i2 < NC; ++i2) {
            const f32x4 u = *(const f32x4*)(us + j * BS + i2 * 64 + c16 * 4);
#pragma unroll
            for (int r2 = 0; r2 < 4; ++r2)
              v[i2 * 4 + r2] = v[i2 * 4 + r2] - e * u[r2];
          }
        }
    return least >= (0x17800000u << 1) - 1u && finite == 0.f;
  };
  // no ordinary weights need the second
  if (__any(!columns(std::false_type{}))) columns(std::true_type{});
}

}  // namespace

// w [n, k] fp32 (read only), ub [nb, nb] the block of U on the diagonal, its
// rows ldu apart,
// columns i1 .. i1 + nb - 1 (nb <= 128).  Writes codes, err [n, nb] and the
// scales and zeros of groups that start in the block; a group that began in
// an earlier block is read from them.
hipError_t lfmq_gptq_block(const void* w, const void* ub, int ldu, void* codes,
                           void* scales, void* zeros, void* err, int n, int k,
                           int G, int i1, int nb, int g, int bits, bool sym,
                           hipStream_t stream) {
  if (nb < 1 || nb > 128 || i1 < 0 || i1 + nb > k || g < 1 || G * (long)g != k)
    return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  const float qmax = (float)((1 << bits) - 1);
  const float inv = sym ? 1.f / ((qmax - 1.f) / 2.f) : 1.f / qmax;
  const dim3 grid((n + ROWS - 1) / ROWS);
  const int bs = nb <= 64 ? 64 : 128;
  const size_t lds = ((size_t)nb * bs + nb) * sizeof(float);
#define GO(NC)                                                              \
  hipLaunchKernelGGL((gptq_block_kernel<NC>), grid, dim3(TPB), lds, stream, \
                     (const float*)w, (const float*)ub, ldu, (i32*)codes,   \
                     (float*)scales, (i32*)zeros, (float*)err, n, k, G, i1, \
                     nb, g, qmax, inv, (int)sym)
  if (bs == 64) GO(1);
  else GO(2);
#undef GO
  return hipGetLastError();
}
