// K13 — GPTQ's inner loop: quantize one block of columns, column by column,
// each column's rounding error pushed onto the block's later ones.
//
//   per group start:  scale, zero from the block's unquantized columns
//   q_j = clamp(round(w_j / s) + z),  e_j = (w_j - (q_j - z) s) / u_jj
//   w_c -= e_j u_jc  for the block's c > j
//
// Rows do not meet, so a row runs in 16 lanes (four rows a wave), its block
// in their registers, and the block of U in LDS for all rows of a workgroup.
// Lane c of a row holds columns 64 i + 4 c + 0..3 at first: a row of U is read
// in 16-byte pieces side by side, the same address for all four rows.  The
// columns in turn are always the first lane's, which a lane permutation hands
// to the others (through LDS, as from any lane, it is 100 cycles of the chain).
// Bound by the chain broadcast -> quotients -> update, 128 times 0.18 us, so
// rows of U are read a column ahead, nothing in the loop waits for stores, and
// few rows go to workgroups of two waves, a wave a SIMD: 2048 rows take 25.1
// us a block of 128 (35.1 in eight waves with the reads in the chain), 8192
// rows 27.2 (35.9), 28672 72 (87).  Four rows that meet numbers whose quotients
// need a division are done again with divisions.
//
// Every operation rounds on its own, in the order of the tensor expressions
// above, so that results are those of a GPU tensor loop, bit by bit: no
// contraction, and a division by a constant is a product with its
// reciprocal.
#include <type_traits>

#include "lds_dma.h"

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef i32 i32x4 __attribute__((ext_vector_type(4)));

#pragma clang fp contract(off)

constexpr int RPW = 4;                       // rows a wave

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

// lane 0's value of each row of 16 lanes, and the next lane's (15: lane 0's)
__device__ __forceinline__ float first_lane(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150,
                                         0xf, 0xf, true));
}
__device__ __forceinline__ float next_lane(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x12F,
                                         0xf, 0xf, true));
}

struct BlockArgs {
  const float *w, *ub;
  i32* codes;
  float* scales;
  i32* zeros;
  float* err;
  int ldu, n, k, G, i1, nb, g;
  float qmax, inv_range;
  bool sym, wide;          // wide: codes and errors in pieces of 16 bytes
};

// DMA: U comes by 16-byte pieces straight into LDS (nb whole chunks)
template <int NC, bool DMA>  // chunks of 64 columns
__global__ __launch_bounds__(512) void gptq_block_kernel(BlockArgs A) {
  constexpr int BS = NC * 64;
  const int n = A.n, k = A.k, G = A.G, i1 = A.i1, nb = A.nb, g = A.g;
  const int tpb = blockDim.x, tid = threadIdx.x;
  const float qmax = A.qmax;
  // U [nb][BS], then {u_jj, 1 / u_jj}
  extern __shared__ __attribute__((aligned(16))) float us[];
  f32x2* diag = (f32x2*)(us + nb * BS);
  if constexpr (DMA) {
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int RL = 256 / BS;           // rows of U a load
    for (int i = wave; i < BS / RL; i += tpb / LFMQ_WAVE) {
      const int e = i * 256 + (tid & 63) * 4;
      load_to_lds(A.ub, ((u32)(e / BS) * (u32)A.ldu + e % BS) * 4, i * 1024);
    }
  } else {
    constexpr int IN = 16;                 // loads in flight
    for (int t0 = tid; t0 < nb * BS; t0 += IN * tpb) {
      float v[IN];
#pragma unroll
      for (int i = 0; i < IN; ++i) {
        const int t = t0 + i * tpb, r = t / BS, c = t % BS;
        v[i] = c < nb && r < nb ? A.ub[(size_t)r * A.ldu + c] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < IN; ++i)
        if (t0 + i * tpb < nb * BS) us[t0 + i * tpb] = v[i];
    }
  }
  const int lane = tid & 63, c16 = lane & 15;
  const int row = blockIdx.x * (tpb / 16) + (tid >> 6) * RPW + (lane >> 4);
  const bool live = row < n;
  const float* wr = A.w + (u64)(live ? row : n - 1) * k;

  struct Fit {
    float s, z, rs;
  };
  // scale and zero of the group from column j of the block on
  auto fit = [&](int j) {
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
    Fit f;
    if (A.sym) {
      f.s = nmax(fabsf(lo), fabsf(hi)) * A.inv_range;
      f.s = f.s == 0.f ? 1.f : f.s;
      f.z = (qmax + 1.f) * 0.5f;
    } else {
      f.s = (hi - lo) * A.inv_range;
      f.s = f.s == 0.f ? 1.f : f.s;
      f.z = (float)(i32)nclamp(rintf(-lo / f.s), qmax);
    }
    f.rs = inverse(f.s);
    return f;
  };
  // the first two groups' while U is on its way
  const int start0 = (g - i1 % g) % g;     // column where the next group starts
  Fit ahead[2] = {};
#pragma unroll
  for (int t = 0; t < 2; ++t)
    if (start0 + t * g < nb) ahead[t] = fit(start0 + t * g);
  Fit begun = {1.f, 0.f, 0.f};
  if (i1 % g != 0) {                       // inside a group begun earlier
    begun.s = A.scales[(u64)(live ? row : n - 1) * G + i1 / g];
    begun.z = (float)A.zeros[(u64)(live ? row : n - 1) * G + i1 / g];
  }
  begun.rs = inverse(begun.s);
  if constexpr (DMA) lds_loads_done();
  else __syncthreads();
  for (int j = tid; j < nb; j += tpb) {
    const float d = us[j * BS + j];
    diag[j] = f32x2{d, inverse(d)};
  }
  __syncthreads();

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
        // here, or every round waits for the stores of the one before
        asm volatile("" : "+v"(v[i * 4 + r]));
      }
    int start = start0, starts = 0;
    Fit f = begun;
    // row j of U and its diagonal, read a column ahead
    struct Row {
      f32x4 u[NC];
      f32x2 d;
    } now, next;
    auto read = [&](Row& o, int j, int from) {
      j = min(j, nb - 1);
      const float* p = us + j * BS + ((c16 + (j >> 2)) & 15) * 4;
#pragma unroll
      for (int i = 0; i < NC; ++i)
        if (i >= from) o.u[i] = *(const f32x4*)(p + i * 64);
      o.d = diag[j];
    };
    read(now, 0, 0);
    u32 least = ~0u;                       // dividend but 0, as bits
    float finite = 0.f;                    // NaN if an error was not

    // the columns of a chunk in turn are lane 0's: after four of them all
    // lanes take the next lane's (a broadcast from lane c goes through LDS)
#pragma unroll
    for (int i = 0; i < NC; ++i)
      for (int c = 0; c < 16; ++c) {
        const int j0 = i * 64 + c * 4;
        if (j0 >= nb) break;
        float q4[4] = {}, e4[4] = {};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = j0 + r;
          if (j >= nb) break;
          if (j == start) {
            f = starts == 0 ? ahead[0] : (starts == 1 ? ahead[1] : fit(j));
            ++starts;
            start += g;
            if (live && c16 == 0) {
              A.scales[(u64)row * G + (i1 + j) / g] = f.s;
              A.zeros[(u64)row * G + (i1 + j) / g] = (i32)f.z;
            }
          }
          read(next, j + 1, i);
          const float x = first_lane(v[i * 4 + r]);
          const float t = EXACT ? x / f.s : quotient(x, f.s, f.rs);
          // (the median of a NaN is not NaN: seen by `finite`)
          const float q = EXACT ? nclamp(rintf(t) + f.z, qmax)
                                : __builtin_amdgcn_fmed3f(rintf(t) + f.z, 0.f,
                                                          qmax);
          const float y = x - (q - f.z) * f.s;
          const float e = EXACT ? y / now.d[0] : quotient(y, now.d[0], now.d[1]);
          least = min(least, (__builtin_bit_cast(u32, y) << 1) - 1u);
          finite = fmaf(t, 0.f, fmaf(e, 0.f, finite));
          q4[r] = q;
          e4[r] = e;
#pragma unroll
          for (int i2 = i; i2 < NC; ++i2)
#pragma unroll
            for (int r2 = 0; r2 < 4; ++r2)
              v[i2 * 4 + r2] = v[i2 * 4 + r2] - e * now.u[i2][r2];
          now = next;
        }
        if (live && c16 == 0) {
          i32* pc = A.codes + (u64)row * k + i1 + j0;
          float* pe = A.err + (u64)row * nb + j0;
          if (A.wide) {
            *(i32x4*)pc = i32x4{(i32)q4[0], (i32)q4[1], (i32)q4[2],
                                (i32)q4[3]};
            *(f32x4*)pe = f32x4{e4[0], e4[1], e4[2], e4[3]};
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (j0 + r < nb) {
                pc[r] = (i32)q4[r];
                pe[r] = e4[r];
              }
          }
        }
#pragma unroll
        for (int t = i * 4; t < NC * 4; ++t) v[t] = next_lane(v[t]);
      }
    return least >= (0x17800000u << 1) - 1u && finite == 0.f;
  };
  // no ordinary weights need the second
  if (__any(!columns(std::false_type{}))) columns(std::true_type{});
}

// w[:, i2:] -= err U[i1:i2, i2:]: the later columns learn of a block's errors.
// A workgroup 64 x 64, K in 64s through LDS, fp32 matrix instructions, the
// product summed apart and rounded once at the size of w.  Bound by the load
// of both operands before the products and, from some 1000 workgroups on, by
// the products.  Over the blocks of 2048 x 2048 11.0 us a product on average
// (the library 14.5), of 4096 x 4096 28.6 (37.4), of 8192 x 2048 28.6 (35.3).  A
// small product repeated on operands that the caches hold takes the library
// less (4.6, here 6.9).  K whole in LDS, two workgroups a CU: 15.1 for 11.4.
constexpr int PT = 64, PK = 64, LA = PK + 4, LB = PT + 16;

__global__ __launch_bounds__(256, 3) void gptq_push_kernel(
    float* __restrict__ w, const float* __restrict__ err,
    const float* __restrict__ u, long ldu, int n, int k, int i2, int nb) {
  // [row][k], banks row * 4 + k; [k][column], banks k * 16 + column
  __shared__ float a[PT * LA], b[PK * LB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l15 = lane & 15, l4 = lane >> 4;
  const int r0 = blockIdx.x * PT, c0 = i2 + blockIdx.y * PT;
  const int ro = wave / 2 * 32, co = wave % 2 * 32;
  constexpr int PL = PT * PK / 256;
  // loads with bounds: rows past the last one are zeros (columns past it, the
  // next row's, are not stored)
  const int R = min(PT, n - r0);
  const auto er = make_rsrc(err + (size_t)r0 * nb, (u32)R * nb * 4);
  const auto ur = make_rsrc(u, (u32)(((nb - 1) * ldu + k) * 4));
  const auto wr = make_rsrc(w + (size_t)r0 * k, (u32)(((size_t)R * k) * 4));
  float va[PL], vb[PL];
  const u32 ao = (u32)(tid / PK * nb + tid % PK) * 4;
  const u32 bo = (u32)(tid / PT * ldu + c0 + tid % PT) * 4;
  auto fetch = [&](int k0) {
    const bool in = k0 + tid % PK < nb;
#pragma unroll
    for (int t = 0; t < PL; ++t) {
      const float x = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(
                     er, ao + (u32)(t * (256 / PK) * nb + k0) * 4, 0, 0));
      va[t] = in ? x : 0.f;
      vb[t] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(
                     ur, bo + (u32)((k0 + t * (256 / PT)) * ldu) * 4, 0, 0));
    }
  };
  f32x4 acc[2][2] = {};
  float old[2][2][4];
  fetch(0);
  for (int k0 = 0; k0 < nb; k0 += PK) {
    if (k0 != 0) __syncthreads();          // the step before is read
#pragma unroll
    for (int t = 0; t < PL; ++t) {
      const int e = t * 256 + tid;
      a[e / PK * LA + e % PK] = va[t];
      b[e / PT * LB + e % PT] = vb[t];
    }
    __syncthreads();
    if (k0 + PK < nb) {
      fetch(k0 + PK);
    } else {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int r = ro + x * 16 + l4 * 4 + i, c = c0 + co + y * 16 + l15;
            old[x][y][i] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(
                           wr, (u32)(r * k + c) * 4, 0, 0));
          }
    }
#pragma unroll 4
    for (int s = 0; s < PK / 4; ++s) {
      float av[2], bv[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        av[x] = a[(ro + x * 16 + l15) * LA + s * 4 + l4];
        bv[x] = b[(s * 4 + l4) * LB + co + x * 16 + l15];
      }
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[x], bv[y],
                                                           acc[x][y], 0, 0, 0);
    }
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = r0 + ro + x * 16 + l4 * 4 + i, c = c0 + co + y * 16 + l15;
        if (r < n && c < k) w[(size_t)r * k + c] = old[x][y][i] - acc[x][y][i];
      }
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
  const bool wide = k % 4 == 0 && i1 % 4 == 0 && nb % 4 == 0 &&
                    ((u64)codes | (u64)err) % 16 == 0;
  const BlockArgs A{(const float*)w, (const float*)ub, (i32*)codes,
                    (float*)scales, (i32*)zeros, (float*)err, ldu, n, k, G, i1,
                    nb, g, qmax, inv, sym, wide};
  // a wave a SIMD while they last (2048 rows 31 us in eight waves, 26 in two),
  // then U read less often
  const int tpb = n <= 4096 ? 128 : (n <= 8192 ? 256 : 512);
  const dim3 grid((n + tpb / 16 - 1) / (tpb / 16));
  const int bs = nb <= 64 ? 64 : 128;
  const size_t lds = ((size_t)nb * bs + 2 * nb) * sizeof(float);
  const bool dma = nb == bs && ldu % 4 == 0 && (u64)ub % 16 == 0 &&
                   (u64)nb * ldu * 4 < 1ull << 32;
#define GO(NC, DMA)                                                          \
  do {                                                                       \
    static bool set = false;                                                 \
    if (NC > 1 && !set) {                                                    \
      LFMQ_CHECK_HIP(hipFuncSetAttribute(                                    \
          (const void*)gptq_block_kernel<NC, DMA>,                           \
          hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024));           \
      set = true;                                                            \
    }                                                                        \
    hipLaunchKernelGGL((gptq_block_kernel<NC, DMA>), grid, dim3(tpb), lds,   \
                       stream, A);                                           \
  } while (0)
  if (bs == 64) {
    if (dma) GO(1, true);
    else GO(1, false);
  } else {
    if (dma) GO(2, true);
    else GO(2, false);
  }
#undef GO
  return hipGetLastError();
}

// w [n, k] fp32, err [n, nb], u: rows i1 .. i1 + nb - 1 of the
// factor, whole (columns 0 .. k - 1), ldu apart; columns i2 .. k - 1 of w
// change
hipError_t lfmq_gptq_push(const void* w, const void* err, const void* u, long ldu,
                          int n, int k, int i2, int nb, hipStream_t stream) {
  if (nb < 1 || (u64)nb * ldu * 4 >= 1ull << 32 || i2 < 0 || i2 > k || (k + PT - 1) / PT > 65535)
    return hipErrorInvalidValue;
  if (n == 0 || i2 == k) return hipSuccess;
  hipLaunchKernelGGL(gptq_push_kernel,
                     dim3((n + PT - 1) / PT, (k - i2 + PT - 1) / PT), dim3(256),
                     0, stream, (float*)w, (const float*)err,
                     (const float*)u, ldu, n, k, i2, nb);
  return hipGetLastError();
}
