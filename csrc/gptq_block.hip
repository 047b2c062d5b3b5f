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
// Bound by the chain broadcast -> quotients -> update, 128 times 0.13 us, so
// rows of U are read a column ahead (held there, or the compiler reads them where
// they are needed), nothing in the loop waits for stores, blocks of whole chunks
// have no tests of their end, and few rows go to workgroups of two waves, a wave a
// SIMD: 2048 rows take 20.6 us a block of 128 (25.9 with rows of U read late, a test
// a column, and a group's fit from one load after the other).  Four rows that meet
// numbers whose quotients need a division are done again with divisions.
//
// Every operation rounds on its own, in the order of the tensor expressions
// above, so that results are those of a GPU tensor loop, bit by bit: no
// contraction, and a division by a constant is a product with its
// reciprocal.
#include <algorithm>
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
  // gptq_step: errors [n, nb] of the block before and its rows of U, from this
  // block's first column on
  const float *before, *ubefore;
};

// w [rows, columns] -= before U, sixteen rows and 128 columns of four waves, as
// gptq_push takes it off (the same sums in the same order), but into LDS
template <int LD>
__device__ __forceinline__ void take_off(const BlockArgs& A, int row0,
                                         float* to) {
  const int lane = threadIdx.x & 63, l15 = lane & 15, l4 = lane >> 4;
  const int c0 = (threadIdx.x >> 6) * 32, nb = A.nb;
  const int R = min(16, A.n - row0);
  const auto er = make_rsrc(A.before + (size_t)row0 * nb, (u32)R * nb * 4);
  const auto wr = make_rsrc(A.w + (size_t)row0 * A.k, (u32)R * A.k * 4);
  auto load = [](__amdgpu_buffer_rsrc_t r, int at) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_raw_buffer_load_b32(r, at * 4, 0, 0));
  };
  constexpr int K = 128 / 4;               // products, 4 of k each
  float e[K], u[2][K], w[2][4];
#pragma unroll
  for (int s = 0; s < K; ++s) {
    e[s] = load(er, l15 * nb + s * 4 + l4);
#pragma unroll
    for (int t = 0; t < 2; ++t)
      u[t][s] = A.ubefore[(size_t)(s * 4 + l4) * A.ldu + c0 + t * 16 + l15];
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      w[t][i] = load(wr, (l4 * 4 + i) * A.k + A.i1 + c0 + t * 16 + l15);
  f32x4 acc[2] = {};
#pragma unroll
  for (int s = 0; s < K; ++s)
#pragma unroll
    for (int t = 0; t < 2; ++t)
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(e[s], u[t][s], acc[t], 0, 0, 0);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      to[(l4 * 4 + i) * LD + c0 + t * 16 + l15] = w[t][i] - acc[t][i];
}

// DMA: U comes by 16-byte pieces straight into LDS (nb whole chunks), and groups
// start on every fourth column at most.  BEFORE: the
// block's columns of w still want the errors of the block before (take_off)
template <int NC, bool DMA, bool BEFORE>   // chunks of 64 columns
__device__ __forceinline__ void block_rows(const BlockArgs& A, int tpb) {
  constexpr int BS = NC * 64, WL = BS + 4;
  const int n = A.n, k = A.k, G = A.G, i1 = A.i1, nb = A.nb, g = A.g;
  const int tid = threadIdx.x;
  const float qmax = A.qmax;
  // U [nb][BS], then {u_jj, 1 / u_jj}; BEFORE: then w [16][WL]
  extern __shared__ __attribute__((aligned(16))) float us[];
  f32x2* diag = (f32x2*)(us + nb * BS);
  float* ws = (float*)(diag + nb);
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
  if constexpr (BEFORE) {
    take_off<WL>(A, blockIdx.x * 16, ws);
    __syncthreads();
  }
  // the row's columns from i1 on
  const float* wr = BEFORE ? ws + (tid >> 4) * WL
                           : A.w + (u64)(live ? row : n - 1) * k + i1;

  struct Fit {
    float s, z, rs;
  };
  // scale and zero of the group from column j of the block on
  auto fit = [&](int j) {
    float lo = INFINITY, hi = -INFINITY;
    constexpr int IN = 8;                  // on their way at once
    for (int t0 = c16; t0 < g; t0 += 16 * IN) {
      float x[IN];
#pragma unroll
      for (int e = 0; e < IN; ++e) x[e] = wr[j + (t0 + 16 * e < g ? t0 + 16 * e : t0)];
#pragma unroll
      for (int e = 0; e < IN; ++e) {
        lo = nmin(lo, x[e]);
        hi = nmax(hi, x[e]);
      }
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
        v[i * 4 + r] = c < nb ? wr[c] : 0.f;
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
        if (!DMA && j0 >= nb) break;
        float q4[4] = {}, e4[4] = {};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = j0 + r;
          if (!DMA && j >= nb) break;
          if ((!DMA || r == 0) && j == start) {
            f = starts == 0 ? ahead[0] : (starts == 1 ? ahead[1] : fit(j));
            ++starts;
            start += g;
            if (live && c16 == 0) {
              A.scales[(u64)row * G + (i1 + j) / g] = f.s;
              A.zeros[(u64)row * G + (i1 + j) / g] = (i32)f.z;
            }
          }
          read(next, j + 1, i);
          __builtin_amdgcn_sched_barrier(0);   // here, not where it is needed
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

template <int NC, bool DMA>
__global__ __launch_bounds__(512) void gptq_block_kernel(BlockArgs A) {
  block_rows<NC, DMA, false>(A, blockDim.x);
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

struct PushArgs {
  float* w;
  const float *err, *u;
  long ldu;
  int n, k, i2, nb;
};

// a, b: PT * LA and PK * LB floats of LDS, [row][k], banks row * 4 + k, and
// [k][column], banks k * 16 + column
__device__ __forceinline__ void push_tile(const PushArgs& A, float* a, float* b,
                                          int bx, int by) {
  float* w = A.w;
  const float *err = A.err, *u = A.u;
  const long ldu = A.ldu;
  const int n = A.n, k = A.k, i2 = A.i2, nb = A.nb;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l15 = lane & 15, l4 = lane >> 4;
  const int r0 = bx * PT, c0 = i2 + by * PT;
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

__global__ __launch_bounds__(256, 3) void gptq_push_kernel(PushArgs A) {
  __shared__ float a[PT * LA], b[PK * LB];
  push_tile(A, a, b, blockIdx.x, blockIdx.y);
}

// A block's columns and what is left of the block before's push, in one launch:
// its first `rows16` workgroups take the errors off their own columns and go
// through them, a wave a SIMD, while the others carry the errors to the columns
// behind this block.  The chain of columns hides the products: a step of 2048
// x 2048 23 us at the end and 29 with all of the push, one after the other 20.6 + 6
// to 17.
__global__ __launch_bounds__(256, 2) void gptq_step_kernel(BlockArgs A,
                                                           PushArgs P,
                                                           int rows16) {
  extern __shared__ __attribute__((aligned(16))) float us[];
  if ((int)blockIdx.x < rows16) {
    __builtin_amdgcn_s_setprio(3);         // before products on the same SIMD
    block_rows<2, true, true>(A, 256);
    return;
  }
  const int id = blockIdx.x - rows16, tiles = (P.n + PT - 1) / PT;
  push_tile(P, us, us + PT * LA, id % tiles, id / tiles);
}

// The diagonal of h [k, k] as the solve wants it: d[0] with ones for zeros (columns
// without inputs), d[1] damped by `percent` of its mean, d[2] whether a column has
// inputs.  One workgroup.
__global__ __launch_bounds__(1024) void gptq_diag_kernel(
    const float* __restrict__ h, float* __restrict__ d, int k, float percent) {
  const int tid = threadIdx.x;
  __shared__ float part[16];
  float sum = 0.f;
#pragma unroll 4
  for (int i = tid; i < k; i += 1024) {
    const float x = h[(size_t)i * k + i];
    const float y = x == 0.f ? 1.f : x;
    d[i] = y;
    d[2 * (size_t)k + i] = x == 0.f ? 0.f : 1.f;
    sum += y;
  }
  sum = wave_reduce_sum(sum);
  if ((tid & 63) == 0) part[tid >> 6] = sum;
  __syncthreads();
  float all = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) all += part[i];
  const float damp = percent * (all / (float)k);
  for (int i = tid; i < k; i += 1024) d[(size_t)k + i] = d[i] + damp;
}

// to = w, zeros in columns without inputs; a row of workgroups a row
__global__ __launch_bounds__(256) void gptq_copy_kernel(
    const float* __restrict__ w, const float* __restrict__ on,
    float* __restrict__ to, int n, int k) {
  const int c = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (c >= k) return;
  for (int r = blockIdx.y; r < n; r += gridDim.y) {
    const float* p = w + (size_t)r * k + c;
    float* q = to + (size_t)r * k + c;
    if (k % 4 == 0 && ((u64)w | (u64)to | (u64)on) % 16 == 0) {
      const f32x4 x = *(const f32x4*)p, o = *(const f32x4*)(on + c);
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = o[e] == 0.f ? 0.f : x[e];
      *(f32x4*)q = y;
    } else {
      for (int e = 0; e < 4 && c + e < k; ++e)
        q[e] = on[c + e] == 0.f ? 0.f : p[e];
    }
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
                    nb, g, qmax, inv, sym, wide, nullptr, nullptr};
  // a wave a SIMD while they last (2048 rows, with rows of U read
  // late, 31 us in eight waves, 26 in two),
  // then U read less often
  const int tpb = n <= 4096 ? 128 : (n <= 8192 ? 256 : 512);
  const dim3 grid((n + tpb / 16 - 1) / (tpb / 16));
  const int bs = nb <= 64 ? 64 : 128;
  const size_t lds = ((size_t)nb * bs + 2 * nb) * sizeof(float);
  const bool dma = nb == bs && g % 4 == 0 && i1 % 4 == 0 && ldu % 4 == 0 && (u64)ub % 16 == 0 &&
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
                     0, stream,
                     PushArgs{(float*)w, (const float*)err, (const float*)u,
                              ldu, n, k, i2, nb});
  return hipGetLastError();
}

// Whether whole blocks of 128 columns go by lfmq_gptq_step: groups that start in a
// block end in it, since the columns behind it change meanwhile; U for 16-byte
// pieces; rows of a workgroup a CU at most (8192 rows: 27 us a block in 256
// workgroups of two waves a SIMD, which leave the products no room).
bool lfmq_gptq_step_ok(const void* u, long ldu, int n, int k, int g) {
  return n >= 1 && n <= 4096 && g >= 4 && 128 % g == 0 && ldu % 4 == 0 &&
         (u64)u % 16 == 0 && 128ull * ldu * 4 < 1ull << 32 &&
         (u64)16 * k * 4 < 1ull << 31 && k / PT <= 65535;
}

// The columns i1 .. i1 + 127 (i1 >= 128), whose w wants the errors `before` [n,
// 128] of the 128 columns in front, and these errors' push to the columns behind.
// u: the whole factor; err another buffer than before.  Otherwise as
// lfmq_gptq_block.
hipError_t lfmq_gptq_step(const void* w, const void* u, long ldu, void* codes,
                          void* scales, void* zeros, const void* before,
                          void* err, int n, int k, int G, int i1, int g,
                          int bits, bool sym, hipStream_t stream) {
  if (!lfmq_gptq_step_ok(u, ldu, n, k, g) || i1 < 128 || i1 + 128 > k ||
      i1 % g != 0 || G * (long)g != k)
    return hipErrorInvalidValue;
  const float qmax = (float)((1 << bits) - 1);
  const float inv = sym ? 1.f / ((qmax - 1.f) / 2.f) : 1.f / qmax;
  const bool wide = k % 4 == 0 && ((u64)codes | (u64)err) % 16 == 0;
  const float* ut = (const float*)u;
  const float* prow = ut + (size_t)(i1 - 128) * ldu;
  const BlockArgs A{(const float*)w, ut + (size_t)i1 * ldu + i1, (i32*)codes,
                    (float*)scales, (i32*)zeros, (float*)err, (int)ldu, n, k, G,
                    i1, 128, g, qmax, inv, sym, wide, (const float*)before,
                    prow + i1};
  const PushArgs P{(float*)w, (const float*)before, prow, ldu, n, k, i1 + 128, 128};
  const int rows16 = (n + 15) / 16;
  const int tiles = (n + PT - 1) / PT * ((k - i1 - 128 + PT - 1) / PT);
  const size_t lds = (128 * 128 + 2 * 128 + 16 * 132) * sizeof(float);
  static_assert(PT * LA + PK * LB <= 128 * 128, "a push fits");
  static bool set = false;
  if (!set) {
    LFMQ_CHECK_HIP(hipFuncSetAttribute(
        (const void*)gptq_step_kernel,
        hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024));
    set = true;
  }
  hipLaunchKernelGGL(gptq_step_kernel, dim3(rows16 + tiles), dim3(256), lds,
                     stream, A, P, rows16);
  return hipGetLastError();
}

// d [3, k] of h [k, k] (gptq_diag_kernel); to = w [n, k] without the columns that
// have no inputs.  Two launches, where tensor operations take twelve and a wait
// for the device.
hipError_t lfmq_gptq_prepare(const void* w, const void* h, void* to, void* d,
                             int n, int k, float percent, hipStream_t stream) {
  if (n < 0 || k < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(gptq_diag_kernel, dim3(1), dim3(1024), 0, stream,
                     (const float*)h, (float*)d, k, percent);
  if (n > 0)
    hipLaunchKernelGGL(gptq_copy_kernel,
                       dim3((k + 1023) / 1024, std::min(n, 65535)), dim3(256), 0,
                       stream, (const float*)w, (const float*)d + 2 * (size_t)k,
                       (float*)to, n, k);
  return hipGetLastError();
}
