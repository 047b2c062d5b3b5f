// K3f/K4f — W4A16 / W8A16 product for prompts of many rows: y[m, n] = x[m, k] ·
// dequant(W)[n, k]^T (+ bias), with the gate behind it, or by expert.
//
// A workgroup of eight waves computes up to 128 rows by 256 columns, a wave all
// rows by 32 columns.  x and the packed weights go from memory straight into
// LDS, three stages of 128 values of k (64 with groups of 64, and 8 bits), so
// that a chunk's loads have two chunks' time; scales and zeros come eight groups
// at a time.  A row tile's products hide the sums of the one before, the
// unpacking of the next chunk's weights and the loads, one after the other; the
// barrier between chunks stands before the last row tile's products.  Nothing
// in the loop branches but on the chunk's place in its four: with a branch a
// row tile for loads past the end, and for the one wave that sums x, 1.05 times
// as long.
//
// sum s (c - z) x = s (sum c x) - (s z) (sum x): the second term is a product
// with one k a chunk, made four chunks at a time by an fp32 matrix instruction,
// instead of as many fp32 additions as the first takes.  int4 codes are exact
// bf16 numbers c here, not 128 + c, so less cancels.
//
// Where the tiles leave a last round of workgroups half empty, its tiles' k is
// split and a second launch adds the parts (3001 rows: n 4096, k 14336 399 us,
// 343 so; n 6144, k 4096 172, 164).
//
// What is large (rows k (n - 2048) from 12 2^30 on, 8 2^30 with stages of 64) is
// dq_panel's now, which measures itself against this kernel; the calls below that
// are marked * are among it, and so is what the next lines are about.
//
// Bound by the matrix cores (busy 57 % of the time), by what the two waves of a
// SIMD wait for together at the barrier, and by 7 us of first loads and last
// stores of a tile of 66 that nothing covers.  us a call, dq_tile and this one
// (4 bits; 8 bits with groups of 64 at k 2048 and 8192):
//                       200 rows      500 rows      1500 rows     3001 rows
//   n 28672, k 4096   80.2 / 63.4*  155 / 137*    438 / 368*    815 / 703*
//   n 6144, k 4096    33.0 / 28.6   51.1 / 41.8   118 / 90.2*   205 / 164*
//   n 4096, k 14336   51.8 / 41.3   91.5 / 77.8*  230 / 180*    451 / 343*
//   n 16384, k 2048   42.6 / 34.7   60.9 / 48.6*  176 / 141*    330 / 272*
//   n 2048, k 8192    30.5 / 27.6   45.5 / 37.8   125 / 88.5    199 / 146
// Without effect: the order of products and sums, wave priorities, x fetched two
// row tiles ahead.  LDS slots that pairs of lanes share (slot_key): 767 us
// instead of 710 at n 28672, 3001 rows.
#include <type_traits>

#include "dq_block.h"
#include "lds_dma.h"

namespace {

typedef DqBlockPlan Plan;

constexpr int NW = 8, TPB = NW * LFMQ_WAVE, NT = 2, BN = NW * NT * 16;
constexpr int ROWS = 128;                        // of a tile, at most
constexpr int D = 3;                             // stages

// LDS: x [D][rows][KC], weights [D][NW][..], two blocks of scales and of zeros
// of eight groups, eight chunks' sums of x
template <int BITS, int KC>
struct Lds {
  static constexpr int XB = ROWS * KC * 2, WB = NT * 16 * KC * BITS / 8;
  static constexpr int W = D * XB, S = W + D * NW * WB;
  static constexpr int SB = BN * 16, ZB = BN * BITS;
  static constexpr int Z = S + 2 * SB, SUM = Z + 2 * ZB;
  static constexpr int BYTES = SUM + 8 * ROWS * 4;
  static_assert(BYTES <= 160 * 1024 && BYTES >= ROWS * (BN + 8) * 2, "");
};

// the result's tile of column block nblk, part of it
template <int BITS, int KC, DqMode MODE, int MT>
__device__ __forceinline__ void dq_block_body(const DqArgs& A, char* smem,
                                              int row0, int rows, int expert,
                                              int nblk, int sp, int parts,
                                              float* part) {
  typedef Lds<BITS, KC> L;
  constexpr int BM = MT * 16, J = KC / 32, WD = J * BITS / 4;
  constexpr int SL = KC / 8;                     // 16-byte slots a row of x
  constexpr int XL = BM * KC * 2 / 1024;         // 1 KiB loads of x a stage
  constexpr int NX = (XL + NW - 1) / NW;         // of a wave, at most
  constexpr int NL = L::WB / 1024;               // of a wave's weights
  constexpr int PC = KC * BITS / 128;            // 16-byte pieces a column
  float* xsum = (float*)(smem + L::SUM);         // [8][ROWS]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4;
  const int C = A.k / KC;
  const int c0 = (int)((long)C * sp / parts);
  const int c1 = (int)((long)C * (sp + 1) / parts);
  const int G = A.k / A.g, zw = (G + 32 / BITS - 1) / (32 / BITS);
  const int cpg = A.g / KC;                      // chunks a group
  const int half = A.n / 2, n0 = nblk * (MODE == GLU ? BN / 2 : BN);
  // column c of this workgroup: row of W.  GLU: a wave's first 16 are gate,
  // the others up
  auto column = [&](int c) {
    if (MODE == GLU)
      return (c >> 4 & 1) * half + min(n0 + (c >> 5) * 16 + (c & 15), half - 1);
    return min(n0 + c, A.n - 1);
  };
  // staging: a lane picks the 16 bytes that belong at its place; rows past
  // the end repeat the last one
  const char* xb = (const char*)(MODE == DENSE ? A.x + (u64)row0 * A.k : A.x);
  const u32 pitch = A.k * 2;
  u32 xo[NX];
  // (where the waves share a stage's loads unevenly, some do the last one again)
  auto nth = [&](int i) {
    return XL % NW == 0 ? i * NW + wave : min(i * NW + wave, XL - 1);
  };
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int at = nth(i) * (64 / SL) + lane / SL;
    int r = min(at, rows - 1);
    if (MODE != DENSE) {
      r += row0;
      if (A.src != nullptr) r = A.src[r];
    }
    xo[i] = (u32)r * pitch + ((lane % SL) ^ slot_key16<SL>(at)) * 16;
  }
  const u32 wrow = A.k * BITS / 8;
  const u64 first = (u64)expert * A.n;           // the expert's rows of W
  const char* wb = A.w + first * wrow;
  u32 wo[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int e = i * 64 + lane, c = e / PC;
    int p = e % PC;
    if constexpr (PC >= 4) p ^= slot_key16<PC>(c & 15);
    wo[i] = (u32)column(wave * NT * 16 + c) * wrow + p * 16;
  }
  auto load_x = [&](int c, int buf, int i) {
    load_to_lds(xb + (u64)c * (KC * 2), xo[i], buf * L::XB + nth(i) * 1024);
  };
  auto load_w = [&](int c, int buf, int i) {
    load_to_lds(wb + (u32)c * (KC * BITS / 8), wo[i],
                L::W + (buf * NW + wave) * L::WB + i * 1024);
  };
  // scales and zeros of groups 8 q .. 8 q + 7: half of the waves each
  const u32 mcol = column((wave & 3) * 64 + lane);
  auto load_meta = [&](int q) {
    if (wave < 4) {
      load_to_lds((const char*)(A.scales + first * G) + q * 16, mcol * (G * 2),
                  L::S + (q & 1) * L::SB + wave * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < BITS / 4; ++i)
        load4_to_lds((const char*)(A.zeros + first * zw) + q * BITS + i * 4,
                     mcol * (zw * 4),
                     L::Z + (q & 1) * L::ZB + i * BN * 4 + (wave - 4) * 256);
    }
  };

  f32x4 acc[MT][NT] = {};
  s16x8 ones = bf16_ones();
  asm volatile("" : "+v"(ones));                // kept, not made anew
  // Scale times zero of four chunks, chunk i in lane group i: of this four, and
  // of the four before until acc -= (scale times zero) (sums of x), in fp32
  float szq[NT] = {}, szp[NT] = {};
  auto sum_of = [&](int quad, int t) {
    return -xsum[((quad & 1) * 4 + l4) * ROWS + t * 16 + l15];
  };
  auto zeros_of = [&](float v, int t, const float (&sz)[NT]) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      acc[t][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, sz[nt], acc[t][nt],
                                                        0, 0, 0);
  };
  auto read_w = [&](int buf, u32 (&w)[NT][WD]) {
    const char* ws = smem + L::W + (buf * NW + wave) * L::WB;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const char* p = ws + (t * 16 + l15) * (PC * 16);
      if constexpr (WD == 2) {
        typedef u32 u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 v = *(const u32x2*)(p + l4 * 8);
        w[t][0] = v[0];
        w[t][1] = v[1];
      } else {
#pragma unroll
        for (int i = 0; i < WD / 4; ++i) {
          const u32x4 v = *(const u32x4*)(
              p + (((l4 * (WD / 4) + i) ^ slot_key16<PC < 4 ? 4 : PC>(l15)) << 4));
#pragma unroll
          for (int e = 0; e < 4; ++e) w[t][i * 4 + e] = v[e];
        }
      }
    }
  };
  struct Meta {
    u32 s, z;
  };
  auto read_meta = [&](int gi, Meta (&o)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int col = (wave * NT + t) * 16 + l15;
      o[t].s = *(const unsigned short*)(smem + L::S + (gi >> 3 & 1) * L::SB +
                                        col * 16 + (gi & 7) * 2);
      o[t].z = *(const u32*)(smem + L::Z + (gi >> 3 & 1) * L::ZB +
                             (BITS == 8 ? (gi >> 2 & 1) * BN * 4 : 0) +
                             col * 4);
    }
  };
  float s[NT], sz[NT];           // of a chunk's group
  auto use_meta = [&](int gi, const Meta (&o)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      s[t] = bf16_bits_to_f32(o[t].s);
      sz[t] = s[t] * (float)(BITS == 4 ? unpack4(o[t].z, gi & 7)
                                       : unpack8(o[t].z, gi & 3));
    }
  };

  int gi = c0 / cpg, gc = c0 % cpg;              // group, chunk in it
  const int q0 = gi >> 3;
  s16x8 b[2][NT][J], xa[2][J];
  u32 w[NT][WD];
  Meta meta[NT];
  int buf = 0;                                   // of chunk c: x, and W before
  auto load = [&](int buf, int row, int j) {
    return *(const s16x8*)(smem + buf * L::XB + row * (KC * 2) +
                           (((l4 * J + j) ^ slot_key16<SL>(l15)) << 4));
  };
  {
#pragma unroll
    for (int i = 0; i < NL; ++i) load_w(c0, 0, i);
    load_meta(q0);
    if (8 * (q0 + 1) < G) load_meta(q0 + 1);
    for (int i = tid; i < 8 * ROWS; i += TPB) xsum[i] = 0.f;
#pragma unroll
    for (int t = 0; t < D - 1; ++t) {
#pragma unroll
      for (int i = 0; i < NX; ++i) load_x(min(c0 + t, c1 - 1), t, i);
#pragma unroll
      for (int i = 0; i < NL; ++i) load_w(min(c0 + t + 1, c1 - 1), t + 1, i);
    }
    loads_but<0>();
    read_w(0, w);
    read_meta(gi, meta);
#pragma unroll
    for (int j = 0; j < J; ++j) xa[0][j] = load(0, l15, j);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < J; ++j)
        b[0][t][j] = codes8_exact<BITS>(&w[t][j * BITS / 4]);
    use_meta(gi, meta);
  }
  // Q: the chunk's place in its four.  Loads past the last chunk repeat it.
  auto chunk = [&](int c, auto place) {
    constexpr int Q = decltype(place)::value, P = Q & 1;
    const int b1 = buf == D - 1 ? 0 : buf + 1, b2 = b1 == D - 1 ? 0 : b1 + 1;
    if (gc == 0 && (gi & 7) == 0 && gi >> 3 != q0 && gi + 8 < G)
      load_meta((gi >> 3) + 1);
    if (++gc == cpg) {
      gc = 0;
      ++gi;
    }
    // the next chunk's weights and scales (past the last one, whatever lies
    // there is read and not used)
    read_w(b1, w);
    read_meta(gi, meta);
    const int quad = (c - c0) >> 2;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if constexpr (Q == 0) {
        szp[t] = szq[t];
        szq[t] = 0.f;
      }
      szq[t] = l4 == Q ? sz[t] : szq[t];
    }
    // a chunk later than its sums of x were written last
    if (Q == 1 && quad > 0) {
      float v[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) v[t] = sum_of(quad - 1, t);
#pragma unroll
      for (int t = 0; t < MT; ++t) zeros_of(v[t], t, szp);
    }
    f32x4 a[2][NT], xsm = {0.f, 0.f, 0.f, 0.f};
    s16x8 xo1[J];                          // this wave's row tile, for its sums
    auto fold = [&](int t) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[t][nt][r] = fmaf(s[nt], a[t & 1][nt][r], acc[t][nt][r]);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) asm volatile("" : "+v"(acc[t][nt]));
    };
    constexpr int ITEMS = NX + NL, F = NT * J;
    const int cx = min(c + 2, c1 - 1), cw = min(c + 3, c1 - 1);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      if (t + 1 < MT) {
#pragma unroll
        for (int j = 0; j < J; ++j)
          xa[(t + 1) & 1][j] = load(buf, (t + 1) * 16 + l15, j);
        // what comes goes where the chunk before has been read
#pragma unroll
        for (int i = t * ITEMS / (MT - 1); i < (t + 1) * ITEMS / (MT - 1); ++i) {
          if (i < NX) load_x(cx, b2, i);
          else load_w(cw, buf, i - NX);
        }
        if (t == 0)
#pragma unroll
          for (int j = 0; j < J; ++j)
            xo1[j] = load(buf, min(wave, MT - 1) * 16 + l15, j);
      } else {
        // x of the next chunk and the weights after it have landed, and all
        // waves have read this one's x: the last products are still to come
        loads_but<NX + NL>();
#pragma unroll
        for (int j = 0; j < J; ++j) xa[0][j] = load(b1, l15, j);
      }
      static_assert(MT % 2 == 0, "the next chunk's first rows go to xa[0]");
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) a[t & 1][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < J; ++j) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          a[t & 1][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              xa[t & 1][j], b[P][nt][j], a[t & 1][nt], 0, 0, 0);
        if (t == (MT > 2 ? 2 : 1))
          xsm = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xo1[j], ones, xsm, 0, 0,
                                                        0);
      }
      if (t > 0) fold(t - 1);
#pragma unroll
      for (int f = t * F / MT; f < (t + 1) * F / MT; ++f)
        b[P ^ 1][f / J][f % J] = codes8_exact<BITS>(&w[f / J][f % J * BITS / 4]);
      __builtin_amdgcn_sched_barrier(0);
    }
    fold(MT - 1);
    if (wave < MT && l15 == 0)
      *(f32x4*)(xsum + ((quad & 1) * 4 + Q) * ROWS + wave * 16 + l4 * 4) = xsm;
    use_meta(gi, meta);
    buf = b1;
  };
  static_assert(MT <= NW, "a row tile's sums of x a wave");
  for (int c = c0; c < c1; c += 4) {
    chunk(c, std::integral_constant<int, 0>{});
    if (c + 1 == c1) break;
    chunk(c + 1, std::integral_constant<int, 1>{});
    if (c + 2 == c1) break;
    chunk(c + 2, std::integral_constant<int, 2>{});
    if (c + 3 == c1) break;
    chunk(c + 3, std::integral_constant<int, 3>{});
  }
  loads_but<0>();
  const int end = c1 - c0 - 1;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    if (end >= 4 && (end & 3) == 0) zeros_of(sum_of((end >> 2) - 1, t), t, szp);
    zeros_of(sum_of(end >> 2, t), t, szq);
  }

  // C fragment: column l15, rows l4 * 4 + r
  if (part != nullptr) {                         // [rows][BN], as the waves lie
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = t * 16 + l4 * 4 + r;
        if (row < rows)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
            part[row * BN + (wave * NT + nt) * 16 + l15] = acc[t][nt][r];
      }
    return;
  }
  if (MODE == SLOTS) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = t * 16 + l4 * 4 + r;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int col = n0 + (wave * NT + nt) * 16 + l15;
          if (row < rows && col < A.n)
            A.y32[(u64)(row0 + row) * A.n + col] = acc[t][nt][r];
        }
      }
    return;
  }
  // through LDS, so that rows are written in 16-byte pieces
  constexpr int BO = MODE == GLU ? BN / 2 : BN, LD = BO + 8;
  const int nout = MODE == GLU ? half : A.n;
  unsigned short* out = (unsigned short*)smem;
  __syncthreads();
#pragma unroll
  for (int nt = 0; nt < (MODE == GLU ? 1 : NT); ++nt) {
    const int c = (MODE == GLU ? wave : wave * NT + nt) * 16 + l15;
    const float bias = MODE == DENSE && A.bias != nullptr && n0 + c < A.n
                           ? bf16_bits_to_f32(A.bias[n0 + c])
                           : 0.f;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float v = MODE == GLU ? silu_mul_f(acc[t][0][r], acc[t][1][r])
                                    : acc[t][nt][r] + bias;
        out[(t * 16 + l4 * 4 + r) * LD + c] =
            (unsigned short)f32_to_bf16_bits_rne(v);
      }
  }
  __syncthreads();
  dq_block_store(out, LD, BM, BO, A.y, row0, rows, n0, nout, tid, TPB);
}

template <int BITS, int KC, DqMode MODE>
__global__ __launch_bounds__(TPB, 2) void dq_block_kernel(DqArgs A, Plan P) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const u32 nb = MODE == GLU ? (A.n / 2 + BN / 2 - 1) / (BN / 2)
                             : (A.n + BN - 1) / BN;
  DqBlockTile T;
  if (!dq_block_tile<MODE>(A, P, nb, BN, T)) return;
  const int nblk = T.nblk, sp = T.sp, parts = T.parts, expert = T.expert;
  const int row0 = T.row0, rows = T.rows;
  float* part = T.part;
  if (rows > 96)
    dq_block_body<BITS, KC, MODE, 8>(A, smem, row0, rows, expert, nblk, sp,
                                     parts, part);
  else if (rows > 64)
    dq_block_body<BITS, KC, MODE, 6>(A, smem, row0, rows, expert, nblk, sp,
                                     parts, part);
  else if (MODE == DENSE || rows > 32)
    dq_block_body<BITS, KC, MODE, 4>(A, smem, row0, rows, expert, nblk, sp,
                                     parts, part);
  else
    // experts with few rows, and what 128s leave of others: a layer of 8
    // (k 4096, 14336) 257 us at 26 rows an expert, 597 at 140; 298 and 630
    // with 64 (k whole).  Tested last: as the first of them it made the others
    // 1 % slower.
    dq_block_body<BITS, KC, MODE, 2>(A, smem, row0, rows, expert, nblk, sp,
                                     parts, part);
}

// the split tiles: sums of their parts, bias or gate
template <DqMode MODE>
__global__ __launch_bounds__(256) void dq_block_sum(DqArgs A, Plan P) {
  const u32 nb = MODE == GLU ? (A.n / 2 + BN / 2 - 1) / (BN / 2)
                             : (A.n + BN - 1) / BN;
  int mt, nblk;
  dq_block_place(P.full + blockIdx.x, P.mb, nb, mt, nblk);
  const int row0 = mt * P.step, rows = min(A.m - row0, P.step);
  const int nout = MODE == GLU ? A.n / 2 : A.n;
  constexpr int BO = MODE == GLU ? BN / 2 : BN, Q = BO / 4;
  const float* part = A.part + (u64)blockIdx.x * P.parts * (P.step * BN);
  const int row = blockIdx.y * (256 / Q) + threadIdx.x / Q;
  const int c = threadIdx.x % Q * 4, col = nblk * BO + c;
  if (row >= rows || col >= nout) return;
  // GLU: 16 of gate, 16 of up a wave
  const float* p = part + row * BN + (MODE == GLU ? (c >> 4) * 32 + (c & 15) : c);
  const f32x4 v = sum_of_parts(p, P.step * BN, P.parts);
  f32x4 u = {};
  if constexpr (MODE == GLU) u = sum_of_parts(p + 16, P.step * BN, P.parts);
  unsigned short* y = A.y + (u64)(row0 + row) * nout + col;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (col + e >= nout) break;
    const float b = MODE == DENSE && A.bias != nullptr
                        ? bf16_bits_to_f32(A.bias[col + e]) : 0.f;
    y[e] = (unsigned short)f32_to_bf16_bits_rne(
        MODE == GLU ? silu_mul_f(v[e], u[e]) : v[e] + b);
  }
}

// y [4 n4]: the sum of part [parts][4 n4]
__global__ __launch_bounds__(256) void dq_block_sum_slots(const float* part,
                                                          float* y, u32 n4,
                                                          int parts) {
  const u32 i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  *(f32x4*)(y + (u64)i * 4) =
      sum_of_parts(part + (u64)i * 4, (u64)n4 * 4, parts);
}

template <int BITS, int KC, DqMode MODE>
hipError_t go(const DqArgs& A, const Plan& P, u32 wgs, hipStream_t stream) {
  constexpr int lds = Lds<BITS, KC>::BYTES;
  static bool set = false;
  if (!set) {
    LFMQ_CHECK_HIP(hipFuncSetAttribute(
        (const void*)dq_block_kernel<BITS, KC, MODE>,
        hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    set = true;
  }
  hipLaunchKernelGGL((dq_block_kernel<BITS, KC, MODE>),
                     dim3(wgs, MODE == SLOTS ? P.parts : 1), dim3(TPB), lds,
                     stream, A, P);
  return hipGetLastError();
}

int chunk_of(int bits, int g) { return bits == 4 && g % 128 == 0 ? 128 : 64; }

template <DqMode MODE>
hipError_t go_bits(const DqArgs& A, const Plan& P, int bits, u32 wgs,
                   hipStream_t stream) {
  if (bits == 4)
    return chunk_of(4, A.g) == 128 ? go<4, 128, MODE>(A, P, wgs, stream)
                                   : go<4, 64, MODE>(A, P, wgs, stream);
  return go<8, 64, MODE>(A, P, wgs, stream);
}

int column_blocks(int n, bool glu) {
  return (int)(glu ? ceil_div_u32(n / 2, BN / 2) : ceil_div_u32(n, BN));
}

}  // namespace

bool lfmq_dq_block_ok(const void* qweight, const void* scales, long n, long k,
                      long g, long bits) {
  return (bits == 4 || bits == 8) && g > 0 && g <= k && g % 64 == 0 &&
         k % g == 0 && k / g % 8 == 0 && n * k / 8 * bits < 1l << 32 &&
         ((u64)qweight | (u64)scales) % 16 == 0;
}

// Rows of a tile, and tiles that are split, by the time this would take: rounds
// of 256 workgroups, 1.8 us each and a chunk's time for each of their chunks,
// 3.8 us and the traffic for the sum of what is split.  Fitted to 700
// measured plans of 33 to 1500 rows, 2048 to 32000 columns (off by 6 % rms; the
// plan it takes is 1.6 % slower than the best of them).
DqBlockPlan lfmq_dq_block_plan(int m, int n, int k, int g, int bits, bool glu) {
  const int kc = chunk_of(bits, g), C = k / kc, nb = column_blocks(n, glu);
  static const float us[3][3] = {{1.13f, 1.39f, 1.69f},     // 64, 96, 128 rows
                                 {0.76f, 0.92f, 1.07f},
                                 {0.84f, 1.00f, 1.15f}};
  const float* chunk = us[bits == 8 ? 2 : (kc == 64 ? 1 : 0)];
  Plan best{};
  float least = INFINITY;
  for (int r = ROWS; r >= 64; r -= 32) {
    Plan p;
    // row tiles alike, in sixteens: 129 rows are two of 80
    p.mb = (int)ceil_div_u32(m, r);
    p.step = (int)ceil_div_u32(ceil_div_u32(m, p.mb), 16) * 16;
    const float c = chunk[p.step <= 64 ? 0 : (p.step <= 96 ? 1 : 2)];
    const long tiles = (long)p.mb * nb;
    const int rest = (int)(tiles % 256);
    const float whole = (C * c + 1.8f) * (float)(tiles / 256);
    for (p.parts = 1; p.parts <= 16; ++p.parts) {
      const int wgs = rest * p.parts;
      if (p.parts > 1 && (rest == 0 || wgs > 512 || C / p.parts < 3)) break;
      float t = whole;
      if (rest) t += ((wgs + 255) / 256) * (ceil_div_u32(C, p.parts) * c + 1.8f);
      if (p.parts > 1) t += 3.8f + 0.00035f * wgs * p.step;
      if (t < least) {
        least = t;
        best = p;
        best.full = (int)(p.parts > 1 ? tiles - rest : tiles);
      }
    }
  }
  best.part = ((long)best.mb * nb - best.full) * best.parts * best.step * BN;
  return best;
}

hipError_t lfmq_dq_block(const void* qweight, const void* scales,
                         const void* qzeros, const void* x, void* y,
                         const void* bias, void* part, void* sums, int m, int n,
                         int k, int g, int bits, bool glu, const DqBlockPlan& P,
                         hipStream_t stream) {
  if (!lfmq_dq_block_ok(qweight, scales, n, k, g, bits) || m < 1 ||
      (glu && (n % 2 || bias != nullptr || (u64)m * k * 2 >= 1ull << 32)))
    return hipErrorInvalidValue;
  const DqArgs A{(const char*)qweight, (const unsigned short*)scales,
                 (const u32*)qzeros, (const unsigned short*)x,
                 (unsigned short*)y, (const unsigned short*)bias, nullptr,
                 (float*)part, m, n, k, g, 1, nullptr, nullptr, nullptr};
  const int rest = P.mb * column_blocks(n, glu) - P.full;
  if (rest > 0 && part == nullptr) return hipErrorInvalidValue;
  const u32 wgs = P.full + rest * P.parts;
  const hipError_t e =
      sums != nullptr
          ? lfmq_dq_panel(A, P, bits, glu ? GLU : DENSE, wgs, sums, m, stream)
      : glu ? go_bits<GLU>(A, P, bits, wgs, stream)
            : go_bits<DENSE>(A, P, bits, wgs, stream);
  if (e != hipSuccess || rest == 0) return e;
  if (glu)
    hipLaunchKernelGGL(dq_block_sum<GLU>, dim3(rest, ceil_div_u32(P.step, 8)),
                       dim3(256), 0, stream, A, P);
  else
    hipLaunchKernelGGL(dq_block_sum<DENSE>, dim3(rest, ceil_div_u32(P.step, 4)),
                       dim3(256), 0, stream, A, P);
  return hipGetLastError();
}

// Without a gate an expert's few rows give few workgroups (n 4096, 8 experts: a
// tile each, 128): their k is split where the parts still fit into one round.
// Rows are taken to be shared out as 9 / 8 of the mean to each, and a part to
// have 8 chunks at least, for what its first loads and the sum cost.  us of a
// layer (gate and this), k whole and in parts, at 26 and 60 rows an expert:
// 8 of 4096, 14336 276, 348 and 238, 304; 8 of 2048, 8192 119 and 76 at 32,
// 145 and 93 at 60; 16 of 1024, 2048 49 and 42 at 60.
int lfmq_dq_block_slot_parts(long slots, long E, int n, int k, int g,
                             int bits) {
  if (slots < 1 || E < 1 || n % 4 || slots * n >= 1l << 32) return 1;
  const long each = (slots * 9 / 8 + E - 1) / E;
  const long wgs = std::min(E, slots) * ((each + ROWS - 1) / ROWS) *
                   column_blocks(n, false);
  int parts = 1;
  while (parts < 4 && wgs * parts * 2 <= 256 &&
         k / chunk_of(bits, g) / (parts * 2) >= 8)
    parts *= 2;
  return parts;
}

hipError_t lfmq_dq_block_experts(const void* qweight, const void* scales,
                                 const void* qzeros, const void* x,
                                 const void* src, const void* tiles, void* y,
                                 void* part, void* sums, long rows, int n_tiles,
                                 int n, int k, int g, int bits, bool glu,
                                 int parts, long slots, hipStream_t stream) {
  if (!lfmq_dq_block_ok(qweight, scales, n, k, g, bits) || (glu && n % 2) ||
      parts < 1 ||
      (parts > 1 && (glu || part == nullptr || n % 4 || slots < 1 ||
                     slots * n >= 1l << 32)))
    return hipErrorInvalidValue;
  DqArgs A{};
  A.w = (const char*)qweight;
  A.scales = (const unsigned short*)scales;
  A.zeros = (const u32*)qzeros;
  A.x = (const unsigned short*)x;
  A.y = (unsigned short*)y;
  A.y32 = (float*)(parts > 1 ? part : y);
  A.src = (const i32*)src;
  A.tiles = (const i32*)tiles;
  A.n = n;
  A.k = k;
  A.g = g;
  A.splits = 1;
  const u32 wgs = n_tiles * column_blocks(n, glu);
  Plan P{};
  P.parts = parts;
  P.part = slots * n;
  const hipError_t e =
      sums != nullptr
          ? lfmq_dq_panel(A, P, bits, glu ? GLU : SLOTS, wgs, sums, rows, stream)
      : glu ? go_bits<GLU>(A, P, bits, wgs, stream)
            : go_bits<SLOTS>(A, P, bits, wgs, stream);
  if (e != hipSuccess || parts == 1) return e;
  const u32 n4 = (u32)(slots * n / 4);
  hipLaunchKernelGGL(dq_block_sum_slots, dim3(ceil_div_u32(n4, 256)), dim3(256),
                     0, stream, (const float*)part, (float*)y, n4, parts);
  return hipGetLastError();
}
