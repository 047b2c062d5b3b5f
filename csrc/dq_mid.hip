// K3h/K4h — W4A16 / W8A16 product for some tens to hundreds of rows: y[m, n] = x[m, k] ·
// dequant(W)[n, k]^T (+ bias) (+ residual), or the gated half of a fused gate and up
// projection.
//
// Eight waves share 64 or 128 columns and k: they lie 2 or 4 side by side and 4 or 2
// along k, by groups in turn, and their sums meet in LDS.  A wave issues some 160
// instructions a step of 64 k, at 4 cycles each the longest of what it does, beside
// products (the sums of x made them a third longer) and reads of LDS: so a step's
// unpacking and scaling stand between the products of the step before, the loads'
// places are kept and moved on, x is read from LDS a row tile ahead and the weights
// come by whole lines, of all of a turn's waves along k (by 32 bytes a column and step
// 3 to 5 % slower).  Stages further ahead (up to six) and x two tiles ahead: the same.
//
// 8 bits: a code minus its zero is an exact bf16 number, a group's scale is applied
// once.  4 bits: sum s (c - z) x = s (sum c x) - (s z) (sum x), the sums of x by the
// matrix cores: each of the waves side by side makes those of its share of the row
// tiles, and all read them two steps later, behind a barrier that there is anyway.
//
// us a call, dq_rows or dq_short (8 bits: this kernel with all of a step one after the
// other) and this one, 4 bits in groups of 128, 8 in groups of 64:
//                               20 rows       48 rows       77 rows       128 rows
//   n 28672, k 4096, gate     25.2 / 23.2   29.4 / 27.1   39.6 / 34.8
//   n 16384, k 2048, gate     12.4 / 10.4   14.9 / 12.4   17.4 / 15.1   20.6 / 18.0
//   n 4096, k 14336           18.0 / 17.6   20.4 / 19.4   27.0 / 25.6
//   n 4096, k 4096                          13.5 / 13.6   15.5 / 16.4   19.6 / 15.1
//   n 32000, k 4096           25.6 / 23.5   31.9 / 28.2   41.1 / 36.7
//   n 28672, k 4096, gate (8) 36.1 / 35.3   41.4 / 36.1   51.6 / 40.2
//   n 2048, k 8192 (8)                      16.9 / 14.3   16.6 / 16.1   23.6 / 17.4
//   n 32000, k 2048 (8)       21.8 / 18.9   23.8 / 21.0   29.2 / 24.5   35.9 / 35.5
//   n 16384, k 2048, gate, groups of 64 (4)  16.8 / 12.1  24.4 / 14.6
// A sum of parts that goes with a norm or rotation that follows (a prompt's layers)
// costs nothing more: there 4096 x 4096 at 48 rows is 2 us ahead.
#include <type_traits>

#include "dq_mid.h"
#include "lds_dma.h"

namespace {

constexpr int NWV = 8, TPB = NWV * 64, NT = 2;   // waves, 16s of columns a wave
constexpr int KS = 64, J = 2;                    // k of a step, products
constexpr int MOST_LDS = 160 * 1024;

// eight codes minus z, exact
__device__ __forceinline__ s16x8 codes8_less(u32 w0, u32 w1, float z) {
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const u32 p = (i >> 1 ? w1 : w0) >> (16 * (i & 1));
    const float lo = (float)(p & 0xFFu) - z, hi = (float)((p >> 8) & 0xFFu) - z;
    o[i] = __builtin_amdgcn_perm(__builtin_bit_cast(u32, hi),
                                 __builtin_bit_cast(u32, lo), 0x07060302u);
  }
  return __builtin_bit_cast(s16x8, o);
}

// NC: waves side by side; GS: steps of a group.  Steps of x: DX, one ahead of the
// products where there is room for three.  Weights: RT turns of a group a k wave,
// whose whole lines come with the steps, DW ahead.
template <int BITS, int GS, int MT, int NC>
struct Lds {
  static constexpr int KW = NWV / NC, BN = NC * NT * 16, BM = MT * 16;
  static constexpr int XB = BM * KS * 2, XS = KW * XB;       // a k wave's, a step's
  static constexpr int CB = KW * GS * KS * BITS / 8;         // a column's of a turn
  static constexpr int WT = BN * CB;
  static constexpr int ROOM = 144 * 1024;
  static constexpr int turns(int dx) { return GS == 1 ? dx + 1 : 3; }
  static constexpr int DX = 3 * XS + turns(3) * WT <= ROOM ? 3 : 2;
  static constexpr int DW = DX + GS, RT = turns(DX);
  // sums of x of the groups of a turn and of the one before (4 bits)
  static constexpr int SUM = KW * BM, SUMS = BITS == 4 ? 2 * SUM * 4 : 0;
  static constexpr int W0 = DX * XS, X0 = W0 + RT * WT, META = X0 + SUMS;
  static constexpr int bytes(int groups) {
    const int loop = META + groups * BN * 4, sums = KW * BM * (BN + 4) * 4;
    return loop > sums ? loop : sums;
  }
};

template <int BITS, int GS, int MT, int NC, DqMode MODE>
__global__ __launch_bounds__(TPB, 2) void dq_mid_kernel(DqArgs A, int mb, int step) {
  typedef Lds<BITS, GS, MT, NC> L;
  constexpr int KW = L::KW, BN = L::BN, BM = L::BM, DX = L::DX, DW = L::DW;
  constexpr int SL = KS / 8;                     // 8 slots of 16 bytes a row
  constexpr int XP = L::XB / 1024, XL = KW * XP, NX = (XL + NWV - 1) / NWV;
  constexpr int NL = L::WT / NWV / GS / 1024;    // of weights, a wave's
  constexpr int PC = L::CB / 16, PG = PC / KW;   // 16-byte pieces a column, a group
  constexpr int WD = J * BITS / 4;               // words of a lane and column
  extern __shared__ __attribute__((aligned(16))) char smem[];
  u32* meta = (u32*)(smem + L::META);            // [groups][BN]
  float* xsum = (float*)(smem + L::X0);          // [2][KW][BM]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = wave % NC, kw = wave / NC;
  const int l15 = lane & 15, l4 = lane >> 4;
  constexpr int BO = MODE == GLU ? BN / 2 : BN;
  const int nout = MODE == GLU ? A.n / 2 : A.n;
  const u32 nb = (nout + BO - 1) / BO;
  u32 id = xcd_swizzle(blockIdx.x, gridDim.x);
  const int row0 = (int)(id % mb) * step;
  id /= mb;
  const int nblk = id % nb, sp = id / nb;
  const int rows = min(A.m - row0, step);
  // groups (A.g's, or parts of them) of this workgroup; a k wave takes every KW-th of
  // them (a division leaves them in vector registers)
  constexpr int g = GS * KS;
  const int G = A.k / A.g, zw = (G + 32 / BITS - 1) / (32 / BITS);
  const int GA = A.k / g, per = A.g / g;
  const int g0 = __builtin_amdgcn_readfirstlane((int)((long)GA * sp / A.splits));
  const int g1 = __builtin_amdgcn_readfirstlane((int)((long)GA * (sp + 1) / A.splits));
  const int ng = g1 - g0, turns = (ng + KW - 1) / KW;
  const int S = turns * GS;                      // steps
  const int half = A.n / 2, n0 = nblk * BO;
  auto column = [&](int c) {
    if (MODE == GLU)
      return (c >> 4 & 1) * half + min(n0 + (c >> 5) * 16 + (c & 15), half - 1);
    return min(n0 + c, A.n - 1);
  };
  const char* xb = (const char*)(A.x + (u64)row0 * A.k);
  const u32 pitch = A.k * 2, last = (u32)(rows - 1) * pitch, wrow = A.k * BITS / 8;
  // x: load i of this wave, for k wave xq
  u32 xo[NX];
  int xq[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int e = min(i * NWV + wave, XL - 1), r = e % XP * 8 + lane / 8;
    xq[i] = e / XP;
    xo[i] = min(r * pitch, last) + ((lane % SL) ^ slot_key16<SL>(r & 15)) * 16 +
            min(xq[i], ng - 1) * (g * 2);
  }
  // weights: load i of a wave in half h of a turn
  u32 wo[GS][NL];
#pragma unroll
  for (int h = 0; h < GS; ++h)
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = ((h * NL + i) * NWV + wave) * 64 + lane, c = e / PC;
      const int p = (e % PC) ^ slot_key<PC < 16 ? PC : 16>(c & 15);
      wo[h][i] = (u32)column(c) * wrow + min(p, ng * PG - 1) * 16;
    }
  // Turns past the last repeat it.  In a last turn of fewer groups than k waves the
  // waves past them get what the last group has (and count nothing): once that turn
  // comes, places change for good.
  const int left = ng - (turns - 1) * KW;        // groups of the last turn
  const char* xp = xb + (u64)g0 * (g * 2);
  const char* wp = A.w + (u64)g0 * (PG * 16);
  auto next_x = [&](int turn) {                  // turn: the one that comes
    if (turn >= turns) return;
    xp += KW * g * 2;
    if (turn == turns - 1 && left < KW) {
#pragma unroll
      for (int i = 0; i < NX; ++i) xo[i] -= max(xq[i] - (left - 1), 0) * (g * 2);
    }
  };
  auto next_w = [&](int turn) {
    if (turn >= turns) return;
    wp += KW * PG * 16;
    if (turn == turns - 1 && left < KW) {
#pragma unroll
      for (int h = 0; h < GS; ++h)
#pragma unroll
        for (int i = 0; i < NL; ++i) {
          const int e = ((h * NL + i) * NWV + wave) * 64 + lane;
          const int p = (e % PC) ^ slot_key<PC < 16 ? PC : 16>(e / PC & 15);
          wo[h][i] -= max(p - (left * PG - 1), 0) * 16;
        }
    }
  };
  // step h of turn's x; half h of turn's weights.  In order: the pointers go along
  auto stage_x = [&](int turn, auto h, int buf) {
    constexpr int H = decltype(h)::value;
#pragma unroll
    for (int i = 0; i < NX; ++i)
      load_to_lds(xp + H * (KS * 2), xo[i],
                  buf * L::XS + min(i * NWV + wave, XL - 1) * 1024);
    if (H == GS - 1) next_x(turn + 1);
  };
  auto stage_w = [&](int turn, auto h, int buf) {
    constexpr int H = decltype(h)::value;
#pragma unroll
    for (int i = 0; i < NL; ++i)
      load_to_lds(wp, wo[H][i],
                  L::W0 + buf * L::WT + ((H * NL + i) * NWV + wave) * 1024);
    if (H == GS - 1) next_w(turn + 1);
  };
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  // (in this order: what the loop waits for is counted)
  auto first_w = [&](auto v) {
    constexpr int V = decltype(v)::value;
    if (V < S) stage_w(V / GS, std::integral_constant<int, V % GS>(), V / GS);
  };
  first_w(even);
  first_w(odd);
  if constexpr (GS == 2) first_w(std::integral_constant<int, 2>());
  stage_x(0, even, 0);
  first_w(std::integral_constant<int, GS + 1>());
  if constexpr (DX == 3) {
    if (S > 1) stage_x(1 / GS, std::integral_constant<int, 1 % GS>(), 1);
    first_w(std::integral_constant<int, GS + 2>());
  }
  if constexpr (BITS == 4)
    for (int i = tid; i < 2 * L::SUM; i += TPB) xsum[i] = 0.f;
  {
    constexpr int IN = 8;
    for (int i0 = tid; i0 < BN * ng; i0 += IN * TPB) {
      u32 s[IN], z[IN];
#pragma unroll
      for (int j = 0; j < IN; ++j) {
        const int i = min(i0 + j * TPB, BN * ng - 1);
        const int gi = (g0 + i % ng) / per;
        const u32 r = column(i / ng);
        s[j] = A.scales[(u64)r * G + gi];
        z[j] = A.zeros[(u64)r * zw + gi / (32 / BITS)];
      }
#pragma unroll
      for (int j = 0; j < IN; ++j) {
        const int i = min(i0 + j * TPB, BN * ng - 1);
        const int gi = (g0 + i % ng) / per;
        meta[i % ng * BN + i / ng] =
            s[j] << 16 | (BITS == 4 ? unpack4(z[j], gi & 7) : unpack8(z[j], gi & 3));
      }
    }
  }
  f32x4 acc[MT][NT] = {}, a[MT][NT] = {};
  // 4 bits: sums of x of every NC-th row tile, which the waves side by side share
  constexpr int XT = (MT + NC - 1) / NC;
  f32x4 xs[XT] = {}, xr[MT];
  const s16x8 ones = bf16_ones();
  s16x8 b[2][NT][J], xa[2][J], xn[J];
  u32 w[NT][WD];
  // the scale and scale times zero of the group in a, the latter of the one before,
  // the zero of the one that is unpacked
  float sc[NT] = {}, z[NT] = {}, zp[NT] = {}, zn[NT];
  // of half h of a turn
  auto read_w = [&](int buf, int h) {
    const char* ws = smem + L::W0 + buf * L::WT;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const char* p = ws + ((wc * NT + t) * 16 + l15) * L::CB;
      const int at = (kw * GS + h) * (KS * BITS / 8) + l4 * WD * 4;
      p += (((at / 16) ^ slot_key<PC < 16 ? PC : 16>(l15)) << 4) + at % 16;
      if constexpr (WD == 2) {
        const u64 v = *(const u64*)p;
        w[t][0] = (u32)v;
        w[t][1] = (u32)(v >> 32);
      } else {
        static_assert(WD == 4, "");
        const u32x4 v = *(const u32x4*)p;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[t][e] = v[e];
      }
    }
  };
  auto read_x = [&](int buf, int t, s16x8 (&x)[J]) {
    const char* p = smem + buf * L::XS + kw * L::XB + (t * 16 + l15) * (KS * 2);
#pragma unroll
    for (int j = 0; j < J; ++j)
      x[j] = *(const s16x8*)(p + (((l4 * J + j) ^ slot_key16<SL>(l15)) << 4));
  };
  auto read_meta = [&](int turn, u32 (&m)[NT]) {
    const int gl = min(turn * KW + kw, ng - 1);
#pragma unroll
    for (int t = 0; t < NT; ++t) m[t] = meta[gl * BN + (wc * NT + t) * 16 + l15];
  };
  auto unpack = [&](s16x8 (&to)[NT][J], int i) {
    const int t = i / J, j = i % J;
    if constexpr (BITS == 4) to[t][j] = codes8_exact<4>(&w[t][j]);
    else to[t][j] = codes8_less(w[t][j * 2], w[t][j * 2 + 1], zn[t]);
    // here and not, as the compiler would have it, where they are used
    asm volatile("" : "+v"(to[t][j]));
  };
  auto fold = [&](int t) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[t][nt][r] = fmaf(sc[nt], a[t][nt][r], acc[t][nt][r]);
      asm volatile("" : "+v"(acc[t][nt]));
    }
  };
  // Zeros' term, of sums that were written two steps ago: a barrier lies between.
  auto read_sums = [&](int turn) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
      xr[t] = *(const f32x4*)(xsum + ((turn & 1) * KW + kw) * BM + t * 16 + l4 * 4);
  };
  auto fold_zeros = [&](int t, const float (&z)[NT]) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[t][nt][r] = fmaf(-z[nt], xr[t][r], acc[t][nt][r]);
      asm volatile("" : "+v"(acc[t][nt]));
    }
  };
  u32 m0[NT], m1[NT];
  constexpr int LATER = (DX - 2) * NX + (DX - 1) * NL;
  if (S >= DW) loads_but<LATER>();
  else loads_but<0>();
  read_meta(0, m0);
#pragma unroll
  for (int t = 0; t < NT; ++t) zn[t] = (float)(m0[t] & 0xFFFFu);
  read_w(0, 0);
  read_x(0, 0, xa[0]);
#pragma unroll
  for (int i = 0; i < NT * J; ++i) unpack(b[0], i);
  int bx = 0, bw = 0;                            // buffers: of the step, of its turn
  // step of a turn with b[PAR], FIRST: of a group
  auto one = [&](int turn, auto par, auto first) {
    constexpr int PAR = decltype(par)::value;
    constexpr bool FIRST = decltype(first)::value;
    constexpr bool ENDS = GS == 1 || !FIRST;     // the next step: of another group
    constexpr bool ZEROS = BITS == 4 && ENDS;    // two steps ago a group ended
    constexpr int H = GS == 1 ? 0 : PAR;
    const int bx1 = bx == DX - 1 ? 0 : bx + 1, bx2 = bx == 0 ? DX - 1 : bx - 1;
    const int bw1 = bw == L::RT - 1 ? 0 : bw + 1;
    // x of DX - 1 steps ahead, half a turn's weights of DW ahead
    constexpr int SX = H + DX - 1, SW = H + DW;
    stage_x(turn + SX / GS, std::integral_constant<int, SX % GS>(), bx2);
    constexpr int BW = SW / GS % L::RT;          // that turn's buffer from bw on
    const int bws = bw + BW >= L::RT ? bw + BW - L::RT : bw + BW;
    stage_w(turn + SW / GS, std::integral_constant<int, SW % GS>(), bws);
    read_w(ENDS ? bw1 : bw, ENDS ? 0 : 1);
    if (ENDS) read_meta(turn + 1, m1);
    if constexpr (ZEROS) read_sums(GS == 1 ? turn : turn + 1);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      if (t + 1 < MT) {
        read_x(bx, t + 1, xa[(t + 1) & 1]);
      } else {
        // x of the next step and the weights of the one after it have landed, and
        // all waves have read this one's x: the last products are still to come
        loads_but<LATER>();
        read_x(bx1, 0, xn);
      }
      if (FIRST) fold(t);
      if constexpr (ZEROS) fold_zeros(t, zp);
      if (t == 0 && ENDS && BITS == 8) {
#pragma unroll
        for (int i = 0; i < NT; ++i) zn[i] = (float)(m1[i] & 0xFFFFu);
      }
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          a[t][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              xa[t & 1][j], b[PAR][nt][j],
              FIRST && j == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : a[t][nt], 0, 0, 0);
      if constexpr (BITS == 4) {
        if (wc == t % NC) {
#pragma unroll
          for (int j = 0; j < J; ++j)
            xs[t / NC] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                xa[t & 1][j], ones,
                FIRST && j == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : xs[t / NC], 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = t * NT * J / MT; i < (t + 1) * NT * J / MT; ++i)
        unpack(b[PAR ^ 1], i);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (FIRST) {                                 // a's group
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        zp[t] = z[t];
        sc[t] = __builtin_bit_cast(float, m0[t] & 0xFFFF0000u);
        z[t] = sc[t] * (float)(m0[t] & 0xFFFFu);
      }
    }
    if (ENDS) {
#pragma unroll
      for (int t = 0; t < NT; ++t) m0[t] = m1[t];
      if (BITS == 4 && l15 == 0) {
#pragma unroll
        for (int i = 0; i < XT; ++i)
          if (wc + i * NC < MT)
            *(f32x4*)(xsum + ((turn & 1) * KW + kw) * BM + (wc + i * NC) * 16 +
                      l4 * 4) = xs[i];
      }
      bw = bw1;
    }
#pragma unroll
    for (int j = 0; j < J; ++j) xa[0][j] = xn[j];
    bx = bx1;
  };
  constexpr std::integral_constant<bool, true> yes{};
  constexpr std::integral_constant<bool, false> no{};
  if constexpr (GS == 2) {
    for (int i = 0; i < turns; ++i) {
      one(i, even, yes);
      one(i, odd, no);
    }
  } else {
    int i = 0;
    for (; i + 1 < turns; i += 2) {
      one(i, even, yes);
      one(i + 1, odd, yes);
    }
    if (i < turns) one(i, even, yes);
  }
  // (waves past the last group have nothing of it, which is not 0 times what they have:
  // that may be infinite)
  const bool in = kw < left;
  if (in) {
#pragma unroll
    for (int t = 0; t < MT; ++t) fold(t);
  }
  loads_but<0>();
  if constexpr (BITS == 4) {
    if (GS == 1) {
      read_sums(turns);
#pragma unroll
      for (int t = 0; t < MT; ++t) fold_zeros(t, zp);
    }
    if (in) {
      read_sums(turns - 1);
#pragma unroll
      for (int t = 0; t < MT; ++t) fold_zeros(t, z);
    }
  }
  // the k waves' sums
  constexpr int LD = BN + 4;
  float* red = (float*)smem;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[(kw * BM + t * 16 + l4 * 4 + r) * LD + (wc * NT + nt) * 16 + l15] =
            acc[t][nt][r];
  __syncthreads();
  for (int i = tid; i < BM * BO / 4; i += TPB) {
    const int row = i / (BO / 4), c = i % (BO / 4) * 4;
    if (row >= rows || n0 + c >= nout) continue;
    auto sum = [&](int col) {
      f32x4 v = *(const f32x4*)(red + row * LD + col);
#pragma unroll
      for (int q = 1; q < KW; ++q) v += *(const f32x4*)(red + (q * BM + row) * LD + col);
      return v;
    };
    const u64 at = (u64)(row0 + row) * nout + n0 + c;
    if (MODE == DENSE && A.splits > 1) {
      *(f32x4*)(A.part + (u64)sp * A.m * nout + at) = sum(c);
      continue;
    }
    const float scale = A.row_scale != nullptr ? A.row_scale[row0 + row] : 1.f;
    f32x4 v;
    if constexpr (MODE == GLU) {
      const int c2 = (c >> 4) * 32 + (c & 15);
      const f32x4 gate = sum(c2) * scale, up = sum(c2 + 16) * scale;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = silu_mul_f(gate[e], up[e]);
    } else {
      v = sum(c) * scale;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (A.bias != nullptr) v[e] += bf16_bits_to_f32(A.bias[n0 + c + e]);
        if (A.resid != nullptr) v[e] += bf16_bits_to_f32(A.resid[at + e]);
      }
    }
    *(u64*)(A.y + at) = pack_bf16x2(v[0], v[1]) | (u64)pack_bf16x2(v[2], v[3]) << 32;
  }
}

template <int BITS, int GS, int MT, int NC, DqMode MODE>
hipError_t go(const DqArgs& A, const DqMidPlan& P, hipStream_t stream) {
  typedef Lds<BITS, GS, MT, NC> L;
  const u32 nb = MODE == GLU ? ceil_div_u32(A.n / 2, L::BN / 2)
                             : ceil_div_u32(A.n, L::BN);
  const int lds = L::bytes((int)ceil_div_u32(A.k / (GS * KS), A.splits));
  if (lds > MOST_LDS) return hipErrorInvalidValue;
  const auto kernel = dq_mid_kernel<BITS, GS, MT, NC, MODE>;
  static bool set = false;
  if (!set) {
    LFMQ_CHECK_HIP(hipFuncSetAttribute(
        (const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, MOST_LDS));
    set = true;
  }
  hipLaunchKernelGGL(kernel, dim3(P.mb * nb * A.splits), dim3(TPB), lds, stream, A,
                     P.mb, P.step);
  return hipGetLastError();
}

template <int BITS, int GS, int NC, DqMode MODE>
hipError_t go_rows(const DqArgs& A, const DqMidPlan& P, hipStream_t stream) {
  switch (P.step / 16) {
    case 2: return go<BITS, GS, 2, NC, MODE>(A, P, stream);
    case 3: return go<BITS, GS, 3, NC, MODE>(A, P, stream);
    case 4: return go<BITS, GS, 4, NC, MODE>(A, P, stream);
    case 5: return go<BITS, GS, 5, NC, MODE>(A, P, stream);
    case 6: return go<BITS, GS, 6, NC, MODE>(A, P, stream);
  }
  return hipErrorInvalidValue;
}

template <int BITS, int GS>
hipError_t go_cols(const DqArgs& A, const DqMidPlan& P, bool glu, hipStream_t stream) {
  if (P.cols == 2)
    return glu ? go_rows<BITS, GS, 2, GLU>(A, P, stream)
               : go_rows<BITS, GS, 2, DENSE>(A, P, stream);
  if (P.cols == 4)
    return glu ? go_rows<BITS, GS, 4, GLU>(A, P, stream)
               : go_rows<BITS, GS, 4, DENSE>(A, P, stream);
  return hipErrorInvalidValue;
}

template <int BITS, int GS>
int lds_of(int mt, int nc, int groups) {
#define S(MT)                                                    \
  if (mt == MT)                                                  \
    return nc == 2 ? Lds<BITS, GS, MT, 2>::bytes(groups)         \
                   : Lds<BITS, GS, MT, 4>::bytes(groups);
  S(2) S(3) S(4) S(5) S(6)
#undef S
  return MOST_LDS + 1;
}
int lds_of(int bits, int g, int mt, int nc, int groups) {
  if (bits == 4)
    return g == 64 ? lds_of<4, 1>(mt, nc, groups) : lds_of<4, 2>(mt, nc, groups);
  return g == 64 ? lds_of<8, 1>(mt, nc, groups) : lds_of<8, 2>(mt, nc, groups);
}

// a group of the kernel's: g, or the part of it that it divides it into
int part_of(int g) { return g % 128 == 0 ? 128 : 64; }

}  // namespace

// Row tiles, columns of a workgroup and parts of k by the time these would take: 256
// workgroups a round, one after the other on a CU; a step 0.5 to 1.3 us, and the
// traffic of the parts and 0.8 us for their launch: mostly a norm, the rotation or
// factors of rows, which are a launch anyway, take the sum along.  A call with nothing
// behind it has the same plan, so that its results are the same bits, and pays 1.6 us
// in a graph and 3.0 called from Python (means of 840 calls).  us in a graph / called /
// with a norm, with this plan and with one that charges 2.2: n 2048, k 2048 (4 bits) at
// 77 rows 10.2 / 12.7 / 10.6, 9.8 / 10.2 / 12.2; n 4096, k 4096 (4) at 77 15.8 / 16.7 /
// 16.5, 14.3 / 14.3 / 16.9; n 3072, k 2048 (8) at 96 12.5 / 13.5 / 13.6, 11.5 / 11.7 /
// 14.2.
// Fitted to half of 101000 measured plans of 9700 calls, 17 to 128 rows (off by 7 %
// rms; the plan it takes is 0.5 % slower than the best); not to more rows.
DqMidPlan lfmq_dq_mid_plan(int m, int n, int k, int g, int bits, bool glu) {
  DqMidPlan best{};
  float least = INFINITY;
  static const float us[4][2] = {
      {0.244f, 0.169f}, {0.222f, 0.153f}, {0.409f, 0.148f}, {0.446f, 0.106f}};
  const int part = part_of(g), G = k / part;
  for (int mb = 1; mb <= 8; ++mb) {
    const int step =
        max(32, (int)ceil_div_u32(ceil_div_u32(m, mb), 16) * 16);
    // (every row tile has a row)
    if (step > 96 || (mb > 1 && m < 17 * mb) || (mb - 1) * step >= m) continue;
    for (int nc = 2; nc <= 4; nc += 2) {
      const int kw = NWV / nc, bo = nc * NT * 16;
      const int nb = (int)(glu ? ceil_div_u32(n / 2, bo / 2) : ceil_div_u32(n, bo));
      const float* t0 = us[(bits == 8 ? 2 : 0) + (nc == 4 ? 1 : 0)];
      for (int wgs = 0, before = 0; wgs <= 512; wgs += wgs == 0 ? 256 : 128) {
        const int sp = max(1, wgs / (nb * mb));
        if (sp == before || (sp > 1 && (glu || sp > G))) continue;
        before = sp;
        const int ng = (int)ceil_div_u32(G, sp), all = mb * nb * sp;
        if (lds_of(bits, part, step / 16, nc, ng) > MOST_LDS) continue;
        const int u = (int)ceil_div_u32(all, 256);
        const float rounds = u == 1 ? 1.f : ((u / 2) + (u & 1) * 0.561f) * 1.95f;
        const int steps = (int)ceil_div_u32(ng, kw) * (part / KS);
        const float chain = steps * (t0[0] + t0[1] * (step / 16)) *
                            (0.866f + 0.134f / 256.f * all / u);
        float t = rounds * (chain + 3.43f);
        if (sp > 1) t += 1.986e-6f * (float)m * (float)n * sp + 0.8f;
        if (t < least) {
          least = t;
          best = {mb, step, nc, sp, all, steps};
        }
      }
    }
  }
  return best;
}

// Whether that is faster than the other kernels for these rows (dq_rows, dq_short,
// dq_tile, dq_block): one round of workgroups, whose chain (steps, times row tiles and
// idle CUs) is not long for what it does.  us of the best of those / of this one:
// - two rounds: n 32000, k 4096 (4 bits, groups of 128) at 128 rows 43.4 / 59.9
// - few rows of 4 bits, where those lose less by idle CUs: n 16832, k 6400 at 32 27.6 /
//   31.6.  A gate has no parts here, nor in dq_rows, but in dq_short and dq_tile: n 8112,
//   k 9728 (8) at 19 29.4 / 49.8, n 2256, k 12032 at 46 21.3 / 31.1; n 2416, k 3840 at
//   40, which dq_rows has, 24.0 / 15.8
// - few rows of a short k, which does not make up for the first loads: n 12584, k 768,
//   gate, at 28 7.9 / 8.6, n 7424, k 640, gate, at 19 6.8 / 8.0; of a small matrix n
//   3712, k 3072 at 19 9.0 / 11.4, n 3072, k 2048 at 32 8.3 / 9.5, but n 25496, k 640 (8)
//   at 32 16.3 / 10.8.  6144 to 8192 columns are 192 to 256 workgroups of dq_rows, which
//   has up to 32 rows at once: n 6944, k 1664 (8) at 26 9.8 / 11.8, n 7440, k 640 (8) at
//   42 10.3 / 8.5
// - groups of 128 of a short k, two steps each: n 16264, k 640 (8) at 119 11.1 / 12.7;
//   n 27200, k 512, gate, at 88 10.2 / 11.7
// - 16384 to 20480 columns, where a workgroup of 128 leaves 96 CUs: n 18688, k 4096 at
//   55 26.3 / 30.1, n 17536, k 1536 at 82 16.6 / 18.7
// - many rows of very long k, 4 bits: n 4096, k 14336 at 126 31.1 / 33.7
// Of 5400 random calls of 17 to 128 rows, 768 to 36000 columns, k 1024 to 14336, groups
// of 64 and 128, 8 in 10 are taken: 1.18 times as fast in the mean, 1.13 with a norm
// behind them, 5 % of them slower by more than 4 %.  (97 to 128 rows of k below 2048
// without parts, on half of the chip: 10 % faster, 8 % slower with a norm, which the sum
// of dq_tile's parts takes along.)
//
// 129 to 768 rows (the most that were measured with these tiles), where dq_block's and
// dq_tile's tiles of 128 rows are few: n 2048, k 2048 at 300 rows 16.7 / 12.0, n 3072, k
// 2048 at 160 15.9 / 10.0, n 4096, k 4096 at 256 24.2 / 19.4, n 16384, k 2048, gate (8),
// at 160 33.1 / 22.6; but long chains, n 4096, k 14336 at 200 41.2 / 49.7, more than a
// round, n 16384, k 2048, gate, at 256 25.0 / 33.9, and short k, n 12000, k 640 2 %; n
// 2048, k 2048 (8) at 768 26.6 / 15.9, but n 2048, k 8192 (4 bits) at 660 37.2 / 42.7.
// Of 9700 random calls more than half are taken: 1.36 times as fast in the mean, 0.8 %
// slower by more than 4 %.
bool lfmq_dq_mid_gains(const DqMidPlan& P, long m, long n, long k, long g, int bits,
                       bool glu) {
  const long size = n * k, M = 1l << 20;
  const bool four = bits == 4, wide = g % 128 == 0;
  if (P.mb < 1 || P.wgs > 256) return false;
  const int work = P.steps * (P.step / 16);      // of a wave
  if (m > 128)
    return k >= 768 &&
           P.steps * P.mb * 256l <= (four && size > 32 * M ? 100l : 200l) * P.wgs;
  const long most = four && !glu && m <= 32 ? 40 : 120;
  if (glu && m <= 48) {
    // (dq_rows with its gate has no parts either, dq_short and dq_tile do)
    const bool others = (n >= 4096 && size >= 16 * M && (k >= 4096 || size >= 48 * M)) ||
                        (m > 32 && k >= 4096 && size >= 24 * M);
    if (others && P.steps * P.mb * 256l > 56l * P.wgs) return false;
  } else if (P.steps * P.mb * 256l > most * P.wgs) {
    return false;
  }
  if (m <= 32) {
    if (four ? P.splits == 1 && P.steps <= (glu ? 5 : 4)
             : glu && wide && P.steps <= 4 && size < 10 * M)
      return false;
    if (k < 768 && (four || size < 10 * M)) return false;
  } else if (m > 48 && k < 1024) {
    if (wide && n > (four && glu ? 2304 : 6144) && work > (k < 768 ? 7 : four ? 9 : 12))
      return false;
    if (k < 768 && four && glu && m > 64 && n > 8192) return false;
  }
  if (!glu && n > 2016 &&
      (m <= 24 ? size < (four ? 20 : 10) * M
               : m <= 48 && size <= (four ? 8 : 6) * M && (four || n < 6144)))
    return false;
  if (!glu && m <= 32 && n >= 6144 && n <= 8192 && size < (four ? 21 : 16) * M)
    return false;
  if (n > 16384 && n <= 20480 && (k <= 2048 ? m > 80 : !glu && k >= 4096)) return false;
  return !(four && m > 96 && k >= 12000);
}

hipError_t lfmq_dq_mid(const DqArgs& A, const DqMidPlan& P, int bits, bool glu,
                       hipStream_t stream) {
  const int nout = glu ? A.n / 2 : A.n;
  if (A.g % 64 || A.g < 64 || A.k % A.g || A.m < 1 || (glu && A.n % 2) ||
      nout % 4 || (u64)A.n * A.k * bits / 8 >= 1ull << 32 || (u64)A.w % 16 ||
      P.mb < 1 || P.step < 32 || P.step > 96 || (P.mb - 1) * P.step >= A.m ||
      P.mb * P.step < A.m || P.splits != A.splits || P.splits < 1 ||
      P.splits > A.k / part_of(A.g) || (P.splits > 1 && (glu || A.part == nullptr)))
    return hipErrorInvalidValue;
  if (bits == 4)
    return part_of(A.g) == 64 ? go_cols<4, 1>(A, P, glu, stream)
                              : go_cols<4, 2>(A, P, glu, stream);
  if (bits == 8)
    return part_of(A.g) == 64 ? go_cols<8, 1>(A, P, glu, stream)
                              : go_cols<8, 2>(A, P, glu, stream);
  return hipErrorInvalidValue;
}
