// K3i/K4i — dq_block's product where it is a large one: y[m, n] = x[m, k] ·
// dequant(W)[n, k]^T (+ bias), with the gate behind it, or by expert.
//
// The card's power bounds these products and not a unit of it: what is left of 691 us
// (3072 rows of n 28672, k 4096) is 557 when only the matrix instructions are left
// (1294 TFLOP/s, what the library's product reaches), at 2.07 GHz and less; without
// the reads of x from LDS it is 604, without the loads to LDS 635, without scaling
// some 650.  So what counts is the work beside the products, done or overlapped.
// Against dq_block (its tile, stages and split of a last round):
//
// - sum s (c - z) x = s (sum c x) - (s z) (sum x), and the sums of x's groups come from
//   a launch before, instead of from each of the workgroups of its rows.  The second
//   term is a product of bf16 parts, exact but for the last (times_sums): 8 k a group of
//   128 and at the rate of the first, an eighth of that in fp32.  It is taken off eight
//   groups at a time, halfway through them, so that what cancels stays small; all of it
//   before the loop is 1 % faster with 8 bits, but of x with a mean of one deviation, k
//   14336, the result was 2.4e-5 off (8 bits, groups of 64; 4 bits, of 128 3.5e-6) and
//   is 6.8e-7 (3.0e-7), with a mean of zero 6.9e-7 and 4.0e-7 (dq_block: 6.6e-7, 1.6e-7
//   and 4.0e-7).
// - 32 x 32 products, half as many instructions; a wave's 32 columns are one, and two
//   row tiles go side by side over half a chunk's k.  A half's products hide the
//   scaling of the chunk before or the unpacking of the half to come.
// - what is unpacked is held where it stands: the compiler moved it to the chunk that
//   uses it, in front of its products.
//
// A wave of 64 columns, which reads x half as often, needs more registers than
// instructions besides matrix ones can address; two waves of 64 rows and columns each
// unpack twice (723 us, 703 with 128 and 32).  Sums of x made from LDS in the loop: 810.
//
// us a call, dq_block and this one with the sums (groups of 128; 8 bits, of 64):
//                            2048 rows     3001 rows
//   n 28672, k 4096          471 / 445     705 / 657
//   n 6144, k 4096           116 / 115     167 / 157
//   n 4096, k 14336          228 / 219     338 / 332
//   n 28672, k 4096 (8)      595 / 562     887 / 838
//   n 8192, k 8192 (8)       341 / 329     486 / 468
#include "dq_block.h"
#include "lds_dma.h"

namespace {

typedef DqBlockPlan Plan;
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef u32 u32x2 __attribute__((ext_vector_type(2)));

constexpr int NW = 8, TPB = NW * LFMQ_WAVE, BN = NW * 32;
constexpr int ROWS = 128;                        // of a tile, at most
constexpr int D = 3;                             // stages
constexpr int SUMS = 48;                         // bytes of eight groups' sums

// LDS: x [D][rows][KC], weights [D][BN][..], two blocks of scales of eight groups;
// zeros and sums of x of one
template <int BITS, int KC>
struct Lds {
  static constexpr int XB = ROWS * KC * 2, WB = BN * KC * BITS / 8;
  static constexpr int W = D * XB, S = W + D * WB;
  static constexpr int SB = BN * 16, Z = S + 2 * SB, SUM = Z + BN * BITS;
  static constexpr int BYTES = SUM + ROWS * SUMS;
  static_assert(BYTES <= 160 * 1024 && BYTES >= ROWS * (BN + 8) * 2, "");
};

// A number of up to 16 significant bits (a scale times a zero) against the parts of
// a sum: two bf16 numbers make it up, three the sum, and of the eight k of a lane six
// are their products.
__device__ __forceinline__ s16x8 times_sums(float v) {
  const u32 b = __builtin_bit_cast(u32, v);
  const float hi = __builtin_bit_cast(float, b & 0xFFFF0000u);
  const u32 h = b >> 16, l = __builtin_bit_cast(u32, v - hi) >> 16;
  return __builtin_bit_cast(s16x8, u32x4{h | h << 16, h, l | l << 16, l});
}

// sums [m, k / g] of x's groups, each as -(a, b, c) in bf16 with a + b + c the sum in
// fp32: of eight groups a and b, and then c.  Eight lanes a group, 128 bytes of a row.
// Bound by reading x: 3001 x 4096 7 us.
__global__ __launch_bounds__(256) void dq_panel_sums(
    const unsigned short* __restrict__ x, char* __restrict__ sums, u32 groups,
    int g) {
  const u32 id = blockIdx.x * 32 + threadIdx.x / 8;
  if (id >= groups) return;
  const u32x4* p = (const u32x4*)(x + (u64)id * g) + threadIdx.x % 8;
  float sum = 0.f;
  for (int i = 0; i < g / 64; ++i) {
    const u32x4 v = p[i * 8];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      sum += bf16_bits_to_f32(v[e] & 0xFFFFu) + bf16_bits_to_f32(v[e] >> 16);
  }
#pragma unroll
  for (int d = 1; d < 8; d *= 2) sum += __shfl_xor(sum, d);
  if (threadIdx.x % 8) return;
  const u32 a = f32_to_bf16_bits_rne(-sum);
  const float ra = -sum - bf16_bits_to_f32(a);
  const u32 b = f32_to_bf16_bits_rne(ra);
  const u32 c = f32_to_bf16_bits_rne(ra - bf16_bits_to_f32(b));
  char* to = sums + (u64)(id / 8) * SUMS;
  ((u32*)to)[id % 8] = a | b << 16;
  ((unsigned short*)to)[16 + id % 8] = (unsigned short)c;
}

// the result's tile of column block nblk, part of it: MT row tiles of 32
template <int BITS, int KC, DqMode MODE, int MT>
__device__ __forceinline__ void dq_panel_body(const DqArgs& A,
                                              const char* sums_of_x, char* smem,
                                              const DqBlockTile& T) {
  typedef Lds<BITS, KC> L;
  constexpr int BM = MT * 32, J = KC / 16;       // products of 16 k a chunk
  constexpr int JH = J / 2, WH = JH * BITS / 4;  // of half a chunk; its words
  constexpr int MP = MT == 4 ? 2 : MT, NG = MT / MP;  // row tiles side by side
  constexpr int SL = KC / 8;                     // 16-byte slots a row of x
  constexpr int XL = BM * KC * 2 / 1024;         // 1 KiB loads of x a stage
  constexpr int NX = (XL + NW - 1) / NW;         // of a wave, at most
  constexpr int NL = L::WB / NW / 1024;          // of weights
  constexpr int PC = KC * BITS / 128;            // 16-byte pieces a column
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, hi = lane >> 5;
  const int row0 = T.row0, rows = T.rows, nblk = T.nblk, sp = T.sp;
  const int parts = T.parts;
  const int C = A.k / KC;
  const int c0 = (int)((long)C * sp / parts);
  const int c1 = (int)((long)C * (sp + 1) / parts);
  const int G = A.k / A.g, zw = (G + 32 / BITS - 1) / (32 / BITS);
  const int cpg = A.g / KC;                      // chunks a group
  const int half = A.n / 2, n0 = nblk * (MODE == GLU ? BN / 2 : BN);
  // column c of this workgroup: row of W.  GLU: a wave's first 16 are gate, the
  // others up
  auto column = [&](int c) {
    if (MODE == GLU)
      return (c >> 4 & 1) * half + min(n0 + (c >> 5) * 16 + (c & 15), half - 1);
    return min(n0 + c, A.n - 1);
  };
  // row of x of this workgroup's row r; rows past the end repeat the last one
  auto x_row = [&](int r) {
    r = min(r, rows - 1) + row0;
    return MODE != DENSE && A.src != nullptr ? A.src[r] : r;
  };
  // staging: a lane picks the 16 bytes that belong at its place
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
    xo[i] = (u32)(x_row(at) - (MODE == DENSE ? row0 : 0)) * pitch +
            ((lane % SL) ^ slot_key<SL>(at)) * 16;
  }
  const u32 wrow = A.k * BITS / 8;
  const u64 first = (u64)T.expert * A.n;           // the expert's rows of W
  const char* wb = A.w + first * wrow;
  u32 wo[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int e = (wave * NL + i) * 64 + lane, c = e / PC;
    wo[i] = (u32)column(c) * wrow + ((e % PC) ^ slot_key<PC>(c)) * 16;
  }
  auto load_x = [&](int c, int buf, int i) {
    load_to_lds(xb + (u64)c * (KC * 2), xo[i], buf * L::XB + nth(i) * 1024);
  };
  auto load_w = [&](int c, int buf, int i) {
    load_to_lds(wb + (u32)c * (KC * BITS / 8), wo[i],
                L::W + buf * L::WB + (wave * NL + i) * 1024);
  };
  // scales of groups 8 q .. 8 q + 7
  const u32 mcol = column((wave & 3) * 64 + lane);
  auto load_meta = [&](int q) {
    if (wave < 4)
      load_to_lds((const char*)(A.scales + first * G) + q * 16, mcol * (G * 2),
                  L::S + (q & 1) * L::SB + wave * 1024);
  };

  // zeros of groups 8 q .. 8 q + 7, and sums of x
  constexpr int NS = (BM * SUMS + 1023) / 1024;  // 1 KiB loads
  const u32 zo = mcol * (zw * 4) + (wave >> 2) * 4;
  u32 so;
  {
    const int e = min(wave * 64 + lane, BM * 3 - 1);
    so = (u32)x_row(e / 3) * (G / 8 * SUMS) + e % 3 * 16;
  }
  auto load_sums = [&](int q) {
    if (BITS == 8 || wave < 4)
      load4_to_lds((const char*)(A.zeros + first * zw) + q * BITS, zo,
                   L::Z + wave * 256);
    if (wave < NS) load_to_lds(sums_of_x + q * SUMS, so, L::SUM + wave * 1024);
  };
  f32x16 acc[MT] = {};
  // acc -= (scale times zero) (sums of x) of these groups, two to a product
  u32x4 ab[MT];                                  // a and b of this lane's four, and c
  u32x2 ec[MT], zs;
  u32 zz;
  auto read_zeros = [&](int q) {
    const int col = wave * 32 + l31;
    zs = *(const u32x2*)(smem + L::S + (q & 1) * L::SB + col * 16 + hi * 8);
    zz = *(const u32*)(smem + L::Z + col * 4 + (BITS == 8 ? hi * 1024 : 0));
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const char* p = smem + L::SUM + (t * 32 + l31) * SUMS;
      ab[t] = *(const u32x4*)(p + hi * 16);
      ec[t] = *(const u32x2*)(p + 32 + hi * 8);
    }
  };
  auto zeros_term = [&]() {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const u32 zero = BITS == 4 ? unpack4(zz, hi * 4 + e) : unpack8(zz, e);
      const u32 scale = e & 1 ? zs[e / 2] >> 16 : zs[e / 2] & 0xFFFFu;
      const s16x8 w = times_sums(bf16_bits_to_f32(scale) * (float)zero);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const u32 lo = ab[t][e];
        const u32 up = e & 1 ? ec[t][e / 2] >> 16 : ec[t][e / 2] & 0xFFFFu;
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(s16x8, u32x4{lo, up, lo, up}), w, acc[t], 0, 0, 0);
      }
    }
  };

  u32 w[2 * WH], meta;
  auto read_w = [&](int buf) {
    const char* p = smem + L::W + buf * L::WB + (wave * 32 + l31) * (PC * 16);
#pragma unroll
    for (int i = 0; i < WH / 2; ++i) {
      const u32x4 v =
          *(const u32x4*)(p + (((hi * (WH / 2) + i) ^ slot_key<PC>(l31)) << 4));
#pragma unroll
      for (int e = 0; e < 4; ++e) w[i * 4 + e] = v[e];
    }
  };
  float s;                                       // of the chunk's group
  auto read_meta = [&](int gi) {
    meta = *(const unsigned short*)(smem + L::S + (gi >> 3 & 1) * L::SB +
                                    (wave * 32 + l31) * 16 + (gi & 7) * 2);
  };
  // halves of a chunk's k, unpacked; x of a group of row tiles and half
  s16x8 b[2][JH], xa[2][MP][JH];
  f32x16 a[MT];
  auto read_x = [&](int buf, int g, int h, s16x8 (&x)[MP][JH]) {
#pragma unroll
    for (int j = 0; j < JH; ++j)
#pragma unroll
      for (int t = 0; t < MP; ++t)
        x[t][j] = *(const s16x8*)(smem + buf * L::XB +
                                  ((g * MP + t) * 32 + l31) * (KC * 2) +
                                  (((hi * J + h * JH + j) ^ slot_key<SL>(l31)) << 4));
  };
  auto unpack = [&](int h, int j) {
    b[h][j] = codes8_exact<BITS>(&w[(h * JH + j) * BITS / 4]);
    // here and not, as the compiler would have it, where they are used
    asm volatile("" : "+v"(b[h][j]));
  };

  int gi = c0 / cpg, gc = c0 % cpg;              // group, chunk in it
  const int m0 = gi >> 3;
  const int first_q = (c0 + 4 * cpg - 1) / (8 * cpg);  // half of it in this part
  {
    load_sums(min(first_q, G / 8 - 1));
#pragma unroll
    for (int i = 0; i < NL; ++i) load_w(c0, 0, i);
    load_meta(m0);
    if (8 * (m0 + 1) < G) load_meta(m0 + 1);
#pragma unroll
    for (int t = 0; t < D - 1; ++t) {
#pragma unroll
      for (int i = 0; i < NX; ++i) load_x(min(c0 + t, c1 - 1), t, i);
#pragma unroll
      for (int i = 0; i < NL; ++i) load_w(min(c0 + t + 1, c1 - 1), t + 1, i);
    }
    loads_but<0>();
    read_w(0);
    read_meta(gi);
    read_x(0, 0, 0, xa[0]);
#pragma unroll
    for (int j = 0; j < JH; ++j) unpack(0, j);
    s = 0.f;
#pragma unroll
    for (int t = 0; t < MT; ++t) a[t] = f32x16{};
  }
  auto fold = [&](int t) {
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = fmaf(s, a[t][r], acc[t][r]);
    asm volatile("" : "+v"(acc[t]));
  };
  int buf = 0;                                   // of chunk c: x, and W before
  for (int c = c0; c < c1; ++c) {
    const int b1 = buf == D - 1 ? 0 : buf + 1, b2 = b1 == D - 1 ? 0 : b1 + 1;
    if (gc == 0 && (gi & 7) == 0 && gi >> 3 != m0 && gi + 8 < G)
      load_meta((gi >> 3) + 1);
    // Zeros' terms of eight groups halfway through them (behind the first products, where
    // there are registers for their operands: 8 bits 2 % slower than without a term in
    // the loop, 1 % so), and the next ones' operands a chunk later, when all waves have
    // read these.
    const int cz = ((gi & 7) - 4) * cpg + gc;
    if (cz == 0) {
      read_zeros(gi >> 3);
      if (KC == 128) zeros_term();
    } else if (cz == 1 && (gi | 7) + 1 < G) {
      load_sums((gi >> 3) + 1);
    }
    if (++gc == cpg) {
      gc = 0;
      ++gi;
    }
    // loads past the last chunk repeat it
    const int cx = min(c + 2, c1 - 1), cw = min(c + 3, c1 - 1);
    constexpr int ITEMS = NX + NL, U = 2 * NG;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int h = u / NG, g = u % NG;
      if (u + 1 < U) {
        read_x(buf, (u + 1) % NG, (u + 1) / NG, xa[(u + 1) & 1]);
        // what comes goes where the chunk before has been read
#pragma unroll
        for (int i = u * ITEMS / (U - 1); i < (u + 1) * ITEMS / (U - 1); ++i) {
          if (i < NX) load_x(cx, b2, i);
          else load_w(cw, buf, i - NX);
        }
      } else {
        // x of the next chunk and the weights after it have landed, and all
        // waves have read this one's x: the last products are still to come
        loads_but<NX + NL>();
        read_x(b1, 0, 0, xa[0]);
      }
      // the next chunk's weights (past the last one, whatever lies there is read
      // and not used)
      if (u == NG) read_w(b1);
#pragma unroll
      for (int j = 0; j < JH; ++j)
#pragma unroll
        for (int t = 0; t < MP; ++t) {
          f32x16& to = a[g * MP + t];
          if (h == 0 && j == 0) {
            fold(g * MP + t);                    // the chunk before
            to = f32x16{};
          }
          to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[u & 1][t][j], b[h][j], to,
                                                       0, 0, 0);
        }
#pragma unroll
      for (int j = g * JH / NG; j < (g + 1) * JH / NG; ++j) unpack(h ^ 1, j);
      if (KC == 64 && u == 0 && cz == 0) zeros_term();
      if (u == NG - 1) s = bf16_bits_to_f32(meta);
      if (u == U - 1) read_meta(gi);
      __builtin_amdgcn_sched_barrier(0);
    }
    buf = b1;
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) fold(t);
  loads_but<0>();

  // result: column l31, rows r % 4 + 8 (r / 4) + 4 hi
  auto row_of = [&](int t, int r) { return t * 32 + r % 4 + r / 4 * 8 + hi * 4; };
  if (float* part = T.part) {                     // [rows][BN], as the waves lie
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (row_of(t, r) < rows)
          part[row_of(t, r) * BN + wave * 32 + l31] = acc[t][r];
    return;
  }
  if (MODE == SLOTS) {
    const int col = n0 + wave * 32 + l31;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (row_of(t, r) < rows && col < A.n)
          A.y32[(u64)(row0 + row_of(t, r)) * A.n + col] = acc[t][r];
    return;
  }
  // through LDS, so that rows are written in 16-byte pieces
  constexpr int BO = MODE == GLU ? BN / 2 : BN, LD = BO + 8;
  const int nout = MODE == GLU ? half : A.n;
  unsigned short* out = (unsigned short*)smem;
  __syncthreads();
  if constexpr (MODE == GLU) {
    // gate and up of a column are 16 lanes apart: of two rows, one lane gets both of
    // the first and the other of the second
    const int second = lane >> 4 & 1, c = wave * 16 + (lane & 15);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float even = acc[t][r], odd = acc[t][r + 1];
        const u32x2 v = __builtin_amdgcn_permlane16_swap(
            __builtin_bit_cast(u32, even), __builtin_bit_cast(u32, odd), false, false);
        const u32 gate = v[0], up = v[1];
        out[(row_of(t, r) + second) * LD + c] =
            (unsigned short)f32_to_bf16_bits_rne(
                silu_mul_f(__builtin_bit_cast(float, gate),
                           __builtin_bit_cast(float, up)));
      }
  } else {
    const int c = wave * 32 + l31;
    const float bias = A.bias != nullptr && n0 + c < A.n
                           ? bf16_bits_to_f32(A.bias[n0 + c])
                           : 0.f;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        out[row_of(t, r) * LD + c] =
            (unsigned short)f32_to_bf16_bits_rne(acc[t][r] + bias);
  }
  __syncthreads();
  dq_block_store(out, LD, BM, BO, A.y, row0, rows, n0, nout, tid, TPB);
}

template <int BITS, int KC, DqMode MODE>
__global__ __launch_bounds__(TPB, 2) void dq_panel_kernel(DqArgs A, Plan P,
                                                          const char* sums) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const u32 nb = MODE == GLU ? (A.n / 2 + BN / 2 - 1) / (BN / 2)
                             : (A.n + BN - 1) / BN;
  DqBlockTile T;
  if (!dq_block_tile<MODE>(A, P, nb, BN, T)) return;
  // (in this order: as the first of them the last made the others 1 % slower)
  if (T.rows > 96)
    dq_panel_body<BITS, KC, MODE, 4>(A, sums, smem, T);
  else if (T.rows > 64)
    dq_panel_body<BITS, KC, MODE, 3>(A, sums, smem, T);
  else if (MODE == DENSE || T.rows > 32)
    dq_panel_body<BITS, KC, MODE, 2>(A, sums, smem, T);
  else
    dq_panel_body<BITS, KC, MODE, 1>(A, sums, smem, T);
}

template <int BITS, int KC, DqMode MODE>
hipError_t go(const DqArgs& A, const Plan& P, u32 wgs, const char* sums,
              hipStream_t stream) {
  constexpr int lds = Lds<BITS, KC>::BYTES;
  static bool set = false;
  if (!set) {
    LFMQ_CHECK_HIP(hipFuncSetAttribute(
        (const void*)dq_panel_kernel<BITS, KC, MODE>,
        hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    set = true;
  }
  hipLaunchKernelGGL((dq_panel_kernel<BITS, KC, MODE>),
                     dim3(wgs, MODE == SLOTS ? P.parts : 1), dim3(TPB), lds,
                     stream, A, P, sums);
  return hipGetLastError();
}

template <DqMode MODE>
hipError_t go_bits(const DqArgs& A, const Plan& P, int bits, u32 wgs,
                   const char* sums, hipStream_t stream) {
  if (bits == 4)
    return A.g % 128 == 0 ? go<4, 128, MODE>(A, P, wgs, sums, stream)
                          : go<4, 64, MODE>(A, P, wgs, sums, stream);
  return go<8, 64, MODE>(A, P, wgs, sums, stream);
}

}  // namespace

// The launch of the sums is 2 us and reads x, which some 2048 columns' gain pays for.
// us of dq_block / this one (4 bits, 128 unless said): n 4096, k 2048 22.5 / 25 at 271
// rows, n 6656, k 4096 54.7 / 53.3 at 806, n 25216, k 4096 63.8 / 61.7 at 234; few
// columns, n 1728, k 10240 51.9 / 53.5 at 895; stages of 64 (8 bits, groups of 64),
// n 7104, k 3584 34.3 / 36.2 at 210, n 6784, k 10752 73.4 / 66.0 at 220.  Of 400 random
// calls of 49 to 1500 rows 1.07 times as fast in the mean where it is taken.
bool lfmq_dq_panel_gains(long rows, long n, long k, long g, long bits) {
  return rows * k * (n - 2048) >= (bits == 4 && g % 128 == 0 ? 12l << 30 : 8l << 30);
}

hipError_t lfmq_dq_panel(const DqArgs& A, const DqBlockPlan& P, int bits, DqMode mode,
                         u32 wgs, void* sums, long rows, hipStream_t stream) {
  const long groups = rows * (A.k / A.g);
  if (groups < 1 || groups * 8 >= 1l << 32) return hipErrorInvalidValue;
  hipLaunchKernelGGL(dq_panel_sums, dim3(ceil_div_u32((u32)groups, 32)), dim3(256), 0,
                     stream, (const unsigned short*)A.x, (char*)sums, (u32)groups, A.g);
  LFMQ_CHECK_HIP(hipGetLastError());
  const char* s = (const char*)sums;
  return mode == DENSE ? go_bits<DENSE>(A, P, bits, wgs, s, stream)
         : mode == GLU ? go_bits<GLU>(A, P, bits, wgs, s, stream)
                       : go_bits<SLOTS>(A, P, bits, wgs, s, stream);
}
