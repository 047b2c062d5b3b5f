// K3b/K4b — W4A16 / W8A16 product for prompts: y[m, n] = x[m, k] ·
// dequant(W)[n, k]^T (+ bias).  Groups that dq_block does not take, 8 bits in
// groups of 128 up to some 200 rows, small matrices a few rows above 128.
//
// A workgroup computes 128 rows by 128 columns, four waves side by side in
// the columns, each all 128 rows by 32 columns.  x goes through LDS (two
// buffers of KC values of k, 16-byte blocks XOR-swizzled by the row), since
// all waves read it; the packed weights do not: a lane reads its columns'
// bytes straight into registers and turns them into operands there
// (dq_frag.h), so that LDS carries one operand only, and a weight is
// unpacked once per 128 rows.  Scales apply per group to the fp32 results.
// The sums of x that the zeros need are shared out: a wave makes a quarter
// of the rows' with products by ones, and all waves apply them a chunk later.
//
// Bound by latencies between the stages of two waves a SIMD (matrix cores
// busy 41 % of the time, vector units 46 %, LDS half: 3001 rows of n 28672, k
// 4096, which are dq_block's now).  128 x 256 tiles with one wave a SIMD: 570
// TFLOP/s and not 832.  slot_key's order of LDS slots, which pairs of lanes
// share: the same within 2 %.  us a call (TFLOP/s):
//                                  100 rows   256 rows   1500 rows   3001 rows
//   n 4096, k 11008 (4 bits)          37         48       195 (692)   403 (672)
//   n 5120, k 13824                   41         67       274 (776)   536 (793)
//   n 28672, k 4096 (8, group 128)    57         95
#include "dq_frag.h"
#include "lds_dma.h"

namespace {

constexpr int NW = 4, TPB = NW * LFMQ_WAVE;

constexpr int ROWS = 128;                        // of a tile, at most

// rows row0 .. of x (or slots), MT * 16 of them at most
template <int BITS, int KC, DqMode MODE, int MT>
__device__ __forceinline__ void dq_tile_body(const DqArgs& A, char* smem,
                                             int row0, int rows, int expert,
                                             int nblk, int sp) {
  constexpr int NT = 2, BM = MT * 16, BN = NW * NT * 16;
  constexpr int J = KC / 32, WD = J * BITS / 4;
  constexpr int SL = KC / 8;                     // 16-byte slots a row
  constexpr int NX = BM * SL / TPB;              // staged slots a thread
  constexpr int XB = ROWS * KC * 2;
  float* xsum = (float*)(smem + 2 * XB);         // [2][BM]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4;
  const int C = A.k / KC;
  const int c0 = (int)((long)C * sp / A.splits);
  const int c1 = (int)((long)C * (sp + 1) / A.splits);
  const int G = A.k / A.g, zw = (G + 32 / BITS - 1) / (32 / BITS);
  auto key = [](int row) { return slot_key16<SL>(row); };
  // columns of this workgroup; GLU: a wave's first 16 are gate, the others up
  const int half = A.n / 2, n0 = nblk * (MODE == GLU ? BN / 2 : BN);

  // staging: a wave's load writes 1 KiB of LDS in lane order, so the lane
  // picks the slot that belongs there; rows past the end repeat the last one
  const unsigned short* xb = MODE == DENSE ? A.x + (u64)row0 * A.k : A.x;
  constexpr int RS = NW * 64 / SL;               // rows between a lane's slots
  static_assert(RS % 16 == 0, "which share one swizzle key");
  const int xrow = wave * 64 / SL + lane / SL;
  const u32 xslot = ((lane % SL) ^ key(xrow)) * 16, pitch = A.k * 2;
  u32 xo[MODE == DENSE ? 1 : NX];                // experts: rows by src
  if constexpr (MODE == DENSE) {
    xo[0] = xrow * pitch;
  } else {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      int r = row0 + min(xrow + i * RS, rows - 1);
      if (A.src != nullptr) r = A.src[r];
      xo[i] = (u32)r * pitch + xslot;
    }
  }
  auto stage = [&](int c, int buf) {
    const char* base = (const char*)(xb + c * KC);
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const u32 off = MODE == DENSE ? min(xo[0] + (u32)(i * RS) * pitch,
                                          (u32)(rows - 1) * pitch) + xslot
                                    : xo[MODE == DENSE ? 0 : i];
      load_to_lds(base, off, buf * XB + (i * NW + wave) * 1024);
    }
  };
  // weights: a matrix is below 4 GiB
  const int wrow = A.k * BITS / 8;
  const char* wb = A.w + (u64)expert * A.n * wrow;
  const unsigned short* sb = A.scales + (u64)expert * A.n * G;
  const u32* zb = A.zeros + (u64)expert * A.n * zw;
  u32 wo[NT], col[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    col[t] = MODE == GLU ? t * half + min(n0 + wave * 16 + l15, half - 1)
                         : min(n0 + (wave * NT + t) * 16 + l15, A.n - 1);
    wo[t] = col[t] * wrow + l4 * (WD * 4);
  }

  u32 wn[NT][WD];
  // scales and zeros of eight groups at a time (fetched per chunk, their
  // lines would be more traffic than the weights), or of one where rows of
  // scales are no multiple of that
  const bool by8 = G % 8 == 0;
  u32x4 sq[NT];
  u32 zq[NT][BITS / 4];
  auto fetch = [&](int c) {
    const int gi = c * KC / A.g;
    const bool next8 = c == c0 || (gi % 8 == 0 && c * KC % A.g == 0);
    if (!by8) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        sq[t][0] = sb[col[t] * G + gi];
        zq[t][0] = zb[col[t] * zw + gi / (32 / BITS)];
      }
    } else if (next8) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        sq[t] = *(const u32x4*)(sb + col[t] * G + (gi & ~7));
#pragma unroll
        for (int i = 0; i < BITS / 4; ++i)
          zq[t][i] = zb[col[t] * zw + (gi & ~7) / (32 / BITS) + i];
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const u32* p = (const u32*)(wb + (wo[t] + (u32)c * (KC * BITS / 8)));
      if constexpr (WD >= 4) {
#pragma unroll
        for (int i = 0; i < WD / 4; ++i) {
          const u32x4 v = *((const u32x4*)p + i);
#pragma unroll
          for (int e = 0; e < 4; ++e) wn[t][i * 4 + e] = v[e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < WD; ++e) wn[t][e] = p[e];
      }
    }
  };

  const s16x8 ones = bf16_ones();
  f32x4 acc[MT][NT] = {};
  float szp[NT] = {};                            // the chunk before's
  // the four lanes of a row tile's sums from the chunk before
  auto xs_of = [&](int par, int t) {
    return *(const f32x4*)(xsum + par * BM + t * 16 + l4 * 4);
  };
  fetch(c0);
  stage(c0, 0);
  if (tid < BM) xsum[BM + tid] = 0.f;            // no chunk before the first
  for (int c = c0; c < c1; ++c) {
    const int par = (c - c0) & 1;
    const char* buf = smem + par * XB;
    // this chunk's loads have landed (a wave waits for its own), the other
    // buffer is consumed
    lds_loads_done();
    s16x8 b[NT][J], xa[2][J];
    float s[NT], sz[NT];
    const int gi = c * KC / A.g;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
      for (int j = 0; j < J; ++j)
        b[nt][j] = codes8<BITS>(&wn[nt][j * BITS / 4]);
      if (by8) {
        const u32 lo = gi & 2 ? sq[nt][1] : sq[nt][0];
        const u32 hi = gi & 2 ? sq[nt][3] : sq[nt][2];
        const u32 d = gi & 4 ? hi : lo;
        s[nt] = bf16_bits_to_f32(gi & 1 ? d >> 16 : d & 0xFFFFu);
      } else {
        s[nt] = bf16_bits_to_f32(sq[nt][0]);
      }
      const u32 z = BITS == 8 && by8 && (gi & 4) ? zq[nt][BITS / 4 - 1]
                                                 : zq[nt][0];
      sz[nt] = s[nt] * zero_bias<BITS>(z, gi);
    }
    if (c + 1 < c1) {
      stage(c + 1, par ^ 1);
      fetch(c + 1);
    }
    auto load = [&](int row, int j) {
      return *(const s16x8*)(buf + row * (KC * 2) +
                             (((l4 * J + j) ^ key(l15)) << 4));
    };
    f32x4 a[2][NT], xp[2];
    auto fold = [&](int t) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[t][nt][r] = fmaf(s[nt], a[t & 1][nt][r],
                               fmaf(-szp[nt], xp[t & 1][r], acc[t][nt][r]));
      // here: sunk behind all products, as the compiler likes it, they leave
      // the matrix cores idle and take 256 registers (3001 x 28672 x 4096: 951
      // us, 907 so; 3001 x 6144 x 4096: 242, 216)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) asm volatile("" : "+v"(acc[t][nt]));
    };
#pragma unroll
    for (int j = 0; j < J; ++j) xa[0][j] = load(l15, j);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      // the next rows on their way, the last ones scaled during the products
      xp[t & 1] = xs_of(par ^ 1, t);
      if (t + 1 < MT) {
#pragma unroll
        for (int j = 0; j < J; ++j)
          xa[(t + 1) & 1][j] = load((t + 1) * 16 + l15, j);
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) a[t & 1][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          a[t & 1][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              xa[t & 1][j], b[nt][j], a[t & 1][nt], 0, 0, 0);
      if (t > 0) fold(t - 1);
      // row tiles kept apart (free, W8 loses 2 %)
      __builtin_amdgcn_sched_barrier(0);
    }
    // this wave's share of the chunk's sums
    constexpr int XS = (MT + NW - 1) / NW;
    f32x4 xs[XS] = {};
#pragma unroll
    for (int i = 0; i < XS; ++i)
      if (MT % NW == 0 || i * NW + wave < MT)
#pragma unroll
        for (int j = 0; j < J; ++j)
          xs[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              load((i * NW + wave) * 16 + l15, j), ones, xs[i], 0, 0, 0);
    fold(MT - 1);
    if (l15 == 0) {
#pragma unroll
      for (int i = 0; i < XS; ++i)
        if (MT % NW == 0 || i * NW + wave < MT)
          *(f32x4*)(xsum + par * BM + (i * NW + wave) * 16 + l4 * 4) = xs[i];
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) szp[t] = sz[t];
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const f32x4 xp = xs_of((c1 - c0 - 1) & 1, t);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[t][nt][r] = fmaf(-szp[nt], xp[r], acc[t][nt][r]);
  }

  // C fragment: column l15, rows l4 * 4 + r
  if (MODE == SLOTS || (MODE == DENSE && A.splits > 1)) {
    float* part = MODE == SLOTS ? A.y32 : A.part + (u64)sp * A.m * A.n;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = t * 16 + l4 * 4 + r;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int col = n0 + (wave * NT + nt) * 16 + l15;
          if (row < rows && col < A.n)
            part[(u64)(row0 + row) * A.n + col] = acc[t][nt][r];
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
  const bool wide = nout % 8 == 0;
  for (int i = tid; i < BM * BO / 8; i += TPB) {
    const int row = i / (BO / 8), c = i % (BO / 8) * 8;
    const int gc = n0 + c;
    if (row >= rows || gc >= nout) continue;
    unsigned short* p = A.y + (u64)(row0 + row) * nout + gc;
    const unsigned short* q = out + row * LD + c;
    if (wide) {
      *(u32x4*)p = *(const u32x4*)q;
    } else {
      for (int e = 0; e < 8 && gc + e < nout; ++e) p[e] = q[e];
    }
  }
}

// step: rows from tile to tile (without a list of them).  A tile takes the smallest body of 64,
// 96 or 128 rows that holds it; LARGE: there is none below 97.
template <int BITS, int KC, DqMode MODE, bool LARGE>
__global__ __launch_bounds__(TPB, 2) void dq_tile_kernel(DqArgs A, int mb,
                                                         int step) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // Up to eight row tiles: an XCD takes a range of columns, row tiles fastest
  // (n 28672, k 4096, 256 rows: 94 us, 97 columns fastest over all XCDs; 8
  // bits, n 32000: 96, 102).  More: columns fastest (2600 rows: 809, 765; 660
  // tokens through 8 experts 924, 869), or, where every eighth row tile is the
  // same XCD's, row tiles (3001 rows: 924 / 865 / 847 in this order).
  const u32 nb = MODE == GLU ? (A.n / 2 + 63) / 64 : (A.n + 127) / 128;
  const bool list = MODE != DENSE && A.tiles != nullptr;
  const bool ranges = !list && mb <= 8;
  u32 id = ranges ? xcd_swizzle(blockIdx.x, gridDim.x) : blockIdx.x;
  u32 mt, nblk;
  if (ranges || (!list && mb % 8 == 0)) {
    mt = id % mb;
    id /= mb;
    nblk = id % nb;
    id /= nb;
  } else {
    nblk = id % nb;
    id /= nb;
    mt = id % mb;
    id /= mb;
  }
  const int sp = (int)id;
  int row0 = (int)mt * step, rows = min(A.m - row0, step), expert = 0;
  if (list) {
    expert = A.tiles[3 * mt];
    if (expert < 0) return;
    row0 = A.tiles[3 * mt + 1];
    rows = A.tiles[3 * mt + 2];
  }
  if (!LARGE && rows <= 64)
    dq_tile_body<BITS, KC, MODE, 4>(A, smem, row0, rows, expert, nblk, sp);
  else if (!LARGE && rows <= 96)
    dq_tile_body<BITS, KC, MODE, 6>(A, smem, row0, rows, expert, nblk, sp);
  else
    dq_tile_body<BITS, KC, MODE, 8>(A, smem, row0, rows, expert, nblk, sp);
}

template <int BITS, int KC, DqMode MODE, bool LARGE>
hipError_t go(const DqArgs& A, int mb, int step, hipStream_t stream) {
  // two buffers and the sums; the result, padded, takes a little more
  constexpr size_t bufs = 2 * ROWS * KC * 2 + 2 * ROWS * 4;
  constexpr size_t out = ROWS * 136 * 2;
  constexpr size_t lds = bufs > out ? bufs : out;
  static bool set = false;
  if (!set && lds > 64 * 1024) {
    LFMQ_CHECK_HIP(hipFuncSetAttribute(
        (const void*)dq_tile_kernel<BITS, KC, MODE, LARGE>,
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    set = true;
  }
  const u32 nb = MODE == GLU ? ceil_div_u32(A.n / 2, 64)
                             : ceil_div_u32(A.n, 128);
  hipLaunchKernelGGL((dq_tile_kernel<BITS, KC, MODE, LARGE>),
                     dim3(mb * nb * A.splits), dim3(TPB), lds, stream, A, mb,
                     step);
  return hipGetLastError();
}

template <DqMode MODE, bool LARGE>
hipError_t go_bits(const DqArgs& A, int bits, int mb, int step,
                   hipStream_t stream) {
  if (bits == 4)
    return A.g % 128 == 0 ? go<4, 128, MODE, LARGE>(A, mb, step, stream)
                          : go<4, 64, MODE, LARGE>(A, mb, step, stream);
  if (bits == 8)
    return A.g % 128 == 0 ? go<8, 128, MODE, LARGE>(A, mb, step, stream)
                          : go<8, 64, MODE, LARGE>(A, mb, step, stream);
  return hipErrorInvalidValue;
}

// Rows of the tiles of a whole k.  Two workgroups a CU take a round, one
// alone 0.69 of it; a tile of 96 rows 0.9 of one of 128, of 64 rows 0.75 (less
// where the rounds are many, but then the last one does not matter).  us with
// 128 / 96 / 64, 4 bits, k 4096: n 6144, 1300 rows 131 / 118 / 103, 1500 rows
// 133 / 118 / 136, 1024 rows 73 / 106 / 92; n 4096, 1500 rows 78 / 70 / 92; n
// 28672, 800 rows 277 / 268 / 302.
int tile_rows(int m, int n, int cols) {
  int best = ROWS;
  float least = INFINITY;
  for (int r = ROWS; r >= 64; r -= 32) {
    const u32 u = ceil_div_u32(ceil_div_u32(m, r) * ceil_div_u32(n, cols), 256);
    const float t = ((u / 2) + (u & 1) * 0.69f) *
                    (r == 128 ? 1.f : (r == 96 ? 0.9f : 0.75f));
    if (t < least * 0.99f) {
      least = t;
      best = r;
    }
  }
  return best;
}

}  // namespace

bool lfmq_dq_tile_ok(int k, int g) {
  return g % 64 == 0 && g <= k && k % g == 0;
}

int lfmq_dq_tile_splits(int m, int n, int k, int g) {
  const int wgs = max(1, (int)(ceil_div_u32(n, 128) * ceil_div_u32(m, 128)));
  const int C = k / (g % 128 == 0 ? 128 : 64);
  // 256 workgroups, or 512 where six chunks are left to each (us at 64 rows,
  // 4 bits: n 28672, k 4096 57 / 48, n 6144 21.8 / 23.8, n 4096, k 14336
  // 34 / 31)
  const int s = max(1, min(256 / wgs, C / 4));
  return 512 / wgs <= C / 6 ? max(s, 512 / wgs) : s;
}

// glu: y [m, n / 2] = silu(gate) up of W = [gate | up], without bias and
// residual.  end: with splits only, what lfmq_dq_rows_sum takes.
hipError_t lfmq_dq_tile(const void* qweight, const void* scales,
                        const void* qzeros, const void* x, void* y,
                        const void* bias, const void* resid, void* part,
                        int m, int n, int k, int g, int bits, int splits,
                        bool glu, hipStream_t stream, const DqRowEnd* end) {
  if (resid != nullptr && splits == 1) return hipErrorInvalidValue;
  if (glu && (n % 2 || bias != nullptr || resid != nullptr ||
              (u64)m * k * 2 >= 1ull << 32))
    return hipErrorInvalidValue;
  if (!lfmq_dq_tile_ok(k, g) || (u64)n * k * bits / 8 >= 1ull << 32)
    return hipErrorInvalidValue;
  const DqArgs A{(const char*)qweight, (const unsigned short*)scales,
                 (const u32*)qzeros, (const unsigned short*)x,
                 (unsigned short*)y, (const unsigned short*)bias, nullptr,
                 (float*)part, m, n, k, g, splits, nullptr, nullptr, nullptr};
  // row tiles alike, in sixteens: 129 rows are two of 80
  const int most = splits == 1 ? tile_rows(m, glu ? n / 2 : n, glu ? 64 : 128)
                               : ROWS;
  const int mb = (int)ceil_div_u32(m, most);
  const int step = (int)ceil_div_u32(ceil_div_u32(m, mb), 16) * 16;
  hipError_t e;
  if (glu && splits == 1)
    e = step <= 96 ? go_bits<GLU, false>(A, bits, mb, step, stream)
                   : go_bits<GLU, true>(A, bits, mb, step, stream);
  else
    e = step <= 96 ? go_bits<DENSE, false>(A, bits, mb, step, stream)
                   : go_bits<DENSE, true>(A, bits, mb, step, stream);
  if (e != hipSuccess || splits == 1) return e;
  return lfmq_dq_rows_sum(part, y, bias, resid, m, n, splits, glu, stream,
                          nullptr, end);
}

// rows of x (or slots) by expert, tiles of up to 128 of them (DqArgs); glu:
// y bf16 [slots, n / 2], else fp32 [slots, n]
hipError_t lfmq_dq_tile_experts(const void* qweight, const void* scales,
                                const void* qzeros, const void* x,
                                const void* src, const void* tiles, void* y,
                                int n_tiles, int n, int k, int g, int bits,
                                bool glu, hipStream_t stream) {
  if (!lfmq_dq_tile_ok(k, g) || (glu && n % 2) ||
      (u64)n * k * bits / 8 >= 1ull << 32)
    return hipErrorInvalidValue;
  DqArgs A{};
  A.w = (const char*)qweight;
  A.scales = (const unsigned short*)scales;
  A.zeros = (const u32*)qzeros;
  A.x = (const unsigned short*)x;
  A.y = (unsigned short*)y;
  A.y32 = (float*)y;
  A.src = (const i32*)src;
  A.tiles = (const i32*)tiles;
  A.n = n;
  A.k = k;
  A.g = g;
  A.splits = 1;
  return glu ? go_bits<GLU, false>(A, bits, n_tiles, 0, stream)
             : go_bits<SLOTS, false>(A, bits, n_tiles, 0, stream);
}
