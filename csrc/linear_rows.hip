// y[m, n] = x[m, k] W[n, k]^T in bf16 for up to 16 rows (decode steps of the
// models with 16-bit weights), sums in fp32; optionally the gated half of a
// fused gate and up projection, silu(y[:, c]) * y[:, c + n / 2].
//
// Bound by reading W once, and at these sizes by latency: eight waves share k
// in chunks of 128.  A load takes a whole 128-byte line of eight columns, so that
// it is asked for once and, from 4 MiB on, passes the caches by; a lane has two
// pieces of it in turn, and lanes of the other eight columns exchange theirs on the
// way into the operands of the matrix instruction.  x is read in the same order
// from the caches; the waves' sums meet in LDS, since a split of k over workgroups
// would take a second launch.
//
// A workgroup has NT tiles of 16 / KS columns (gate: a tile and its up).
// KS 2: up to eight rows.  Row and column i of the tile then stand for row and
// column i % 8 in share i / 8 of k, the even or the odd pieces; what meets in the
// two squares on the diagonal is added, the rest is not read.
//
// us by 64 bytes of 16 columns a load and tiles of 16 columns, and now, weights not
// cached: 32000 x 4096 at 1 row 46.6 / 43.6 (6.0 TB/s), 8 rows 52.6 / 46.9, 16 rows
// 64.2 / 48.4; 10240 x 5120 at 8 rows 31.4 / 22.7; at 3 rows 6144 x 2048 8.3 / 7.2
// (the library 12.3), 2048 x 2048 5.1 / 4.2 (8.4), 16384 x 2048 with silu 14.7 / 13.3
// (21.0), 32000 x 2048 25.1 / 24.3 (31); 2048 x 8192 at 4 rows 11.2 / 9.3.
#include "common.h"

namespace {

constexpr int KC = 128, NW = 8, TPB = NW * 64;

struct LArgs {
  const unsigned short *x, *w;
  unsigned short* y;
  u64 ldx;
  int m, n, k;
};

template <bool HI>
__device__ __forceinline__ s16x8 other8(s16x8 a, s16x8 b) {
  const u32x4 x = __builtin_bit_cast(u32x4, a), y = __builtin_bit_cast(u32x4, b);
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = ::other8<HI>(x[e], y[e]);
  return __builtin_bit_cast(s16x8, o);
}

template <int NT, int U, int KS, bool GLU, bool PAST>
__global__ __launch_bounds__(TPB) void linear_rows_kernel(LArgs A) {
  static_assert(KS == 1 || KS == 2, "");
  constexpr int S = 16 / KS, BN = GLU ? S : NT * S;
  __shared__ f32x4 red[NW][NT][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4, l7 = l15 & 7, odd = l15 >> 3;
  const int cols = GLU ? A.n / 2 : A.n, n0 = blockIdx.x * BN;
  // a load takes a 128-byte line of eight columns: pieces l4 * 2 and l4 * 2 + 1 of
  // column l7, the second in the upper eight lanes
  constexpr int H = 2 / KS;                // eights of columns a tile
  const unsigned short* wp[NT][H];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int h = 0; h < H; ++h)
      wp[t][h] = A.w + (l4 * 2 + odd) * 8 + (u64)A.k *
                 (GLU ? min(n0 + h * 8 + l7, cols - 1) + t * cols
                      : min(n0 + t * S + h * 8 + l7, cols - 1));
  // KS 1: row l15, both pieces; KS 2: row l7, the piece of the columns' lanes
  const unsigned short* xp = A.x + (u64)min(KS == 1 ? l15 : l7, A.m - 1) * A.ldx +
                             l4 * 16 + (KS == 1 ? 0 : odd * 8);

  f32x4 acc[NT] = {};
  const int C = A.k / KC;
  for (int c0 = wave; c0 < C; c0 += NW * U) {
    s16x8 b[U][NT][H][2], a[U][2][H];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = min(c0 + u * NW, C - 1);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int h = 0; h < H; ++h) {
            const s16x8* p = (const s16x8*)(wp[t][h] + c * KC + j * 64);
            b[u][t][h][j] = PAST ? __builtin_nontemporal_load(p) : *p;
          }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = min(c0 + u * NW, C - 1);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int h = 0; h < H; ++h)
          a[u][j][h] = *(const s16x8*)(xp + c * KC + j * 64 + h * 8);
    }
    __builtin_amdgcn_sched_barrier(0);     // all loads before the first use
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // past the end the last chunk came again: times zero weights, so that
      // nothing of x (infinities too) counts twice
      const bool live = c0 + u * NW < C;
      const s16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const s16x8 x = live ? a[u][j][h] : zero;
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            s16x8 w = b[u][t][h][j];
            if constexpr (H == 2)
              w = h == 0 ? other8<true>(b[u][t][0][j], b[u][t][1][j])
                         : other8<false>(b[u][t][1][j], b[u][t][0][j]);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                x, live ? w : zero, acc[t], 0, 0, 0);
          }
        }
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) red[wave][t][lane] = acc[t];
  __syncthreads();
  // row r of column c (of tile o): in lane r / 4 * 16 + c, element r % 4
  for (int e = tid; e < S * BN; e += TPB) {
    const int r = e / BN, o = e % BN / S, c = e % S;
    float v[NT];
#pragma unroll
    for (int t = 0; t < (GLU ? NT : 1); ++t) {
      v[t] = 0.f;
#pragma unroll
      for (int g = 0; g < NW; ++g)
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const int i = s * S + r;
          v[t] += red[g][o + t][i / 4 * 16 + s * S + c][i % 4];
        }
    }
    const int col = n0 + o * S + c;
    if (r < A.m && col < cols) {
      const float z = GLU ? v[0] / (1.f + __expf(-v[0])) * v[NT - 1] : v[0];
      A.y[(u64)r * cols + col] = (unsigned short)f32_to_bf16_bits_rne(z);
    }
  }
}

// From how many weights on they pass the caches by (4 MiB).  us by them / past them:
// 1024 x 1024 at 4 rows 3.3 / 3.4, 2048 x 2048 5.3 / 5.0, 32000 x 4096 at 1 row
// 46.3 / 45.0, 128256 x 4096 at 9 194 / 190.
constexpr long PAST_CACHES = 2l << 20;

// Columns of a workgroup.  Few rows want many workgroups, more rows few that read
// x; and a chip of 256 CUs, whole rounds of them: so the least of rounds times
// (columns / 16 + 0.75 rows / 16), a round of what is left counted whole up to 8
// rounds, and up to 5 rows of long k the wide tiles 1.1 times.  Up to 2 rows
// always 8 (a gate up to 4).  Over 630 measured shapes of 1 to 16 rows, 1024 to 50304
// columns, k 1024 to 14336 the choice is 0.7 % slower than the best of these tiles
// (16 columns but for a few shapes, as it was: 18 %).  us at 16 and the columns
// chosen: 32000 x 4096, 1 row 45.0 / 39.9 (8), 8 rows 50.3 / 46.7 (64), 16 rows 61.8
// / 48.8 (64); 10240 x 5120, 8 rows 30.0 / 21.1 (48); 1024 x 2048, 4 rows 4.6 / 3.7
// (8); with a gate 16384 x 2048, 1 row 14.0 / 12.9 (8).
int columns(int m, int cols, int k, bool glu) {
  if (m <= (glu ? 4 : 2)) return 8;
  int best = 0;
  float least = INFINITY;
  static const int tiles[] = {16, 32, 64, 48, 8};
  for (int c : tiles) {
    if ((c == 8 && m > 8) || (glu && c > 16)) continue;
    const int wgs = (cols + c - 1) / c, whole = (wgs + 255) / 256;
    const float rounds = whole > 8 ? wgs / 256.f : (float)whole;
    float t = rounds * ((glu ? 2 : 1) * c / 16.f + 0.75f * m / 16.f);
    if (c > 16 && m <= 5 && k >= 4096) t *= 1.1f;
    if (t < least) {
      least = t;
      best = c;
    }
  }
  return best;
}

}  // namespace

bool lfmq_linear_rows_ok(const void* x, long ldx, const void* w, int m, int n,
                         int k) {
  // few columns, long sums and too many rows to share k: the library splits
  // k (2048 x 8192: 12.3 us at 16 rows, 17.5 here)
  if (m > 8 && n <= 4096 && k > 4096) return false;
  return m >= 1 && m <= 16 && n >= 1 && k >= KC && k % KC == 0 &&
         ldx % 8 == 0 && ((u64)x | (u64)w) % 16 == 0;
}

// x [m, k], rows ldx apart; w [n, k]; y [m, n], or [m, n / 2] with glu
hipError_t lfmq_linear_rows(const void* x, long ldx, const void* w, void* y,
                            int m, int n, int k, bool glu,
                            hipStream_t stream) {
  if (!lfmq_linear_rows_ok(x, ldx, w, m, n, k) || (glu && n % 2))
    return hipErrorInvalidValue;
  const LArgs A{(const unsigned short*)x, (const unsigned short*)w,
                (unsigned short*)y, (u64)ldx, m, n, k};
  const bool past = (long)n * k >= PAST_CACHES;
  const int cols = glu ? n / 2 : n, tile = columns(m, cols, k, glu);
  const dim3 grid((cols + tile - 1) / tile);
  const int Q = (k / KC + NW - 1) / NW;    // chunks of a wave
#define GO(NT, U, KS, GLU)                                                     \
  do {                                                                         \
    if (past)                                                                  \
      hipLaunchKernelGGL((linear_rows_kernel<NT, U, KS, GLU, true>), grid,     \
                         dim3(TPB), 0, stream, A);                             \
    else                                                                       \
      hipLaunchKernelGGL((linear_rows_kernel<NT, U, KS, GLU, false>), grid,    \
                         dim3(TPB), 0, stream, A);                             \
  } while (0)
  // Two chunks of a wave in flight where it has an even number and few columns,
  // and both where it has two: a third chunk of two would come twice (8 columns,
  // 1 row, 32000 x 2560 33.1 us with two, 27.3 with one; 32000 x 4096 39.9, 44.8;
  // 32 columns, 3 rows, 6144 x 2048 7.6, 8.1; 32000 x 4096 52, 51).  A gate's two
  // tiles are enough (16384 x 2048, 4 rows 14.2, 13.2).
  if (tile == 8) {
    if (glu) {
      if (Q % 2 == 0) GO(2, 2, 2, true);
      else GO(2, 1, 2, true);
    } else {
      if (Q % 2 == 0) GO(1, 2, 2, false);
      else GO(1, 1, 2, false);
    }
  } else if (glu) {
    GO(2, 1, 1, true);
  } else if (tile == 16) {
    if (Q == 2) GO(1, 2, 1, false);
    else GO(1, 1, 1, false);
  } else if (tile == 32) {
    if (Q == 2) GO(2, 2, 1, false);
    else GO(2, 1, 1, false);
  } else if (tile == 48) {
    GO(3, 1, 1, false);
  } else {
    GO(4, 1, 1, false);
  }
#undef GO
  return hipGetLastError();
}
