// y[m, n] = x[m, k] W[n, k]^T in bf16 for up to 16 rows (decode steps of the
// models with 16-bit weights), sums in fp32; optionally the gated half of a
// fused gate and up projection, silu(y[:, c]) * y[:, c + n / 2].
//
// Bound by reading W once, and at these sizes by latency: eight waves share k
// in chunks of 128, all chunks of a wave in flight where k <= 2048.  A lane's
// weights come from memory straight into operands of the matrix instruction,
// 64 consecutive bytes of a column; x is read in the same order from the
// caches; the waves' sums meet in LDS, since a split of k over workgroups
// would take a second launch.
//
// A workgroup has NT tiles of 16 / KS columns (gate: a tile and its up).
// KS > 1: narrow outputs and rows to spare.  Row and column i of the tile then
// stand for row and column i % (16 / KS) in share i / (16 / KS) of k; what
// meets in the KS squares on the diagonal is added, the rest is not read.
//
// us at 3 rows, the library's product and this one, weights not cached:
// 6144 x 2048 12.3 / 7.4, 2048 x 2048 8.4 / 4.9, 3392 x 2048 11.8 / 5.8,
// 16384 x 2048 with silu 21.0 / 15.1 (floor 14.2), 32000 x 2048 31 / 24.
#include "common.h"

namespace {

constexpr int KC = 128, NW = 8, TPB = NW * 64;

struct LArgs {
  const unsigned short *x, *w;
  unsigned short* y;
  u64 ldx;
  int m, n, k;
};

template <int NT, int U, int KS, bool GLU>
__global__ __launch_bounds__(TPB) void linear_rows_kernel(LArgs A) {
  constexpr int S = 16 / KS, BN = GLU ? S : NT * S;
  __shared__ f32x4 red[NW][NT][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4, share = l15 / S;
  const int cols = GLU ? A.n / 2 : A.n, n0 = blockIdx.x * BN;
  const unsigned short* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    wp[t] = A.w + l4 * 32 + (u64)A.k *
            (GLU ? min(n0 + l15 % S, cols - 1) + t * cols
                 : min(n0 + t * S + l15 % S, cols - 1));
  const unsigned short* xp =
      A.x + (u64)min(l15 % S, A.m - 1) * A.ldx + l4 * 32;

  f32x4 acc[NT] = {};
  const int C = A.k / KC;                  // chunk c: KS of them, one a share
  for (int c0 = wave; c0 * KS < C; c0 += NW * U) {
    s16x8 b[U][NT][4], a[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = min((c0 + u * NW) * KS + share, C - 1);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          b[u][t][i] = ((const s16x8*)(wp[t] + c * KC))[i];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = min((c0 + u * NW) * KS + share, C - 1);
#pragma unroll
      for (int i = 0; i < 4; ++i) a[u][i] = ((const s16x8*)(xp + c * KC))[i];
    }
    __builtin_amdgcn_sched_barrier(0);     // all loads before the first use
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // past the end the last chunk came again: times zero weights, so that
      // nothing of x (infinities too) counts twice
      const bool live = (c0 + u * NW) * KS + share < C;
      const s16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[u][i] = live ? a[u][i] : zero;
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a[u][i], live ? b[u][t][i] : zero, acc[t], 0, 0, 0);
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
#define GO(NT, U, KS, GLU, COLS)                                           \
  hipLaunchKernelGGL((linear_rows_kernel<NT, U, KS, GLU>),                 \
                     dim3(((GLU ? n / 2 : n) + COLS - 1) / COLS),          \
                     dim3(TPB), 0, stream, A)
  if (glu) {
    if (k <= NW * KC) GO(2, 1, 1, true, 16);
    else GO(2, 2, 1, true, 16);
  } else if (n <= 2048 && k > 2048 && m <= 8) {
    // 256 workgroups instead of 128 (2048 x 8192: 10.6 us, 13.5; 4096 x 14336
    // has 256 either way: 31.4, 25.2)
    GO(1, 2, 2, false, 8);
  } else if (n >= 6144 && k > NW * KC && k <= 2 * NW * KC) {
    // x half as often, enough workgroups (6144 x 2048: 7.4 us, 8.5), all in
    // flight at once (28672 x 4096: 52, 43)
    GO(2, 2, 1, false, 32);
  } else if (k <= NW * KC) {
    GO(1, 1, 1, false, 16);
  } else {
    GO(1, 2, 1, false, 16);
  }
#undef GO
  return hipGetLastError();
}
