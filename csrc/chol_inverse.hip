// K14 — the factor GPTQ propagates errors with: U upper triangular with
// U^T U = H^-1, from one Cholesky factorisation.
//
// With J the reversal of rows (and columns), J H J = L L^T gives U = J L^-1 J:
// neither H^-1 nor a second factorisation is formed.  L^-1 grows beside L:
// the elimination steps that turn J H J into L^T turn the identity into
// L^-1.  Step j, over blocks of 64 (M is the matrix below the diagonal right
// of block column j, and the rows of what was the identity left of it):
//
//   panel   S_i = M_ij D^T (i > j),  S_i = (D M_ji)^T (i < j),  S_j = D^T,
//           D = L_jj^-1; the rows S_i, i <= j, are row j of L^-1: to U
//   update  M_rc -= S_r S_c^T for r > j, c <= r; the first workgroup then
//           factors M_j+1,j+1 and inverts the factor for the next panel
//
// Up to 3072 both are one launch: a tile's workgroup makes the two panels it
// needs itself and reads one copy of M while it writes the other.  Above, three
// products a tile instead of one would cost more than the launch.
//
// Both halves of the work share one square of memory, since column j of L is
// read by its panel only.  Products are fp32 matrix instructions fed from
// global memory (L2): a lane's 16 values of k lie side by side.
//
// Bound by the chain of the diagonal blocks, 15 us a step at n 2048 as clocks within
// count it, 14.2 timed: 4 from the
// end of a launch to the next one's first workgroup, 2.5 until its panel's
// operands are there (other XCDs wrote them), 2 of products, 6.5 of factor and
// inverse; from 8192 on by the traffic of M.  In the factor every wave carries
// the diagonal block's 16 columns, a lane a column, beside 16 rows of its own,
// so that a column is a reciprocal and one instruction a row, and the inverse
// grows beside it (a lane a row in one wave, other waves waiting, then the
// inverse: 10 us).  n 512: 101 us (133 so), 1024 192 (256), 2048 470 (638; 12.7
// ms for factor, inverse and factor from the library), 3072 975 (1170), 4096
// 1615 (1732), 8192 8140 (8250).  The error of U against 64 bits is a third of
// that path's (n 2048: 2.1e-7 of its norm; 2.5e-7 with the factor before).
#include <float.h>

#include <utility>

#include "common.h"

namespace {

constexpr int NB = 64, TPB = 256, LD = NB + 4;

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

struct Diag {
  float a[NB][LD];           // the block; its lower blocks of 16 become L's
  float x[NB][LD];           // L^-T, its upper blocks of 16
  float diag[4][16][20];     // a wave's diagonal block (20: over all banks)
};

// lane J's value of each row of 16 lanes
template <int J>
__device__ __forceinline__ float row_lane(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                         0x150 + J, 0xf, 0xf, true));
}

// v[i] += f * lane J's v[i], one instruction each (the compiler makes a move
// and a sum of it, with waits between).  Lanes of a register may be read two
// instructions after it was written: the wait in front covers what comes before
// a block, and within a block no register is written and read again.
#define LFMQ_ADD(i, f, J)                                       \
  "v_fmac_f32_dpp %" #i ", %" #i ", %" #f " row_newbcast:%" #J \
  " row_mask:0xf bank_mask:0xf\n\t"

template <int J, int N>
__device__ __forceinline__ void add_lane(float* v, float f) {
  if constexpr (N >= 6) {
    asm("s_nop 1\n\t" LFMQ_ADD(0, 6, 7) LFMQ_ADD(1, 6, 7) LFMQ_ADD(2, 6, 7)
            LFMQ_ADD(3, 6, 7) LFMQ_ADD(4, 6, 7) LFMQ_ADD(5, 6, 7)
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]),
          "+v"(v[5])
        : "v"(f), "n"(J));
    add_lane<J, N - 6>(v + 6, f);
  } else if constexpr (N >= 3) {
    asm("s_nop 1\n\t" LFMQ_ADD(0, 3, 4) LFMQ_ADD(1, 3, 4) LFMQ_ADD(2, 3, 4)
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2])
        : "v"(f), "n"(J));
    add_lane<J, N - 3>(v + 3, f);
  } else if constexpr (N == 2) {
    asm("s_nop 1\n\t" LFMQ_ADD(0, 2, 3) LFMQ_ADD(1, 2, 3)
        : "+v"(v[0]), "+v"(v[1])
        : "v"(f), "n"(J));
  } else if constexpr (N == 1) {
    asm("s_nop 1\n\t" LFMQ_ADD(0, 1, 2) : "+v"(v[0]) : "v"(f), "n"(J));
  }
}

// Column J of a panel leaves the columns behind it, without square roots: the
// diagonal block's rows v, and four rows o of another block.  A lane is a
// column; piv is the pivot, then the next one (read four instructions after it
// was written: the chain of a panel runs through it).
template <int J>
__device__ __forceinline__ void column(float (&v)[16], float (&o)[4],
                                       float& piv, int l15) {
  if constexpr (J < 15) {
    float r = __builtin_amdgcn_rcpf(piv);
    r = fmaf(fmaf(-piv, r, 1.f), r, r);
    const float f = l15 > J ? -v[J] * r : 0.f;
    asm("s_nop 1\n\t" LFMQ_ADD(0, 6, 7) LFMQ_ADD(1, 6, 7) LFMQ_ADD(2, 6, 7)
            LFMQ_ADD(3, 6, 7)
        "v_mov_b32_dpp %5, %0 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
            LFMQ_ADD(4, 6, 7)
        : "+v"(v[J + 1]), "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]),
          "=&v"(piv)
        : "v"(f), "n"(J), "n"(J + 1));
    add_lane<J, 14 - J>(v + J + 2, f);
  }
}
template <int... J>
__device__ __forceinline__ void columns(float (&v)[16], float (&o)[4], int l15,
                                        std::integer_sequence<int, J...>) {
  float piv = row_lane<0>(v[0]);
  (column<J>(v, o, piv, l15), ...);
}

// d.a = L L^T; L^-1 to inv [64, 64], upper part zero.  The columns of L act on
// the rows of the identity too, which become L^-T: in panel p a wave has one
// block of 16 rows, of d.a below the diagonal block or of the identity beside
// and above it (below that it is still zero), and everybody the diagonal block.
// A panel's blocks first take what the panels before it leave them.
__device__ __forceinline__ void factor(Diag& d, float* inv, int* info, bool first) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l15 = lane & 15, l4 = lane >> 4;
  bool bad = false;
#pragma unroll 1
  for (int p = 0; p < 4; ++p) {
    __syncthreads();
    const bool below = wave > p;
    float (*rows)[LD] = below ? d.a : d.x;
    f32x4 dg, sd = {0.f, 0.f, 0.f, 0.f}, so = sd;
    float o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      dg[i] = d.a[16 * p + 4 * l4 + i][16 * p + l15];
      o[i] = below ? d.a[16 * wave + 4 * l4 + i][16 * p + l15]
                   : (wave == p && l15 == 4 * l4 + i ? 1.f : 0.f);
    }
    f32x4 va[3], vb[3];
#pragma unroll
    for (int m = 0; m < 3; ++m)
      if (m < p) {
        vb[m] = *(f32x4*)&d.a[16 * p + l15][16 * m + 4 * l4];
        va[m] = *(f32x4*)&rows[16 * wave + l15][16 * m + 4 * l4];
      }
#pragma unroll
    for (int m = 0; m < 3; ++m)
      if (m < p)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sd = mfma(vb[m][i], vb[m][i], sd);
          if (below || m >= wave) so = mfma(va[m][i], vb[m][i], so);
        }
    float v[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[i] -= so[i];
      d.diag[wave][4 * l4 + i][l15] = dg[i] - sd[i];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = d.diag[wave][i][l15];
    columns(v, o, l15, std::make_integer_sequence<int, 16>());
    float piv = v[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) piv = l15 == i ? v[i] : piv;
    // (above, its reciprocal leaves the normal range)
    bad |= !(piv >= FLT_MIN && piv <= 0x1p125f);
    float rs = __builtin_amdgcn_rsqf(piv);
    rs = fmaf(fmaf(-piv * rs, rs, 1.f), 0.5f * rs, rs);
    f32x4 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      out[i] = o[i] * rs;
      rows[16 * wave + 4 * l4 + i][16 * p + l15] = out[i];
    }
    *(f32x4*)(inv + (16 * p + l15) * NB + 16 * wave + 4 * l4) =
        below ? f32x4{0.f, 0.f, 0.f, 0.f} : out;
  }
  bad = __any(bad);
  if (tid == 0 && (first || bad)) *info = bad;
}

// tile t of the lower triangle, a row's tiles from the diagonal to the left
__device__ __forceinline__ void tile_of(int t, int& r, int& c) {
  r = (int)((sqrtf(8.f * t + 1.f) - 1.f) * 0.5f);
  while (r * (r + 1) / 2 > t) --r;
  while ((r + 1) * (r + 2) / 2 <= t) ++r;
  c = r - (t - r * (r + 1) / 2);
}

// M = J H J, lower triangle (of H also), identity past n; factors block 0.
// diag: H's diagonal instead of its own, or null
__global__ __launch_bounds__(TPB, 4) void chol_begin_kernel(
    const float* __restrict__ h, const float* __restrict__ diag,
    float* __restrict__ m, float* __restrict__ inv, int* __restrict__ info,
    int n, int np) {
  __shared__ Diag d;
  int r, c;
  tile_of(blockIdx.x, r, c);
  for (int t = threadIdx.x; t < NB * NB; t += TPB) {
    // neighbouring threads: neighbouring i, which H's rows run along
    const int i = r * NB + t % NB, k = c * NB + t / NB;
    const int lo = max(i, k), hi = min(i, k);
    const float* p = i == k && diag != nullptr
                         ? diag + (n - 1 - i)
                         : h + (size_t)(n - 1 - hi) * n + n - 1 - lo;
    const float v = lo < n ? *p : (i == k ? 1.f : 0.f);
    if (r == 0) d.a[t % NB][t / NB] = v;
    else m[(size_t)i * np + k] = v;
  }
  if (blockIdx.x == 0) factor(d, inv, info, true);
}

// 64 values of k of 16 rows, the lane's 16
__device__ __forceinline__ void load_rows(const float* p, f32x4 (&v)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = ((const f32x4*)p)[i];
}

// S_b of step j: rows wave * 16 + l4 * 4 + i, columns t * 16 + l15.  SIDE: where
// b lies from j; each has its loads and products to itself, or the compiler
// waits for the first loads before it issues the rest.
enum Side { LEFT, AT, BELOW };

template <Side SIDE>
__device__ __forceinline__ void panel_of(const float* __restrict__ m,
                                         const float* __restrict__ inv, int b,
                                         int j, int np, f32x4 (&acc)[4]) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int l15 = lane & 15, l4 = lane >> 4, row = (tid >> 6) * 16 + l15;
  if constexpr (SIDE == AT) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc[t][i] = inv[(t * 16 + l15) * NB + (tid >> 6) * 16 + l4 * 4 + i];
  } else {
    f32x4 va[4], vb[4][4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if constexpr (SIDE == BELOW) {
        va[q] = *(const f32x4*)(m + (size_t)(b * NB + row) * np + j * NB +
                                q * 16 + l4 * 4);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          va[q][i] = m[(size_t)(j * NB + q * 16 + l4 * 4 + i) * np + b * NB + row];
      }
    // D is lower triangular: its rows of block t end with block t of k
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int q = 0; q <= t; ++q)
        vb[t][q] = *(const f32x4*)(inv + (t * 16 + l15) * NB + q * 16 + l4 * 4);
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = q; t < 4; ++t)
          acc[t] = mfma(va[q][i], vb[t][q][i], acc[t]);
  }
}
__device__ __forceinline__ void panel(const float* __restrict__ m,
                                      const float* __restrict__ inv, int b,
                                      int j, int np, f32x4 (&acc)[4]) {
  if (b > j) panel_of<BELOW>(m, inv, b, j, np, acc);
  else if (b < j) panel_of<LEFT>(m, inv, b, j, np, acc);
  else panel_of<AT>(m, inv, b, j, np, acc);
}

// S_b, b <= j: row j of L^-1, to U
__device__ __forceinline__ void to_u(const f32x4 (&acc)[4],
                                     float* __restrict__ u, int b, int j,
                                     int n) {
  const int tid = threadIdx.x, l15 = tid & 15, l4 = tid >> 4 & 3;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = b * NB + (tid >> 6) * 16 + l4 * 4 + i;
      const int at = j * NB + t * 16 + l15;      // element (at, r) of L^-1
      if (at < n && r <= at)
        u[(size_t)(n - 1 - at) * n + n - 1 - r] = acc[t][i];
    }
}

// A step in one launch: a tile's workgroup makes both panels it needs again,
// so everything is read from one copy of M (and D) and written to another.
__global__ __launch_bounds__(TPB, 4) void chol_step_kernel(
    const float* __restrict__ m, float* __restrict__ mn,
    const float* __restrict__ inv, float* __restrict__ invn,
    float* __restrict__ u, int* __restrict__ info, int j, int n, int np) {
  __shared__ Diag d;                       // S_r, S_c; then the next block
  // rows from j on, tile (j + 1, j + 1), whose factor the next step waits for,
  // first
  const int first = (j + 1) * NB < np ? j + 1 : 0;
  u32 id = blockIdx.x + first;
  id = id < gridDim.x ? id : id - gridDim.x;
  int r, c;
  tile_of(id + j * (j + 1) / 2, r, c);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l15 = lane & 15, l4 = lane >> 4;
  f32x4 p[4];
  if (r == j) {
    panel(m, inv, c, j, np, p);
    to_u(p, u, c, j, n);
    return;
  }
  const int row0 = wave / 2 * 32, col0 = wave % 2 * 32;
  const size_t mt = (size_t)(r * NB + row0 + l4 * 4) * np + c * NB + col0 + l15;
  f32x4 old[2][2];                         // at c = j M still holds the panel
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        old[t][v][i] = m[mt + (size_t)(t * 16 + i) * np + v * 16];
  auto keep = [&](float (*s)[LD]) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        s[wave * 16 + l4 * 4 + i][t * 16 + l15] = p[t][i];
  };
  panel_of<BELOW>(m, inv, r, j, np, p);
  keep(d.a);
  if (c != r) {
    panel(m, inv, c, j, np, p);
    keep(d.x);
  }
  __syncthreads();
  const float (*sc)[LD] = c == r ? d.a : d.x;
  f32x4 acc[2][2] = {};                    // summed apart (chol_update_kernel)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f32x4 a[2], b[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      a[t] = *(const f32x4*)&d.a[row0 + t * 16 + l15][l4 * 16 + i * 4];
      b[t] = *(const f32x4*)&sc[col0 + t * 16 + l15][l4 * 16 + i * 4];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 2; ++v)
          acc[t][v] = mfma(a[t][e], b[v][e], acc[t][v]);
  }
  const bool next = r == j + 1 && c == r;
  if (next) __syncthreads();               // the panel is read
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = (c == j ? 0.f : old[t][v][i]) - acc[t][v][i];
        if (next) d.a[row0 + t * 16 + l4 * 4 + i][col0 + v * 16 + l15] = x;
        else mn[mt + (size_t)(t * 16 + i) * np + v * 16] = x;
      }
  if (next) factor(d, invn, info, false);
}

__global__ __launch_bounds__(TPB) void chol_panel_kernel(
    const float* __restrict__ m, const float* __restrict__ inv,
    float* __restrict__ s, float* __restrict__ u, int j, int n, int np) {
  const int b = blockIdx.x, tid = threadIdx.x, l15 = tid & 15, l4 = tid >> 4 & 3;
  f32x4 acc[4];
  panel(m, inv, b, j, np, acc);
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      s[(size_t)(b * NB + (tid >> 6) * 16 + l4 * 4 + i) * NB + t * 16 + l15] =
          acc[t][i];
  if (b <= j) to_u(acc, u, b, j, n);
}

__global__ __launch_bounds__(TPB, 4) void chol_update_kernel(
    float* __restrict__ m, const float* __restrict__ s,
    float* __restrict__ inv, int* __restrict__ info, int j, int np) {
  __shared__ Diag d;
  int r, c;
  tile_of(blockIdx.x + (j + 1) * (j + 2) / 2, r, c);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l15 = lane & 15, l4 = lane >> 4;
  const int row0 = wave / 2 * 32, col0 = wave % 2 * 32;
  f32x4 a[2][4], b[2][4], acc[2][2], old[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    load_rows(s + (size_t)(r * NB + row0 + t * 16 + l15) * NB + l4 * 16, a[t]);
    load_rows(s + (size_t)(c * NB + col0 + t * 16 + l15) * NB + l4 * 16, b[t]);
  }
  float* mt = m + (size_t)(r * NB + row0 + l4 * 4) * np + c * NB + col0 + l15;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // summed apart: rounded once at the size of M, not 16 times
        acc[t][v][i] = 0.f;
        old[t][v][i] = mt[(size_t)(t * 16 + i) * np + v * 16];
      }
#pragma unroll
  for (int i = 0; i < 16; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 2; ++v)
        acc[t][v] = mfma(a[t][i / 4][i % 4], b[v][i / 4][i % 4], acc[t][v]);
  // at c = j M still holds the panel
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 2; ++v)
      acc[t][v] = (c == j ? f32x4{0.f, 0.f, 0.f, 0.f} : old[t][v]) - acc[t][v];
  if (blockIdx.x != 0) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 2; ++v)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          mt[(size_t)(t * 16 + i) * np + v * 16] = acc[t][v][i];
    return;
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)              // block (j + 1, j + 1)
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        d.a[row0 + t * 16 + l4 * 4 + i][col0 + v * 16 + l15] = acc[t][v][i];
  factor(d, inv, info, false);
}

}  // namespace

int lfmq_chol_pad(int n) { return (n + NB - 1) / NB * NB; }

// One launch a step or two: us at n 512 101 / 127, 1024 192 / 251, 2048 470 / 575,
// 2560 720 / 806, 3072 975 / 1043, but 3584 1340 / 1315 and 4096 1790 / 1630,
// where three products a tile are more than the chain.
static bool one_launch(int N) { return N <= 48; }

// floats of scratch memory: M and inverse twice where a step is one launch,
// else M, inverse and panel
long lfmq_chol_scratch(int n) {
  const long np = lfmq_chol_pad(n), N = np / NB;
  return one_launch((int)N) ? 2 * (np * np + NB * NB)
                            : np * np + NB * NB + np * NB;
}

// h [n, n] fp32 (its lower triangle), diag [n] to take its diagonal's place or
// null, u [n, n] zeros, scratch of lfmq_chol_scratch; info: 1 if a pivot was not
// positive.
hipError_t lfmq_chol_inverse(const void* h, const void* diag, void* u,
                             void* scratch, void* info, int n,
                             hipStream_t stream) {
  const int np = lfmq_chol_pad(n), N = np / NB;
  if (n < 1 || N > 32768) return hipErrorInvalidValue;
  const size_t sq = (size_t)np * np;
  float* m = (float*)scratch;
  float* inv = m + sq;
  float* s = inv + NB * NB;                // panel, or the other M and inverse
  hipLaunchKernelGGL(chol_begin_kernel, dim3(N * (N + 1) / 2), dim3(TPB), 0,
                     stream, (const float*)h, (const float*)diag, m, inv,
                     (int*)info, n, np);
  if (one_launch(N)) {
    for (int j = 0; j < N; ++j) {
      float* m1 = j & 1 ? s : m;
      float* m2 = j & 1 ? m : s;
      hipLaunchKernelGGL(chol_step_kernel,
                         dim3(N * (N + 1) / 2 - j * (j + 1) / 2), dim3(TPB), 0,
                         stream, m1, m2, m1 + sq, m2 + sq, (float*)u,
                         (int*)info, j, n, np);
    }
    return hipGetLastError();
  }
  for (int j = 0; j < N; ++j) {
    hipLaunchKernelGGL(chol_panel_kernel, dim3(N), dim3(TPB), 0, stream, m, inv,
                       s, (float*)u, j, n, np);
    if (j + 1 < N)
      hipLaunchKernelGGL(chol_update_kernel,
                         dim3(N * (N + 1) / 2 - (j + 1) * (j + 2) / 2),
                         dim3(TPB), 0, stream, m, s, inv, (int*)info, j, np);
  }
  return hipGetLastError();
}
