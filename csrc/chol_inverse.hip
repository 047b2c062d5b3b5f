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
// Up to 2048 both are one launch: a tile's workgroup makes the two panels it
// needs itself and reads one copy of M while it writes the other.  Above, three
// products a tile instead of one would cost more than the launch.
//
// Both halves of the work share one square of memory, since column j of L is
// read by its panel only.  Products are fp32 matrix instructions fed from
// global memory (L2): a lane's 16 values of k lie side by side.
//
// Bound by the chain of the diagonal blocks (the factor of 64 in panels of 16
// by one wave, inverse by blocks of 16: 15 us with its update, 20 with the
// panels and the launch); from 8192 on by the traffic of M.  n 2048: 0.63 ms
// (two launches a step 0.70), 12.7 for factor, inverse and factor from the
// library; 14336: 50 and 261.  The error of U against 64 bits is a third to a
// half of that path's (n 2048: 1.4e-7, condition 3600: 4.6e-6).
#include <float.h>

#include "common.h"

namespace {

constexpr int NB = 64, TPB = 256, LD = NB + 4;

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

struct Diag {
  float a[NB][LD];   // the block, its lower triangle becomes L
  float x[NB][LD];   // L^-1
};

// d.a: factor and inverse; the inverse to inv [64, 64], upper part zero
__device__ __forceinline__ void factor(Diag& d, float* inv, int* info, bool first) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l15 = lane & 15, l4 = lane >> 4;
  bool bad = false;
  __syncthreads();
#pragma unroll 1
  for (int p = 0; p < 4; ++p) {
    if (wave == 0) {                       // a lane a row, 16 columns
      f32x4 v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = *(f32x4*)&d.a[lane][16 * p + 4 * i];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float piv = lane_value(v[j / 4][j % 4], 16 * p + j);
        bad |= !(piv >= FLT_MIN && piv <= FLT_MAX);
        float rs = __builtin_amdgcn_rsqf(piv);
        rs = fmaf(fmaf(-piv * rs, rs, 1.f), 0.5f * rs, rs);
        const float l = v[j / 4][j % 4] * rs;
        v[j / 4][j % 4] = l;
#pragma unroll
        for (int c = j + 1; c < 16; ++c)
          v[c / 4][c % 4] -= l * lane_value(l, 16 * p + c);
      }
      if (lane >= 16 * p)
#pragma unroll
        for (int i = 0; i < 4; ++i) *(f32x4*)&d.a[lane][16 * p + 4 * i] = v[i];
    }
    __syncthreads();
    int t = 0;
    for (int r = p + 1; r < 4; ++r)
      for (int c = p + 1; c <= r; ++c, ++t) {
        if ((t & 3) != wave) continue;
        const f32x4 va = *(f32x4*)&d.a[16 * r + l15][16 * p + 4 * l4];
        const f32x4 vb = *(f32x4*)&d.a[16 * c + l15][16 * p + 4 * l4];
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = mfma(va[i], vb[i], acc);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          d.a[16 * r + l4 * 4 + i][16 * c + l15] -= acc[i];
      }
    __syncthreads();
  }
  if (tid == 0 && (first || bad)) *info = bad;

  {                                        // a wave a diagonal block of 16
    f32x4 l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      l[i] = *(f32x4*)&d.a[16 * wave + l15][16 * wave + 4 * i];
    const float rd = 1.f / d.a[16 * wave + l15][16 * wave + l15];
    f32x4 x[4];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i / 4][i % 4] = i == l15 ? 1.f : 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const float xk = x[k / 4][k % 4] * lane_value(rd, k);
      x[k / 4][k % 4] = xk;
#pragma unroll
      for (int i = k + 1; i < 16; ++i)
        x[i / 4][i % 4] -= lane_value(l[k / 4][k % 4], i) * xk;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = x[i][0];
      v = l4 == 1 ? x[i][1] : v;
      v = l4 == 2 ? x[i][2] : v;
      v = l4 == 3 ? x[i][3] : v;
      d.x[16 * wave + 4 * i + l4][16 * wave + l15] = v;
    }
  }
#pragma unroll
  for (int dist = 1; dist < 4; ++dist) {   // X_rc = -X_rr sum L_rm X_mc
    __syncthreads();
    const int c = wave, r = c + dist;
    if (r < 4) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      for (int m = c; m < r; ++m) {
        const f32x4 l = *(f32x4*)&d.a[16 * r + l15][16 * m + 4 * l4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc = mfma(l[i], d.x[16 * m + 4 * l4 + i][16 * c + l15], acc);
      }
      const f32x4 xr = *(f32x4*)&d.x[16 * r + l15][16 * r + 4 * l4];
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) o = mfma(xr[i], acc[i], o);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        d.x[16 * r + l4 * 4 + i][16 * c + l15] = -o[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NB * NB / 4; t += TPB) {
    const int r = (t + tid) / (NB / 4), c = (t + tid) % (NB / 4) * 4;
    ((f32x4*)inv)[t + tid] = c / 16 <= r / 16 ? *(f32x4*)&d.x[r][c]
                                              : f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

// tile t of the lower triangle, a row's tiles from the diagonal to the left
__device__ __forceinline__ void tile_of(int t, int& r, int& c) {
  r = (int)((sqrtf(8.f * t + 1.f) - 1.f) * 0.5f);
  while (r * (r + 1) / 2 > t) --r;
  while ((r + 1) * (r + 2) / 2 <= t) ++r;
  c = r - (t - r * (r + 1) / 2);
}

// M = J H J, lower triangle (of H also), identity past n; factors block 0
__global__ __launch_bounds__(TPB, 4) void chol_begin_kernel(
    const float* __restrict__ h, float* __restrict__ m,
    float* __restrict__ inv, int* __restrict__ info, int n, int np) {
  __shared__ Diag d;
  int r, c;
  tile_of(blockIdx.x, r, c);
  for (int t = threadIdx.x; t < NB * NB; t += TPB) {
    // neighbouring threads: neighbouring i, which H's rows run along
    const int i = r * NB + t % NB, k = c * NB + t / NB;
    const int lo = max(i, k), hi = min(i, k);
    const float v = lo < n ? h[(size_t)(n - 1 - hi) * n + n - 1 - lo]
                           : (i == k ? 1.f : 0.f);
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

// S_b of step j: rows wave * 16 + l4 * 4 + i, columns t * 16 + l15
__device__ __forceinline__ void panel(const float* __restrict__ m,
                                      const float* __restrict__ inv, int b,
                                      int j, int np, f32x4 (&acc)[4]) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int l15 = lane & 15, l4 = lane >> 4, row = (tid >> 6) * 16 + l15;
  if (b == j) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc[t][i] = inv[(t * 16 + l15) * NB + (tid >> 6) * 16 + l4 * 4 + i];
  } else {
    f32x4 va[4], vb[4];
    if (b > j) {
      load_rows(m + (size_t)(b * NB + row) * np + j * NB + l4 * 16, va);
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        va[i / 4][i % 4] = m[(size_t)(j * NB + l4 * 16 + i) * np + b * NB + row];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      load_rows(inv + (t * 16 + l15) * NB + l4 * 16, vb);
      acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 16; ++i)
        acc[t] = mfma(va[i / 4][i % 4], vb[i / 4][i % 4], acc[t]);
    }
  }
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
        old[t][v][i] = c == j ? 0.f : m[mt + (size_t)(t * 16 + i) * np + v * 16];
  auto keep = [&](float (*s)[LD]) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        s[wave * 16 + l4 * 4 + i][t * 16 + l15] = p[t][i];
  };
  panel(m, inv, r, j, np, p);
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
        const float x = old[t][v][i] - acc[t][v][i];
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

// One launch a step or two: us at n 512 130 / 156, 1024 256 / 314, 2048 629 / 701,
// but 3072 1427 / 1174, where three products a tile are more than the chain.
static bool one_launch(int N) { return N <= 32; }

// floats of scratch memory: M and inverse twice where a step is one launch,
// else M, inverse and panel
long lfmq_chol_scratch(int n) {
  const long np = lfmq_chol_pad(n), N = np / NB;
  return one_launch((int)N) ? 2 * (np * np + NB * NB)
                            : np * np + NB * NB + np * NB;
}

// h [n, n] fp32 (its lower triangle), u [n, n] zeros, scratch of
// lfmq_chol_scratch; info: 1 if a pivot was not positive.
hipError_t lfmq_chol_inverse(const void* h, void* u, void* scratch, void* info,
                             int n, hipStream_t stream) {
  const int np = lfmq_chol_pad(n), N = np / NB;
  if (n < 1 || N > 32768) return hipErrorInvalidValue;
  const size_t sq = (size_t)np * np;
  float* m = (float*)scratch;
  float* inv = m + sq;
  float* s = inv + NB * NB;                // panel, or the other M and inverse
  hipLaunchKernelGGL(chol_begin_kernel, dim3(N * (N + 1) / 2), dim3(TPB), 0,
                     stream, (const float*)h, m, inv, (int*)info, n, np);
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
