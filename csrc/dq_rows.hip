// K3c/K4c — W4A16 / W8A16 product for a few to a hundred rows of x:
// y[m, n] = x[m, k] · dequant(W)[n, k]^T (+ bias) (+ residual).
//
// Between the GEMV (m <= 4) and the large product the packed weights are
// still most of the traffic, so they are read once, straight into
// registers, and turned into matrix-core operands there: int4 as the exact
// bf16 numbers 128 + c, int8 as c.  Scale and zero are applied per group to
// the fp32 result:  sum s (c - z) x = s (sum c x - z sum x), the second sum
// from one more product, with ones.
//
// A wave computes MT x 16 rows by NT x 16 columns over a share of k.  Its
// lanes read 16 bytes of a packed row at a time (a chunk of KC values of k
// is split over the four lane groups, x is read in the same order), the next
// chunk's weights are on their way during this one's products, and no
// barrier is needed until the waves of a workgroup, which share k, add
// their results in LDS.  Where that does not fill the chip, k is also split
// over workgroups; their fp32 sums meet in dq_rows_sum.
//
// What a decode layer has around its products rides along: the root mean
// square of a row of x is the diagonal of x xT, one more product a chunk,
// and scales the sums; silu(gate) * up; bias and residual.
//
// us a call, before (16-column GEMV tiles up to 16 rows, 128 x 128 tiles
// above) and now, of what is not dq_wide's or dq_short's:
//                       8 rows       24 rows       48 rows
//   n 4096, k 14336   45.0 -> 17.4
//   n 2048, k 8192    25.5 -> 12.0  203 -> 14.1   203 -> 16.6   (8 bits,
//   n 16384, k 2048                  57 -> 15.1    58 -> 18.2   group 64)
#include "dq_frag.h"

namespace {

__device__ __forceinline__ float epilogue(const DqArgs& A, float v, int row,
                                          int col) {
  if (A.bias != nullptr) v += bf16_bits_to_f32(A.bias[col]);
  if (A.resid != nullptr)
    v += bf16_bits_to_f32(A.resid[(u64)row * A.n + col]);
  return v;
}

// SCALED: whole sums of rows of x times A.row_scale
template <int BITS, int MT, int NT, int NW, int KC, DqMode MODE, bool SCALED>
__global__ __launch_bounds__(NW * 64) void dq_rows_kernel(DqArgs A) {
  constexpr int TPB = NW * 64;
  constexpr int J = KC / 32;                 // products a chunk
  constexpr int WD = J * BITS / 4;           // packed dwords a lane, a chunk
  constexpr int BM = MT * 16, BN = NT * 16, LD = BN + 4;
  // first [groups][BN] scales and zeros, then [NW][BM][LD] results
  extern __shared__ __attribute__((aligned(16))) float red[];
  u32* meta = (u32*)red;
  const int lane = threadIdx.x & 63, l15 = lane & 15, l4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // this workgroup's rows, from row0 of x (or slot) on
  int row0 = blockIdx.z * BM, rows = A.m - row0, expert = 0;
  if (MODE != DENSE && A.tiles != nullptr) {
    expert = A.tiles[3 * blockIdx.z];
    if (expert < 0) return;
    row0 = A.tiles[3 * blockIdx.z + 1];
    rows = A.tiles[3 * blockIdx.z + 2];
  }
  const bool rms = MODE != SLOTS && A.rms_eps >= 0.f;
  // columns; GLU: the first half of the 16s is gate, the second up
  constexpr int HT = MODE == GLU ? NT / 2 : NT;
  const int n0 = blockIdx.x * (HT * 16), half = A.n / 2;
  auto column = [&](int c) {               // of this workgroup -> of W
    if (MODE == GLU && c >= HT * 16)
      return half + min(n0 + c - HT * 16, half - 1);
    return min(n0 + c, (MODE == GLU ? half : A.n) - 1);
  };
  const int C = A.k / KC;
  // this wave's chunks: workgroups, then waves, share them evenly
  const int u = blockIdx.y * NW + wave, U = gridDim.y * NW;
  const int c0 = (int)((long)C * u / U), c1 = (int)((long)C * (u + 1) / U);
  const int G = A.k / A.g, zw = (G + 32 / BITS - 1) / (32 / BITS);
  const u64 first = (u64)expert * A.n;     // the expert's rows of W

  // one word a column and group of this workgroup: scale (bf16) above,
  // zero bias below.  Read from memory once; per chunk, its lines of 2-byte
  // scales would be most of the traffic.
  const int w0 = (int)((long)C * blockIdx.y * NW / U);
  const int w1 = (int)((long)C * (blockIdx.y + 1) * NW / U);
  const int g0 = w0 * KC / A.g, ng = w1 > w0 ? (w1 - 1) * KC / A.g - g0 + 1 : 0;
  for (int i = threadIdx.x; i < BN * ng; i += TPB) {
    const int col = i / ng, gi = g0 + i % ng;
    const u64 r = first + column(col);
    const u32 z = A.zeros[r * zw + gi / (32 / BITS)];
    meta[(gi - g0) * BN + col] =
        (u32)A.scales[r * G + gi] << 16 |
        (BITS == 4 ? unpack4(z, gi & 7) + 128u : unpack8(z, gi & 3));
  }
  const char* wr[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const u64 r = first + column(t * 16 + l15);
    wr[t] = A.w + r * (A.k * BITS / 8) + l4 * (WD * 4);
  }
  u32 xo[MT];                                // byte offsets into x
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    int r = row0 + min(t * 16 + l15, rows - 1);
    if (MODE != DENSE && A.src != nullptr) r = A.src[r];
    xo[t] = ((u32)r * A.k + l4 * (KC / 4)) * 2;
  }

  const s16x8 ones = bf16_ones();
  f32x4 acc[MT][NT] = {};
  f32x4 sq[MT] = {};                         // x xT: its diagonal
  // WR chunks of weights and XR of x are on their way
  constexpr int WR = MT == 1 ? 4 : 2, XR = MT <= 2 ? 2 : 1;
  u32 wq[WR][NT][WD];
  s16x8 xq[XR][MT][J];
  auto fetch_w = [&](int c, u32 (&w)[NT][WD]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const u32* p = (const u32*)(wr[t] + (u64)c * (KC * BITS / 8));
      if constexpr (WD >= 4) {
#pragma unroll
        for (int i = 0; i < WD / 4; ++i) {
          const u32x4 v = __builtin_nontemporal_load((const u32x4*)p + i);
#pragma unroll
          for (int e = 0; e < 4; ++e) w[t][i * 4 + e] = v[e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < WD; ++e) w[t][e] = p[e];
      }
    }
  };
  auto fetch_x = [&](int c, s16x8 (&x)[MT][J]) {
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int t = 0; t < MT; ++t)
        x[t][j] = *(const s16x8*)((const char*)A.x + xo[t] +
                                  (u32)(c * KC + j * 8) * 2);
  };
  auto multiply = [&](int c, const u32 (&w)[NT][WD], const s16x8 (&x)[MT][J]) {
    const u32* mt = meta + (c * KC / A.g - g0) * BN + l15;
    f32x4 xs[MT] = {};
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int t = 0; t < MT; ++t)
        xs[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[t][j], ones, xs[t],
                                                        0, 0, 0);
    if (rms)
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          sq[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[t][j], x[t][j],
                                                          sq[t], 0, 0, 0);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      f32x4 a[MT] = {};
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const s16x8 b = codes8<BITS>(&w[nt][j * BITS / 4]);
#pragma unroll
        for (int t = 0; t < MT; ++t)
          a[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[t][j], b, a[t], 0,
                                                         0, 0);
      }
      const u32 e = mt[nt * 16];
      const float s = __builtin_bit_cast(float, e & 0xFFFF0000u);
      const float sz = s * (float)(e & 0xFFu);
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[t][nt][i] = fmaf(-sz, xs[t][i], fmaf(s, a[t][i], acc[t][nt][i]));
    }
  };
#pragma unroll
  for (int i = 0; i < WR; ++i) {
    if (c0 + i < c1) fetch_w(c0 + i, wq[i]);
    if (i < XR && XR > 1 && c0 + i < c1) fetch_x(c0 + i, xq[i]);
  }
  __syncthreads();                           // meta is there
  for (int c = c0; c < c1; c += WR) {
#pragma unroll
    for (int i = 0; i < WR; ++i) {
      if (c + i >= c1) break;
      if constexpr (XR == 1) fetch_x(c + i, xq[0]);
      multiply(c + i, wq[i], xq[i % XR]);
      if (c + i + WR < c1) fetch_w(c + i + WR, wq[i]);
      if (XR > 1 && c + i + XR < c1) fetch_x(c + i + XR, xq[i % XR]);
    }
  }

  // ---- the waves' shares of k ----
  __syncthreads();                           // meta is read
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[((u32)wave * BM + t * 16 + l4 * 4 + r) * LD + nt * 16 + l15] =
            acc[t][nt][r];
  float* rs = red + NW * BM * LD;            // [BM], after [NW][BM]
  if (SCALED && threadIdx.x < BM)
    rs[threadIdx.x] = A.row_scale[row0 + min((int)threadIdx.x, rows - 1)];
  if (rms) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (l15 == l4 * 4 + r) rs[BM + wave * BM + t * 16 + l15] = sq[t][r];
  }
  __syncthreads();
  if (rms) {
    if (threadIdx.x < BM) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) v += rs[BM + w * BM + threadIdx.x];
      rs[threadIdx.x] = rsqrtf(v / (float)A.k + A.rms_eps);
    }
    __syncthreads();
  }
  const int nout = MODE == GLU ? half : A.n;
  const bool wide = nout % 4 == 0;
  for (int id = threadIdx.x; id < BM * HT * 4; id += TPB) {
    const int row = id / (HT * 4), c4 = id % (HT * 4) * 4;
    const int gr = row0 + row, gc = n0 + c4;
    if (row >= rows || gc >= nout) continue;
    auto sum = [&](int c) {
      f32x4 v = *(const f32x4*)(red + (u32)row * LD + c);
#pragma unroll
      for (int w = 1; w < NW; ++w)
        v += *(const f32x4*)(red + ((u32)w * BM + row) * LD + c);
      return v;
    };
    f32x4 v = sum(c4);
    const float scale = SCALED || rms ? rs[row] : 1.f;
    if constexpr (MODE == GLU) {
      const f32x4 up = sum(HT * 16 + c4);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = silu_mul_f(v[e] * scale, up[e] * scale);
    } else if (SCALED || rms) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= scale;
    }
    if (MODE == SLOTS || (MODE == DENSE && gridDim.y > 1)) {
      float* p = (MODE == SLOTS ? A.y32 : A.part + (u64)blockIdx.y * A.m * nout)
                 + (u64)gr * nout + gc;
      if (wide) {
        *(f32x4*)p = v;
      } else {
        for (int e = 0; e < 4 && gc + e < nout; ++e) p[e] = v[e];
      }
      continue;
    }
    unsigned short* p = A.y + (u64)gr * nout + gc;
    if constexpr (MODE == DENSE) {
      for (int e = 0; e < 4; ++e)
        if (gc + e < nout) v[e] = epilogue(A, v[e], gr, gc + e);
    }
    if (wide) {
      *(u64*)p = pack_bf16x2(v[0], v[1]) | (u64)pack_bf16x2(v[2], v[3]) << 32;
    } else {
      for (int e = 0; e < 4 && gc + e < nout; ++e)
        p[e] = (unsigned short)f32_to_bf16_bits_rne(v[e]);
    }
  }
}

// y = sum of the splits' parts (+ bias) (+ residual); GLU: silu(gate) * up of
// the sums, y half as wide.  Bound by the launch and one latency: all parts on
// their way at once, no division for a place (48 x 4096: 5.1 us with a grid over
// all elements and parts four by four, 4.8 so).
template <bool GLU, bool SCALED>
__global__ __launch_bounds__(256) void dq_rows_sum(DqArgs A) {
  const u64 part = (u64)A.m * A.n;
  const int nout = GLU ? A.n / 2 : A.n;
  const u64 total = (u64)A.m * nout;
  if (nout % 4 == 0) {                     // a row of workgroups a row
    const int col = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (col >= nout) return;
    for (int row = blockIdx.y; row < A.m; row += gridDim.y) {
      const float* p = A.part + (u64)row * A.n + col;
      float add[4] = {};
      if constexpr (!GLU)
#pragma unroll
        for (int e = 0; e < 4; ++e) add[e] = epilogue(A, 0.f, row, col + e);
      f32x4 v = sum_of_parts(p, part, A.splits);
      if constexpr (SCALED) v *= A.row_scale[row];
      if constexpr (GLU) {
        f32x4 up = sum_of_parts(p + nout, part, A.splits);
        if constexpr (SCALED) up *= A.row_scale[row];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = silu_mul_f(v[e], up[e]);
      } else if (A.bias != nullptr || A.resid != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += add[e];
      }
      *(u64*)(A.y + (u64)row * nout + col) =
          pack_bf16x2(v[0], v[1]) | (u64)pack_bf16x2(v[2], v[3]) << 32;
    }
    return;
  }
  for (u64 id = (u64)blockIdx.x * 256 + threadIdx.x; id < total;
       id += (u64)gridDim.x * 256) {
    const int row = id / nout, col = id % nout;
    float v = 0.f, up = 0.f;
    for (int s = 0; s < A.splits; ++s) {
      v += A.part[s * part + (u64)row * A.n + col];
      if (GLU) up += A.part[s * part + (u64)row * A.n + nout + col];
    }
    if constexpr (SCALED) {
      v *= A.row_scale[row];
      up *= A.row_scale[row];
    }
    A.y[id] = (unsigned short)f32_to_bf16_bits_rne(
        GLU ? silu_mul_f(v, up) : epilogue(A, v, row, col));
  }
}

// A whole row of the result a workgroup, and what DqRowEnd says of it: the sum of
// parts, the residual and the norm in one launch.  V pieces of four columns a
// thread, B parts of them on their way at once.  Bound as dq_rows_sum by launch
// and latency: 77 rows of 2048 with the norm 4.0 us (dq_rows_sum 3.9, the norm
// alone 3.2); 48 rows of 4096, six parts, 4.7 us (dq_rows_sum 4.8, and the norm
// of its rows 5.0, or in the next product the squares of every workgroup's rows,
// n 6144, k 4096 22 us where the product without is 10.5).
constexpr int ROW_TPB = 512;

template <int V, int B, bool NORM>
__global__ __launch_bounds__(ROW_TPB) void dq_rows_sum_row(DqArgs A) {
  typedef u32 u32x2 __attribute__((ext_vector_type(2)));
  const u64 part = (u64)A.m * A.n;
  const int n4 = A.n / 4, tid = threadIdx.x;
  const u64 at = (u64)blockIdx.x * A.n;
  auto four = [](const u32x2 t) {
    float a, b, c, d;
    bf16x2_to_f32(t[0], a, b);
    bf16x2_to_f32(t[1], c, d);
    return f32x4{a, b, c, d};
  };
  const float scale = A.row_scale != nullptr ? A.row_scale[blockIdx.x] : 1.f;
  const unsigned short* resid = NORM ? A.end.to : A.resid;
  u32x2 add[V] = {}, wv[V];
  f32x4 v[V] = {}, bias[V] = {};
#pragma unroll
  for (int i = 0; i < V; ++i) {
    // past the end the last piece again, not counted and not stored
    const int c = min(tid + i * ROW_TPB, n4 - 1);
    if (resid != nullptr) add[i] = ((const u32x2*)(resid + at))[c];
    if (NORM) wv[i] = ((const u32x2*)A.end.w)[c];
    if (A.bias != nullptr) bias[i] = four(((const u32x2*)A.bias)[c]);
  }
  for (int s0 = 0; s0 < A.splits; s0 += B) {
    f32x4 t[B][V];
#pragma unroll
    for (int s = 0; s < B; ++s)
#pragma unroll
      for (int i = 0; i < V; ++i)
        t[s][i] = ((const f32x4*)(A.part + at + min(s0 + s, A.splits - 1) * part))
            [min(tid + i * ROW_TPB, n4 - 1)];
#pragma unroll
    for (int s = 0; s < B; ++s)
#pragma unroll
      for (int i = 0; i < V; ++i)
        if (s0 + s < A.splits) v[i] += t[s][i];
  }
  __shared__ float red[ROW_TPB / LFMQ_WAVE];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = tid + i * ROW_TPB;
    f32x4 r = v[i] * scale + bias[i];
    if (!NORM) r += four(add[i]);
    const u32x2 out = {pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3])};
    v[i] = four(out);                      // the result as it is stored
    if (NORM) v[i] += four(add[i]);
    if (c < n4) {
      if (!NORM) ((u32x2*)(A.y + at))[c] = out;
#pragma unroll
      for (int e = 0; e < 4; ++e) ss = fmaf(v[i][e], v[i][e], ss);
    }
  }
  ss = wave_reduce_sum_dpp(ss);
  if (tid % LFMQ_WAVE == 0) red[tid / LFMQ_WAVE] = ss;
  __syncthreads();
  ss = 0.f;
#pragma unroll
  for (int i = 0; i < ROW_TPB / LFMQ_WAVE; ++i) ss += red[i];
  const float inv = rsqrtf(ss / (float)A.n + A.end.eps);
  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int c = tid + i * ROW_TPB;
      if (c >= n4) break;
      const f32x4 w = four(wv[i]);
      ((u32x2*)(A.y + at))[c] =
          u32x2{pack_bf16x2(v[i][0], v[i][1]), pack_bf16x2(v[i][2], v[i][3])};
      ((u32x2*)(A.end.normed + at))[c] =
          u32x2{pack_bf16x2(v[i][0] * inv * w[0], v[i][1] * inv * w[1]),
                pack_bf16x2(v[i][2] * inv * w[2], v[i][3] * inv * w[3])};
    }
  } else if (tid == 0) {
    A.end.scale[blockIdx.x] = inv;
  }
}

template <bool NORM>
void sum_row(const DqArgs& A, hipStream_t stream) {
#define GO(V, B)                                                          \
  hipLaunchKernelGGL((dq_rows_sum_row<V, B, NORM>), dim3(A.m), dim3(ROW_TPB), \
                     0, stream, A)
  const int v = (int)ceil_div_u32(A.n, 4 * ROW_TPB);
  if (v <= 1) {
    if (A.splits <= 4) GO(1, 4);
    else GO(1, 8);
  } else if (v == 2) {
    if (A.splits <= 4) GO(2, 4);
    else GO(2, 8);
  } else if (v <= 4) {
    GO(4, 4);
  } else {
    GO(8, 2);
  }
#undef GO
}

void sum_parts(const DqArgs& A, bool glu, hipStream_t stream) {
  if (A.end.normed != nullptr) return sum_row<true>(A, stream);
  if (A.end.scale != nullptr) return sum_row<false>(A, stream);
  const int nout = glu ? A.n / 2 : A.n;
  const dim3 grid =
      nout % 4 == 0
          ? dim3(ceil_div_u32(nout, 1024), min(A.m, 65535))
          : dim3((u32)min(((u64)A.m * nout + 255) / 256, (u64)1024));
  const bool scaled = A.row_scale != nullptr;
  const auto kernel = glu ? (scaled ? dq_rows_sum<true, true>
                                    : dq_rows_sum<true, false>)
                          : (scaled ? dq_rows_sum<false, true>
                                    : dq_rows_sum<false, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, A);
}

int chunk_of(int g) { return g % 128 == 0 ? 128 : (g % 64 == 0 ? 64 : 32); }

// scales and zeros of a workgroup: its share of the chunks, which may begin
// and end inside a group
size_t meta_bytes(int k, int g, int splits, int nt) {
  const int kc = chunk_of(g), chunks = (k / kc + splits - 1) / splits + 1;
  return ((size_t)chunks * kc / g + 2) * nt * 16 * 4;
}

template <int BITS, int MT, int NT, int NW, int KC, DqMode MODE = DENSE,
          bool SCALED = false>
hipError_t go(const DqArgs& A, int tiles, hipStream_t stream) {
  if constexpr (!SCALED && MT > 1 && MODE != SLOTS)
    if (A.row_scale != nullptr && A.splits == 1)
      return go<BITS, MT, NT, NW, KC, MODE, true>(A, tiles, stream);
  const size_t sums =
      ((size_t)NW * MT * 16 * (NT * 16 + 4) + (NW + 1) * MT * 16) * 4;
  const size_t lds = max(sums, meta_bytes(A.k, A.g, A.splits, NT));
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  static size_t set = 64 * 1024;
  if (lds > set) {
    LFMQ_CHECK_HIP(hipFuncSetAttribute(
        (const void*)dq_rows_kernel<BITS, MT, NT, NW, KC, MODE, SCALED>,
        hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    set = 160 * 1024;
  }
  const int cols = MODE == GLU ? NT * 8 : NT * 16;
  const dim3 grid(ceil_div_u32(MODE == GLU ? A.n / 2 : A.n, cols), A.splits,
                  tiles);
  hipLaunchKernelGGL((dq_rows_kernel<BITS, MT, NT, NW, KC, MODE, SCALED>), grid, dim3(NW * 64),
                     lds, stream, A);
  if (A.splits > 1) sum_parts(A, false, stream);
  return hipGetLastError();
}

// rows and columns (in 16s) of a wave, waves of a workgroup; whole: they
// take all of k, else it is also split over workgroups
struct Tile {
  int mt, nt, nw;
  bool whole;
};

// fused: norm or gate, which need whole sums.  us per call, whole / split and
// summed by a second launch (4 bits but for the last):
//   n 6144, k 4096        8 rows  9.4 / 10.2    24 rows 13.1 / 14.3
//   n 4096, k 4096                8.0 /  9.0            11.6 / 12.0
//   n 4096, k 14336              17.4 / 17.9  16 rows   21.8 / 19.0
//   n 2048, k 8192               10.9 /  9.7            18.3 / 12.2
//   n 3072, k 2048                5.6 /  7.5             7.4 / 10.2
//   n 2048, k 2048 (8 bits)       6.5 /  7.5             8.3 /  9.8
// 48 rows: n 3072, k 2048 10.0 / 11.9, n 4096, k 4096 18.2 / 14.5; n 16384,
// k 2048 four or eight waves 17.8 / 14.9.
Tile tile_of(int m, int n, int k, int g, bool glu, bool fused) {
  const int mt = m <= 16 ? 1 : (m <= 32 ? 2 : 3);
  if (g % 64 != 0) return {mt, mt == 1 ? 2 : 4, 4, fused};
  const bool few = n < 6144 && !glu;         // columns: tiles of 16
  if (mt == 1) {
    if (!few) return {1, 2, n >= 16384 ? 4 : 8, true};
    if (fused || (n >= 2048 && (k <= 4096 || (n >= 4096 && m <= 8))))
      return {1, 1, 8, true};
    return {1, 2, 4, false};
  }
  if (mt == 2) {
    if (few && (fused || (n >= 2048 && k <= 4096))) return {2, 1, 8, true};
    if (!few && !glu && n < 16384 && (fused || k <= 4096))
      return {2, 2, 4, true};
    return {2, 4, 4, fused};
  }
  if (few && (fused || (n >= 2048 && k <= 2048))) return {3, 1, 8, true};
  if (glu || n >= 16384) return {3, 4, 8, true};
  if (fused) return {3, 2, 8, true};
  return {3, 4, 4, false};
}

template <int BITS, int KC>
hipError_t go_tile(const DqArgs& A, bool glu, hipStream_t stream) {
  const Tile t = tile_of(A.m, A.n, A.k, A.g, glu, glu || A.rms_eps >= 0.f);
  const int tiles = ceil_div_u32(A.m, t.mt * 16);
#define V(MT, NT, NW)                              \
  if (t.mt == MT && t.nt == NT && t.nw == NW) \
    return go<BITS, MT, NT, NW, KC>(A, tiles, stream)
#define VG(MT, NT, NW)                                                 \
  if (t.mt == MT && t.nt == NT && t.nw == NW)                          \
    return glu ? go<BITS, MT, NT, NW, KC, GLU>(A, tiles, stream)       \
               : go<BITS, MT, NT, NW, KC>(A, tiles, stream)
  VG(1, 2, 4);
  VG(2, 4, 4);
  if constexpr (KC == 32) {
    VG(3, 4, 4);
  } else {
    V(3, 4, 4);
    VG(1, 2, 8);
    V(1, 1, 8);
    V(2, 1, 8);
    V(2, 2, 4);
    V(3, 1, 8);
    V(3, 2, 8);
    VG(3, 4, 8);
  }
#undef V
#undef VG
  return hipErrorInvalidValue;
}

}  // namespace

// false: the shape belongs to another kernel.  fused: norm or gate
bool lfmq_dq_rows_ok(int m, int n, int k, int g, bool fused) {
  if (g % 32 || g > k || k % g || (u64)m * k * 2 >= 1ull << 32) return false;
  // whole sums: scales and zeros of all groups in LDS
  return !fused || (m <= 48 && meta_bytes(k, g, 1, 4) <= 96 * 1024);
}

// workgroups that share k
int lfmq_dq_rows_splits(int m, int n, int k, int g) {
  const Tile t = tile_of(m, n, k, g, false, false);
  if (t.whole && meta_bytes(k, g, 1, t.nt) <= 64 * 1024) return 1;
  const int wgs = max(1, (int)(ceil_div_u32(n, t.nt * 16) *
                               ceil_div_u32(m, t.mt * 16)));
  const int C = k / chunk_of(g);
  // 256 workgroups, or 512 where a wave keeps six chunks (us at 8 rows, 2 / 4
  // splits: n 4096, k 4096 9.0 / 9.7, k 14336 18.3 / 17.8)
  int s = max(1, min(256 / wgs, C / (t.nw * 2)));
  if (512 / wgs <= C / (t.nw * 6)) s = max(s, 512 / wgs);
  while (meta_bytes(k, g, s, t.nt) > 64 * 1024) ++s;     // LDS of a workgroup
  return s;
}

// part: splits > 1 only, [splits, m, n] fp32.  rms_eps >= 0: rows of x are
// scaled by 1 / sqrt(mean x^2 + eps) first; glu: y [m, n / 2] = silu(gate)
// up of W = [gate | up].  Both with splits 1.  row_scale: rows of x times it.
// end: with splits only, what lfmq_dq_rows_sum takes.
hipError_t lfmq_dq_rows(const void* qweight, const void* scales,
                        const void* qzeros, const void* x, void* y,
                        const void* bias, const void* resid, void* part,
                        int m, int n, int k, int g, int bits, int splits,
                        float rms_eps, bool glu, hipStream_t stream,
                        const float* row_scale, const DqRowEnd* end) {
  const bool fused = glu || rms_eps >= 0.f;
  if (!lfmq_dq_rows_ok(m, n, k, g, fused) || (fused && splits != 1) ||
      (glu && n % 2))
    return hipErrorInvalidValue;
  if (bits != 4 && bits != 8) return hipErrorInvalidValue;
  const DqArgs A{(const char*)qweight, (const unsigned short*)scales,
                 (const u32*)qzeros, (const unsigned short*)x,
                 (unsigned short*)y, (const unsigned short*)bias,
                 (const unsigned short*)resid, (float*)part, m, n, k, g,
                 splits, nullptr, nullptr, nullptr, rms_eps, row_scale,
                 end != nullptr ? *end : DqRowEnd{}};
  const int kc = chunk_of(g);
  if (bits == 4) {
    if (kc == 128) return go_tile<4, 128>(A, glu, stream);
    if (kc == 64) return go_tile<4, 64>(A, glu, stream);
    return go_tile<4, 32>(A, glu, stream);
  }
  if (kc == 128) return go_tile<8, 128>(A, glu, stream);
  if (kc == 64) return go_tile<8, 64>(A, glu, stream);
  return go_tile<8, 32>(A, glu, stream);
}

bool lfmq_dq_row_end_ok(int n) { return n % 8 == 0 && n <= 32 * ROW_TPB; }

hipError_t lfmq_dq_rows_sum(const void* part, void* y, const void* bias,
                            const void* resid, int m, int n, int splits,
                            bool glu, hipStream_t stream,
                            const float* row_scale, const DqRowEnd* end) {
  DqArgs A{};
  A.part = (float*)part;
  A.y = (unsigned short*)y;
  A.bias = (const unsigned short*)bias;
  A.resid = (const unsigned short*)resid;
  A.m = m;
  A.n = n;
  A.splits = splits;
  A.row_scale = row_scale;
  if (end != nullptr) A.end = *end;
  sum_parts(A, glu, stream);
  return hipGetLastError();
}

// rows of x (or slots) by expert, tiles of up to 16 of them (DqArgs); glu: y
// bf16 [slots, n / 2], else fp32 [slots, n]
hipError_t lfmq_dq_rows_experts(const void* qweight, const void* scales,
                                const void* qzeros, const void* x,
                                const void* src, const void* tiles, void* y,
                                int n_tiles, int n, int k, int g, int bits,
                                bool glu, hipStream_t stream) {
  if (g % 32 || g > k || k % g || (glu && n % 2)) return hipErrorInvalidValue;
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
  const int kc = chunk_of(g);
#define GO(B, KC)                                             \
  return glu ? go<B, 1, 2, 4, KC, GLU>(A, n_tiles, stream)       \
             : go<B, 1, 2, 4, KC, SLOTS>(A, n_tiles, stream)
#define GOB(B)              \
  do {                      \
    if (kc == 128) GO(B, 128); \
    if (kc == 64) GO(B, 64);   \
    GO(B, 32);              \
  } while (0)
  if (bits == 4) GOB(4);
  if (bits == 8) GOB(8);
#undef GOB
#undef GO
  return hipErrorInvalidValue;
}
