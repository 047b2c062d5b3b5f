// K3b/K4b — W4A16 / W8A16 product for prompts: y[m, n] = x[m, k] ·
// dequant(W)[n, k]^T (+ bias).
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
// Bound by the issue of products, unpacking and scaling together: 768
// TFLOP/s at 3001 x 28672 x 4096 (4 bits, groups of 128), where 128 x 128
// tiles of weights unpacked into LDS reached 418.  us a call, before and now:
//                       64 rows      256 rows      3001 rows
//   n 28672, k 4096   107 -> 50.7   178 -> 87.9   1690 -> 918
//   n 4096, k 14336   369 -> 33.1   361 -> 53.7    890 -> 496   (4 bits)
//   n 6144, k 4096    101 -> 25.2   103 -> 34.4    422 -> 230
//   n 16384, k 2048    58 -> 28.3    59 -> 45.9    501 -> 377   (8 bits,
//   n 2048, k 8192    203 -> 24.5   203 -> 32.5    343 -> 233    group 64)
#include "dq_frag.h"
#include "lds_dma.h"

namespace {

constexpr int NW = 4, TPB = NW * LFMQ_WAVE;

struct TArgs {
  const char* w;                 // [n, k * BITS / 8] bytes
  const unsigned short* scales;  // [n, G]
  const u32* zeros;              // [n, zw]
  const unsigned short* x;       // [m, k]
  unsigned short* y;             // [m, n]
  const unsigned short* bias;
  float* part;                   // [splits, m, n], splits > 1
  int m, n, k, g, splits;
};

template <int BITS, int KC>
__global__ __launch_bounds__(TPB, 2) void dq_tile_kernel(TArgs A) {
  constexpr int MT = 8, NT = 2, BM = MT * 16, BN = NW * NT * 16;
  constexpr int J = KC / 32, WD = J * BITS / 4;
  constexpr int SL = KC / 8;                     // 16-byte slots a row
  constexpr int NX = BM * SL / TPB;              // staged slots a thread
  constexpr int XB = BM * KC * 2;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* xsum = (float*)(smem + 2 * XB);         // [2][BM]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4;
  // an XCD's workgroups share columns: rows run fastest
  const u32 mb = (A.m + BM - 1) / BM, nb = (A.n + BN - 1) / BN;
  u32 id = xcd_swizzle(blockIdx.x, gridDim.x);
  const int m0 = (int)(id % mb) * BM;
  id /= mb;
  const int n0 = (int)(id % nb) * BN, sp = (int)(id / nb);
  const int C = A.k / KC;
  const int c0 = (int)((long)C * sp / A.splits);
  const int c1 = (int)((long)C * (sp + 1) / A.splits);
  const int G = A.k / A.g, zw = (G + 32 / BITS - 1) / (32 / BITS);
  auto key = [](int row) { return slot_key<SL>(row); };

  // staging: a wave's load writes 1 KiB of LDS in lane order, so the lane
  // picks the slot that belongs there; rows past m repeat the last one
  u32 xo[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int p = (i * NW + wave) * 64 + lane, row = p / SL;
    xo[i] = ((u32)min(row, A.m - 1 - m0) * A.k +
             ((p % SL) ^ key(row)) * 8) * 2;
  }
  auto stage = [&](int c, int buf) {
    const char* base = (const char*)(A.x + (u64)m0 * A.k + c * KC);
#pragma unroll
    for (int i = 0; i < NX; ++i)
      load_to_lds(base, xo[i], buf * XB + (i * NW + wave) * 1024);
  };
  // weights: rows of this workgroup's columns, within 4 GiB of the first
  const int wrow = A.k * BITS / 8;
  const char* wb = A.w + (u64)n0 * wrow;
  u32 wo[NT], so[NT], zo[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int col = min(n0 + (wave * NT + t) * 16 + l15, A.n - 1);
    wo[t] = (u32)(col - n0) * wrow + l4 * (WD * 4);
    so[t] = (u32)col * G;
    zo[t] = (u32)col * zw;
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
        sq[t][0] = A.scales[so[t] + gi];
        zq[t][0] = A.zeros[zo[t] + gi / (32 / BITS)];
      }
    } else if (next8) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        sq[t] = *(const u32x4*)(A.scales + so[t] + (gi & ~7));
#pragma unroll
        for (int i = 0; i < BITS / 4; ++i)
          zq[t][i] = A.zeros[zo[t] + (gi & ~7) / (32 / BITS) + i];
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
      // kept apart, the stages fit 256 registers (W4: 774 against 731 TFLOP/s
      // at 3001 x 28672 x 4096; W8 spills so: 672 against 687)
      if constexpr (BITS == 4) __builtin_amdgcn_sched_barrier(0);
    }
    // this wave's share of the chunk's sums
    f32x4 xs[MT / NW] = {};
#pragma unroll
    for (int i = 0; i < MT / NW; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j)
        xs[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            load((wave * (MT / NW) + i) * 16 + l15, j), ones, xs[i], 0, 0, 0);
    fold(MT - 1);
    if (l15 == 0) {
#pragma unroll
      for (int i = 0; i < MT / NW; ++i)
        *(f32x4*)(xsum + par * BM + (wave * (MT / NW) + i) * 16 + l4 * 4) =
            xs[i];
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
  if (A.splits > 1) {
    float* part = A.part + (u64)sp * A.m * A.n;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + t * 16 + l4 * 4 + r;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int col = n0 + (wave * NT + nt) * 16 + l15;
          if (row < A.m && col < A.n)
            part[(u64)row * A.n + col] = acc[t][nt][r];
        }
      }
    return;
  }
  // through LDS, so that rows are written in 16-byte pieces
  constexpr int LD = BN + 8;
  unsigned short* out = (unsigned short*)smem;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int c = (wave * NT + nt) * 16 + l15;
    const float bias = A.bias != nullptr && n0 + c < A.n
                           ? bf16_bits_to_f32(A.bias[n0 + c])
                           : 0.f;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        out[(t * 16 + l4 * 4 + r) * LD + c] =
            (unsigned short)f32_to_bf16_bits_rne(acc[t][nt][r] + bias);
  }
  __syncthreads();
  const bool wide = A.n % 8 == 0;
  for (int i = tid; i < BM * BN / 8; i += TPB) {
    const int row = i / (BN / 8), c = i % (BN / 8) * 8;
    const int gr = m0 + row, gc = n0 + c;
    if (gr >= A.m || gc >= A.n) continue;
    unsigned short* p = A.y + (u64)gr * A.n + gc;
    const unsigned short* q = out + row * LD + c;
    if (wide) {
      *(u32x4*)p = *(const u32x4*)q;
    } else {
      for (int e = 0; e < 8 && gc + e < A.n; ++e) p[e] = q[e];
    }
  }
}

template <int BITS, int KC>
hipError_t go(const TArgs& A, hipStream_t stream) {
  // two buffers and the sums; the result, padded, takes a little more
  constexpr size_t bufs = 2 * 128 * KC * 2 + 2 * 128 * 4, out = 128 * 136 * 2;
  constexpr size_t lds = bufs > out ? bufs : out;
  static bool set = false;
  if (!set && lds > 64 * 1024) {
    LFMQ_CHECK_HIP(hipFuncSetAttribute(
        (const void*)dq_tile_kernel<BITS, KC>,
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    set = true;
  }
  const u32 grid = ceil_div_u32(A.m, 128) * ceil_div_u32(A.n, 128) * A.splits;
  hipLaunchKernelGGL((dq_tile_kernel<BITS, KC>), dim3(grid), dim3(TPB), lds,
                     stream, A);
  return hipGetLastError();
}

}  // namespace

bool lfmq_dq_tile_ok(int k, int g) {
  return g % 64 == 0 && g <= k && k % g == 0;
}

int lfmq_dq_tile_splits(int m, int n, int k, int g) {
  const int wgs = (int)(ceil_div_u32(n, 128) * ceil_div_u32(m, 128));
  const int C = k / (g % 128 == 0 ? 128 : 64);
  // 256 workgroups, or 512 where six chunks are left to each (us at 64 rows,
  // 4 bits: n 28672, k 4096 57 / 48, n 6144 21.8 / 23.8, n 4096, k 14336
  // 34 / 31)
  const int s = max(1, min(256 / wgs, C / 4));
  return 512 / wgs <= C / 6 ? max(s, 512 / wgs) : s;
}

hipError_t lfmq_dq_rows_sum(const void* part, void* y, const void* bias,
                            const void* resid, int m, int n, int splits,
                            hipStream_t stream);

hipError_t lfmq_dq_tile(const void* qweight, const void* scales,
                        const void* qzeros, const void* x, void* y,
                        const void* bias, void* part, int m, int n, int k,
                        int g, int bits, int splits, hipStream_t stream) {
  if (!lfmq_dq_tile_ok(k, g)) return hipErrorInvalidValue;
  const TArgs A{(const char*)qweight, (const unsigned short*)scales,
                (const u32*)qzeros, (const unsigned short*)x,
                (unsigned short*)y, (const unsigned short*)bias, (float*)part,
                m, n, k, g, splits};
  hipError_t e;
  if (bits == 4)
    e = g % 128 == 0 ? go<4, 128>(A, stream) : go<4, 64>(A, stream);
  else if (bits == 8)
    e = g % 128 == 0 ? go<8, 128>(A, stream) : go<8, 64>(A, stream);
  else
    return hipErrorInvalidValue;
  if (e != hipSuccess || splits == 1) return e;
  return lfmq_dq_rows_sum(part, y, bias, nullptr, m, n, splits, stream);
}
