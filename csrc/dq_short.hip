// K3g/K4g — W4A16 / W8A16 product for a few tens to a hundred rows: y[m, n] =
// x[m, k] · dequant(W)[n, k]^T (+ bias) (+ residual), or the gated half of a
// fused gate and up projection.
//
// As dq_tile (128 columns a workgroup, four waves side by side), but row tiles
// of every 16 rows, x and the packed weights by way of LDS in as many stages as
// leave room for a second workgroup, and scales and zeros of 32 groups there
// too: a wave waits for what it asked for two to five chunks ago, where dq_tile's
// one chunk was less than the latency.  Bound by the chain of a chunk (weights,
// unpacking, products, sums), which two waves a SIMD do not fill: at 77 rows of n
// 16384, k 2048 (8 bits) loads alone take 13 us, all but the loads 20, both 22.
// us a call, dq_rows or dq_tile and this one:
//                            20 rows      48 rows      77 rows      96 rows
//   n 28672, k 4096, gate  31.2 / 26.1  38.5 / 29.8
//   n 6144, k 4096         13.0 / 12.2  17.6 / 15.0  21.8 / 19.1  23.2 / 21.2
//   n 4096, k 4096         11.0 / 10.5  14.2 / 13.0  18.9 / 15.1  19.8 / 15.9
//   n 4096, k 14336        22.3 / 17.8  24.1 / 20.2  30.1 / 26.6  31.1 / 28.3
//   n 3072, k 2048 (8)      8.0 / 10.0  10.7 / 11.2  15.2 / 12.9  16.7 / 13.6
//   n 2048, k 8192 (8)     13.8 / 13.7  17.0 / 16.4  22.5 / 19.7  24.0 / 20.5
//   n 32000, k 4096 (8)    49.5 / 38.9  43.5 / 36.8  54.3 / 47.9  57.0 / 51.7
#include "dq_short.h"
#include "lds_dma.h"

namespace {

typedef u32 u32x2 __attribute__((ext_vector_type(2)));

constexpr int NW = 4, TPB = NW * LFMQ_WAVE, NT = 2, BN = NW * NT * 16;
constexpr int MG = 32;                   // groups whose scales LDS holds

template <int BITS, int KC, int MT, int D>
struct Lds {
  static constexpr int BM = MT * 16;
  static constexpr int XB = BM * KC * 2, WB = NT * 16 * KC * BITS / 8;
  static constexpr int STAGE = XB + NW * WB;
  static constexpr int META = D * STAGE, SUM = META + MG * BN * 4;
  static constexpr int ALL = SUM + 2 * BM * 4;
  static constexpr int OUT = BM * (BN + 8) * 2;
  static constexpr int BYTES = ALL > OUT ? ALL : OUT;
};

// SCALED: rows of x times A.row_scale, whole sums
template <int BITS, int KC, int MT, int D, DqMode MODE, bool SCALED>
__global__ __launch_bounds__(TPB, 2) void dq_short_kernel(DqArgs A, int mb,
                                                          int step) {
  typedef Lds<BITS, KC, MT, D> L;
  constexpr int BM = L::BM, J = KC / 32, WD = J * BITS / 4;
  constexpr int SL = KC / 8;                     // 16-byte slots a row of x
  constexpr int XL = L::XB / 1024;               // 1 KiB loads of x a stage
  constexpr int NX = (XL + NW - 1) / NW;         // of a wave, at most
  constexpr int NL = L::WB / 1024;               // of a wave's weights
  constexpr int PC = KC * BITS / 128;            // 16-byte pieces a column
  constexpr bool EVEN = XL % NW == 0;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  u32* meta = (u32*)(smem + L::META);            // [groups][BN]
  float* xsum = (float*)(smem + L::SUM);         // [2][BM]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, l4 = lane >> 4;
  const u32 nb = MODE == GLU ? (A.n / 2 + 63) / 64 : (A.n + 127) / 128;
  u32 id = xcd_swizzle(blockIdx.x, gridDim.x);
  const int row0 = (int)(id % mb) * step;
  id /= mb;
  const int nblk = id % nb, sp = id / nb;
  const int rows = min(A.m - row0, step);
  const int C = A.k / KC;
  const int c0 = (int)((long)C * sp / A.splits);
  const int c1 = (int)((long)C * (sp + 1) / A.splits);
  const int G = A.k / A.g, zw = (G + 32 / BITS - 1) / (32 / BITS);
  const int half = A.n / 2, n0 = nblk * (MODE == GLU ? BN / 2 : BN);
  // column c of this workgroup: row of W.  GLU: a wave's first 16 are gate,
  // the others up
  auto column = [&](int c) {
    if (MODE == GLU)
      return (c >> 4 & 1) * half + min(n0 + (c >> 5) * 16 + (c & 15), half - 1);
    return min(n0 + c, A.n - 1);
  };
  // staging (dq_tile): a lane picks the 16 bytes that belong at its place
  const char* xb = (const char*)(A.x + (u64)row0 * A.k);
  constexpr int RS = NW * 64 / SL;
  static_assert(RS % 16 == 0, "the loads of a lane share one swizzle key");
  const int xrow = wave * 64 / SL + lane / SL;
  const u32 pitch = A.k * 2;
  const u32 xslot = ((lane % SL) ^ slot_key16<SL>(xrow)) * 16;
  const u32 last = (u32)(rows - 1) * pitch;
  const u32 wrow = A.k * BITS / 8;
  u32 wo[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int e = i * 64 + lane, c = e / PC;
    int p = e % PC;
    if constexpr (PC >= 4) p ^= slot_key16<PC>(c & 15);
    wo[i] = (u32)column(wave * NT * 16 + c) * wrow + p * 16;
  }
  auto stage = [&](int c, int buf) {
    const char* base = xb + (u64)c * (KC * 2);
    const u32 at = buf * L::STAGE;
#pragma unroll
    for (int i = 0; i < NX; ++i)
      if (EVEN || i * NW + wave < XL)
        load_to_lds(base, min((xrow + i * RS) * pitch, last) + xslot,
                    at + (i * NW + wave) * 1024);
    const char* wb = A.w + (u32)c * (KC * BITS / 8);
#pragma unroll
    for (int i = 0; i < NL; ++i)
      load_to_lds(wb, wo[i], at + L::XB + wave * L::WB + i * 1024);
  };
  // loads of stage c have landed, D - 2 later ones may be on their way
  auto arrived = [&](int c) {
    if (c + D - 2 < c1) {
      if (EVEN || wave < XL % NW) loads_but<(D - 2) * (NX + NL)>();
      else loads_but<(D - 2) * (NX - 1 + NL)>();
    } else {
      loads_but<0>();
    }
  };
  int gm = 0;                                    // first group in LDS
  auto fill = [&](int c) {
    gm = c * KC / A.g;
    const int ng = min(MG, (c1 * KC - 1) / A.g + 1 - gm);
    constexpr int IN = 8;
    for (int i0 = tid; i0 < BN * ng; i0 += IN * TPB) {
      u32 s[IN], z[IN];
#pragma unroll
      for (int j = 0; j < IN; ++j) {
        const int i = min(i0 + j * TPB, BN * ng - 1);
        const int gi = gm + i % ng;
        const u32 r = column(i / ng);
        s[j] = A.scales[(u64)r * G + gi];
        z[j] = A.zeros[(u64)r * zw + gi / (32 / BITS)];
      }
#pragma unroll
      for (int j = 0; j < IN; ++j) {
        const int i = min(i0 + j * TPB, BN * ng - 1);
        const int gi = gm + i % ng;
        meta[i % ng * BN + i / ng] =
            s[j] << 16 | (BITS == 4 ? unpack4(z[j], gi & 7) : unpack8(z[j], gi & 3));
      }
    }
  };

  const s16x8 ones = bf16_ones();
  f32x4 acc[MT][NT] = {};
  float szp[NT] = {};                            // the chunk before's
  auto xs_of = [&](int par, int t) {
    return *(const f32x4*)(xsum + par * BM + t * 16 + l4 * 4);
  };
#pragma unroll
  for (int i = 0; i < D - 1; ++i)
    if (c0 + i < c1) stage(c0 + i, i);
  fill(c0);
  if (tid < BM) xsum[BM + tid] = 0.f;            // no chunk before the first
  int buf = 0;
  for (int c = c0; c < c1; ++c) {
    const int par = (c - c0) & 1;
    const int gi = c * KC / A.g;
    if (gi - gm == MG) {
      __syncthreads();                           // the scales before are read
      fill(c);
      loads_but<0>();
    }
    arrived(c);
    if (c + D - 1 < c1) stage(c + D - 1, buf == 0 ? D - 1 : buf - 1);
    const char* xs = smem + buf * L::STAGE;
    const char* ws = xs + L::XB + wave * L::WB;
    s16x8 b[NT][J], xa[2][J];
    float s[NT], sz[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const u32 m = meta[(gi - gm) * BN + (wave * NT + t) * 16 + l15];
      s[t] = __builtin_bit_cast(float, m & 0xFFFF0000u);
      sz[t] = s[t] * (float)(m & 0xFFFFu);
      u32 w[WD];
      const char* p = ws + (t * 16 + l15) * (PC * 16);
      if constexpr (WD == 2) {
        const u32x2 v = *(const u32x2*)(p + l4 * 8);
        w[0] = v[0];
        w[1] = v[1];
      } else {
#pragma unroll
        for (int i = 0; i < WD / 4; ++i) {
          const u32x4 v = *(const u32x4*)(
              p + (((l4 * (WD / 4) + i) ^ slot_key16<PC < 4 ? 4 : PC>(l15)) << 4));
#pragma unroll
          for (int e = 0; e < 4; ++e) w[i * 4 + e] = v[e];
        }
      }
#pragma unroll
      for (int j = 0; j < J; ++j) b[t][j] = codes8_exact<BITS>(&w[j * BITS / 4]);
    }
    auto load = [&](int row, int j) {
      return *(const s16x8*)(xs + row * (KC * 2) +
                             (((l4 * J + j) ^ slot_key16<SL>(l15)) << 4));
    };
    f32x4 a[2][NT], xp[2];
    auto fold = [&](int t) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[t][nt][r] = fmaf(s[nt], a[t & 1][nt][r],
                               fmaf(-szp[nt], xp[t & 1][r], acc[t][nt][r]));
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) asm volatile("" : "+v"(acc[t][nt]));
    };
#pragma unroll
    for (int j = 0; j < J; ++j) xa[0][j] = load(l15, j);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
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
      __builtin_amdgcn_sched_barrier(0);
    }
    // this wave's share of the chunk's sums
    constexpr int XS = (MT + NW - 1) / NW;
    f32x4 xsm[XS] = {};
#pragma unroll
    for (int i = 0; i < XS; ++i)
      if (MT % NW == 0 || i * NW + wave < MT)
#pragma unroll
        for (int j = 0; j < J; ++j)
          xsm[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              load((i * NW + wave) * 16 + l15, j), ones, xsm[i], 0, 0, 0);
    fold(MT - 1);
    if (l15 == 0) {
#pragma unroll
      for (int i = 0; i < XS; ++i)
        if (MT % NW == 0 || i * NW + wave < MT)
          *(f32x4*)(xsum + par * BM + (i * NW + wave) * 16 + l4 * 4) = xsm[i];
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) szp[t] = sz[t];
    buf = buf == D - 1 ? 0 : buf + 1;
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
  if (MODE == DENSE && A.splits > 1) {
    float* part = A.part + (u64)sp * A.m * A.n;
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
  if constexpr (SCALED) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float scale =
            A.row_scale[row0 + min(t * 16 + l4 * 4 + r, rows - 1)];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[t][nt][r] *= scale;
      }
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
        const int row = t * 16 + l4 * 4 + r;
        float v = MODE == GLU ? silu_mul_f(acc[t][0][r], acc[t][1][r])
                              : acc[t][nt][r] + bias;
        if (MODE == DENSE && A.resid != nullptr && row < rows && n0 + c < A.n)
          v += bf16_bits_to_f32(A.resid[(u64)(row0 + row) * A.n + n0 + c]);
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

// stages: as many as leave room for a second workgroup on the CU
template <int BITS, int KC, int MT>
constexpr int depth() {
  constexpr int room = 80 * 1024 - Lds<BITS, KC, MT, 1>::ALL +
                       Lds<BITS, KC, MT, 1>::STAGE;
  constexpr int d = room / Lds<BITS, KC, MT, 1>::STAGE;
  constexpr int m = 3 * Lds<BITS, KC, MT, 1>::STAGE < 140 * 1024 ? 3 : 2;
  return d < m ? m : (d > 6 ? 6 : d);
}

template <int BITS, int KC, int MT, DqMode MODE, bool SCALED = false>
hipError_t go(const DqArgs& A, int mb, int step, hipStream_t stream) {
  // (17 to 48 rows)
  if (!SCALED && A.row_scale != nullptr && A.splits == 1) {
    if constexpr (MT <= 3) return go<BITS, KC, MT, MODE, true>(A, mb, step, stream);
    return hipErrorInvalidValue;
  }
  constexpr int D = depth<BITS, KC, MT>();
  constexpr int lds = Lds<BITS, KC, MT, D>::BYTES;
  static_assert(lds <= 160 * 1024, "");
  static bool set = false;
  if (!set && lds > 64 * 1024) {
    LFMQ_CHECK_HIP(hipFuncSetAttribute(
        (const void*)dq_short_kernel<BITS, KC, MT, D, MODE, SCALED>,
        hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    set = true;
  }
  const u32 nb = MODE == GLU ? ceil_div_u32(A.n / 2, 64)
                             : ceil_div_u32(A.n, 128);
  hipLaunchKernelGGL((dq_short_kernel<BITS, KC, MT, D, MODE, SCALED>),
                     dim3(mb * nb * A.splits), dim3(TPB), lds, stream, A, mb,
                     step);
  return hipGetLastError();
}

template <int BITS, int KC, DqMode MODE>
hipError_t go_rows(const DqArgs& A, int mb, int step, hipStream_t stream) {
  switch ((step + 15) / 16) {
    case 1:
    case 2: return go<BITS, KC, 2, MODE>(A, mb, step, stream);
    case 3: return go<BITS, KC, 3, MODE>(A, mb, step, stream);
    case 4: return go<BITS, KC, 4, MODE>(A, mb, step, stream);
    case 5: return go<BITS, KC, 5, MODE>(A, mb, step, stream);
    case 6: return go<BITS, KC, 6, MODE>(A, mb, step, stream);
    case 7:
    case 8: return go<BITS, KC, 8, MODE>(A, mb, step, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace

// Row tiles and parts of k by the time these would take: 256 workgroups a
// round, two on a CU 1.56 times the time of one, a chunk 0.2 to 0.8 us and some
// for each 16 rows, and the traffic of the parts.  Fitted to 1200 measured
// plans of 20 to 200 rows, 2048 to 32000 columns (off by 7 % rms; the plan it
// takes is 2.6 % slower than the best of them).
DqShortPlan lfmq_dq_short_plan(int m, int n, int k, int g, int bits, bool glu) {
  const int kc = g % 128 == 0 ? 128 : 64, C = k / kc;
  static const float us[4][2] = {
      {0.22f, 0.19f}, {0.38f, 0.068f}, {0.82f, 0.127f}, {0.34f, 0.081f}};
  const float* t0 = us[(bits == 8 ? 2 : 0) + (kc == 64 ? 1 : 0)];
  const int nb = (int)(glu ? ceil_div_u32(n / 2, 64) : ceil_div_u32(n, 128));
  DqShortPlan best{};
  float least = INFINITY;
  static const int most[] = {32, 48, 64, 80, 96, 128};
  for (int r : most) {
    DqShortPlan p;
    p.mb = (int)ceil_div_u32(m, r);
    p.step = (int)ceil_div_u32(ceil_div_u32(m, p.mb), 16) * 16;
    const int mt = max(2, p.step / 16 == 7 ? 8 : p.step / 16);
    for (int wgs = 256; wgs <= 512; wgs += 256) {
      p.splits = max(1, min(wgs / (p.mb * nb), C / 3));
      const int u = (int)ceil_div_u32(p.mb * nb * p.splits, 256);
      const float rounds = u == 1 ? 1.f : ((u / 2) + (u & 1) * 0.6f) * 1.56f;
      float t = rounds * (ceil_div_u32(C, p.splits) * (t0[0] + t0[1] * mt) +
                          0.32f);
      if (p.splits > 1) t += 1.9e-6f * (float)m * (float)n * p.splits;
      if (t < least) {
        least = t;
        best = p;
      }
    }
  }
  return best;
}

hipError_t lfmq_dq_short(const DqArgs& A, const DqShortPlan& P, int bits,
                         bool glu, hipStream_t stream) {
  if (A.g % 64 || A.k % A.g || A.m < 1 || (glu && A.n % 2) ||
      (u64)A.n * A.k * bits / 8 >= 1ull << 32 || (u64)A.w % 16 ||
      P.splits != A.splits || P.splits < 1 || P.step > 128 ||
      (P.splits > 1 && A.part == nullptr))
    return hipErrorInvalidValue;
  const bool whole = glu && P.splits == 1;
#define GO(B, K)                                              \
  return whole ? go_rows<B, K, GLU>(A, P.mb, P.step, stream)  \
               : go_rows<B, K, DENSE>(A, P.mb, P.step, stream)
  if (bits == 4) {
    if (A.g % 128 == 0) GO(4, 128);
    GO(4, 64);
  }
  if (bits != 8) return hipErrorInvalidValue;
  if (A.g % 128 == 0) GO(8, 128);
  GO(8, 64);
#undef GO
}
