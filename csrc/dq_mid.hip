// K4h — W8A16 product for some tens of rows: y[m, n] = x[m, k] · dequant(W)[n, k]^T
// (+ bias) (+ residual), or the gated half of a fused gate and up projection.
//
// dq_short's workgroup of four waves takes 128 columns and all of k, one chunk
// after the other, each as long as its chain of unpacking, products and sums.  Here
// eight waves share k too: a workgroup has 64 or 128 columns, its waves lie 2 or 4
// side by side and 4 or 2 along k, by groups in turn, and their sums meet in LDS.
// So half as many columns fill the chip, and half or a quarter of the chain is left.
// A code minus its zero is an exact bf16 number, so no sums of x are needed and a
// group's scale is applied once.  x comes a step ahead and the weights two, by way
// of LDS.  Bound by that chain still: at 77 rows of n 16384, k 2048 the loads alone
// are 9 of 16 us.
//
// us a call, dq_short or dq_rows and this one (groups of 64):
//                             20 rows       40 rows       77 rows       96 rows
//   n 16384, k 2048, gate   17.8 / 13.8   18.0 / 15.5   25.6 / 18.6   27.9 / 18.5
//   n 32000, k 2048         25.7 / 24.6   29.8 / 26.0   36.6 / 31.4   36.2 / 31.5
//   n 2048, k 8192                                      20.4 / 17.2   21.7 / 18.4
//   n 12288, k 3072 (128)   21.9 / 17.3   27.2 / 19.1   28.9 / 21.9   26.7 / 23.7
//   n 4096, k 4096 (128)                                19.0 / 16.6   21.4 / 16.9
#include "dq_mid.h"
#include "lds_dma.h"

namespace {

constexpr int NWV = 8, TPB = NWV * 64, NT = 2;   // waves, 16s of columns a wave
constexpr int KS = 64, J = 2;                    // k of a step, products
constexpr int DX = 2;                            // steps of x in LDS
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

// NC: waves side by side
template <int MT, int NC>
struct Lds {
  static constexpr int KW = NWV / NC, BN = NC * NT * 16, BM = MT * 16;
  static constexpr int XB = BM * KS * 2, WB = NT * 16 * KS;  // a k wave's, a wave's
  static constexpr int XS = KW * XB, WS = NWV * WB;          // a step's
  static constexpr int ROOM = 150 * 1024 - DX * XS;
  static constexpr int DW = ROOM / WS >= DX + 2 ? DX + 2 : DX + 1;
  static constexpr int W0 = DX * XS, META = W0 + DW * WS;
  static constexpr int bytes(int groups) {
    const int loop = META + groups * BN * 4, sums = KW * BM * (BN + 4) * 4;
    return loop > sums ? loop : sums;
  }
};

template <int MT, int NC, DqMode MODE>
__global__ __launch_bounds__(TPB, 2) void dq_mid_kernel(DqArgs A, int mb, int step) {
  typedef Lds<MT, NC> L;
  constexpr int KW = L::KW, BN = L::BN, DW = L::DW;
  constexpr int BM = L::BM;
  constexpr int SL = KS / 8;                     // 8 slots of 16 bytes a row
  constexpr int XP = L::XB / 1024, XL = KW * XP, NX = (XL + NWV - 1) / NWV;
  constexpr int NL = L::WB / 1024;               // of a wave's weights
  constexpr int PC = KS / 16;                    // 16-byte pieces a column
  extern __shared__ __attribute__((aligned(16))) char smem[];
  u32* meta = (u32*)(smem + L::META);            // [groups][BN]
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
  const int G = A.k / A.g, zw = (G + 3) / 4;
  // groups of this workgroup; a k wave takes every KW-th of them
  const int g0 = (int)((long)G * sp / A.splits), g1 = (int)((long)G * (sp + 1) / A.splits);
  const int gs = A.g / KS;                       // steps a group
  const int S = (g1 - g0 + KW - 1) / KW * gs;    // steps
  const int half = A.n / 2, n0 = nblk * BO;
  auto column = [&](int c) {
    if (MODE == GLU) return (c >> 4 & 1) * half + min(n0 + (c >> 5) * 16 + (c & 15), half - 1);
    return min(n0 + c, A.n - 1);
  };
  const char* xb = (const char*)(A.x + (u64)row0 * A.k);
  const u32 pitch = A.k * 2, last = (u32)(rows - 1) * pitch, wrow = A.k;
  // x: load i of this wave
  u32 xo[NX];
  int xq[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int e = min(i * NWV + wave, XL - 1), q = e / XP, r = e % XP * 8 + lane / 8;
    xq[i] = q;
    xo[i] = min(r * pitch, last) + ((lane % SL) ^ slot_key16<SL>(r & 15)) * 16;
  }
  u32 wo[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int e = i * 64 + lane, c = e / PC;
    wo[i] = (u32)column(wc * NT * 16 + c) * wrow +
            ((e % PC) ^ slot_key16<PC>(c & 15)) * 16;
  }
  // k of step s for k wave q
  auto kat = [&](int s, int q) {
    const int grp = min(g0 + (s / gs) * KW + q, g1 - 1);
    return grp * A.g + s % gs * KS;
  };
  auto stage_x = [&](int s) {
    const u32 at = s % DX * L::XS;
#pragma unroll
    for (int i = 0; i < NX; ++i)
      load_to_lds(xb + kat(s, xq[i]) * 2, xo[i], at + min(i * NWV + wave, XL - 1) * 1024);
  };
  auto stage_w = [&](int s) {
    const u32 at = L::W0 + s % DW * L::WS + wave * L::WB;
    const char* wb = A.w + (u32)kat(s, kw);
#pragma unroll
    for (int i = 0; i < NL; ++i) load_to_lds(wb, wo[i], at + i * 1024);
  };
#pragma unroll
  for (int i = 0; i < DW - 1; ++i) {
    if (i < DX - 1 && i < S) stage_x(i);
    if (i < S) stage_w(i);
  }
  {
    const int ng = g1 - g0;
    constexpr int IN = 8;
    for (int i0 = tid; i0 < BN * ng; i0 += IN * TPB) {
      u32 s[IN], z[IN];
#pragma unroll
      for (int j = 0; j < IN; ++j) {
        const int i = min(i0 + j * TPB, BN * ng - 1);
        const int gi = g0 + i % ng;
        const u32 r = column(i / ng);
        s[j] = A.scales[(u64)r * G + gi];
        z[j] = A.zeros[(u64)r * zw + gi / 4];
      }
#pragma unroll
      for (int j = 0; j < IN; ++j) {
        const int i = min(i0 + j * TPB, BN * ng - 1);
        const int gi = g0 + i % ng;
        meta[i % ng * BN + i / ng] = s[j] << 16 | unpack8(z[j], gi & 3);
      }
    }
  }
  f32x4 acc[MT][NT] = {}, a[MT][NT] = {};
  float sc[NT] = {}, z[NT] = {};
  for (int s = 0; s < S; ++s) {
    const int si = s % gs, gl = (s / gs) * KW + kw;        // group, local
    if (s > 0 && s + DW - 2 < S) loads_but<(DX - 1) * NL + (DX - 2) * NX>();
    else loads_but<0>();
    if (s + DX - 1 < S) stage_x(s + DX - 1);
    if (s + DW - 1 < S) stage_w(s + DW - 1);
    const char* xs_ = smem + s % DX * L::XS + kw * L::XB;
    const char* ws = smem + L::W0 + s % DW * L::WS + wave * L::WB;
    if (gl >= g1 - g0) continue;                 // (no more of its groups)
    if (si == 0) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const u32 m = meta[gl * BN + (wc * NT + t) * 16 + l15];
        sc[t] = __builtin_bit_cast(float, m & 0xFFFF0000u);
        z[t] = (float)(m & 0xFFFFu);
      }
    }
    s16x8 b[NT][J];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const u32x4 w = *(const u32x4*)(ws + (t * 16 + l15) * (PC * 16) +
                                      ((l4 ^ slot_key16<PC>(l15)) << 4));
#pragma unroll
      for (int j = 0; j < J; ++j)
        b[t][j] = codes8_less(w[j * 2], w[j * 2 + 1], z[t]);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      s16x8 xa[J];
#pragma unroll
      for (int j = 0; j < J; ++j)
        xa[j] = *(const s16x8*)(xs_ + (t * 16 + l15) * (KS * 2) + (((l4 * J + j) ^ slot_key16<SL>(l15)) << 4));
#pragma unroll
      for (int j = 0; j < J; ++j) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          a[t][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[j], b[nt][j], a[t][nt], 0, 0, 0);
      }
    }
    if (si == gs - 1) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[t][nt][r] = fmaf(sc[nt], a[t][nt][r], acc[t][nt][r]);
          a[t][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
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
        red[(kw * BM + t * 16 + l4 * 4 + r) * LD + (wc * NT + nt) * 16 + l15] = acc[t][nt][r];
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

template <int MT, int NC, DqMode MODE>
hipError_t go(const DqArgs& A, const DqMidPlan& P, hipStream_t stream) {
  typedef Lds<MT, NC> L;
  const u32 nb = MODE == GLU ? ceil_div_u32(A.n / 2, L::BN / 2)
                             : ceil_div_u32(A.n, L::BN);
  const int lds = L::bytes((int)ceil_div_u32(A.k / A.g, A.splits));
  if (lds > MOST_LDS) return hipErrorInvalidValue;
  static bool set = false;
  if (!set) {
    LFMQ_CHECK_HIP(hipFuncSetAttribute(
        (const void*)dq_mid_kernel<MT, NC, MODE>,
        hipFuncAttributeMaxDynamicSharedMemorySize, MOST_LDS));
    set = true;
  }
  hipLaunchKernelGGL((dq_mid_kernel<MT, NC, MODE>), dim3(P.mb * nb * A.splits),
                     dim3(TPB), lds, stream, A, P.mb, P.step);
  return hipGetLastError();
}

template <int NC, DqMode MODE>
hipError_t go_rows(const DqArgs& A, const DqMidPlan& P, hipStream_t stream) {
  switch (P.step / 16) {
    case 2: return go<2, NC, MODE>(A, P, stream);
    case 3: return go<3, NC, MODE>(A, P, stream);
    case 4: return go<4, NC, MODE>(A, P, stream);
    case 5: return go<5, NC, MODE>(A, P, stream);
    case 6: return go<6, NC, MODE>(A, P, stream);
  }
  return hipErrorInvalidValue;
}

int lds_of(int mt, int nc, int groups) {
#define S(MT)                                                    \
  if (mt == MT)                                                  \
    return nc == 2 ? Lds<MT, 2>::bytes(groups) : Lds<MT, 4>::bytes(groups);
  S(2) S(3) S(4) S(5) S(6)
#undef S
  return MOST_LDS + 1;
}

}  // namespace

// Row tiles, columns of a workgroup and parts of k by the time these would take: 256
// workgroups a round, one after the other on a CU; a step 0.9 to 1.4 us, and the
// traffic and the launch of the parts.  Fitted to 1500 measured plans of 217 shapes,
// 17 to 128 rows (off by 6 % rms; the plan it takes is 0.2 % slower than the best).
DqMidPlan lfmq_dq_mid_plan(int m, int n, int k, int g, bool glu) {
  DqMidPlan best{};
  float least = INFINITY;
  const int G = k / g;
  for (int mb = 1; mb <= 4; ++mb) {
    const int step =
        max(32, (int)ceil_div_u32(ceil_div_u32(m, mb), 16) * 16);
    // (every row tile has a row)
    if (step > 96 || (mb > 1 && m < 17 * mb) || (mb - 1) * step >= m) continue;
    for (int nc = 2; nc <= 4; nc += 2) {
      const int kw = NWV / nc, bo = nc * NT * 16;
      const int nb = (int)(glu ? ceil_div_u32(n / 2, bo / 2) : ceil_div_u32(n, bo));
      for (int wgs = 0; wgs <= 512; wgs += wgs == 0 ? 256 : 128) {
        const int sp = max(1, wgs / (nb * mb));
        if (sp > 1 && (glu || sp > G / kw)) continue;
        const int ng = (int)ceil_div_u32(G, sp);
        if (lds_of(step / 16, nc, ng) > MOST_LDS) continue;
        const int u = (int)ceil_div_u32(mb * nb * sp, 256);
        const float rounds = u == 1 ? 1.f : ((u / 2) + (u & 1) * 0.527f) * 2.022f;
        const float chain =
            (int)ceil_div_u32(ng, kw) * (g / KS) *
            (nc == 2 ? 0.625f + 0.146f * (step / 16) : 0.641f + 0.122f * (step / 16));
        float t = rounds * (chain + 2.434f);
        if (sp > 1) t += 0.919e-6f * (float)m * (float)n * sp + 3.4f;
        if (t < least) {
          least = t;
          best = {mb, step, nc, sp};
        }
      }
    }
  }
  return best;
}

hipError_t lfmq_dq_mid(const DqArgs& A, const DqMidPlan& P, bool glu,
                       hipStream_t stream) {
  const int nout = glu ? A.n / 2 : A.n;
  if (A.g % 64 || A.g < 64 || A.k % A.g || A.m < 1 || (glu && A.n % 2) ||
      nout % 4 || (u64)A.n * A.k >= 1ull << 32 || (u64)A.w % 16 || P.mb < 1 ||
      P.step < 32 || P.step > 96 || (P.mb - 1) * P.step >= A.m ||
      P.mb * P.step < A.m || P.splits != A.splits || P.splits < 1 ||
      P.splits > A.k / A.g || (P.splits > 1 && (glu || A.part == nullptr)))
    return hipErrorInvalidValue;
  if (P.cols == 2)
    return glu ? go_rows<2, GLU>(A, P, stream) : go_rows<2, DENSE>(A, P, stream);
  if (P.cols == 4)
    return glu ? go_rows<4, GLU>(A, P, stream) : go_rows<4, DENSE>(A, P, stream);
  return hipErrorInvalidValue;
}
