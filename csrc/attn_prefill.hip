// Flash-style prefill attention on MFMA: o = softmax(q·Kᵀ·scale + causal)·V
// against the KV cache, s >= 1 queries at positions [pos0, pos0+s).
//
//   q   [b, s, hq*128] bf16, already roped (qkv_rope_append output view)
//   k/v [b, hkv, tmax, 128] bf16 caches holding positions [0, pos0+s)
//   out [b, s, hq*128] bf16
//
// One workgroup = 4 waves x QT * 16 queries of one head, key tiles of 64.
// Keys and values go from the cache straight into LDS as they are (two
// buffers, XOR-swizzled).  Scores are computed transposed (keys as rows,
// queries as columns), so that a lane holds 16 keys of one query: the softmax
// needs two shuffles a tile, and the rounded weights are already the right
// operand of the product with the values, transposed as well: the transposing
// LDS read brings four keys of a lane's value column in the scores' order.
// Scores, softmax and sums stay in fp32 registers.  The last queries see the
// most keys and start first.
//
// Bound by the LDS reads of both operands and the softmax's vector work.
// 32 heads on 8, us before (values transposed by 2-byte LDS writes, weights
// through LDS) and now:
//   1 x 512          32.2 ->  15.1    1 x 3001 after 1000   866 -> 186
//   2 x 330          33.9 ->  12.8    1 x 8192             3785 -> 620
//   1 x 2048          367 ->  65      (663 and 887 TFLOP/s)
#include "lds_dma.h"

namespace {

constexpr int TPB = 256, NW = 4;
constexpr int BN = 64;                       // keys a tile
constexpr int HD = 128;                      // head dim (only supported size)
constexpr int ROW = HD * 2, TILE = BN * ROW; // bytes
constexpr int KS = HD / 32, VT = HD / 16;
constexpr float LOG2E = 1.4426950408889634f;

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;

struct PArgs {
  const unsigned short *q, *kc, *vc;
  unsigned short* o;
  int s, b, hq, hkv, tmax, pos0, T;
  float scale, sign;       // scale > 0; what queries are multiplied by first
};

__device__ __forceinline__ u32 pack2(float a, float b) {
  const bf16x2_native v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(u32, v);
}

template <int QT>
__global__ __launch_bounds__(TPB, 2) void attn_prefill_kernel(PArgs A) {
  constexpr int BM = NW * QT * 16;
  extern __shared__ __attribute__((aligned(16))) char smem[];  // [2][K | V]
  // An XCD (every eighth workgroup) takes an eighth of the heads, if that
  // divides them, so that its L2 holds the keys and values they share: heads
  // fastest, last queries first (8192 queries 851 us, so 620)
  const u32 nq = (A.s + BM - 1) / BM, all = A.hq * A.b, per = all / 8;
  u32 id = blockIdx.x, hb = id / nq, qt = id % nq;
  if (all % 8 == 0) {
    hb = id % 8 * per + id / 8 % per;
    qt = id / 8 / per;
  }
  const int q0 = (int)(nq - 1 - qt) * BM;
  const int h = hb % A.hq, bb = hb / A.hq, hk = h / (A.hq / A.hkv);
  const int lane = threadIdx.x & 63, l15 = lane & 15, l4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned short* K = A.kc + ((u64)bb * A.hkv + hk) * A.tmax * HD;
  const unsigned short* V = A.vc + ((u64)bb * A.hkv + hk) * A.tmax * HD;

  // keys below hi are visible to the workgroup's last query
  const int hi = min(A.T, A.pos0 + q0 + BM);
  // staging: a wave's load fills 4 keys; keys past the end repeat the last
  auto stage = [&](int t0, int buf) {
#pragma unroll
    for (int i = 0; i < TILE / 1024 / NW; ++i) {
      const int r = (i * NW + wave) * 4 + (lane >> 4);
      const u32 row = (u32)min(t0 + r, hi - 1) * ROW;
      const u32 lds = buf * 2 * TILE + (i * NW + wave) * 1024;
      load_to_lds(K, row + ((l15 ^ slot_key<16>(r)) << 4), lds);
      load_to_lds(V, row + ((((l15 >> 1) ^ (r & 7)) << 5) | (l15 & 1) << 4),
                  lds + TILE);
    }
  };
  stage(0, 0);

  const int w0 = q0 + wave * (QT * 16);          // the wave's first query
  s16x8 qf[QT][KS];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const u64 row = (u64)bb * A.s + min(w0 + qt * 16 + l15, A.s - 1);
    const unsigned short* p = A.q + (row * A.hq + h) * HD;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[qt][ks] = *(const s16x8*)(p + ks * 32 + l4 * 8);
  }
  if (A.sign != 1.f) {
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          qf[qt][ks][e] = (short)f32_to_bf16_bits_rne(
              bf16_bits_to_f32((unsigned short)qf[qt][ks][e]) * A.sign);
  }
  const float sc2 = A.scale * LOG2E;             // softmax in powers of two
  const int w_lo = A.pos0 + w0, w_hi = w_lo + QT * 16 - 1;   // positions
  float m[QT], l[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    m[qt] = -INFINITY;
    l[qt] = 0.f;
  }
  f32x4 oacc[QT][VT] = {};

  for (int t0 = 0, par = 0; t0 < hi; t0 += BN, par ^= 1) {
    lds_loads_done();
    if (t0 + BN < hi) stage(t0 + BN, par ^ 1);
    if (t0 + BN > hi) {
      // values past the end: 0, which their weight of 0 leaves 0 (an infinite
      // one would be NaN)
      const u32x4 z = {0, 0, 0, 0};
      for (int i = (hi - t0) * (ROW / 16) + threadIdx.x; i < TILE / 16; i += TPB)
        *(u32x4*)(smem + par * 2 * TILE + TILE + i * 16) = z;
      __syncthreads();
    }
    if (t0 > w_hi) continue;                     // none seen
    const char* lk = smem + par * 2 * TILE;
    const char* lv = lk + TILE;

    f32x4 sc[QT][BN / 16] = {};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int nt = 0; nt < BN / 16; ++nt) {
        const s16x8 kf = *(const s16x8*)(
            lk + (nt * 16 + l15) * ROW +
            (((ks * 4 + l4) ^ slot_key<16>(l15)) << 4));
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
          sc[qt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              kf, qf[qt][ks], sc[qt][nt], 0, 0, 0);
      }
    // a tile that every query of this wave sees whole needs no mask
    const bool whole = t0 + BN - 1 <= w_lo && t0 + BN <= hi;
    s16x8 pf[QT][BN / 32];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      if (!whole) {
        const int last = min(w_lo + qt * 16 + l15, hi - 1) - t0 - l4 * 4;
#pragma unroll
        for (int nt = 0; nt < BN / 16; ++nt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            sc[qt][nt][r] = nt * 16 + r <= last ? sc[qt][nt][r] : -INFINITY;
      }
      float mx = sc[qt][0][0];
#pragma unroll
      for (int nt = 0; nt < BN / 16; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sc[qt][nt][r]);
      mx *= sc2;
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      mx = fmaxf(mx, m[qt]);                     // finite: key 0 came first
      if (__any(mx > m[qt])) {
        const float al = __builtin_amdgcn_exp2f(m[qt] - mx);
        m[qt] = mx;
        l[qt] *= al;
#pragma unroll
        for (int on = 0; on < VT; ++on) oacc[qt][on] *= al;
      }
      float ps = 0.f;
#pragma unroll
      for (int nt = 0; nt < BN / 16; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sc[qt][nt][r] =
              __builtin_amdgcn_exp2f(fmaf(sc[qt][nt][r], sc2, -mx));
          ps += sc[qt][nt][r];
        }
      l[qt] += ps;                               // of this lane's keys
#pragma unroll
      for (int k2 = 0; k2 < BN / 32; ++k2) {
        const f32x4 a = sc[qt][2 * k2], b = sc[qt][2 * k2 + 1];
        const u32x4 v = {pack2(a[0], a[1]), pack2(a[2], a[3]),
                         pack2(b[0], b[1]), pack2(b[2], b[3])};
        pf[qt][k2] = __builtin_bit_cast(s16x8, v);
      }
    }
    // keys of a step, in the scores' order: 16 (2 k2) + 4 l4 + 0..3, then
    // the same of the next 16
#pragma unroll
    for (int k2 = 0; k2 < BN / 32; ++k2)
#pragma unroll
      for (int on = 0; on < VT; ++on) {
        s16x8 vf;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int key = k2 * 32 + e * 16 + l4 * 4 + (l15 >> 2);
          const char* p =
              lv + key * ROW + ((on ^ (key & 7)) << 5) + (l15 & 3) * 8;
          const s16x4_t v =
              __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
#pragma unroll
          for (int i = 0; i < 4; ++i) vf[e * 4 + i] = v[i];
        }
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
          oacc[qt][on] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              vf, pf[qt][k2], oacc[qt][on], 0, 0, 0);
      }
  }

  // a lane holds four consecutive columns of one query
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int qr = w0 + qt * 16 + l15;
    float sum = l[qt];
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (qr >= A.s) continue;
    const float inv = 1.f / sum;
    unsigned short* p = A.o + (((u64)bb * A.s + qr) * A.hq + h) * HD + l4 * 4;
#pragma unroll
    for (int on = 0; on < VT; ++on)
      *(u64*)(p + on * 16) =
          pack2(oacc[qt][on][0] * inv, oacc[qt][on][1] * inv) |
          (u64)pack2(oacc[qt][on][2] * inv, oacc[qt][on][3] * inv) << 32;
  }
}

template <int QT>
hipError_t launch(const PArgs& A, int b, hipStream_t stream) {
  constexpr int lds = 4 * TILE;
  const dim3 grid((A.s + NW * QT * 16 - 1) / (NW * QT * 16) * A.hq * A.b);
  hipLaunchKernelGGL(attn_prefill_kernel<QT>, grid, dim3(TPB), lds, stream, A);
  return hipGetLastError();
}

}  // namespace

// q [b,s,hq*d] roped; caches [b,hkv,tmax,d] already hold rows [0, pos0+s).
// d == 128 only (callers fall back to the matmul-chain path otherwise).
hipError_t lfmq_attn_prefill(const void* q, const void* kc, const void* vc,
                             void* o, int b, int s, int hq, int hkv, int tmax,
                             int pos0, int d, float scale,
                             hipStream_t stream) {
  if (d != HD) return hipErrorInvalidValue;
  if (hq % hkv) return hipErrorInvalidValue;
  const int T = pos0 + s;
  if (T > tmax) return hipErrorInvalidValue;
  // The kernel compares scores before it scales them.  A scale that turns
  // their order or makes them equal goes to the queries instead: -1 and 0 are
  // exact there, and NaN makes all of them NaN.
  const bool up = scale > 0.f;
  const PArgs A{(const unsigned short*)q, (const unsigned short*)kc,
                (const unsigned short*)vc, (unsigned short*)o, s, b, hq, hkv,
                tmax, pos0, T, up ? scale : (scale < 0.f ? -scale : 1.f),
                up ? 1.f : (scale < 0.f ? -1.f : scale)};
  // 128 queries a workgroup where they fill the chip, else 64 (us of 64 / 128:
  // 512 queries 14.9 / 17.4, 1024 32.1 / 33.4, 2048 109 / 79, heads in turn)
  if ((long)((s + 127) / 128) * hq * b >= 384) return launch<2>(A, b, stream);
  return launch<1>(A, b, stream);
}
