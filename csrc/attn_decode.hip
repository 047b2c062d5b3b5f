// K8 — GQA decode attention: o = softmax(q·Kᵀ·scale)·V over the KV cache,
// one query token per sequence.
//
// Bound by the read of the cache, so a key/value row is read once for all
// the query heads that share it: a workgroup = one key range x up to GH
// query heads of one key/value head, 4 waves.  A wave takes 32 keys at a
// time on its own, no barriers: scores on the matrix cores with the keys
// as rows (a lane reads 16 bytes of a key straight from the cache), the
// online softmax per head across the lanes, weights in fp32 through a small
// LDS slab, and the weighted sum in fp32 on the vector units (a lane owns 8
// value columns, so values need no transposition; the multiplications hide
// behind the read).  The waves' results meet once at the end.
//
// FUSED: the input is the raw [q | k | v] projection row.  The prologue
// rotates this kv head's queries and its new key; workgroup 0 of the head
// writes the new cache row.  The new key's score and value never come from
// the cache: the score is the product of the unrounded rotated rows.
//
// With several key ranges the partial {o fp32[D], m, l} of each goes to
// scratch, and the last workgroup of the head to arrive merges them (a
// ticket counter) or, without tickets, a second kernel does.
//
// One layer of an 8B model (32 query heads on 8), one kernel, against a
// workgroup a query head and 64 keys:
//   b 1,  T 129       8.4 us (10.3)
//   b 1,  T 7901     20.2 us (199)
//   b 8,  T 1000     20.4 us (165)
//   b 48, T 2047     117 us (2157), 3.4 TB/s
#include "common.h"

namespace {

constexpr int TPB = 256, NW = 4, KT = 32;
constexpr int MAX_SPLITS = 64;       // a wave merges them, one a lane
// Two rounds of a wave's 32 keys cost 1.6 us more than one, a merge 4 us:
// ranges of 128 / 256 / 512 keys take 10.0 / 8.4 / 8.4 us at 129 keys,
// 13.4 / 13.6 / 17.2 at 2000, 23.7 / 20.2 / 19.1 at 7901 (b 1).
constexpr int LEAST_KEYS = 256;
// No more workgroups than are resident at once: 384 heads in 2 / 3 / 6
// ranges take 117 / 143 / 199 us (b 48, 2047 keys).
constexpr int FULL_WGS = 1024;

struct DArgs {
  const unsigned short* q;           // [b, hq, D], or [b, (hq + 2 hkv) D]
  unsigned short *kc, *vc;           // [b, hkv, tmax, D]
  float* part;                       // [b, hq, splits, D + 2]
  u32* o;                            // [b, hq, D]
  const float* inv_freq;
  const i32* T_dev;
  u32* tickets;                      // [b * hkv * head tiles], zero
  int hq, hkv, tmax, T, splits, least;
  float scale;
};

// keys a range: all ranges alike, whole wave tiles, not below `least`
__device__ __forceinline__ int range_keys(int T, int splits, int least) {
  const int per = max((T + splits - 1) / splits, least);
  return (per + KT - 1) / KT * KT;
}

// weights of `used` partial results of one head: lane c holds range c's
__device__ __forceinline__ float merge_weight(const float* p, int used,
                                              int stride, int D, int lane) {
  const bool on = lane < used;
  const float m = on ? p[lane * stride + D] : -INFINITY;
  const float l = on ? p[lane * stride + D + 1] : 0.f;
  const float M = wave_reduce_max(m);
  const float e = on ? __expf(m - M) : 0.f;
  return e / wave_reduce_sum(e * l);
}

template <int D, int GH, bool FUSED>
__global__ __launch_bounds__(TPB) void attn_decode_kernel(DArgs A) {
  constexpr int KS = D / 32, LPR = D / 8;
  constexpr int RPP = 64 / LPR;          // value rows a pass
  constexpr int NP = KT / RPP;           // passes a tile
  __shared__ __attribute__((aligned(16))) float ps[NW][KT][GH];
  __shared__ __attribute__((aligned(16))) float al_s[NW][GH];
  __shared__ float ml[NW][GH][2];
  __shared__ float ws[NW][GH][D + 1];
  __shared__ __attribute__((aligned(16))) unsigned short qs[GH][D];
  __shared__ float s_new[GH];            // FUSED: scores of the new key

  const int T = A.T_dev != nullptr ? *A.T_dev : A.T;
  const int group = A.hq / A.hkv, htiles = (group + GH - 1) / GH;
  const int kh = blockIdx.y / htiles, ht = blockIdx.y % htiles;
  const int bb = blockIdx.z;
  const int h0 = kh * group + ht * GH;             // first query head
  const int nh = min(GH, group - ht * GH);
  const int len = min(T, A.tmax);
  const int per = range_keys(len, A.splits, A.least);
  const int used = (len + per - 1) / per;
  const int lo = blockIdx.x * per, hi = min(len, lo + per);
  if (lo >= hi) return;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l15 = lane & 15, l4 = lane >> 4;
  const int vrow = lane / LPR, vcol = (lane % LPR) * 8;
  unsigned short* K = A.kc + ((u64)bb * A.hkv + kh) * A.tmax * D;
  unsigned short* V = A.vc + ((u64)bb * A.hkv + kh) * A.tmax * D;
  const s16x8 z8 = {0, 0, 0, 0, 0, 0, 0, 0};

  s16x8 qf[KS];
  u32x4 v_new = {0, 0, 0, 0};
  const int pos = FUSED ? T - 1 : -1;    // the new key
  if constexpr (FUSED) {
    const unsigned short* row = A.q + (u64)bb * (A.hq + 2 * A.hkv) * D;
    const unsigned short* kr = row + (u64)(A.hq + kh) * D;
    const unsigned short* vr = row + (u64)(A.hq + A.hkv + kh) * D;
    v_new = *(const u32x4*)(vr + vcol);
    // a wave rotates heads wave, wave + 4, ..: one angle a lane
    const int i = lane & (D / 2 - 1);
    float sn, cs;
    __sincosf((float)pos * A.inv_freq[i], &sn, &cs);
    const float k1 = bf16_bits_to_f32(kr[i]);
    const float k2 = bf16_bits_to_f32(kr[i + D / 2]);
    const float ka = k1 * cs - k2 * sn, kb = k1 * sn + k2 * cs;
    if (blockIdx.x == 0 && ht == 0 && wave == 0 && pos < A.tmax) {
      if (lane < D / 2) {
        K[(u64)pos * D + i] = (unsigned short)f32_to_bf16_bits_rne(ka);
        K[(u64)pos * D + i + D / 2] = (unsigned short)f32_to_bf16_bits_rne(kb);
      }
      if (vrow == 0) *(u32x4*)(V + (u64)pos * D + vcol) = v_new;
    }
    for (int g = wave; g < nh; g += NW) {
      const unsigned short* qr = row + (u64)(h0 + g) * D;
      const float q1 = bf16_bits_to_f32(qr[i]);
      const float q2 = bf16_bits_to_f32(qr[i + D / 2]);
      const float qa = q1 * cs - q2 * sn, qb = q1 * sn + q2 * cs;
      if (lane < D / 2) {
        qs[g][i] = (unsigned short)f32_to_bf16_bits_rne(qa);
        qs[g][i + D / 2] = (unsigned short)f32_to_bf16_bits_rne(qb);
      }
      const float s = wave_reduce_sum(lane < D / 2 ? qa * ka + qb * kb : 0.f);
      if (lane == 0) s_new[g] = s;
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = l15 < nh ? *(const s16x8*)&qs[l15 < GH ? l15 : 0][ks * 32 + l4 * 8]
                        : z8;
  } else {
    const unsigned short* qr = A.q + ((u64)bb * A.hq + h0 + l15) * D;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = l15 < nh ? *(const s16x8*)(qr + ks * 32 + l4 * 8) : z8;
  }
  const float sn_h = FUSED && l15 < nh ? s_new[l15 < GH ? l15 : 0] : 0.f;

  float m = -INFINITY, l = 0.f;          // of head l15
  float acc[GH][8] = {};
  for (int t0 = lo + wave * KT; t0 < hi; t0 += NW * KT) {
    s16x8 kf[2][KS];
    u32x4 vv[NP];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const unsigned short* kr = K + (u64)min(t0 + mt * 16 + l15, hi - 1) * D;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kf[mt][ks] = *(const s16x8*)(kr + ks * 32 + l4 * 8);
    }
#pragma unroll
    for (int i = 0; i < NP; ++i)
      vv[i] = *(const u32x4*)(V + (u64)min(t0 + i * RPP + vrow, hi - 1) * D +
                              vcol);
    f32x4 sc[2] = {};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
        sc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[mt][ks], qf[ks],
                                                         sc[mt], 0, 0, 0);
    float mx = -INFINITY;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = t0 + mt * 16 + l4 * 4 + r;
        const float s = FUSED && t == pos ? sn_h : sc[mt][r];
        sc[mt][r] = t < hi ? s * A.scale : -INFINITY;
        mx = fmaxf(mx, sc[mt][r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx);             // a tile has a visible key
    const float al = __expf(m - mn);
    float sum = 0.f;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = __expf(sc[mt][r] - mn);
        sum += p;
        if (l15 < GH) ps[wave][mt * 16 + l4 * 4 + r][l15] = p;
      }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    l = l * al + sum;
    m = mn;
    if (lane < GH) al_s[wave][lane] = al;
    // wave-local slabs: LDS operations of a wave retire in order
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int h = 0; h < GH; ++h) {
      const float a = al_s[wave][h];
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[h][e] *= a;
    }
    // rows past the range are the last one again: 0, which their weight of 0
    // leaves 0 (an infinite value would be NaN)
    if (t0 + KT > hi) {
#pragma unroll
      for (int i = 0; i < NP; ++i)
        if (t0 + i * RPP + vrow >= hi) vv[i] = u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if (FUSED && t0 + i * RPP + vrow == pos) vv[i] = v_new;
      float v[8];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        bf16x2_to_f32(vv[i][e], v[2 * e], v[2 * e + 1]);
      const float* pr = ps[wave][i * RPP + vrow];
#pragma unroll
      for (int h = 0; h < GH; ++h) {
        const float p = pr[h];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[h][e] = fmaf(p, v[e], acc[h][e]);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // ps is read
  }

  // rows of one wave, then the waves
#pragma unroll
  for (int h = 0; h < GH; ++h)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int o = LPR; o < 64; o <<= 1)
        acc[h][e] += __shfl_xor(acc[h][e], o, 64);
      if (lane < LPR) ws[wave][h][vcol + e] = acc[h][e];
    }
  if (lane < GH) {
    ml[wave][lane][0] = m;
    ml[wave][lane][1] = l;
  }
  __syncthreads();
  float* part = A.part + (((u64)bb * A.hq + h0) * A.splits + blockIdx.x) *
                             (D + 2);
  const int hstep = A.splits * (D + 2);
  for (int id = tid; id < nh * (D / 2); id += TPB) {
    const int h = id / (D / 2), e = id % (D / 2) * 2;
    const float M = fmaxf(fmaxf(ml[0][h][0], ml[1][h][0]),
                          fmaxf(ml[2][h][0], ml[3][h][0]));
    float o0 = 0.f, o1 = 0.f, L = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float c = __expf(ml[w][h][0] - M);
      o0 = fmaf(c, ws[w][h][e], o0);
      o1 = fmaf(c, ws[w][h][e + 1], o1);
      L = fmaf(c, ml[w][h][1], L);
    }
    if (used == 1) {
      A.o[((u64)bb * A.hq + h0 + h) * (D / 2) + e / 2] =
          pack_bf16x2(o0 / L, o1 / L);
      continue;
    }
    // written through to where the merging workgroup reads
    typedef __attribute__((address_space(1))) float gfloat;
    float* p = part + (u64)h * hstep;
    __hip_atomic_store((gfloat*)(p + e), o0, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store((gfloat*)(p + e + 1), o1, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    if (e == 0) {
      __hip_atomic_store((gfloat*)(p + D), M, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store((gfloat*)(p + D + 1), L, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (used == 1 || A.tickets == nullptr) return;

  // the last to arrive merges.  vmcnt is a per-wave counter: every wave
  // drains its own stores, and the barrier orders all of them before the
  // ticket.  The merging workgroup puts the ticket back to zero, so a
  // replayed graph finds it as the first launch did.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  __shared__ int last_s;
  typedef __attribute__((address_space(1))) unsigned gu32;
  gu32* ticket = (gu32*)(A.tickets + (u64)bb * gridDim.y + blockIdx.y);
  if (tid == 0) {
    const unsigned old = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_ACQ_REL,
                                                __HIP_MEMORY_SCOPE_AGENT);
    last_s = (int)old == used - 1;
    if (last_s)
      __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last_s) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  const float* head = A.part + ((u64)bb * A.hq + h0) * hstep;
  float(*wt)[GH] = (float(*)[GH])&ps[0][0][0];       // [MAX_SPLITS][GH]
  static_assert(MAX_SPLITS <= NW * KT, "weights fit the slab");
  for (int g = wave; g < nh; g += NW)
    wt[lane][g] = merge_weight(head + (u64)g * hstep, used, D + 2, D, lane);
  __syncthreads();
  for (int id = tid; id < nh * (D / 2); id += TPB) {
    const int h = id / (D / 2), e = id % (D / 2) * 2;
    const float* p = head + (u64)h * hstep + e;
    float a0 = 0.f, a1 = 0.f;
#pragma unroll 8
    for (int c = 0; c < used; ++c) {
      a0 = fmaf(wt[c][h], p[c * (D + 2)], a0);
      a1 = fmaf(wt[c][h], p[c * (D + 2) + 1], a1);
    }
    A.o[((u64)bb * A.hq + h0 + h) * (D / 2) + e / 2] = pack_bf16x2(a0, a1);
  }
}

// the merge as a kernel of its own: one head a wave
template <int D>
__global__ __launch_bounds__(64) void attn_decode_merge(DArgs A) {
  const int len = min(A.T_dev != nullptr ? *A.T_dev : A.T, A.tmax);
  const int per = range_keys(len, A.splits, A.least);
  const int used = (len + per - 1) / per;
  if (used <= 1) return;
  __shared__ float wt[MAX_SPLITS];
  const float* p = A.part + (u64)blockIdx.x * A.splits * (D + 2);
  const int lane = threadIdx.x;
  wt[lane] = merge_weight(p, used, D + 2, D, lane);
  __syncthreads();
  if (2 * lane >= D) return;
  float a0 = 0.f, a1 = 0.f;
#pragma unroll 8
  for (int c = 0; c < used; ++c) {
    a0 = fmaf(wt[c], p[c * (D + 2) + 2 * lane], a0);
    a1 = fmaf(wt[c], p[c * (D + 2) + 2 * lane + 1], a1);
  }
  A.o[(u64)blockIdx.x * (D / 2) + lane] = pack_bf16x2(a0, a1);
}

// query heads a workgroup
int head_tile(int group) {
  return group <= 1 ? 1 : (group <= 2 ? 2 : (group <= 4 ? 4 : 8));
}

template <int D, bool FUSED>
hipError_t launch(const DArgs& A, int b, hipStream_t stream) {
  const int group = A.hq / A.hkv, gh = head_tile(group);
  const dim3 grid(A.splits, A.hkv * ((group + gh - 1) / gh), b);
#define GO(G)                                                               \
  hipLaunchKernelGGL((attn_decode_kernel<D, G, FUSED>), grid, dim3(TPB), 0, \
                     stream, A)
  if (gh == 1) GO(1);
  else if (gh == 2) GO(2);
  else if (gh == 4) GO(4);
  else GO(8);
#undef GO
  if (A.splits > 1 && A.tickets == nullptr)
    hipLaunchKernelGGL((attn_decode_merge<D>), dim3(b * A.hq), dim3(64), 0,
                       stream, A);
  return hipGetLastError();
}

}  // namespace

// Key ranges a head for up to T keys.
int lfmq_attn_decode_splits(int b, int hq, int hkv, int T) {
  const int group = hq / hkv, gh = head_tile(group);
  const int wgs = b * hkv * ((group + gh - 1) / gh);
  const int n = FULL_WGS / max(wgs, 1);
  const int most = (T + LEAST_KEYS - 1) / LEAST_KEYS;
  return max(1, min(min(n, most), MAX_SPLITS));
}

// q [b, hq, d]; scratch: b*hq*splits*(d+2) floats.  T_dev != null: the
// number of keys is read on the device (T sized the splits).
hipError_t lfmq_attn_decode(const void* q, const void* kc, const void* vc,
                            void* o, void* scratch, int b, int hq, int hkv,
                            int tmax, int T, const void* T_dev, int d,
                            int splits, float scale, hipStream_t stream) {
  if (d != 128 && d != 64) return hipErrorInvalidValue;
  if (hq % hkv || T < 1) return hipErrorInvalidValue;
  const DArgs A{(const unsigned short*)q, (unsigned short*)kc,
                (unsigned short*)vc, (float*)scratch, (u32*)o, nullptr,
                (const i32*)T_dev, nullptr, hq, hkv, tmax, T, splits,
                LEAST_KEYS, scale};
  return d == 128 ? launch<128, false>(A, b, stream)
                  : launch<64, false>(A, b, stream);
}

// Rotation, cache append and attention from the raw [b, (hq+2hkv)*d]
// projection; the new token sits at T-1.  tickets (null: a second kernel
// merges): zero-initialized u32[b*hq].
hipError_t lfmq_attn_decode_fused(const void* qkv, void* kc, void* vc,
                                  void* o, void* scratch,
                                  const void* inv_freq, int b, int hq,
                                  int hkv, int tmax, int T, const void* T_dev,
                                  int d, int splits, float scale,
                                  void* tickets, hipStream_t stream) {
  if (d != 128 && d != 64) return hipErrorInvalidValue;
  if (hq % hkv || T < 1) return hipErrorInvalidValue;
  const DArgs A{(const unsigned short*)qkv, (unsigned short*)kc,
                (unsigned short*)vc, (float*)scratch, (u32*)o,
                (const float*)inv_freq, (const i32*)T_dev, (u32*)tickets, hq,
                hkv, tmax, T, splits, LEAST_KEYS, scale};
  return d == 128 ? launch<128, true>(A, b, stream)
                  : launch<64, true>(A, b, stream);
}
