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
// A launch that only reads 402 MB takes 66 us, one of 33 MB 6.5, and so does this
// one from some 60 MB on since its loads are whole lines that pass the caches by
// (b 48, T 2047 by half lines of keys 76.6, values past the caches 69, keys too
// 72, keys by whole lines alike 67).  Below, the rest is a
// chain from the length over the keys and the rotation to the scores, sums over
// the lanes, and the merge's trips to memory.  So a wave's first keys and values
// are on their way before the rotation and the next ones during a round, by loads
// that stop at the range's end and wait by count; sums over the lanes are taken two
// at a time by exchanges of lanes and not through LDS.  One layer of an 8B model
// (32 query heads on 8), cold, us before (loads in the round that needs them, in the
// caches' way) and now:
//   b 1,  T 129         8.1 ->  6.0      b 8,  T 4000     31.3 -> 26.5
//   b 1,  T 7901       16.8 -> 13.9      b 20, T 900      21.9 -> 18.1
//   b 8,  T 1000       14.3 -> 11.8      b 48, T 2047     80.0 -> 67.7 (5.9 TB/s)
#include <type_traits>

#include "common.h"

namespace {

constexpr int KT = 32;               // keys of a wave and round
constexpr int MAX_SPLITS = 64;       // a wave merges them, one a lane
// A merge costs 2 us, two rounds of a wave's 32 keys 1.5 more than one.  Up to
// ONE_RANGE keys are one range; longer ranges than LEAST_KEYS where there would
// be more than MANY of them, of the keys that there are: a cache that is half
// full has as many.  us (32 heads on 8, b 1) with one range up to 128 / 256 keys
// 6.6 / 6.2 at 150 keys (b 4 7.0 / 6.3); with least ranges of 128 / 256 7.0 / 8.1
// at 700, 8.0 / 8.8 at 1500, 10.3 / 10.3 at 4000, but b 12 10.4 / 9.4 at 400 and
// 12.4 / 13.2 at 700.
constexpr int ONE_RANGE = 256, LEAST_KEYS = 128, MANY = 24;
// Two workgroups a CU, three where a range has very many keys: us with 512 / 768
// workgroups 26.5 / 27.6 (b 8, 4000 keys), 15.6 / 16.2 (b 16, 900), 71.6 / 67.7
// (b 48, 2047; with 1536 70.4).  Not where a workgroup has eight heads, of which two fit: 23.3 /
// 32.8 (28 heads on 4, b 13, 2000 keys of 16384).
constexpr int FULL_WGS = 512, MORE_WGS = 768, LONG_RANGE = 1024;

struct DArgs {
  const unsigned short* q;           // [b, hq, D], or [b, (hq + 2 hkv) D]
  unsigned short *kc, *vc;           // [b, hkv, tmax, D]
  float* part;                       // [b, hq, splits, D + 2]
  u32* o;                            // [b, hq, D]
  const float* inv_freq;
  const i32* T_dev;
  u32* tickets;                      // [b * hkv * head tiles], zero
  int hq, hkv, tmax, T, splits;
  float scale;
  int group, htiles;                 // hq / hkv, workgroups a key/value head
  u32 inv_splits;                    // 2^32 / splits, rounded up
};

// keys a range: all ranges alike, whole wave tiles
template <int NW>
__device__ __forceinline__ int range_keys(const DArgs& A, int len) {
  // (len + splits - 1) / splits, exact below 2^26 keys
  const int per = A.splits == 1 ? len
                                : (int)(((u64)(u32)(len + A.splits - 1) *
                                         A.inv_splits) >> 32);
  const int least = NW == 8 || len <= ONE_RANGE ? ONE_RANGE
                    : len <= MANY * LEAST_KEYS ? LEAST_KEYS : 2 * LEAST_KEYS;
  return (max(per, least) + KT - 1) / KT * KT;
}

// the other half's value, or the other 16 lanes' of this half
__device__ __forceinline__ float max_across(float v) {
  const u32 x = __builtin_bit_cast(u32, v);
  const auto p = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  const u32 p0 = p[0], p1 = p[1];
  const u32 y = __builtin_bit_cast(u32, fmaxf(__builtin_bit_cast(float, p0),
                                              __builtin_bit_cast(float, p1)));
  const auto q = __builtin_amdgcn_permlane16_swap(y, y, false, false);
  const u32 q0 = q[0], q1 = q[1];
  return fmaxf(__builtin_bit_cast(float, q0), __builtin_bit_cast(float, q1));
}

__device__ __forceinline__ float sum_across(float v) {
  const u32 x = __builtin_bit_cast(u32, v);
  const auto p = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  const u32 p0 = p[0], p1 = p[1];
  const u32 y = __builtin_bit_cast(u32, __builtin_bit_cast(float, p0) +
                                            __builtin_bit_cast(float, p1));
  const auto q = __builtin_amdgcn_permlane16_swap(y, y, false, false);
  const u32 q0 = q[0], q1 = q[1];
  return __builtin_bit_cast(float, q0) + __builtin_bit_cast(float, q1);
}
// a of both halves in the lower one, b in the upper one
__device__ __forceinline__ float sum_halves(float a, float b) {
  const auto p = __builtin_amdgcn_permlane32_swap(
      __builtin_bit_cast(u32, a), __builtin_bit_cast(u32, b), false, false);
  const u32 p0 = p[0], p1 = p[1];
  return __builtin_bit_cast(float, p0) + __builtin_bit_cast(float, p1);
}
// the same in each half: 16 lanes and 16
__device__ __forceinline__ float sum_quarters(float a, float b) {
  const auto p = __builtin_amdgcn_permlane16_swap(
      __builtin_bit_cast(u32, a), __builtin_bit_cast(u32, b), false, false);
  const u32 p0 = p[0], p1 = p[1];
  return __builtin_bit_cast(float, p0) + __builtin_bit_cast(float, p1);
}

// a's lower half and b's, plus the upper halves eight columns away
__device__ __forceinline__ float sum_pieces(float a, float b) {
  const auto p = __builtin_amdgcn_permlane32_swap(
      __builtin_bit_cast(u32, a), __builtin_bit_cast(u32, b), false, false);
  const u32 p0 = p[0], p1 = p[1];
  return __builtin_bit_cast(float, p0) +
         __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                                       0, (int)p1, 0x128, 0xf, 0xf, true));
}

// Two floats of a partial result, past the caches of the XCD: a workgroup of
// another one may be the reader.
__device__ __forceinline__ void put2(float* p, float a, float b) {
  typedef __attribute__((address_space(1))) u64 gu64;
  __hip_atomic_store((gu64*)p,
                     (u64)__builtin_bit_cast(u32, b) << 32 |
                         __builtin_bit_cast(u32, a),
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void get2(const float* p, float& a, float& b) {
  typedef __attribute__((address_space(1))) u64 gu64;
  const u64 v = __hip_atomic_load((gu64*)p, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
  a = __builtin_bit_cast(float, (u32)v);
  b = __builtin_bit_cast(float, (u32)(v >> 32));
}

// weights of `used` partial results of one head: lane c holds range c's
__device__ __forceinline__ float merge_weight(const float* p, int used,
                                              int stride, int D, int lane) {
  const bool on = lane < used;
  float m = -INFINITY, l = 0.f;
  if (on) get2(p + lane * stride + D, m, l);
  const float M = wave_reduce_max_dpp(m);
  const float e = on ? __expf(m - M) : 0.f;
  return e / wave_reduce_sum_dpp(e * l);
}

// NT: keys and values pass the caches by (cache policy 2)
template <int D, int GH, bool FUSED, int NW, bool NT>
__global__ __launch_bounds__(NW * 64, NW == 8 || D * GH > 512 ? 2 : 3)
void attn_decode_kernel(DArgs A) {
  constexpr int TPB = NW * 64, AUX = NT ? 2 : 0;
  constexpr int KL = D / 64, LPR = D / 8;  // lines of 128 bytes a key
  constexpr int RPP = 64 / LPR;          // value rows a pass
  constexpr int NP = KT / RPP;           // passes a tile
  __shared__ __attribute__((aligned(16))) float ps[NW][KT][GH];
  __shared__ __attribute__((aligned(16))) float al_s[NW][GH];
  __shared__ float ml[NW][GH][2];
  __shared__ float ws[NW][GH][D + 1];
  __shared__ __attribute__((aligned(16))) unsigned short qs[GH][D];
  __shared__ float s_new[GH];            // FUSED: scores of the new key

  const int T = A.T_dev != nullptr ? *A.T_dev : A.T;
  const int group = A.group, htiles = A.htiles;
  const int kh = htiles == 1 ? blockIdx.x : blockIdx.x / htiles;
  const int ht = htiles == 1 ? 0 : blockIdx.x % htiles;
  const int bb = blockIdx.y, range = blockIdx.z;
  const int h0 = kh * group + ht * GH;             // first query head
  const int nh = min(GH, group - ht * GH);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l15 = lane & 15, l4 = lane >> 4, lh = l15 & 7;
  const int vrow = lane / LPR, vcol = (lane % LPR) * 8;
  const s16x8 z8 = {0, 0, 0, 0, 0, 0, 0, 0};

  s16x8 qf[KL];
  auto piece = [&](int j) { return j * 64 + (l4 * 2 + (l15 >> 3)) * 8; };
  u32x4 v_new = {0, 0, 0, 0};
  // what does not depend on the number of keys is on its way with it: a wave
  // rotates heads wave, wave + 4, one angle a lane
  constexpr int QW = (GH + NW - 1) / NW;
  float freq, k1, k2, q1[QW], q2[QW];
  const int i = lane & (D / 2 - 1);
  if constexpr (FUSED) {
    const unsigned short* row = A.q + (u64)bb * (A.hq + 2 * A.hkv) * D;
    const unsigned short* kr = row + (u64)(A.hq + kh) * D;
    v_new = *(const u32x4*)(row + (u64)(A.hq + A.hkv + kh) * D + vcol);
    freq = A.inv_freq[i];
    k1 = bf16_bits_to_f32(kr[i]);
    k2 = bf16_bits_to_f32(kr[i + D / 2]);
#pragma unroll
    for (int g = 0; g < QW; ++g) {
      const unsigned short* qr =
          row + (u64)(h0 + min(wave + g * NW, nh - 1)) * D;
      q1[g] = bf16_bits_to_f32(qr[i]);
      q2[g] = bf16_bits_to_f32(qr[i + D / 2]);
    }
  }
  const int len = min(T, A.tmax);
  const int per = range_keys<NW>(A, len);
  const int lo = range * per, hi = min(len, lo + per);
  if (lo >= hi) return;
  unsigned short* K = A.kc + ((u64)bb * A.hkv + kh) * A.tmax * D;
  unsigned short* V = A.vc + ((u64)bb * A.hkv + kh) * A.tmax * D;
  // A wave's keys and values from t0 on, zeros past the range.  The first are on
  // their way beside the rotation, the next ones as soon as there is room for
  // them; the loads are there without keys too, or the compiler waits for all.
  // A load of keys takes a whole line of 128 bytes of 8 of them: lane l15 has key
  // l15 % 8, piece l4 * 2 of the line below l15 8 and l4 * 2 + 1 from there.  As
  // rows of a product, keys' first pieces and keys' second ones; its columns are
  // heads' first pieces and, 8 on, heads' second ones.
  s16x8 kf[KT / 8][KL];
  u32x4 vv[NP];
  auto rows_of = [&](const unsigned short* base, int t0) {
    const int n = max(0, min(KT, hi - t0));
    return make_rsrc_uniform(base + (u64)(n > 0 ? t0 : 0) * D, (u32)n * D * 2);
  };
  auto load_keys = [&](int t0) {
    const auto r = rows_of(K, t0);
#pragma unroll
    for (int g = 0; g < KT / 8; ++g)
#pragma unroll
      for (int j = 0; j < KL; ++j)
        kf[g][j] = __builtin_bit_cast(
            s16x8, __builtin_amdgcn_raw_buffer_load_b128(
                       r, ((g * 8 + (l15 & 7)) * D + piece(j)) * 2, 0, AUX));
  };
  auto load_values = [&](int t0) {
    const auto r = rows_of(V, t0);
#pragma unroll
    for (int i = 0; i < NP; ++i)
      vv[i] = __builtin_amdgcn_raw_buffer_load_b128(
          r, ((i * RPP + vrow) * D + vcol) * 2, 0, AUX);
  };
  const int first = lo + __builtin_amdgcn_readfirstlane(wave) * KT;
  load_keys(first);
  load_values(first);
  const int pos = FUSED ? T - 1 : -1;    // the new key
  if constexpr (FUSED) {
    float sn, cs;
    __sincosf((float)pos * freq, &sn, &cs);
    const float ka = k1 * cs - k2 * sn, kb = k1 * sn + k2 * cs;
    if (range == 0 && ht == 0 && wave == 0 && pos < A.tmax) {
      if (lane < D / 2) {
        K[(u64)pos * D + i] = (unsigned short)f32_to_bf16_bits_rne(ka);
        K[(u64)pos * D + i + D / 2] = (unsigned short)f32_to_bf16_bits_rne(kb);
      }
      if (vrow == 0) *(u32x4*)(V + (u64)pos * D + vcol) = v_new;
    }
#pragma unroll
    for (int j = 0; j < QW; ++j) {
      const int g = wave + j * NW;
      if (g >= nh) break;
      const float qa = q1[j] * cs - q2[j] * sn, qb = q1[j] * sn + q2[j] * cs;
      if (lane < D / 2) {
        qs[g][i] = (unsigned short)f32_to_bf16_bits_rne(qa);
        qs[g][i + D / 2] = (unsigned short)f32_to_bf16_bits_rne(qb);
      }
      const float s =
          wave_reduce_sum_dpp(lane < D / 2 ? qa * ka + qb * kb : 0.f);
      if (lane == 0) s_new[g] = s;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < KL; ++j)
      qf[j] = lh < nh ? *(const s16x8*)&qs[lh < GH ? lh : 0][piece(j)] : z8;
  } else {
    const unsigned short* qr = A.q + ((u64)bb * A.hq + h0 + lh) * D;
#pragma unroll
    for (int j = 0; j < KL; ++j)
      qf[j] = lh < nh ? *(const s16x8*)(qr + piece(j)) : z8;
  }
  const float sn_h = FUSED && l15 < nh ? s_new[l15 < GH ? l15 : 0] : 0.f;

  float m = -INFINITY, l = 0.f;          // of head l15
  float acc[GH][8] = {};
  for (int t0 = first; t0 < hi; t0 += NW * KT) {
    f32x4 pt[KT / 8] = {};
#pragma unroll
    for (int j = 0; j < KL; ++j)
#pragma unroll
      for (int g = 0; g < KT / 8; ++g)
        pt[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[g][j], qf[j], pt[g],
                                                        0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);         // not before: other registers
    load_keys(t0 + NW * KT);
    // a result's rows: first pieces in the lower half of the wave, second ones in
    // the upper half; what pairs a first with a second stays in lanes from 8 on
    f32x4 sc[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sc[mt][r] = sum_pieces(pt[mt * 2][r], pt[mt * 2 + 1][r]);
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
    const float mn = fmaxf(m, max_across(mx));  // a tile has a visible key
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
    l = l * al + sum;                          // this lane's keys only
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
    // (rows past the range are zeros, which their weight of 0 leaves 0)
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
    __builtin_amdgcn_sched_barrier(0);
    load_values(t0 + NW * KT);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // ps is read
  }

  // lanes and rows of one wave, then the waves.  Two sums at a time: halves, then
  // quarters of the wave end up with one each, in all R of GH * 8
  l = sum_across(l);
  constexpr int NV = GH * 8, R = NV / 4;
  float* a1 = &acc[0][0];
  if constexpr (LPR == 8)
#pragma unroll
    for (int v = 0; v < NV; ++v)
      a1[v] += __builtin_bit_cast(
          float, __builtin_amdgcn_update_dpp(
                     0, __builtin_bit_cast(int, a1[v]), 0x128, 0xf, 0xf, true));
#pragma unroll
  for (int v = 0; v < NV / 2; ++v) a1[v] = sum_halves(a1[v], a1[v + NV / 2]);
#pragma unroll
  for (int v = 0; v < R; ++v) {
    const float x = sum_quarters(a1[v], a1[v + R]);
    const int at = l4 * R + v;               // of the heads' columns
    if (l15 < LPR) ws[wave][at / 8][vcol + at % 8] = x;
  }
  if (lane < GH) {
    ml[wave][lane][0] = m;
    ml[wave][lane][1] = l;
  }
  __syncthreads();
  const int used = (len + per - 1) / per;
  float* part = A.part + (((u64)bb * A.hq + h0) * A.splits + range) *
                             (D + 2);
  const int hstep = A.splits * (D + 2);
  for (int id = tid; id < nh * (D / 2); id += TPB) {
    const int h = id / (D / 2), e = id % (D / 2) * 2;
    float M = ml[0][h][0];
#pragma unroll
    for (int w = 1; w < NW; ++w) M = fmaxf(M, ml[w][h][0]);
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
    float* p = part + (u64)h * hstep;
    put2(p + e, o0, o1);
    if (e == 0) put2(p + D, M, L);
  }
  if (used == 1 || A.tickets == nullptr) return;

  // The last to arrive merges.  vmcnt is a per-wave counter: every wave
  // drains its own stores, which are past the XCDs' caches when they are done,
  // and the barrier orders all of them before the ticket; the merging workgroup
  // reads past its caches, too.  So the ticket orders nothing: as a release and
  // acquire, which any chip would need that keeps agent scope in its L2s, it
  // writes back and empties an XCD's L2, once for each of these workgroups (48 x
  // 300 keys, 384 of them: 58 us).  The merging workgroup
  // puts the ticket back to zero, so a replayed graph finds it as the first
  // launch did.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  __shared__ int last_s;
  typedef __attribute__((address_space(1))) unsigned gu32;
  gu32* ticket = (gu32*)(A.tickets + (u64)bb * gridDim.x + blockIdx.x);
  if (tid == 0) {
    const unsigned old = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
    last_s = (int)old == used - 1;
    if (last_s)
      __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last_s) return;
  // the first results of a thread are on their way with the weights
  const float* head = A.part + ((u64)bb * A.hq + h0) * hstep;
  constexpr int AT = 32;                             // ranges at a time
  float r0[AT], r1[AT];
  auto fetch = [&](int id, int c0) {
    const float* p = head + (u64)(id / (D / 2)) * hstep + id % (D / 2) * 2;
#pragma unroll
    for (int c = 0; c < AT; ++c)
      if (c0 + c < used) get2(p + (c0 + c) * (D + 2), r0[c], r1[c]);
  };
  const int ids = nh * (D / 2);
  if (tid < ids) fetch(tid, 0);
  float(*wt)[GH] = (float(*)[GH])&ps[0][0][0];       // [MAX_SPLITS][GH]
  static_assert(MAX_SPLITS <= NW * KT, "weights fit the slab");
  for (int g = wave; g < nh; g += NW)
    wt[lane][g] = merge_weight(head + (u64)g * hstep, used, D + 2, D, lane);
  __syncthreads();
  for (int id = tid; id < ids; id += TPB) {
    const int h = id / (D / 2);
    float a0 = 0.f, a1 = 0.f;
    for (int c0 = 0; c0 < used; c0 += AT) {
      if (id != tid || c0 > 0) fetch(id, c0);
#pragma unroll
      for (int c = 0; c < AT; ++c)
        if (c0 + c < used) {
          a0 = fmaf(wt[c0 + c][h], r0[c], a0);
          a1 = fmaf(wt[c0 + c][h], r1[c], a1);
        }
    }
    A.o[((u64)bb * A.hq + h0 + h) * (D / 2) + id % (D / 2)] =
        pack_bf16x2(a0, a1);
  }
}

// the merge as a kernel of its own: one head a wave
template <int D, int NW>
__global__ __launch_bounds__(64) void attn_decode_merge(DArgs A) {
  const int len = min(A.T_dev != nullptr ? *A.T_dev : A.T, A.tmax);
  const int per = range_keys<NW>(A, len);
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

// Eight waves a workgroup, ranges of one round of theirs: eight heads of 128,
// whose rounds are the longest, where that is a workgroup a CU or less.  us with
// four / eight (8 heads on one key head, of 128): 11.9 / 10.2 at 1500 keys (b 1, 4
// key heads), 18.5 / 14.1 at 8000, 16.6 / 13.8 (b 3, 4000), 5.7 / 6.1 at 60; of 64
// 10.6 / 9.6 to 7.0 / 7.8; 4 heads of 128 7.0 / 8.4 at 600 keys, 10.2 / 10.5 at 4000.
bool eight_waves(int d, int gh, int wgs, int T) {
  return d == 128 && gh == 8 && T <= MAX_SPLITS * ONE_RANGE &&
         (long)wgs * ((T + ONE_RANGE - 1) / ONE_RANGE) <= 256;
}

// From how many bytes of keys and values on they pass the caches by: less than
// this, of all layers, may still be there at the next token (b 1, 129 keys in a
// step of four layers 0.25 us a launch).  us in the caches' way / past them, cold: b 1, 600 keys (2.5 MB) 7.1 / 7.1, b 4,
// 300 (4.9 MB) 7.4 / 7.3, b 16, 129 (8.5 MB) 7.2 / 6.8, b 48, 300 16.5 / 15.3.
constexpr long PAST_CACHES = 4l << 20;

template <int D, bool FUSED>
hipError_t launch(DArgs A, int b, hipStream_t stream) {
  const int group = A.hq / A.hkv, gh = head_tile(group);
  A.group = group;
  A.htiles = (group + gh - 1) / gh;
  A.inv_splits = (u32)(((1ull << 32) + A.splits - 1) / A.splits);
  // Ranges last: XCDs, and the parts of one, take workgroups in turn, and where
  // every second or fourth has keys (a graph's cache that is not full) some
  // would get all of those.  us with ranges first / second / last: 32 heads on
  // 32, b 4, 200 keys of 500 9.6 / 8.4 / 7.2; 28 on 4, b 20 15.7 / 15.1 / 13.4.
  const dim3 grid(A.hkv * A.htiles, b, A.splits);
  const bool nt = (long)b * A.hkv * A.T * D * 4 >= PAST_CACHES;
  auto go = [&](auto heads, auto waves) {
    constexpr int G = decltype(heads)::value, NW = decltype(waves)::value;
    if (nt)
      hipLaunchKernelGGL((attn_decode_kernel<D, G, FUSED, NW, true>), grid,
                         dim3(NW * 64), 0, stream, A);
    else
      hipLaunchKernelGGL((attn_decode_kernel<D, G, FUSED, NW, false>), grid,
                         dim3(NW * 64), 0, stream, A);
    if (A.splits > 1 && A.tickets == nullptr)
      hipLaunchKernelGGL((attn_decode_merge<D, NW>), dim3(b * A.hq), dim3(64), 0,
                         stream, A);
  };
  constexpr std::integral_constant<int, 4> four{};
  if (gh == 1) go(std::integral_constant<int, 1>(), four);
  else if (gh == 2) go(std::integral_constant<int, 2>(), four);
  else if (gh == 4) go(four, four);
  else if (eight_waves(D, gh, b * A.hkv * A.htiles, A.T))
    go(std::integral_constant<int, 8>(), std::integral_constant<int, 8>());
  else
    go(std::integral_constant<int, 8>(), four);
  return hipGetLastError();
}

}  // namespace

// Key ranges a head for up to T keys.
int lfmq_attn_decode_splits(int b, int hq, int hkv, int T, int d) {
  const int group = hq / hkv, gh = head_tile(group);
  const int wgs = b * hkv * ((group + gh - 1) / gh);
  if (eight_waves(d, gh, wgs, T)) return max(1, (T + ONE_RANGE - 1) / ONE_RANGE);
  int n = FULL_WGS / max(wgs, 1);
  // (eight heads a workgroup: two of them a CU)
  if (gh < 8 && T > max(n, 1) * LONG_RANGE) n = MORE_WGS / max(wgs, 1);
  const int most = max(min((T + LEAST_KEYS - 1) / LEAST_KEYS, MANY),
                       (T + 2 * LEAST_KEYS - 1) / (2 * LEAST_KEYS));
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
                scale, 0, 0, 0};
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
                hkv, tmax, T, splits, scale, 0, 0, 0};
  return d == 128 ? launch<128, true>(A, b, stream)
                  : launch<64, true>(A, b, stream);
}
