// K3e/K4e — W4A16 / W8A16 product of one row of x with a large matrix:
// y[n] = dequant(W)[n, k] x[k] (+ bias) (+ residual), with the norm in front or
// the gate behind it.  The step of one sequence is mostly this.
//
// Bound by instructions more than by the read: a launch of these sizes that
// only reads takes 10.0 us for n 28672, k 4096, and the GEMV (dq_gemv.hip)
// takes 17.0 with weights that lie in the cache, 18.3 without.  So a wave
// keeps 2048 values of k for many rows of W, and what belongs to x (its sums,
// its squares, its order) is done once; int4 codes are taken as bf16 pairs 0 2,
// 4 6, 1 3, 5 7 of a dword, seven instructions for eight, and x is put in that
// order; the scales and zeros of the workgroup's rows come as one piece, first
// of all, into LDS; and four rows are summed over the lanes at once.  A row of
// W is read by KW waves, 1 or 2 KiB in a piece, four rows ahead.
//
// Loads wait by count: x, scales and weights are asked for in this order and
// without conditions (past an end the buffer's bounds give zeros), or the
// compiler waits for all of them at every turn.
//
// us a call, the GEMV, this one with conditions and now (4 bits; the last three 8):
//   n 28672, k 4096, norm and gate  18.3 / 13.1 / 12.8
//   n 4096, k 14336, residual       11.2 /  9.7 /  8.9
//   n 6144, k 4096, norm             6.6 /  6.4 /  5.8
//   n 4096, k 4096, residual         5.2 /      /  4.6
//   n 2048, k 8192                   6.2 /  5.5 /  4.9
//   n 32000, k 4096                 33.3 / 27.6 / 23.9
//   n 16384, k 2048, norm and gate       /  9.7 /  8.5
//   n 2048, k 8192                   8.0 /  7.1 /  6.3
// 8 bits, where a load took 16 of every 32 bytes and each line was asked for twice:
// 26.1 for n 32000, 9.3 for n 16384, 24.6 for n 28672, k 4096, norm and gate (21.7;
// the loads as they were, but by way of the caches 22.8).
// (a launch that only reads: 10.0 for n 28672, k 4096.)  Eight rows ahead: 15.4;
// 1024 workgroups: 14.8 (n 28672).
#include "dq_frag.h"

namespace {

constexpr int AHEAD = 4;                 // rows of W on their way; a group
constexpr int MOST = 8;                  // waves of a workgroup

struct Row {
  DqArgs A;
  int q, r;                              // groups of four rows of a workgroup:
                                         // q, or q + 1 of the first r
  int G, zw;
  int kw, cw;                            // waves along k, groups at a time
};

// sums over the 64 lanes of four values: in the n-th 16 lanes the n-th one's
__device__ __forceinline__ float sum4(float a, float b, float c, float d) {
  auto bits = [](float v) { return __builtin_bit_cast(u32, v); };
  auto value = [](u32 v) { return __builtin_bit_cast(float, v); };
  const auto p = __builtin_amdgcn_permlane32_swap(bits(a), bits(c), false, false);
  const u32 p0 = p[0], p1 = p[1];
  const auto q = __builtin_amdgcn_permlane32_swap(bits(b), bits(d), false, false);
  const u32 q0 = q[0], q1 = q[1];
  const auto r = __builtin_amdgcn_permlane16_swap(
      bits(value(p0) + value(p1)), bits(value(q0) + value(q1)), false, false);
  const u32 r0 = r[0], r1 = r[1];
  float v = value(r0) + value(r1);
#define LFMQ_ADD(ctrl)                                                        \
  v += value(__builtin_amdgcn_update_dpp(0, bits(v), ctrl, 0xf, 0xf, true))
  LFMQ_ADD(0xB1);                        // the neighbour
  LFMQ_ADD(0x4E);                        // the other two of four
  LFMQ_ADD(0x141);                       // eight, mirrored
  LFMQ_ADD(0x140);                       // sixteen, mirrored
#undef LFMQ_ADD
  return v;
}

// the lower four of eight lanes a, the upper ones b
__device__ __forceinline__ u32 own16(u32 a, u32 b) {
  return (u32)__builtin_amdgcn_update_dpp((int)a, (int)b, 0xE4, 0xf, 0xa, false);
}
// the same of the lane that mirrors this one in eight
__device__ __forceinline__ u32 mirrored16(u32 a, u32 b) {
  const int lo = __builtin_amdgcn_update_dpp((int)a, (int)a, 0x141, 0xf, 0x5, false);
  return (u32)__builtin_amdgcn_update_dpp(lo, (int)b, 0x141, 0xf, 0xa, false);
}

// block (64, KW, CW): KW waves along k, CW groups of rows at a time
template <int BITS, bool GATE>
__global__ __launch_bounds__(MOST * 64, 4) void dq_row_kernel(Row W) {
  const DqArgs& A = W.A;
  constexpr int WB = BITS / 4;                   // 16-byte pieces a lane
  constexpr int H = GATE ? 2 : 1, TC = 4 / H;    // columns of a group
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x, KW = W.kw, CW = W.cw;
  const int kw = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int cw = __builtin_amdgcn_readfirstlane(threadIdx.z);
  const int tid = (cw * KW + kw) * 64 + lane, T = KW * CW * 64;
  const bool rms = A.rms_eps >= 0.f;
  const int k = A.k, nout = A.n / H, G = W.G, zw = W.zw;
  const int bi = blockIdx.x, ga = bi * W.q + min(bi, W.r);
  const int ng = W.q + (bi < W.r ? 1 : 0);
  // columns of y, and of either half of W
  const int r0 = ga * TC, nr = min(ng * TC, nout - r0);

  // scales and zeros as they lie, [H][nr][G] and [H][nr][zw]
  const int sd = nr * G / 2, zd = nr * zw, all = H * (sd + zd);
  u32* meta = (u32*)smem;
  const unsigned short* ms = (const unsigned short*)smem;
  const u32* mz = meta + H * sd;
  float* part = (float*)(meta + all);            // [KW][ng][4]
  float* sqs = part + KW * ng * 4;               // [KW]
  const u32* S0 = (const u32*)(A.scales + (u64)r0 * G);
  const u32* Z0 = A.zeros + (u64)r0 * zw;
  // (selects, no branches, and a load for everybody: waits by count)
  auto meta_at = [&](int i) {
    const bool zero = i >= H * sd;
    i -= zero ? H * sd : 0;
    const int one = zero ? zd : sd;
    const u64 up = zero ? (u64)nout * zw : (u64)nout * G / 2;
    const u32* p = zero ? Z0 : S0;
    return p[GATE && i >= one ? up + (u64)(i - one) : (u64)i];
  };
  // this lane's 32 values of x: none past the end
  const int k0 = kw * 2048 + lane * 32;
  const bool in = k0 < k;
  const auto xr = make_rsrc(A.x, k * 2);
  u32x4 xv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    xv[i] = __builtin_amdgcn_raw_buffer_load_b128(xr, k0 * 2 + i * 16, 0, 0);
  constexpr int MQ = 4;
  u32 mq[MQ];
#pragma unroll
  for (int i = 0; i < MQ; ++i) mq[i] = meta_at(min(tid + i * T, all - 1));
  for (int i = tid + MQ * T; i < all; i += T) meta[i] = meta_at(i);
  // row j of group g, inside the workgroup's: gate, gate, up, up
  auto column = [&](int g, int j) { return g * TC + (GATE ? j & 1 : j); };
  const u32 pitch = k * BITS / 8;
  // 8 bits: a load takes whole lines of 128 bytes, by eight lanes; a lane has 16 of
  // its own 32 bytes and 16 of those of the lane that mirrors it
  const int l7 = lane & 7;
  const u32 byte = kw * 256 * BITS + (BITS == 4 ? lane * 16 : lane / 8 * 256);
  const u32 at[2] = {BITS == 4 ? 0u : (l7 < 4 ? 2 * l7 : 15 - 2 * l7) * 16u,
                     128 + (l7 < 4 ? 7 - 2 * l7 : 2 * l7 - 8) * 16u};
  u32x4 w[AHEAD][WB];
  // (past the last group nothing is read, but the load is there: where loads of
  // a loop depend on conditions the compiler waits for all of them)
  auto fetch = [&](int g, int j, u32x4 (&b)[WB]) {
    const u64 row = (u64)(r0 + min(column(g, j), nr - 1)) +
                    (GATE ? (u64)(j >> 1) * nout : 0);
    const auto rsrc = make_rsrc_uniform(A.w + row * pitch, g < ng ? pitch : 0);
#pragma unroll
    for (int i = 0; i < WB; ++i)
      b[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, byte + at[i], 0, 2);
  };
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) fetch(cw, j, w[j]);
#pragma unroll
  for (int i = 0; i < MQ; ++i)
    if (tid + i * T < all) meta[tid + i * T] = mq[i];

  float xs = 0.f, ss = 0.f;
  u32 xp[16];                                    // as the codes come
  float xf[BITS == 8 ? 32 : 1];
  if constexpr (BITS == 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        xs = dot2_bf16(0x3F803F80u, xv[i][e], xs);
        ss = dot2_bf16(xv[i][e], xv[i][e], ss);
      }
      const u32x4 d = __builtin_bit_cast(
          u32x4, deal8(__builtin_bit_cast(s16x8, xv[i])));
#pragma unroll
      for (int e = 0; e < 4; ++e) xp[i * 4 + e] = d[e];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      bf16x2_to_f32(xv[i >> 2][i & 3], xf[2 * i], xf[2 * i + 1]);
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      xs += xf[i];
      ss = fmaf(xf[i], xf[i], ss);
    }
  }
  if (rms && cw == 0) {
    const float v = wave_reduce_sum_dpp(ss);
    if (lane == 0) sqs[kw] = v;
  }
  const int gi = in ? (int)((u32)k0 / (u32)A.g) : 0;
  const int zi = gi / (32 / BITS), zs = gi % (32 / BITS) * BITS;
  __syncthreads();
  for (int g = cw; g < ng; g += CW) {
    float v[4];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      float c0 = 0.f, c1 = 0.f;
      if constexpr (BITS == 4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const u32x4 d =
              __builtin_bit_cast(u32x4, codes8_dealt(w[j][0][e]));
          c0 = dot2_bf16(d[0], xp[e * 4], c0);
          c1 = dot2_bf16(d[1], xp[e * 4 + 1], c1);
          c0 = dot2_bf16(d[2], xp[e * 4 + 2], c0);
          c1 = dot2_bf16(d[3], xp[e * 4 + 3], c1);
        }
      } else {
#pragma unroll
        for (int b = 0; b < WB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const u32 d = b == 0 ? own16(w[j][0][e], w[j][WB - 1][e])
                                 : mirrored16(w[j][0][e], w[j][WB - 1][e]);
            const float* x = xf + (b * 16 + e * 4) % (BITS == 8 ? 32 : 1);
            c0 = fmaf((float)(d & 0xFFu), x[0], c0);
            c1 = fmaf((float)((d >> 8) & 0xFFu), x[1], c1);
            c0 = fmaf((float)((d >> 16) & 0xFFu), x[2], c0);
            c1 = fmaf((float)(d >> 24), x[3], c1);
          }
      }
      // (above the products it would go to other registers, and be waited for)
      __builtin_amdgcn_sched_barrier(0);
      fetch(g + CW, j, w[j]);
      const int lr = min(column(g, j), nr - 1) + (GATE ? (j >> 1) * nr : 0);
      const float s = bf16_bits_to_f32(ms[lr * G + gi]);
      const u32 z = (mz[lr * zw + zi] >> zs) & ((1u << BITS) - 1);
      // the bits of 128 + z, and z
      const float zb = BITS == 4 ? __builtin_bit_cast(float, z << 16 | 0x43000000u)
                                 : (float)z;
      float t = s * fmaf(-zb, xs, c0 + c1);
      asm volatile("" : "+v"(t));                // a select, no branch
      v[j] = in ? t : 0.f;
    }
    const float t = sum4(v[0], v[1], v[2], v[3]);
    if ((lane & 15) == 0) part[(kw * ng + g) * 4 + (lane >> 4)] = t;
  }
  __syncthreads();
  float inv = 1.f;
  if (rms) {
    float s = 0.f;
    for (int i = 0; i < KW; ++i) s += sqs[i];
    inv = rsqrtf(s / (float)k + A.rms_eps);
  }
  for (int c = tid; c < nr; c += T) {
    const int p = GATE ? (c >> 1) * 4 + (c & 1) : c;
    float y = 0.f, u = 0.f;
    for (int i = 0; i < KW; ++i) {
      y += part[i * ng * 4 + p];
      if (GATE) u += part[i * ng * 4 + p + 2];
    }
    y *= inv;
    if constexpr (GATE) {
      y = silu_mul_f(y, u * inv);
    } else {
      if (A.bias != nullptr) y += bf16_bits_to_f32(A.bias[r0 + c]);
      if (A.resid != nullptr) y += bf16_bits_to_f32(A.resid[r0 + c]);
    }
    A.y[r0 + c] = (unsigned short)f32_to_bf16_bits_rne(y);
  }
}

template <int BITS, bool GATE>
hipError_t go(const DqArgs& A, hipStream_t stream) {
  constexpr int H = GATE ? 2 : 1, TC = 4 / H;
  const int groups = (int)ceil_div_u32(A.n / H, TC);
  const int G = A.k / A.g, zw = (G + 32 / BITS - 1) / (32 / BITS);
  const int KW = (int)ceil_div_u32(A.k, 2048);
  // Two workgroups of eight waves a CU, of four where they would not get a
  // group a wave (n 6144, k 4096: 6.4 us, 7.0) or a row is one wave's (n 16384,
  // k 2048: 6.9, 7.1; 8 bits 9.2, 10.0), with as many more of them
  int waves = MOST, wgs = 512;
  if (KW == 1) {
    waves = 4;
  } else if (KW <= 4 && groups < 512 * (MOST / KW)) {
    waves = 4;
    wgs = 1024;
  }
  const int CW = max(1, waves / KW);
  size_t lds;
  int grid;
  // (rows whose scales do not fit LDS: more workgroups)
  for (;; wgs *= 2) {
    grid = min(wgs, (int)ceil_div_u32(groups, CW));
    const size_t ng = ceil_div_u32(groups, grid);
    lds = (ng * 4 * (G / 2 + zw) + KW * ng * 4 + KW) * 4;
    if (lds <= 64 * 1024 || wgs >= groups) break;
  }
  if (lds > 64 * 1024) return hipErrorInvalidValue;
  const Row W{A, groups / grid, groups % grid, G, zw, KW, CW};
  hipLaunchKernelGGL((dq_row_kernel<BITS, GATE>), dim3(grid), dim3(64, KW, CW),
                     lds, stream, W);
  return hipGetLastError();
}

}  // namespace

// Up to eight waves along k; an even number of groups, each a lane's values or
// more.  Smaller matrices are the GEMV's, us of both: n 2048, k 2048 3.4 / 3.4, n
// 1024, k 4096 3.4 / 3.4 (from there on this one: n 3072, k 2048 3.7 / 3.5, n 1024, k
// 8192 5.2 / 3.7, n 4096, k 2048 with norm and gate 5.0 / 3.8).
bool lfmq_dq_row_ok(int n, int k, int g) {
  return n >= 1 && k <= MOST * 2048 && g % 32 == 0 && k % (2 * g) == 0 &&
         (long)n * k >= 4l << 20;
}

// rms_eps >= 0: x over its root mean square; glu: y [n / 2] = silu(gate) up of
// W = [gate | up], without bias and residual
hipError_t lfmq_dq_row(const void* qweight, const void* scales,
                       const void* qzeros, const void* x, void* y,
                       const void* bias, const void* resid, int n, int k, int g,
                       int bits, float rms_eps, bool glu, hipStream_t stream) {
  if (!lfmq_dq_row_ok(n, k, g) || (glu && n % 2)) return hipErrorInvalidValue;
  const DqArgs A{(const char*)qweight, (const unsigned short*)scales,
                 (const u32*)qzeros, (const unsigned short*)x,
                 (unsigned short*)y, (const unsigned short*)bias,
                 (const unsigned short*)resid, nullptr, 1, n, k, g, 1, nullptr,
                 nullptr, nullptr, rms_eps};
  if (bits == 4) return glu ? go<4, true>(A, stream) : go<4, false>(A, stream);
  if (bits == 8) return glu ? go<8, true>(A, stream) : go<8, false>(A, stream);
  return hipErrorInvalidValue;
}
