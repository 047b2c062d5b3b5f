// K3d/K4d — W4A16 / W8A16 product of up to 16 rows of x with many columns:
// y[m, n] = x[m, k] · dequant(W)[n, k]^T (+ bias) (+ residual), with the norm
// in front or the gate behind it, or by expert (dq_frag.h).
//
// A workgroup keeps its operands of x in registers and walks over tiles of 16
// columns (of 8 and their gates): its waves share k, a wave holds 256 values of
// k of every row (and reads others only where k is longer than 4096), so that
// x, its sums and its squares cost one pass a workgroup and not one a tile.
// The scales and zeros of the tiles lie in one piece and come by whole lines
// first of all; fetched a lane at a time they were as many requests as the
// weights (loads alone 16 us instead of 13 at n 28672, k 4096).  The sums of
// the waves meet in LDS after the last tile.
//
// Bound by the instructions that unpack the weights, which run beside the
// reads only as far as the waves are out of step, and by the first loads and
// the last sums, which nothing covers.  us a call, dq_rows and this one (4
// bits but for the last):
//                                   2 rows       8 rows       16 rows
//   n 28672, k 4096, norm, gate   21.5 / 16.0  25.0 / 17.2  30.2 / 18.4
//   n 6144, k 4096, norm           8.9 /  7.6   9.4 /  8.7  10.8 / 10.0
//   n 2048, k 2048, residual       4.9 /  4.1   5.5 /  4.9   6.3 /  5.6
//   n 16384, k 2048, norm, gate    9.8 /  8.3  10.4 /  9.3  11.4 / 10.5
//   n 32000, k 4096 (8 bits)      31.0 / 26.2  34.5 / 27.0  40.5 / 27.3
// 8 experts of n 28672, k 4096 and n 4096, k 14336, one to four rows each:
// 130.6 -> 110.8, 72.5 -> 70.9.  Two steps of weights in flight a wave: 17.1
// us instead of 16.9 at 8 rows; eight waves with twice the k 17.9; batches of
// tiles whose sums are taken during the next batch: registers spill, 20 % slower.
// (Groups of 64 with k above 4096 spill 2 to 20 registers: ext.hip's rules were
// measured with that.)
//
// Where k is longer than a workgroup's 4096, it may also be shared by workgroups of
// which the last one to end adds up: a merge by way of memory costs 2 to 3 us, one
// part after the other of a tile more from some 50 million weights on.  us a call,
// dq_rows or several steps a workgroup, and in parts (4 bits; 5120 x 17408 of 8 bits):
//                                   3 rows       8 rows       16 rows
//   n 4096, k 14336               13.6 / 13.5  16.4 / 14.4  18.7 / 15.7
//   n 6144, k 8192                12.3 / 11.2  13.9 / 12.2  16.7 / 13.4
//   n 5120, k 17408               26.1 / 19.0  33.3 / 20.3  27.3 / 21.7
//   n 5120, k 17408 (8 bits)      37.6 / 25.3  45.5 / 26.4  35.5 / 28.0
#include "dq_frag.h"

int lfmq_dq_wide_part_blocks(int n, int parts);

namespace {

constexpr int KS = 256;                  // values of k of a wave and step
constexpr int MAX_TILES = 8;             // of a workgroup
constexpr int MOST_PARTS = 5;            // of k

struct Wide {
  DqArgs A;
  int q, r;                              // tiles of a workgroup: q, or q + 1
                                         // of the first r
  int G, zw, steps;                      // groups, words of zeros; steps of k
  u32* tickets;                          // PARTS: a counter a workgroup, zero
};

// A partial result, past the caches of the XCD: a workgroup of another one may be
// the reader.
__device__ __forceinline__ void put4(float* p, f32x4 v) {
  typedef __attribute__((address_space(1))) u64 gu64;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float a = v[2 * i], b = v[2 * i + 1];
    __hip_atomic_store((gu64*)p + i,
                       (u64)__builtin_bit_cast(u32, b) << 32 |
                           __builtin_bit_cast(u32, a),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}
__device__ __forceinline__ f32x4 get4(const float* p) {
  typedef __attribute__((address_space(1))) u64 gu64;
  f32x4 v;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const u64 b = __hip_atomic_load((gu64*)p + i, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
    v[2 * i] = __builtin_bit_cast(float, (u32)b);
    v[2 * i + 1] = __builtin_bit_cast(float, (u32)(b >> 32));
  }
  return v;
}

__host__ __device__ __forceinline__ int lanes_of(int rows) {
  return rows <= 4 ? 16 : (rows <= 8 ? 32 : 64);
}

// MORE: more than one step of k.  LINES: a load takes a whole 128-byte line of eight
// rows of W, past the caches: pieces of two chunks (PAIR), or the halves of one;
// lanes of the two eights exchange theirs on the way into the operands.  PARTS: k is
// shared by A.splits workgroups, of which the last one to end adds up.
template <int BITS, int KC, DqMode MODE, bool MORE, int NW, bool LINES, bool PARTS>
__global__ __launch_bounds__(NW * 64, 4) void dq_wide_kernel(Wide W) {
  const DqArgs& A = W.A;
  constexpr int TPB = NW * 64;
  constexpr int J = KC / 32, S = KS / KC;        // products, chunks
  constexpr int UW = BITS / 4, WD = J * UW;      // dwords of 8 codes, a chunk
  constexpr int H = MODE == GLU ? 2 : 1, TC = 16 / H;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15, l4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int row0 = 0, rows = A.m, expert = 0;
  if (MODE != DENSE && A.tiles != nullptr) {
    expert = A.tiles[3 * blockIdx.y];
    if (expert < 0) return;
    row0 = A.tiles[3 * blockIdx.y + 1];
    rows = A.tiles[3 * blockIdx.y + 2];
  }
  const bool rms = MODE != SLOTS && A.rms_eps >= 0.f;
  const int nout = A.n / H, G = W.G, zw = W.zw;
  // (parts end with a line, two chunks)
  const int c0 = PARTS ? A.k / KC / 2 * (int)blockIdx.y / A.splits * 2 : 0;
  const int C = PARTS ? A.k / KC / 2 * (int)(blockIdx.y + 1) / A.splits * 2
                      : A.k / KC;
  const int bi = blockIdx.x, ta = bi * W.q + min(bi, W.r);
  const int nt = W.q + (bi < W.r ? 1 : 0);
  // rows of W of this workgroup: r0 .. (GLU: of either half)
  const int r0 = ta * TC, nr = min(nt * TC, nout - r0);
  const int sd = nr * G / 2, zd = nr * zw, all = H * (sd + zd);
  const u64 first = (u64)expert * A.n;

  // scales and zeros as they lie, [H][nr][G] and [H][nr][zw]
  u32* meta = (u32*)smem;
  const unsigned short* ms = (const unsigned short*)smem;
  const u32* mz = meta + H * sd;
  const u32* S0 = (const u32*)(A.scales + (first + r0) * G);
  const u32* Z0 = A.zeros + (first + r0) * zw;
  auto meta_at = [&](int i) {
    if (i < H * sd)
      return H == 2 && i >= sd ? S0[(u64)nout * G / 2 + i - sd] : S0[i];
    i -= H * sd;
    return H == 2 && i >= zd ? Z0[(u64)nout * zw + i - zd] : Z0[i];
  };
  constexpr int MQ = 48 / NW;
  u32 mq[MQ];
#pragma unroll
  for (int i = 0; i < MQ; ++i)
    if (tid + i * TPB < all) mq[i] = meta_at(tid + i * TPB);
  for (int i = tid + MQ * TPB; i < all; i += TPB) meta[i] = meta_at(i);

  // rows past the last one repeat it
  int xr = row0 + min(l15, rows - 1);
  if (MODE != DENSE && A.src != nullptr) xr = A.src[xr];
  // halves of a chunk: its values of x are read in that order
  constexpr bool PAIR = LINES && WD == 4, HALVES = LINES && WD == 8;
  static_assert(!LINES || PAIR || HALVES, "");
  constexpr int XP = HALVES ? 16 : KC / 4;         // values of x in a piece
  const char* xp = (const char*)A.x + ((u64)xr * A.k + l4 * XP) * 2;
  auto chunk = [&](int p) { return c0 + (p * NW + wave) * S; };
  s16x8 xq[S][J];
  auto fetch_x = [&](int p) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int c = min(chunk(p) + s, C - 1);
#pragma unroll
      for (int j = 0; j < J; ++j)
        xq[s][j] = *(const s16x8*)(
            xp + (u32)(c * KC + (HALVES ? j / 2 * 64 + j % 2 * 8 : j * 8)) * 2);
    }
  };
  // this lane's row of W in tile t, from r0 on (GLU: gate, then up)
  auto local = [&](int t) {
    return min(t * TC + (H == 2 ? l15 & 7 : l15), nr - 1);
  };
  const u64 wrow = (u64)A.k * BITS / 8;
  const int l7 = l15 & 7, odd = l15 >> 3;
  const char* wp = A.w + (first + r0 + (H == 2 && !LINES ? odd * nout : 0)) * wrow +
                   l4 * (LINES ? 16 : WD * 4) + (HALVES ? odd * 64 : 0);
  u32 w[S][WD];                          // LINES: of rows l7, then of l7 + 8
  auto fetch_w = [&](int p, int t) {
    if constexpr (LINES) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const char* row =
            wp + (u64)(min(t * TC + (H == 2 ? l7 : h * 8 + l7), nr - 1) +
                       (H == 2 ? h * nout : 0)) * wrow;
#pragma unroll
        for (int s = 0; s < (PAIR ? S / 2 : S); ++s) {
          const int c = min(chunk(p) + (PAIR ? 2 * s + odd : s), C - 1);
          const u32x4 v = __builtin_nontemporal_load(
              (const u32x4*)(row + (u32)c * (KC * BITS / 8)));
#pragma unroll
          for (int e = 0; e < 4; ++e)
            w[PAIR ? 2 * s + h : s][(PAIR ? 0 : h * 4) + e] = v[e];
        }
      }
    } else {
      const char* row = wp + local(t) * wrow;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const u32* a = (const u32*)(
            row + (u32)min(chunk(p) + s, C - 1) * (KC * BITS / 8));
        if constexpr (WD >= 4) {
#pragma unroll
          for (int i = 0; i < WD / 4; ++i) {
            const u32x4 v = ((const u32x4*)a)[i];
#pragma unroll
            for (int e = 0; e < 4; ++e) w[s][i * 4 + e] = v[e];
          }
        } else {
#pragma unroll
          for (int e = 0; e < WD; ++e) w[s][e] = a[e];
        }
      }
    }
  };
  // this lane's row's dword e of chunk s
  auto word = [&](int s, int e) {
    if constexpr (!LINES) return w[s][e];
    const bool hi = PAIR ? s & 1 : e >= 4;
    const u32 x = PAIR ? w[s & ~1][e] : w[s][e & 3];
    const u32 y = PAIR ? w[s | 1][e] : w[s][e | 4];
    return hi ? other8<false>(y, x) : other8<true>(x, y);
  };
  fetch_x(0);
  fetch_w(0, 0);
#pragma unroll
  for (int i = 0; i < MQ; ++i)
    if (tid + i * TPB < all) meta[tid + i * TPB] = mq[i];

  // sums: of the lanes that hold rows, [nt][NW][lanes]
  const int lanes = lanes_of(rows);
  f32x4* red = (f32x4*)(smem + ((all * 4 + 15) & ~15));
  float* sqs = (float*)(red + nt * NW * lanes);          // [NW][16]
  const s16x8 ones = bf16_ones();
  s16x8 xf[S][J];
  f32x4 xs[S], sq = {0.f, 0.f, 0.f, 0.f};
  for (int p = 0; p < (MORE ? W.steps : 1); ++p) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      xs[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < J; ++j)
        xf[s][j] = BITS == 4 ? deal8(xq[s][j]) : xq[s][j];
      if (chunk(p) + s < C) {
#pragma unroll
        for (int j = 0; j < J; ++j)
          xs[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[s][j], ones, xs[s],
                                                          0, 0, 0);
        if (rms)
#pragma unroll
          for (int j = 0; j < J; ++j)
            sq = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[s][j], xf[s][j], sq,
                                                         0, 0, 0);
      }
    }
    if (p == 0) __syncthreads();                         // meta is there
    if (MORE && p + 1 < W.steps) fetch_x(p + 1);
    for (int t = 0; t < nt; ++t) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      f32x4* mine = red + (t * NW + wave) * lanes + lane;
      if (MORE && p > 0 && lane < lanes) acc = *mine;
      const int lr = local(t) + (H == 2 ? (l15 >> 3) * nr : 0);
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int c = chunk(p) + s;
        if (c < C) {
          f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int j = 0; j < J; ++j) {
            const u32 two[2] = {word(s, j * UW), word(s, j * UW + UW - 1)};
            const s16x8 b = BITS == 4 ? codes8_dealt(two[0]) : codes8<BITS>(two);
            a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[s][j], b, a, 0, 0, 0);
          }
          const float sc = bf16_bits_to_f32(ms[lr * G + c]);
          const float sz =
              sc * zero_bias<BITS>(mz[lr * zw + c / (32 / BITS)], c);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[e] = fmaf(-sz, xs[s][e], fmaf(sc, a[e], acc[e]));
        }
      }
      if (t + 1 < nt) fetch_w(p, t + 1);
      else if (MORE && p + 1 < W.steps) fetch_w(p + 1, 0);
      if (lane < lanes) *mine = acc;
    }
  }
  if (rms) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (l15 == l4 * 4 + e) sqs[wave * 16 + l15] = sq[e];
  }
  __syncthreads();
  // a wave a tile: column l15, rows l4 * 4 + e
  if (!PARTS && wave >= nt) return;
  float inv = 1.f;                                       // of row l15
  if (rms) {
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) v += sqs[i * 16 + l15];
    inv = rsqrtf(v / (float)A.k + A.rms_eps);
  }
  const int t = wave;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (lane < lanes && (!PARTS || t < nt)) {
#pragma unroll
    for (int i = 0; i < NW; ++i) v += red[(t * NW + i) * lanes + lane];
  }
  if constexpr (PARTS) {
    // As the decode attention's merge: results are written through to where the
    // workgroup that adds up reads, every wave waits for its own, and the barrier
    // stands before the ticket, which is put back to zero.
    float* part = A.part + ((u64)(ta + t) * A.splits * 64 + lane) * 4;
    if (t < nt && lane < lanes) put4(part + blockIdx.y * 256, v);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* last_s = (int*)smem;              // (scales, read)
    typedef __attribute__((address_space(1))) unsigned gu32;
    gu32* ticket = (gu32*)(W.tickets + blockIdx.x);
    if (tid == 0) {
      const unsigned old = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
      *last_s = (int)old == A.splits - 1;
      if (*last_s)
        __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!*last_s || t >= nt) return;
    f32x4 all[MOST_PARTS];
    const bool on = lane < lanes;
#pragma unroll
    for (int i = 0; i < MOST_PARTS; ++i)
      if (i < A.splits && on) all[i] = get4(part + i * 256);
    v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < MOST_PARTS; ++i)
      if (i < A.splits && on) v += all[i];
  }
  const int col = (ta + t) * TC + (H == 2 ? l15 & 7 : l15);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = l4 * 4 + e;
    float y = v[e];
    if (rms) y *= __shfl(inv, row, 64);
    if (MODE == GLU)
      y = silu_mul_f(y, __shfl(y, (lane & 48) | 8 | (l15 & 7), 64));
    if (row >= rows || col >= nout || (H == 2 && l15 >= 8)) continue;
    const u64 at = (u64)(row0 + row) * nout + col;
    if (MODE == SLOTS) {
      A.y32[at] = y;
      continue;
    }
    if (MODE == DENSE) {
      if (A.bias != nullptr) y += bf16_bits_to_f32(A.bias[col]);
      if (A.resid != nullptr) y += bf16_bits_to_f32(A.resid[at]);
    }
    A.y[at] = (unsigned short)f32_to_bf16_bits_rne(y);
  }
}

static_assert(MAX_TILES <= 8, "a wave ends a tile");

size_t lds_bytes(int nt, int rows, int G, int zw, int NW) {
  return (size_t)nt * 16 * (G * 2 + zw * 4) + 16 +
         (size_t)nt * NW * lanes_of(rows) * 16 + NW * 64;
}

int words_of(int G, int bits) { return (G + 32 / bits - 1) / (32 / bits); }

// waves of a workgroup, and the LDS that it may take of a CU's
int waves_of(int k) { return k <= 8 * KS ? 8 : 16; }
size_t room_of(int NW) { return 160 * 1024 / (16 / NW); }

// rows: the most that a tile of rows has; lists: tiles of rows
template <int BITS, int KC, DqMode MODE, bool MORE, int NW, bool LINES = false>
hipError_t go(const DqArgs& A, int rows, int lists, hipStream_t stream) {
  constexpr int TC = MODE == GLU ? 8 : 16;
  const int tiles = (int)ceil_div_u32(MODE == GLU ? A.n / 2 : A.n, TC);
  const int G = A.k / KC, zw = words_of(G, BITS);
  const size_t room = room_of(NW);
  // Tiles of a workgroup, whose scales and sums lie in LDS: what takes the
  // fewest rounds of workgroups that run at once, a round as long as its tiles
  // and about two more.  (4 experts, n 28672, k 4096: 3.5 rounds of 8 tiles 61.1
  // us, 4 of 7 56.9; n 4096, k 14336 with 9 lists of rows, 2 rounds of 7 72.3,
  // 3 of 4 59.8.)
  const long once = 256l * (16 / NW);
  int nt = 0;
  long least = 0;
  for (int i = 1; i <= MAX_TILES; ++i) {
    if (lds_bytes(i, rows, G, zw, NW) > room) break;
    const long wgs = (long)ceil_div_u32(tiles, i) * lists;
    const long cost = (wgs + once - 1) / once * (i + 2);
    if (nt == 0 || cost <= least) {
      nt = i;
      least = cost;
    }
  }
  if (nt == 0) return hipErrorInvalidValue;
  const int grid = (int)ceil_div_u32(tiles, nt);
  const auto kernel = dq_wide_kernel<BITS, KC, MODE, MORE, NW, LINES, false>;
  static bool set = false;
  if (!set) {
    LFMQ_CHECK_HIP(hipFuncSetAttribute(
        (const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
        (int)room));
    set = true;
  }
  const Wide W{A, tiles / grid, tiles % grid, G, zw,
               (int)ceil_div_u32(A.k, NW * KS), nullptr};
  hipLaunchKernelGGL(kernel, dim3(grid, lists), dim3(NW * 64),
                     lds_bytes((int)ceil_div_u32(tiles, grid), rows, G, zw, NW),
                     stream, W);
  return hipGetLastError();
}

template <int BITS, int KC, DqMode MODE>
hipError_t go_k(const DqArgs& A, int rows, int lists, hipStream_t stream) {
  // Whole lines from 8 MiB on: below, the exchange costs more.  us by 64 bytes of 16
  // rows / by lines: n 28672, k 4096 (4 bits, norm and gate, 16 rows) 18.8 / 18.7, n
  // 6144, k 4096 (12 MiB) 10.3 / 10.0, n 4096, k 4096 (8) 8.8 / 8.7; n 32000, k 4096 (8
  // bits, groups of 128) 30.4 / 27.3, n 16384, k 2048 (32 MiB) 13.4 / 13.1; n 3072, k
  // 2048 (6, 2 rows) 5.1 / 5.3.  With more steps there is no room for it (n 10240, k
  // 8192, 4 bits 15.4 / 16.3); 4 bits in groups of 64 have 32 bytes a chunk; and an
  // expert's second tile of rows reads again what the first one has read (8 experts, 120
  // rows, n 28672, k 4096 164 / 170).
  if constexpr (BITS * KC >= 512 && MODE != SLOTS) {
    if (A.tiles == nullptr && (u64)A.n * A.k * BITS / 8 >= 8u << 20) {
      if (A.k <= 8 * KS)
        return go<BITS, KC, MODE, false, 8, true>(A, rows, lists, stream);
      if (A.k <= 16 * KS)
        return go<BITS, KC, MODE, false, 16, true>(A, rows, lists, stream);
    }
  }
  if (A.k <= 8 * KS) return go<BITS, KC, MODE, false, 8>(A, rows, lists, stream);
  if (A.k <= 16 * KS)
    return go<BITS, KC, MODE, false, 16>(A, rows, lists, stream);
  return go<BITS, KC, MODE, true, 16>(A, rows, lists, stream);
}

// column tiles of a workgroup where k is in parts of up to 4096: a workgroup a CU, and
// no second round of a few (n 8176, k 8960, 3 rows: 258 of 6 tiles 23.6 us, in one
// launch without parts 15.2)
int part_tiles(int n, int parts) {
  const u32 tiles = ceil_div_u32(n, 16);
  u32 nt = ceil_div_u32(tiles * parts, 256);
  while (ceil_div_u32(tiles, nt) * parts > 256) ++nt;
  return (int)nt;
}

template <int BITS, int KC>
hipError_t go_parts(const DqArgs& A, void* tickets, hipStream_t stream) {
  constexpr int NW = 16;
  constexpr bool LINES = BITS * KC >= 512;
  const int tiles = (int)ceil_div_u32(A.n, 16), G = A.k / KC, zw = words_of(G, BITS);
  const int grid = lfmq_dq_wide_part_blocks(A.n, A.splits);
  const size_t lds = lds_bytes((int)ceil_div_u32(tiles, grid), A.m, G, zw, NW);
  const auto kernel = dq_wide_kernel<BITS, KC, DENSE, false, NW, LINES, true>;
  static bool set = false;
  if (!set) {
    LFMQ_CHECK_HIP(hipFuncSetAttribute(
        (const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
        (int)room_of(NW)));
    set = true;
  }
  const Wide W{A, tiles / grid, tiles % grid, G, zw, 1, (u32*)tickets};
  hipLaunchKernelGGL(kernel, dim3(grid, A.splits), dim3(NW * 64), lds, stream, W);
  return hipGetLastError();
}

template <DqMode MODE>
hipError_t go_bits(const DqArgs& A, int bits, int rows, int lists,
                   hipStream_t stream) {
  if (bits == 4)
    return A.g == 128 ? go_k<4, 128, MODE>(A, rows, lists, stream)
                      : go_k<4, 64, MODE>(A, rows, lists, stream);
  if (bits == 8)
    return A.g == 128 ? go_k<8, 128, MODE>(A, rows, lists, stream)
                      : go_k<8, 64, MODE>(A, rows, lists, stream);
  return hipErrorInvalidValue;
}

}  // namespace

// groups of 64 or 128, an even number of them, and as many as LDS holds the
// scales of for a tile of columns (16 rows, groups of 64: k up to 233 000 with 4
// bits, 194 000 with 8)
bool lfmq_dq_wide_ok(int m, int n, int k, int g, int bits) {
  return m >= 1 && m <= 16 && n >= 1 && (g == 64 || g == 128) &&
         k % (2 * g) == 0 && (bits == 4 || bits == 8) &&
         lds_bytes(1, m, k / g, words_of(k / g, bits), waves_of(k)) <=
             room_of(waves_of(k));
}

// as lfmq_dq_rows, without splits of k
hipError_t lfmq_dq_wide(const void* qweight, const void* scales,
                        const void* qzeros, const void* x, void* y,
                        const void* bias, const void* resid, int m, int n,
                        int k, int g, int bits, float rms_eps, bool glu,
                        hipStream_t stream) {
  if (!lfmq_dq_wide_ok(m, n, k, g, bits) || (glu && n % 2))
    return hipErrorInvalidValue;
  const DqArgs A{(const char*)qweight, (const unsigned short*)scales,
                 (const u32*)qzeros, (const unsigned short*)x,
                 (unsigned short*)y, (const unsigned short*)bias,
                 (const unsigned short*)resid, nullptr, m, n, k, g, 1, nullptr,
                 nullptr, nullptr, rms_eps};
  return glu ? go_bits<GLU>(A, bits, m, 1, stream)
             : go_bits<DENSE>(A, bits, m, 1, stream);
}

// Workgroups of a part of k.
int lfmq_dq_wide_part_blocks(int n, int parts) {
  return (int)ceil_div_u32(ceil_div_u32(n, 16), part_tiles(n, parts));
}

// Parts of k of a product that one launch does in parts; 0: it does not.
int lfmq_dq_wide_parts(int m, int n, int k, int g, int bits) {
  const int parts = (int)ceil_div_u32(k, 16 * KS);
  if (parts < 2 || parts > MOST_PARTS || !lfmq_dq_wide_ok(m, n, k, g, bits)) return 0;
  const int nt = part_tiles(n, parts), G = k / g;
  return nt <= MAX_TILES &&
                 lds_bytes(nt, m, G, words_of(G, bits), 16) <= room_of(16)
             ? parts
             : 0;
}

// as lfmq_dq_wide, without a norm; part: [n / 16, rounded up][parts][256] floats of
// scratch memory; tickets: a zero a workgroup of a part, which no other launch uses
// meanwhile, and zeros again afterwards
hipError_t lfmq_dq_wide_in_parts(const void* qweight, const void* scales,
                                 const void* qzeros, const void* x, void* y,
                                 const void* bias, const void* resid, void* part,
                                 void* tickets, int m, int n, int k, int g, int bits,
                                 hipStream_t stream) {
  const int parts = lfmq_dq_wide_parts(m, n, k, g, bits);
  if (parts == 0 || part == nullptr || tickets == nullptr)
    return hipErrorInvalidValue;
  const DqArgs A{(const char*)qweight, (const unsigned short*)scales,
                 (const u32*)qzeros, (const unsigned short*)x,
                 (unsigned short*)y, (const unsigned short*)bias,
                 (const unsigned short*)resid, (float*)part, m, n, k, g, parts,
                 nullptr, nullptr, nullptr};
  if (bits == 4)
    return g == 128 ? go_parts<4, 128>(A, tickets, stream)
                    : go_parts<4, 64>(A, tickets, stream);
  return g == 128 ? go_parts<8, 128>(A, tickets, stream)
                  : go_parts<8, 64>(A, tickets, stream);
}

// as lfmq_dq_rows_experts
hipError_t lfmq_dq_wide_experts(const void* qweight, const void* scales,
                                const void* qzeros, const void* x,
                                const void* src, const void* tiles, void* y,
                                int n_tiles, int n, int k, int g, int bits,
                                bool glu, hipStream_t stream) {
  if (!lfmq_dq_wide_ok(16, n, k, g, bits) || (glu && n % 2) || n_tiles < 1)
    return hipErrorInvalidValue;
  DqArgs A{};
  A.w = (const char*)qweight;
  A.scales = (const unsigned short*)scales;
  A.zeros = (const u32*)qzeros;
  A.x = (const unsigned short*)x;
  A.y = (unsigned short*)y;
  A.y32 = (float*)y;
  A.src = (const i32*)src;
  A.tiles = (const i32*)tiles;
  A.m = 16;
  A.n = n;
  A.k = k;
  A.g = g;
  A.splits = 1;
  return glu ? go_bits<GLU>(A, bits, 16, n_tiles, stream)
             : go_bits<SLOTS>(A, bits, 16, n_tiles, stream);
}
