// K1 — GPTQ Hessian accumulate: H += 2·XᵀX (X bf16 [t, k], H fp32 [k, k]).
//
// Both operands of a product are columns of X, consecutive tokens a lane.
// Rows of X go from memory straight into LDS as they are, and the transposing
// LDS read (16 lanes get the 16 columns of a 4 x 16 block) makes operands of
// them.  H is symmetric but for what it held before: only tiles on and below
// the diagonal are computed, and each is added to its own place and to its
// mirror image.
//
// A workgroup = 128 x 128, 4 waves of 64 x 64, tokens in steps of 64 through
// two LDS buffers.  Tiles run in blocks of 4 x 4, a range of blocks to an XCD,
// whose L2 then serves a row of tiles four times (8 x 8 leave more of the
// triangle's edge empty: 102 x 7416 99 us, 82 so).
//
// Where H is large its traffic is as long as the products (128 x 14336: 346 us
// at 4.8 TB/s; the products of 2048 x 14336 alone: 465), and the two overlap
// only as far as a workgroup's loads are under way before it needs them and
// leave X in the L2.  So elements of the tile's own place load beside the last
// step, those of the mirror while the result goes through LDS, and H
// passes by the caches where its rows are whole lines.  2048 x 14336: 673 us
// with H read after the products, 629 with loads ahead, 545 past the caches
// too (772 TFLOP/s of the half computed); 512 x 8192: 122 and 100;
// 2048 x 4096: 78 and 65; 2048 x 2048: 33, 64 x 512: 7.9 (one round of
// workgroups, below).  Matrix cores are busy 40 % of the time, memory 65 %:
// two workgroups of one wave a SIMD each hide no more of each other.
#include "lds_dma.h"

namespace {

constexpr int TPB = 256, NW = 4;
constexpr int BC = 128, BK = 64;             // tile side, tokens a step
constexpr int SB = 4;                        // tiles a side of a block
constexpr int BUF = 2 * BC * BK * 2;         // both operands of a step
constexpr int LD = BC + 1;                   // of the result in LDS

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;

// a step's operand in LDS: [BK tokens][BC columns], 32-byte chunks of a row
// (16 columns) XOR-swizzled by the token so that the four tokens of a
// transposing read, and those of neighbouring lane groups, use other banks
__device__ __forceinline__ int chunk_key(int token) {
  return (token & 7) ^ ((token >> 1) & 4);
}

// How H is read and written.  DIRECT: a single round of workgroups, one a CU, which
// wait for memory once, straight from the fragments, with registers for all of a
// thread's elements (64 x 512 with clearing H: 9.6 us, 11.0 row by row in half the
// registers; 478 x 1616 21.8, 23.3).  WHOLE: more workgroups, rows of H whole lines, past the caches.
// CACHED: the same where neighbouring tiles share lines, which then have to
// meet in a cache (102 x 7416: 81 us, 107 past it).
enum Way { DIRECT, WHOLE, CACHED };

template <Way WAY>
__global__ __launch_bounds__(TPB, WAY == DIRECT ? 1 : 2) void hessian_kernel(
    const unsigned short* __restrict__ x, float* h, int t, int k) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // block (bi, bj) of the lower triangle, tile (r, c) of it
  const u32 id = xcd_swizzle(blockIdx.x, gridDim.x);
  const u32 blk = id / (SB * SB);
  u32 bi = (u32)((sqrtf(8.f * blk + 1.f) - 1.f) * 0.5f);
  while (bi * (bi + 1) / 2 > blk) --bi;
  while ((bi + 1) * (bi + 2) / 2 <= blk) ++bi;
  bi = __builtin_amdgcn_readfirstlane(bi);   // the root is a vector operation
  const u32 bj = blk - bi * (bi + 1) / 2;
  const int ti = bi * SB + id / SB % SB, tj = bj * SB + id % SB;
  const int i0 = ti * BC, j0 = tj * BC;
  if (tj > ti || i0 >= k) return;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wi = wave >> 1, wj = wave & 1;
  const int l15 = lane & 15, l4 = lane >> 4;
  // staging: a wave's load fills 4 tokens of 256 bytes; tokens past the end
  // repeat the last one and are cleared below, columns past k are not stored
  constexpr int NL = BC * BK * 2 / 1024 / NW;          // loads an operand
  u32 ci[NL], cj[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int tok = (i * NW + wave) * 4 + (lane >> 4);
    const int c = (((lane & 15) >> 1) ^ chunk_key(tok)) * 16 + (lane & 1) * 8;
    ci[i] = (i0 + c < k ? c : 0) * 2;
    cj[i] = (j0 + c < k ? c : 0) * 2;
  }
  auto stage = [&](int t0, int buf) {
    const unsigned short* a = x + (u64)t0 * k + i0;
    const unsigned short* b = x + (u64)t0 * k + j0;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int tok = (i * NW + wave) * 4 + (lane >> 4);
      const u32 row = (u32)min(tok, t - 1 - t0) * (u32)(k * 2);
      load_to_lds(a, row + ci[i], buf * BUF + (i * NW + wave) * 1024);
      load_to_lds(b, row + cj[i], buf * BUF + BUF / 2 + (i * NW + wave) * 1024);
    }
  };
  // operand: 8 tokens of column c * 16 + l15, in two reads of four
  auto frag = [&](const char* buf, int ks, int c) {
    s16x8 f;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int tok = ks * 32 + l4 * 8 + e * 4 + (l15 >> 2);
      const char* p = buf + tok * (BC * 2) + ((c ^ chunk_key(tok)) << 5) +
                      (l15 & 3) * 8;
      const s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
#pragma unroll
      for (int i = 0; i < 4; ++i) f[e * 4 + i] = v[i];
    }
    return f;
  };
  // rows of a tile of H in fours of a thread: 512 bytes of a row together
  constexpr int NF = BC * BC / 4 / TPB;
  const int c4 = tid % (BC / 4) * 4, r0 = tid / (BC / 4);
  auto fours_load = [&](f32x4 (&v)[NF], int row0, int col0) {
    const float* p = h + (u64)row0 * k + min(col0 + c4, k - 4);
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      const int r = min(r0 + e * (TPB * 4 / BC), k - 1 - row0);
      const f32x4* q = (const f32x4*)(p + (u32)(r * k));
      v[e] = WAY == WHOLE ? __builtin_nontemporal_load(q) : *q;
    }
  };
  f32x4 acc[4][4] = {}, own[NF];
  auto products = [&](int par) {
    const char* la = smem + par * BUF;
    const char* lb = la + BUF / 2;
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      s16x8 a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = frag(la, ks, wi * 4 + i);
        b[i] = frag(lb, ks, wj * 4 + i);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a[i], b[j], acc[i][j], 0, 0, 0);
    }
  };
  // tokens past the end of the last step
  auto clear = [&](int t0, int par) {
    if (t0 + BK <= t) return;
    const u32x4 z = {0, 0, 0, 0};
    for (int i = (t - t0) * 16 + tid; i < BK * 16; i += TPB) {
      *(u32x4*)(smem + par * BUF + i * 16) = z;
      *(u32x4*)(smem + par * BUF + BUF / 2 + i * 16) = z;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  int par = 0;
  stage(0, 0);
  if constexpr (WAY == DIRECT) {
    for (int t0 = 0; t0 < t; t0 += BK, par ^= 1) {
      loads_but<0>();
      if (t0 + BK < t) stage(t0 + BK, par ^ 1);
      else clear(t0, par);
      products(par);
    }
  } else {
    // The last step by itself: behind its loads those of H are on their way (in
    // the same loop their registers are copied at each turn: 724 us for 545).  A
    // second copy of the products costs a single round 1.2 us of fetching it.
    const int end = (t - 1) / BK * BK;
    for (int t0 = 0; t0 < end; t0 += BK, par ^= 1) {
      loads_but<0>();
      stage(t0 + BK, par ^ 1);
      products(par);
    }
    // counted: what comes between the stage's loads and the wait is these NF (h is
    // not __restrict__, so that the waits' memory clobbers hold for them as well)
    __builtin_amdgcn_sched_barrier(0);
    fours_load(own, i0, j0);
    __builtin_amdgcn_sched_barrier(0);
    loads_but<NF>();
    clear(end, par);
    products(par);
  }
  // H += 2 acc, here and mirrored
  if constexpr (WAY == DIRECT) {
    // All of a thread's elements on their way at once, places past the end out of
    // the buffer's bounds (by rows of fragments, in conditions: 1.1 us more)
    const auto hr = make_rsrc(h, (u32)k * (u32)k * 4);
    float v[4][4][4];
    f32x4 u[4][4];
    auto place = [&](int row, int col, bool in) {
      return in && row < k && col < k ? (u32)(row * k + col) * 4 : ~0u;
    };
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = i0 + wi * 64 + i * 16 + l4 * 4;
        const int col = j0 + wj * 64 + j * 16 + l15;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[i][j][r] = __builtin_bit_cast(
              float, __builtin_amdgcn_raw_buffer_load_b32(
                         hr, place(row + r, col, true), 0, 0));
        u[i][j] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       hr, place(col, row, ti != tj), 0, 0));
      }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = i0 + wi * 64 + i * 16 + l4 * 4;
        const int col = j0 + wj * 64 + j * 16 + l15;
        f32x4 w;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          __builtin_amdgcn_raw_buffer_store_b32(
              __builtin_bit_cast(u32, fmaf(2.f, acc[i][j][r], v[i][j][r])), hr,
              place(row + r, col, true), 0, 0);
          w[r] = fmaf(2.f, acc[i][j][r], u[i][j][r]);
        }
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, w), hr,
                                               place(col, row, ti != tj), 0, 0);
      }
  } else {
    // (LD: rows and columns both spread over the banks)
    float* out = (float*)smem;
    loads_but<NF>();
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          out[(wi * 64 + i * 16 + l4 * 4 + r) * LD + wj * 64 + j * 16 + l15] =
              acc[i][j][r];
    f32x4 mirror[NF];
    if (ti != tj) fours_load(mirror, j0, i0);
    // only LDS: the loads stay under way
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // v + 2 out at (row0, col0) of H; out by ro a row and co a column
    auto add = [&](const f32x4 (&v)[NF], int row0, int col0, int ro, int co) {
      if (col0 + c4 >= k) return;            // k in eights: four columns alike
      float* p = h + (u64)row0 * k + col0 + c4;
#pragma unroll
      for (int e = 0; e < NF; ++e) {
        const int r = r0 + e * (TPB * 4 / BC);
        f32x4 w;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          w[q] = fmaf(2.f, out[r * ro + (c4 + q) * co], v[e][q]);
        if (row0 + r >= k) continue;
        f32x4* to = (f32x4*)(p + (u32)(r * k));
        if (WAY == WHOLE)
          __builtin_nontemporal_store(w, to);
        else
          *to = w;
      }
    };
    add(own, i0, j0, LD, 1);
    if (ti != tj) add(mirror, j0, i0, 1, LD);
  }
}

}  // namespace

hipError_t lfmq_hessian_accum(const void* x, void* h, int t, int k,
                              hipStream_t stream) {
  if (k % 8) return hipErrorInvalidValue;
  if (t == 0 || k == 0) return hipSuccess;
  const u32 n = ceil_div_u32(k, BC * SB), wgs = n * (n + 1) / 2 * SB * SB;
  // (of 336, 231 with a tile, some XCD has more than CUs: 1469 x 2584 59 us, 51
  // the other way)
  const bool direct = wgs <= 256;
  const int lds = direct ? 2 * BUF : max(2 * BUF, BC * LD * 4);
  auto* kernel = direct ? hessian_kernel<DIRECT>
                        : (k % 32 == 0 && (u64)h % 128 == 0
                               ? hessian_kernel<WHOLE>
                               : hessian_kernel<CACHED>);
  hipLaunchKernelGGL(kernel, dim3(wgs), dim3(TPB), lds,
                     stream, (const unsigned short*)x, (float*)h, t, k);
  return hipGetLastError();
}
