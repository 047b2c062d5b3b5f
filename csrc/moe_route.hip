// MoE routing in ONE kernel (Mixtral top-k), on the device from the router's
// logits to what the grouped kernels read, so that a step of any size can be
// captured: top-k and softmax of every token, slots sorted by expert, row
// tiles.  One workgroup: a thread a token at a time, counters and cursors in
// LDS.  The order of an expert's slots is the cursors' and has no effect: a
// row's result does not depend on its place.
#include "common.h"

namespace {

constexpr int MAXE = 64;
constexpr int MAXK = 4;

struct RouteArgs {
  const unsigned short* logits;  // [t, E] bf16
  i32* src;                      // [t * topk] token of a slot
  float* slot_w;                 // [t * topk] weight of a slot, or null
  i32* pos;                      // [t, topk] slot of a token's choice
  float* w;                      // [t, topk] its weight
  i32* offsets;                  // [E + 1] slots of the experts, or null
  i32* active;                   // [E] experts with slots, then -1, or null
  i32* tiles;                    // [n_tiles, 3] expert (or -1), slot, slots
  int t, E, topk, bm, n_tiles;
};

__global__ __launch_bounds__(1024) void moe_route_kernel(RouteArgs A) {
  __shared__ int cnt[MAXE], offs[MAXE + 1], tile0[MAXE + 1], cur[MAXE];
  const int tid = threadIdx.x, E = A.E, topk = A.topk;
  if (tid < MAXE) cnt[tid] = 0;
  __syncthreads();
  for (int tok = tid; tok < A.t; tok += blockDim.x) {
    // serial top-k over E logits (E <= 64, k <= 4); first of equals wins
    float best[MAXK];
    int id[MAXK];
#pragma unroll
    for (int j = 0; j < MAXK; ++j) {
      best[j] = -INFINITY;
      id[j] = 0;
    }
    for (int e = 0; e < E; ++e) {
      float v = bf16_bits_to_f32(A.logits[(u64)tok * E + e]);
      int i = e;
#pragma unroll
      for (int j = 0; j < MAXK; ++j) {
        if (j < topk && v > best[j]) {       // the displaced one moves down
          const float tv = best[j];
          const int ti = id[j];
          best[j] = v;
          id[j] = i;
          v = tv;
          i = ti;
        }
      }
    }
    float den = 0.f;
#pragma unroll
    for (int j = 0; j < MAXK; ++j)
      if (j < topk) den += __expf(best[j] - best[0]);
#pragma unroll
    for (int j = 0; j < MAXK; ++j)
      if (j < topk) {
        A.w[(u64)tok * topk + j] = __expf(best[j] - best[0]) / den;
        A.pos[(u64)tok * topk + j] = id[j];  // the expert, for now
        atomicAdd(&cnt[id[j]], 1);
      }
  }
  __syncthreads();
  if (tid == 0) {
    int at = 0, ti = 0, na = 0;
    for (int e = 0; e < E; ++e) {
      offs[e] = at;
      tile0[e] = ti;
      cur[e] = at;
      if (A.active != nullptr && cnt[e] > 0) A.active[na++] = e;
      at += cnt[e];
      ti += (cnt[e] + A.bm - 1) / A.bm;
    }
    offs[E] = at;
    tile0[E] = ti;
    if (A.active != nullptr)
      for (int j = na; j < E; ++j) A.active[j] = -1;
  }
  __syncthreads();
  if (A.offsets != nullptr)                // one more than there may be threads
    for (int e = tid; e <= E; e += blockDim.x) A.offsets[e] = offs[e];
  if (A.tiles != nullptr) {
    for (int i = tid; i < A.n_tiles; i += blockDim.x) {
      int e = -1;
      if (i < tile0[E])
        for (e = 0; tile0[e + 1] <= i; ++e) {}
      const int first = e < 0 ? 0 : offs[e] + (i - tile0[e]) * A.bm;
      A.tiles[3 * i] = e;
      A.tiles[3 * i + 1] = first;
      A.tiles[3 * i + 2] = e < 0 ? 0 : min(A.bm, offs[e + 1] - first);
    }
  }
  for (int tok = tid; tok < A.t; tok += blockDim.x)
    for (int j = 0; j < topk; ++j) {
      const u64 i = (u64)tok * topk + j;
      const int slot = atomicAdd(&cur[A.pos[i]], 1);
      A.src[slot] = tok;
      if (A.slot_w != nullptr) A.slot_w[slot] = A.w[i];
      A.pos[i] = slot;
    }
}

// tiles of sorted slots, given where each expert's begin
__global__ __launch_bounds__(64) void moe_tiles_kernel(
    const i32* __restrict__ offsets, i32* __restrict__ tiles, int E, int bm,
    int n_tiles) {
  for (int i = threadIdx.x; i < n_tiles; i += 64) {
    int e = 0, left = i;
    for (; e < E; ++e) {
      const int n = (offsets[e + 1] - offsets[e] + bm - 1) / bm;
      if (left < n) break;
      left -= n;
    }
    const int first = e < E ? offsets[e] + left * bm : 0;
    tiles[3 * i] = e < E ? e : -1;
    tiles[3 * i + 1] = first;
    tiles[3 * i + 2] = e < E ? min(bm, offsets[e + 1] - first) : 0;
  }
}

// y[t] = sum over a token's choices of w * rows[pos], fp32 -> bf16
__global__ __launch_bounds__(256) void moe_sum_kernel(
    const float* __restrict__ rows, const i32* __restrict__ pos,
    const float* __restrict__ w, unsigned short* __restrict__ y, int t, int n,
    int topk) {
  const int c = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (c >= n) return;
  for (u64 tok = blockIdx.y; tok < (u64)t; tok += gridDim.y) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < topk; ++j) {
      const float wj = w[tok * topk + j];
      const f32x4 r = *(const f32x4*)(rows + (u64)pos[tok * topk + j] * n + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = fmaf(wj, r[e], v[e]);
    }
    *(u64*)(y + tok * n + c) =
        pack_bf16x2(v[0], v[1]) | (u64)pack_bf16x2(v[2], v[3]) << 32;
  }
}

}  // namespace

hipError_t lfmq_moe_route(const void* logits, void* src, void* slot_w,
                          void* pos, void* w, void* offsets, void* active,
                          void* tiles, int t, int E, int topk, int bm,
                          int n_tiles, hipStream_t stream) {
  if (E > MAXE || topk > MAXK || topk > E || bm < 1)
    return hipErrorInvalidValue;
  const RouteArgs A{(const unsigned short*)logits, (i32*)src, (float*)slot_w,
                    (i32*)pos, (float*)w, (i32*)offsets, (i32*)active,
                    (i32*)tiles, t, E, topk, bm, n_tiles};
  const int threads = t <= 64 ? 64 : (t <= 256 ? 256 : 1024);
  hipLaunchKernelGGL(moe_route_kernel, dim3(1), dim3(threads), 0, stream, A);
  return hipGetLastError();
}

hipError_t lfmq_moe_tiles(const void* offsets, void* tiles, int E, int bm,
                          int n_tiles, hipStream_t stream) {
  hipLaunchKernelGGL(moe_tiles_kernel, dim3(1), dim3(64), 0, stream,
                     (const i32*)offsets, (i32*)tiles, E, bm, n_tiles);
  return hipGetLastError();
}

hipError_t lfmq_moe_sum(const void* rows, const void* pos, const void* w,
                        void* y, int t, int n, int topk, hipStream_t stream) {
  if (n % 4) return hipErrorInvalidValue;
  if (t == 0) return hipSuccess;
  hipLaunchKernelGGL(moe_sum_kernel,
                     dim3((n / 4 + 255) / 256, min(t, 65535)), dim3(256), 0,
                     stream, (const float*)rows, (const i32*)pos,
                     (const float*)w, (unsigned short*)y, t, n, topk);
  return hipGetLastError();
}
