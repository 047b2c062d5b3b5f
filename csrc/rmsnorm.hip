// K6 — fused RMSNorm: y = x · rsqrt(mean(x²)+ε) · w, optional fused
// residual add in the same pass (one read, one write — the op is
// HBM-bound).
// One workgroup per row, which it keeps in registers (rmsnorm_row_kernel): 16
// bytes a load, the row, the residual and the weights on their way at once, one
// barrier for the sum.  Bound by that one latency and the launch for few rows,
// by the traffic for many.  us a call with the residual, 4096 wide, reading the
// row twice by four bytes and this one: 1 row 4.1 / 2.1, 48 rows 5.0 / 2.5, 660
// rows 9.6 / 5.4, 3001 rows 25.6 / 16.9 (5.8 TB/s); 14336 wide, 77 rows 17.5 / 4.6.
// Rows that are no multiple of eight, unaligned or above 16384 wide take
// the kernels below.
#include "common.h"

namespace {

constexpr int TPB = 256;

// MODE: 0 = plain, 1 = fused residual-in (y = norm(x+r)),
//       2 = fused residual-in + write new residual (r_out = x+r)
// V: pieces of eight values a thread
template <int MODE, int V>
__global__ __launch_bounds__(TPB) void rmsnorm_row_kernel(
    const u32x4* __restrict__ x, const u32x4* __restrict__ res_in,
    const u32x4* __restrict__ w, u32x4* __restrict__ y,
    u32x4* __restrict__ res_out, int hidden, float eps) {
  const int n = hidden / 8, tid = threadIdx.x;
  const u64 at = (u64)blockIdx.x * n;
  u32x4 xv[V], rv[V], wv[V];
#pragma unroll
  for (int i = 0; i < V; ++i) {
    // past the end the last piece again, not counted and not stored
    const int c = min(tid + i * TPB, n - 1);
    xv[i] = x[at + c];
    if (MODE) rv[i] = res_in[at + c];
    wv[i] = w[c];
  }
  __shared__ float red[TPB / LFMQ_WAVE];
  float v[V][8], ss = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    float part = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float a, b;
      bf16x2_to_f32(xv[i][e], a, b);
      if (MODE) {
        float c, d;
        bf16x2_to_f32(rv[i][e], c, d);
        a += c;
        b += d;
      }
      v[i][2 * e] = a;
      v[i][2 * e + 1] = b;
      part = fmaf(a, a, part);
      part = fmaf(b, b, part);
    }
    if (tid + i * TPB < n) ss += part;
  }
  ss = wave_reduce_sum_dpp(ss);
  if (tid % LFMQ_WAVE == 0) red[tid / LFMQ_WAVE] = ss;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < TPB / LFMQ_WAVE; ++i) t += red[i];
  const float inv = rsqrtf(t / (float)hidden + eps);
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = tid + i * TPB;
    if (c >= n) break;
    u32x4 o, r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = v[i][2 * e], b = v[i][2 * e + 1];
      float wa, wb;
      bf16x2_to_f32(wv[i][e], wa, wb);
      o[e] = pack_bf16x2(a * inv * wa, b * inv * wb);
      if (MODE == 2) r[e] = pack_bf16x2(a, b);
    }
    y[at + c] = o;
    if (MODE == 2) res_out[at + c] = r;
  }
}

template <int MODE>
__global__ __launch_bounds__(TPB) void rmsnorm_kernel(
    const u32* __restrict__ x, const u32* __restrict__ res_in,
    const u32* __restrict__ w, u32* __restrict__ y, u32* __restrict__ res_out,
    int hidden, float eps) {
  const int row = blockIdx.x;
  const int dw = hidden / 2;  // dwords per row (hidden even)
  const u32* xr = x + (u64)row * dw;
  const u32* rr = MODE ? res_in + (u64)row * dw : nullptr;
  u32* yr = y + (u64)row * dw;
  u32* ro = MODE == 2 ? res_out + (u64)row * dw : nullptr;

  __shared__ float red[TPB / LFMQ_WAVE];

  float ss = 0.f;
  // the row is read twice, the second time mostly from the caches
  for (int i = threadIdx.x; i < dw; i += TPB) {
    float a, b;
    bf16x2_to_f32(xr[i], a, b);
    if (MODE) {
      float c, d;
      bf16x2_to_f32(rr[i], c, d);
      a += c;
      b += d;
    }
    ss = fmaf(a, a, ss);
    ss = fmaf(b, b, ss);
  }
  ss = wave_reduce_sum(ss);
  const int wave = threadIdx.x / LFMQ_WAVE;
  const int lane = threadIdx.x % LFMQ_WAVE;
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < TPB / LFMQ_WAVE; ++i) t += red[i];
  const float inv = rsqrtf(t / (float)hidden + eps);

  for (int i = threadIdx.x; i < dw; i += TPB) {
    float a, b, wa, wb;
    bf16x2_to_f32(xr[i], a, b);
    bf16x2_to_f32(w[i], wa, wb);
    if (MODE) {
      float c, d;
      bf16x2_to_f32(rr[i], c, d);
      a += c;
      b += d;
      if (MODE == 2) ro[i] = pack_bf16x2(a, b);
    }
    yr[i] = pack_bf16x2(a * inv * wa, b * inv * wb);
  }
}

// A wave a row, which it keeps in registers: no LDS, no barrier.  Up to 16 rows
// of up to 1024 that rmsnorm_row_kernel does not take (widths not in eights,
// rows not on 16 bytes).
template <int MODE, int DWPL>  // dwords per lane
__global__ __launch_bounds__(LFMQ_WAVE) void rmsnorm_wave_kernel(
    const u32* __restrict__ x, const u32* __restrict__ res_in,
    const u32* __restrict__ w, u32* __restrict__ y, u32* __restrict__ res_out,
    int hidden, float eps) {
  const int row = blockIdx.x;
  const int dw = hidden / 2;
  const int lane = threadIdx.x;
  const u32* xr = x + (u64)row * dw;
  const u32* rr = MODE ? res_in + (u64)row * dw : nullptr;
  u32* yr = y + (u64)row * dw;
  u32* ro = MODE == 2 ? res_out + (u64)row * dw : nullptr;

  float va[DWPL * 2];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < DWPL; ++i) {
    const int idx = lane + i * LFMQ_WAVE;
    float a = 0.f, b = 0.f;
    if (idx < dw) {
      bf16x2_to_f32(xr[idx], a, b);
      if (MODE) {
        float c, d;
        bf16x2_to_f32(rr[idx], c, d);
        a += c;
        b += d;
        if (MODE == 2) ro[idx] = pack_bf16x2(a, b);
      }
    }
    va[2 * i] = a;
    va[2 * i + 1] = b;
    ss = fmaf(a, a, ss);
    ss = fmaf(b, b, ss);
  }
  ss = wave_reduce_sum(ss);
  const float inv = rsqrtf(ss / (float)hidden + eps);
#pragma unroll
  for (int i = 0; i < DWPL; ++i) {
    const int idx = lane + i * LFMQ_WAVE;
    if (idx < dw) {
      float wa, wb;
      bf16x2_to_f32(w[idx], wa, wb);
      yr[idx] = pack_bf16x2(va[2 * i] * inv * wa, va[2 * i + 1] * inv * wb);
    }
  }
}

// 1 / sqrt(mean x^2 + eps) of each row alone: a launch and a latency, 48 rows of
// 4096 4.7 us on a busy queue (the whole norm 5.0).
__global__ __launch_bounds__(TPB) void row_scale_kernel(
    const unsigned short* __restrict__ x, float* __restrict__ scale, int hidden,
    float eps, bool wide) {
  const unsigned short* row = x + (u64)blockIdx.x * hidden;
  float ss = 0.f;
  const int n8 = wide ? hidden / 8 : 0;
  for (int i = threadIdx.x; i < n8; i += TPB) {
    const u32x4 v = ((const u32x4*)row)[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float a, b;
      bf16x2_to_f32(v[e], a, b);
      ss = fmaf(b, b, fmaf(a, a, ss));
    }
  }
  for (int i = n8 * 8 + threadIdx.x; i < hidden; i += TPB) {
    const float a = bf16_bits_to_f32(row[i]);
    ss = fmaf(a, a, ss);
  }
  __shared__ float red[TPB / LFMQ_WAVE];
  ss = wave_reduce_sum_dpp(ss);
  if (threadIdx.x % LFMQ_WAVE == 0) red[threadIdx.x / LFMQ_WAVE] = ss;
  __syncthreads();
  if (threadIdx.x == 0) {
    ss = 0.f;
    for (int i = 0; i < TPB / LFMQ_WAVE; ++i) ss += red[i];
    scale[blockIdx.x] = rsqrtf(ss / (float)hidden + eps);
  }
}

template <int MODE>
bool launch_row(const void* x, const void* r, const void* w, void* y, void* ro,
                int rows, int hidden, float eps, hipStream_t stream) {
  if (hidden % 8 || (((u64)x | (u64)r | (u64)w | (u64)y | (u64)ro) & 15))
    return false;
#define RCASE(V)                                                            \
  if (hidden <= 8 * V * TPB) {                                              \
    hipLaunchKernelGGL((rmsnorm_row_kernel<MODE, V>), dim3(rows), dim3(TPB), \
                       0, stream, (const u32x4*)x, (const u32x4*)r,          \
                       (const u32x4*)w, (u32x4*)y, (u32x4*)ro, hidden, eps); \
    return true;                                                            \
  }
  RCASE(1)
  RCASE(2)
  RCASE(4)
  RCASE(8)
#undef RCASE
  return false;
}

template <int MODE>
bool launch_wave(const u32* x, const u32* r, const u32* w, u32* y, u32* ro,
                 int rows, int hidden, float eps, hipStream_t stream) {
  const int dw = hidden / 2;
#define WCASE(D)                                                           \
  if (dw <= LFMQ_WAVE * D) {                                               \
    hipLaunchKernelGGL((rmsnorm_wave_kernel<MODE, D>), dim3(rows),         \
                       dim3(LFMQ_WAVE), 0, stream, x, r, w, y, ro, hidden, \
                       eps);                                               \
    return true;                                                           \
  }
  WCASE(8)
#undef WCASE
  return false;
}

}  // namespace

hipError_t lfmq_rmsnorm(const void* x, const void* residual, const void* w,
                        void* y, void* res_out, int rows, int hidden,
                        float eps, hipStream_t stream) {
  if (hidden % 2) return hipErrorInvalidValue;
  if (residual == nullptr
          ? launch_row<0>(x, nullptr, w, y, nullptr, rows, hidden, eps, stream)
          : (res_out == nullptr ? launch_row<1>(x, residual, w, y, nullptr, rows,
                                                hidden, eps, stream)
                                : launch_row<2>(x, residual, w, y, res_out, rows,
                                                hidden, eps, stream)))
    return hipGetLastError();
  if (rows <= 16 && hidden <= 1024) {  // tiny rows: wave-per-row path
    bool ok;
    if (residual == nullptr)
      ok = launch_wave<0>((const u32*)x, nullptr, (const u32*)w, (u32*)y,
                          nullptr, rows, hidden, eps, stream);
    else if (res_out == nullptr)
      ok = launch_wave<1>((const u32*)x, (const u32*)residual, (const u32*)w,
                          (u32*)y, nullptr, rows, hidden, eps, stream);
    else
      ok = launch_wave<2>((const u32*)x, (const u32*)residual, (const u32*)w,
                          (u32*)y, (u32*)res_out, rows, hidden, eps, stream);
    if (ok) return hipGetLastError();
  }
  dim3 grid(rows), block(TPB);
  if (residual == nullptr)
    hipLaunchKernelGGL((rmsnorm_kernel<0>), grid, block, 0, stream,
                       (const u32*)x, nullptr, (const u32*)w, (u32*)y, nullptr,
                       hidden, eps);
  else if (res_out == nullptr)
    hipLaunchKernelGGL((rmsnorm_kernel<1>), grid, block, 0, stream,
                       (const u32*)x, (const u32*)residual, (const u32*)w,
                       (u32*)y, nullptr, hidden, eps);
  else
    hipLaunchKernelGGL((rmsnorm_kernel<2>), grid, block, 0, stream,
                       (const u32*)x, (const u32*)residual, (const u32*)w,
                       (u32*)y, (u32*)res_out, hidden, eps);
  return hipGetLastError();
}

hipError_t lfmq_row_scale(const void* x, void* scale, int rows, int hidden,
                          float eps, hipStream_t stream) {
  if (rows < 1) return hipSuccess;
  const bool wide = hidden % 8 == 0 && (u64)x % 16 == 0;
  hipLaunchKernelGGL(row_scale_kernel, dim3(rows), dim3(TPB), 0, stream,
                     (const unsigned short*)x, (float*)scale, hidden, eps, wide);
  return hipGetLastError();
}
