// Fused decode epilogue of the qkv projection (K7 + K10 in one pass):
// reads the raw fused qkv GEMV output [b*s, (hq+2hkv)*d] bf16 and in one
// launch (a) applies NeoX rotary to q -> q_out [b, s, hq, d] (== the
// [b, hq, 1, d] attention layout at s == 1, so decode never transposes),
// (b) applies rotary to k and scatters it into k_cache at its position,
// (c) scatters v into v_cache.  Replaces rope + kv_append + two reshape
// copies on the decode path — these tensors are tiny, so the win is
// launch/latency count, the thing the decode step is bound by.
#include "common.h"

namespace {

__global__ void qkv_rope_append_kernel(
    const u32* __restrict__ qkv, u32* __restrict__ q_out,
    u32* __restrict__ kc, u32* __restrict__ vc,
    const i32* __restrict__ positions, const float* __restrict__ inv_freq,
    int b, int s, int hq, int hkv, int d, int tmax, int pos0,
    const i32* __restrict__ pos_dev) {
  if (pos_dev != nullptr) pos0 = *pos_dev;  // hipGraph mode
  const int dp = d / 4;          // dword-pairs per rotated half
  const int dw = d / 2;          // dwords per head
  const int qkv_dw = (hq + 2 * hkv) * dw;
  const u64 q_pairs = (u64)b * s * hq * dp;
  const u64 k_pairs = (u64)b * s * hkv * dp;
  const u64 v_dwords = (u64)b * s * hkv * dw;
  const u64 total = q_pairs + k_pairs + v_dwords;

  for (u64 idx = (u64)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (u64)gridDim.x * blockDim.x) {
    if (idx < q_pairs + k_pairs) {
      const bool is_q = idx < q_pairs;
      const u64 rel = is_q ? idx : idx - q_pairs;
      const int nh = is_q ? hq : hkv;
      const int j = rel % dp;
      const int hh = (rel / dp) % nh;
      const int tok = rel / ((u64)dp * nh);
      const int si = tok % s;
      const int bb = tok / s;
      const int pos = positions[si];
      const u32* src = qkv + (u64)tok * qkv_dw +
                       (is_q ? hh * dw : (hq + hh) * dw);
      const u32 a = src[j], bv = src[j + dp];
      float a0, a1, b0, b1;
      bf16x2_to_f32(a, a0, a1);
      bf16x2_to_f32(bv, b0, b1);
      const float ang0 = (float)pos * inv_freq[2 * j];
      const float ang1 = (float)pos * inv_freq[2 * j + 1];
      float c0, s0, c1, s1;
      __sincosf(ang0, &s0, &c0);
      __sincosf(ang1, &s1, &c1);
      const u32 lo = pack_bf16x2(a0 * c0 - b0 * s0, a1 * c1 - b1 * s1);
      const u32 hi = pack_bf16x2(a0 * s0 + b0 * c0, a1 * s1 + b1 * c1);
      if (is_q) {
        u32* dst = q_out + ((u64)tok * hq + hh) * dw;
        dst[j] = lo;
        dst[j + dp] = hi;
      } else {
        u32* dst = kc + (((u64)bb * hkv + hh) * tmax + pos0 + si) * dw;
        dst[j] = lo;
        dst[j + dp] = hi;
      }
    } else {
      const u64 rel = idx - q_pairs - k_pairs;
      const int j = rel % dw;
      const int hh = (rel / dw) % hkv;
      const int tok = rel / ((u64)dw * hkv);
      const int si = tok % s;
      const int bb = tok / s;
      const u32 v = qkv[(u64)tok * qkv_dw + (hq + hkv + hh) * dw + j];
      vc[(((u64)bb * hkv + hh) * tmax + pos0 + si) * dw + j] = v;
    }
  }
}

// The same from the parts of the projection, part [splits, b s, n] fp32 (+ bias),
// whose sums are rounded to bf16 as a launch of their own would store them: one
// launch and the projection's way to memory and back less.  A thread has four
// values of each half of a head, up to four parts of them on their way at once.
// 77 tokens of 3072, us: the sum of parts 3.8 and the rotation 3.4, both here 3.8.
__global__ __launch_bounds__(256) void qkv_sum_rope_append_kernel(
    const float* __restrict__ part, int splits,
    const unsigned short* __restrict__ bias, u64* __restrict__ q_out,
    u64* __restrict__ kc, u64* __restrict__ vc,
    const i32* __restrict__ positions, const float* __restrict__ inv_freq,
    int s, int hq, int hkv, int d, int tmax, int pos0) {
  const int item = blockIdx.x * 256 + threadIdx.x, per = d / 8;
  const int head = item / per, j = item % per, tok = blockIdx.y;
  if (head >= hq + 2 * hkv) return;
  const int n = (hq + 2 * hkv) * d, c0 = head * d + j * 4, c1 = c0 + d / 2;
  const int si = tok % s, bb = tok / s;
  const u64 stride = (u64)gridDim.y * n;
  const float* row = part + (u64)tok * n;
  const float pos = (float)positions[si];
  const f32x4 freq = *(const f32x4*)(inv_freq + j * 4);
  f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
  for (int s0 = 0; s0 < splits; s0 += 4) {
    f32x4 ta[4], tb[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* p = row + (u64)min(s0 + i, splits - 1) * stride;
      ta[i] = *(const f32x4*)(p + c0);
      tb[i] = *(const f32x4*)(p + c1);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (s0 + i < splits) {
        a += ta[i];
        b += tb[i];
      }
  }
  if (bias != nullptr)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      a[e] += bf16_bits_to_f32(bias[c0 + e]);
      b[e] += bf16_bits_to_f32(bias[c1 + e]);
    }
  u32 lo[2], hi[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    lo[e] = pack_bf16x2(a[2 * e], a[2 * e + 1]);
    hi[e] = pack_bf16x2(b[2 * e], b[2 * e + 1]);
  }
  const bool rotated = head < hq + hkv;
  if (rotated) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      float a0, a1, b0, b1, sn0, cs0, sn1, cs1;
      bf16x2_to_f32(lo[e], a0, a1);
      bf16x2_to_f32(hi[e], b0, b1);
      __sincosf(pos * freq[2 * e], &sn0, &cs0);
      __sincosf(pos * freq[2 * e + 1], &sn1, &cs1);
      lo[e] = pack_bf16x2(a0 * cs0 - b0 * sn0, a1 * cs1 - b1 * sn1);
      hi[e] = pack_bf16x2(a0 * sn0 + b0 * cs0, a1 * sn1 + b1 * cs1);
    }
  }
  u64* dst;
  if (head < hq)
    dst = q_out + ((u64)tok * hq + head) * (d / 4);
  else
    dst = (rotated ? kc : vc) +
          (((u64)bb * hkv + (head - hq) % hkv) * tmax + pos0 + si) * (d / 4);
  dst[j] = lo[0] | (u64)lo[1] << 32;
  dst[j + per] = hi[0] | (u64)hi[1] << 32;
}

}  // namespace

// part [splits, b s, (hq + 2 hkv) d]; heads in eights, caches and frequencies on 16
// bytes
hipError_t lfmq_qkv_sum_rope_append(const void* part, int splits,
                                    const void* bias, void* q_out, void* kc,
                                    void* vc, const void* positions,
                                    const void* inv_freq, int b, int s, int hq,
                                    int hkv, int d, int tmax, int pos0,
                                    hipStream_t stream) {
  const int items = (hq + 2 * hkv) * (d / 8);
  if (d % 8 || splits < 1 || b < 1 || s < 1 || (long)b * s > 65535 ||
      pos0 < 0 || pos0 > tmax - s ||
      (((u64)kc | (u64)vc | (u64)q_out | (u64)inv_freq) & 15))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(qkv_sum_rope_append_kernel,
                     dim3((items + 255) / 256, b * s), dim3(256), 0, stream,
                     (const float*)part, splits, (const unsigned short*)bias,
                     (u64*)q_out, (u64*)kc, (u64*)vc, (const i32*)positions,
                     (const float*)inv_freq, s, hq, hkv, d, tmax, pos0);
  return hipGetLastError();
}

hipError_t lfmq_qkv_rope_append(const void* qkv, void* q_out, void* kc,
                                void* vc, const void* positions,
                                const void* inv_freq, int b, int s, int hq,
                                int hkv, int d, int tmax, int pos0,
                                const void* pos_dev, hipStream_t stream) {
  if (d % 4) return hipErrorInvalidValue;
  const u64 total = (u64)b * s * ((hq + hkv) * (d / 4) + hkv * (d / 2));
  u32 blocks = (u32)((total + 255) / 256);
  if (blocks > 2048) blocks = 2048;
  if (blocks == 0) blocks = 1;
  hipLaunchKernelGGL(qkv_rope_append_kernel, dim3(blocks), dim3(256), 0,
                     stream, (const u32*)qkv, (u32*)q_out, (u32*)kc, (u32*)vc,
                     (const i32*)positions, (const float*)inv_freq, b, s, hq,
                     hkv, d, tmax, pos0, (const i32*)pos_dev);
  return hipGetLastError();
}
