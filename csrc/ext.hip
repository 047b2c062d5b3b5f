// lfmq_hip — torch-extension bindings for the gfx950 kernels.
// Every entry validates dtype/contiguity/device and launches on the
// current HIP stream.  No fallbacks: errors raise.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include <hip/hip_runtime.h>

#include "dq_mid.h"
#include "dq_short.h"

hipError_t lfmq_pack(const void*, void*, long, int, int, hipStream_t);
hipError_t lfmq_unpack(const void*, void*, long, int, int, hipStream_t);
hipError_t lfmq_dq_gemv(const void*, const void*, const void*, const void*,
                        void*, const void*, const void*, int, int, int, int,
                        int, float, int, hipStream_t);
bool lfmq_dq_rows_ok(int, int, int, int, bool);
int lfmq_dq_rows_splits(int, int, int, int);
hipError_t lfmq_dq_rows(const void*, const void*, const void*, const void*,
                        void*, const void*, const void*, void*, int, int, int,
                        int, int, int, float,
                        bool, hipStream_t, const float* row_scale = nullptr,
                        const DqRowEnd* end = nullptr);
bool lfmq_dq_row_ok(int, int, int);
hipError_t lfmq_dq_row(const void*, const void*, const void*, const void*,
                       void*, const void*, const void*, int, int, int, int,
                       float, bool, hipStream_t);
bool lfmq_dq_wide_ok(int, int, int, int, int);
hipError_t lfmq_dq_wide(const void*, const void*, const void*, const void*,
                        void*, const void*, const void*, int, int, int, int,
                        int, float, bool, hipStream_t);
int lfmq_dq_wide_parts(int, int, int, int, int);
int lfmq_dq_wide_part_blocks(int, int);
hipError_t lfmq_dq_wide_in_parts(const void*, const void*, const void*, const void*,
                                 void*, const void*, const void*, void*, void*, int,
                                 int, int, int, int, hipStream_t);
hipError_t lfmq_dq_wide_experts(const void*, const void*, const void*,
                                const void*, const void*, const void*, void*,
                                int, int, int, int, int, bool, hipStream_t);
bool lfmq_dq_tile_ok(int, int);
int lfmq_dq_tile_splits(int, int, int, int);
hipError_t lfmq_dq_tile(const void*, const void*, const void*, const void*,
                        void*, const void*, const void*, void*, int, int, int,
                        int, int, int, bool, hipStream_t,
                        const DqRowEnd* end = nullptr);
hipError_t lfmq_row_scale(const void*, void*, int, int, float, hipStream_t);
hipError_t lfmq_rmsnorm(const void*, const void*, const void*, void*, void*,
                        int, int, float, hipStream_t);
hipError_t lfmq_rope(void*, void*, const void*, const void*, int, int, int,
                     int, int, hipStream_t);
hipError_t lfmq_silu_mul(const void*, const void*, void*, long, hipStream_t);
hipError_t lfmq_silu_mul_fused(const void*, void*, long, int, hipStream_t);
hipError_t lfmq_residual_add(const void*, const void*, void*, long,
                             hipStream_t);
hipError_t lfmq_kv_append(void*, void*, const void*, const void*, int, int,
                          int, int, int, int, hipStream_t);
hipError_t lfmq_attn_decode(const void*, const void*, const void*, void*,
                            void*, int, int, int, int, int, const void*, int,
                            int, float, hipStream_t);
hipError_t lfmq_attn_decode_fused(const void*, void*, void*, void*, void*,
                                  const void*, int, int, int, int, int,
                                  const void*, int, int, float, void*,
                                  hipStream_t);
int lfmq_attn_decode_splits(int, int, int, int, int);
hipError_t lfmq_attn_prefill(const void*, const void*, const void*, void*,
                             int, int, int, int, int, int, int, float,
                             hipStream_t);
hipError_t lfmq_hessian_accum(const void*, void*, int, int, hipStream_t);
long lfmq_chol_scratch(int n);
hipError_t lfmq_chol_inverse(const void*, const void*, void*, void*, void*, int,
                             hipStream_t);
hipError_t lfmq_gptq_prepare(const void*, const void*, void*, void*, int, int,
                             float, hipStream_t);
hipError_t lfmq_gptq_block(const void*, const void*, int, void*, void*, void*,
                           void*, int, int, int, int, int, int, int, bool,
                           hipStream_t);
hipError_t lfmq_gptq_push(const void*, const void*, const void*, long, int, int,
                          int, int, hipStream_t);
bool lfmq_gptq_step_ok(const void*, long, int, int, int);
hipError_t lfmq_gptq_step(const void*, const void*, long, void*, void*, void*,
                          const void*, void*, int, int, int, int, int, int, bool,
                          hipStream_t);
hipError_t lfmq_dq_gemv_gateup(const void*, const void*, const void*,
                               const void*, void*, int, int, int, int, int,
                               float, int, hipStream_t);
hipError_t lfmq_qkv_rope_append(const void*, void*, void*, void*, const void*,
                                const void*, int, int, int, int, int, int,
                                int, const void*, hipStream_t);
hipError_t lfmq_advance_record(void*, void*, const void*, void*, int, int,
                               hipStream_t);
hipError_t lfmq_moe_route(const void*, void*, void*, void*, void*, void*,
                          void*, void*, int, int, int, int, int, hipStream_t);
hipError_t lfmq_moe_tiles(const void*, void*, int, int, int, hipStream_t);
hipError_t lfmq_moe_sum(const void*, const void*, const void*, void*, int, int,
                        int, hipStream_t);
hipError_t lfmq_dq_rows_experts(const void*, const void*, const void*,
                                const void*, const void*, const void*, void*,
                                int, int, int, int, int, bool, hipStream_t);
hipError_t lfmq_dq_tile_experts(const void*, const void*, const void*,
                                const void*, const void*, const void*, void*,
                                int, int, int, int, int, bool, hipStream_t);
hipError_t lfmq_argmax_rows(const void*, void*, void*, void*, int, int,
                            hipStream_t);
hipError_t lfmq_read_probe(const void*, void*, long, long, int, int, int,
                           hipStream_t);
hipError_t lfmq_qkv_sum_rope_append(const void*, int, const void*, void*, void*,
                                    void*, const void*, const void*, int, int,
                                    int, int, int, int, int, hipStream_t);
#include "dq_block.h"
#include "engine_args.h"

namespace {

#define CHECK_HIP(call)                                                     \
  do {                                                                      \
    hipError_t e = (call);                                                  \
    TORCH_CHECK(e == hipSuccess, "lfmq HIP error: ", hipGetErrorString(e)); \
  } while (0)

void check_t(const torch::Tensor& t, torch::ScalarType dt, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be on GPU");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
  TORCH_CHECK(t.scalar_type() == dt, name, " has wrong dtype ",
              t.scalar_type(), " expected ", dt);
}

hipStream_t stream() {
  return (hipStream_t)at::cuda::getCurrentCUDAStream().stream();
}

torch::Tensor pack(torch::Tensor codes, long bits) {
  check_t(codes, torch::kInt32, "codes");
  const long n = codes.size(0), k = codes.size(1);
  const long per = 32 / bits;
  TORCH_CHECK(k % per == 0, "k must be divisible by ", per);
  auto out = torch::empty({n, k / per}, codes.options());
  CHECK_HIP(lfmq_pack(codes.data_ptr(), out.data_ptr(), n, (int)k, (int)bits,
                      stream()));
  return out;
}

torch::Tensor unpack(torch::Tensor packed, long bits, long k) {
  check_t(packed, torch::kInt32, "packed");
  const long n = packed.size(0);
  auto out = torch::empty({n, k}, packed.options());
  CHECK_HIP(lfmq_unpack(packed.data_ptr(), out.data_ptr(), n, (int)k,
                        (int)bits, stream()));
  return out;
}

// dq_row and dq_wide read scales two at a time
bool in_pairs(const torch::Tensor& scales) {
  return (uintptr_t)scales.data_ptr() % 4 == 0;
}

// rows from which the rows kernel is taken and not the GEMV, whose lanes hold
// the scales of 128 groups at most.  us of both (4 bits, groups of 128): n 4096, k
// 14336 11.3 / 13.0 at 1 row, 15.6 / 13.1 at 2; n 2048, k 8192 5.9 / 8.4, 7.6 / 8.3
// and 9.3 / 8.5 at 3 (8 bits, groups of 64: 8.1 / 11.0, 10.8 / 10.8).
int rows_from(long bits, long n, long k, long g) {
  if (k > 128 * g) return 1;
  return bits == 8 || n * k >= 32l << 20 ? 2 : 3;
}

// the product through LDS addresses a matrix below 4 GiB, the others any
bool tile_addresses(long n, long k, long bits) {
  return n * k / 8 * bits < 1l << 32;
}

// The kernel that keeps x and walks over columns (dq_wide), or rows.  Its 8 or
// 16 waves hold 256 values of k each and as many steps of them as k takes, so
// what counts first is how full the last step is; then, that rows runs one
// column tile of 16 to 32 a workgroup, in whole rounds of them up to 8192
// columns (10240: one and a quarter).  us of rows / wide:
//   4 bits, groups of 128        4 rows         16 rows
//     n 4096, k 4096 (full)    7.2 / 6.7       9.2 / 8.5
//     n 4096, k 2560 (0.62)    6.2 / 6.5       7.2 / 8.2
//     n 8192, k 2560           7.7 / 7.9       8.8 / 9.7
//     n 10240, k 2560         10.3 / 9.1      12.5 / 11.0
//     n 6144, k 5120 (0.62)   10.9 / 11.0     13.3 / 14.6
//     n 28672, k 4096         22.4 / 16.2     30.2 / 18.1
// With groups of 64 the bodies for several steps spill (gate, 4 rows: n 5120, k
// 5120 14.9 / 20.7; n 10240, k 8192 31.3 / 26.9).  A gate makes twice the tiles:
// of 5120 to 8192 columns and k 2048, where that is one a workgroup, 7.0 / 6.7
// at 4 rows, 7.6 / 8.5 at 16.  With k of many groups rows has the gate apart (n
// 8192, k 28672, groups of 64: 94 / 68).  Two rows of a smaller matrix of 4 bits
// are otherwise the GEMV's, which takes, groups of 128, 0.9 of wide's time at n
// 2048, 1.1 at n 4096; of 64, 0.75 to 1.05 up to 10240 columns, with a gate 0.9
// to 1.1, and 0.65 to 0.7 for several steps.
bool wide_rows(int m, int n, int k, long g, long bits, bool glu) {
  if (m < 2 || n < 2048 || k < 2048 ||
      !lfmq_dq_wide_ok(m, n, k, (int)g, (int)bits))
    return false;
  const bool more = k > 4096;                    // than one step
  if (more && n < (k <= 8192 ? 5120 : 8192)) return false;
  if (m == 2 && rows_from(bits, n, k, g) > 2)
    return g == 128 ? glu || n > 2048 : (glu ? !more : n >= 12288);
  const int step = k <= 2048 ? 2048 : 4096;
  const int full = (int)(100l * k / (((long)k + step - 1) / step * step));
  int least;                                     // percent of the steps
  if (n > 8192) {
    least = !more || g == 128 ? 50 : (glu && n <= 16384 ? 70 : 60);
  } else if (more && g == 64) {
    if (glu) return !lfmq_dq_rows_ok(m, n, k, (int)g, true);
    if (bits == 8 && k > 8192) return false;
    least = bits == 4 ? 70 : 80;
  } else if (glu && k <= 2048 && n > 4096) {
    return m <= 8;
  } else if (glu ? n <= 4096 : n > 4096 && n < 6144) {
    least = glu ? 50 : 60;
  } else {
    least = bits == 8 || (more && !glu) ? 70 : 80;
  }
  return full >= least;
}

// Whether that kernel gains by k in parts, of up to 4096 each, which its last
// workgroup adds up (dq_wide).  us of the other way / this one: n 4096, k 8192 (4 bits,
// groups of 128) 11.4 / 10.9 at 8 rows, 13.6 / 12.1 at 16, 10.1 / 10.4 at 4; n 4096, k
// 14336 14.2 / 13.7 at 4; n 2048, k 8192 9.9 / 10.7 at 16; n 4096, k 5120 10.9 / 12.1; n
// 12288, k 8192 17.0 / 16.0 at 3, groups of 64 21.5 / 21.9; seven parts, n 4096, k 27648
// 26.7 / 34.6 at 7, of few columns n 1904, k 25600 20.9 / 22.6 at 13.  Of 22000 random
// calls that it takes 1.23 times as fast in the mean, 0.8 % slower by more than 4 %:
// groups of 64 below 44 million weights, n 2136, k 16384 at 16 17.1 / 18.8.
bool part_rows(long m, long n, long k, long g, long bits) {
  const long size = n * k, M = 1l << 20, parts = (k + 4095) / 4096;
  return m >= 3 && m <= 16 && n >= 2048 && k >= 8192 && parts <= 5 &&
         size >= (m > 8 ? 32 : 48) * M && 10 * k >= 7 * 4096 * parts &&
         (bits == 8 || g != 64 || n <= 8192) && tile_addresses(n, k, bits);
}

// The product for many rows: tiles of 256 columns instead of 128, which few
// columns leave most of the chip without.  The time of dq_tile / of this one, the
// mean over 4400 measured calls of 129 to 700 rows and 6700 of 17 to 128, by n k
// in millions (2^20):
//   4 bits, 128  49-96 rows: 0.85 to 1.05 up to 66, 1.08 from 67 on.  129-160:
//                0.97 up to 10, 1.08 from there on; 161 and more: 1.05 to 1.3
//   4 bits, 64   49-96: 1.05 from 26 on, 1.15 from 50 on (n 12288, k 3072 at 96
//                rows 29.4 / 26.6 us).  129-160: 0.97 up to 7, then 1.1 to 1.4
//   8 bits, 64   49-96: 1.08 from 50 on.  129 and more as 4 bits
//   8 bits, 128  up to 128 rows 0.85 to 1.0.  129-160: 0.86 to 0.99 up to 66,
//                then 1.03; 161-256: 0.9 to 1.0 up to 34, then 1.04; 257 and
//                more: 1.0 to 1.1.  With a gate up to 256 rows 1.0 up to 120 and
//                1.1 at 224, but n 16384, k 8192 82 / 116 us at 144 rows
// us, 4 bits, k 4096: n 28672 438 / 368 at 1500 rows; n 6144 118 / 90.
bool block_rows(const torch::Tensor& qweight, const torch::Tensor& scales,
                long m, long n, long k, long g, long bits, bool glu) {
  const long size = n * k, M = 1l << 20;
  const bool wide = g % 128 == 0;                // groups
  bool gains;
  if (bits == 8 && wide)
    gains = m > 256 ||
            (m > 128 && size > (glu ? 160 : m <= 160 ? 66 : 34) * M);
  else if (m > 128)
    gains = m > 160 || size > (wide ? 10 : 7) * M;
  else
    gains = m > 96 || size >= 62 * M ||
            (m > 64 && bits == 4 && !wide && size > 26 * M);
  return gains && lfmq_dq_block_ok(qweight.data_ptr(), scales.data_ptr(), n, k,
                                   g, bits);
}

// room for the sums of x's groups, where a product of `rows` rows gains by them
torch::Tensor panel_sums(const torch::Tensor& x, long rows, long n, long g,
                         long bits) {
  const long k = x.size(1), groups = x.size(0) * (k / g);
  if (!lfmq_dq_panel_gains(rows, n, k, g, bits) || groups * 8 >= 1l << 32) return {};
  return torch::empty({groups * 3 / 2}, x.options().dtype(torch::kInt32));
}

void dq_block(const torch::Tensor& x, const torch::Tensor& qweight,
              const torch::Tensor& scales, const torch::Tensor& qzeros,
              const void* bias, torch::Tensor& y, long g, long bits, bool glu) {
  const int m = (int)x.size(0), k = (int)x.size(1), n = (int)qweight.size(0);
  const DqBlockPlan P =
      lfmq_dq_block_plan(m, n, k, (int)g, (int)bits, glu);
  torch::Tensor part;
  if (P.part > 0)
    part = torch::empty({P.part}, x.options().dtype(torch::kFloat32));
  const torch::Tensor sums = panel_sums(x, m, n, g, bits);
  CHECK_HIP(lfmq_dq_block(qweight.data_ptr(), scales.data_ptr(),
                          qzeros.data_ptr(), x.data_ptr(), y.data_ptr(), bias,
                          P.part > 0 ? part.data_ptr() : nullptr,
                          sums.defined() ? sums.data_ptr() : nullptr, m, n, k,
                          (int)g, (int)bits, glu, P, stream()));
}

// The product for 17 to 128 rows whose loads are several stages ahead: where it
// is faster than dq_rows (up to 48 rows), dq_tile and dq_block.  The time of
// those / of this one (m rows), the mean over 6700 measured calls by size, that
// is n k in millions (2^20):
//   4 bits, 128  49-96 rows: 1.05 to 1.2 up to 66 (dq_block 0.97 to 1.05), 0.94
//                from 67 on (1.08).  97-128: 1.25 up to 17, then dq_block
//   4 bits, 64   49-64: 1.1 (and so dq_block).  65-96: 1.08 up to 26, then 1.02
//                and dq_block 1.12
//   8 bits, 64   49-64: 1.15 to 1.3, dq_block 1.0 to 1.15.  65-96: 1.1 up to 60,
//                then the same as dq_block.  97-128: 1.08 up to 34, 1.04 (1.07)
//   8 bits, 128  49-128: 1.1 up to 58 and for k 2048 (n 32000 1.2), 0.93 from 64
//                on (dq_block 0.98)
// Up to 48 rows of 16 million weights, groups of 64: n 4096, k 4096 10.9 / 12.6
// at 17 rows, with a gate 24 / 13.  81 to 104 blocks of 128 columns in groups of
// 128 fill two thirds of the CUs with two parts, and gain nothing by a third: n
// 11008, k 4096 27.0 / 30.8 at 80 rows, 10240 29.3 / 23.8.  97 rows of short k,
// groups of 128: n 24576, k 1024 18.1 / 23.8 (dq_block 16.1).
// block: dq_block would take the call.
// Below 4 million weights rows of x in registers up to 96 (n 2048, k 2048 9.7 /
// 9.9 at 96 rows).
bool short_rows(const torch::Tensor& qweight, long m, long n, long k, long g,
                long bits, bool glu, bool block) {
  const long size = n * k, M = 1l << 20;
  const bool wide = g % 128 == 0;                // groups
  bool gains;
  if (m <= 48)
    gains = n >= 4096 && size >= (wide || glu ? 16 : 20) * M &&
            (k >= 4096 || size >= 48 * M);
  else if (bits == 8 && wide)
    gains = k <= 2048 || size < (m <= 96 ? 58 : 63) * M;
  else if (m > 96)
    gains = (k <= 4096 && size <= 17 * M) ||
            (size <= 34 * M &&
             (bits == 8 || (k <= 2048 && (n <= 16384 || !wide))));
  else if (bits == 8)
    gains = m <= 64 || size < (m <= 80 ? 66 : 62) * M;
  else
    gains = wide || m <= 64 ? size < 66 * M : size < 62 * M && !block;
  const long blocks = (n + 127) / 128;
  if (wide && m > 48 && k >= 4096 && blocks > 80 && blocks <= 104) gains = false;
  return m > 16 && m <= 128 && n > 0 && gains && tile_addresses(n, k, bits) &&
         lfmq_dq_tile_ok((int)k, (int)g) &&
         (uintptr_t)qweight.data_ptr() % 16 == 0;
}

// What goes with whole rows of a product: a factor of x's rows, and what follows
// rows of the result, which the sum of parts takes along if there is one.
struct RowWays {
  const float* scale = nullptr;
  const DqRowEnd* end = nullptr;
  bool* ended = nullptr;
  // where the parts go that a launch of the caller's adds up (dq_mid, dq_short)
  torch::Tensor* parts = nullptr;
  int* count = nullptr;
  bool keeps(const torch::Tensor& part, int splits) const {
    if (parts == nullptr) return false;
    *parts = part;
    *count = splits;
    return true;
  }
  const DqRowEnd* ends() const {           // for a launch that sums parts
    if (end != nullptr) *ended = true;
    return end;
  }
};

// The product whose workgroups share k among eight waves (dq_mid), where it is faster;
// mb 0: it is not.
DqMidPlan mid_plan(const torch::Tensor& qweight, long m, long n, long k, long g,
                   long bits, bool glu) {
  if (m <= 16 || m > 768 || n <= 0 || n % 8 || !tile_addresses(n, k, bits) ||
      !lfmq_dq_tile_ok((int)k, (int)g) || (uintptr_t)qweight.data_ptr() % 16)
    return {};
  const DqMidPlan P =
      lfmq_dq_mid_plan((int)m, (int)n, (int)k, (int)g, (int)bits, glu);
  return lfmq_dq_mid_gains(P, m, n, k, g, (int)bits, glu) ? P : DqMidPlan{};
}

void dq_short(const torch::Tensor& x, const torch::Tensor& qweight,
              const torch::Tensor& scales, const torch::Tensor& qzeros,
              const void* bias, const void* resid, torch::Tensor& y, long g,
              long bits, bool glu, const RowWays& ways) {
  const int m = (int)x.size(0), k = (int)x.size(1), n = (int)qweight.size(0);
  const DqShortPlan P = lfmq_dq_short_plan(m, n, k, (int)g, (int)bits, glu);
  DqArgs A{};
  torch::Tensor part;
  if (P.splits > 1) {
    part = torch::empty({(long)P.splits * m * n},
                        x.options().dtype(torch::kFloat32));
    A.part = part.data_ptr<float>();
  }
  A.w = (const char*)qweight.data_ptr();
  A.scales = (const unsigned short*)scales.data_ptr();
  A.zeros = (const u32*)qzeros.data_ptr();
  A.x = (const unsigned short*)x.data_ptr();
  A.y = (unsigned short*)y.data_ptr();
  A.bias = (const unsigned short*)bias;
  A.resid = (const unsigned short*)resid;
  A.m = m;
  A.n = n;
  A.k = k;
  A.g = (int)g;
  A.splits = P.splits;
  A.row_scale = ways.scale;
  CHECK_HIP(lfmq_dq_short(A, P, (int)bits, glu, stream()));
  if (P.splits > 1 && !ways.keeps(part, P.splits))
    CHECK_HIP(lfmq_dq_rows_sum(part.data_ptr(), y.data_ptr(), bias, resid, m, n,
                               P.splits, glu, stream(), ways.scale,
                               ways.ends()));
}

void dq_mid(const DqMidPlan& P, const torch::Tensor& x, const torch::Tensor& qweight,
            const torch::Tensor& scales, const torch::Tensor& qzeros,
            const void* bias, const void* resid, torch::Tensor& y, long g,
            long bits, bool glu, const RowWays& ways) {
  const int m = (int)x.size(0), k = (int)x.size(1), n = (int)qweight.size(0);
  DqArgs A{};
  torch::Tensor part;
  if (P.splits > 1) {
    part = torch::empty({(long)P.splits * m * n},
                        x.options().dtype(torch::kFloat32));
    A.part = part.data_ptr<float>();
  }
  A.w = (const char*)qweight.data_ptr();
  A.scales = (const unsigned short*)scales.data_ptr();
  A.zeros = (const u32*)qzeros.data_ptr();
  A.x = (const unsigned short*)x.data_ptr();
  A.y = (unsigned short*)y.data_ptr();
  A.bias = (const unsigned short*)bias;
  A.resid = (const unsigned short*)resid;
  A.m = m;
  A.n = n;
  A.k = k;
  A.g = (int)g;
  A.splits = P.splits;
  A.row_scale = ways.scale;
  CHECK_HIP(lfmq_dq_mid(A, P, (int)bits, glu, stream()));
  if (P.splits > 1 && !ways.keeps(part, P.splits))
    CHECK_HIP(lfmq_dq_rows_sum(part.data_ptr(), y.data_ptr(), bias, resid, m, n,
                               P.splits, false, stream(), ways.scale,
                               ways.ends()));
}

torch::Tensor rmsnorm(torch::Tensor x, torch::Tensor w, double eps,
                      c10::optional<torch::Tensor> residual);
torch::Tensor silu_mul_fused(torch::Tensor gate_up);

torch::Tensor linear(torch::Tensor x, const torch::Tensor& qweight,
                     const torch::Tensor& scales, const torch::Tensor& qzeros,
                     long bits, long g, const c10::optional<torch::Tensor>& bias,
                     const c10::optional<torch::Tensor>& resid, double rms_eps,
                     long cols_hint, const RowWays& ways) {
  check_t(x, torch::kBFloat16, "x");
  check_t(qweight, torch::kInt32, "qweight");
  check_t(scales, torch::kBFloat16, "scales");
  check_t(qzeros, torch::kInt32, "qzeros");
  TORCH_CHECK(x.dim() == 2, "x must be [m, k]");
  TORCH_CHECK(g > 0, "groups have at least one column");
  const int m = (int)x.size(0), k = (int)x.size(1);
  const int n = (int)qweight.size(0);
  TORCH_CHECK(qweight.size(1) == (long)k * bits / 32, "qweight/k mismatch");
  const bool one = cols_hint == 0 && m == 1 && in_pairs(scales) &&
                   lfmq_dq_row_ok(n, k, (int)g);
  // more groups than the kernels with the norm in them hold scales of (381
  // and 128): the norm apart
  if (rms_eps >= 0 && m <= 4 && k > 128 * g && !one &&
      !lfmq_dq_rows_ok(m, n, k, (int)g, true)) {
    x = rmsnorm(x, torch::ones({k}, x.options()), rms_eps, c10::nullopt);
    rms_eps = -1;
  }
  if ((uintptr_t)x.data_ptr() % 16) x = x.clone();  // 16-byte loads to LDS
  const void* bptr = nullptr;
  if (bias.has_value()) {
    check_t(*bias, torch::kBFloat16, "bias");
    bptr = bias->data_ptr();
  }
  const void* rptr = nullptr;
  if (resid.has_value()) {
    check_t(*resid, torch::kBFloat16, "resid");
    rptr = resid->data_ptr();
  }
  auto y = torch::empty({m, n}, x.options());
  // What is left by dq_row, dq_wide, dq_mid, dq_short and dq_block, whose rules go
  // first: a wave a few columns (GEMV), rows of x in registers, x through LDS.  us
  // of the last two: n 3072, k 8192 (4 bits) 14.5 / 17.1 at 32 rows, 17.7 / 17.1 at
  // 33, 25.5 / 18.7 at 49; n 16384, k 2048 (8 bits, groups of 64) 18.4 / 21.4 at 48,
  // 30.7 / 21.6 at 49.
  const bool rms = rms_eps >= 0, scaled = ways.scale != nullptr;
  const bool tile = tile_addresses(n, k, bits);
  const bool large = tile && !rms && k >= 4096 && (long)n * k >= 24l << 20 &&
                     (rptr == nullptr ||
                      lfmq_dq_tile_splits(m, n, k, (int)g) > 1);
  // a product that a few workgroups do whole: n 2048, k 2048 9.7 / 12.9 at 77
  // rows; n 3072 14.1 / 13.6
  const bool small = !rms && rptr == nullptr && (long)n * k <= 4l << 20;
  const bool by_rows = (cols_hint == 0 ? m >= rows_from(bits, n, k, g)
                                       : cols_hint == 6 && m > 4) &&
                       (!tile || m <= (scaled ? 48 : large ? 32 : small ? 96 : 48)) &&
                       lfmq_dq_rows_ok(m, n, k, (int)g, rms);
  const bool block = rptr == nullptr && !scaled &&
                     block_rows(qweight, scales, m, n, k, g, bits, false);
  const DqMidPlan plan = cols_hint == 0 && !rms
                             ? mid_plan(qweight, m, n, k, g, bits, false)
                             : DqMidPlan{};
  const bool mid = plan.mb > 0;
  const bool few = cols_hint == 0 && !rms && !(small && by_rows) &&
                   short_rows(qweight, m, n, k, g, bits, false, block);
  TORCH_CHECK(!scaled || (m > 16 && m <= 48 && (by_rows || few || mid)),
              "factors of rows are for 17 to 48 of them");
  if (m > 16) {
    TORCH_CHECK((by_rows || !rms) && (m <= 48 || rptr == nullptr),
                "fused rms/resid is a decode (m <= 48) path");
    TORCH_CHECK(lfmq_dq_tile_ok(k, (int)g),
                "more than 16 rows need groups of a multiple of 64 that "
                "divide k");
  }
  torch::Tensor part;
  auto parts = [&](int splits) -> void* {
    if (splits == 1) return nullptr;
    part = torch::empty({(long)splits * m * n},
                        x.options().dtype(torch::kFloat32));
    return part.data_ptr();
  };
  if (one) {
    CHECK_HIP(lfmq_dq_row(qweight.data_ptr(), scales.data_ptr(),
                          qzeros.data_ptr(), x.data_ptr(), y.data_ptr(), bptr,
                          rptr, n, k, (int)g, (int)bits, (float)rms_eps, false,
                          stream()));
  } else if (cols_hint == 0 && in_pairs(scales) &&
             wide_rows(m, n, k, g, bits, false)) {
    CHECK_HIP(lfmq_dq_wide(qweight.data_ptr(), scales.data_ptr(),
                           qzeros.data_ptr(), x.data_ptr(), y.data_ptr(), bptr,
                           rptr, m, n, k, (int)g, (int)bits, (float)rms_eps,
                           false, stream()));
  } else if (mid) {
    dq_mid(plan, x, qweight, scales, qzeros, bptr, rptr, y, g, bits, false, ways);
  } else if (few) {
    dq_short(x, qweight, scales, qzeros, bptr, rptr, y, g, bits, false,
             ways);
  } else if (by_rows) {
    const int splits = rms ? 1 : lfmq_dq_rows_splits(m, n, k, (int)g);
    CHECK_HIP(lfmq_dq_rows(qweight.data_ptr(), scales.data_ptr(),
                           qzeros.data_ptr(), x.data_ptr(), y.data_ptr(), bptr,
                           rptr, parts(splits), m, n, k, (int)g, (int)bits,
                           splits, (float)rms_eps, false, stream(), ways.scale,
                           splits > 1 ? ways.ends() : nullptr));
  } else if (m <= 16) {
    CHECK_HIP(lfmq_dq_gemv(qweight.data_ptr(), scales.data_ptr(),
                           qzeros.data_ptr(), x.data_ptr(), y.data_ptr(), bptr,
                           rptr, m, n, k, (int)g, (int)bits, (float)rms_eps,
                           (int)cols_hint, stream()));
  } else if (block) {
    dq_block(x, qweight, scales, qzeros, bptr, y, g, bits, false);
  } else {
    const int splits = lfmq_dq_tile_splits(m, n, k, (int)g);
    CHECK_HIP(lfmq_dq_tile(qweight.data_ptr(), scales.data_ptr(),
                           qzeros.data_ptr(), x.data_ptr(), y.data_ptr(), bptr,
                           rptr, parts(splits), m, n, k, (int)g, (int)bits,
                           splits, false, stream(),
                           splits > 1 ? ways.ends() : nullptr));
  }
  return y;
}

torch::Tensor dq_linear(torch::Tensor x, torch::Tensor qweight,
                        torch::Tensor scales, torch::Tensor qzeros, long bits,
                        long g, c10::optional<torch::Tensor> bias,
                        c10::optional<torch::Tensor> resid, double rms_eps,
                        long cols_hint) {
  return linear(x, qweight, scales, qzeros, bits, g, bias, resid, rms_eps,
                cols_hint, {});
}

// dq_linear of 3 to 16 rows whose k is in parts that one launch adds up, with
// `tickets` (zeros before and afterwards, of nobody else meanwhile); None: it gains
// nothing by them.
c10::optional<torch::Tensor> dq_linear_parts(
    torch::Tensor x, torch::Tensor qweight, torch::Tensor scales,
    torch::Tensor qzeros, long bits, long g, c10::optional<torch::Tensor> bias,
    c10::optional<torch::Tensor> resid, torch::Tensor tickets) {
  check_t(x, torch::kBFloat16, "x");
  check_t(qweight, torch::kInt32, "qweight");
  check_t(scales, torch::kBFloat16, "scales");
  check_t(qzeros, torch::kInt32, "qzeros");
  check_t(tickets, torch::kInt32, "tickets");
  TORCH_CHECK(x.dim() == 2, "x must be [m, k]");
  TORCH_CHECK(g > 0, "groups have at least one column");
  const long m = x.size(0), k = x.size(1), n = qweight.size(0);
  TORCH_CHECK(qweight.size(1) == k * bits / 32, "qweight/k mismatch");
  if (!part_rows(m, n, k, g, bits) || !in_pairs(scales) ||
      (uintptr_t)x.data_ptr() % 16 || (uintptr_t)qweight.data_ptr() % 16)
    return c10::nullopt;
  const int parts = lfmq_dq_wide_parts((int)m, (int)n, (int)k, (int)g, (int)bits);
  if (parts == 0 || tickets.numel() < lfmq_dq_wide_part_blocks((int)n, parts))
    return c10::nullopt;
  auto vector = [&](const c10::optional<torch::Tensor>& t, const char* name,
                    long size) -> const void* {
    if (!t.has_value()) return nullptr;
    check_t(*t, torch::kBFloat16, name);
    TORCH_CHECK(t->numel() == size, name, " has another size");
    return t->data_ptr();
  };
  const void* b = vector(bias, "bias", n);
  const void* r = vector(resid, "resid", m * n);
  auto y = torch::empty({m, n}, x.options());
  auto part = torch::empty({(n + 15) / 16 * parts * 256}, x.options().dtype(torch::kFloat32));
  CHECK_HIP(lfmq_dq_wide_in_parts(
      qweight.data_ptr(), scales.data_ptr(), qzeros.data_ptr(), x.data_ptr(),
      y.data_ptr(), b, r, part.data_ptr(), tickets.data_ptr(), (int)m, (int)n, (int)k,
      (int)g, (int)bits, stream()));
  return y;
}

// 1 / sqrt(mean x^2 + eps) of each row, fp32
torch::Tensor row_scale(torch::Tensor x, double eps) {
  check_t(x, torch::kBFloat16, "x");
  TORCH_CHECK(x.dim() == 2, "x must be [m, k]");
  auto s = torch::empty({x.size(0)}, x.options().dtype(torch::kFloat32));
  CHECK_HIP(lfmq_row_scale(x.data_ptr(), s.data_ptr(), (int)x.size(0),
                           (int)x.size(1), (float)eps, stream()));
  return s;
}

const float* factors(const c10::optional<torch::Tensor>& scale, long m) {
  if (!scale.has_value()) return nullptr;
  check_t(*scale, torch::kFloat32, "row scale");
  TORCH_CHECK(scale->numel() == m, "one factor a row");
  return scale->data_ptr<float>();
}

// whether a workgroup of the sum of parts can hold a row and read beside it
bool rows_end(int n, const c10::optional<torch::Tensor>& bias,
              const c10::optional<torch::Tensor>& add, const void* w) {
  auto even = [](const c10::optional<torch::Tensor>& t) {
    return !t.has_value() || (uintptr_t)t->data_ptr() % 8 == 0;
  };
  return lfmq_dq_row_end_ok(n) && even(bias) && even(add) &&
         (uintptr_t)w % 8 == 0;
}

// y = x W^T (+ bias) in bf16, then {rmsnorm(y + residual) w, y + residual}: in the
// launch that adds up the product's parts where it has some
std::vector<torch::Tensor> dq_linear_norm(
    torch::Tensor x, torch::Tensor qweight, torch::Tensor scales,
    torch::Tensor qzeros, long bits, long g, c10::optional<torch::Tensor> bias,
    torch::Tensor residual, torch::Tensor w, double eps) {
  check_t(residual, torch::kBFloat16, "residual");
  check_t(w, torch::kBFloat16, "w");
  const int m = (int)x.size(0), n = (int)qweight.size(0);
  TORCH_CHECK(residual.numel() == (long)m * n && w.numel() == n,
              "a residual and a weight for each column of the result");
  auto h = torch::empty({m, n}, x.options());
  RowWays ways{};
  DqRowEnd end{};
  bool ended = false;
  end.normed = (unsigned short*)h.data_ptr();
  end.to = (const unsigned short*)residual.data_ptr();
  end.w = (const unsigned short*)w.data_ptr();
  end.eps = (float)eps;
  ways.ended = &ended;
  if (rows_end(n, bias, residual, w.data_ptr())) ways.end = &end;
  auto y = linear(x, qweight, scales, qzeros, bits, g, bias, c10::nullopt, -1.0,
                  0, ways);
  if (ended) return {h, y};
  auto sum = torch::empty_like(y);
  CHECK_HIP(lfmq_rmsnorm(y.data_ptr(), residual.data_ptr(), w.data_ptr(),
                         h.data_ptr(), sum.data_ptr(), m, n, (float)eps,
                         stream()));
  return {h, sum};
}

// Rows of x times their factors (17 to 48 rows); eps >= 0: also row_scale of the
// result, from the sum of the product's parts where it has some, else by a launch
// of its own, and not at all without `apart`
std::vector<torch::Tensor> dq_linear_scaled(
    torch::Tensor x, c10::optional<torch::Tensor> scale, torch::Tensor qweight,
    torch::Tensor scales, torch::Tensor qzeros, long bits, long g,
    c10::optional<torch::Tensor> bias, c10::optional<torch::Tensor> resid,
    double eps, bool apart) {
  const int m = (int)x.size(0), n = (int)qweight.size(0);
  if (resid.has_value())
    TORCH_CHECK(resid->numel() == (long)m * n, "one residual a result");
  RowWays ways{factors(scale, m)};
  DqRowEnd end{};
  bool ended = false;
  torch::Tensor out;
  if (eps >= 0) {
    out = torch::empty({m}, x.options().dtype(torch::kFloat32));
    end.scale = out.data_ptr<float>();
    end.eps = (float)eps;
    ways.ended = &ended;
    if (rows_end(n, bias, resid, nullptr)) ways.end = &end;
  }
  auto y = linear(x, qweight, scales, qzeros, bits, g, bias, resid, -1.0, 0,
                  ways);
  if (eps < 0 || (!ended && !apart)) return {y};
  if (!ended)
    CHECK_HIP(lfmq_row_scale(y.data_ptr(), out.data_ptr(), m, n, (float)eps,
                             stream()));
  return {y, out};
}


torch::Tensor rmsnorm(torch::Tensor x, torch::Tensor w, double eps,
                      c10::optional<torch::Tensor> residual) {
  check_t(x, torch::kBFloat16, "x");
  check_t(w, torch::kBFloat16, "w");
  const int hidden = (int)x.size(-1);
  const int rows = (int)(x.numel() / hidden);
  auto y = torch::empty_like(x);
  const void* rptr = nullptr;
  if (residual.has_value()) {
    check_t(*residual, torch::kBFloat16, "residual");
    rptr = residual->data_ptr();
  }
  CHECK_HIP(lfmq_rmsnorm(x.data_ptr(), rptr, w.data_ptr(), y.data_ptr(),
                         nullptr, rows, hidden, (float)eps, stream()));
  return y;
}

std::vector<torch::Tensor> rmsnorm_residual(torch::Tensor x,
                                            torch::Tensor residual,
                                            torch::Tensor w, double eps) {
  check_t(x, torch::kBFloat16, "x");
  check_t(residual, torch::kBFloat16, "residual");
  check_t(w, torch::kBFloat16, "w");
  const int hidden = (int)x.size(-1);
  const int rows = (int)(x.numel() / hidden);
  auto y = torch::empty_like(x);
  auto res_out = torch::empty_like(x);
  CHECK_HIP(lfmq_rmsnorm(x.data_ptr(), residual.data_ptr(), w.data_ptr(),
                         y.data_ptr(), res_out.data_ptr(), rows, hidden,
                         (float)eps, stream()));
  return {y, res_out};
}

void rope(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
          torch::Tensor inv_freq) {
  check_t(q, torch::kBFloat16, "q");
  check_t(k, torch::kBFloat16, "k");
  check_t(positions, torch::kInt32, "positions");
  check_t(inv_freq, torch::kFloat32, "inv_freq");
  TORCH_CHECK(q.dim() == 4 && k.dim() == 4, "q/k must be [b, s, h, d]");
  const int b = (int)q.size(0), s = (int)q.size(1);
  const int hq = (int)q.size(2), d = (int)q.size(3);
  const int hkv = (int)k.size(2);
  TORCH_CHECK(positions.numel() == s, "positions must have s entries");
  CHECK_HIP(lfmq_rope(q.data_ptr(), k.data_ptr(), positions.data_ptr(),
                      inv_freq.data_ptr(), b * s, s, hq, hkv, d, stream()));
}

torch::Tensor silu_mul(torch::Tensor gate, torch::Tensor up) {
  check_t(gate, torch::kBFloat16, "gate");
  check_t(up, torch::kBFloat16, "up");
  auto y = torch::empty_like(gate);
  CHECK_HIP(lfmq_silu_mul(gate.data_ptr(), up.data_ptr(), y.data_ptr(),
                          gate.numel(), stream()));
  return y;
}

torch::Tensor silu_mul_fused(torch::Tensor gate_up) {
  check_t(gate_up, torch::kBFloat16, "gate_up");
  const long inter = gate_up.size(-1) / 2;
  const long rows = gate_up.numel() / (2 * inter);
  auto sizes = gate_up.sizes().vec();
  sizes.back() = inter;
  auto y = torch::empty(sizes, gate_up.options());
  CHECK_HIP(lfmq_silu_mul_fused(gate_up.data_ptr(), y.data_ptr(), rows,
                                (int)inter, stream()));
  return y;
}

torch::Tensor residual_add(torch::Tensor a, torch::Tensor b) {
  check_t(a, torch::kBFloat16, "a");
  check_t(b, torch::kBFloat16, "b");
  auto y = torch::empty_like(a);
  CHECK_HIP(lfmq_residual_add(a.data_ptr(), b.data_ptr(), y.data_ptr(),
                              a.numel(), stream()));
  return y;
}

void kv_append(torch::Tensor kc, torch::Tensor vc, torch::Tensor kn,
               torch::Tensor vn, long pos0) {
  check_t(kc, torch::kBFloat16, "k_cache");
  check_t(vc, torch::kBFloat16, "v_cache");
  check_t(kn, torch::kBFloat16, "k_new");
  check_t(vn, torch::kBFloat16, "v_new");
  // caches [b, hkv, tmax, d]; new [b, s, hkv, d] (token-major)
  const int b = (int)kc.size(0), hkv = (int)kc.size(1);
  const int tmax = (int)kc.size(2), d = (int)kc.size(3);
  const int s = (int)kn.size(1);
  TORCH_CHECK(kn.size(0) == b && kn.size(2) == hkv && kn.size(3) == d,
              "k_new shape mismatch");
  CHECK_HIP(lfmq_kv_append(kc.data_ptr(), vc.data_ptr(), kn.data_ptr(),
                           vn.data_ptr(), b, s, hkv, d, tmax, (int)pos0,
                           stream()));
}

torch::Tensor attn_decode(torch::Tensor q, torch::Tensor kc, torch::Tensor vc,
                          long seq_len, double scale,
                          c10::optional<torch::Tensor> t_dev) {
  check_t(q, torch::kBFloat16, "q");
  check_t(kc, torch::kBFloat16, "k_cache");
  check_t(vc, torch::kBFloat16, "v_cache");
  const int b = (int)q.size(0), hq = (int)q.size(1), d = (int)q.size(3);
  const int hkv = (int)kc.size(1), tmax = (int)kc.size(2);
  // graph mode (t_dev set): seq_len is MAX T; grid fixed, T read on device
  TORCH_CHECK(hq % hkv == 0, "query heads must share key heads evenly");
  const int splits = lfmq_attn_decode_splits(b, hq, hkv, (int)seq_len, d);
  auto scratch = torch::empty({(long)b * hq * splits * (d + 2)},
                              q.options().dtype(torch::kFloat32));
  auto o = torch::empty_like(q);
  const void* tptr = nullptr;
  if (t_dev.has_value()) {
    check_t(*t_dev, torch::kInt32, "t_dev");
    tptr = t_dev->data_ptr();
  }
  CHECK_HIP(lfmq_attn_decode(q.data_ptr(), kc.data_ptr(), vc.data_ptr(),
                             o.data_ptr(), scratch.data_ptr(), b, hq, hkv,
                             tmax, (int)seq_len, tptr, d, splits,
                             (float)scale, stream()));
  return o;
}

// flash prefill (csrc/attn_prefill.hip): q [b,s,hq*d] roped,
// caches [b,hkv,tmax,d] holding rows [0, pos0+s).  d == 128 only.
torch::Tensor attn_prefill(torch::Tensor q, torch::Tensor kc,
                           torch::Tensor vc, long hq, long pos0,
                           double scale) {
  check_t(q, torch::kBFloat16, "q");
  check_t(kc, torch::kBFloat16, "k_cache");
  check_t(vc, torch::kBFloat16, "v_cache");
  const int b = (int)q.size(0), s = (int)q.size(1);
  const int hkv = (int)kc.size(1), tmax = (int)kc.size(2);
  const int d = (int)kc.size(3);
  TORCH_CHECK(q.size(2) == hq * d, "q last dim != hq*d");
  TORCH_CHECK(pos0 + s <= tmax, "cache too small");
  // 16-byte loads to LDS
  if ((uintptr_t)kc.data_ptr() % 16) kc = kc.clone();
  if ((uintptr_t)vc.data_ptr() % 16) vc = vc.clone();
  auto o = torch::empty_like(q);
  CHECK_HIP(lfmq_attn_prefill(q.data_ptr(), kc.data_ptr(), vc.data_ptr(),
                              o.data_ptr(), b, s, (int)hq, hkv, tmax,
                              (int)pos0, d, (float)scale, stream()));
  return o;
}

torch::Tensor dq_gemv_gateup(torch::Tensor x, torch::Tensor qweight,
                             torch::Tensor scales, torch::Tensor qzeros,
                             long bits, long g, double rms_eps,
                             long cols_hint) {
  check_t(x, torch::kBFloat16, "x");
  check_t(qweight, torch::kInt32, "qweight");
  TORCH_CHECK(g > 0, "groups have at least one column");
  const int m = (int)x.size(0), k = (int)x.size(1);
  const int n = (int)qweight.size(0);
  TORCH_CHECK(qweight.size(1) == (long)k * bits / 32, "qweight/k mismatch");
  auto y = torch::empty({m, n / 2}, x.options());
  // as dq_linear
  const bool tile = tile_addresses(n, k, bits) && (long)m * k < 1l << 31;
  const bool large =
      tile && rms_eps < 0 && k >= 4096 && (long)n * k >= 24l << 20;
  const bool block = block_rows(qweight, scales, m, n, k, g, bits, true);
  const DqMidPlan plan = cols_hint == 0 && rms_eps < 0
                             ? mid_plan(qweight, m, n, k, g, bits, true)
                             : DqMidPlan{};
  if (plan.mb > 0) {
    if ((uintptr_t)x.data_ptr() % 16) x = x.clone();
    dq_mid(plan, x, qweight, scales, qzeros, nullptr, nullptr, y, g, bits, true, {});
    return y;
  }
  if (cols_hint == 0 && rms_eps < 0 && n % 2 == 0 &&
      short_rows(qweight, m, n, k, g, bits, true, block)) {
    if ((uintptr_t)x.data_ptr() % 16) x = x.clone();
    dq_short(x, qweight, scales, qzeros, nullptr, nullptr, y, g, bits, true, {});
    return y;
  }
  if (cols_hint == 0 && tile && n % 2 == 0 && m > (large ? 32 : 48) &&
      lfmq_dq_tile_ok(k, (int)g)) {
    TORCH_CHECK(rms_eps < 0, "fused rms is a decode (m <= 48) path");
    if ((uintptr_t)x.data_ptr() % 16) x = x.clone();
    if (block) {
      dq_block(x, qweight, scales, qzeros, nullptr, y, g, bits, true);
      return y;
    }
    const int splits = lfmq_dq_tile_splits(m, n, k, (int)g);
    torch::Tensor part;
    if (splits > 1)
      part = torch::empty({(long)splits * m * n},
                          x.options().dtype(torch::kFloat32));
    CHECK_HIP(lfmq_dq_tile(qweight.data_ptr(), scales.data_ptr(),
                           qzeros.data_ptr(), x.data_ptr(), y.data_ptr(),
                           nullptr, nullptr,
                           splits > 1 ? part.data_ptr() : nullptr, m, n, k,
                           (int)g, (int)bits, splits, true, stream()));
    return y;
  }
  if (cols_hint == 0 && n % 2 == 0 && in_pairs(scales) &&
      (m == 1 ? lfmq_dq_row_ok(n, k, (int)g) : wide_rows(m, n, k, g, bits, true))) {
    if ((uintptr_t)x.data_ptr() % 16) x = x.clone();
    if (m == 1)
      CHECK_HIP(lfmq_dq_row(qweight.data_ptr(), scales.data_ptr(),
                            qzeros.data_ptr(), x.data_ptr(), y.data_ptr(),
                            nullptr, nullptr, n, k, (int)g, (int)bits,
                            (float)rms_eps, true, stream()));
    else
      CHECK_HIP(lfmq_dq_wide(qweight.data_ptr(), scales.data_ptr(),
                             qzeros.data_ptr(), x.data_ptr(), y.data_ptr(),
                             nullptr, nullptr, m, n, k, (int)g, (int)bits,
                             (float)rms_eps, true, stream()));
    return y;
  }
  if (cols_hint == 0 && m >= rows_from(bits, n, k, g) && m <= 48 &&
      n % 2 == 0 && lfmq_dq_rows_ok(m, n, k, (int)g, true)) {
    if ((uintptr_t)x.data_ptr() % 16) x = x.clone();
    CHECK_HIP(lfmq_dq_rows(qweight.data_ptr(), scales.data_ptr(),
                           qzeros.data_ptr(), x.data_ptr(), y.data_ptr(),
                           nullptr, nullptr, nullptr, m, n, k, (int)g,
                           (int)bits, 1, (float)rms_eps, true, stream()));
    return y;
  }
  // what no kernel with the gate in it takes (the GEMV: 128 groups)
  if (k > 128 * g || (cols_hint == 0 && !tile && m > 48))
    return silu_mul_fused(dq_linear(x, qweight, scales, qzeros, bits, g,
                                    c10::nullopt, c10::nullopt, rms_eps, 0));
  CHECK_HIP(lfmq_dq_gemv_gateup(qweight.data_ptr(), scales.data_ptr(),
                                qzeros.data_ptr(), x.data_ptr(), y.data_ptr(),
                                m, n, k, (int)g, (int)bits, (float)rms_eps,
                                (int)cols_hint, stream()));
  return y;
}

// dq_gemv_gateup of rows of x times their factors (17 to 48 rows)
torch::Tensor dq_gateup_scaled(torch::Tensor x, torch::Tensor scale,
                               torch::Tensor qweight, torch::Tensor scales,
                               torch::Tensor qzeros, long bits, long g) {
  check_t(x, torch::kBFloat16, "x");
  check_t(qweight, torch::kInt32, "qweight");
  check_t(scales, torch::kBFloat16, "scales");
  check_t(qzeros, torch::kInt32, "qzeros");
  TORCH_CHECK(x.dim() == 2, "x must be [m, k]");
  TORCH_CHECK(g > 0, "groups have at least one column");
  const int m = (int)x.size(0), k = (int)x.size(1);
  const int n = (int)qweight.size(0);
  TORCH_CHECK(qweight.size(1) == (long)k * bits / 32, "qweight/k mismatch");
  TORCH_CHECK(m > 16 && m <= 48 && n % 2 == 0 &&
                  lfmq_dq_rows_ok(m, n, k, (int)g, true),
              "factors of rows are for 17 to 48 of them");
  RowWays ways{factors(scale, m)};
  if ((uintptr_t)x.data_ptr() % 16) x = x.clone();
  auto y = torch::empty({m, n / 2}, x.options());
  const DqMidPlan plan = mid_plan(qweight, m, n, k, g, bits, true);
  if (plan.mb > 0)
    dq_mid(plan, x, qweight, scales, qzeros, nullptr, nullptr, y, g, bits, true, ways);
  else if (short_rows(qweight, m, n, k, g, bits, true, false))
    dq_short(x, qweight, scales, qzeros, nullptr, nullptr, y, g, bits, true,
             ways);
  else
    CHECK_HIP(lfmq_dq_rows(qweight.data_ptr(), scales.data_ptr(),
                           qzeros.data_ptr(), x.data_ptr(), y.data_ptr(),
                           nullptr, nullptr, nullptr, m, n, k, (int)g,
                           (int)bits, 1, -1.f, true, stream(), ways.scale));
  return y;
}

// s rows from pos0 on for caches [b, hkv, tmax, d], before anything writes them:
// their places in the caches, an angle's factors and positions are there
void check_append(const torch::Tensor& kc, const torch::Tensor& vc,
                  const torch::Tensor& positions, const torch::Tensor& inv_freq,
                  long s, long pos0) {
  check_t(kc, torch::kBFloat16, "k_cache");
  check_t(vc, torch::kBFloat16, "v_cache");
  check_t(positions, torch::kInt32, "positions");
  check_t(inv_freq, torch::kFloat32, "inv_freq");
  TORCH_CHECK(kc.dim() == 4 && kc.sizes() == vc.sizes(),
              "caches must be [b, hkv, tmax, d]");
  TORCH_CHECK(pos0 >= 0 && s <= kc.size(2) && pos0 <= kc.size(2) - s,
              "KV cache overflow: ", pos0, " + ", s, " > ", kc.size(2));
  TORCH_CHECK(positions.numel() >= s, "positions must have s entries");
  TORCH_CHECK(inv_freq.numel() >= kc.size(3) / 2,
              "inv_freq must have d / 2 entries");
}

torch::Tensor qkv_rope_append(torch::Tensor qkv, torch::Tensor kc,
                              torch::Tensor vc, torch::Tensor positions,
                              torch::Tensor inv_freq, long hq, long pos0,
                              c10::optional<torch::Tensor> pos_dev) {
  check_t(qkv, torch::kBFloat16, "qkv");
  TORCH_CHECK(kc.dim() == 4 && kc.size(0) > 0 && (hq + 2 * kc.size(1)) * kc.size(3) > 0,
              "caches must be [b, hkv, tmax, d]");
  const int b = (int)kc.size(0), hkv = (int)kc.size(1);
  const int tmax = (int)kc.size(2), d = (int)kc.size(3);
  const int s = (int)(qkv.numel() / ((hq + 2 * hkv) * d)) / b;
  check_append(kc, vc, positions, inv_freq, s, pos0);
  auto q_out = torch::empty({b, s, hq, (long)d}, qkv.options());
  const void* pdev = nullptr;
  if (pos_dev.has_value()) {
    check_t(*pos_dev, torch::kInt32, "pos_dev");
    pdev = pos_dev->data_ptr();
  }
  CHECK_HIP(lfmq_qkv_rope_append(qkv.data_ptr(), q_out.data_ptr(),
                                 kc.data_ptr(), vc.data_ptr(),
                                 positions.data_ptr(), inv_freq.data_ptr(), b,
                                 s, (int)hq, hkv, d, tmax, (int)pos0, pdev,
                                 stream()));
  return q_out;
}

// A layer's kernels for a prompt, one after the other, from its normed input h [b,
// s, hidden] and what that was: {the next layer's normed input, what that was}.
// packed: weights, scales and zeros of qkv, o, gate and up, down; forms: bits and
// groups of each; biases of qkv, o and down.  Called one by one from Python these
// take the host 85 us a layer, this way 58.
std::vector<torch::Tensor> prompt_layer(
    torch::Tensor h, torch::Tensor residual, torch::Tensor kc, torch::Tensor vc,
    torch::Tensor positions, torch::Tensor inv_freq, long hq, long pos0,
    double scale, const std::vector<torch::Tensor>& packed,
    const std::vector<long>& forms,
    const std::vector<c10::optional<torch::Tensor>>& biases,
    torch::Tensor post_norm, double post_eps, torch::Tensor next_norm,
    double next_eps) {
  TORCH_CHECK(h.dim() == 3 && kc.dim() == 4 && packed.size() == 12 &&
                  forms.size() == 8 && biases.size() == 3,
              "a layer has four packed products");
  const auto sizes = h.sizes().vec();
  const long b = sizes[0], s = sizes[1];
  check_append(kc, vc, positions, inv_freq, s, pos0);
  TORCH_CHECK(kc.size(0) == b, "a cache of ", kc.size(0), " for ", b, " sequences");
  auto rows = [&](const torch::Tensor& t) { return t.view({b * s, t.size(-1)}); };
  torch::Tensor part, q;
  int splits = 0;
  RowWays ways{};
  const long d = kc.size(3), hkv = kc.size(1);
  if (d % 8 == 0 && b * s <= 65535 && packed[0].size(0) == (hq + 2 * hkv) * d &&
      ((uintptr_t)kc.data_ptr() | (uintptr_t)vc.data_ptr() |
       (uintptr_t)inv_freq.data_ptr()) % 16 == 0) {
    ways.parts = &part;
    ways.count = &splits;
  }
  auto qkv = linear(rows(h), packed[0], packed[1], packed[2], forms[0], forms[1],
                    biases[0], c10::nullopt, -1.0, 0, ways);
  if (splits > 1) {
    q = torch::empty({b, s, hq, d}, h.options());
    CHECK_HIP(lfmq_qkv_sum_rope_append(
        part.data_ptr(), splits,
        biases[0].has_value() ? biases[0]->data_ptr() : nullptr, q.data_ptr(),
        kc.data_ptr(), vc.data_ptr(), positions.data_ptr(), inv_freq.data_ptr(),
        (int)b, (int)s, (int)hq, (int)hkv, (int)d, (int)kc.size(2), (int)pos0,
        stream()));
  } else {
    q = qkv_rope_append(qkv, kc, vc, positions, inv_freq, hq, pos0, c10::nullopt);
  }
  auto o = attn_prefill(q.view({b, s, hq * q.size(3)}), kc, vc, hq, pos0, scale);
  auto r = dq_linear_norm(rows(o), packed[3], packed[4], packed[5], forms[2],
                          forms[3], biases[1], residual, post_norm, post_eps);
  auto g = dq_gemv_gateup(r[0], packed[6], packed[7], packed[8], forms[4],
                          forms[5], -1.0, 0);
  r = dq_linear_norm(g, packed[9], packed[10], packed[11], forms[6], forms[7],
                     biases[2], r[1], next_norm, next_eps);
  return {r[0].view(sizes), r[1].view(sizes)};
}

torch::Tensor greedy_sample(torch::Tensor logits) {
  check_t(logits, torch::kBFloat16, "logits");
  TORCH_CHECK(logits.dim() == 2, "logits must be [b, vocab]");
  const int b = (int)logits.size(0), vocab = (int)logits.size(1);
  auto out = torch::empty({b}, logits.options().dtype(torch::kInt64));
  auto sf = torch::empty({b * 64}, logits.options().dtype(torch::kFloat32));
  auto si = torch::empty({b * 64}, logits.options().dtype(torch::kInt32));
  CHECK_HIP(lfmq_argmax_rows(logits.data_ptr(), out.data_ptr(), sf.data_ptr(),
                             si.data_ptr(), b, vocab, stream()));
  return out;
}

void read_probe(torch::Tensor src, torch::Tensor sink, long row_bytes,
                long n_rows, long nt, long streams, long mode) {
  CHECK_HIP(lfmq_read_probe(src.data_ptr(), sink.data_ptr(), row_bytes,
                            n_rows, (int)nt, (int)streams, (int)mode,
                            stream()));
}

// one-kernel MoE routing: logits [t, E] bf16 -> (token of a slot, slot
// weights, first slots of the experts, experts that have any)
std::vector<torch::Tensor> moe_route(torch::Tensor logits, long topk) {
  check_t(logits, torch::kBFloat16, "logits");
  const int t = (int)logits.size(0), E = (int)logits.size(1);
  TORCH_CHECK(t <= 64, "moe_route takes up to 64 tokens");
  const auto i32 = logits.options().dtype(torch::kInt32);
  const auto f32 = logits.options().dtype(torch::kFloat32);
  auto src_tok = torch::empty({(long)t * topk}, i32);
  auto slot_w = torch::empty({(long)t * topk}, f32);
  auto pos = torch::empty({(long)t * topk}, i32);
  auto w = torch::empty({(long)t * topk}, f32);
  auto offsets = torch::empty({(long)E + 1}, i32);
  auto active = torch::empty({(long)E}, i32);
  CHECK_HIP(lfmq_moe_route(logits.data_ptr(), src_tok.data_ptr(),
                           slot_w.data_ptr(), pos.data_ptr(), w.data_ptr(),
                           offsets.data_ptr(), active.data_ptr(), nullptr, t,
                           E, (int)topk, 1, 0, stream()));
  return {src_tok, slot_w, offsets, active};
}

// Tiles of 16 rows, `lists` of them, of the grouped products that keep x and walk
// over columns, against those of dq_rows.  The time of rows / wide: k 2048 to
// 4096 and 8192 1.05 to 1.5, up to 4 lists up to 1.9; where k leaves many waves
// without a step (wide_rows) k 5632, n 2048 0.7 to 0.9 from 9 lists on, 1.1 with
// 4 bits in groups of 128; k 5120, n 16384 with a gate, groups of 64 0.8 to 0.95;
// k 3072, 4 bits in groups of 64 0.9 from 17 lists on.
bool wide_experts(int n, int k, long g, long bits, bool glu, long lists) {
  if (n < 2048 || k < 2048 ||
      !lfmq_dq_wide_ok(16, n, k, (int)g, (int)bits))
    return false;
  const int step = k <= 2048 ? 2048 : 4096;
  const int full = (int)(100l * k / (((long)k + step - 1) / step * step));
  if (k > 4096 && full < 70)
    return g == 128 ? bits == 4 || glu || lists <= 8 : !glu && lists <= 8;
  return bits == 8 || g == 128 || full >= 80 || lists <= 16;
}

// Rows a tile of the grouped products for `slots` rows over E experts.  us of
// a layer with tiles of 16 / 128 (4 bits but the third):
//   rows an expert             14         18         26         40
//   E 8,  k 4096, 14336    214 / 218  259 / 223  340 / 230  461 / 272
//   E 8,  k 2048, 8192      63 / 64    67 / 65    99 / 74   126 / 82
//   E 8,  k 2048, 4096      57 / 53    56 / 53    88 / 60   110 / 62
//   E 64, k 2048, 2048     118 / 133  142 / 131  186 / 145  246 / 165
//   E 16, k 1024, 2048      32 / 29    39 / 29    49 / 34    63 / 35
// With dq_tile (for groups that dq_block does not take) the first line's 128
// wins from 26: 364 us at 14 rows, 369 at 32; where there are more experts, and
// so tiles, from 18 (k 3072, 1536, 8 bits in groups of 128, at 19 rows: E 16 116
// / 83, E 64 387 / 282; E 8 at 16 0.9 of the time, at 25 1.1).  The last line's
// tiles of 16 are dq_rows', which reads x for each column.
long moe_tile(long slots, long E, long k_in, long g_in, long k_out,
              long g_out) {
  TORCH_CHECK(g_in > 0 && g_out > 0, "groups have at least one column");
  // (the first product has 2 k_out columns, the second k_in)
  const bool wide =
      wide_experts(2048, (int)k_in, g_in, 8, true, 1) && k_out >= 1024;
  const bool block =
      lfmq_dq_block_ok(nullptr, nullptr, 2 * k_out, k_in, g_in, 8) &&
      lfmq_dq_block_ok(nullptr, nullptr, k_in, k_out, g_out, 8);
  return slots > (!wide ? 14 : block ? 16 : E > 8 ? 18 : 26) * E &&
                 lfmq_dq_tile_ok((int)k_in, (int)g_in) &&
                 lfmq_dq_tile_ok((int)k_out, (int)g_out)
             ? 128
             : 16;
}

// routing for the grouped products: (token of a slot, slot and weight of a
// token's choice [t, topk], tiles of bm rows)
std::vector<torch::Tensor> moe_plan(torch::Tensor logits, long topk, long bm) {
  check_t(logits, torch::kBFloat16, "logits");
  TORCH_CHECK(bm > 0, "tiles have at least one row");
  const int t = (int)logits.size(0), E = (int)logits.size(1);
  const long slots = (long)t * topk;
  const int n_tiles = (int)(slots / bm + std::min((long)E, slots));
  const auto i32 = logits.options().dtype(torch::kInt32);
  auto src = torch::empty({slots}, i32);
  auto pos = torch::empty({t, topk}, i32);
  auto w = torch::empty({t, topk}, logits.options().dtype(torch::kFloat32));
  auto tiles = torch::empty({n_tiles, 3}, i32);
  CHECK_HIP(lfmq_moe_route(logits.data_ptr(), src.data_ptr(), nullptr,
                           pos.data_ptr(), w.data_ptr(), nullptr, nullptr,
                           tiles.data_ptr(), t, E, (int)topk, (int)bm, n_tiles,
                           stream()));
  return {src, pos, w, tiles};
}

// rows of x by expert (src: the row of a slot, else the slot itself): glu:
// bf16 [slots, n / 2] silu(gate) * up of W = [gate | up], else fp32 [slots, n]
torch::Tensor moe_linear(torch::Tensor x, c10::optional<torch::Tensor> src,
                         torch::Tensor tiles, torch::Tensor qweight,
                         torch::Tensor scales, torch::Tensor qzeros, long bits,
                         long g, bool glu, long bm) {
  check_t(x, torch::kBFloat16, "x");
  check_t(tiles, torch::kInt32, "tiles");
  check_t(qweight, torch::kInt32, "qweight");
  check_t(scales, torch::kBFloat16, "scales");
  check_t(qzeros, torch::kInt32, "qzeros");
  const int n = (int)qweight.size(1), k = (int)x.size(1);
  TORCH_CHECK(qweight.size(2) == (long)k * bits / 32, "qweight/k mismatch");
  TORCH_CHECK(g > 0, "groups have at least one column");
  TORCH_CHECK(x.numel() * 2 < 1l << 32, "x of 4 GiB or more");
  if ((uintptr_t)x.data_ptr() % 16) x = x.clone();  // 16-byte loads to LDS
  const void* sptr = nullptr;
  long slots = x.size(0);
  if (src.has_value()) {
    check_t(*src, torch::kInt32, "src");
    sptr = src->data_ptr();
    slots = src->numel();
  }
  TORCH_CHECK(bm == 16 || bm == 128, "tiles of 16 or 128 rows");
  // Tiles of 128 rows.  The time of dq_tile / dq_block is 1.1 to 4 but for 8 bits
  // in groups of 128: with a gate 0.8 to 1.0 from 25 rows an expert on, without
  // one (k in parts) 1.0 to 2.5, but 0.7 to 0.95 at k 1024.
  const bool block =
      bm == 128 && !(bits == 8 && g % 128 == 0 && (glu || k <= 1024)) &&
      lfmq_dq_block_ok(qweight.data_ptr(), scales.data_ptr(), n, k, g, bits);
  const int parts = block && !glu
                        ? lfmq_dq_block_slot_parts(slots, qweight.size(0), n, k,
                                                   (int)g, (int)bits)
                        : 1;
  const auto f32 = x.options().dtype(torch::kFloat32);
  auto y = glu ? torch::empty({slots, (long)n / 2}, x.options())
               : torch::empty({slots, (long)n}, f32);
  const int nt = (int)tiles.size(0);
  if (nt == 0) return y;
  torch::Tensor part;
  if (parts > 1) part = torch::empty({parts * slots, (long)n}, f32);
  if (block) {
    const torch::Tensor sums = panel_sums(x, slots, n, g, bits);
    CHECK_HIP(lfmq_dq_block_experts(
        qweight.data_ptr(), scales.data_ptr(), qzeros.data_ptr(), x.data_ptr(),
        sptr, tiles.data_ptr(), y.data_ptr(),
        parts > 1 ? part.data_ptr() : nullptr,
        sums.defined() ? sums.data_ptr() : nullptr, x.size(0), nt, n, k, (int)g,
        (int)bits, glu, parts, slots, stream()));
  } else if (bm == 128)
    CHECK_HIP(lfmq_dq_tile_experts(
        qweight.data_ptr(), scales.data_ptr(), qzeros.data_ptr(), x.data_ptr(),
        sptr, tiles.data_ptr(), y.data_ptr(), nt, n, k, (int)g, (int)bits, glu,
        stream()));
  else if (in_pairs(scales) && wide_experts(n, k, g, bits, glu, nt))
    CHECK_HIP(lfmq_dq_wide_experts(
        qweight.data_ptr(), scales.data_ptr(), qzeros.data_ptr(), x.data_ptr(),
        sptr, tiles.data_ptr(), y.data_ptr(), nt, n, k, (int)g, (int)bits, glu,
        stream()));
  else
    CHECK_HIP(lfmq_dq_rows_experts(
        qweight.data_ptr(), scales.data_ptr(), qzeros.data_ptr(), x.data_ptr(),
        sptr, tiles.data_ptr(), y.data_ptr(), nt, n, k, (int)g, (int)bits, glu,
        stream()));
  return y;
}

// y[t] = sum of a token's rows, weighted
torch::Tensor moe_sum(torch::Tensor rows, torch::Tensor pos, torch::Tensor w) {
  check_t(rows, torch::kFloat32, "rows");
  check_t(pos, torch::kInt32, "pos");
  check_t(w, torch::kFloat32, "w");
  const long t = pos.size(0), topk = pos.size(1), n = rows.size(1);
  auto y = torch::empty({t, n}, rows.options().dtype(torch::kBFloat16));
  CHECK_HIP(lfmq_moe_sum(rows.data_ptr(), pos.data_ptr(), w.data_ptr(),
                         y.data_ptr(), (int)t, (int)n, (int)topk, stream()));
  return y;
}

// slots already sorted by expert: `offsets` [E + 1] says where each begins
torch::Tensor grouped_tiles(torch::Tensor offsets, long slots) {
  check_t(offsets, torch::kInt32, "offsets");
  const int E = (int)offsets.numel() - 1;
  const int n_tiles = (int)(slots / 16 + std::min((long)E, slots));
  auto tiles = torch::empty({n_tiles, 3}, offsets.options());
  if (n_tiles > 0)
    CHECK_HIP(lfmq_moe_tiles(offsets.data_ptr(), tiles.data_ptr(), E, 16,
                             n_tiles, stream()));
  return tiles;
}

// For callers with sorted slots of their own.  `active`, the experts that have
// any, says nothing that `offsets` does not: not read.
torch::Tensor grouped_dq_gateup(torch::Tensor x, torch::Tensor src_tok,
                                torch::Tensor offsets, torch::Tensor qweight,
                                torch::Tensor scales, torch::Tensor qzeros,
                                long bits, long g,
                                c10::optional<torch::Tensor> active) {
  return moe_linear(x, src_tok, grouped_tiles(offsets, src_tok.numel()),
                    qweight, scales, qzeros, bits, g, true, 16);
}

torch::Tensor grouped_dq_linear(torch::Tensor x, torch::Tensor offsets,
                                torch::Tensor qweight, torch::Tensor scales,
                                torch::Tensor qzeros, long bits, long g) {
  return moe_linear(x, c10::nullopt, grouped_tiles(offsets, x.size(0)),
                    qweight, scales, qzeros, bits, g, false, 16)
      .to(torch::kBFloat16);
}

// y_f32[dst_tok[s]] += slot_w[s] * (x[s] W_e^T)
void grouped_dq_linear_scatter(torch::Tensor x, torch::Tensor offsets,
                               torch::Tensor dst_tok, torch::Tensor slot_w,
                               torch::Tensor y_f32, torch::Tensor qweight,
                               torch::Tensor scales, torch::Tensor qzeros,
                               long bits, long g,
                               c10::optional<torch::Tensor> active) {
  check_t(y_f32, torch::kFloat32, "y_f32");
  check_t(dst_tok, torch::kInt32, "dst_tok");
  check_t(slot_w, torch::kFloat32, "slot_w");
  TORCH_CHECK(y_f32.size(1) == qweight.size(1), "y_f32 width mismatch");
  const long slots = x.size(0);
  TORCH_CHECK(dst_tok.numel() >= slots && slot_w.numel() >= slots,
              "a token and a weight for every slot");
  auto rows = moe_linear(x, c10::nullopt, grouped_tiles(offsets, slots),
                         qweight, scales, qzeros, bits, g, false, 16);
  rows.mul_(slot_w.view({-1}).narrow(0, 0, slots).unsqueeze(1));
  // no expert's: not written
  auto none = at::arange(slots, offsets.options()).ge(offsets.select(0, -1));
  rows.masked_fill_(none.unsqueeze(1), 0);
  y_f32.index_add_(0, dst_tok.view({-1}).narrow(0, 0, slots), rows);
}

void advance_record(torch::Tensor state, torch::Tensor tok_buf,
                    torch::Tensor sampled, torch::Tensor ring) {
  check_t(state, torch::kInt32, "state");
  const int b = (int)tok_buf.size(0);
  const int ring_len = (int)ring.size(-1);
  CHECK_HIP(lfmq_advance_record(state.data_ptr(), tok_buf.data_ptr(),
                                sampled.data_ptr(), ring.data_ptr(), b,
                                ring_len, stream()));
}

torch::Tensor attn_decode_fused(torch::Tensor qkv, torch::Tensor kc,
                                torch::Tensor vc, long seq_len, double scale,
                                torch::Tensor inv_freq, long hq,
                                c10::optional<torch::Tensor> t_dev,
                                c10::optional<torch::Tensor> tickets) {
  check_t(qkv, torch::kBFloat16, "qkv");
  check_t(kc, torch::kBFloat16, "k_cache");
  check_t(vc, torch::kBFloat16, "v_cache");
  check_t(inv_freq, torch::kFloat32, "inv_freq");
  const int b = (int)kc.size(0), hkv = (int)kc.size(1);
  const int tmax = (int)kc.size(2), d = (int)kc.size(3);
  TORCH_CHECK(hq % hkv == 0, "query heads must share key heads evenly");
  const int splits = lfmq_attn_decode_splits(b, (int)hq, hkv, (int)seq_len, d);
  auto scratch = torch::empty({(long)b * hq * splits * (d + 2)},
                              qkv.options().dtype(torch::kFloat32));
  auto o = torch::empty({(long)b, 1L, hq * (long)d}, qkv.options());
  const void* tptr = nullptr;
  if (t_dev.has_value()) tptr = t_dev->data_ptr();
  void* tk = nullptr;
  if (tickets.has_value()) {
    check_t(*tickets, torch::kInt32, "tickets");
    TORCH_CHECK(tickets->numel() >= (long)b * hq, "tickets too small");
    tk = tickets->data_ptr();
  }
  CHECK_HIP(lfmq_attn_decode_fused(qkv.data_ptr(), kc.data_ptr(),
                                   vc.data_ptr(), o.data_ptr(),
                                   scratch.data_ptr(), inv_freq.data_ptr(), b,
                                   (int)hq, hkv, tmax, (int)seq_len, tptr, d,
                                   splits, (float)scale, tk, stream()));
  return o;
}

// persistent decode engine: one launch = one whole decode step (layers
// only; lm_head/sampling stay separate).  Granule buffers must be zeroed
// by the CALLER before every call (lfmq/models/engine.py does, inside the
// captured graph).  Returns nothing; output lands in xout.
void engine_step(torch::Tensor stream_t, long stream_per_cu, long nslot_ring,
                 long n_layers, long hidden, long inter, long nqkv, long hq,
                 long hkv, long log2g, double rms_eps, double attn_scale,
                 torch::Tensor inv_freq, torch::Tensor kc, torch::Tensor vc,
                 torch::Tensor state, torch::Tensor tok, torch::Tensor embed,
                 torch::Tensor final_w, torch::Tensor xout,
                 torch::Tensor g_qkv, torch::Tensor g_attn, torch::Tensor g_o,
                 torch::Tensor g_h, torch::Tensor g_down, torch::Tensor g_scr,
                 torch::Tensor tmo, c10::optional<torch::Tensor> prof,
                 long debug) {
  check_t(kc, torch::kBFloat16, "k_cache");
  check_t(vc, torch::kBFloat16, "v_cache");
  check_t(embed, torch::kBFloat16, "embed");
  check_t(final_w, torch::kBFloat16, "final_w");
  check_t(xout, torch::kBFloat16, "xout");
  check_t(inv_freq, torch::kFloat32, "inv_freq");
  check_t(state, torch::kInt32, "state");
  TORCH_CHECK(tok.scalar_type() == torch::kInt64, "tok must be int64");
  TORCH_CHECK(stream_t.scalar_type() == torch::kUInt8, "stream uint8");
  // kc: [L, 1, hkv, tmax, d] (stacked) or list-stacked contiguous
  const int tmax = (int)kc.size(-2), d = (int)kc.size(-1);
  EngineArgs a{};
  a.stream = (const char*)stream_t.data_ptr();
  a.stream_per_cu = (unsigned long long)stream_per_cu;
  a.n_slots_total = (int)((stream_per_cu + 16383) / 16384);
  a.nslot_ring = (int)nslot_ring;
  a.n_layers = (int)n_layers;
  a.hidden = (int)hidden;
  a.inter = (int)inter;
  a.nqkv = (int)nqkv;
  a.hq = (int)hq;
  a.hkv = (int)hkv;
  a.log2g = (int)log2g;
  a.rms_eps = (float)rms_eps;
  a.attn_scale = (float)attn_scale;
  a.inv_freq = (const float*)inv_freq.data_ptr();
  a.kc = (const unsigned short*)kc.data_ptr();
  a.vc = (const unsigned short*)vc.data_ptr();
  a.kv_layer_stride = (unsigned long long)hkv * tmax * d;
  a.tmax = tmax;
  a.nch_max = (tmax + 255) / 256;
  TORCH_CHECK(a.nch_max <= 64, "engine needs tmax <= 16384");
  a.T_dev = (const int*)state.data_ptr() + 1;  // state = {pos0, T, step}
  a.tok = (const long long*)tok.data_ptr();
  a.embed = (const unsigned short*)embed.data_ptr();
  a.final_w = (const unsigned short*)final_w.data_ptr();
  a.xout = (unsigned short*)xout.data_ptr();
  a.g_qkv = g_qkv.data_ptr();
  a.g_attn = g_attn.data_ptr();
  a.g_o = g_o.data_ptr();
  a.g_h = g_h.data_ptr();
  a.g_down = g_down.data_ptr();
  a.g_scr = g_scr.data_ptr();
  a.tmo = tmo.data_ptr();
  a.prof = prof.has_value()
               ? (unsigned long long*)prof->data_ptr()
               : nullptr;
  a.debug = (unsigned)debug;
  CHECK_HIP(lfmq_engine_step(&a, d, stream()));
}

void hessian_accum(torch::Tensor h, torch::Tensor x) {
  check_t(h, torch::kFloat32, "H");
  check_t(x, torch::kBFloat16, "x");
  const int t = (int)x.size(0), k = (int)x.size(1);
  TORCH_CHECK(h.size(0) == k && h.size(1) == k, "H must be [k, k]");
  if ((uintptr_t)x.data_ptr() % 16) x = x.clone();  // 16-byte loads to LDS
  CHECK_HIP(lfmq_hessian_accum(x.data_ptr(), h.data_ptr(), t, k, stream()));
}

// U upper triangular, U^T U = h^-1, and [1]: not 0 if h (its lower triangle)
// is not positive definite in fp32.  diag takes the place of h's diagonal
std::vector<torch::Tensor> chol_inverse(torch::Tensor h,
                                        c10::optional<torch::Tensor> diag) {
  check_t(h, torch::kFloat32, "h");
  TORCH_CHECK(h.dim() == 2 && h.size(0) == h.size(1) && h.size(0) > 0,
              "h must be [n, n]");
  const int n = (int)h.size(0);
  const void* dptr = nullptr;
  if (diag.has_value()) {
    check_t(*diag, torch::kFloat32, "diag");
    TORCH_CHECK(diag->numel() == n, "diag must be [n]");
    dptr = diag->data_ptr();
  }
  auto u = torch::zeros_like(h);
  auto scratch = torch::empty({lfmq_chol_scratch(n)}, h.options());
  auto info = torch::empty({1}, h.options().dtype(torch::kInt32));
  CHECK_HIP(lfmq_chol_inverse(h.data_ptr(), dptr, u.data_ptr(),
                              scratch.data_ptr(), info.data_ptr(), n, stream()));
  return {u, info};
}

// w, a copy without columns that have no inputs (zeros on h's diagonal), and [3, k]:
// h's diagonal with ones there, the same damped, whether a column has inputs
std::vector<torch::Tensor> gptq_prepare(torch::Tensor w, torch::Tensor h,
                                        double percent) {
  check_t(w, torch::kFloat32, "w");
  check_t(h, torch::kFloat32, "h");
  TORCH_CHECK(w.dim() == 2 && h.dim() == 2 && w.size(1) > 0 &&
                  h.size(0) == w.size(1) && h.size(1) == w.size(1) &&
                  h.device() == w.device(),
              "w [n, k], h [k, k] on one device");
  auto to = torch::empty_like(w);
  auto d = torch::empty({3, w.size(1)}, w.options());
  CHECK_HIP(lfmq_gptq_prepare(w.data_ptr(), h.data_ptr(), to.data_ptr(),
                              d.data_ptr(), (int)w.size(0), (int)w.size(1),
                              (float)percent, stream()));
  return {to, d};
}

// one column block of the GPTQ solve; returns its errors [n, nb]
torch::Tensor gptq_block(torch::Tensor w, torch::Tensor ub,
                         torch::Tensor codes, torch::Tensor scales,
                         torch::Tensor zeros, long i1, long g, long bits,
                         bool sym) {
  check_t(w, torch::kFloat32, "w");
  TORCH_CHECK(ub.is_cuda() && ub.scalar_type() == torch::kFloat32 &&
                  ub.dim() == 2 && ub.stride(1) == 1 &&
                  ub.stride(0) >= ub.size(1) && ub.stride(0) <= INT32_MAX,
              "ub must be rows of fp32 on GPU");
  check_t(codes, torch::kInt32, "codes");
  check_t(scales, torch::kFloat32, "scales");
  check_t(zeros, torch::kInt32, "zeros");
  TORCH_CHECK(w.dim() == 2 && ub.dim() == 2 && ub.size(0) == ub.size(1),
              "w [n, k], ub [nb, nb]");
  const long n = w.size(0), k = w.size(1), nb = ub.size(0);
  TORCH_CHECK(codes.sizes() == w.sizes(), "codes must be [n, k]");
  TORCH_CHECK(g > 0 && k % g == 0 && scales.numel() == n * (k / g) &&
                  zeros.numel() == n * (k / g),
              "scales and zeros must be [n, k / g]");
  auto err = torch::empty({n, nb}, w.options());
  CHECK_HIP(lfmq_gptq_block(w.data_ptr(), ub.data_ptr(),
                            (int)ub.stride(0), codes.data_ptr(),
                            scales.data_ptr(), zeros.data_ptr(),
                            err.data_ptr(), (int)n, (int)k, (int)(k / g),
                            (int)i1, (int)nb, (int)g, (int)bits, sym,
                            stream()));
  return err;
}

// w[:, i1 + nb:] -= err U[i1:i1 + nb, i1 + nb:]
void gptq_push(torch::Tensor w, torch::Tensor err, torch::Tensor u, long i1) {
  check_t(w, torch::kFloat32, "w");
  check_t(err, torch::kFloat32, "err");
  TORCH_CHECK(w.dim() == 2 && err.dim() == 2 && err.size(0) == w.size(0),
              "w [n, k], err [n, nb]");
  const long n = w.size(0), k = w.size(1), nb = err.size(1);
  TORCH_CHECK(u.is_cuda() && u.scalar_type() == torch::kFloat32 &&
                  u.dim() == 2 && u.size(0) == k && u.size(1) == k &&
                  u.stride(1) == 1 && u.stride(0) >= k,
              "u must be [k, k], rows of fp32 on GPU");
  TORCH_CHECK(i1 >= 0 && i1 + nb <= k, "block past the last column");
  CHECK_HIP(lfmq_gptq_push(w.data_ptr(), err.data_ptr(),
                           u.data_ptr<float>() + i1 * u.stride(0), u.stride(0),
                           (int)n, (int)k, (int)(i1 + nb), (int)nb, stream()));
}

// All columns of a solve, `block` at a time: w, which changes, with the factor u
// to codes, scales and zeros
void gptq_columns(torch::Tensor w, torch::Tensor u, torch::Tensor codes,
                  torch::Tensor scales, torch::Tensor zeros, long block, long g,
                  long bits, bool sym) {
  check_t(w, torch::kFloat32, "w");
  check_t(u, torch::kFloat32, "u");
  check_t(codes, torch::kInt32, "codes");
  check_t(scales, torch::kFloat32, "scales");
  check_t(zeros, torch::kInt32, "zeros");
  TORCH_CHECK(w.dim() == 2 && codes.sizes() == w.sizes(),
              "w and codes must be [n, k]");
  const long n = w.size(0), k = w.size(1);
  TORCH_CHECK(u.dim() == 2 && u.size(0) == k && u.size(1) == k,
              "u must be [k, k]");
  TORCH_CHECK(g > 0 && k % g == 0 && scales.numel() == n * (k / g) &&
                  zeros.numel() == n * (k / g),
              "scales and zeros must be [n, k / g]");
  TORCH_CHECK(block > 0, "a block has columns");
  const bool steps = block == 128 && lfmq_gptq_step_ok(u.data_ptr(), k, (int)n,
                                                       (int)k, (int)g);
  torch::Tensor before, other;             // errors of the last two blocks
  for (long i1 = 0; i1 < k; i1 += block) {
    const long nb = std::min(block, k - i1);
    if (i1 > 0 && steps && nb == block) {
      if (!other.defined()) other = torch::empty_like(before);
      CHECK_HIP(lfmq_gptq_step(w.data_ptr(), u.data_ptr(), k, codes.data_ptr(),
                               scales.data_ptr(), zeros.data_ptr(),
                               before.data_ptr(), other.data_ptr(), (int)n,
                               (int)k, (int)(k / g), (int)i1, (int)g, (int)bits,
                               sym, stream()));
      std::swap(before, other);
      continue;
    }
    if (i1 > 0) gptq_push(w, before, u, i1 - block);
    before = gptq_block(w, u.narrow(0, i1, nb).narrow(1, i1, nb), codes, scales,
                        zeros, i1, g, bits, sym);
  }
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("pack", &pack, "pack int codes");
  m.def("unpack", &unpack, "unpack int codes");
  m.def("dq_linear", &dq_linear, "fused dequant GEMV/GEMM");
  m.def("dq_linear_parts", &dq_linear_parts, "dq_linear with k in parts, or None");
  m.def("row_scale", &row_scale, "1 / root mean square of rows");
  m.def("dq_linear_scaled", &dq_linear_scaled,
        "dq_linear of rows times factors, and the result's own",
        pybind11::arg("x"), pybind11::arg("scale"), pybind11::arg("qweight"),
        pybind11::arg("scales"), pybind11::arg("qzeros"), pybind11::arg("bits"),
        pybind11::arg("g"), pybind11::arg("bias"), pybind11::arg("resid"),
        pybind11::arg("eps"), pybind11::arg("apart") = true);
  m.def("prompt_layer", &prompt_layer, "a layer's kernels for a prompt");
  m.def("dq_linear_norm", &dq_linear_norm,
        "dq_linear, the residual and the next norm");
  m.def("dq_gateup_scaled", &dq_gateup_scaled,
        "dq_gemv_gateup of rows times factors");
  m.def("rmsnorm", &rmsnorm, "fused rmsnorm");
  m.def("rmsnorm_residual", &rmsnorm_residual, "fused rmsnorm + residual");
  m.def("rope", &rope, "fused rope (in-place)");
  m.def("silu_mul", &silu_mul, "silu(gate) * up");
  m.def("silu_mul_fused", &silu_mul_fused, "silu-mul on fused gate_up");
  m.def("residual_add", &residual_add, "bf16 add");
  m.def("kv_append", &kv_append, "KV cache append");
  m.def("attn_decode", &attn_decode, "GQA decode attention");
  m.def("attn_prefill", &attn_prefill,
        "flash prefill attention (LFMQ_FLASH_PREFILL)");
  m.def("hessian_accum", &hessian_accum, "H += 2 X^T X");
  m.def("gptq_prepare", &gptq_prepare, "weights and diagonal of a GPTQ solve");
  m.def("chol_inverse", &chol_inverse,
        "upper Cholesky factor of the inverse, and whether there is none",
        pybind11::arg("h"), pybind11::arg("diag") = pybind11::none());
  m.def("gptq_push", &gptq_push, "a GPTQ block's errors to later columns");
  m.def("gptq_columns", &gptq_columns, "all column blocks of the GPTQ solve");
  m.def("gptq_block", &gptq_block, "one column block of the GPTQ solve");
  m.def("dq_gemv_gateup", &dq_gemv_gateup, "fused gate_up GEMV + silu*mul");
  m.def("qkv_rope_append", &qkv_rope_append, "fused rope + KV append");
  m.def("greedy_sample", &greedy_sample, "row argmax");
  m.def("read_probe", &read_probe, "bw probe");
  m.def("advance_record", &advance_record, "graph decode-state advance");
  m.def("attn_decode_fused", &attn_decode_fused,
        "fused rope+KV-append+attention decode");
  m.def("grouped_dq_gateup", &grouped_dq_gateup, "MoE grouped gate_up+silu");
  m.def("grouped_dq_linear", &grouped_dq_linear, "MoE grouped linear");
  m.def("grouped_dq_linear_scatter", &grouped_dq_linear_scatter,
        "MoE grouped linear, weighted rows added to their tokens'");
  m.def("moe_route", &moe_route, "one-kernel MoE top-k routing");
  m.def("moe_tile", &moe_tile, "rows a tile of the grouped products");
  m.def("moe_plan", &moe_plan, "MoE routing with tiles");
  m.def("moe_linear", &moe_linear, "MoE grouped product over tiles");
  m.def("moe_sum", &moe_sum, "MoE weighted sum of a token's rows");
  m.def("engine_step", &engine_step, "persistent decode engine step");
}
