// Packed product for many rows (dq_block.hip).
#pragma once
#include "dq_frag.h"

// Tiles from `full` on are split over `parts` workgroups, whose sums meet in a
// second launch.
struct DqBlockPlan {
  int mb, step;                  // row tiles and their rows
  int full, parts;
  long part;                     // floats of scratch memory
};

// groups in eights, whose scales and zeros come by 16-byte pieces
bool lfmq_dq_block_ok(const void* qweight, const void* scales, long n, long k,
                      long g, long bits);

DqBlockPlan lfmq_dq_block_plan(int m, int n, int k, int g, int bits, bool glu);

// glu: y [m, n / 2] = silu(gate) up of W = [gate | up], without bias
hipError_t lfmq_dq_block(const void* qweight, const void* scales,
                         const void* qzeros, const void* x, void* y,
                         const void* bias, void* part, int m, int n, int k,
                         int g, int bits, bool glu, const DqBlockPlan& P,
                         hipStream_t stream);

// parts of k that pay for an fp32 product of `slots` rows over E experts
int lfmq_dq_block_slot_parts(long slots, long E, int n, int k, int g, int bits);

// rows of x (or slots) by expert, tiles of up to 128 of them (DqArgs); glu:
// y bf16 [slots, n / 2], else fp32 [slots, n]; part: parts > 1 only, fp32
// [parts, slots, n]
hipError_t lfmq_dq_block_experts(const void* qweight, const void* scales,
                                 const void* qzeros, const void* x,
                                 const void* src, const void* tiles, void* y,
                                 void* part, int n_tiles, int n, int k, int g,
                                 int bits, bool glu, int parts, long slots,
                                 hipStream_t stream);
