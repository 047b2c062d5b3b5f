// Packed product for a few tens to a hundred rows (dq_short.hip).
#pragma once
#include "dq_frag.h"

struct DqShortPlan {
  int mb, step, splits;          // row tiles and their rows; parts of k
};

DqShortPlan lfmq_dq_short_plan(int m, int n, int k, int g, int bits, bool glu);

// groups of 64's multiples that divide k, a matrix below 4 GiB that starts on
// 16 bytes; splits > 1: A.part gets [splits, m, n] fp32, and nothing else is
// done, else glu: y [m, n / 2] = silu(gate) up without bias and residual, and
// rows of x times A.row_scale
hipError_t lfmq_dq_short(const DqArgs& A, const DqShortPlan& P, int bits,
                         bool glu, hipStream_t stream);
