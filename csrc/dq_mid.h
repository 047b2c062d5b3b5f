// Packed 8-bit product for some tens of rows (dq_mid.hip).
#pragma once
#include "dq_frag.h"

struct DqMidPlan {
  int mb, step, cols, splits;    // row tiles and their rows; waves side by side;
                                 // parts of k.  mb 0: none fits
};

// groups of 64's multiples that divide k, y's rows in fours
DqMidPlan lfmq_dq_mid_plan(int m, int n, int k, int g, bool glu);

// a matrix below 4 GiB that starts on 16 bytes; splits > 1 (not with glu): A.part
// gets [splits, m, n] fp32, and nothing else is done; else rows of x times
// A.row_scale, bias and residual, or y [m, n / 2] = silu(gate) up
hipError_t lfmq_dq_mid(const DqArgs& A, const DqMidPlan& P, bool glu,
                       hipStream_t stream);
