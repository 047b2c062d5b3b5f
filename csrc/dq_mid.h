// Packed product for some tens to hundreds of rows (dq_mid.hip).
#pragma once
#include "dq_frag.h"

struct DqMidPlan {
  int mb, step, cols, splits;    // row tiles and their rows; waves side by side;
                                 // parts of k.  mb 0: none fits
  int wgs, steps;                // workgroups, their steps
};

// groups of 64's multiples that divide k, y's rows in fours
DqMidPlan lfmq_dq_mid_plan(int m, int n, int k, int g, int bits, bool glu);

// whether that is the faster way
bool lfmq_dq_mid_gains(const DqMidPlan& P, long m, long n, long k, long g, int bits,
                       bool glu);

// a matrix below 4 GiB that starts on 16 bytes; splits > 1 (not with glu): A.part
// gets [splits, m, n] fp32, and nothing else is done; else rows of x times
// A.row_scale, bias and residual, or y [m, n / 2] = silu(gate) up
hipError_t lfmq_dq_mid(const DqArgs& A, const DqMidPlan& P, int bits, bool glu,
                       hipStream_t stream);
