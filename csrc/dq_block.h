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

// row tile and column block of a tile: bands of 8 row tiles, row tiles fastest
__device__ __forceinline__ void dq_block_place(u32 id, int mb, u32 nb, int& mt,
                                               int& nblk) {
  const u32 band = id / (8 * nb), in = id - band * 8 * nb;
  const u32 w = min(8u, (u32)mb - band * 8);
  mt = band * 8 + in % w;
  nblk = in / w;
}

// What a workgroup computes: `rows` rows from row0 on, of x or of an expert's slots,
// by column block nblk, part sp of k's parts; to `part` where a second launch adds
// these up.
struct DqBlockTile {
  int nblk, sp = 0, parts = 1, expert = 0, row0, rows;
  float* part = nullptr;
};

// of workgroup blockIdx of a product of nb column blocks, step rows of bn columns
// a part; false: nothing
template <DqMode MODE>
__device__ __forceinline__ bool dq_block_tile(DqArgs& A, const DqBlockPlan& P, u32 nb,
                                              int bn, DqBlockTile& T) {
  int mt;
  if (MODE != DENSE && A.tiles != nullptr) {
    T.nblk = blockIdx.x % nb;
    mt = blockIdx.x / nb;
    T.expert = A.tiles[3 * mt];
    if (T.expert < 0) return false;
    T.row0 = A.tiles[3 * mt + 1];
    T.rows = A.tiles[3 * mt + 2];
    if (MODE == SLOTS) {
      T.sp = blockIdx.y;
      T.parts = P.parts;
      A.y32 += (u64)T.sp * P.part;
    }
    return true;
  }
  u32 id = blockIdx.x;
  if ((int)id < P.full) {
    id = xcd_swizzle(id, P.full);
  } else {
    T.parts = P.parts;
    T.part = A.part + (u64)(id - P.full) * (P.step * bn);
    T.sp = (id - P.full) % T.parts;
    id = P.full + (id - P.full) / T.parts;
  }
  dq_block_place(id, P.mb, nb, mt, T.nblk);
  T.row0 = mt * P.step;
  T.rows = min(A.m - T.row0, P.step);
  return true;
}

// `tile` rows of bo columns in LDS, ld apart, to rows row0 .. row0 + rows of y
__device__ __forceinline__ void dq_block_store(const unsigned short* out, int ld,
                                               int tile, int bo, unsigned short* y,
                                               int row0, int rows, int n0, int nout,
                                               int tid, int tpb) {
  const bool wide = nout % 8 == 0;
  for (int i = tid; i < tile * bo / 8; i += tpb) {
    const int row = i / (bo / 8), c = i % (bo / 8) * 8;
    const int gc = n0 + c;
    if (row >= rows || gc >= nout) continue;
    unsigned short* p = y + (u64)(row0 + row) * nout + gc;
    const unsigned short* q = out + row * ld + c;
    if (wide) {
      *(u32x4*)p = *(const u32x4*)q;
    } else {
      for (int e = 0; e < 8 && gc + e < nout; ++e) p[e] = q[e];
    }
  }
}

// groups in eights, whose scales and zeros come by 16-byte pieces
bool lfmq_dq_block_ok(const void* qweight, const void* scales, long n, long k,
                      long g, long bits);

DqBlockPlan lfmq_dq_block_plan(int m, int n, int k, int g, int bits, bool glu);

// Whether a product of `rows` rows (of all experts) gains by the sums of x's groups
// being made first, into scratch memory of 8 bytes each (dq_panel.hip); null sums,
// here and below: not.
bool lfmq_dq_panel_gains(long rows, long n, long k, long g, long bits);

// glu: y [m, n / 2] = silu(gate) up of W = [gate | up], without bias
hipError_t lfmq_dq_block(const void* qweight, const void* scales,
                         const void* qzeros, const void* x, void* y,
                         const void* bias, void* part, void* sums, int m, int n,
                         int k, int g, int bits, bool glu, const DqBlockPlan& P,
                         hipStream_t stream);

// parts of k that pay for an fp32 product of `slots` rows over E experts
int lfmq_dq_block_slot_parts(long slots, long E, int n, int k, int g, int bits);

// rows of x (or slots) by expert, tiles of up to 128 of them (DqArgs); glu:
// y bf16 [slots, n / 2], else fp32 [slots, n]; rows: of x; part: parts > 1 only, fp32
// [parts, slots, n]
hipError_t lfmq_dq_block_experts(const void* qweight, const void* scales,
                                 const void* qzeros, const void* x,
                                 const void* src, const void* tiles, void* y,
                                 void* part, void* sums, long rows, int n_tiles,
                                 int n, int k, int g, int bits, bool glu,
                                 int parts, long slots, hipStream_t stream);

// lfmq_dq_block's and lfmq_dq_block_experts' kernel after the sums of x's `rows`
// rows, for their wgs workgroups
hipError_t lfmq_dq_panel(const DqArgs& A, const DqBlockPlan& P, int bits, DqMode mode,
                         u32 wgs, void* sums, long rows, hipStream_t stream);
