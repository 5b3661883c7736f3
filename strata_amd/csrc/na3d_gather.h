// NA3D in fp32 arithmetic on the matrix cores (na3d_gather.hip): the forward for
// fp32 tensors, the backward for fp32 and for the bf16 shapes the LDS kernels of
// na3d_bwd.hip do not take.
#pragma once

#include "common.h"

namespace strata {

enum GatherMode { GATHER_FWD = 0, GATHER_DQ = 1, GATHER_DKV = 2 };

// A wave owns 16 "column" tokens (queries; keys in GATHER_DKV) and streams the
// "row" tokens their windows (inverse windows) reach.
struct GatherParams {
  const void *c0, *c1;  // columns: q | q, dout | k, v
  const void *s0, *s1;  // rows:    k, v | k, v | q, dout
  void *o0, *o1;        // out | dq | dk, dv
  int B, H, D;
  int L[3], org[3], ext[3], ker[3], dil[3];
  float scale;
  int64_t cs[5], ss0[5], ss1[5], os[5];  // element strides (b, z, y, x, h); c1 as c0, o1 as o0
  float* lse;         // forward: log2-sum-exp out or null; backward: the statistics read
  const float* dsum;  // backward: dO . O per query
  int lse_ext1;       // forward: y extent of the lse array
  // set by gather_plan
  int tl[3];    // log2 of the column tile's extent per axis, summing to 4
  int nt[3];    // tiles per axis (largest over the dilation residue classes)
  int nres, tiles;
};

// Sets the tile shape and counts.  False: a shape or layout these kernels do not take (the
// caller keeps its general kernel).
bool gather_plan(GatherParams& p, int mode, int elem_bytes);
int gather_split(const GatherParams& p);
// p as gather_plan left it; bf16: T = bf16 (the backward), else float.
int launch_gather(const GatherParams& p, int mode, bool is_bf16, hipStream_t st);

}  // namespace strata
