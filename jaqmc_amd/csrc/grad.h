// Weight-gradient contractions of the reverse pass (grad.hip) and the queue of
// their slice sums.
#pragma once

#include "kernels.h"

// dW[k][n] = sum_r X[r][k] dY[r][n] over `rows` rows (k < Kx, n < Ny), added to
// the FP64 accumulator; with `bias`, also db[n] = sum_r dY[r][n].  X null (Kx 0)
// forms the column sums only.
//   rgrp > 0: row r is row (r / rgrp) * rstride + r % rgrp of X and dY (the
//     rows of one spin channel of walker-major units).
// Where the sums go: feature k is pack row k, or k + kskip from ksplit on;
// output column n is column n % seg of the kernel n / seg, whose kernels are
// segstride entries apart (seg = Ny: one kernel).
struct WgradArgs {
  long rows;
  const float* X;
  long ldx;
  int Kx;
  const float* dY;
  long ldy;
  int Ny;
  int rgrp, rstride;
  long off;  // dW's first entry in the accumulator, rows ld entries apart
  int ld;
  bool bias;
  long boff;  // db's first entry
  int ksplit, kskip;
  int seg;
  long segstride;
};
inline WgradArgs wgrad_args(long rows, const float* X, long ldx, int Kx, const float* dY, long ldy, int Ny, long off,
                            bool bias, long boff) {
  WgradArgs a{};
  a.rows = rows;
  a.X = X;
  a.ldx = ldx;
  a.Kx = Kx;
  a.dY = dY;
  a.ldy = ldy;
  a.Ny = Ny;
  a.off = off;
  a.ld = Ny;
  a.bias = bias;
  a.boff = boff;
  a.ksplit = Kx;
  a.seg = Ny;
  return a;
}

// One contraction's slices P[s][k][n] (row Kx: the column sums) waiting to be
// added to the accumulator.
struct SliceJob {
  const float* P;
  int ns, nrow, Ny;
  int ld, ksplit, kskip, seg, Kx;
  long off, boff, segstride;
};
constexpr int kSliceJobs = 24;
struct SliceJobs {
  SliceJob j[kSliceJobs];
  int first[kSliceJobs + 1];  // first workgroup of each job
  int n;
};

// Contractions of one reverse sweep: each launches at once and leaves FP32
// slices in the workspace; their FP64 sums run together when the workspace or
// the job table is full, when a contraction adds to entries that a waiting one
// adds to, and at the end (flush).  Nothing outlives the sweep.
class WgradQueue {
 public:
  WgradQueue(float* P, long cap, double* acc, hipStream_t s) : P_(P), cap_(cap), acc_(acc), s_(s) { jobs_.n = 0; }
  int add(const WgradArgs& a);
  void flush();

 private:
  float* P_;
  long cap_, used_ = 0;
  double* acc_;
  hipStream_t s_;
  SliceJobs jobs_;
};
