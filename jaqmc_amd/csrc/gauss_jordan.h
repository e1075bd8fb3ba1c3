// FP64 elimination with the matrix in registers: Gauss-Jordan inversion of the
// augmented matrix [A | I], shared by the determinant kernels (det.hip) and their
// adjoint (grad.hip), and the LU of small matrices (det.hip, ferminet_small.hip).
//
// Gauss-Jordan: no rows are exchanged: the pivot of column p is the unused row with the
// largest |entry| (the smallest row on ties; any unused row is taken, even a
// non-finite one), and at the end row p of A^-1 is the right half of the pivot
// row of column p.  The parity of that row permutation is perm_sign's.
#pragma once

#include "common.h"

// log|prod_p v_p| over the pivots without one log per factor: the running
// product is kept as a mantissa in [0.5, 1) and a binary exponent (both
// factors split with frexp, so it neither overflows nor underflows), and one
// log is taken at the end.  A zero factor gives -inf, a NaN or inf factor
// propagates, as the sum of logs would.  The value-only eliminations (fwd_col_steps,
// fwd_lu_steps) go on past a zero pivot, so a singular matrix gives -inf there; the
// ones that form an inverse divide by it, and give NaN.
struct LogAbsProduct {
  double m = 1.0;
  int e = 0;
  __device__ void mul(double v) {
    int ev, em;
    const double mv = frexp(fabs(v), &ev);
    m = frexp(m * mv, &em);
    e += ev + em;
  }
  __device__ double log_abs() const { return log(m) + (double)e * 0.69314718055994530942; }
};

// Sign of the permutation perm[0 .. n-1] (n <= 64), from its cycles.
__device__ inline int perm_sign(const int* perm, int n) {
  unsigned long long seen = 0ull;
  int sgn = 1;
  for (int p = 0; p < n; ++p) {
    if ((seen >> p) & 1ull) continue;
    int len = 0, c = p;
    while (len < n && c < n && !((seen >> c) & 1ull)) {
      seen |= 1ull << c;
      c = perm[c];
      ++len;
    }
    if ((len & 1) == 0) sgn = -sgn;
  }
  return sgn;
}

// ---- one workgroup of 256 threads, NP a multiple of 16 up to 64 ------------
// Thread (ti, tj) = (tid % 16, tid / 16) owns rows i = ti + 16a and columns
// j = tj + 16b of the NP x 2NP augmented matrix.  Per pivot: the owners of
// column p (16 lanes of one DPP row) have already reduced their candidates to
// (q, A[q][p]); barrier; the owners of row q and of column p publish them;
// barrier; every thread updates its elements and the owners of column p + 1
// reduce the next candidates.
// Scratch: 3 NP + 2 doubles, then NP ints, the pivot row of each column.
template <int NP>
constexpr int gj_wg_scratch() {  // in doubles
  return 3 * NP + 2 + NP / 2;
}
template <int NP>
__device__ inline int* gj_wg_perm(double* scratch) {
  return (int*)(scratch + 3 * NP + 2);
}

// Returns with scratch still being read by other threads; the pivots' product
// and signs are in logdet, sgn of thread 0, and inv_pos[a] is the pivot index of
// the thread's row ti + 16a.  The matrix is worked on in arrays of this function
// (with the caller's, referenced, the compiler leaves it in scratch memory).
template <int NP>
__device__ __forceinline__ void gj_wg(double (&aug)[NP / 16][NP / 8], int (&inv_pos)[NP / 16], double* scratch,
                                      LogAbsProduct& logdet, int& sgn) {
  constexpr int RA = NP / 16, CB = NP / 8;
  const int tid = threadIdx.x, ti = tid & 15, tj = tid >> 4;
  double* prow = scratch;             // pivot row, 2NP
  double* pcol = scratch + 2 * NP;    // pivot column, NP
  double* cval = scratch + 3 * NP;    // signed pivot value
  int* cidx = (int*)(scratch + 3 * NP + 1);
  int* perm = gj_wg_perm<NP>(scratch);
  unsigned used = 0;
  double x[RA][CB];
  int pos[RA];
#pragma unroll
  for (int a = 0; a < RA; ++a)
#pragma unroll
    for (int b = 0; b < CB; ++b) x[a][b] = aug[a][b];
  // candidates of a column held in x[.][b] by the 16 lanes of this DPP row
  auto candidates = [&](int b) __attribute__((always_inline)) {
    double v = -1.0, sv = 0.0;
    int bi = NP;
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      const double y = fabs(x[a][b]);
      if (!((used >> a) & 1u) && (bi == NP || y > v)) {  // any unused row, even a non-finite one
        v = y;
        sv = x[a][b];
        bi = ti + 16 * a;
      }
    }
    // lanes without an unused row (bi == NP) take any offered candidate, so
    // the result is a valid unused row whenever one exists
    auto pick = [&](double ov, double osv, int oi) __attribute__((always_inline)) {
      if (oi != NP && (bi == NP || ov > v || (ov == v && oi < bi))) {
        v = ov;
        sv = osv;
        bi = oi;
      }
    };
    pick(dpp_d<0xB1>(v), dpp_d<0xB1>(sv), __builtin_amdgcn_mov_dpp(bi, 0xB1, 0xF, 0xF, false));
    pick(dpp_d<0x4E>(v), dpp_d<0x4E>(sv), __builtin_amdgcn_mov_dpp(bi, 0x4E, 0xF, 0xF, false));
    pick(dpp_d<0x141>(v), dpp_d<0x141>(sv), __builtin_amdgcn_mov_dpp(bi, 0x141, 0xF, 0xF, false));
    pick(dpp_d<0x140>(v), dpp_d<0x140>(sv), __builtin_amdgcn_mov_dpp(bi, 0x140, 0xF, 0xF, false));
    if (ti == 0) {
      *cval = sv;
      *cidx = bi;
    }
  };
  if (tj == 0) candidates(0);
#pragma unroll
  for (int pb = 0; pb < RA; ++pb) {
    for (int pr = 0; pr < 16; ++pr) {
      const int p = 16 * pb + pr;
      __syncthreads();
      const int q = *cidx;
      const double piv = *cval;
      const double rp = 1.0 / piv;
      if (tid == 0) {
        logdet.mul(piv);
        if (piv < 0) sgn = -sgn;
        perm[p] = q;
      }
      if (ti == (q & 15)) {
#pragma unroll
        for (int a = 0; a < RA; ++a)
          if (a == (q >> 4)) {
#pragma unroll
            for (int b = 0; b < CB; ++b) prow[tj + 16 * b] = x[a][b];
          }
      }
      if (tj == pr) {
#pragma unroll
        for (int a = 0; a < RA; ++a) pcol[ti + 16 * a] = x[a][pb];
      }
      __syncthreads();
      double r[CB];
#pragma unroll
      for (int b = 0; b < CB; ++b) r[b] = prow[tj + 16 * b] * rp;
#pragma unroll
      for (int a = 0; a < RA; ++a) {
        const int i = ti + 16 * a;
        if (i == q) {
#pragma unroll
          for (int b = 0; b < CB; ++b) x[a][b] = r[b];
          used |= 1u << a;
          pos[a] = p;
        } else {
          const double f = pcol[i];
#pragma unroll
          for (int b = 0; b < CB; ++b) x[a][b] -= f * r[b];
        }
      }
      if (p + 1 < NP && tj == ((p + 1) & 15)) {
        if (pr == 15) {
          candidates(pb + 1 < RA ? pb + 1 : pb);  // p + 1 < NP implies pb + 1 < RA here
        } else {
          candidates(pb);
        }
      }
    }
  }
#pragma unroll
  for (int a = 0; a < RA; ++a) {
    inv_pos[a] = pos[a];
#pragma unroll
    for (int b = 0; b < CB; ++b) aug[a][b] = x[a][b];
  }
}

// ---- one wavefront, 16 x 16 ------------------------------------------------
// Lane (ti, tj) = (lane % 16, lane / 16) owns row ti, columns tj + 4b
// (b = 0..7) of the 16 x 32 augmented matrix.  The pivot is reduced with DPP
// inside the 16-lane row that holds column p; the pivot row and column are
// published through LDS.  Scratch: 48 doubles, then 16 ints (the pivot row of
// each column).
constexpr int kGjWave = 16;
constexpr int kGjWaveScratch = 48 + kGjWave / 2;  // in doubles
__device__ inline int* gj_wave_perm(double* scratch) { return (int*)(scratch + 48); }

// (value, row) with the largest value over a 16-lane DPP row, the smallest row
// on ties; row kGjWave offers nothing.
__device__ inline void gj_pick16(double& v, int& bi) {
  auto pick = [&](double ov, int oi) __attribute__((always_inline)) {
    if (oi != kGjWave && (bi == kGjWave || ov > v || (ov == v && oi < bi))) {
      v = ov;
      bi = oi;
    }
  };
  pick(dpp_d<0xB1>(v), __builtin_amdgcn_mov_dpp(bi, 0xB1, 0xF, 0xF, false));
  pick(dpp_d<0x4E>(v), __builtin_amdgcn_mov_dpp(bi, 0x4E, 0xF, 0xF, false));
  pick(dpp_d<0x141>(v), __builtin_amdgcn_mov_dpp(bi, 0x141, 0xF, 0xF, false));
  pick(dpp_d<0x140>(v), __builtin_amdgcn_mov_dpp(bi, 0x140, 0xF, 0xF, false));
}

// pos: the pivot index of the lane's row; logdet and sgn in every lane.
__device__ __forceinline__ void gj_wave16(double (&x)[8], int& pos, double* scratch, LogAbsProduct& logdet, int& sgn) {
  const int lane = threadIdx.x & 63, ti = lane & 15, tj = lane >> 4;
  bool used = false;
  double* prow = scratch;       // 32 doubles
  double* pcol = scratch + 32;  // 16 doubles
  int* perm = gj_wave_perm(scratch);
  for (int p = 0; p < kGjWave; ++p) {
    const int pb = p >> 2, pr = p & 3;
    double xp = 0.0;
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if (b == pb) xp = x[b];
    double v = used ? -1.0 : fabs(xp);
    int bi = used ? kGjWave : ti;
    gj_pick16(v, bi);
    int q = __builtin_amdgcn_readlane(bi, 16 * pr);
    if (q >= kGjWave) q = 0;  // unreachable: an unused row always remains
    const double piv = readlane_d(xp, 16 * pr + q);
    logdet.mul(piv);
    if (piv < 0) sgn = -sgn;
    if (lane == 0) perm[p] = q;
    if (ti == q) {
#pragma unroll
      for (int b = 0; b < 8; ++b) prow[tj + 4 * b] = x[b];
    }
    if (tj == pr) pcol[ti] = xp;
    wave_sync();
    const double rp = 1.0 / piv;
    const double f = ti == q ? 0.0 : pcol[ti];
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const double r = prow[tj + 4 * b] * rp;
      x[b] = ti == q ? r : x[b] - f * r;
    }
    if (ti == q) {
      used = true;
      pos = p;
    }
    wave_sync();
  }
}

// ---- LU of 16-lane rows: log|det| and sign, no inverse ---------------------
// Lane j of a DPP row holds column j of an NP x NP matrix (NP <= 16).  Step P
// broadcasts column P from lane P (a DPP move, no LDS), every lane finds the
// pivot in it (the first row of the largest |entry|), exchanges its own rows P
// and q and subtracts; the column loop is unrolled at compile time.  Call with
// P = 0; every lane of the wave takes part.
template <int P, int NP>
__device__ __forceinline__ void fwd_col_steps(double (&m)[NP], LogAbsProduct& logdet, int& neg) {
  if constexpr (P < NP) {
    double c[NP];
#pragma unroll
    for (int i = P; i < NP; ++i) c[i] = dpp_d<0x150 + P>(m[i]);  // row_newbcast:P
    double best = fabs(c[P]), pv = c[P];
    int q = P;
#pragma unroll
    for (int i = P + 1; i < NP; ++i) {  // the first of the largest
      const bool more = fabs(c[i]) > best;
      best = more ? fabs(c[i]) : best;
      pv = more ? c[i] : pv;
      q = more ? i : q;
    }
    logdet.mul(pv);
    neg ^= (pv < 0.0) != (q != P) ? 1 : 0;
    const double mp = m[P], cp = c[P];
    double r = mp;
#pragma unroll
    for (int i = P + 1; i < NP; ++i) {
      const bool sel = i == q;
      r = sel ? m[i] : r;
      m[i] = sel ? mp : m[i];
      c[i] = sel ? cp : c[i];
    }
    // A zero pivot has nothing beside it to eliminate, and the step leaves the other
    // columns as they are (0 / 0 would turn them, and the identity that pads the
    // matrix, into NaN); a non-finite r stays in the result as NaN.
    r = pv == 0.0 ? r * 0.0 : r / pv;
#pragma unroll
    for (int i = P + 1; i < NP; ++i) m[i] = fma(-c[i], r, m[i]);
    fwd_col_steps<P + 1, NP>(m, logdet, neg);
  }
}
