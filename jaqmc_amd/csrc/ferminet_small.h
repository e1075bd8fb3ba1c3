// The value path of small FermiNets and their Metropolis moves in one kernel
// (ferminet_small.hip).
#pragma once

#include "kernels.h"

constexpr int kSmallLayers = 4;

struct SmallLayer {
  const float *Wm, *Wg, *b;  // (d1, kmain), (d1, kg) transposed; (d1)
  const float *W2, *b2;      // pair layer (f2, d2), or null in the last layer
  int f1, f2, d1, d2, kmain, kg;
  int res1, res2;
};
struct SmallNet {
  SmallLayer l[kSmallLayers];
  int L, N, n_up, n_dn, nch, M, K, korb, env_kind;
  const float* Worb[2];  // per channel: (K N, korb) transposed
  const float *pi[2], *sigma[2];
  const float* atoms;
  int G;                      // walkers per workgroup
  int max_groups, max_moves;  // workgroups up to which log|psi|, and the moves, are the faster path
  // LDS layout, in floats
  int ldx, ldg, ldG, ldh, ldo, o_X[2], o_g, o_G, o_h2[2], o_phi, o_env, o_geo, o_det, o_misc, lds_floats;
};
// Fills G, the lines and the LDS layout; false where the network does not fit the kernel.
bool small_net_plan(SmallNet& n);

// log|psi| and sign (sign may be null) of B walkers.
int launch_small_logpsi(const SmallNet& n, const float* elec, int B, float* logpsi, float* sign, hipStream_t s);
// n_steps Metropolis moves of B walkers, as launch_propose, the value path and
// launch_accept make them.  refresh: logp is first set to 2 log|psi|.
struct SmallMoves {
  float* elec;
  float* logp;
  int B, n_steps;
  float width;
  const double* width_dev;  // null: width
  const float *normals, *uniforms;  // (n_steps, B, ...), or null: Philox
  uint64_t seed, ctr;
  int32_t* n_accept;
  int refresh;
};
int launch_small_moves(const SmallNet& n, const SmallMoves& m, hipStream_t s);
