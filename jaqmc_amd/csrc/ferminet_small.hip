// The value path of a small FermiNet (FP32, up to 16 electrons, pair widths up
// to 16) with everything between the positions and log|psi| in one workgroup's
// LDS, and whole Metropolis runs of it in one launch.
//
// A move of such a network is about twenty kernels of 3-5 us whose work fits one
// CU, so launches bound it.  Walkers are independent: a workgroup takes as many
// as fill one 16-row MFMA tile (G = 16 / N), keeps their positions and
// activations in LDS, reads the weights (tens of KB) from L2 and makes all the
// moves of the call.  Each step is computed as the general path computes it, in
// the same order, on the same instructions -- the GEMM's k order and epilogue
// (gemm_impl.h), the features, means, pair layers and envelope (ferminet.hip),
// the determinants (gauss_jordan.h, det.hip), the draws and the decision
// (mcmc.hip) -- so a walker's trajectory is the same bit for bit on either.
// Bound by the latency of the steps between barriers: 19 us a move (3 electrons,
// 1024 walkers, 4 determinants, layers of 64), against 67 in the general path's
// kernels (128 before their tiles fitted such sizes).

#include <algorithm>

#include "ferminet_small.h"
#include "gauss_jordan.h"
#include "philox.h"

namespace {

constexpr int kRows = 16;
constexpr int kThreads = 256;
constexpr size_t kMaxLds = 96 * 1024;

// acc of the 16 rows x 16 columns [16 ct, 16 ct + 16) of X W^T, column tile ct of
// every fourth wave, handed to epi(row, col, value).  The k order is gemm_kernel's:
// chunks of 32 from chunk kst on, lane group g the entries 8 g .. 8 g + 7.
template <typename Epi>
__device__ inline void tile_gemm(const float* X, int ldx, const float* __restrict__ W, int K, int kst, int ncols,
                                 const Epi& epi) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lg = lane >> 4;
  const int nk = K / 32;
  for (int ct = wave; 16 * ct < ncols; ct += kThreads / 64) {
    const int col = 16 * ct + lr;
    const float* wp = W + (long)(col < ncols ? col : 0) * K + 8 * lg;
    auto kof = [&](int it) {
      const int c = it + kst;
      return (c >= nk ? c - nk : c) * 32;
    };
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 b0 = *(const f32x4*)(wp + kof(0)), b1 = *(const f32x4*)(wp + kof(0) + 4);
    for (int it = 0; it < nk; ++it) {
      const int kn = kof(it + 1 < nk ? it + 1 : it);
      const f32x4 n0 = *(const f32x4*)(wp + kn), n1 = *(const f32x4*)(wp + kn + 4);
      const float* xp = X + lr * ldx + kof(it) + 8 * lg;
      const f32x4 a0 = *(const f32x4*)xp, a1 = *(const f32x4*)(xp + 4);
#pragma unroll
      for (int kk = 0; kk < 8; ++kk)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(kk < 4 ? a0[kk & 3] : a1[kk & 3], kk < 4 ? b0[kk & 3] : b1[kk & 3],
                                                   acc, 0, 0, 0);
      b0 = n0;
      b1 = n1;
    }
    if (col < ncols)
#pragma unroll
      for (int v = 0; v < 4; ++v) epi(4 * lg + v, col, acc[v]);
  }
}

template <int NP>
__device__ inline void small_dets(const SmallNet& n, const float* phi, const float* env, double* det, int nw) {
  const int j = threadIdx.x & 15, N = n.N, KN = n.K * N, total = nw * n.K;
  for (int q0 = 0; q0 < total; q0 += kThreads / 16) {
    const int id = q0 + (threadIdx.x >> 4);
    const int idc = id < total ? id : total - 1;  // every lane takes part in the moves
    const int w = idc / n.K, k = idc % n.K;
    double m[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      m[i] = i == j ? 1.0 : 0.0;
      if (i < N && j < N)
        m[i] = (double)phi[(w * N + i) * n.ldo + k * N + j] * (double)env[(w * N + i) * KN + k * N + j];
    }
    LogAbsProduct logdet;
    int neg = 0;
    fwd_col_steps<0, NP>(m, logdet, neg);
    if (j == 0 && id < total) {
      det[2 * id] = logdet.log_abs();
      det[2 * id + 1] = neg ? -1.0 : 1.0;
    }
  }
}

// log|psi| and sign of the workgroup's nw walkers at pos[w][3 N] (LDS) into
// lp[w], sg[w] (LDS).  Starts behind a barrier; its results are behind one.
__device__ inline void small_forward(const SmallNet& n, float* sm, const float* pos, int nw, float* lp, float* sg) {
  const int tid = threadIdx.x, N = n.N, M = n.M, rows = nw * N;
  float* X = sm + n.o_X[0];
  float* Xn = sm + n.o_X[1];
  float* h2 = sm + n.o_h2[0];
  float* h2n = sm + n.o_h2[1];
  float* g = sm + n.o_g;
  float* G = sm + n.o_G;
  float* geo = sm + n.o_geo;  // r log2(e) of every row and nucleus
  // features (ae_features_kernel, ee_features_kernel)
  for (int e = tid; e < rows * M; e += kThreads) {
    const int row = e / M, I = e % M;
    const float* xi = pos + row * 3;
    const float dx = xi[0] - n.atoms[3 * I], dy = xi[1] - n.atoms[3 * I + 1], dz = xi[2] - n.atoms[3 * I + 2];
    const float r = sqrtf(dx * dx + dy * dy + dz * dz);
    float* x = X + row * n.ldx + 4 * I;
    x[0] = r;
    x[1] = dx;
    x[2] = dy;
    x[3] = dz;
    geo[e] = r * 1.4426950408889634f;
  }
  for (int p = tid; p < rows * N; p += kThreads) {
    const int b = p % N, a = p / N % N, w = p / (N * N);
    const float* xa = pos + (w * N + a) * 3;
    const float* xb = pos + (w * N + b) * 3;
    const float dv[3] = {xa[0] - xb[0], xa[1] - xb[1], xa[2] - xb[2]};
    float* o = h2 + p * n.ldh;
    o[0] = a == b ? 0.f : sqrtf(dv[0] * dv[0] + dv[1] * dv[1] + dv[2] * dv[2]);
    o[1] = dv[0];
    o[2] = dv[1];
    o[3] = dv[2];
  }
  __syncthreads();
  for (int l = 0; l < n.L; ++l) {
    const SmallLayer& y = n.l[l];
    // pair means over the first index (pair_means_fwd_kernel), zero padding
    const int nc = y.kmain - y.f1;
    for (int e = tid; e < rows * nc; e += kThreads) {
      const int row = e / nc, cc = e % nc, w = row / N, i = row % N;
      float out = 0.f;
      if (cc < n.nch * y.f2) {
        const int s = cc / y.f2, f = cc % y.f2;
        const int j0 = n.nch == 1 ? 0 : (s == 0 ? 0 : n.n_up);
        const int ns = n.nch == 1 ? N : (s == 0 ? n.n_up : n.n_dn);
        const float* p = h2 + ((w * N + j0) * N + i) * n.ldh + f;
        float acc = 0.f;
        for (int j = 0; j < ns; ++j) acc += p[j * N * n.ldh];
        out = acc / ns;
      }
      X[row * n.ldx + y.f1 + cc] = out;
    }
    // spin means (spin_means4_kernel), zero padding
    for (int e = tid; e < nw * y.kg; e += kThreads) {
      const int w = e / y.kg, c = e % y.kg;
      float acc = 0.f;
      if (c < n.nch * y.f1) {
        const int s = c / y.f1, f = c % y.f1;
        const int i0 = n.nch == 1 ? 0 : (s == 0 ? 0 : n.n_up);
        const int ns = n.nch == 1 ? N : (s == 0 ? n.n_up : n.n_dn);
        const float inv = 1.f / ns;
        for (int k = 0; k < ns; ++k) acc += X[(w * N + i0 + k) * n.ldx + f];
        acc *= inv;
      }
      g[w * n.ldg + c] = acc;
    }
    __syncthreads();
    tile_gemm(g, n.ldg, y.Wg, y.kg, 0, y.d1, [&](int row, int col, float v) { G[row * n.ldG + col] = v; });
    // pair layer (pair_layer_kernel adds the bias first, the generic one last)
    if (y.W2) {
      const bool bias_first = (y.f2 == 4 || y.f2 == 16) && y.d2 == 16;
      for (int e = tid; e < rows * N * y.d2; e += kThreads) {
        const int p = e / y.d2, f = e % y.d2;
        const float* x = h2 + p * n.ldh;
        float acc = bias_first ? y.b2[f] : 0.f;
        for (int k = 0; k < y.f2; ++k) acc += x[k] * y.W2[k * y.d2 + f];
        if (!bias_first) acc += y.b2[f];
        float o = tanhf(acc);
        if (y.res2) o = (o + x[f]) * 0.70710678118654752f;
        h2n[p * n.ldh + f] = o;
      }
    }
    __syncthreads();
    // one-electron layer; the residual's k order as in gemm_kernel
    const int nk = y.kmain / 32, kst = y.res1 ? ((y.d1 + 31) / 32) % nk : 0;
    tile_gemm(X, n.ldx, y.Wm, y.kmain, kst, y.d1, [&](int row, int col, float v) {
      if (row >= rows) return;
      v += G[(row / N) * n.ldG + col];
      v += y.b[col];
      v = tanhf(v);
      if (y.res1) v = (v + X[row * n.ldx + col]) * 0.70710678118654752f;
      Xn[row * n.ldx + col] = v;
    });
    __syncthreads();
    float* t = X;
    X = Xn;
    Xn = t;
    if (y.W2) {
      t = h2;
      h2 = h2n;
      h2n = t;
    }
  }
  // orbitals per spin channel, envelopes (envelope_kernel), determinants
  float* phi = sm + n.o_phi;
  float* env = sm + n.o_env;
  const int KN = n.K * N;
  for (int c = 0; c < n.nch; ++c)
    tile_gemm(X, n.ldx, n.Worb[c], n.korb, 0, KN, [&](int row, int col, float v) {
      if (row < rows && (n.nch == 1 || (row % N < n.n_up) == (c == 0))) phi[row * n.ldo + col] = v;
    });
  for (int e = tid; e < rows * KN; e += kThreads) {
    const int row = e / KN, ko = e % KN;
    float v = 0.f;
    if (n.env_kind == 2) {
      v = 1.f;
    } else {
      const int c = n.nch == 1 || row % N < n.n_up ? 0 : 1;
      for (int I = 0; I < M; ++I) {
        const float sg = n.sigma[c][(long)I * KN + ko];
        const float a = n.env_kind == 1 ? fabsf(sg) : sg;
        const float f = n.pi[c][(long)I * KN + ko] * __builtin_amdgcn_exp2f(-a * geo[row * M + I]);
        v += f;
      }
    }
    env[e] = v;
  }
  __syncthreads();
  double* det = (double*)(sm + n.o_det);
  if (N <= 4)
    small_dets<4>(n, phi, env, det, nw);
  else if (N <= 8)
    small_dets<8>(n, phi, env, det, nw);
  else if (N <= 12)
    small_dets<12>(n, phi, env, det, nw);
  else
    small_dets<16>(n, phi, env, det, nw);
  __syncthreads();
  if (tid < nw) {  // combine_kernel
    const double* dw = det + 2 * tid * n.K;
    double m = -INFINITY;
    for (int k = 0; k < n.K; ++k) m = fmax(m, dw[2 * k]);
    double S = 0.0;
    for (int k = 0; k < n.K; ++k) S += dw[2 * k + 1] * exp(dw[2 * k] - m);
    const double logpsi = log(fabs(S)) + m;
    lp[tid] = (float)logpsi;
    sg[tid] = (float)(S > 0 ? 1.0 : (S < 0 ? -1.0 : 0.0));
  }
  __syncthreads();
}

// Rows past the last walker's stay zero: they feed products that are not used.
__device__ inline void small_clear(const SmallNet& n, float* sm) {
  for (int e = threadIdx.x; e < n.lds_floats; e += kThreads) sm[e] = 0.f;
  __syncthreads();
}

__global__ __launch_bounds__(kThreads) void small_logpsi_kernel(SmallNet n, const float* __restrict__ elec, int B,
                                                                float* __restrict__ logpsi, float* __restrict__ sign) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int tid = threadIdx.x, N3 = 3 * n.N, w0 = blockIdx.x * n.G, nw = min(n.G, B - w0);
  float* pos = sm + n.o_misc;
  float* lp = pos + kRows * 3;
  small_clear(n, sm);
  for (int e = tid; e < nw * N3; e += kThreads) pos[e] = elec[(long)w0 * N3 + e];
  __syncthreads();
  small_forward(n, sm, pos, nw, lp, lp + kRows);
  if (tid < nw) {
    logpsi[w0 + tid] = lp[tid];
    if (sign) sign[w0 + tid] = lp[kRows + tid];
  }
}

__global__ __launch_bounds__(kThreads) void small_moves_kernel(SmallNet n, SmallMoves m) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int tid = threadIdx.x, N3 = 3 * n.N, w0 = blockIdx.x * n.G, nw = min(n.G, m.B - w0);
  float* pos = sm + n.o_misc;
  float* lp = pos + kRows * 3;
  float* prop = lp + 2 * kRows;
  float* logp = prop + kRows * 3;
  int* acc = (int*)(logp + kRows);
  small_clear(n, sm);
  for (int e = tid; e < nw * N3; e += kThreads) pos[e] = m.elec[(long)w0 * N3 + e];
  if (tid < nw && !m.refresh) logp[tid] = m.logp[w0 + tid];
  __syncthreads();
  const float width = m.width_dev ? (float)m.width_dev[0] : m.width;
  const int groups = (N3 + 3) / 4;
  int count = 0;
  for (int t = m.refresh ? -1 : 0; t < m.n_steps; ++t) {  // -1: log|psi| where the walkers are
    const uint64_t step = m.ctr + t;
    for (int e = tid; e < nw * groups; e += kThreads) {
      const int w = e / groups, gi = e % groups;
      float z[4] = {0.f, 0.f, 0.f, 0.f};
      if (t < 0) {
      } else if (m.normals) {
        for (int q = 0; q < 4; ++q) {
          const int c = 4 * gi + q;
          z[q] = c < N3 ? m.normals[((long)t * m.B + w0 + w) * N3 + c] : 0.f;
        }
      } else {
        philox_normals(m.seed, step, (uint32_t)(w0 + w), (uint32_t)gi, z);
      }
      for (int q = 0; q < 4; ++q) {
        const int c = 4 * gi + q;
        if (c < N3) prop[w * N3 + c] = t < 0 ? pos[w * N3 + c] : pos[w * N3 + c] + width * z[q];
      }
    }
    __syncthreads();
    small_forward(n, sm, prop, nw, lp, lp + kRows);
    if (tid < nw) {
      const float lp2 = 2.f * lp[tid];
      bool yes = false;
      if (t < 0) {
        logp[tid] = lp2;
      } else {
        const float u = m.uniforms ? m.uniforms[(long)t * m.B + w0 + tid]
                                   : philox_uniform(m.seed, step, (uint32_t)(w0 + tid));
        const float ratio = lp2 - logp[tid];
        yes = ratio > logf(u);
        if (yes) logp[tid] = lp2;
        count += yes ? 1 : 0;
      }
      acc[tid] = yes ? 1 : 0;
    }
    __syncthreads();
    for (int e = tid; e < nw * N3; e += kThreads)
      if (acc[e / N3]) pos[e] = prop[e];
    __syncthreads();
  }
  for (int e = tid; e < nw * N3; e += kThreads) m.elec[(long)w0 * N3 + e] = pos[e];
  if (tid < nw) {
    m.logp[w0 + tid] = logp[tid];
    m.n_accept[w0 + tid] += count;
  }
}

// Workgroups up to which this path is the faster one.  A CU runs a round of as many
// as its LDS holds at once, two at most in the moves (their registers); every round
// takes the same time, while the general path's launches cost `layer_us` a layer and
// once more for the features and determinants, and little more for more walkers.  One
// round is always taken, further ones while they fit that.  The time of a round is an
// estimate, within 4 % (mean) of the moves of 152 networks of 1 to 16 electrons: steps
// between barriers, a wave's 32 x 64 chunks of weights, pair products, envelope terms,
// elimination.  Where three workgroups fit a CU every launch measured, up to five per
// CU, was faster.
int faster_groups(const SmallNet& n, double layer_us) {
  constexpr int kCus = 256, kCuLds = 160 * 1024;
  const int fit = kCuLds / (n.lds_floats * 4);
  if (fit >= 3) return 5 * kCus;
  const int rows = n.G * n.N, KN = n.K * n.N, np = round_up(n.N, 4);
  long chunks = (long)n.nch * ceil_div(KN, 64) * (n.korb / 32), pair = 0;
  for (int l = 0; l < n.L; ++l) {
    const SmallLayer& y = n.l[l];
    chunks += (long)ceil_div(y.d1, 64) * ((y.kmain + y.kg) / 32);
    if (y.W2) pair += (long)ceil_div((long)rows * n.N * y.d2, kThreads) * y.f2;
  }
  const long env = (long)ceil_div((long)rows * KN, kThreads) * n.M;
  const long det = (long)ceil_div((long)n.G * n.K, kThreads / 16) * np * np;
  const double round_us = 3.2 + 4.8 * n.L + 0.31 * chunks + 0.08 * pair + 0.11 * env + 0.036 * det;
  const int rounds = std::max(1, (int)(layer_us * (1 + n.L) / round_us));
  return std::min(5, std::min(fit, 2) * rounds) * kCus;
}
// Measured, here and in the general path (us), four determinants: layers 2 x 64, three
// electrons, log|psi| of 1280 walkers 24 and 67, 6400 48 and 111; fourteen, 512 43 and
// 93, 1024 80 and 106, general from there (1280: 108 and 118).  Ten moves: 4 x 128,
// fourteen electrons, 512 walkers 1181 and 1748, general from there (640: 2103 and
// 1839); sixteen, one workgroup per CU, 256 1104 and 1625, 384 2194 and 1732.
constexpr double kLayerUs = 28.0, kMoveLayerUs = 36.0;

}  // namespace

bool small_net_plan(SmallNet& n) {
  if (n.N > kRows || n.L < 1 || n.L > kSmallLayers) return false;
  int kx = n.korb, kg = 0, d1 = 0, f2 = 4;
  for (int l = 0; l < n.L; ++l) {
    const SmallLayer& y = n.l[l];
    if (y.d1 % 32 || y.d1 > 256 || y.f1 % 4 || (y.W2 && (y.d2 > 16 || y.d2 < 1))) return false;
    kx = std::max(kx, y.kmain);
    kg = std::max(kg, y.kg);
    d1 = std::max(d1, y.d1);
    if (y.W2) f2 = std::max(f2, y.d2);
  }
  n.G = kRows / n.N;
  // row strides of 4 mod 32 floats: 16-byte aligned, 16-byte reads of 8 rows on distinct banks
  n.ldx = kx + 4;
  n.ldg = kg + 4;
  n.ldG = d1 + 4;
  n.ldh = round_up(f2, 4) + 1;  // scalar reads down the pairs
  n.ldo = n.K * n.N + 1;
  int at = 0;
  auto take = [&](long floats) {
    const int o = at;
    at += round_up((int)floats, 4);
    return o;
  };
  const long KN = (long)n.K * n.N;
  if (KN > 1024 || (long)n.M * kRows > 4096) return false;
  for (int q = 0; q < 2; ++q) n.o_X[q] = take((long)kRows * n.ldx);
  n.o_g = take((long)kRows * n.ldg);
  n.o_G = take((long)kRows * n.ldG);
  for (int q = 0; q < 2; ++q) n.o_h2[q] = take((long)n.G * n.N * n.N * n.ldh);
  n.o_phi = take((long)kRows * n.ldo);
  n.o_env = take((long)kRows * KN);
  n.o_geo = take((long)kRows * n.M);
  n.o_det = take(4L * n.G * n.K);
  n.o_misc = take(2L * kRows * 3 + 4 * kRows);  // positions, proposals; log|psi|, sign, logp, decisions
  n.lds_floats = at;
  if ((size_t)at * 4 > kMaxLds) return false;
  n.max_groups = faster_groups(n, kLayerUs);
  n.max_moves = faster_groups(n, kMoveLayerUs);
  return true;
}

template <typename K>
static int small_attr(K kernel) {
  return hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds) == hipSuccess
             ? 0
             : -1;
}

int launch_small_logpsi(const SmallNet& n, const float* elec, int B, float* logpsi, float* sign, hipStream_t s) {
  static const int attr = small_attr(small_logpsi_kernel);
  if (attr) return -1;
  hipLaunchKernelGGL(small_logpsi_kernel, dim3(ceil_div(B, n.G)), dim3(kThreads), (size_t)n.lds_floats * 4, s, n, elec,
                     B, logpsi, sign);
  return 0;
}

int launch_small_moves(const SmallNet& n, const SmallMoves& m, hipStream_t s) {
  static const int attr = small_attr(small_moves_kernel);
  if (attr) return -1;
  hipLaunchKernelGGL(small_moves_kernel, dim3(ceil_div(m.B, n.G)), dim3(kThreads), (size_t)n.lds_floats * 4, s, n, m);
  return 0;
}
