// Reverse pass of FermiNet log|psi| with respect to the parameters, seeded per
// walker:  g = sum_w c_w grad_theta log|psi(x_w)|  (the vector-Jacobian product
// jax.value_and_grad forms per walker in LossAndGrad.evaluate_single_walker,
// estimator/loss_grad.py:70-103, already contracted with the walker weights of
// LossAndGrad.finalize_stats, :115-128).
//
// Derivatives restated from the forward definitions:
//   log|psi| = log|sum_k det A_k|:  d/dA_k = w_k A_k^-T,
//            w_k = s_k e^{l_k - m} / sum_j s_j e^{l_j - m}   (output/logdet.py:55-79)
//   A_k = Phi_k * env_k  (elementwise; app/molecule/wavefunction/ferminet.py:93-95)
//   env[k,i,o] = sum_I pi[o,I,k] exp(-a r_iI), a = |sigma| or sigma  (output/envelope.py:124-140)
//   Phi = h_L W_orb per spin channel                               (output/orbital.py:60-78)
//   h_{l+1} = tanh(X_l W_m + g_l W_g + b) (+ h_l, / sqrt 2)        (backbone/ferminet.py:51-63)
//   h2_{l+1} = tanh(h2_l W_2 + b_2) (+ h2_l, / sqrt 2)
//   g_l = spin means of h_l;  X_l = [h_l | means over the first index of h2_l]
// The kernels here are the pieces that are not plain GEMMs: the FP64
// determinant adjoint, the envelope parameter sums, the tanh/residual
// adjoint, the walker sums and the mean adjoints, and the weight-gradient
// contraction X^T dY over walker rows (FP32 MFMA, deterministic slices).

#include "gauss_jordan.h"
#include "grad.h"

namespace {

// w_k of determinant k of a walker (stride-3 determinant records), formed
// by one wavefront; uniform result.
__device__ inline double det_weight(const double* __restrict__ dw, int K, int k) {
  const int lane = threadIdx.x & 63;
  double m = -INFINITY;
  for (int j = lane; j < K; j += 64) m = fmax(m, dw[j * 3]);
  m = wave_max_d(m);
  double S = 0.0;
  for (int j = lane; j < K; j += 64) S += dw[j * 3 + 1] * exp(dw[j * 3] - m);
  S = wave_sum_d(S);
  return dw[k * 3 + 1] * exp(dw[k * 3] - m) / S;
}

// dA_k = c_w w_k A_k^-T for one (walker, det), by FP64 Gauss-Jordan in
// registers (gauss_jordan.h): one workgroup each for 16 < N <= 64, one
// wavefront for N <= 16.  Writes
//   dPhi[unit(w,i)][k N + o] = dA[i][o] env[i][o]
//   denv[w][i][k N + o]      = dA[i][o] Phi[i][o]
// A walker with c_w = 0 writes zeros without touching its matrices (a zero
// weight stays exact even for a singular walker).  Bound by the latency of the
// pivot steps (two barriers each; wavefronts have none): 4096 matrices of 42 in
// 270 us (1184 with the matrix in LDS and a barrier tree for each pivot), 16384
// of 14 in 73 us (800).  A workgroup inverts a matrix of up to 16 in the same
// steps as one wavefront, at four times the waves: hence the line at 16.
struct DetVjp {
  FermiDims d;
  const float* Phi;
  long ldphi;
  const float* env;
  const double* det;
  const double* cot;
  int b0;
  float* dPhi;
  long lddphi;
  float* denv;
};
// thread t of nt writes its share of (walker w, det k); Inv row o, column i at Inv[o * is + i]
__device__ inline void det_vjp_out(const DetVjp& a, int w, int k, double scale, const double* Inv, int is, int t,
                                   int nt) {
  const int N = a.d.N, KN = a.d.K * N;
  for (int e = t; e < N * N; e += nt) {
    const int i = e / N, o = e % N;
    const long u = unit_idx(a.d, w, i), ie = ((long)w * N + i) * KN + k * N + o;
    float gp = 0.f, ge = 0.f;
    if (Inv) {
      const double da = scale * Inv[o * is + i];
      gp = (float)(da * a.env[ie * env_stride(a.d)]);
      ge = (float)(da * a.Phi[u * a.ldphi + k * N + o]);
    }
    a.dPhi[u * a.lddphi + k * N + o] = gp;
    a.denv[ie] = ge;
  }
}

template <int NP>
__global__ __launch_bounds__(256) void det_vjp_wg_kernel(DetVjp a) {
  constexpr int IS = NP + 1;  // odd row stride: transposed reads hit distinct banks
  __shared__ double M[NP * IS];
  __shared__ double wk_s;
  static_assert(NP * IS >= gj_wg_scratch<NP>(), "the scratch takes the matrix's place");
  const int w = blockIdx.x / a.d.K, k = blockIdx.x % a.d.K, N = a.d.N, tid = threadIdx.x;
  const double c = a.cot[a.b0 + w];
  if (c == 0.0) {
    det_vjp_out(a, w, k, 0.0, nullptr, 0, tid, 256);
    return;
  }
  if (tid < 64) {
    const double wk = det_weight(a.det + (long)w * a.d.K * 3, a.d.K, k);
    if (tid == 0) wk_s = wk;
  }
  for (int e = tid; e < NP * NP; e += 256) {
    const int i = e / NP, o = e % NP;
    double v = i == o ? 1.0 : 0.0;
    if (i < N && o < N)
      v = (double)a.Phi[(long)unit_idx(a.d, w, i) * a.ldphi + k * N + o] *
          (double)a.env[(((long)w * N + i) * a.d.K * N + k * N + o) * env_stride(a.d)];
    M[i * IS + o] = v;
  }
  __syncthreads();
  constexpr int RA = NP / 16, CB = NP / 8;
  const int ti = tid & 15, tj = tid >> 4;
  double x[RA][CB];
#pragma unroll
  for (int r = 0; r < RA; ++r)
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const int i = ti + 16 * r, j = tj + 16 * b;
      x[r][b] = j < NP ? M[i * IS + j] : (i == j - NP ? 1.0 : 0.0);
    }
  __syncthreads();  // M is scratch from here on
  int pos[RA];
  LogAbsProduct logdet;
  int sgn = 1;
  gj_wg<NP>(x, pos, M, logdet, sgn);
  __syncthreads();  // the scratch is read; M takes the inverse
#pragma unroll
  for (int r = 0; r < RA; ++r)
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const int j = tj + 16 * b;
      if (j >= NP) M[pos[r] * IS + (j - NP)] = x[r][b];
    }
  __syncthreads();
  det_vjp_out(a, w, k, c * wk_s, M, IS, tid, 256);
}

__global__ __launch_bounds__(256) void det_vjp_wave_kernel(DetVjp a) {
  constexpr int NP = kGjWave, IS = NP + 1;
  __shared__ double Ms[4][NP * IS];
  __shared__ double scratch[4][kGjWaveScratch];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, N = a.d.N, K = a.d.K;
  const int kb = (K + 3) / 4, w = blockIdx.x / kb, k = 4 * (blockIdx.x % kb) + wave;
  if (k >= K) return;  // the whole wave; no workgroup barriers below
  const double c = a.cot[a.b0 + w];
  if (c == 0.0) {
    det_vjp_out(a, w, k, 0.0, nullptr, 0, lane, 64);
    return;
  }
  const double wk = det_weight(a.det + (long)w * K * 3, K, k);
  double* M = Ms[wave];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int e = lane + 64 * t, i = e >> 4, o = e & 15;
    double v = i == o ? 1.0 : 0.0;
    if (i < N && o < N)
      v = (double)a.Phi[(long)unit_idx(a.d, w, i) * a.ldphi + k * N + o] *
          (double)a.env[(((long)w * N + i) * K * N + k * N + o) * env_stride(a.d)];
    M[i * IS + o] = v;
  }
  wave_sync();
  const int ti = lane & 15, tj = lane >> 4;
  double x[8];
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const int j = tj + 4 * b;
    x[b] = j < NP ? M[ti * IS + j] : (ti == j - NP ? 1.0 : 0.0);
  }
  int pos = 0;
  LogAbsProduct logdet;
  int sgn = 1;
  gj_wave16(x, pos, scratch[wave], logdet, sgn);
#pragma unroll
  for (int b = 4; b < 8; ++b) M[pos * IS + tj + 4 * b - NP] = x[b];
  wave_sync();
  det_vjp_out(a, w, k, c * wk, M, IS, lane, 64);
}

// Envelope parameter gradients:
//   d pi[o,I,k]    += sum_{w, i in set} denv[w][i][k N + o] e_iI
//   d sigma[o,I,k] += sum denv pi e_iI (-r_iI) (sign(sigma) for abs_isotropic)
// accumulated in FP64 into acc (pack layout (N, M, K) per set: pi then sigma,
// at off0 / off1).  The device keeps pi, sigma as [I][k][o].
// A workgroup owns 64 consecutive (k, o) of one set, one per lane, so that a
// row of denv is read coalesced, EG_I nuclei, for which the row is used, and a
// slice of the (walker, electron) rows, which its waves take in turn, EG_R rows
// in flight.  Its FP64 sums go to the workspace, P[slice][set][pi | sigma][I][k
// N + o], and env_sum_kernel adds the slices in order.  Bound by latency and the
// exponentials (42 electrons, 12 nuclei, 16 determinants, 256 walkers: 408 ->
// 85 us; 14, 2, 16, 1024: 60 -> 18 us): a wavefront per parameter gathered denv
// at a row stride and read it once per nucleus.
constexpr int EG_WAVES = 4, EG_I = 4, EG_R = 4;
struct EnvGrad {
  FermiDims d;
  const float *elec, *atoms;
  const float *pi[2], *sg[2];
  int kind, nsets;
  const float* denv;
};
__global__ __launch_bounds__(64 * EG_WAVES) void env_grad_kernel(EnvGrad a, int slices, double* __restrict__ P) {
  __shared__ double red[EG_WAVES][64];
  const FermiDims& d = a.d;
  const int N = d.N, M = d.M, KN = d.K * N;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ko = blockIdx.x * 64 + lane, I0 = blockIdx.y * EG_I, set = blockIdx.z % a.nsets, sl = blockIdx.z / a.nsets;
  const bool in = ko < KN;
  float pi[EG_I], sa[EG_I], sgn[EG_I];
  double gp[EG_I], gs[EG_I];
  // distances are the same for all lanes: lane EG_I u + q forms that of row u
  // to nucleus q
  const int lu = lane / EG_I % EG_R, lI = I0 + lane % EG_I < M ? I0 + lane % EG_I : M - 1;
  const float Rx = a.atoms[3 * lI], Ry = a.atoms[3 * lI + 1], Rz = a.atoms[3 * lI + 2];
#pragma unroll
  for (int q = 0; q < EG_I; ++q) {
    const int I = I0 + q < M ? I0 + q : M - 1;
    const long qd = (long)I * KN + (in ? ko : 0);  // device layout [I][k][o]
    pi[q] = a.pi[set][qd];
    const float sg = a.sg[set][qd];
    sa[q] = a.kind == 1 ? fabsf(sg) : sg;
    sgn[q] = a.kind == 1 ? (sg > 0.f ? 1.f : (sg < 0.f ? -1.f : 0.f)) : 1.f;
    gp[q] = gs[q] = 0.0;
  }
  int i0 = 0, i1 = N;
  if (a.nsets == 2) {
    i0 = set == 0 ? 0 : d.n_up;
    i1 = set == 0 ? d.n_up : N;
  }
  const int ni = i1 - i0, rows = d.Bc * ni;
  for (int r0 = sl * EG_WAVES + wave; r0 < rows; r0 += EG_R * EG_WAVES * slices) {
    auto walker_row = [&](int u) __attribute__((always_inline)) {
      const int r = r0 + u * EG_WAVES * slices, rc = r < rows ? r : r0;
      return (long)(rc / ni) * N + i0 + rc % ni;
    };
    float de[EG_R];
#pragma unroll
    for (int u = 0; u < EG_R; ++u)
      de[u] = in && r0 + u * EG_WAVES * slices < rows ? a.denv[walker_row(u) * KN + ko] : 0.f;
    const float* x = a.elec + walker_row(lu) * 3;
    const float dx = x[0] - Rx, dy = x[1] - Ry, dz = x[2] - Rz;
    const int rl = __float_as_int(sqrtf(dx * dx + dy * dy + dz * dz));
#pragma unroll
    for (int u = 0; u < EG_R; ++u)
#pragma unroll
      for (int q = 0; q < EG_I; ++q) {
        const float rr = __int_as_float(__builtin_amdgcn_readlane(rl, EG_I * u + q));
        const float e = expf(-sa[q] * rr);
        gp[q] += (double)de[u] * e;
        gs[q] += (double)de[u] * (double)(pi[q] * e * (-rr) * sgn[q]);
      }
  }
  double* Ps = P + ((long)sl * a.nsets + set) * 2 * M * KN;
#pragma unroll
  for (int q = 0; q < 2 * EG_I; ++q) {
    __syncthreads();
    red[wave][lane] = q < EG_I ? gp[q % EG_I] : gs[q % EG_I];
    __syncthreads();
    const int I = I0 + q % EG_I;
    if (wave == 0 && in && I < M) {
      double t = 0.0;
#pragma unroll
      for (int v = 0; v < EG_WAVES; ++v) t += red[v][lane];
      Ps[((long)(q < EG_I ? 0 : M) + I) * KN + ko] = t;
    }
  }
}
__global__ void env_sum_kernel(int N, int M, int K, int nsets, int slices, const double* __restrict__ P,
                               double* __restrict__ acc, long off0, long off1) {
  const int KN = K * N, per = M * KN;
  const int e = blockIdx.x * 256 + threadIdx.x;  // [set][pi | sigma][I][k N + o]
  if (e >= 2 * per * nsets) return;
  double s = 0.0;
  int z = 0;
  for (; z + 8 <= slices; z += 8) {  // eight slices in flight, added in order
    double t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = P[(long)(z + u) * 2 * per * nsets + e];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += t[u];
  }
  for (; z < slices; ++z) s += P[(long)z * 2 * per * nsets + e];
  const int set = e / (2 * per), part = e / per % 2, I = e / KN % M, k = e % KN / N, o = e % N;
  acc[(set ? off1 : off0) + (long)part * per + ((long)o * M + I) * K + k] += s;
}

// tanh and residual adjoint of h_new = tanh(z) (+ h_old) / sqrt 2:
//   t  = res ? sqrt2 h_new - h_old : h_new,   dz = dh_new s (1 - t^2)
//   dh_old = res ? dh_new / sqrt 2 : 0   (initialises the next adjoint)
// s = 1/sqrt 2 with the residual, 1 without.
__global__ void tanh_bwd_kernel(long rows, int n, const float* __restrict__ hnew, long ldn,
                                const float* __restrict__ hold, long ldo, const float* __restrict__ dhnew, long lddn,
                                int res, float* __restrict__ dz, long lddz, float* __restrict__ dhold, long lddo) {
  const long tot = rows * n;
  const float r2 = 0.70710678118654752f;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < tot; e += (long)gridDim.x * blockDim.x) {
    const long r = e / n;
    const int c = (int)(e % n);
    const float hn = hnew[r * ldn + c];
    const float g = dhnew[r * lddn + c];
    float t = hn;
    if (res) t = 1.41421356237309515f * hn - hold[r * ldo + c];
    dz[r * lddz + c] = (res ? g * r2 : g) * (1.f - t * t);
    if (dhold) dhold[r * lddo + c] = res ? g * r2 : 0.f;
  }
}

// dG[w][n] = sum over the walker's units of dz[unit][n]
__global__ void walker_sum_kernel(FermiDims d, const float* __restrict__ dz, long lddz, int n,
                                  float* __restrict__ dG, long lddg) {
  const long tot = (long)d.Bc * n;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < tot; e += (long)gridDim.x * blockDim.x) {
    const int w = (int)(e / n), c = (int)(e % n);
    float s = 0.f;
    for (int i = 0; i < d.N; ++i) s += dz[(long)unit_idx(d, w, i) * lddz + c];
    dG[(long)w * lddg + c] = s;
  }
}

// dh[unit(w,i)][f] += dX[unit(w,i)][f] + dg[w][ch(i) f1 + f] / n_ch(i)   (f < f1)
__global__ void one_adj_kernel(FermiDims d, int f1, const float* __restrict__ dX, long lddx,
                               const float* __restrict__ dg, long lddg, float* __restrict__ dh, long lddh) {
  const long tot = (long)d.Bc * d.N * f1;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < tot; e += (long)gridDim.x * blockDim.x) {
    const int f = (int)(e % f1);
    const long wi = e / f1;
    const int w = (int)(wi / d.N), i = (int)(wi % d.N);
    const int ch = (d.nch == 2 && i >= d.n_up) ? 1 : 0;
    const int nc = d.nch == 2 ? (ch ? d.n_dn : d.n_up) : d.N;
    const long u = unit_idx(d, w, i);
    dh[u * lddh + f] += dX[u * lddx + f] + dg[(long)w * lddg + ch * f1 + f] / (float)nc;
  }
}

// Adjoint of the pair stream's input of one layer, for pair (w, j, i):
//   dh2[f] = sum_n dz2[n] W2[f][n] (+ dh2_new[f] / sqrt 2 with the residual)   (dz2 set)
//          + dX[unit(w,i)][col0 + ch(j) f2 + f] / n_ch(j)
// (the layer's own pair product, then the pair means over the first index j
// within its spin channel).  A workgroup stages W2 and the dz2 rows of PD_P
// pairs in LDS; a thread owns one f and several pairs, so a weight is read once
// for PD_V of them.  Memory-bound: 200704 pairs of 32 in 36 us, where the
// product alone took 379 us with W2 gathered from global memory and the means
// another 25.
constexpr int PD_P = 64, PD_V = 8;
__global__ __launch_bounds__(256) void pair_bwd_kernel(FermiDims d, long npairs, int f2, int fout,
                                                       const float* __restrict__ dz2, const float* __restrict__ W2,
                                                       int res, const float* __restrict__ dh2new,
                                                       const float* __restrict__ dX, long lddx, int col0,
                                                       float* __restrict__ dh2) {
  extern __shared__ float sm[];
  const int tid = threadIdx.x, SW = fout + 1;
  float* Ws = sm;              // [f2][fout + 1]
  float* Zs = Ws + f2 * SW;    // [PD_P][fout]
  const long p0 = (long)blockIdx.x * PD_P;
  if (dz2) {
    for (int e = tid; e < f2 * fout; e += 256) Ws[(e / fout) * SW + e % fout] = W2[e];
    const long lim = (npairs - p0) * fout;
    for (int e = tid; e < PD_P * fout; e += 256) Zs[e] = e < lim ? dz2[p0 * fout + e] : 0.f;
    __syncthreads();
  }
  const int groups = 256 / f2 > 0 ? 256 / f2 : 1;  // pairs side by side
  const int NN = d.N * d.N;
  for (int f = f2 <= 256 ? tid % f2 : tid; f < f2; f += f2 <= 256 ? f2 : 256) {
    const int g = f2 <= 256 ? tid / f2 : 0;
    if (g >= groups) break;
    for (int pb = g; pb < PD_P; pb += groups * PD_V) {
      float s[PD_V];
#pragma unroll
      for (int v = 0; v < PD_V; ++v) s[v] = 0.f;
      if (dz2)
        for (int n = 0; n < fout; ++n) {
          const float wv = Ws[f * SW + n];
#pragma unroll
          for (int v = 0; v < PD_V; ++v) {
            const int q = pb + v * groups;
            s[v] += Zs[(q < PD_P ? q : 0) * fout + n] * wv;
          }
        }
#pragma unroll
      for (int v = 0; v < PD_V; ++v) {
        const int q = pb + v * groups;
        const long p = p0 + q;
        if (q >= PD_P || p >= npairs) continue;
        const int w = (int)(p / NN), rem = (int)(p % NN), j = rem / d.N, i = rem % d.N;
        const int ch = (d.nch == 2 && j >= d.n_up) ? 1 : 0;
        const int nc = d.nch == 2 ? (ch ? d.n_dn : d.n_up) : d.N;
        float t = s[v];
        if (dz2 && res) t += dh2new[p * fout + f] * 0.70710678118654752f;
        dh2[p * f2 + f] = t + dX[(long)unit_idx(d, w, i) * lddx + col0 + ch * f2 + f] / (float)nc;
      }
    }
  }
}

// Wider pair streams than the staged weights' LDS: one thread per entry.
__global__ void pair_bwd_wide_kernel(FermiDims d, long npairs, int f2, int fout, const float* __restrict__ dz2,
                                     const float* __restrict__ W2, int res, const float* __restrict__ dh2new,
                                     const float* __restrict__ dX, long lddx, int col0, float* __restrict__ dh2) {
  const long tot = npairs * f2;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < tot; e += (long)gridDim.x * blockDim.x) {
    const long p = e / f2;
    const int f = (int)(e % f2);
    float s = 0.f;
    for (int n = 0; n < fout; ++n) s += dz2[p * fout + n] * W2[f * fout + n];
    if (res) s += dh2new[p * fout + f] * 0.70710678118654752f;
    const int i = (int)(p % d.N), j = (int)((p / d.N) % d.N), w = (int)(p / ((long)d.N * d.N));
    const int ch = (d.nch == 2 && j >= d.n_up) ? 1 : 0;
    const int nc = d.nch == 2 ? (ch ? d.n_dn : d.n_up) : d.N;
    dh2[e] = s + dX[(long)unit_idx(d, w, i) * lddx + col0 + ch * f2 + f] / (float)nc;
  }
}

// Weight-gradient contraction over rows on FP32 MFMA (v_mfma_f32_16x16x4f32):
//   P[s][k][n] = sum_{r in slice s} X[r][k] dY[r][n]   (k < Kx, n < Ny)
//   P[s][Kx][n] = sum_{r in slice s} dY[r][n]          (BIAS)
// The A operand of a 16x16x4 step is X^T (row m = feature k, inner = row r),
// the B operand dY: lane l reads X[r0 + l/16][k0 + l%16] and dY[r0 + l/16][n0 +
// l%16], 64-byte row segments per lane group, no LDS staging.  A workgroup
// (4 waves) owns a 64 x 64 output tile of one slice; the waves take every
// fourth group of 4 rows, the next group's operands in flight while one is
// multiplied, and their partial tiles are summed through LDS.  The column sums
// are the operands of the first row of tiles, added in registers.
// One launch serves a dense layer: its kernel (Q, K and V side by side), its
// bias and, in FermiNet, both parts of its input; the slices are summed for
// many layers at once (grad.h).  MFMA-bound in the large ones: 10752 rows x 256
// x 768 in 68 us against 27 at the FP32 rate.  42 electrons, 256 walkers: 69
// launches of 21.9 us and as many slice sums of 29.7 became 36 of 29 and 6 of
// 16 us (the whole gradient 7.76 -> 5.26 ms; 14 electrons, 1024 walkers 4.08 ->
// 2.99 ms).
constexpr int WG_T = 4;  // 16x16 blocks per wave tile side

template <bool HASX>
__global__ __launch_bounds__(256) void wgrad_kernel(WgradArgs a, long rows_per_slice, float* __restrict__ P) {
  __shared__ float red[HASX ? 64 * 65 : 1];
  __shared__ float csum[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  const int k0 = blockIdx.x * 64, n0 = blockIdx.y * 64;
  const long r_beg = (long)blockIdx.z * rows_per_slice;
  const long r_end = r_beg + rows_per_slice < a.rows ? r_beg + rows_per_slice : a.rows;
  const float* const __restrict__ X = a.X;
  const float* const __restrict__ dY = a.dY;
  f32x4 acc[WG_T][WG_T];
  float cs[WG_T];
#pragma unroll
  for (int i = 0; i < WG_T; ++i) {
    cs[i] = 0.f;
#pragma unroll
    for (int j = 0; j < WG_T; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  bool kin[WG_T], nin[WG_T];
#pragma unroll
  for (int i = 0; i < WG_T; ++i) {
    kin[i] = HASX && k0 + i * 16 + lr < a.Kx;
    nin[i] = n0 + i * 16 + lr < a.Ny;
  }
  // the lane's row: number r of the contraction, row `row` of the operands
  long r = r_beg + 4 * wave + lg;
  long row = r;
  int in_group = 0;
  if (a.rgrp > 0) {
    in_group = (int)(r % a.rgrp);
    row = r / a.rgrp * a.rstride + in_group;
  }
  auto load = [&](float (&av)[WG_T], float (&bv)[WG_T]) __attribute__((always_inline)) {
    const bool rok = r < r_end;
#pragma unroll
    for (int i = 0; i < WG_T; ++i) {
      if (HASX) av[i] = rok && kin[i] ? X[row * a.ldx + k0 + i * 16 + lr] : 0.f;
      bv[i] = rok && nin[i] ? dY[row * a.ldy + n0 + i * 16 + lr] : 0.f;
    }
    r += 16;
    if (a.rgrp > 0) {
      in_group += 16;
      row += 16;
      while (in_group >= a.rgrp) {
        in_group -= a.rgrp;
        row += a.rstride - a.rgrp;
      }
    } else {
      row += 16;
    }
  };
  float av[WG_T], bv[WG_T];
  load(av, bv);
  for (long r0 = r_beg + 4 * wave; r0 < r_end; r0 += 16) {
    float an[WG_T], bn[WG_T];
    load(an, bn);
#pragma unroll
    for (int j = 0; j < WG_T; ++j) cs[j] += bv[j];
    if constexpr (HASX) {
#pragma unroll
      for (int i = 0; i < WG_T; ++i)
#pragma unroll
        for (int j = 0; j < WG_T; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bv[j], acc[i][j], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < WG_T; ++i) {
      av[i] = an[i];
      bv[i] = bn[i];
    }
  }
  const int nrow = a.Kx + (a.bias ? 1 : 0);
  float* Ps = P + (long)blockIdx.z * nrow * a.Ny;
  if (a.bias && blockIdx.x == 0) {
#pragma unroll
    for (int j = 0; j < WG_T; ++j) {
      float t = cs[j] + __shfl_xor(cs[j], 16);
      t += __shfl_xor(t, 32);
      if (lg == 0) csum[wave][j * 16 + lr] = t;
    }
    __syncthreads();
    const int n = threadIdx.x;
    if (n < 64 && n0 + n < a.Ny)
      Ps[(long)a.Kx * a.Ny + n0 + n] = (csum[0][n] + csum[1][n]) + (csum[2][n] + csum[3][n]);
  }
  if constexpr (HASX) {
    // acc[i][j][v]: output row k0 + i*16 + 4*lg + v, column n0 + j*16 + lr
    for (int src = 0; src < 4; ++src) {
      if (wave == src) {
#pragma unroll
        for (int i = 0; i < WG_T; ++i)
#pragma unroll
          for (int j = 0; j < WG_T; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              float* t = &red[(i * 16 + 4 * lg + v) * 65 + j * 16 + lr];
              *t = (src == 0 ? 0.f : *t) + acc[i][j][v];
            }
      }
      __syncthreads();
    }
    for (int e = threadIdx.x; e < 64 * 64; e += 256) {
      const int kk = e / 64, nn = e % 64;
      if (k0 + kk < a.Kx && n0 + nn < a.Ny) Ps[(long)(k0 + kk) * a.Ny + n0 + nn] = red[kk * 65 + nn];
    }
  }
}

// acc[place of (k, n)] += sum_s P[s][k][n] of every waiting contraction (FP64,
// fixed slice order), one thread per entry.
__global__ __launch_bounds__(256) void slice_sum_kernel(SliceJobs jobs, double* __restrict__ acc) {
  int q = 0;
  while (q + 1 < jobs.n && (int)blockIdx.x >= jobs.first[q + 1]) ++q;
  const SliceJob& j = jobs.j[q];
  const int tot = j.nrow * j.Ny;
  const int e = ((int)blockIdx.x - jobs.first[q]) * 256 + threadIdx.x;
  if (e >= tot) return;
  const float* __restrict__ P = j.P + e;
  double s = 0.0;
  int z = 0;
  for (; z + 8 <= j.ns; z += 8) {  // eight slices in flight, added in order
    float t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = P[(long)(z + u) * tot];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += t[u];
  }
  for (; z < j.ns; ++z) s += P[(long)z * tot];
  const int k = e / j.Ny, n = e % j.Ny;
  const long col = (long)(n / j.seg) * j.segstride + n % j.seg;
  acc[k == j.Kx ? j.boff + col : j.off + (long)(k < j.ksplit ? k : k + j.kskip) * j.ld + col] += s;
}

__global__ void fill_f64_kernel(double* p, long n, double v) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) p[e] = v;
}
__global__ void fill_f32_kernel(float* p, long n, float v) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) p[e] = v;
}
__global__ void f64_to_f32_kernel(const double* a, long n, float* out) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x)
    out[e] = (float)a[e];
}

inline int grid_of(long total) {
  long g = (total + 255) / 256;
  if (g > 65536L * 4) g = 65536L * 4;
  return (int)(g < 1 ? 1 : g);
}

}  // namespace

int launch_det_vjp(const FermiDims& d, const float* Phi, long ldphi, const float* env, const double* det,
                   const double* cot, int b0, float* dPhi, long lddphi, float* denv, hipStream_t s) {
  const DetVjp a{d, Phi, ldphi, env, det, cot, b0, dPhi, lddphi, denv};
  if (d.N <= kGjWave)
    hipLaunchKernelGGL(det_vjp_wave_kernel, dim3(d.Bc * ((d.K + 3) / 4)), dim3(256), 0, s, a);
  else if (d.N <= 32)
    hipLaunchKernelGGL(det_vjp_wg_kernel<32>, dim3(d.Bc * d.K), dim3(256), 0, s, a);
  else if (d.N <= 48)
    hipLaunchKernelGGL(det_vjp_wg_kernel<48>, dim3(d.Bc * d.K), dim3(256), 0, s, a);
  else if (d.N <= 64)
    hipLaunchKernelGGL(det_vjp_wg_kernel<64>, dim3(d.Bc * d.K), dim3(256), 0, s, a);
  else
    return -1;
  return 0;
}

// P: workspace of cap doubles
int launch_env_grad(const FermiDims& d, const float* elec, const float* atoms, const float* const* pi,
                    const float* const* sg, int kind, int nsets, const float* denv, double* P, long cap, double* acc,
                    long off0, long off1, hipStream_t s) {
  const EnvGrad a{d, elec, atoms, {pi[0], pi[1]}, {sg[0], sg[1]}, kind, nsets, denv};
  const int bx = ceil_div((long)d.K * d.N, 64), by = ceil_div(d.M, EG_I);
  // about 1024 workgroups, but at least two turns of its rows for each wave
  const long entries = 2L * d.M * d.K * d.N * nsets, turns = ceil_div((long)d.Bc * d.N, 2 * EG_R * EG_WAVES);
  long slices = 1024 / ((long)bx * by * nsets);
  slices = slices > turns ? turns : slices;
  while (slices > 1 && slices * entries > cap) slices >>= 1;
  slices = slices < 1 ? 1 : slices;
  if (entries > cap) return -1;
  hipLaunchKernelGGL(env_grad_kernel, dim3(bx, by, (unsigned)(nsets * slices)), dim3(64 * EG_WAVES), 0, s, a,
                     (int)slices, P);
  hipLaunchKernelGGL(env_sum_kernel, dim3(ceil_div(entries, 256)), dim3(256), 0, s, d.N, d.M, d.K, nsets, (int)slices,
                     P, acc, off0, off1);
  return 0;
}

int launch_tanh_bwd(long rows, int n, const float* hnew, long ldn, const float* hold, long ldo, const float* dhnew,
                    long lddn, int res, float* dz, long lddz, float* dhold, long lddo, hipStream_t s) {
  hipLaunchKernelGGL(tanh_bwd_kernel, dim3(grid_of(rows * n)), dim3(256), 0, s, rows, n, hnew, ldn, hold, ldo, dhnew,
                     lddn, res, dz, lddz, dhold, lddo);
  return 0;
}

int launch_walker_sum(const FermiDims& d, const float* dz, long lddz, int n, float* dG, long lddg, hipStream_t s) {
  hipLaunchKernelGGL(walker_sum_kernel, dim3(grid_of((long)d.Bc * n)), dim3(256), 0, s, d, dz, lddz, n, dG, lddg);
  return 0;
}

int launch_one_adj(const FermiDims& d, int f1, const float* dX, long lddx, const float* dg, long lddg, float* dh,
                   long lddh, hipStream_t s) {
  hipLaunchKernelGGL(one_adj_kernel, dim3(grid_of((long)d.Bc * d.N * f1)), dim3(256), 0, s, d, f1, dX, lddx, dg,
                     lddg, dh, lddh);
  return 0;
}

// dz2 null: the means' part alone (fout, W2, res, dh2new unused)
int launch_pair_bwd(const FermiDims& d, int f2, int fout, const float* dz2, const float* W2, int res,
                    const float* dh2new, const float* dX, long lddx, int col0, float* dh2, hipStream_t s) {
  const long npairs = (long)d.Bc * d.N * d.N;
  if (!dz2) fout = 0;
  const size_t smem = dz2 ? ((size_t)f2 * (fout + 1) + (size_t)PD_P * fout) * 4 : 0;
  if (smem <= 64 * 1024)
    hipLaunchKernelGGL(pair_bwd_kernel, dim3(ceil_div(npairs, PD_P)), dim3(256), smem, s, d, npairs, f2, fout, dz2, W2,
                       res, dh2new, dX, lddx, col0, dh2);
  else
    hipLaunchKernelGGL(pair_bwd_wide_kernel, dim3(grid_of(npairs * f2)), dim3(256), 0, s, d, npairs, f2, fout, dz2, W2,
                       res, dh2new, dX, lddx, col0, dh2);
  return 0;
}

// Slices of a contraction: about 1024 workgroups (four per CU, what the 64 x 64
// tiles' registers allow) of at least 64 rows each.
static int wgrad_slices(const WgradArgs& a, long cap) {
  const long tiles = (long)(a.Kx > 0 ? (a.Kx + 63) / 64 : 1) * ((a.Ny + 63) / 64);
  long ns = 1024 / tiles;
  ns = ns < 1 ? 1 : (ns > 256 ? 256 : ns);
  const long by_rows = (a.rows + 63) / 64;
  if (ns > by_rows) ns = by_rows > 0 ? by_rows : 1;
  while (ns > 1 && ns * (a.Kx + 1) * a.Ny > cap) ns >>= 1;
  return (int)ns;
}

int WgradQueue::add(const WgradArgs& a) {
  if (a.rows <= 0 || a.Ny <= 0 || (a.Kx <= 0 && !a.bias)) return 0;
  const int ns = wgrad_slices(a, cap_);
  const int nrow = a.Kx + (a.bias ? 1 : 0);
  const long need = (long)ns * nrow * a.Ny;
  if (need > cap_ || (long)nrow * a.Ny > 0x7FFFFFFFL) return -1;
  bool wait = jobs_.n == kSliceJobs || used_ + need > cap_;
  for (int i = 0; i < jobs_.n; ++i) wait = wait || jobs_.j[i].off == a.off || (a.bias && jobs_.j[i].boff == a.boff);
  if (wait) flush();
  long rps = (a.rows + ns - 1) / ns;
  rps = (rps + 3) / 4 * 4;
  float* P = P_ + used_;
  const dim3 grid(a.Kx > 0 ? (a.Kx + 63) / 64 : 1, (a.Ny + 63) / 64, ns);
  if (a.Kx > 0)
    hipLaunchKernelGGL(wgrad_kernel<true>, grid, dim3(256), 0, s_, a, rps, P);
  else
    hipLaunchKernelGGL(wgrad_kernel<false>, grid, dim3(256), 0, s_, a, rps, P);
  used_ += need;
  if (jobs_.n == 0) jobs_.first[0] = 0;
  jobs_.j[jobs_.n] = SliceJob{P, ns, nrow, a.Ny, a.ld, a.ksplit, a.kskip, a.seg, a.Kx, a.off, a.boff, a.segstride};
  jobs_.first[jobs_.n + 1] = jobs_.first[jobs_.n] + ceil_div((long)nrow * a.Ny, 256);
  ++jobs_.n;
  return 0;
}

void WgradQueue::flush() {
  if (jobs_.n > 0)
    hipLaunchKernelGGL(slice_sum_kernel, dim3(jobs_.first[jobs_.n]), dim3(256), 0, s_, jobs_, acc_);
  jobs_.n = 0;
  used_ = 0;
}

int launch_fill_f64(double* p, long n, double v, hipStream_t s) {
  hipLaunchKernelGGL(fill_f64_kernel, dim3(grid_of(n)), dim3(256), 0, s, p, n, v);
  return 0;
}
int launch_fill_f32(float* p, long n, float v, hipStream_t s) {
  hipLaunchKernelGGL(fill_f32_kernel, dim3(grid_of(n)), dim3(256), 0, s, p, n, v);
  return 0;
}
int launch_f64_to_f32(const double* a, long n, float* out, hipStream_t s) {
  hipLaunchKernelGGL(f64_to_f32_kernel, dim3(grid_of(n)), dim3(256), 0, s, a, n, out);
  return 0;
}
