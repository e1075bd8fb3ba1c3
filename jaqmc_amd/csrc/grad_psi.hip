// Reverse pass of the Psiformer value path with respect to the parameters:
// the pieces that are not plain GEMMs (the dense layers' adjoints and weight
// gradients run on the GEMM family and wgrad_kernel, grad.hip).  Derivatives
// restated from the forward definitions (wavefunction/backbone/psiformer.py:
// 29-98, wavefunction/jastrow.py:60-122):
//   LayerNorm  y = s xh + b,  xh = (x - mu) / sigma,  sigma = sqrt(var + eps):
//     g = dy s,  dx = (g - mean(g) - xh mean(g xh)) / sigma,
//     ds = sum_rows dy xh,  db = sum_rows dy
//   attention per (walker, head), q carrying 1/sqrt(dh):  a = softmax_j(q.k),
//   o = a v:  dv = a^T do,  da = do v^T,  ds = a (da - rowsum(a da)),
//     dq = ds k,  dk = ds^T q
//   Jastrow  -c alpha^2 / (alpha + r):  d/d alpha = -c alpha (alpha + 2 r) / (alpha + r)^2

#include "kernels.h"

namespace {

constexpr int LN_MAXV = 8;  // features per lane (D <= 512)

// One wavefront per row.  out = base + dx (base may alias out; null: out =
// dx); P = dy xh (the rows of the scale gradient).
__global__ __launch_bounds__(256) void ln_bwd_kernel(long rows, int D, const float* __restrict__ x, long ldx,
                                                     const float* __restrict__ s, const float* __restrict__ dy,
                                                     long lddy, float eps, const float* base, long ldb, float* out,
                                                     long ldo, float* __restrict__ P, long ldp) {
  const long r = blockIdx.x * 4L + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= rows) return;
  float xv[LN_MAXV], gv[LN_MAXV], dv[LN_MAXV];
  float sum = 0.f;
#pragma unroll
  for (int q = 0; q < LN_MAXV; ++q) {
    const int c = lane + 64 * q;
    xv[q] = c < D ? x[r * ldx + c] : 0.f;
    dv[q] = c < D ? dy[r * lddy + c] : 0.f;
    sum += xv[q];
  }
  const float mu = wave_sum(sum) / (float)D;
  float sq = 0.f;
#pragma unroll
  for (int q = 0; q < LN_MAXV; ++q) {
    const float t = lane + 64 * q < D ? xv[q] - mu : 0.f;
    sq += t * t;
  }
  const float rs = 1.f / sqrtf(wave_sum(sq) / (float)D + eps);
  float sg = 0.f, sgx = 0.f;
#pragma unroll
  for (int q = 0; q < LN_MAXV; ++q) {
    const int c = lane + 64 * q;
    const float xh = c < D ? (xv[q] - mu) * rs : 0.f;
    const float g = c < D ? dv[q] * s[c] : 0.f;
    xv[q] = xh;
    gv[q] = g;
    sg += g;
    sgx += g * xh;
  }
  const float mg = wave_sum(sg) / (float)D, mgx = wave_sum(sgx) / (float)D;
#pragma unroll
  for (int q = 0; q < LN_MAXV; ++q) {
    const int c = lane + 64 * q;
    if (c < D) {
      out[r * ldo + c] = (base ? base[r * ldb + c] : 0.f) + (gv[q] - mg - xv[q] * mgx) * rs;
      P[r * ldp + c] = dv[q] * xv[q];
    }
  }
}

// One workgroup per (walker, head).  Q, K, V come head-split
// ([w][part][h][i][dh], one row per electron), dO row-major with the head's
// features at columns h*dh; dq, dk, dv go to row-major [unit][part*D + h*dh + d].
// Bound by LDS reads: threads work on register blocks, 2 x 4 scores with
// 16-byte reads along d, then 4 rows x 4 features of dq, dk, dv (two thirds of
// the reads of one output per thread go); softmax and its adjoint take a
// wavefront per row.  42 electrons, 64-wide heads, 1024 walker-heads: 116 -> 87
// us at two workgroups per CU.  Rows N .. N4 of the arrays are zeros.
constexpr int AB_PAD = 4;  // row strides dh + 4, N4 + 4: 16-byte aligned, rows on shifted banks
__global__ __launch_bounds__(256) void attn_bwd_kernel(const float* __restrict__ QKV, const float* __restrict__ dO,
                                                       long lddo, float* __restrict__ dQKV, long ldq, int N, int H,
                                                       int dh) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int N4 = (N + 3) & ~3, SR = dh + AB_PAD, SN = N4 + AB_PAD;
  float* Qs = sm;
  float* Ks = Qs + N4 * SR;
  float* Vs = Ks + N4 * SR;
  float* Gs = Vs + N4 * SR;  // dO
  float* As = Gs + N4 * SR;  // scores, then a
  float* Ds = As + N4 * SN;  // da, then ds
  const int w = blockIdx.x / H, h = blockIdx.x % H, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long blk = (long)N * dh;
  const float* q = QKV + ((long)w * 3 * H + h) * blk;
  for (int e = tid; e < N4 * dh; e += 256) {
    const int i = e / dh, d = e % dh;
    const bool in = i < N;
    Qs[i * SR + d] = in ? q[e] : 0.f;
    Ks[i * SR + d] = in ? q[(long)H * blk + e] : 0.f;
    Vs[i * SR + d] = in ? q[2L * H * blk + e] : 0.f;
    Gs[i * SR + d] = in ? dO[((long)w * N + i) * lddo + h * dh + d] : 0.f;
  }
  __syncthreads();
  auto dot4 = [](float s, const float4& a, const float4& b) __attribute__((always_inline)) {
    s += a.x * b.x;
    s += a.y * b.y;
    s += a.z * b.z;
    return s + a.w * b.w;
  };
  const int nj = N4 / 4;
  for (int e = tid; e < (N4 / 2) * nj; e += 256) {
    const int i = 2 * (e / nj), j = 4 * (e % nj);
    float sa[2][4] = {}, da[2][4] = {};
    for (int d = 0; d < dh; d += 4) {
      float4 x[2], g[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        x[u] = *(const float4*)&Qs[(i + u) * SR + d];
        g[u] = *(const float4*)&Gs[(i + u) * SR + d];
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float4 k4 = *(const float4*)&Ks[(j + v) * SR + d], v4 = *(const float4*)&Vs[(j + v) * SR + d];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          sa[u][v] = dot4(sa[u][v], x[u], k4);
          da[u][v] = dot4(da[u][v], g[u], v4);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        As[(i + u) * SN + j + v] = sa[u][v];
        Ds[(i + u) * SN + j + v] = da[u][v];
      }
  }
  __syncthreads();
  for (int i = wave; i < N4; i += 4) {  // N <= 64: one column per lane
    const bool in = lane < N && i < N;
    const float s = in ? As[i * SN + lane] : -INFINITY;
    const float m = wave_max(s);
    const float e = in ? expf(s - m) : 0.f;
    const float a = i < N ? e * (1.f / wave_sum(e)) : 0.f;
    const float da = in ? Ds[i * SN + lane] : 0.f;
    const float rsum = wave_sum(a * da);
    if (lane < N4) {
      As[i * SN + lane] = a;
      Ds[i * SN + lane] = a * (da - rsum);
    }
  }
  __syncthreads();
  const int D = H * dh, nd = dh / 4;
  float* out = dQKV + (long)w * N * ldq + h * dh;
  auto fma4 = [](float4& s, float a, const float4& b) __attribute__((always_inline)) {
    s.x += a * b.x;
    s.y += a * b.y;
    s.z += a * b.z;
    s.w += a * b.w;
  };
  for (int e = tid; e < (N4 / 4) * nd; e += 256) {
    const int i = 4 * (e / nd), d = 4 * (e % nd);
    float4 gq[4] = {}, gk[4] = {}, gv[4] = {};
    for (int j = 0; j < N; ++j) {
      const float4 k4 = *(const float4*)&Ks[j * SR + d], q4 = *(const float4*)&Qs[j * SR + d],
                   g4 = *(const float4*)&Gs[j * SR + d];
      const float4 ds = *(const float4*)&Ds[j * SN + i], aj = *(const float4*)&As[j * SN + i];
      const float dsj[4] = {ds.x, ds.y, ds.z, ds.w}, ajj[4] = {aj.x, aj.y, aj.z, aj.w};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        fma4(gq[u], Ds[(i + u) * SN + j], k4);
        fma4(gk[u], dsj[u], q4);
        fma4(gv[u], ajj[u], g4);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i + u < N) {
        float* o = out + (long)(i + u) * ldq + d;
        *(float4*)o = gq[u];
        *(float4*)(o + D) = gk[u];
        *(float4*)(o + 2 * D) = gv[u];
      }
  }
}

// out[w][0..1] = c_w dJ_w / d(alpha_par, alpha_anti), one wavefront per walker
// of the chunk (walker b0 + w of the weights), its lanes taking the pairs in turn
__global__ __launch_bounds__(64) void jastrow_grad_kernel(const float* __restrict__ elec, int Bc, int N, int n_up,
                                                          float ap, float aa, const double* __restrict__ cot, int b0,
                                                          float* __restrict__ out) {
  const int w = blockIdx.x, lane = threadIdx.x;
  const float* x = elec + (long)w * N * 3;
  double gp = 0.0, ga = 0.0;
  for (int e = lane; e < N * N; e += 64) {
    const int i = e / N, j = e % N;
    if (j <= i) continue;
    const double dx = x[3 * i] - x[3 * j], dy = x[3 * i + 1] - x[3 * j + 1], dz = x[3 * i + 2] - x[3 * j + 2];
    const double r = sqrt(dx * dx + dy * dy + dz * dz);
    if ((i < n_up) == (j < n_up)) {
      const double q = ap + r;
      gp += -0.25 * ap * (ap + 2.0 * r) / (q * q);
    } else {
      const double q = aa + r;
      ga += -0.5 * aa * (aa + 2.0 * r) / (q * q);
    }
  }
  gp = wave_sum_d(gp);
  ga = wave_sum_d(ga);
  if (lane == 0) {
    const double c = cot[b0 + w];
    out[2 * w] = (float)(c * gp);
    out[2 * w + 1] = (float)(c * ga);
  }
}

// out[r][c] = a[r][c] + b[r][c]
__global__ void add_rows_kernel(long rows, int n, const float* a, long lda, const float* b, long ldb, float* out,
                                long ldo) {
  const long tot = rows * n;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < tot; e += (long)gridDim.x * blockDim.x) {
    const long r = e / n;
    const int c = (int)(e % n);
    out[r * ldo + c] = a[r * lda + c] + b[r * ldb + c];
  }
}

__global__ void scale_f64_kernel(double* p, long n, double v) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) p[e] *= v;
}

inline int grid_for(long total) {
  long g = (total + 255) / 256;
  if (g > 65536L * 4) g = 65536L * 4;
  return (int)(g < 1 ? 1 : g);
}

}  // namespace

int launch_ln_bwd(long rows, int D, const float* x, long ldx, const float* s, const float* dy, long lddy, float eps,
                  const float* base, long ldb, float* out, long ldo, float* P, long ldp, hipStream_t st) {
  if (D > 64 * LN_MAXV || rows <= 0) return rows <= 0 ? 0 : -1;
  hipLaunchKernelGGL(ln_bwd_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, st, rows, D, x, ldx, s, dy, lddy,
                     eps, base, ldb, out, ldo, P, ldp);
  return 0;
}

size_t attn_bwd_smem(int N, int dh) {
  const int N4 = round_up(N, 4);
  return (size_t)(4 * N4 * (dh + AB_PAD) + 2 * N4 * (N4 + AB_PAD)) * 4;
}

int launch_attn_bwd(const float* QKV, const float* dO, long lddo, float* dQKV, long ldq, int Bc, int N, int H, int dh,
                    hipStream_t st) {
  const size_t smem = attn_bwd_smem(N, dh);
  if (N > 64 || dh > 64 || dh % 4 || ldq % 4 || Bc <= 0) return Bc <= 0 ? 0 : -1;
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)attn_bwd_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)attn_bwd_smem(64, 64));
    attr = true;
  }
  hipLaunchKernelGGL(attn_bwd_kernel, dim3((unsigned)(Bc * H)), dim3(256), smem, st, QKV, dO, lddo, dQKV, ldq, N, H,
                     dh);
  return 0;
}

int launch_jastrow_grad(const float* elec, int Bc, int N, int n_up, float ap, float aa, const double* cot, int b0,
                        float* out, hipStream_t st) {
  if (Bc <= 0) return 0;
  hipLaunchKernelGGL(jastrow_grad_kernel, dim3((unsigned)Bc), dim3(64), 0, st, elec, Bc, N, n_up, ap, aa,
                     cot, b0, out);
  return 0;
}

int launch_add_rows(long rows, int n, const float* a, long lda, const float* b, long ldb, float* out, long ldo,
                    hipStream_t st) {
  hipLaunchKernelGGL(add_rows_kernel, dim3(grid_for(rows * n)), dim3(256), 0, st, rows, n, a, lda, b, ldb, out, ldo);
  return 0;
}

int launch_scale_f64(double* p, long n, double v, hipStream_t st) {
  hipLaunchKernelGGL(scale_f64_kernel, dim3(grid_for(n)), dim3(256), 0, st, p, n, v);
  return 0;
}
