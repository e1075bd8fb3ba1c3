// Outlier clipping of per-walker losses for the VMC gradient
// (estimator/loss_grad.py:91-128, utils/clip.py:11-60), on the device in FP64:
//   "mad":  median m = nanmedian(x), d = nanmedian(|x - m|), clip to m -+ s d
//   "iqr":  q1, q3 = nanquantile(x, .25 / .75), clip to [q1 - s iqr, q3 + s iqr]
//   "none": no clipping
// then the gradient weights  w_i = 2 (c_i - mean(c)) / n  over the n walkers
// whose clipped loss c_i is not NaN (0 for the others), so that
//   sum_i w_i grad log|psi_i| = 2 (mean(grad.c) - mean(c) mean(grad)),
// LossAndGrad.finalize_stats's gradient.
//
// Quantiles follow jnp.nanquantile's default ("linear"): position q (n - 1)
// between the order statistics floor and ceil of it, NaN entries ignored.  The
// order statistics of one quantile (or of both of "iqr") are found together by
// an MSB-first radix select over the FP64 values mapped to order-preserving
// 64-bit keys: the digits start at the highest bit in which the smallest and
// the largest key differ, each pass histograms the digit of the keys that
// match a target's prefix, and the digit holding the target's rank extends it.
//
// Two forms, by the batch alone (both exact, and deterministic: histograms are
// integer counts and every floating sum has a fixed order):
//   B <= 16384: one workgroup, the values in its registers, the histograms in
//     LDS, one launch for everything.  Bound by the barriers of its 2 x ~4
//     passes and by launch latency.  A call on 2048 values ("mad"): 421 -> 19
//     us (70 launches of two kernels per 8-bit pass and statistic ran before,
//     the digit picked by a single thread); on 16384: 555 -> 57 us.
//   larger: a histogram pass per 11-bit digit over up to 256 workgroups; the
//     last workgroup to finish a pass picks the digits (mad: two selections of a range
//     and six digit passes, 17 launches with the set-up, the means and the weights).
//     200000 values: 1906 -> 401 us, 2^20: 2819 -> 524 us.
// The line between them is the register budget of one workgroup of 1024
// threads: 16 values each (the second form takes 223 us just past it).
//
// The scratch buffer (histograms + selection state, used by the second form)
// is a caller workspace of jq_loss_clip_workspace_bytes() bytes, or, for
// jq_loss_clip_noalloc, a static device array of the same size.

#include <algorithm>
#include <mutex>
#include <string>

#include "../../include/jaqmc_amd.h"
#include "kernels.h"

int jq_fail(int code, const std::string& msg);

namespace {

typedef unsigned long long u64;

constexpr int kOneThreads = 1024;  // the one-workgroup form
constexpr int kOneMax = 16;        // values per thread at most
constexpr int kGridBlocks = 256;   // workgroups of a pass (at most)
constexpr int kGridThreads = 256;
constexpr int kDigit = 11;         // digit bits of a pass
constexpr int kBins = 1 << kDigit;
constexpr int kTargets = 4;        // order statistics found together (two quantiles x floor / ceil)

// State of the many-workgroup form, in the scratch buffer.
struct ClipState {
  u64 kmin, kmax;  // smallest and largest key of the selection
  u64 n;           // its non-NaN entries
  u64 prefix[kTargets], mask;
  long long k[kTargets];  // rank still to find below the prefix
  int shift;              // lowest bit of the prefix found so far
  unsigned ticket;        // workgroups that have finished the pass
  double q[2];            // quantile values
  double lo, hi;          // window
  double mean_x, mean_c, count;
};
constexpr size_t kStateBytes = 256;
static_assert(sizeof(ClipState) <= kStateBytes, "the state precedes the histograms");
// Scratch layout: [ClipState][kTargets x kBins counts][kGridBlocks x 3 partial sums]
constexpr size_t kScratchBytes = JQ_LOSS_CLIP_SCRATCH_BYTES;
static_assert(kStateBytes + kTargets * kBins * 4 + kGridBlocks * 3 * 8 <= kScratchBytes, "scratch size of the header");

__device__ inline u64 key_of(double v) {
  const u64 b = __builtin_bit_cast(u64, v);
  return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__device__ inline double val_of(u64 k) {
  const u64 b = (k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k;
  return __builtin_bit_cast(double, b);
}

// Targets of a selection: nt / 2 quantiles, target 2j the floor and 2j + 1 the
// ceil order statistic of quantile j.
struct Plan {
  int nt;
  double q[2];
};
__device__ inline double position(const Plan& p, int t, u64 n) { return p.q[t >> 1] * (double)((long long)n - 1); }
__device__ inline long long rank_of(const Plan& p, int t, u64 n) {
  if (n == 0) return 0;
  const double pos = position(p, t, n);
  return (long long)((t & 1) ? ceil(pos) : floor(pos));
}
// quantile from its floor / ceil order statistics, weighted as jnp.quantile's
// linear method: lo (1 - f) + hi f with f = pos - floor(pos) (at q = 0.5 this
// equals nanmedian's midpoint (lo + hi) / 2 exactly)
__device__ inline double quantile_of(double q, u64 n, double lo, double hi) {
  if (n == 0) return __builtin_nan("");
  const double pos = q * (double)((long long)n - 1);
  const double f = pos - floor(pos);
  return lo * (1.0 - f) + hi * f;
}
__device__ inline void window_of(int method, double scale, double q0, double q1, double& lo, double& hi) {
  if (method == 0) {  // mad: q0 median, q1 median absolute deviation
    lo = q0 - scale * q1;
    hi = q0 + scale * q1;
  } else if (method == 1) {  // iqr: q0 q1, q1 q3
    const double iqr = q1 - q0;
    lo = q0 - scale * iqr;
    hi = q1 + scale * iqr;
  } else {
    lo = -__builtin_inf();
    hi = __builtin_inf();
  }
}
__device__ inline double clip_to(double v, double lo, double hi) {
  return v < lo ? lo : (v > hi ? hi : v);  // NaN stays NaN (jnp.clip)
}

__device__ inline u64 shfl_xor_u64(u64 v, int o) {
  const unsigned lo = __shfl_xor((unsigned)v, o), hi = __shfl_xor((unsigned)(v >> 32), o);
  return ((u64)hi << 32) | lo;
}
__device__ inline u64 wave_min_u64(u64 v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const u64 w = shfl_xor_u64(v, o);
    v = w < v ? w : v;
  }
  return v;
}
__device__ inline u64 wave_max_u64(u64 v) { return ~wave_min_u64(~v); }

// One wavefront: the digit of nbins counts (nbins <= 32 * 64, a power of two)
// that holds rank k, and the rank below it.
__device__ inline int pick_digit(const unsigned* h, int nbins, long long& k, unsigned& count) {
  const int lane = threadIdx.x & 63;
  const int per = nbins > 64 ? nbins / 64 : 1;
  unsigned own = 0;
  for (int j = 0; j < per; ++j) own += lane * per + j < nbins ? h[lane * per + j] : 0u;
  unsigned incl = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned v = __shfl_up(incl, o);
    if (lane >= o) incl += v;
  }
  // the first lane whose running total exceeds k (the last one with a count
  // otherwise: k below the total always has one)
  const u64 over = __ballot((long long)incl > k);
  const int src = over ? __builtin_ctzll(over) : 63;
  long long kk = k - (long long)(incl - own);
  int d = lane * per;
  unsigned c = 0;
  if (lane == src) {
    for (int j = 0; j < per; ++j) {
      c = lane * per + j < nbins ? h[lane * per + j] : 0u;
      if (kk < (long long)c || j == per - 1) {
        d = lane * per + j;
        break;
      }
      kk -= c;
    }
  }
  k = (long long)((u64)(unsigned)__shfl((int)kk, src) | ((u64)(unsigned)__shfl((int)(kk >> 32), src) << 32));
  count = (unsigned)__shfl((int)c, src);
  return __shfl(d, src);
}

// ---- one workgroup --------------------------------------------------------
struct OneShared {
  unsigned h[kTargets][256];
  u64 red[3][16];
  double sum[3][16];
  u64 prefix[kTargets];
  long long k[kTargets];
  unsigned count[kTargets];
  double value[kTargets];
};

// The order statistics of p among the workgroup's values v[j], or |v[j] - center|
// where dev is set (valid: bit j set where the value counts), into S.value;
// returns their number.  The keys are formed at each use: kept, they would
// take the registers of the largest batch.
template <int V>
__device__ u64 one_select(const double (&v)[V], bool dev, double center, unsigned valid, const Plan& p, OneShared& S) {
  auto key = [&](int j) __attribute__((always_inline)) { return key_of(dev ? fabs(v[j] - center) : v[j]); };
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  u64 mn = ~0ull, mx = 0ull;
#pragma unroll
  for (int j = 0; j < V; ++j)
    if ((valid >> j) & 1u) {
      const u64 k = key(j);
      mn = k < mn ? k : mn;
      mx = k > mx ? k : mx;
    }
  mn = wave_min_u64(mn);
  mx = wave_max_u64(mx);
  int c = __builtin_popcount(valid);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if (lane == 0) {
    S.red[0][wave] = mn;
    S.red[1][wave] = mx;
    S.red[2][wave] = (u64)c;
  }
  __syncthreads();
  u64 n = 0;
  for (int i = 0; i < kOneThreads / 64; ++i) {
    const u64 a = S.red[0][i], b = S.red[1][i];
    mn = a < mn ? a : mn;
    mx = b > mx ? b : mx;
    n += S.red[2][i];
  }
  const u64 diff = n > 0 ? mn ^ mx : 0ull;
  if (diff == 0) {  // none, or all equal
    if (tid < p.nt) S.value[tid] = n > 0 ? val_of(mn) : __builtin_nan("");
    __syncthreads();
    return n;
  }
  int shift = 64 - __builtin_clzll(diff);  // bits below it are still open
  u64 mask = shift < 64 ? ~0ull << shift : 0ull;
  if (tid < p.nt) {
    S.prefix[tid] = mn & mask;
    S.k[tid] = rank_of(p, tid, n);
  }
  bool single = false;
  while (shift > 0 && !single) {
    const int low = shift > 8 ? shift - 8 : 0;
    const unsigned dm = (1u << (shift - low)) - 1u;
    S.h[tid >> 8][tid & 255] = 0;  // kTargets * 256 counts
    __syncthreads();
    // targets that share a prefix share the histogram of the first of them
    u64 pre[kTargets];
    int rep[kTargets];
    for (int t = 0; t < p.nt; ++t) {
      pre[t] = S.prefix[t];
      rep[t] = t;
      for (int u = 0; u < t; ++u)
        if (pre[u] == pre[t]) {
          rep[t] = u;
          break;
        }
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
      if (!((valid >> j) & 1u)) continue;
      const u64 k = key(j), top = k & mask;
      for (int t = 0; t < p.nt; ++t)
        if (rep[t] == t && top == pre[t]) atomicAdd(&S.h[t][(unsigned)(k >> low) & dm], 1u);
    }
    __syncthreads();
    if (wave < p.nt) {  // wave t extends target t's prefix
      long long k = S.k[wave];
      unsigned cnt;
      const int d = pick_digit(S.h[rep[wave]], 256, k, cnt);
      if (lane == 0) {
        S.k[wave] = k;
        S.count[wave] = cnt;
        S.prefix[wave] = pre[wave] | ((u64)(unsigned)d << low);
      }
    }
    shift = low;
    mask = ~0ull << shift;
    __syncthreads();
    single = true;
    for (int t = 0; t < p.nt; ++t) single = single && S.count[t] == 1;
  }
  if (shift == 0) {
    if (tid < p.nt) S.value[tid] = val_of(S.prefix[tid]);
  } else {  // one key left under each prefix: it is the order statistic
#pragma unroll
    for (int j = 0; j < V; ++j)
      if ((valid >> j) & 1u)
        for (int t = 0; t < p.nt; ++t)
          if ((key(j) & mask) == S.prefix[t]) S.value[t] = val_of(key(j));
  }
  __syncthreads();
  return n;
}

template <int V>
__global__ __launch_bounds__(kOneThreads) void clip_one_kernel(const double* __restrict__ x, int B, int method,
                                                               double scale, double* __restrict__ clipped,
                                                               double* __restrict__ w, double* __restrict__ stats) {
  __shared__ OneShared S;
  const int tid = threadIdx.x;
  double v[V];
  unsigned in = 0, valid = 0;
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int i = tid + j * kOneThreads;
    v[j] = i < B ? x[i] : 0.0;
    if (i < B) in |= 1u << j;
    if (i < B && !isnan(v[j])) valid |= 1u << j;
  }
  double q0 = 0.0, q1 = 0.0, lo, hi;
  if (method == 0) {
    const Plan p{2, {0.5, 0.5}};
    u64 n = one_select<V>(v, false, 0.0, valid, p, S);
    q0 = quantile_of(0.5, n, S.value[0], S.value[1]);
    unsigned dev = 0;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      if (((valid >> j) & 1u) && !isnan(v[j] - q0)) dev |= 1u << j;
    }
    __syncthreads();  // S.value and the reductions are read before they are reused
    n = one_select<V>(v, true, q0, dev, p, S);
    q1 = quantile_of(0.5, n, S.value[0], S.value[1]);
  } else if (method == 1) {
    const Plan p{4, {0.25, 0.75}};
    const u64 n = one_select<V>(v, false, 0.0, valid, p, S);
    q0 = quantile_of(0.25, n, S.value[0], S.value[1]);
    q1 = quantile_of(0.75, n, S.value[2], S.value[3]);
  }
  window_of(method, scale, q0, q1, lo, hi);
  // nanmeans of x and of the clipped values
  double a = 0.0, c = 0.0;
  double cnt = (double)__builtin_popcount(valid);
#pragma unroll
  for (int j = 0; j < V; ++j)
    if ((valid >> j) & 1u) {
      a += v[j];
      c += clip_to(v[j], lo, hi);
    }
  a = wave_sum_d(a);
  c = wave_sum_d(c);
  cnt = wave_sum_d(cnt);
  if ((tid & 63) == 0) {
    S.sum[0][tid >> 6] = a;
    S.sum[1][tid >> 6] = c;
    S.sum[2][tid >> 6] = cnt;
  }
  __syncthreads();
  double A = 0.0, C = 0.0, n = 0.0;
  for (int i = 0; i < kOneThreads / 64; ++i) {
    A += S.sum[0][i];
    C += S.sum[1][i];
    n += S.sum[2][i];
  }
  const double mc = C / n;
#pragma unroll
  for (int j = 0; j < V; ++j)
    if ((in >> j) & 1u) {
      const double cv = clip_to(v[j], lo, hi);
      if (clipped) clipped[tid + j * kOneThreads] = cv;
      w[tid + j * kOneThreads] = isnan(cv) ? 0.0 : 2.0 * (cv - mc) / n;
    }
  if (tid == 0 && stats) {
    stats[0] = A / n;
    stats[1] = mc;
    stats[2] = lo;
    stats[3] = hi;
    stats[4] = n;
  }
}

// ---- many workgroups ------------------------------------------------------
// Value fed to a selection: x, or |x - center| (center = a quantile result).
struct Src {
  const double* x;
  int B;
  const double* center;  // null: plain x
};
__device__ inline double src_val(const Src& s, int i) {
  const double v = s.x[i];
  return s.center ? fabs(v - *s.center) : v;
}

// True in every thread of the pass's last workgroup: all others' atomics and
// stores before it are visible to it.
__device__ inline bool last_block(ClipState* st) {
  __shared__ unsigned mine;
  __threadfence();
  __syncthreads();
  if (threadIdx.x == 0) mine = atomicAdd(&st->ticket, 1u);
  __syncthreads();
  const bool last = mine == gridDim.x - 1;
  if (last) {
    __threadfence();
    if (threadIdx.x == 0) st->ticket = 0;
  }
  return last;
}

__global__ void state_init_kernel(ClipState* st, unsigned* __restrict__ h) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kTargets * kBins) h[i] = 0;
  if (i == 0) {
    st->kmin = ~0ull;
    st->kmax = 0ull;
    st->n = 0;
    st->ticket = 0;
    st->q[0] = st->q[1] = 0.0;
  }
}

// smallest and largest key, the count, and from them the first prefix and the ranks
__global__ __launch_bounds__(kGridThreads) void range_kernel(Src s, Plan p, ClipState* st) {
  u64 mn = ~0ull, mx = 0ull;
  int c = 0;
  for (int i = blockIdx.x * kGridThreads + threadIdx.x; i < s.B; i += gridDim.x * kGridThreads) {
    const double v = src_val(s, i);
    if (isnan(v)) continue;
    const u64 k = key_of(v);
    mn = k < mn ? k : mn;
    mx = k > mx ? k : mx;
    ++c;
  }
  mn = wave_min_u64(mn);
  mx = wave_max_u64(mx);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if ((threadIdx.x & 63) == 0 && c > 0) {
    atomicMin(&st->kmin, mn);
    atomicMax(&st->kmax, mx);
    atomicAdd(&st->n, (u64)c);
  }
  if (!last_block(st) || threadIdx.x != 0) return;
  const u64 n = __hip_atomic_load(&st->n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const u64 lo = __hip_atomic_load(&st->kmin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const u64 hi = __hip_atomic_load(&st->kmax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const u64 diff = n > 0 ? lo ^ hi : 0ull;
  const int shift = diff ? 64 - __builtin_clzll(diff) : 0;  // 0: none, or all equal
  st->shift = shift;
  st->mask = shift < 64 ? ~0ull << shift : 0ull;
  for (int t = 0; t < kTargets; ++t) {
    st->prefix[t] = lo & st->mask;
    st->k[t] = t < p.nt ? rank_of(p, t, n) : 0;
  }
}

// One digit of every target.  Passes past the last digit find shift 0 and only
// leave the result: the quantiles into q[slot ...] (the last pass launched).
__global__ __launch_bounds__(kGridThreads) void digit_kernel(Src s, Plan p, ClipState* st, unsigned* __restrict__ gh,
                                                             int last_pass, int slot) {
  __shared__ unsigned h[kTargets][kBins];
  const int shift = st->shift;
  if (shift > 0) {
    const int low = shift > kDigit ? shift - kDigit : 0;
    const unsigned dm = (1u << (shift - low)) - 1u;
    const u64 mask = st->mask;
    u64 pre[kTargets];
    int rep[kTargets];
    for (int t = 0; t < p.nt; ++t) {
      pre[t] = st->prefix[t];
      rep[t] = t;
      for (int u = 0; u < t; ++u)
        if (pre[u] == pre[t]) {
          rep[t] = u;
          break;
        }
    }
    for (int i = threadIdx.x; i < p.nt * kBins; i += kGridThreads) h[i / kBins][i % kBins] = 0;
    __syncthreads();
    for (int i = blockIdx.x * kGridThreads + threadIdx.x; i < s.B; i += gridDim.x * kGridThreads) {
      const double v = src_val(s, i);
      if (isnan(v)) continue;
      const u64 k = key_of(v), top = k & mask;
      for (int t = 0; t < p.nt; ++t)
        if (rep[t] == t && top == pre[t]) atomicAdd(&h[t][(unsigned)(k >> low) & dm], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < p.nt * kBins; i += kGridThreads) {
      const unsigned c = h[i / kBins][i % kBins];
      if (c) atomicAdd(&gh[i], c);
    }
    if (!last_block(st)) return;
    for (int i = threadIdx.x; i < p.nt * kBins; i += kGridThreads) {
      h[i / kBins][i % kBins] = __hip_atomic_load(&gh[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      gh[i] = 0;  // for the next pass
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6;
    if (wave < p.nt) {
      long long k = st->k[wave];
      unsigned cnt;
      const int d = pick_digit(h[rep[wave]], kBins, k, cnt);
      if ((threadIdx.x & 63) == 0) {
        st->k[wave] = k;
        st->prefix[wave] = pre[wave] | ((u64)(unsigned)d << low);
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      st->shift = low;
      st->mask = ~0ull << low;
    }
  } else if (blockIdx.x != 0) {
    return;
  }
  if (last_pass && threadIdx.x == 0) {
    for (int j = 0; 2 * j < p.nt; ++j)
      st->q[slot + j] = quantile_of(p.q[j], st->n, val_of(st->prefix[2 * j]), val_of(st->prefix[2 * j + 1]));
    // ready for a second selection
    st->kmin = ~0ull;
    st->kmax = 0ull;
    st->n = 0;
  }
}

// clipped values, then nanmeans of x and of the clipped values
__global__ __launch_bounds__(kGridThreads) void clip_mean_kernel(const double* __restrict__ x, int B, int method,
                                                                 double scale, ClipState* st, double* part,
                                                                 double* __restrict__ clipped) {
  __shared__ double s1[kGridThreads], s2[kGridThreads], s3[kGridThreads];
  double lo, hi;
  window_of(method, scale, st->q[0], st->q[1], lo, hi);
  double a = 0.0, c = 0.0, n = 0.0;
  for (int i = blockIdx.x * kGridThreads + threadIdx.x; i < B; i += gridDim.x * kGridThreads) {
    const double v = x[i];
    const double cv = clip_to(v, lo, hi);
    if (clipped) clipped[i] = cv;
    if (!isnan(v)) {
      a += v;
      c += cv;
      n += 1.0;
    }
  }
  auto block_sum = [&](double p1, double p2, double p3) {
    p1 = wave_sum_d(p1);
    p2 = wave_sum_d(p2);
    p3 = wave_sum_d(p3);
    if ((threadIdx.x & 63) == 0) {
      s1[threadIdx.x >> 6] = p1;
      s2[threadIdx.x >> 6] = p2;
      s3[threadIdx.x >> 6] = p3;
    }
    __syncthreads();
    a = c = n = 0.0;
    for (int i = 0; i < kGridThreads / 64; ++i) {
      a += s1[i];
      c += s2[i];
      n += s3[i];
    }
  };
  block_sum(a, c, n);
  if (threadIdx.x == 0) {
    __hip_atomic_store(&part[3 * blockIdx.x], a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&part[3 * blockIdx.x + 1], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&part[3 * blockIdx.x + 2], n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (!last_block(st)) return;
  static_assert(kGridBlocks <= kGridThreads, "one partial per thread");
  double p[3] = {0.0, 0.0, 0.0};
  if (threadIdx.x < gridDim.x)
    for (int j = 0; j < 3; ++j)
      p[j] = __hip_atomic_load(&part[3 * threadIdx.x + j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  block_sum(p[0], p[1], p[2]);
  if (threadIdx.x == 0) {
    st->lo = lo;
    st->hi = hi;
    st->mean_x = a / n;
    st->mean_c = c / n;
    st->count = n;
  }
}

__global__ void weights_kernel(const double* __restrict__ x, int B, const ClipState* st,
                               double* __restrict__ w, double* __restrict__ stats) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const double lo = st->lo, hi = st->hi, mc = st->mean_c, n = st->count;
  if (i < B) {
    const double cv = clip_to(x[i], lo, hi);
    w[i] = isnan(cv) ? 0.0 : 2.0 * (cv - mc) / n;
  }
  if (i == 0 && stats) {
    stats[0] = st->mean_x;
    stats[1] = mc;
    stats[2] = lo;
    stats[3] = hi;
    stats[4] = n;
  }
}

void select_into(const Src& src, const Plan& p, ClipState* st, unsigned* h, int nblk, int slot, hipStream_t s) {
  hipLaunchKernelGGL(range_kernel, dim3(nblk), dim3(kGridThreads), 0, s, src, p, st);
  constexpr int passes = (64 + kDigit - 1) / kDigit;
  for (int i = 0; i < passes; ++i)
    hipLaunchKernelGGL(digit_kernel, dim3(nblk), dim3(kGridThreads), 0, s, src, p, st, h, i == passes - 1 ? 1 : 0,
                       slot);
}

template <int V>
void launch_one(const double* x, int B, int method, double scale, double* clipped, double* weights, double* stats,
                hipStream_t s) {
  hipLaunchKernelGGL(clip_one_kernel<V>, dim3(1), dim3(kOneThreads), 0, s, x, B, method, scale, clipped, weights,
                     stats);
}

int loss_clip(const double* x, int B, int method, double scale, double* clipped, double* weights, double* stats,
              void* scratch, hipStream_t s) {
  if (B <= kOneMax * kOneThreads) {
    const int per = (B + kOneThreads - 1) / kOneThreads;
    if (per <= 2)
      launch_one<2>(x, B, method, scale, clipped, weights, stats, s);
    else if (per <= 8)
      launch_one<8>(x, B, method, scale, clipped, weights, stats, s);
    else
      launch_one<kOneMax>(x, B, method, scale, clipped, weights, stats, s);
    return 0;
  }
  ClipState* st = (ClipState*)scratch;
  unsigned* h = (unsigned*)((char*)scratch + kStateBytes);
  double* part = (double*)(h + kTargets * kBins);
  const int nblk = std::min(kGridBlocks, ceil_div(B, kGridThreads * 4));
  hipLaunchKernelGGL(state_init_kernel, dim3(kTargets * kBins / 256), dim3(256), 0, s, st, h);
  const Src plain{x, B, nullptr};
  if (method == 0) {
    const Plan p{2, {0.5, 0.5}};
    select_into(plain, p, st, h, nblk, 0, s);
    select_into(Src{x, B, &st->q[0]}, p, st, h, nblk, 1, s);
  } else if (method == 1) {
    select_into(plain, Plan{4, {0.25, 0.75}}, st, h, nblk, 0, s);
  }
  hipLaunchKernelGGL(clip_mean_kernel, dim3(nblk), dim3(kGridThreads), 0, s, x, B, method, scale, st, part, clipped);
  hipLaunchKernelGGL(weights_kernel, dim3(ceil_div(B, 256)), dim3(256), 0, s, x, B, st, weights, stats);
  return 0;
}

// The static scratch of jq_loss_clip_noalloc: one copy per device, held until
// the process ends.  Host code never uses the array's name as an address; it
// uses the device address from hipGetSymbolAddress, looked up once per device.
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

static void* scratch_address() {
  static std::mutex mu;
  static void* ptr[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  std::lock_guard<std::mutex> lk(mu);
  if (!ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
    ptr[dev] = p;
  }
  return ptr[dev];
}

int check_args(const double* x, int B, int method, double* weights) {
  if (B < 1 || B > JQ_LOSS_CLIP_MAX_B || !x || !weights || method < 0 || method > 2)
    return jq_fail(JQ_EINVAL, "jq_loss_clip: bad argument (1 <= B <= JQ_LOSS_CLIP_MAX_B, method 0 mad / 1 iqr / 2 none)");
  return 0;
}

}  // namespace

extern "C" {

size_t jq_loss_clip_workspace_bytes(int B) {
  (void)B;
  return kScratchBytes;
}

int jq_loss_clip(const double* x, int B, int method, double scale, double* clipped, double* weights, double* stats,
                 void* workspace, size_t ws_bytes, void* stream) {
  int rc = check_args(x, B, method, weights);
  if (rc) return rc;
  if (!workspace || ws_bytes < kScratchBytes)
    return jq_fail(JQ_EINVAL, "jq_loss_clip: workspace smaller than jq_loss_clip_workspace_bytes()");
  loss_clip(x, B, method, scale, clipped, weights, stats, workspace, (hipStream_t)stream);
  if (hipGetLastError() != hipSuccess) return jq_fail(JQ_EHIP, "kernel launch failed in jq_loss_clip");
  return JQ_OK;
}

int jq_loss_clip_noalloc(const double* x, int B, int method, double scale, double* clipped, double* weights,
                         double* stats, void* stream) {
  int rc = check_args(x, B, method, weights);
  if (rc) return rc;
  if (B > JQ_LOSS_CLIP_NOALLOC_MAX_B)
    return jq_fail(JQ_EINVAL, "jq_loss_clip_noalloc: B exceeds JQ_LOSS_CLIP_NOALLOC_MAX_B");
  void* p = scratch_address();
  if (!p) return jq_fail(JQ_EHIP, "jq_loss_clip_noalloc: device address of the static scratch not found");
  loss_clip(x, B, method, scale, clipped, weights, stats, p, (hipStream_t)stream);
  if (hipGetLastError() != hipSuccess) return jq_fail(JQ_EHIP, "kernel launch failed in jq_loss_clip_noalloc");
  return JQ_OK;
}

}  // extern "C"
