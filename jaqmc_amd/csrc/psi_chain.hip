// The row-wise part of a pre-LN Psiformer layer in one kernel (Laplacian mode,
// FP16X3, 256 features, 128-row units): for every unit
//   x1 = x + O Wo + bo;  t = LN2(x1);  t = tanh(t Wm + bm), ...;  x = x1 + t;
//   QKV = LN1'(x) Wqkv' + bqkv'   (the next layer's, head-split; none after the last)
// by the forward-Laplacian rules of gemm_kernel, in its order: the results are the same
// bit for bit as those of a GEMM a stage with the LayerNorms in their epilogues
// (JQ_OPT_SEPARATE_LAUNCHES; test_psiformer_chain_is_bit_identical holds both to it).
//
// Bound by the FP16 matrix rate, the LayerNorms and the memory together: as one
// GEMM a stage, with the LayerNorms in their epilogues, a layer read and wrote
// fourteen times the (rows, 256) stream, at the copy rate more than its products
// take.  Here a tile's rows stay on chip from the attention output to q, k, v: six
// streams (O and x in; x, q, k, v out).  One workgroup of eight waves per CU
// (the two FP16 planes of 128 x 256 fill the LDS) walks over the tiles; a wave
// owns 32 columns of every row, so accumulators (64 registers), the residual
// stream x1 (64) and two chunks of weight fragments fit the 256 registers of two
// waves per SIMD.  The columns of a lane are adjacent: x, q, k, v move as 128-byte
// row segments straight from registers, past the L2's weights (nontemporal).
// Vector-memory results return in order, so a load from HBM issued between the
// weights' delays them: O of the next tile is requested before the second
// LayerNorm and x as soon as the panel is written, the weights two chunks ahead
// (the next stage's before this one's stores), and no barrier waits for any of
// them.
// Measured, the four layers of 768 walkers of 42 electrons (4.1M rows of 128-row
// units, two-layer MLP): 61.1 ms in separate launches, 45.6 ms here (0.75 PFLOP/s
// issued).  A tile takes about 200k cycles: 74k are the products' at the matrix
// rate (what they take where no store is draining), the rest the LayerNorms' sums
// and the waits for the stores of x, q, k and v.  Taken back: loads of x and O
// spread over the chunks of a stage (+20k cycles), workgroups started at
// staggered times (no change), LayerNorm sums by halving steps over a lane row
// (10k cycles less, another rounding).
#include "kernels.h"

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
constexpr int kD = 256;          // features of every stage
constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kLS = kD + 8;      // f16 per panel row
constexpr int kFS = kD + 4;      // floats per row of the LayerNorm
constexpr int kNK = kD / 32;     // k chunks of a stage
constexpr int kCus = 256;
constexpr float kJScale = 64.f;  // fixed scale of Jacobian rows (gemm_impl.h)
constexpr int kMB = 8;           // 16-row blocks of a unit
constexpr int kProj = 3;         // column blocks of the projection

constexpr int kLds = 2 * 16 * kMB * kLS * 2 + 4 * (256 + 2 * 16 * kMB + 2 * kWaves + 4) +
                     4 * kD * (2 * (1 + kChainMlp + kProj) + 4);

// Maximum over the 16 lanes of a DPP row.
__device__ inline float max16(float t) {
  t = fmaxf(t, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0xB1, 0xF, 0xF, false)));
  t = fmaxf(t, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0x4E, 0xF, 0xF, false)));
  t = fmaxf(t, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0x141, 0xF, 0xF, false)));
  return fmaxf(t, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0x140, 0xF, 0xF, false)));
}
// x * sc (sc a power of two) as the sum of two FP16; each one mixed-precision
// multiply-add, which rounds once.
__device__ inline void split(float x, float sc, f16* h, f16* l) {
  *h = (f16)__builtin_fmaf(x, sc, 0.f);
  *l = (f16)__builtin_fmaf(x, sc, -(float)*h);
}
template <int CTRL>
__device__ inline float dpp_f(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, false));
}
// Sum over the wavefront's 64 lanes: 16-lane rows first, then (0 + 1) + (2 + 3).
__device__ inline float row_sum(float t) {
  t += dpp_f<0xB1>(t);
  t += dpp_f<0x4E>(t);
  t += dpp_f<0x141>(t);
  t += dpp_f<0x140>(t);
  t += __shfl_xor(t, 16);
  return t + __shfl_xor(t, 32);
}
// Power of two that brings mx into [2^13, 2^14), and its inverse.
__device__ inline void pow2_scale(float mx, float* sc, float* si) {
  *sc = *si = 1.f;
  if (mx > 0.f && mx <= 3.0e38f) {
    int e;
    (void)frexpf(mx, &e);
    int sh = 14 - e;
    sh = sh < -60 ? -60 : (sh > 60 ? 60 : sh);
    *sc = ldexpf(1.f, sh);
    *si = ldexpf(1.f, -sh);
  }
}

// PROJ: with the projection
template <bool PROJ>
__global__ __launch_bounds__(kThreads, 2) void psi_chain_kernel(const PsiChainArgs a, int tiles) {
  constexpr int MB = kMB, BM = 16 * MB, NJ = BM / kWaves;
  constexpr int MP = 6;  // row blocks from here on can hold padding rows (R > 96)
  static_assert(BM * kFS * 4 <= 2 * BM * kLS * 2, "the rows fit the panel");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  f16* const P0 = (f16*)smem;  // high plane, then the low plane
  f16* const P1 = P0 + BM * kLS;
  float* const sqp = (float*)(P1 + BM * kLS);   // [4][64] sums of squares
  float* const rowm = sqp + 256;                // [BM] row means
  float* const rowv = rowm + BM;                // [BM] J_v,r
  float* const mx8 = rowv + BM;                 // [2][waves] maxima of value and Laplacian rows
  float* const mx1 = mx8 + 2 * kWaves;          // [2] the same of a loaded panel
  float* const scal = mx1 + 2;                 // <d_r, d_0> of the value and Laplacian rows
  float* const pv = scal + 2;                  // per stage: inverse column scales, then biases
  const int nst = 1 + a.nm + (PROJ ? kProj : 0);
  float* const pbias = pv + nst * kD;
  float* const pln = pbias + nst * kD;          // scale and bias of LN2, then of the next LN1

  const int tid = threadIdx.x, lane_id = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Each part derives its addresses from a lane number of its own, which the
  // compiler takes as new: hoisted out of the tile loop they would spill.
#define LANE                                    \
  int lane = lane_id;                           \
  __asm__ volatile("" : "+v"(lane));            \
  const int lr = lane & 15, lg = lane >> 4;     \
  const int col = wave * 32 + 2 * lr; /* this lane's two columns of a block */
  auto planes = [&](const void* wlo, long wplane) __attribute__((always_inline)) {
    return (const f16*)((const bf16*)wlo + 3 * wplane);
  };
  for (int i = tid; i < nst * kD; i += kThreads) {
    const int st = i / kD, c = i % kD;
    if (st <= a.nm) {
      const long wp = (long)kD * kD;
      pv[i] = ((const float*)(planes(a.W[st], wp) + 2 * wp))[c];
      pbias[i] = a.bias[st] ? a.bias[st][c] : 0.f;
    } else {
      const long wp = (long)kProj * kD * kD;
      const int pc = (st - 1 - a.nm) * kD + c;
      pv[i] = ((const float*)(planes(a.Wp, wp) + 2 * wp))[pc];
      pbias[i] = a.bp ? a.bp[pc] : 0.f;
    }
  }
  for (int i = tid; i < kD; i += kThreads) {
    pln[i] = a.ln2_s[i];
    pln[kD + i] = a.ln2_b[i];
    pln[2 * kD + i] = PROJ ? a.ln1_s[i] : 0.f;
    pln[3 * kD + i] = PROJ ? a.ln1_b[i] : 0.f;
  }

  // XCD x = b % 8 takes a contiguous range of tiles, its workgroups neighbours
  const int tpx = (tiles + kXcds - 1) / kXcds;
  const int t0 = (int)(blockIdx.x % kXcds) * tpx, t1 = t0 + tpx < tiles ? t0 + tpx : tiles;
  const int slot = (int)blockIdx.x / kXcds, step = (int)gridDim.x / kXcds;
  const int rows = a.units * BM;

  f32x4 acc[MB][2], aux[2 * MB];  // aux: x, x1 (two rows of two columns each), or the next panel
  uint4 b[2][2][2];               // [set][plane][column of the pair]
  auto bload = [&](int set, const f16* W, long wp, int c, int boff) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) b[set][s][nb] = *(const uint4*)(W + s * wp + (boff + nb * kD + c * 32));
  };
  // row j of this wave's share of tile t's panel
  auto load_row = [&](int t, int j, int lane) __attribute__((always_inline)) {
    int r = t * BM + wave + kWaves * j;
    r = r < rows ? r : rows - 1;
    aux[j] = __builtin_nontemporal_load((const f32x4*)(a.O + (long)r * a.ldo + 4 * lane));
  };
  // One stage: acc = panel . W^T over this wave's 32 columns, every row.  Its
  // first two chunks' fragments are there; those of the next stage's (Wn) are
  // requested after their sets' last products, before the epilogue's stores.
  auto products = [&](const f16* W, long wp, const f16* Wn, long wpn) __attribute__((always_inline)) {
    LANE
    const int boff = col * kD + 8 * lg;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < kNK; ++c) {
      const f16* ap = P0 + lr * kLS + c * 32 + 8 * lg;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const f16x8 a0 = *(const f16x8*)(ap + 16 * mb * kLS), a1 = *(const f16x8*)(ap + (16 * mb + BM) * kLS);
        const uint4(&bs)[2][2] = b[c & 1];
        // small terms first
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, __builtin_bit_cast(f16x8, bs[0][nb]), acc[mb][nb], 0, 0, 0);
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, __builtin_bit_cast(f16x8, bs[1][nb]), acc[mb][nb], 0, 0, 0);
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, __builtin_bit_cast(f16x8, bs[0][nb]), acc[mb][nb], 0, 0, 0);
      }
      if (c + 2 < kNK)
        bload(c & 1, W, wp, c + 2, boff);
      else
        bload(c & 1, Wn, wpn, c + 2 - kNK, boff);
      __builtin_amdgcn_sched_barrier(0);  // no other chunk's operands in registers
    }
  };
  // inverse scales of the panel's value and Laplacian rows
  float ival = 1.f, ilap = 1.f;
  // acc without the power-of-two scales, the bias on the value rows
  auto unscale = [&](int st) __attribute__((always_inline)) {
    LANE
    const float2 cs = *(const float2*)&pv[st * kD + col], bv = *(const float2*)&pbias[st * kD + col];
    const float csi[2] = {cs.x, cs.y}, bb[2] = {bv.x, bv.y};
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float ir = 1.f / kJScale;
        if (mb == 0 && v < ROW_J0) ir = lg == 0 ? (v == ROW_VAL ? ival : ilap) : ir;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          acc[mb][nb][v] *= ir * csi[nb];
          if (mb == 0 && v == ROW_VAL) acc[mb][nb][v] += lg == 0 ? bb[nb] : 0.f;
        }
      }
  };
  // (the fused multiply-adds of this rule and of the LayerNorm are written out as
  // gemm_kernel's are compiled)
  auto tanh_rule = [&]() __attribute__((always_inline)) {
#pragma clang fp contract(off)
    LANE
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      float sq = 0.f;
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float j = acc[m][nb][v];
          if (m == 0 && v == 0)
            sq = lg == 0 ? 0.f : fmaf(j, j, acc[0][nb][1] * acc[0][nb][1]);
          else if (m > 0 || v > 1)
            sq = fmaf(j, j, sq);
        }
      sq += __shfl_xor(sq, 16);
      sq += __shfl_xor(sq, 32);
      const float y0 = __shfl(acc[0][nb][ROW_VAL], lr);
      const float y1 = __shfl(acc[0][nb][ROW_LAP], lr);
      const float th = tanhf(y0);
      const float d1 = fmaf(-th, th, 1.f);
      const float lap = fmaf(d1, y1, -2.f * th * d1 * sq);
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[m][nb][v] *= d1;
      if (lg == 0) {
        acc[0][nb][ROW_VAL] = th;
        acc[0][nb][ROW_LAP] = lap;
      }
    }
  };
  // acc = LN(acc).  The rows go through LDS (the panel is free), where a
  // wave sums sixteen of them whole, a row's 256 columns over its lanes:
  // position 4 l + q of a row holds column 64 (l / 16) + 16 q + l % 16.
  // Sums are taken in gemm_kernel's order.
  auto layernorm = [&](const float* ln) __attribute__((always_inline)) {
#pragma clang fp contract(off)
    LANE
    constexpr float invD = 1.f / kD;
    float* const F = (float*)smem;
    lds_barrier();  // every wave is done with the panel
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      float* const fp = F + 4 * lg * kFS + (wave >> 1) * 64 + ((2 * lr + nb) & 15) * 4 + (wave & 1) * 2 + (lr >> 3);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int v = 0; v < 4; ++v) fp[(mb * 16 + v) * kFS] = acc[mb][nb][v];
    }
    lds_barrier();
    {
      auto sum4 = [](const f32x4& x) __attribute__((always_inline)) {
        return row_sum(((x.x + x.y) + x.z) + x.w);
      };
      f32x4 z = *(const f32x4*)&F[4 * lane];
      z -= sum4(z) * invD;  // centred value row
      float mean = 0.f, dot = 0.f;  // of row 16 wave + lane % 16
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int r = 16 * wave + k;
        f32x4 x = *(const f32x4*)&F[r * kFS + 4 * lane];
        const float m = sum4(x) * invD;
        x -= m;
        const float t = row_sum(fmaf(x.w, z.w, fmaf(x.z, z.z, fmaf(x.y, z.y, x.x * z.x))));
        mean = lr == k ? m : mean;
        dot = lr == k ? t : dot;
        if (r > 0) F[r * kFS + 4 * lane] = fmaf(x.w, x.w, fmaf(x.z, x.z, fmaf(x.x, x.x, x.y * x.y)));
      }
      if (lane < 16) {
        const int r = 16 * wave + lane;
        rowm[r] = mean;
        rowv[r] = r >= ROW_J0 && r < a.R ? 2.f * invD * dot : 0.f;  // J_v,r = 2/D <d_r, d_0>
        if (r < ROW_J0) scal[r] = dot;
      }
    }
    lds_barrier();
    // sums of |d_r|^2 over the Jacobian rows, a lane group's rows in turn
    if (wave < 4) {
      float sq = 0.f;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int r = mb * 16 + 4 * wave + v;
          if (r >= ROW_J0 && r < a.R) sq += F[r * kFS + 4 * lane];
        }
      sqp[wave * 64 + lane] = sq;
    }
    float d0[2];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const f32x4 m = *(const f32x4*)&rowm[mb * 16 + 4 * lg];
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) acc[mb][nb] -= m;
    }
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) d0[nb] = __shfl(acc[0][nb][ROW_VAL], lr);
    const float j0 = rowv[lane], j1 = rowv[64 + lane];
    const float jv2 = wave_sum(j0 * j0) + wave_sum(j1 * j1);
    lds_barrier();
    float sqt = (sqp[lane] + sqp[128 + lane]) + (sqp[64 + lane] + sqp[192 + lane]);
    sqt += __shfl_xor(sqt, 8);
    sqt += __shfl_xor(sqt, 4);
    sqt += __shfl_xor(sqt, 2);
    sqt += __shfl_xor(sqt, 1);
    sqt += __shfl_xor(sqt, 16);
    sqt += __shfl_xor(sqt, 32);
    // the variance, its Laplacian, s = (v + eps)^-1/2 and its derivatives
    const float lapv = 2.f * invD * (scal[ROW_LAP] + sqt);
    const float ve = fmaf(scal[ROW_VAL], invD, a.eps);
    const float sv = rsqrtf(ve);
    const float s1 = -0.5f * sv / ve;
    const float s2 = 0.75f * sv / (ve * ve);
    const float laps = fmaf(s1, lapv, s2 * jv2);
    const float2 g2 = *(const float2*)&ln[col], b2 = *(const float2*)&ln[kD + col];
    const float g[2] = {g2.x, g2.y}, bb[2] = {b2.x, b2.y};
    float cross[2] = {0.f, 0.f};
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const f32x4 jv = *(const f32x4*)&rowv[mb * 16 + 4 * lg];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float js = s1 * jv[v];  // 0 outside the Jacobian rows
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          const float d = acc[mb][nb][v];
          cross[nb] = fmaf(d, js, cross[nb]);
          float y = g[nb] * fmaf(sv, d, js * d0[nb]);
          if (mb >= MP) y = mb * 16 + 4 * lg + v < a.R ? y : 0.f;
          if (mb == 0 && v == ROW_VAL) {
            // (gemm_kernel's rounding of this row block: from the second 16
            // columns of a 64-column group on, sv d is the rounded product)
            const float p = sv * d;
            if ((wave & 1) != 0 || lr >= 8) y = g[nb] * fmaf(js, d0[nb], p);
            y = lg == 0 ? fmaf(p, g[nb], bb[nb]) : y;
          }
          if (mb == 0 && v == ROW_LAP) y = lg == 0 ? d : y;
          acc[mb][nb][v] = y;
        }
      }
    }
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      float t = cross[nb] + __shfl_xor(cross[nb], 16);
      t += __shfl_xor(t, 32);
      if (lg == 0) acc[0][nb][ROW_LAP] = g[nb] * fmaf(2.f, t, fmaf(acc[0][nb][ROW_LAP], sv, d0[nb] * laps));
    }
  };
  // acc into the panel: value and Laplacian rows scaled to [2^13, 2^14)
  auto put_panel = [&]() __attribute__((always_inline)) {
    LANE
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const float m = max16(fmaxf(fabsf(acc[0][0][p]), fabsf(acc[0][1][p])));
      if (lane == 0) mx8[p * kWaves + wave] = m;
    }
    lds_barrier();  // every wave is done with the panel
    float m[2], sval, slap;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const f32x4 q0 = *(const f32x4*)&mx8[p * kWaves], q1 = *(const f32x4*)&mx8[p * kWaves + 4];
      m[p] = fmaxf(fmaxf(fmaxf(q0.x, q0.y), fmaxf(q0.z, q0.w)), fmaxf(fmaxf(q1.x, q1.y), fmaxf(q1.z, q1.w)));
    }
    pow2_scale(m[0], &sval, &ival);
    pow2_scale(m[1], &slap, &ilap);
    f16 *p0 = P0 + 4 * lg * kLS + col, *p1 = P1 + 4 * lg * kLS + col;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float sc = kJScale;
        if (mb == 0 && v < ROW_J0) sc = lg == 0 ? (v == ROW_VAL ? sval : slap) : sc;
        f16 h[2], l[2];
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) split(acc[mb][nb][v], sc, &h[nb], &l[nb]);
        *(unsigned*)(p0 + (mb * 16 + v) * kLS) = *(const unsigned*)h;
        *(unsigned*)(p1 + (mb * 16 + v) * kLS) = *(const unsigned*)l;
      }
    lds_barrier();  // the panel is ready
  };

  const long wpD = (long)kD * kD, wpP = (long)kProj * kD * kD;
  const f16* const W0 = planes(a.W[0], wpD);
  const f16* const Wp = PROJ ? planes(a.Wp, wpP) : W0;
  int t = t0 + slot;
  if (t >= t1) return;
  {
    LANE
    bload(0, W0, wpD, 0, col * kD + 8 * lg);
    bload(1, W0, wpD, 1, col * kD + 8 * lg);
#pragma unroll
    for (int j = 0; j < NJ; ++j) load_row(t, j, lane);
  }
  // none outstanding from before the loop (vmcnt 0), so that its waits cover
  // the loads of the tile before and not the stores behind them
  __builtin_amdgcn_s_waitcnt(0x0F70);
  for (; t < t1; t += step) {
    // ---- the panel of O; wave w holds rows w, w + 8, ... ----
    lds_barrier();  // every wave is done with the previous tile
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      LANE
      float sc = kJScale;
      if (j == 0 && wave < ROW_J0) {
        const f32x4 v = aux[j];
        const float mx = wave_max(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        float si;
        pow2_scale(mx, &sc, &si);
        if (lane == 0) mx1[wave] = si;
      }
      f16 h[4], l[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) split(aux[j][e], sc, &h[e], &l[e]);
      const int at = (wave + kWaves * j) * kLS + 4 * lane;
      *(uint2*)(P0 + at) = *(const uint2*)h;
      *(uint2*)(P1 + at) = *(const uint2*)l;
    }
    float* const xt = a.x + (long)t * BM * kD;
    {
      LANE
      const int xoff = 4 * lg * kD + col;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const f32x2 q = __builtin_nontemporal_load((const f32x2*)(xt + (mb * 16 + v) * kD + xoff));
          aux[2 * mb + v / 2][2 * (v & 1)] = q.x;
          aux[2 * mb + v / 2][2 * (v & 1) + 1] = q.y;
        }
    }
    lds_barrier();
    ival = mx1[ROW_VAL];
    ilap = mx1[ROW_LAP];
    // ---- x1 = x + O Wo + bo, LN2 ----
    products(W0, wpD, planes(a.W[1], wpD), wpD);
    unscale(0);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          acc[mb][nb][v] += aux[2 * mb + v / 2][2 * (v & 1) + nb];
          aux[2 * mb + v / 2][2 * (v & 1) + nb] = acc[mb][nb][v];
        }
    layernorm(pln);
    put_panel();
    // ---- the MLP; x = x1 + its output ----
#pragma unroll 1
    for (int st = 1; st <= a.nm; ++st) {
      const bool last = st == a.nm;
      const f16* const Wn = last ? Wp : planes(a.W[st + 1], wpD);
      products(planes(a.W[st], wpD), wpD, Wn, last && PROJ ? wpP : wpD);
      unscale(st);
      tanh_rule();
      if (!last) put_panel();
    }
    {
      LANE
      const int xoff = 4 * lg * kD + col;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
#pragma unroll
          for (int nb = 0; nb < 2; ++nb) acc[mb][nb][v] += aux[2 * mb + v / 2][2 * (v & 1) + nb];
          __builtin_nontemporal_store(f32x2{acc[mb][0][v], acc[mb][1][v]}, (f32x2*)(xt + (mb * 16 + v) * kD + xoff));
        }
    }
    {  // the next tile's O
      LANE
      const int tn = t + step < t1 ? t + step : t;
#pragma unroll
      for (int j = 0; j < NJ; ++j) load_row(tn, j, lane);
    }
    if constexpr (!PROJ) continue;
    // ---- LN1 and the projection of the next layer ----
    layernorm(pln + 2 * kD);
    put_panel();
    auto store = [&](int cb) __attribute__((always_inline)) {
      unscale(1 + a.nm + cb);
      LANE
      const int n0 = cb * kD + wave * 32;  // 32 columns of one head
      const int prt = n0 / kD, hh = (n0 % kD) / a.dh, dd = n0 % a.dh;
      const int w = t / a.N, i = t % a.N;
      float* const y = a.Y + ((((long)w * kProj + prt) * a.H + hh) * a.N + i) * ((long)BM * a.dh) + dd;
      const int yoff = 4 * lg * a.dh + 2 * lr;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          __builtin_nontemporal_store(f32x2{acc[mb][0][v], acc[mb][1][v]},
                                      (f32x2*)(y + (long)(mb * 16 + v) * a.dh + yoff));
    };
#pragma unroll 1
    for (int cb = 0; cb < kProj; ++cb) {
      const bool last = cb == kProj - 1;
      products(Wp + cb * wpD, wpP, last ? W0 : Wp + (cb + 1) * wpD, last ? wpD : wpP);
      store(cb);
    }
  }
}

#undef LANE

template <bool PROJ>
int launch_chain(const PsiChainArgs& a, hipStream_t s) {
  constexpr int lds = kLds;
  static_assert(lds <= 160 * 1024, "one workgroup per CU");
  static const hipError_t attr = hipFuncSetAttribute((const void*)psi_chain_kernel<PROJ>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return -1;
  hipLaunchKernelGGL((psi_chain_kernel<PROJ>), dim3(kCus), dim3(kThreads), lds, s, a, a.units);
  return 0;
}
}  // namespace

// 128-row units (32 to 42 electrons) alone: there the stages in a GEMM each round
// alike, whatever the batch.  Both sides measured, energies of 42 electrons: 1 walker
// 2785 us in separate launches, 2652 us here; 16 walkers 4147 and 3916 us; 64 walkers
// 10180 and 8551 us.
bool psi_chain_supported(int Rp, int D, int prec, int n_mlp, const int* width) {
  if (prec != PREC_FP16X3 || Rp != 128 || D != kD || n_mlp < 1 || n_mlp > kChainMlp) return false;
  for (int j = 0; j <= n_mlp; ++j)
    if (width[j] != kD) return false;
  return true;
}

int launch_psi_chain(const PsiChainArgs& a, hipStream_t s) { return a.Wp ? launch_chain<true>(a, s) : launch_chain<false>(a, s); }
