// The row-wise part of a pre-LN Psiformer layer in one kernel (Laplacian mode,
// FP16X3, 256 features): for every tile of whole units
//   x1 = x + O Wo + bo;  t = LN2(x1);  t = tanh(t Wm + bm), ...;  x = x1 + t;
//   QKV = LN1'(x) Wqkv' + bqkv'   (the next layer's, head-split; none after the last)
// by the forward-Laplacian rules of gemm_kernel and layernorm_lap_kernel.
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
// row segments straight from registers.  Loads hide behind products: weights two
// chunks ahead (the next stage's before this one's stores), x row block by row
// block during the first stage, the next tile's O during the first q, k, v block.
// Measured, the four layers of 768 walkers of 42 electrons (4.1M rows of 128-row
// units, two-layer MLP): 61.1 ms in separate launches, 44.2 ms here (0.77 PFLOP/s
// issued); their energies 111.0 -> 92.9 ms.
#include "kernels.h"

namespace {

constexpr int kD = 256;          // features of every stage
constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kLS = kD + 8;      // f16 per panel row
constexpr int kNK = kD / 32;     // k chunks of a stage
constexpr int kCus = 256;
constexpr float kJScale = 64.f;  // fixed scale of Jacobian rows (gemm_impl.h)
constexpr int kProj = 3;         // column blocks of the projection

template <int MB>
constexpr int chain_lds() {
  return 2 * 16 * MB * kLS * 2 + 4 * (kWaves * 16 * MB + 16 * MB + 16 * kWaves + 2 * 16 + 2 * 16) +
         4 * kD * (2 * (1 + kChainMlp + kProj) + 4);
}

// Sum and maximum over the 16 lanes of a DPP row.
__device__ inline float sum16(float t) {
  t += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0xB1, 0xF, 0xF, false));
  t += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0x4E, 0xF, 0xF, false));
  t += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0x141, 0xF, 0xF, false));
  return t + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0x140, 0xF, 0xF, false));
}
__device__ inline float max16(float t) {
  t = fmaxf(t, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0xB1, 0xF, 0xF, false)));
  t = fmaxf(t, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0x4E, 0xF, 0xF, false)));
  t = fmaxf(t, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0x141, 0xF, 0xF, false)));
  return fmaxf(t, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0x140, 0xF, 0xF, false)));
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

// MB: 16-row blocks of a tile; MBU: of a unit
template <int MB, int MBU>
__global__ __launch_bounds__(kThreads, 2) void psi_chain_kernel(const PsiChainArgs a, int tiles) {
  constexpr int BM = 16 * MB, RU = 16 * MBU, UPT = MB / MBU, NJ = BM / kWaves;
  static_assert(MB % MBU == 0 && MB <= kNK && UPT <= 4, "whole units; one row block a chunk");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  f16* const P0 = (f16*)smem;  // high plane, then the low plane
  f16* const P1 = P0 + BM * kLS;
  float* const part = (float*)(P1 + BM * kLS);  // [waves][BM] row partials
  float* const rowv = part + kWaves * BM;       // [BM] row means, then J_v,r
  float* const mx8 = rowv + BM;                 // [2 UPT][waves] maxima of value and Laplacian rows
  float* const mx1 = mx8 + 16 * kWaves;         // [2 UPT] the same of a loaded panel
  float* const scal = mx1 + 32;                 // [waves][4] sums of squares per unit
  float* const pv = scal + 32;                  // per stage: inverse column scales, then biases
  const int nst = 1 + a.nm + (a.Wp ? kProj : 0);
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
    pln[2 * kD + i] = a.Wp ? a.ln1_s[i] : 0.f;
    pln[3 * kD + i] = a.Wp ? a.ln1_b[i] : 0.f;
  }

  // XCD x = b % 8 takes a contiguous range of tiles, its workgroups neighbours
  const int tpx = (tiles + kXcds - 1) / kXcds;
  const int t0 = (int)(blockIdx.x % kXcds) * tpx, t1 = t0 + tpx < tiles ? t0 + tpx : tiles;
  const int slot = (int)blockIdx.x / kXcds, step = (int)gridDim.x / kXcds;
  const int rows = a.units * RU;

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
    aux[j] = *(const f32x4*)(a.O + (long)r * a.ldo + 4 * lane);
  };
  // One stage: acc = panel . W^T over this wave's 32 columns, every row.  Its
  // first two chunks' fragments are there; those of the next stage's (Wn) are
  // requested after their sets' last products, before the epilogue's stores.
  // extra(c) issues other loads after chunk c.
  auto products = [&](const f16* W, long wp, const f16* Wn, long wpn, auto extra) __attribute__((always_inline)) {
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
      extra(c, lane);
      __builtin_amdgcn_sched_barrier(0);  // no other chunk's operands in registers
    }
  };
  // inverse scales of the panel's value and Laplacian rows
  float ival[UPT], ilap[UPT];
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
        if (mb % MBU == 0 && v < ROW_J0) ir = lg == 0 ? (v == ROW_VAL ? ival[mb / MBU] : ilap[mb / MBU]) : ir;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          acc[mb][nb][v] *= ir * csi[nb];
          if (mb % MBU == 0 && v == ROW_VAL) acc[mb][nb][v] += lg == 0 ? bb[nb] : 0.f;
        }
      }
  };
  // (the fused multiply-adds of this rule and of the LayerNorm are written out,
  // so that a unit's result does not depend on its place in the tile)
  auto tanh_rule = [&]() __attribute__((always_inline)) {
#pragma clang fp contract(off)
    LANE
#pragma unroll
    for (int u = 0; u < UPT; ++u)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        float sq = 0.f;
#pragma unroll
        for (int m = 0; m < MBU; ++m)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float j = acc[u * MBU + m][nb][v];
            const bool jrow = !(m == 0 && lg == 0 && v < ROW_J0);
            sq = fmaf(jrow ? j : 0.f, j, sq);
          }
        sq += __shfl_xor(sq, 16);
        sq += __shfl_xor(sq, 32);
        const float y0 = __shfl(acc[u * MBU][nb][ROW_VAL], lr);
        const float y1 = __shfl(acc[u * MBU][nb][ROW_LAP], lr);
        const float th = tanhf(y0);
        const float d1 = fmaf(-th, th, 1.f);
        const float lap = fmaf(d1, y1, -2.f * th * d1 * sq);
#pragma unroll
        for (int m = 0; m < MBU; ++m)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[u * MBU + m][nb][v] *= d1;
        if (lg == 0) {
          acc[u * MBU][nb][ROW_VAL] = th;
          acc[u * MBU][nb][ROW_LAP] = lap;
        }
      }
  };
  // acc = LN(acc).  A row statistic is a sum over the 16 lanes of a lane group,
  // combined over the waves in LDS.
  auto layernorm = [&](const float* ln) __attribute__((always_inline)) {
#pragma clang fp contract(off)
    LANE
    constexpr float invD = 1.f / kD;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float t = sum16(acc[mb][0][v] + acc[mb][1][v]);
        if (lr == 0) part[wave * BM + mb * 16 + 4 * lg + v] = t;
      }
    __syncthreads();
    auto total = [&](int r) __attribute__((always_inline)) {
      float t[kWaves];
#pragma unroll
      for (int w = 0; w < kWaves; ++w) t[w] = part[w * BM + r];
      return ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
    };
    if (tid < BM) rowv[tid] = total(tid) * invD;
    __syncthreads();
    float d0[UPT][2];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const f32x4 m = *(const f32x4*)&rowv[mb * 16 + 4 * lg];
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) acc[mb][nb] -= m;
      if (mb % MBU == 0)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) d0[mb / MBU][nb] = __shfl(acc[mb][nb][ROW_VAL], lr);
    }
    // <d_r, d_0> per row; sum of |d_r|^2 over the Jacobian rows of a unit
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      float sq = 0.f;
#pragma unroll
      for (int m = 0; m < MBU; ++m)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int mb = u * MBU + m, r = m * 16 + 4 * lg + v;
          const float x0 = acc[mb][0][v], x1 = acc[mb][1][v];
          sq += (r >= ROW_J0 && r < a.R) ? fmaf(x1, x1, x0 * x0) : 0.f;
          const float t = sum16(fmaf(x1, d0[u][1], x0 * d0[u][0]));
          if (lr == 0) part[wave * BM + u * RU + r] = t;
        }
      sq = wave_sum(sq);
      if (lane == 0) scal[wave * 4 + u] = sq;
    }
    __syncthreads();
    // J_v,r = 2/D <d_r, d_0> of the Jacobian rows; per unit the variance, its
    // Laplacian, s = (v + eps)^-1/2 and its derivatives
    float sv[UPT], s1[UPT], s2[UPT], lapv[UPT];
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      float q[kWaves];
#pragma unroll
      for (int w = 0; w < kWaves; ++w) q[w] = scal[w * 4 + u];
      const float sqt = ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
      lapv[u] = 2.f * invD * (total(u * RU + ROW_LAP) + sqt);
      const float ve = fmaf(total(u * RU + ROW_VAL), invD, a.eps);
      sv[u] = rsqrtf(ve);
      s1[u] = -0.5f * sv[u] / ve;
      s2[u] = 0.75f * sv[u] / (ve * ve);
    }
    if (tid < BM) {
      const int r = tid % RU;
      rowv[tid] = (r >= ROW_J0 && r < a.R) ? 2.f * invD * total(tid) : 0.f;
    }
    __syncthreads();
    const float2 g2 = *(const float2*)&ln[col], b2 = *(const float2*)&ln[kD + col];
    const float g[2] = {g2.x, g2.y}, bb[2] = {b2.x, b2.y};
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      float cross[2] = {0.f, 0.f}, jv2 = 0.f;
#pragma unroll
      for (int m = 0; m < MBU; ++m) {
        const int mb = u * MBU + m;
        const f32x4 jv = *(const f32x4*)&rowv[mb * 16 + 4 * lg];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int r = m * 16 + 4 * lg + v;
          const float js = s1[u] * jv[v];  // 0 outside the Jacobian rows
          jv2 = fmaf(jv[v], jv[v], jv2);
          const bool jr = r >= ROW_J0 && r < a.R;
#pragma unroll
          for (int nb = 0; nb < 2; ++nb) {
            const float d = acc[mb][nb][v];
            cross[nb] = fmaf(d, js, cross[nb]);
            const float y = jr ? g[nb] * fmaf(d, sv[u], d0[u][nb] * js) : 0.f;
            if (m == 0 && v == ROW_VAL)
              acc[mb][nb][v] = lg == 0 ? fmaf(g[nb], d * sv[u], bb[nb]) : y;
            else if (m == 0 && v == ROW_LAP)
              acc[mb][nb][v] = lg == 0 ? d : y;
            else
              acc[mb][nb][v] = y;
          }
        }
      }
      jv2 += __shfl_xor(jv2, 16);
      jv2 += __shfl_xor(jv2, 32);
      const float laps = fmaf(s1[u], lapv[u], s2[u] * jv2);
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        float t = cross[nb] + __shfl_xor(cross[nb], 16);
        t += __shfl_xor(t, 32);
        if (lg == 0)
          acc[u * MBU][nb][ROW_LAP] = g[nb] * fmaf(2.f, t, fmaf(acc[u * MBU][nb][ROW_LAP], sv[u], d0[u][nb] * laps));
      }
    }
  };
  // acc into the panel: value and Laplacian rows scaled to [2^13, 2^14)
  auto put_panel = [&]() __attribute__((always_inline)) {
    LANE
#pragma unroll
    for (int u = 0; u < UPT; ++u)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const float m = max16(fmaxf(fabsf(acc[u * MBU][0][p]), fabsf(acc[u * MBU][1][p])));
        if (lane == 0) mx8[(2 * u + p) * kWaves + wave] = m;
      }
    __syncthreads();  // every wave is done with the panel
    float sval[UPT], slap[UPT];
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      float m[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const f32x4 q0 = *(const f32x4*)&mx8[(2 * u + p) * kWaves], q1 = *(const f32x4*)&mx8[(2 * u + p) * kWaves + 4];
        m[p] = fmaxf(fmaxf(fmaxf(q0.x, q0.y), fmaxf(q0.z, q0.w)), fmaxf(fmaxf(q1.x, q1.y), fmaxf(q1.z, q1.w)));
      }
      pow2_scale(m[0], &sval[u], &ival[u]);
      pow2_scale(m[1], &slap[u], &ilap[u]);
    }
    f16 *p0 = P0 + 4 * lg * kLS + col, *p1 = P1 + 4 * lg * kLS + col;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float sc = kJScale;
        if (mb % MBU == 0 && v < ROW_J0) sc = lg == 0 ? (v == ROW_VAL ? sval[mb / MBU] : slap[mb / MBU]) : sc;
        f16 h[2], l[2];
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          const float y = acc[mb][nb][v] * sc;
          h[nb] = (f16)y;
          l[nb] = (f16)(y - (float)h[nb]);
        }
        *(unsigned*)(p0 + (mb * 16 + v) * kLS) = *(const unsigned*)h;
        *(unsigned*)(p1 + (mb * 16 + v) * kLS) = *(const unsigned*)l;
      }
    __syncthreads();  // the panel is ready
  };

  const long wpD = (long)kD * kD, wpP = (long)kProj * kD * kD;
  const f16* const W0 = planes(a.W[0], wpD);
  const f16* const Wp = a.Wp ? planes(a.Wp, wpP) : W0;
  int t = t0 + slot;
  if (t >= t1) return;
  {
    LANE
    bload(0, W0, wpD, 0, col * kD + 8 * lg);
    bload(1, W0, wpD, 1, col * kD + 8 * lg);
#pragma unroll
    for (int j = 0; j < NJ; ++j) load_row(t, j, lane);
  }
  for (; t < t1; t += step) {
    // ---- the panel of O; wave w holds rows w, w + 8, ... ----
    __syncthreads();  // every wave is done with the previous tile
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      LANE
      float sc = kJScale;
      if (j % (2 * MBU) == 0 && wave < ROW_J0) {
        const f32x4 v = aux[j];
        const float mx = wave_max(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        float si;
        pow2_scale(mx, &sc, &si);
        if (lane == 0) mx1[j / (2 * MBU) * 2 + wave] = si;
      }
      f16 h[4], l[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float y = aux[j][e] * sc;
        h[e] = (f16)y;
        l[e] = (f16)(y - (float)h[e]);
      }
      const int at = (wave + kWaves * j) * kLS + 4 * lane;
      *(uint2*)(P0 + at) = *(const uint2*)h;
      *(uint2*)(P1 + at) = *(const uint2*)l;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      ival[u] = mx1[2 * u];
      ilap[u] = mx1[2 * u + 1];
    }
    // ---- x1 = x + O Wo + bo, LN2 ----
    const long row0 = (long)t * BM;
    float* const xt = a.x + row0 * kD;
    products(W0, wpD, planes(a.W[1], wpD), wpD, [&](int c, int lane) __attribute__((always_inline)) {
      const int xoff = (lane >> 4) * 4 * kD + wave * 32 + 2 * (lane & 15);
      if (c < MB && (UPT == 1 || row0 + (c / MBU + 1) * RU <= rows))
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float2 q = *(const float2*)(xt + (c * 16 + v) * kD + xoff);
          aux[2 * c + v / 2][2 * (v & 1)] = q.x;
          aux[2 * c + v / 2][2 * (v & 1) + 1] = q.y;
        }
    });
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
      products(planes(a.W[st], wpD), wpD, Wn, last && a.Wp ? wpP : wpD, [](int, int) {});
      unscale(st);
      tanh_rule();
      if (!last) put_panel();
    }
    {
      LANE
      const int xoff = 4 * lg * kD + col;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        if (UPT == 1 || row0 + (mb / MBU + 1) * RU <= rows)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) acc[mb][nb][v] += aux[2 * mb + v / 2][2 * (v & 1) + nb];
            *(float2*)(xt + (mb * 16 + v) * kD + xoff) = float2{acc[mb][0][v], acc[mb][1][v]};
          }
    }
    const int tn = t + step < t1 ? t + step : t;
    if (!a.Wp) {
      LANE
#pragma unroll
      for (int j = 0; j < NJ; ++j) load_row(tn, j, lane);
      continue;
    }
    // ---- LN1 and the projection of the next layer ----
    layernorm(pln + 2 * kD);
    put_panel();
    auto store = [&](int cb) __attribute__((always_inline)) {
      unscale(1 + a.nm + cb);
      LANE
      const int n0 = cb * kD + wave * 32;  // 32 columns of one head
      const int prt = n0 / kD, hh = (n0 % kD) / a.dh, dd = n0 % a.dh;
#pragma unroll
      for (int u = 0; u < UPT; ++u) {
        const int unit = t * UPT + u;
        if (UPT > 1 && unit >= a.units) break;
        const int w = unit / a.N, i = unit % a.N;
        float* const yu = a.Y + ((((long)w * kProj + prt) * a.H + hh) * a.N + i) * ((long)RU * a.dh) + dd;
        const int yoff = 4 * lg * a.dh + 2 * lr;
#pragma unroll
        for (int m = 0; m < MBU; ++m)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            *(float2*)(yu + (long)(m * 16 + v) * a.dh + yoff) = float2{acc[u * MBU + m][0][v], acc[u * MBU + m][1][v]};
      }
    };
    products(Wp, wpP, Wp + wpD, wpP, [&](int c, int lane) __attribute__((always_inline)) {
      if (c < MB) {
        load_row(tn, 2 * c, lane);
        load_row(tn, 2 * c + 1, lane);
      }
    });
    store(0);
#pragma unroll 1
    for (int cb = 1; cb < kProj; ++cb) {
      const bool last = cb == kProj - 1;
      products(Wp + cb * wpD, wpP, last ? W0 : Wp + (cb + 1) * wpD, last ? wpD : wpP, [](int, int) {});
      store(cb);
    }
  }
}

#undef LANE

template <int MB, int MBU>
int launch_chain(const PsiChainArgs& a, hipStream_t s) {
  constexpr int lds = chain_lds<MB>();
  static_assert(lds <= 160 * 1024, "one workgroup per CU");
  static const hipError_t attr = hipFuncSetAttribute((const void*)psi_chain_kernel<MB, MBU>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return -1;
  const int tiles = ceil_div(a.units, MB / MBU);
  hipLaunchKernelGGL((psi_chain_kernel<MB, MBU>), dim3(kCus), dim3(kThreads), lds, s, a, tiles);
  return 0;
}

}  // namespace

bool psi_chain_supported(int Rp, int D, int prec, int n_mlp, const int* width) {
  if (prec != PREC_FP16X3 || D != kD || n_mlp < 1 || n_mlp > kChainMlp) return false;
  for (int j = 0; j <= n_mlp; ++j)
    if (width[j] != kD) return false;
  return Rp == 128 || Rp == 96 || Rp == 64 || Rp == 48 || Rp == 32;
}

int launch_psi_chain(const PsiChainArgs& a, int Rp, hipStream_t s) {
  // One unit a tile while every unit has a CU of its own; beyond that 96- and
  // 128-row tiles, whose weights are read once for several units.  Both sides
  // measured, energies: 10 electrons (32-row
  // units) x 16 walkers 682 us in 128-row tiles, 547 us in 32-row tiles; 14 electrons
  // x 16 walkers 751 and 696 us.  At any size below the separate launches' times
  // (7 to 42 electrons, 1 to 768 walkers).
  const bool few = a.units <= kCus;
  switch (Rp) {
    case 128: return launch_chain<8, 8>(a, s);
    case 96: return launch_chain<6, 6>(a, s);
    case 64: return few ? launch_chain<4, 4>(a, s) : launch_chain<8, 4>(a, s);
    case 48: return few ? launch_chain<3, 3>(a, s) : launch_chain<6, 3>(a, s);
    case 32: return few ? launch_chain<2, 2>(a, s) : launch_chain<8, 2>(a, s);
  }
  return -1;
}
