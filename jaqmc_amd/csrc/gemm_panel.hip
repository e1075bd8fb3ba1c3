// Persistent FP16X3 layer GEMM on whole row panels (Laplacian mode).
//
// Bound by the FP16 matrix rate and the stores together.  gemm_kernel's workgroups
// stream their X tile chunk by chunk, once for every column block, one chunk ahead,
// and end with their stores, behind which other workgroups' loads wait: a launch
// takes about the sum of its products and its stores.  Here one workgroup per CU
// walks over row tiles: four producer waves keep the whole X panel of the next
// tile (BM rows, every k) in flight in their registers while eight consumer waves
// multiply the present one, which lies in LDS split into its two FP16 planes, once
// for all column blocks; nothing waits for a store.  Two barriers a tile: the
// consumers are done with the panel, and the producers have split the next one
// into it.
//   consumers: wave c owns columns 32 c .. 32 c + 31 of each 256-column block and
//     every row (two 16-column blocks, BM / 16 row blocks of accumulators), its
//     weight fragments one 32-k chunk ahead from L2;
//   producers: wave p owns rows p, p + 4, ...; a row's 256 first k are one load of
//     16 bytes per lane, so the power-of-two scale of a value or Laplacian row is
//     a wave maximum of registers, without gemm_kernel's scan.
// Products, scales and the epilogue are gemm_kernel's in its order; the results
// are the same bit for bit.
// Measured at 1.23M rows, gemm_kernel -> here (us): 128-row units 1393 -> 1211 (512
// columns), 1935 -> 1590 (672), 2056 -> 1657 (768: 0.87 PFLOP/s issued and 3.0 TB/s);
// 48-row units 2137 -> 1772, 96-row units 2149 -> 1746 (768).  Splitting the next
// panel while the consumers still multiply spilled and was no faster.
#include <type_traits>

#include "kernels.h"

namespace {

constexpr int kConsumers = 8, kProducers = 4, kThreads = 64 * (kConsumers + kProducers);
constexpr float kJScale = 64.f;  // fixed scale of Jacobian rows (gemm_impl.h)
constexpr int kCus = 256;
constexpr int kK = 256;          // k of every launch
constexpr int kStride = 36;      // floats between staged output rows of 32

// MB: 16-row blocks of a panel; MBU: of a unit
template <int MB>
constexpr int panel_lds() {
  return 2 * 16 * MB * (kK + 8) * 2 + kConsumers * 16 * kStride * 4 + 2 * 16 * MB * 4;
}

template <int MB, int MBU>
__global__ __launch_bounds__(kThreads, 3) void panel_kernel(const GemmArgs a, int tiles_per_batch, int tiles) {
  constexpr int BM = 16 * MB, RU = 16 * MBU, UPT = MB / MBU, LS = kK + 8, NK = kK / 32;
  static_assert(MB % MBU == 0, "whole units");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  f16* const P0 = (f16*)smem;  // high plane, then the low plane
  f16* const P1 = P0 + BM * LS;
  float* const stage = (float*)(P1 + BM * LS);
  float* const rsc = stage + kConsumers * 16 * kStride;  // row scales and their inverses
  float* const rsi = rsc + BM;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // XCD x = b % 8 takes a contiguous range of tiles, its workgroups neighbours
  const int tpx = (tiles + kXcds - 1) / kXcds;
  const int t0 = (int)(blockIdx.x % kXcds) * tpx, t1 = t0 + tpx < tiles ? t0 + tpx : tiles;
  const int slot = (int)blockIdx.x / kXcds, step = (int)gridDim.x / kXcds;

  if (wave >= kConsumers) {
    // ---- producers ----
    const int p = wave - kConsumers;
    constexpr int NJ = BM / 4;                  // rows of this wave: p + 4 j
    f32x4 x[NJ];
    auto load = [&](int t) __attribute__((always_inline)) {
      const int z = t / tiles_per_batch;
      const long row0 = (long)(t - z * tiles_per_batch) * BM;
      const float* X = (const float*)a.X + (long)z * a.sxb;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const long r = row0 + p + 4 * j;
        x[j] = *(const f32x4*)(X + (r < a.rows ? r : (long)a.rows - 1) * a.ldx + 4 * lane);
      }
    };
    int t = t0 + slot;
    if (t < t1) load(t);
    for (; t < t1; t += step) {
      lds_barrier();  // the panel is free
      float sk = kJScale, ik = 1.f / kJScale;  // lane j keeps the scales of row p + 4 j
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        float sc = kJScale;
        if (j % (4 * MBU) == 0 && p < 2) {  // a value or Laplacian row, scaled to [2^13, 2^14)
          const f32x4 v = x[j];
          const float mx = wave_max(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
          float si = 1.f;
          sc = 1.f;
          if (mx > 0.f && mx <= 3.0e38f) {
            int e;
            (void)frexpf(mx, &e);
            int sh = 14 - e;
            sh = sh < -60 ? -60 : (sh > 60 ? 60 : sh);
            sc = ldexpf(1.f, sh);
            si = ldexpf(1.f, -sh);
          }
          if (lane == j) {
            sk = sc;
            ik = si;
          }
        }
        f16 h[4], l[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y = x[j][e] * sc;
          h[e] = (f16)y;
          l[e] = (f16)(y - (float)h[e]);
        }
        const int at = (p + 4 * j) * LS + 4 * lane;
        *(uint2*)(P0 + at) = *(const uint2*)h;
        *(uint2*)(P1 + at) = *(const uint2*)l;
      }
      if (lane < NJ) {
        rsc[p + 4 * lane] = sk;
        rsi[p + 4 * lane] = ik;
      }
      lds_barrier();  // the panel is ready
      if (t + step < t1) load(t + step);
    }
    return;
  }

  // ---- consumers ----
  const int lr = lane & 15, lg = lane >> 4;
  const f16* Wb = (const f16*)((const bf16*)a.Wt_lo + 3 * a.wplane);
  const float* csinv = (const float*)(Wb + 2 * a.wplane);
  const int ncb = (a.ncols - wave * 32 + 255) / 256;  // 256-column blocks with columns of this wave
  uint4 b[2][2][2];  // [set][plane][column block]
  auto bload = [&](auto set, int cb, int it) __attribute__((always_inline)) {
    constexpr int S = decltype(set)::value;
    const int k0 = it * 32;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const int gc = cb * 256 + wave * 32 + nb * 16 + lr;
      const f16* wp = Wb + (long)(gc < a.ncols ? gc : 0) * a.ldw + k0 + 8 * lg;
#pragma unroll
      for (int s = 0; s < 2; ++s) b[S][s][nb] = *(const uint4*)(wp + s * a.wplane);
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  float* const stg = stage + wave * 16 * kStride;
  f32x4 acc[MB][2];
  auto products = [&](auto set, int it) __attribute__((always_inline)) {
    constexpr int S = decltype(set)::value;
    const int k0 = it * 32;
    const f16* ap = P0 + lr * LS + k0 + 8 * lg;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const f16x8 a0 = *(const f16x8*)(ap + 16 * mb * LS), a1 = *(const f16x8*)(ap + (16 * mb + BM) * LS);
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        const f16x8 b0 = __builtin_bit_cast(f16x8, b[S][0][nb]), b1 = __builtin_bit_cast(f16x8, b[S][1][nb]);
        acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, b0, acc[mb][nb], 0, 0, 0);  // small terms first
        acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, b1, acc[mb][nb], 0, 0, 0);
        acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, b0, acc[mb][nb], 0, 0, 0);
      }
    }
  };
  bload(S0{}, 0, 0);
  for (int t = t0 + slot; t < t1; t += step) {
    lds_barrier();  // every consumer is done with the panel
    lds_barrier();  // the producers have filled it
    const int z = t / tiles_per_batch;
    const long row0 = (long)(t - z * tiles_per_batch) * BM;
    for (int cb = 0; cb < ncb; ++cb) {
      int ncol[2];
      bool cok[2];
      float csi[2];
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        ncol[nb] = cb * 256 + wave * 32 + nb * 16 + lr;
        cok[nb] = ncol[nb] < a.ncols;
        csi[nb] = cok[nb] ? csinv[ncol[nb]] : 1.f;
      }
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      const int cbn = cb + 1 < ncb ? cb + 1 : 0;
#pragma unroll 1
      for (int it = 0; it < NK; it += 2) {
        bload(S1{}, cb, it + 1);
        products(S0{}, it);
        const bool more = it + 2 < NK;
        bload(S0{}, more ? cb : cbn, more ? it + 2 : 0);
        products(S1{}, it + 1);
      }
      // remove the power-of-two row and column scales
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float ir = rsi[mb * 16 + 4 * lg + v];
#pragma unroll
          for (int nb = 0; nb < 2; ++nb) acc[mb][nb][v] *= ir * csi[nb];
        }
      if (a.bias) {  // on the value rows
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          const float bv = (cok[nb] && lg == 0) ? a.bias[cok[nb] ? ncol[nb] : 0] : 0.f;
#pragma unroll
          for (int u = 0; u < UPT; ++u) acc[u * MBU][nb][ROW_VAL] += bv;
        }
      }
      // store: 16 rows of 32 columns at a time through the wave's
      // slice of LDS, 8 lanes per row
      const int c4 = (lane & 7) * 4, rl = lane >> 3, n = cb * 256 + wave * 32 + c4;
      const bool nok = n < a.ncols;
      float* Y = (float*)a.Y + (long)z * a.syb;
      long hcol = 0;
      int hw0 = 0, hi0 = 0;
      if (a.hs_H > 0) {
        const int part = n / a.hs_D, hh = (n % a.hs_D) / a.hs_dh, dd = n % a.hs_dh;
        hcol = ((long)part * a.hs_H + hh) * a.hs_N * ((long)RU * a.hs_dh) + dd;
        const int u0 = (int)(row0 / RU);
        hw0 = u0 / a.hs_N;
        hi0 = u0 % a.hs_N;
      }
#pragma unroll 1
      for (int mb0 = 0; mb0 < MB; ++mb0) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          if (mb == mb0) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
              for (int v = 0; v < 4; ++v) stg[(4 * lg + v) * kStride + nb * 16 + lr] = acc[mb][nb][v];
          }
        wave_sync();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int r = rl + 8 * i;
          const long grow = row0 + mb0 * 16 + r;
          if (grow >= a.rows || !nok) continue;
          const f32x4 y = *(const f32x4*)&stg[r * kStride + c4];
          float* dst;
          if (a.hs_H > 0) {
            int w = hw0, e = hi0 + (mb0 * 16 + r) / RU;
            while (e >= a.hs_N) {
              e -= a.hs_N;
              ++w;
            }
            dst = Y + ((((long)w * 3 * a.hs_H) * a.hs_N + e) * RU + (mb0 * 16 + r) % RU) * (long)a.hs_dh + hcol;
          } else {
            dst = Y + grow * a.ldy + n;
          }
          *(f32x4*)dst = y;
        }
        wave_sync();
      }
    }
  }
}

template <int MB, int MBU>
int launch_panel(const GemmArgs& a, hipStream_t s) {
  constexpr int lds = panel_lds<MB>();
  static_assert(lds <= 160 * 1024, "one workgroup per CU");
  static const hipError_t attr = hipFuncSetAttribute((const void*)panel_kernel<MB, MBU>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return -1;
  const long per = ceil_div(a.rows, 16 * MB), tiles = per * (a.nbatch > 1 ? a.nbatch : 1);
  if (tiles > 0x7FFFFFFFL) return -1;
  hipLaunchKernelGGL((panel_kernel<MB, MBU>), dim3(kCus), dim3(kThreads), lds, s, a, (int)per, (int)tiles);
  return 0;
}

}  // namespace

// Takes a projection (no activation, broadcast term or residual) of 256 k onto
// more columns than one block, with 16-byte rows and stores, of 48-, 96- and
// 128-row units (the panel of 192 rows does not fit LDS; 16-, 32- and 64-row units
// stay with gemm_kernel, not measured here).  Both sides measured: the panel is
// split once for all column blocks, which wins from the second on (1.23M rows of
// 128-row units: 1239 -> 1019 us at 320 columns) and loses with only one (733 -> 854
// us at 256, 657 -> 791 at 224); and the last round of tiles idles the fewer CUs the
// more tiles each has (768 columns: 264 -> 225 us at 4.5 tiles per CU).
bool gemm_panel_ok(const GemmArgs& a) {
  const int bm = a.R == 128 ? 128 : (a.R == 48 || a.R == 96 ? 96 : 0);
  if (bm == 0 || a.K != kK || a.ncols <= 256 || a.act != ACT_NONE || a.G || a.Res || a.Yln || a.rgrp > 0 || a.linear_tiles)
    return false;
  if (a.ncols % 4 || a.zpad > a.ncols || a.ldx % 4 || a.sxb % 4 || a.ldy % 4 || a.syb % 4 || (a.hs_H > 0 && a.hs_dh % 4))
    return false;
  return (long)ceil_div(a.rows, bm) * (a.nbatch > 1 ? a.nbatch : 1) >= 4L * kCus;
}

int gemm_panel(const GemmArgs& a, hipStream_t s) {
  if (a.R == 128) return launch_panel<8, 8>(a, s);
  return a.R == 48 ? launch_panel<6, 3>(a, s) : launch_panel<6, 6>(a, s);
}
