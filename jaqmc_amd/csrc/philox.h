// The sampler's randomness: Philox-4x32-10 (Salmon et al., "Parallel random
// numbers: as easy as 1, 2, 3", SC'11) with key = seed and counter = (block
// index, walker, step low word, step high word ^ stream tag); normals by the
// Box-Muller transform.  Streams are keyed by (seed, step, walker, element),
// never by launch geometry, so a walker's trajectory does not depend on the
// batch it is evaluated in.
#pragma once

#include "common.h"

struct u32x4 {
  uint32_t x, y, z, w;
};

__device__ inline uint32_t mulhilo(uint32_t a, uint32_t b, uint32_t& hi) {
  const uint64_t p = (uint64_t)a * b;
  hi = (uint32_t)(p >> 32);
  return (uint32_t)p;
}

__device__ inline u32x4 philox4x32_10(u32x4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    uint32_t hi0, hi1;
    const uint32_t lo0 = mulhilo(0xD2511F53u, c.x, hi0);
    const uint32_t lo1 = mulhilo(0xCD9E8D57u, c.z, hi1);
    c = u32x4{hi1 ^ c.y ^ k0, lo1, hi0 ^ c.w ^ k1, lo0};
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return c;
}

// (0, 1], never 0 so log(u) is finite
__device__ inline float u01(uint32_t v) { return ((v >> 8) + 1u) * (1.0f / 16777216.0f); }

constexpr uint32_t TAG_NORMAL = 0u;
constexpr uint32_t TAG_UNIFORM = 0x80000000u;

// Normals 4 g .. 4 g + 3 of a walker's move.
__device__ inline void philox_normals(uint64_t seed, uint64_t step, uint32_t walker, uint32_t g, float (&z)[4]) {
  const u32x4 r = philox4x32_10(u32x4{g, walker, (uint32_t)step, (uint32_t)(step >> 32) ^ TAG_NORMAL}, (uint32_t)seed,
                                (uint32_t)(seed >> 32));
  const float u1 = u01(r.x), u2 = u01(r.y), u3 = u01(r.z), u4 = u01(r.w);
  const float m1 = sqrtf(-2.f * logf(u1)), m2 = sqrtf(-2.f * logf(u3));
  float s1, c1, s2, c2;
  sincospif(2.f * u2, &s1, &c1);
  sincospif(2.f * u4, &s2, &c2);
  z[0] = m1 * c1;
  z[1] = m1 * s1;
  z[2] = m2 * c2;
  z[3] = m2 * s2;
}

// The uniform of a walker's accept decision.
__device__ inline float philox_uniform(uint64_t seed, uint64_t step, uint32_t walker) {
  const u32x4 r = philox4x32_10(u32x4{0u, walker, (uint32_t)step, (uint32_t)(step >> 32) ^ TAG_UNIFORM}, (uint32_t)seed,
                                (uint32_t)(seed >> 32));
  return u01(r.x);
}
