// decode_common.hpp — device helpers shared by the decode step's kernels
// (decode.hip) and the prompt's (prefill.hip): the three-term bf16 split of
// an activation and the total order of logits.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mlxhip {
namespace dec {

constexpr int WAVE = 64;
constexpr int KSTEP = 32;   // k per MFMA
constexpr int TILE_N = 16;  // output features per MFMA tile

__device__ inline uint32_t bf16_rne(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return u >> 16;
}
__device__ inline float bf16_f32(uint32_t h) { return __uint_as_float(h << 16); }

// The hi / mid / lo bf16 terms of v: hi + mid + lo is v.
__device__ inline void split_terms(float v, uint16_t (&t)[3]) {
    const uint32_t h = bf16_rne(v);
    const float r1 = v - bf16_f32(h);
    const uint32_t m = bf16_rne(r1);
    const float r2 = r1 - bf16_f32(m);
    t[0] = (uint16_t)h;
    t[1] = (uint16_t)m;
    t[2] = (uint16_t)bf16_rne(r2);
}

// Total order of finite floats as unsigned integers, larger value = larger key.
__device__ inline uint32_t order_key(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// A logit's key: the larger logit, then the lower index, has the larger key.
__device__ inline uint64_t logit_key(float v, int n) {
    return ((uint64_t)order_key(v) << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)n);
}

__device__ inline uint64_t max_u64(uint64_t a, uint64_t b) { return a > b ? a : b; }

__device__ inline uint64_t shfl_xor_u64(uint64_t v, int o) {
    const uint32_t lo = __shfl_xor((uint32_t)v, o, WAVE);
    const uint32_t hi = __shfl_xor((uint32_t)(v >> 32), o, WAVE);
    return ((uint64_t)hi << 32) | lo;
}

// v[w] of (v0, v1, v2, v3) by value selects on the bits of w (0 <= w < 4).
__device__ inline float pick4(int w, float v0, float v1, float v2, float v3) {
    const float lo = (w & 1) ? v1 : v0;
    const float hi = (w & 1) ? v3 : v2;
    return (w & 2) ? hi : lo;
}

}  // namespace dec
}  // namespace mlxhip
