// Shared by the split-x products (eff_gemm_sx.hip, eff_gemm_sxt.hip): the
// prepared x's slots and the exact fp16 weight decoders.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "eff_device.h"

namespace eff {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// Types with group minima (their group sums of x form a 17th slot)
template <int TYPE>
constexpr bool sx_mins() {
  return TYPE == Q2_K || TYPE == Q4_K;
}

template <int TYPE>
constexpr uint32_t sx_slots() {  // x slots of 1 KB per (token tile, block): 16 steps (+ group sums)
  return sx_mins<TYPE>() ? 17u : 16u;
}

// 4 bytes b (each < 1024 after the caller's masking) -> 1024 + b as fp16 pairs
__device__ __forceinline__ half2v h1024_lo(uint32_t v) {
  return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u));
}
__device__ __forceinline__ half2v h1024_hi(uint32_t v) {
  return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u));
}

// 8 unsigned bytes q (v0: q0..q3, v1: q4..q7) -> sc * q as fp16, exact
// (sc * q < 2048; the fused multiply-add rounds once: (1024 + q) sc - 1024 sc)
__device__ __forceinline__ half8 dec_scaled(uint32_t v0, uint32_t v1, uint32_t sc) {
  const _Float16 s = (_Float16)(float)sc, o = (_Float16)(-1024.f * (float)sc);
  const half2v s2 = {s, s}, o2 = {o, o};
  const half2v a = __builtin_elementwise_fma(h1024_lo(v0), s2, o2);
  const half2v b = __builtin_elementwise_fma(h1024_hi(v0), s2, o2);
  const half2v c = __builtin_elementwise_fma(h1024_lo(v1), s2, o2);
  const half2v d = __builtin_elementwise_fma(h1024_hi(v1), s2, o2);
  return half8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}

// 8 unsigned bytes -> fp16 (exact below 1024)
__device__ __forceinline__ half8 dec_plain(uint32_t v0, uint32_t v1) {
  const half2v o2 = {(_Float16)-1024.f, (_Float16)-1024.f};
  const half2v a = h1024_lo(v0) + o2, b = h1024_hi(v0) + o2, c = h1024_lo(v1) + o2, d = h1024_hi(v1) + o2;
  return half8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}

__device__ __forceinline__ uint32_t byte_of(const uint32_t *w, uint32_t i) { return (w[i >> 2] >> (8u * (i & 3u))) & 0xFFu; }

// 8 signed bytes q -> q as fp16 (exact): 1024 + (q + 128) - 1152
__device__ __forceinline__ half8 dec_signed(uint32_t v0, uint32_t v1) {
  const half2v o2 = {(_Float16)-1152.f, (_Float16)-1152.f};
  v0 ^= 0x80808080u;
  v1 ^= 0x80808080u;
  const half2v a = h1024_lo(v0) + o2, b = h1024_hi(v0) + o2, c = h1024_lo(v1) + o2, d = h1024_hi(v1) + o2;
  return half8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}

}  // namespace eff
