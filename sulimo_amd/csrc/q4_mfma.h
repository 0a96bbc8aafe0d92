// q4_mfma.h - device helpers the Q4_0 GEMM kernels share: buffer descriptors and
// global -> LDS DMA, the nibble dequantization, waits, and lane-quad transposes.
#pragma once

#include <type_traits>
#include <utility>

#include "common.h"

namespace sulimo {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __amdgpu_buffer_rsrc_t rsrc_t;

constexpr int kBK = 64;                   // k per stage
constexpr uint32_t kOob = 0x80000000u;    // buffer offset past every buffer: reads as zero
constexpr uint32_t kRsrcWord3 = 0x00020000u;  // raw buffer, 32-bit data format (gfx9)
constexpr int kXcds = 8;                      // XCDs of an MI355X

template <int J>
using ic = std::integral_constant<int, J>;

template <typename F, int... J>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, J...>) {
  (f(ic<J>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

__device__ __forceinline__ half2v as_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, (int)kRsrcWord3);
}

// One buffer -> LDS DMA: active lane i writes 16 bytes at dst + 16*i.
__device__ __forceinline__ void dma16(rsrc_t r, void *dst, uint32_t voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)dst, 16, (int)voff, soff, 0, 0);
}

// Four nibbles, one per byte in bits [3:0] (HI = false) or [7:4] (HI = true) with the
// other bits clear -> two half2 of (q-8)*d.
template <bool HI>
__device__ __forceinline__ void dq4(uint32_t nib, half2v d2, half2v &a, half2v &b) {
  // bytes [n0, 0x64, n1, 0x64] -> half2(1024 + n0, 1024 + n1), exact
  const uint32_t p0 = __builtin_amdgcn_perm(0x64646464u, nib, 0x04010400u);
  const uint32_t p1 = __builtin_amdgcn_perm(0x64646464u, nib, 0x04030402u);
  if constexpr (HI) {  // 1024 + 16q: /16 - 72 = q - 8, one exact fma
    const half2v s = {(_Float16)0.0625f, (_Float16)0.0625f};
    const half2v o = {(_Float16)-72.0f, (_Float16)-72.0f};
    a = __builtin_elementwise_fma(as_h2(p0), s, o) * d2;
    b = __builtin_elementwise_fma(as_h2(p1), s, o) * d2;
  } else {
    const half2v o = {(_Float16)1032.0f, (_Float16)1032.0f};
    a = (as_h2(p0) - o) * d2;
    b = (as_h2(p1) - o) * d2;
  }
}

// The same four nibbles -> two half2 of q-8 (exact, unscaled).
template <bool HI>
__device__ __forceinline__ void dq4_raw(uint32_t nib, half2v &a, half2v &b) {
  const uint32_t p0 = __builtin_amdgcn_perm(0x64646464u, nib, 0x04010400u);
  const uint32_t p1 = __builtin_amdgcn_perm(0x64646464u, nib, 0x04030402u);
  if constexpr (HI) {
    const half2v s = {(_Float16)0.0625f, (_Float16)0.0625f};
    const half2v o = {(_Float16)-72.0f, (_Float16)-72.0f};
    a = __builtin_elementwise_fma(as_h2(p0), s, o);
    b = __builtin_elementwise_fma(as_h2(p1), s, o);
  } else {
    const half2v o = {(_Float16)1032.0f, (_Float16)1032.0f};
    a = as_h2(p0) - o;
    b = as_h2(p1) - o;
  }
}

// s_waitcnt vmcnt(n) with expcnt and lgkmcnt left unconstrained (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// Workgroup barrier that orders LDS accesses only: global loads and stores in flight
// stay in flight (__syncthreads also waits for those).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Lane exchanges within a quad of lanes (DPP quad_perm): partner lane j^1, j^2.
__device__ __forceinline__ uint32_t dpp_xor1(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t dpp_xor2(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t fu(float v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ float uf(uint32_t v) { return __builtin_bit_cast(float, v); }

// 4 x 4 transposes across a lane quad. Lane j of the quad holds rows 0..3 of column j;
// afterwards it holds row j, columns 0..3. Every lane of the quad must be active.
// f16: p = rows 0,1 and q = rows 2,3 (packed); returns columns 0,1 and 2,3 (packed).
__device__ __forceinline__ uint2 quad_t16(uint32_t p, uint32_t q, int j) {
  const uint32_t sel = (j & 1) ? 0x03020706u : 0x05040100u;
  const uint32_t x = __builtin_amdgcn_perm(dpp_xor1(p), p, sel);  // row j&1 (odd) or 0, columns pair of j
  const uint32_t y = __builtin_amdgcn_perm(dpp_xor1(q), q, sel);  // row 2 + (j&1)
  const uint32_t r = dpp_xor2((j & 2) ? x : y);
  return (j & 2) ? uint2{r, y} : uint2{x, r};
}
__device__ __forceinline__ float4 quad_t32(float a0, float a1, float a2, float a3, int j) {
  const bool odd = j & 1, h = j & 2;
  const float r1 = uf(dpp_xor1(fu(odd ? a0 : a1)));
  const float r2 = uf(dpp_xor1(fu(odd ? a2 : a3)));
  const float x0 = odd ? r1 : a0, x1 = odd ? a1 : r1;  // row j&1, the pair of columns holding j
  const float y0 = odd ? r2 : a2, y1 = odd ? a3 : r2;  // row 2 + (j&1)
  const float t0 = uf(dpp_xor2(fu(h ? x0 : y0))), t1 = uf(dpp_xor2(fu(h ? x1 : y1)));
  return h ? float4{t0, t1, y0, y1} : float4{x0, x1, t0, t1};
}
// Four consecutive K-split partials as f32, stored as f16 or f32.
template <bool F16>
__device__ __forceinline__ float4 load_part4(const float *part, size_t idx) {
  if constexpr (F16) {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    const h4 v = *reinterpret_cast<const h4 *>(reinterpret_cast<const _Float16 *>(part) + idx);
    return float4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
  } else {
    return *reinterpret_cast<const float4 *>(part + idx);
  }
}
__device__ __forceinline__ uint32_t pack_h2(float lo, float hi) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)lo) | ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)hi) << 16);
}

}  // namespace
}  // namespace sulimo
