// Device helpers of the recurrences in chunks of 16 tokens with decays per channel (chunk_delta.hip, chunk_channel.hip): fp32 operands of the
// bf16 matrix instructions in three parts, products of decays over the tokens around a lane's own.
#pragma once

#include "common.h"

namespace die {

namespace {

constexpr int CT = 16;        // tokens of a chunk
constexpr int TP = CT + 4;    // pitch of the 16-wide arrays (floats): 16-byte reads of 16 rows fall on different banks

__device__ __forceinline__ f32x4_t mm(float a, float b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ float dpp_ror8(float x) {   // of lane ^ 8
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, false));
}
__device__ __forceinline__ f32x4_t ld4(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }

// x - low (x - high) value of a packed pair, by the dot product with (-1, 0) or (0, -1) in one instruction. (The constants come from
// registers: as an immediate the instruction would take -1 for both halves.)
__device__ __forceinline__ uint32_t opaque(uint32_t c) {
  asm("" : "+s"(c));
  return c;
}
__device__ __forceinline__ float less(float x, uint32_t pair, uint32_t which) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pair), __builtin_bit_cast(bf16x2_t, which), x, false);
}
__device__ __forceinline__ uint32_t top2(float x, float y) {   // the upper halves of two values' bits
  return __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);
}
// x = h + m + l in bf16 parts, exact: twice 8 bits rounded to nearest, so that what is left has either sign (cut off, the products that are
// not formed would add up, 1 - 7 % of the error), then the rest. Pairs of values, packed. (A conversion takes the time of two other
// instructions.)
template <int N> __device__ __forceinline__ void split3(float (&x)[2 * N], uint32_t (&p)[3][N]) {
  const uint32_t lo = opaque(0x0000bf80u), hi = opaque(0xbf800000u);
  auto rest = [&](const uint32_t (&q)[N]) {
#pragma unroll
    for (int e = 0; e < N; ++e) x[2 * e] = less(x[2 * e], q[e], lo), x[2 * e + 1] = less(x[2 * e + 1], q[e], hi);
  };
#pragma unroll
  for (int e = 0; e < N; ++e) p[0][e] = pack2(x[2 * e], x[2 * e + 1]);
  rest(p[0]);
#pragma unroll
  for (int e = 0; e < N; ++e) p[1][e] = pack2(x[2 * e], x[2 * e + 1]);
  rest(p[1]);
#pragma unroll
  for (int e = 0; e < N; ++e) p[2][e] = top2(x[2 * e], x[2 * e + 1]);
}
__device__ __forceinline__ void split3(float x, float y, uint32_t (&p)[3]) {
  float v[2] = {x, y};
  uint32_t q[3][1];
  split3<1>(v, q);
#pragma unroll
  for (int i = 0; i < 3; ++i) p[i] = q[i][0];
}
// the same of products x a, y b, which are not rounded before they are cut (24 bits and the sign of what is left)
__device__ __forceinline__ void split3(float x, float a, float y, float b, uint32_t (&p)[3]) {
  const uint32_t lo = opaque(0x0000bf80u), hi = opaque(0xbf800000u);
  p[0] = pack2(x * a, y * b);
  const float u = fmaf(x, a, -__uint_as_float(p[0] << 16)), v = fmaf(y, b, -__uint_as_float(p[0] & 0xffff0000u));
  p[1] = pack2(u, v);
  p[2] = pack2(less(u, p[1], lo), less(v, p[1], hi));
}
// base (the same for all lanes) + a lane's offset in bytes: one scalar and one 32-bit address register
template <typename T> __device__ __forceinline__ const T* at_bytes(const void* base, uint32_t off) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
}
typedef float float2_at4 __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t uint32_at2 __attribute__((aligned(2)));
// 4 consecutive places of a contraction as operands of 8 places: (h, m) and (h, l)
__device__ __forceinline__ void split_store(char* to, const float* x, const float* y) {   // of products x y
  uint32_t a[3], b[3];
  split3(x[0], y[0], x[1], y[1], a);
  split3(x[2], y[2], x[3], y[3], b);
  *reinterpret_cast<uint4*>(to) = make_uint4(a[0], b[0], a[1], b[1]);
  *reinterpret_cast<uint4*>(to + 16) = make_uint4(a[0], b[0], a[2], b[2]);
}
__device__ __forceinline__ bf16x8_t ldf(const char* p) { return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(p)); }
__device__ __forceinline__ bf16x8_t frag(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return __builtin_bit_cast(bf16x8_t, make_uint4(a, b, c, d));
}
__device__ __forceinline__ f32x4_t mm(bf16x8_t a, bf16x8_t b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// A lane's 4 tokens are quarter lg = lane / 16 of a chunk; own: the product of their decays. The products over the quarters before and behind.
__device__ __forceinline__ void around(float own, int lg, float& before, float& behind) {
  const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(own), __float_as_uint(own), false, false);
  const float one = __uint_as_float(lg & 1 ? x[0] : x[1]);            // of the other quarter of the own half
  const float half = own * one;
  const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(half), __float_as_uint(half), false, false);
  const float two = __uint_as_float(lg & 2 ? y[0] : y[1]);            // of the other half
  before = (lg & 1 ? one : 1.0f) * (lg & 2 ? two : 1.0f);
  behind = (lg & 1 ? 1.0f : one) * (lg & 2 ? 1.0f : two);
}

}  // namespace

}  // namespace die
