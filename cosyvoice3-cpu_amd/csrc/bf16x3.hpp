// Three-plane bfloat16 form of float32 values: x = hi + mid + lo, each plane the
// round-to-nearest bfloat16 of what the planes before it leave.  Each residual is
// exact in float32 (x minus a rounding of x to fewer bits), so |x - (hi + mid + lo)|
// <= 2^-8 |x - hi - mid| <= 2^-24 |x|: the planes carry all 24 bits of the float, from 2^-110 up.
// Below, the last bits fall under the smallest bfloat16 and |x - (hi + mid + lo)| <= 2^-134 instead:
// 2e-6 of a value of 2^-116, 4e-5 of one of 2^-120 (the matrix cores keep subnormal operands).
// ops.linear and ops.sdpa form such outputs again in float32; the models' own layers do not.
// A product a.b is then the six plane products whose weights reach 2^-16
// (hh, hm, mh, hl, mm, lh), each exact in the matrix core's float32 accumulate;
// the three dropped (ml, lm, ll) weigh at most ~2^-23 |a b|.
#pragma once

#include "common.hpp"

namespace cv3 {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// Two floats -> their hi, mid and lo planes, two bfloat16 per 32-bit word (a in the
// low half).  v_cvt_pk_bf16_f32 rounds to nearest even.
__device__ __forceinline__ void split_x3(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  const f32x2_t x = {a, b};
  const bf16x2_t h = __builtin_convertvector(x, bf16x2_t);
  const f32x2_t r1 = x - __builtin_convertvector(h, f32x2_t);
  const bf16x2_t m = __builtin_convertvector(r1, bf16x2_t);
  const f32x2_t r2 = r1 - __builtin_convertvector(m, f32x2_t);
  const bf16x2_t l = __builtin_convertvector(r2, bf16x2_t);
  hi = __builtin_bit_cast(uint32_t, h);
  mid = __builtin_bit_cast(uint32_t, m);
  lo = __builtin_bit_cast(uint32_t, l);
}

// Eight floats (two float4) -> one 16-byte word of each plane.
__device__ __forceinline__ void split_x3(const float4& a, const float4& b, uint4& hi, uint4& mid, uint4& lo) {
  split_x3(a.x, a.y, hi.x, mid.x, lo.x);
  split_x3(a.z, a.w, hi.y, mid.y, lo.y);
  split_x3(b.x, b.y, hi.z, mid.z, lo.z);
  split_x3(b.z, b.w, hi.w, mid.w, lo.w);
}

// The same planes for a weight or a linear's rows, whose largest values count too: past the largest bfloat16 (3.39e38)
// the rounding above is an infinity, and x - inf loses the value.  Here hi stays at that largest and mid and lo hold
// the rest, exact as everywhere; an infinity is (inf, 0, 0), so that lo + mid + hi, summed in this order, is x.
__device__ __forceinline__ void split_x3_full(float a, uint16_t& hi, uint16_t& mid, uint16_t& lo) {
  const float top = 3.3895313892515355e38f;
  const bool finite = fabsf(a) <= 3.4028234663852886e38f;
  const __bf16 h = (__bf16)(finite ? fminf(fmaxf(a, -top), top) : a);
  const float r1 = finite ? a - (float)h : 0.f;
  const __bf16 m = (__bf16)r1;
  const __bf16 l = (__bf16)(r1 - (float)m);
  hi = __builtin_bit_cast(uint16_t, h);
  mid = __builtin_bit_cast(uint16_t, m);
  lo = __builtin_bit_cast(uint16_t, l);
}

__device__ __forceinline__ void split_x3_full(const float4& a, const float4& b, uint4& hi, uint4& mid, uint4& lo) {
  const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  uint32_t *h = &hi.x, *m = &mid.x, *l = &lo.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint16_t p[2][3];
    split_x3_full(v[2 * i], p[0][0], p[0][1], p[0][2]);
    split_x3_full(v[2 * i + 1], p[1][0], p[1][1], p[1][2]);
    h[i] = p[0][0] | (uint32_t)p[1][0] << 16;
    m[i] = p[0][1] | (uint32_t)p[1][1] << 16;
    l[i] = p[0][2] | (uint32_t)p[1][2] << 16;
  }
}

// Whether outputs of one row are what planes give in full: all finite, and all zero or one of 2^-90 or more.
__device__ __forceinline__ bool in_range(uint32_t largest) {
  const uint32_t low = (127u - 90u) << 23;
  return largest == 0 || largest - low <= 0x7f7fffffu - low;
}
__device__ __forceinline__ uint32_t magnitude(float v) { return __float_as_uint(v) & 0x7fffffffu; }
__device__ __forceinline__ bool in_range(const float4& v) {
  return in_range(max(max(magnitude(v.x), magnitude(v.y)), max(magnitude(v.z), magnitude(v.w))));
}

// Scheduling groups: R times, N1 instructions of class M1, then N2 of class M2 (0x8 MFMA, 0x20 VMEM read,
// 0x100 LDS read).
template <int M, int N>
__device__ __forceinline__ void sched_n() {
  if constexpr (N > 0) __builtin_amdgcn_sched_group_barrier(M, N, 0);
}
template <int M1, int N1, int M2, int N2, int R>
__device__ __forceinline__ void interleave() {
  if constexpr (R > 0) {
    sched_n<M1, N1>();
    sched_n<M2, N2>();
    interleave<M1, N1, M2, N2, R - 1>();
  }
}

// 16 bytes per lane, global -> LDS.  (A function of its own: called inside a kernel template's lambda the
// builtin makes clang drop the kernel's host stub.)
__device__ __forceinline__ void dma16(const uint4* g, uint4* l) { __builtin_amdgcn_global_load_lds(g, l, 16, 0, 0); }

typedef float f32x16_t __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f32x16_t mfma_bf16(const uint4& a, const uint4& b, const f32x16_t& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                 0, 0, 0);
}

}  // namespace cv3

// s_waitcnt for at most n vector-memory operations in flight (loads complete in order), others untouched.
#define CV3_VM(n) (((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))
