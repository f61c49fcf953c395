// fp32 products on the bf16 matrix cores: every fp32 operand is taken apart into three bf16 values
// x = h + m + l (8 + 8 + 8 significant bits, each rounded to nearest even, so the sum is x itself),
// and a product is six of the nine partial products, a.l*b.h + a.h*b.l + a.m*b.m + a.m*b.h +
// a.h*b.m + a.h*b.h, accumulated in fp32. The three that are left out are below 2^-25 of |a*b|
// together, under the rounding of the fp32 accumulation itself. Relative 2-norm errors of a dot of
// K normal values against 64 bits, the fp32 MFMA first: K 48 1.24e-7 / 0.83e-7, K 384 3.6e-7 /
// 2.7e-7, K 1536 6.8e-7 / 6.0e-7, K 4096 1.12e-6 / 1.05e-6 (one 16-deep MFMA rounds once where the
// 2-deep fp32 MFMA rounds eight times). Exponents are bf16's, that is fp32's: only below about
// 2^-110 does the low part run out of range (an absolute error of 2^-134 times the other operand).
//
// Why: v_mfma_f32_32x32x2_f32 runs at 154 TFLOP/s here and the VALU stands still beside it;
// v_mfma_f32_32x32x16_bf16 runs at 2300 with up to six VALU instructions per MFMA for free, so six
// products are 2.5 times the fp32 rate and the operands' splitting hides beneath them.
//
// Operands or sums that are not finite (and values above 2^128 - 2^119, which bf16 rounds to
// infinity) turn into NaN parts: kernels check their accumulators and compute such a tile again
// with fp32 products, so infinities and NaN come out as they always did.
#pragma once

#include "device_utils.hpp"

namespace mnn {
namespace dev {

struct Split8 {
  bf16x8 h, m, l;
};

// Parts of eight consecutive values. The conversions are written as the instruction on purpose:
// from C++ the compiler converts each value once more on its own (5 conversions a pair, not 3).
__device__ __forceinline__ unsigned cvt_pk_bf16(float a, float b) {
  unsigned r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ Split8 split8(const float4& a, const float4& b) {
  const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  unsigned h[4], m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    h[i] = cvt_pk_bf16(x[2 * i], x[2 * i + 1]);
    const float r0 = x[2 * i] - __builtin_bit_cast(float, h[i] << 16);
    const float r1 = x[2 * i + 1] - __builtin_bit_cast(float, h[i] & 0xffff0000u);
    m[i] = cvt_pk_bf16(r0, r1);
    l[i] = cvt_pk_bf16(r0 - __builtin_bit_cast(float, m[i] << 16),
                       r1 - __builtin_bit_cast(float, m[i] & 0xffff0000u));
  }
  typedef unsigned uint4v __attribute__((ext_vector_type(4)));
  Split8 s;
  s.h = __builtin_bit_cast(bf16x8, (uint4v){h[0], h[1], h[2], h[3]});
  s.m = __builtin_bit_cast(bf16x8, (uint4v){m[0], m[1], m[2], m[3]});
  s.l = __builtin_bit_cast(bf16x8, (uint4v){l[0], l[1], l[2], l[3]});
  return s;
}

// Parts of eight consecutive values by truncation: bit operations at full rate, where the rounding
// conversion is not (44 against 54 cycles a pair). The parts sum to the value and share its sign, so
// one operand of a product may be truncated if the other is rounded: the dropped products then have
// no bias.
__device__ __forceinline__ Split8 split8_trunc(const float* x) {
  unsigned h[4], m[4], l[4];
  auto hi = [](float v) { return __builtin_bit_cast(unsigned, v) & 0xffff0000u; };
  auto pack = [](unsigned a, unsigned b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = x[2 * i], b = x[2 * i + 1];
    const float ra = a - __builtin_bit_cast(float, hi(a)), rb = b - __builtin_bit_cast(float, hi(b));
    const float sa = ra - __builtin_bit_cast(float, hi(ra)),
                sb = rb - __builtin_bit_cast(float, hi(rb));
    h[i] = pack(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b));
    m[i] = pack(__builtin_bit_cast(unsigned, ra), __builtin_bit_cast(unsigned, rb));
    l[i] = pack(__builtin_bit_cast(unsigned, sa), __builtin_bit_cast(unsigned, sb));
  }
  typedef unsigned uint4v __attribute__((ext_vector_type(4)));
  Split8 s;
  s.h = __builtin_bit_cast(bf16x8, (uint4v){h[0], h[1], h[2], h[3]});
  s.m = __builtin_bit_cast(bf16x8, (uint4v){m[0], m[1], m[2], m[3]});
  s.l = __builtin_bit_cast(bf16x8, (uint4v){l[0], l[1], l[2], l[3]});
  return s;
}

// Parts of a weight: as split8, but a value that bf16 would round to infinity keeps a truncated
// high part, so the three parts of every finite weight sum to it. An infinite weight (loaded ones are
// finite, a product with a LayerNorm's scale may overflow) is its high part alone.
__device__ __forceinline__ void split_weight(float x, __bf16& h, __bf16& m, __bf16& l) {
  h = (__bf16)x;
  if (__builtin_isinf((float)h))
    h = __builtin_bit_cast(__bf16, (unsigned short)(__builtin_bit_cast(unsigned, x) >> 16));
  const float r = __builtin_isinf(x) ? 0.f : x - (float)h;
  m = (__bf16)r;
  l = (__bf16)(r - (float)m);
}

// The p-th of the six partial products, small ones first.
__device__ __forceinline__ floatx16 mfma_x3(const Split8& a, const Split8& b, floatx16 c, int p) {
  const bf16x8& x = p == 0 ? a.l : (p == 2 || p == 3) ? a.m : a.h;
  const bf16x8& y = p == 1 ? b.l : (p == 2 || p == 4) ? b.m : b.h;
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, c, 0, 0, 0);
}

// Whether a value among the calling wave's accumulators is not finite.
template <int N, int M>
__device__ __forceinline__ bool any_not_finite(const floatx16 (&acc)[N][M]) {
  float t[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) t[v & 3] = fmaf(acc[i][j][v], 0.f, t[v & 3]);
  return __any(!((t[0] + t[1]) + (t[2] + t[3]) == 0.f));
}

}  // namespace dev
}  // namespace mnn
