// fp32 products on the bf16 matrix cores: every fp32 operand is taken apart into three bf16 values
// x = h + m + l (8 + 8 + 8 significant bits, each rounded to nearest even, so the sum is x itself),
// and a product is six of the nine partial products, accumulated in fp32: a.l*b.h, a.h*b.l, a.m*b.m,
// a.m*b.h, a.h*b.m, and a.h*b.h. |m| <= 2^-8 |x| and |l| <= 2^-17 |x|, so the three that are left
// out (m*l, l*m, l*l) are at most 1.001 * 2^-24 |a*b| together, one fp32 rounding (rms 2^-27.4). The
// matrix instruction rounds its sums to 1.5 * 2^-24 (measured on single products; an fp32 one to
// 2^-24). The GEMM and the scores give a.h*b.h an accumulator of its own, and the small products, which would
// each be rounded to the large ones' last bits, another; the two are added at the end.
// Errors against 64 bits, the fp32 MFMA first: 2-norm of a dot of K normal values, K 32 1.04e-7 /
// 0.39e-7, K 384 3.5e-7 / 0.83e-7, K 1536 7.0e-7 / 1.6e-7, K 4096 1.14e-6 / 0.27e-6; a single product rms
// 0.42 / 0.44 and at most 1.0 / 1.7 (of 10^6) times 2^-24.
// Exponents are bf16's, that is fp32's: only below about 2^-110 does the low part run out of range
// (an absolute error below 2^-133).
//
// Why: v_mfma_f32_32x32x2_f32 runs at 154 TFLOP/s here and the VALU stands still beside it;
// v_mfma_f32_32x32x16_bf16 runs at 2300 with up to six VALU instructions per MFMA for free, so six
// products are 2.5 times the fp32 rate and the splitting of an operand hides beneath them where a wave uses
// each part in four MFMAs (128-wide tiles; a 64x64 tile splits 7 to 9 instructions per MFMA and is bound by it).
//
// Operands or sums that are not finite (and values above 2^128 - 2^119, which bf16 rounds to
// infinity) turn into NaN parts, sums of tiny operands are tiny: kernels check their accumulators and
// compute such a tile again with fp32 products, so infinities and NaN come out as they always did and
// activations below 2^-110 keep their bits. (A weight is its parts, 2^-134 at the finest.)
#pragma once

#include "device_utils.hpp"

namespace mnn {
namespace dev {

struct Split8 {
  bf16x8 h, m, l;
};

// Parts of eight consecutive values: 11 instructions a pair, whose two conversions run at about half
// rate (50 cycles; by truncation alone 44, but the dropped products are then up to three times as large,
// 2^-22.5). After two rounded parts at most 7 bits are left: the low part needs no rounding. The rounded
// parts are read back by byte permutes: from shifts, masks or casts the compiler sees a conversion of one
// value and converts each of the pair once more on its own. (Conversions in inline asm are no way out: the
// compiler knows no hazards there, and probabilities fresh from v_exp_f32 were read too early.)
__device__ __forceinline__ unsigned cvt_pk_bf16(float a, float b) {
  typedef float float2v __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, __builtin_convertvector((float2v){a, b}, bf16x2));
}
__device__ __forceinline__ Split8 split8(const float* x) {
  unsigned h[4], m[4], l[4];
  auto bits = [](float v) { return __builtin_bit_cast(unsigned, v); };
  auto lo = [](unsigned p) {
    return __builtin_bit_cast(float, __builtin_amdgcn_perm(0u, p, 0x01000c0cu));
  };
  auto hi = [](unsigned p) {
    return __builtin_bit_cast(float, __builtin_amdgcn_perm(0u, p, 0x03020c0cu));
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    h[i] = cvt_pk_bf16(x[2 * i], x[2 * i + 1]);
    const float r0 = x[2 * i] - lo(h[i]), r1 = x[2 * i + 1] - hi(h[i]);
    m[i] = cvt_pk_bf16(r0, r1);
    l[i] = __builtin_amdgcn_perm(bits(r1 - hi(m[i])), bits(r0 - lo(m[i])), 0x07060302u);
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

// Sums below this (and not zero) are computed again in fp32: an operand whose low part is out of bf16's
// range is off by less than 2^-133, so larger sums are off by a relative 2^-24 at most as long as the other
// operand's values add up to less than 2^23.
constexpr float kTinySum = 0x1p-86f;

// Whether a value among the calling wave's accumulators is not finite or tiny: their largest and smallest
// magnitude first (half an instruction each a value; maximum keeps NaN). With none below the limit, zeros
// included, there is nothing more to look at.
template <int N, int M>
__device__ __forceinline__ bool any_out_of_range(const floatx16 (&acc)[N][M]) {
  float hi[2] = {1.f, 1.f}, lo[2] = {1.f, 1.f};
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < M; ++j)
#pragma unroll
      for (int v = 0; v < 16; v += 2) {
        const float a = fabsf(acc[i][j][v]), b = fabsf(acc[i][j][v + 1]);
        float &h = hi[(v >> 1) & 1], &l = lo[(v >> 1) & 1];
        h = __builtin_elementwise_maximum(__builtin_elementwise_maximum(h, a), b);
        l = fminf(fminf(l, a), b);
      }
  bool out = !(__builtin_elementwise_maximum(hi[0], hi[1]) < __builtin_inff());
  if (__any(fminf(lo[0], lo[1]) < kTinySum)) {
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int j = 0; j < M; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          out |= (acc[i][j][v] != 0.f) & (fabsf(acc[i][j][v]) < kTinySum);
  }
  return __any(out);
}

}  // namespace dev
}  // namespace mnn
