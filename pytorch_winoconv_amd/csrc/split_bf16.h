#pragma once
#include "wc_common.h"

namespace wc {

// fp32 products of the Winograd domain on the bf16 matrix cores: x = h + m + l with three bf16 numbers of 8 bits each, h the
// upper half of x, m and l rounded to nearest, which together are x exactly, and x y = hh + hm + mh + mm + hl + lh, six of
// the nine products.  What is left out, ml + lm + ll, is at most 2^-22 and in the root mean square 2^-26 of the product, less
// than a rounding of fp32, and a sum of 16 products is rounded six times where eight v_mfma_f32_32x32x2_f32 round it eight.
// 16-bit products have 16 times the rate of fp32 ones.
// They cut their sums off, though, where the fp32 instructions round them.  Against fp64 in the 2-norm, fp32 | this (T=4, 1024 x 256 normal
// numbers): one channel 2.5e-8 | 4.1e-8 (with ml and lm as well still 3.4e-8), 4 channels 4.0e-8 | 3.9e-8, 32 1.0e-7 | 7.2e-8, 512 4.1e-7 | 3.4e-7, 4096
// 1.1e-6 | 1.0e-6; half of V zeros, whose products are not rounded: 32 7.5e-8 | 7.1e-8, 128 1.4e-7 | 1.6e-7; sums of one sign: 512 3.5e-7 | 2.9e-7,
// 2048 7.0e-7 | 1.2e-6, 4096 9.9e-7 | 3.2e-6.  So the parts are for sums of some to a thousand products of transformed operands
// (fp32_in_parts in gemm.hip; wc_conv_backward_weight, whose kernel adds up longer ones in fp32 outside of the instructions).
//
// h of an infinity is the infinity and m is no number, which it makes of every sum it enters.  The kernels take such sums again
// with fp32 products: a plan whose tile has one tap, or a caller of the product alone, gets the infinity and its sign.
typedef uint32_t SplitWords __attribute__((ext_vector_type(4)));
struct Split { uint32_t h[2], m[2], l[2]; };
__device__ __forceinline__ Split split_bf16(SplitWords c) {
  Split s;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t a = c[2 * i], b = c[2 * i + 1];
    s.h[i] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    const float ra = __uint_as_float(a) - __uint_as_float(a & 0xffff0000u), rb = __uint_as_float(b) - __uint_as_float(b & 0xffff0000u);
    const Pack<bf16_t, 2> m = {{static_cast<bf16_t>(ra), static_cast<bf16_t>(rb)}};
    s.m[i] = __builtin_bit_cast(uint32_t, m);
    const Pack<bf16_t, 2> l = {{static_cast<bf16_t>(ra - __uint_as_float(s.m[i] << 16)), static_cast<bf16_t>(rb - __uint_as_float(s.m[i] & 0xffff0000u))}};
    s.l[i] = __builtin_bit_cast(uint32_t, l);
  }
  return s;
}

}  // namespace wc
