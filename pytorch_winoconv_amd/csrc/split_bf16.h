#pragma once
#include "wc_common.h"

namespace wc {

// fp32 products of the Winograd domain on the bf16 matrix cores: x = h + m + l with three bf16 numbers of 8 bits each, h the
// upper half of x, m and l rounded to nearest, which together are x exactly, and x y = hh + hm + mh + mm + hl + lh, six of
// the nine products.  What is left out, ml + lm + ll, is at most 2^-22 and in the root mean square 2^-26 of the product, less
// than a rounding of fp32, and a sum of 16 products is rounded six times where eight v_mfma_f32_32x32x2_f32 round it eight.
// 16-bit products have 16 times the rate of fp32 ones.  Against fp64 in the 2-norm, fp32 | this (T=4, 2048 x 512): 32 channels 1.1e-7 |
// 7.2e-8, 8 channels 6.1e-8 | 3.8e-8, 4 channels 4.7e-8 | 3.9e-8, but a product that stands alone 2.5e-8 | 4.1e-8 (6e-8 | 2.9e-7 of it at
// most), as the instruction cuts its sums off: with ml and lm as well still 3.4e-8.
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
