// The tile of the row form (conv_row.hip, conv_row_tall.hip), F(4, 3) or F(2, 5): its points, the arithmetic of one channel,
// MFMA.
//
// Points of the tile: 0, +-a, +-1/a, infinity with a^2 = 0.425 instead of the customary 0, +-1, +-2.  They spread the
// rounding of U and V evenly: with independent roundings of relative size e in both, the output's is 3.1 e in the root
// mean square against 4.6 e with integer points, and against 2.4 e (products rounded to the storage type on top) for
// F(2x2, 3x3).  Measured over 64 channels, fp16: 6e-4 of the output in the 2-norm, as F(2x2, 3x3), and a sixth of
// F(4x4, 3x3)'s 3.7e-3.
#pragma once
#include "wc_transform.h"

namespace wc {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kA2 = 0.425f, kB2 = 1.0f / 0.425f;             // a^2 and 1 / a^2
constexpr float kA = 0.65192024f, kB = 1.0f / 0.65192024f;      // a (its square differs from kA2 by 5e-9)
constexpr float kS = kA2 + kB2;

template <typename T> struct MfmaRow;
template <> struct MfmaRow<half_t> {
  using Frag = f16x8;
  static __device__ __forceinline__ f32x16 run(Frag a, Frag b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};
template <> struct MfmaRow<bf16_t> {
  using Frag = bf16x8;
  static __device__ __forceinline__ f32x16 run(Frag a, Frag b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};

// d + f in fp32, rounded to T
__device__ __forceinline__ bf16_t plus(bf16_t d, float f) { return static_cast<bf16_t>(static_cast<float>(d) + f); }
__device__ __forceinline__ half_t plus(half_t d, float f) {
  float one = 1.0f;
  asm("" : "+s"(one));                  // d * 1 + f stays one v_fma_mix instead of a conversion, an addition and a conversion
  return static_cast<half_t>(__builtin_fmaf(static_cast<float>(d), one, f));
}

// channel e of two neighbouring ones: the six inputs of x become the six elements of the tile, in place
template <typename T>
__device__ __forceinline__ void row_input_channel(Pack<T, 2> (&x)[6], int e) {
  float d[6];
#pragma unroll
  for (int j = 0; j < 6; ++j) d[j] = static_cast<float>(x[j].v[e]);
  const float ea = __builtin_fmaf(-kB2, d[2], d[4]), oa = __builtin_fmaf(-kB2, d[1], d[3]);
  const float eb = __builtin_fmaf(-kA2, d[2], d[4]), ob = __builtin_fmaf(-kA2, d[1], d[3]);
  const float e0 = __builtin_fmaf(-kS, d[2], d[4]), o0 = __builtin_fmaf(-kS, d[3], d[5]);
  x[0].v[e] = plus(x[0].v[e], e0);
  x[5].v[e] = plus(x[1].v[e], o0);
  x[1].v[e] = static_cast<T>(__builtin_fmaf(kA, oa, ea));
  x[2].v[e] = static_cast<T>(__builtin_fmaf(-kA, oa, ea));
  x[3].v[e] = static_cast<T>(__builtin_fmaf(kB, ob, eb));
  x[4].v[e] = static_cast<T>(__builtin_fmaf(-kB, ob, eb));
}

// The pair of elements at +p and -p (p^2 = p2) of a row of five taps: three leave g3 and g4 zero.  Explicit, so that kernels
// that transform a filter for themselves find the numbers of those that do it for them
struct RowPair { float plus, minus; };
__device__ __forceinline__ RowPair row_filter_pair(float g0, float g1, float g2, float g3, float g4, float p, float p2, float f) {
  const float even = __builtin_fmaf(p2, __builtin_fmaf(p2, g4, g2), g0), odd = __builtin_fmaf(p2, g3, g1);
  RowPair o = {__builtin_fmaf(p, odd, even) * f, __builtin_fmaf(-p, odd, even) * f};
  asm("" : "+v"(o.plus), "+v"(o.minus));          // a product in fp32: not rounded to T within one instruction here and in two there
  return o;
}
// denominators: prod over the other points; 1 for 0 (a^2 b^2), 2 a^2 (a^2 - b^2) for +-a, 2 b^2 (b^2 - a^2) for +-b
constexpr float kRowFa = 1.f / (2.f * kA2 * (kA2 - kB2)), kRowFb = 1.f / (2.f * kB2 * (kB2 - kA2));

// Outputs of a tile: the six elements carry F(4, 3), F(2, 5) and F(3, 4) alike, whose tiles start 4, 2 and 3 pixels apart.  A row
// of 7 taps is two of F(3, 4): the first three taps, and the other four on the tile after, three pixels on.
__host__ __device__ constexpr int row_outputs_of(int taps) { return taps == 7 ? 3 : 7 - taps; }
__host__ __device__ constexpr int row_pieces(int taps) { return taps == 7 ? 2 : 1; }

// One output channel of a tile from the two halves of its elements, each reduced to (x, s, d): the element at 0 or infinity,
// and sum and difference of the pair at +-a (first half) or +-1/a (second)
template <int OUT> struct RowOutputs { float o[OUT]; };
template <int OUT>
__device__ __forceinline__ RowOutputs<OUT> row_outputs(float m0, float sa, float da, float mi, float sb, float db, float b) {
  if constexpr (OUT == 3) {
    return {{m0 + sa + sb + b, __builtin_fmaf(kA, da, __builtin_fmaf(kB, db, b)), __builtin_fmaf(kA2, sa, __builtin_fmaf(kB2, sb, mi + b))}};
  } else if constexpr (OUT == 2) {
    return {{m0 + sa + sb + b, __builtin_fmaf(kA, da, __builtin_fmaf(kB, db, mi + b))}};
  } else {
    return {{m0 + sa + sb + b, __builtin_fmaf(kA, da, __builtin_fmaf(kB, db, b)), __builtin_fmaf(kA2, sa, __builtin_fmaf(kB2, sb, b)),
             __builtin_fmaf(kA * kA2, da, __builtin_fmaf(kB * kB2, db, mi + b))}};
  }
}

// the first n < 8 of eight 16-bit elements, in at most three stores
template <typename T>
__device__ __forceinline__ void store_some(T* dst, u32x4 v, int n) {
  unsigned next = v[0], after = v[1];
  if (n & 4) {
    __builtin_memcpy(dst, &v, 8);
    dst += 4; next = v[2]; after = v[3];
  }
  if (n & 2) {
    __builtin_memcpy(dst, &next, 4);
    dst += 2; next = after;
  }
  if (n & 1) __builtin_memcpy(dst, &next, 2);
}

constexpr int kRowPitch = 64;     // LDS bytes per (element, row of a tile): 32 channels in four chunks of 16 bytes
// Chunk g of row s lies at position g ^ (s / 4 % 4).  A 16-byte read is served in four phases of sixteen lanes over 64
// banks, lanes 0-3, 12-15, 20-27 in the first, 4-11, 16-19, 28-31 in the second and the same 32 further up: of the lanes of
// a phase with the same row modulo 4 each has another row / 4 modulo 4, so one chunk of 32 consecutive rows, from any
// row on, is read without conflicts, and so is what a store writes, all chunks of 16 rows.  Two lanes of a phase whose
// different rows agree modulo 16 take a cycle each: what the boxes make of that, see choose_box.
__device__ __forceinline__ int v_offset(int s, int g) { return s * kRowPitch + ((g ^ (s >> 2)) & 3) * 16; }

// eight 16-bit elements without the first `by` < 8, zeros behind them
__device__ __forceinline__ u32x4 shift_channels(u32x4 v, int by) {
  if (by & 4) v = u32x4{v[2], v[3], 0u, 0u};
  if (by & 2) v = u32x4{v[1], v[2], v[3], 0u};
  if (by & 1) v = u32x4{v[0] >> 16 | v[1] << 16, v[1] >> 16 | v[2] << 16, v[2] >> 16 | v[3] << 16, v[3] >> 16};
  return v;
}

// The box of output tiles of a workgroup (conv_row.hip): images, planes, rows, tiles of a row, how many along each axis, the LDS rows of a plane and an image
struct RowBox { int bn, bd, bh, bw, n_n, n_d, n_h, n_w, prow, irow; long long boxes; };
RowBox choose_box(int N, int oD, int oH, int nW, int kd, int kh, int tiles, int slots);

// Few tiles (conv_row_few.hip): the workgroups of the kernel where it is taken for `planes` output planes, and their box, else 0 (padded: x with channels
// padded to a multiple of 8), and the launch with the arguments of row_conv (box null: to be searched)
int row_few_workgroups(long long planes, int oH, int nW, int kd, int kh, int K, int C, bool padded, RowBox* box);
bool row_few_takes_filter(const wc_conv_desc* d, const void* w, const int64_t s[5]);      // whether the kernel can take it as it is, instead of U
bool row_few_filter_pays(const wc_conv_desc* d, int workgroups);                          // and is the faster then
int row_few_conv(const wc_conv_desc* d, const void* x, int x_row, int n_images, const RowBox* box, const void* U, const void* w, const int64_t* w_strides, const void* bias, void* y,
                 void* stream);

}  // namespace wc
