// Change of layout between channel-first (N, C, S) and channel-last (N, S, C) memory, S = [D] H W: a bit-exact
// copy.  Replaces the permute passes the reference runs in torch on both sides of its kernels
// (dwm.py:129-133,143-144; Split_and_Concat.py:25,47,64,81) for the plans whose transform kernels cannot read or
// write channel-first memory themselves.
//
// Per image this is the transpose of an R x Q matrix into a Q x R one.  A thread turns a square block of 16 bytes a side
// in registers (8 x 8 elements of two bytes, 4 x 4 of four); the 64 blocks of a wavefront form a square, so that every access
// of a wavefront is eight runs of 128 contiguous bytes.  Rows start at any multiple of the element size: accesses of 16 bytes
// need no alignment here.  No LDS and no barrier: a small copy is a few loads in flight per wavefront and its stores.  us,
// tiles of 64 x 64 through LDS in accesses of 2 or 4 bytes | this, 16 bit: 6 x 100 x 2745 7.8 | 3.9, 64 x 256 x 3136 51 | 35 (5.8 TB/s),
// back 50 | 35, 64 x 128 x 3136 20.4 | 18.2; 32 bit, 64 x 256 x 3136 102 | 74, 8 x 256 x 3136 12.0 | 9.9; 32 x 3 x 50176 (a thread to a
// column) 42 | 9.
#include "wc_transform.h"

#include <algorithm>

namespace wc {

struct TransposeArgs {
  const void* src;     // (n, R, Q)
  void* dst;           // (n, Q, Rd), Rd >= R, zeros beyond R
  long long R, Q, Rd;
  int tiles_r, tiles_q;
  long long n_blocks;
};

typedef uint32_t Words __attribute__((ext_vector_type(4)));

template <typename U>
__global__ __launch_bounds__(256) void transpose_kernel(TransposeArgs a) {
  constexpr int E = 16 / sizeof(U);
  const long long blk = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (blk >= a.n_blocks) return;
  const int tq = (int)(blk % a.tiles_q);
  const long long rest = blk / a.tiles_q;
  const int tr = (int)(rest % a.tiles_r);
  const long long n = rest / a.tiles_r;
  const int lane = threadIdx.x & 63;
  // loads: the lanes of a row of blocks run along Q; stores: along R
  long long q0 = (long long)tq * 8 * E + (lane & 7) * E, r0 = (long long)tr * 8 * E + (lane >> 3) * E;
  if (q0 >= a.Q || r0 >= a.Rd) return;
  // a block that would reach beyond the end overlaps its neighbour instead, and both write the same values there
  if (q0 + E > a.Q) q0 = a.Q - E;
  if (r0 + E > a.Rd) r0 = a.Rd - E;
  const U* const src = static_cast<const U*>(a.src) + (n * a.R + r0) * a.Q + q0;
  U* const dst = static_cast<U*>(a.dst) + (n * a.Q + q0) * a.Rd + r0;
  Words in[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    in[r] = Words{0u, 0u, 0u, 0u};
    if (r0 + r < a.R) __builtin_memcpy(&in[r], src + r * a.Q, 16);
  }
#pragma unroll
  for (int c = 0; c < E; ++c) {
    Words out;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      out[k] = sizeof(U) == 4 ? in[k][c % 4]
                              : __builtin_amdgcn_perm(in[(2 * k + 1) % E][c / 2 % 4], in[2 * k % E][c / 2 % 4], c % 2 ? 0x07060302u : 0x05040100u);
    __builtin_memcpy(dst + c * a.Rd, &out, 16);
  }
}

// Matrices narrower than a block on either side: a thread takes all of the narrow side
template <typename U>
__global__ __launch_bounds__(256) void transpose_narrow_kernel(TransposeArgs a) {
  const bool rows = a.Rd < a.Q;                    // few rows: a thread takes a column
  const long long wide = rows ? a.Q : a.Rd, i = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long n = i / wide, at = i - n * wide;
  if (i >= a.n_blocks) return;
  const U* const src = static_cast<const U*>(a.src) + n * a.R * a.Q;
  U* const dst = static_cast<U*>(a.dst) + n * a.Rd * a.Q;
  if (rows)
    for (int r = 0; r < (int)a.Rd; ++r) dst[at * a.Rd + r] = r < a.R ? src[r * a.Q + at] : U(0);
  else
    for (int q = 0; q < (int)a.Q; ++q) dst[q * a.Rd + at] = at < a.R ? src[at * a.Q + q] : U(0);
}

static int transpose_padded(const void* src, void* dst, long long n, long long R, long long Q, long long Rd, int elem_size, void* stream) {
  WC_CHECK_ARG(src && dst && n > 0 && R > 0 && Q > 0, "layout copy: null pointer or empty tensor");
  WC_CHECK_ARG(elem_size == 2 || elem_size == 4, "layout copy: element size %d", elem_size);
  TransposeArgs a;
  a.src = src; a.dst = dst; a.R = R; a.Q = Q; a.Rd = Rd;
  const int block = 16 / elem_size, side = 8 * block;
  const bool narrow = Rd < block || Q < block;
  a.tiles_r = (int)ceil_div_ll(Rd, side); a.tiles_q = (int)ceil_div_ll(Q, side);
  a.n_blocks = narrow ? n * std::max(Rd, Q) : n * a.tiles_r * a.tiles_q;
  const long long groups = ceil_div_ll(a.n_blocks, narrow ? 256 : 4);
  WC_CHECK_ARG(groups < (1ll << 31), "layout copy: problem too large");
  auto launch = [&](auto u) {
    using U = decltype(u);
    const auto fn = narrow ? transpose_narrow_kernel<U> : transpose_kernel<U>;
    hipLaunchKernelGGL(fn, dim3((unsigned)groups), dim3(256), 0, as_stream(stream), a);
  };
  if (elem_size == 2) launch((unsigned short)0);
  else launch(0u);
  WC_CHECK_LAUNCH("transpose_kernel");
  return WC_OK;
}

// src (n, R, Q) -> dst (n, Q, R), elements of 2 or 4 bytes
int transpose_images(const void* src, void* dst, long long n, long long R, long long Q, int elem_size, void* stream) {
  return transpose_padded(src, dst, n, R, Q, R, elem_size, stream);
}

// Rows of C 16-bit elements to rows of Cx, a multiple of 8: a thread moves 16 bytes, from wherever its row starts; the last of a row
// comes from the row's last eight elements, shifted (rows of less than eight: element by element).
struct PadArgs {
  const unsigned short* src; void* dst;
  int C, chunks;               // chunks of 8 elements in a row of dst
  long long total;             // rows x chunks
  FastDiv f_chunks;
};

__global__ __launch_bounds__(256) void pad_rows_kernel(PadArgs a) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.total) return;
  const long long row = a.total < (1ll << 31) ? fast_div((int)i, a.f_chunks) : i / a.chunks;
  const int c = (int)(i - row * a.chunks) * 8;
  const unsigned short* p = a.src + row * a.C + c;
  unsigned long long v[2] = {0, 0};
  if (c + 8 <= a.C) {
    __builtin_memcpy(v, p, 16);
  } else if (a.C >= 8) {
    const int bits = (c + 8 - a.C) * 16;         // 16 to 112
    __builtin_memcpy(v, p - bits / 16, 16);
    if (bits >= 64) v[0] = v[1] >> (bits - 64), v[1] = 0;
    else v[0] = v[0] >> bits | v[1] << (64 - bits), v[1] >>= bits;
  } else {
#pragma unroll
    for (int e = 0; e < 7; ++e)
      if (e < a.C) v[e / 4] |= (unsigned long long)p[e] << e % 4 * 16;
  }
  __builtin_memcpy(static_cast<unsigned char*>(a.dst) + i * 16, v, 16);
}

int pad_channels(const void* src, void* dst, long long n, int C, int Cx, long long S, bool channel_first, void* stream) {
  WC_CHECK_ARG(src && dst && n > 0 && C > 0 && Cx >= C && Cx % 8 == 0 && S > 0, "pad_channels: null pointer or empty tensor");
  if (channel_first) return transpose_padded(src, dst, n, C, S, Cx, 2, stream);
  PadArgs a;
  a.src = static_cast<const unsigned short*>(src); a.dst = dst; a.C = C; a.chunks = Cx / 8; a.total = n * S * a.chunks; a.f_chunks = make_fast_div(a.chunks);
  const long long blocks = ceil_div_ll(a.total, 256);
  WC_CHECK_ARG(blocks < (1ll << 31), "pad_channels: problem too large");
  hipLaunchKernelGGL(pad_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream), a);
  WC_CHECK_LAUNCH("pad_rows_kernel");
  return WC_OK;
}

// The fp32 parameters of a layer in its activations' type, weight and bias in one launch: as two casts they were two launches of some
// 5 us of host time each, in a training step that waits for the host (us, fp16 N=64 128 -> 128, 28x28, twelve processes each: 93-96 | 91-93 where autograd's thread
// wakes quickly, a matter of the process, and 114-122 | 110-115 where it does not).
struct CastArgs {
  const float* src[2]; void* dst[2];
  long long n[2];
  int blocks;                      // of the first, 1024 elements each; the second's behind them
};
template <typename T>
__global__ __launch_bounds__(256) void cast_kernel(CastArgs a) {
  const int which = (int)blockIdx.x >= a.blocks;
  const float* const src = a.src[which];
  T* const dst = static_cast<T*>(a.dst[which]);
  const long long i = ((long long)(blockIdx.x - (which ? a.blocks : 0)) * 256 + threadIdx.x) * 4, n = a.n[which];
  if (i >= n) return;
  if (i + 4 <= n) {                // either tensor may start at any element
    float v[4];
    Pack<T, 4> o;
    __builtin_memcpy(v, src + i, 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(v[e]);
    __builtin_memcpy(dst + i, &o, 8);
  } else {
    for (long long e = i; e < n; ++e) dst[e] = static_cast<T>(src[e]);
  }
}

}  // namespace wc

using namespace wc;

extern "C" int wc_cast_parameters(const float* w, void* w_out, long long n_w, const float* bias, void* bias_out, long long n_bias, int dtype, void* stream) {
  WC_CHECK_ARG(w && w_out && n_w > 0 && (n_bias == 0 || (n_bias > 0 && bias && bias_out)), "wc_cast_parameters: null pointer or empty tensor");
  WC_CHECK_ARG(dtype == WC_F16 || dtype == WC_BF16, "wc_cast_parameters: dtype %d, a 16-bit type is needed", dtype);
  const long long blocks = ceil_div_ll(n_w, 1024), more = ceil_div_ll(n_bias, 1024);
  WC_CHECK_ARG(blocks + more < (1ll << 31), "wc_cast_parameters: problem too large");
  const CastArgs a = {{w, bias}, {w_out, bias_out}, {n_w, n_bias}, (int)blocks};
  hipLaunchKernelGGL(dtype == WC_F16 ? &cast_kernel<half_t> : &cast_kernel<bf16_t>, dim3((unsigned)(blocks + more)), dim3(256), 0, as_stream(stream), a);
  WC_CHECK_LAUNCH("cast_kernel");
  return WC_OK;
}

extern "C" int wc_layout_copy(const void* src, void* dst, int n_images, int channels, long long spatial,
                              int to_channel_last, int elem_size, void* stream) {
  WC_CHECK_ARG(n_images > 0 && channels > 0 && spatial > 0, "wc_layout_copy: %d images, %d channels, %lld positions",
               n_images, channels, spatial);
  // channel-first (n, C, S) -> channel-last (n, S, C) is the transpose of C x S matrices, and back
  return to_channel_last ? transpose_images(src, dst, n_images, channels, spatial, elem_size, stream)
                         : transpose_images(src, dst, n_images, spatial, channels, elem_size, stream);
}
