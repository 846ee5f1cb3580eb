// The row form (conv_row.hip) for few tiles: 16 tiles x 16 output channels per workgroup, the reduction shared out over up to sixteen
// wavefronts.
//
// A layer with hardly any pixels is bound by the length of the chain from the launch to the stores and by the way of its filter into the few compute
// units that have a box of it.  The smallest shape of conv_row.hip gives 32 channels to a workgroup and walks over the channel blocks
// in steps, each with its barriers, its loads a step ahead.  Here a workgroup takes half the channels, and a pair of wavefronts one channel
// block (3-D: and plane of taps), an "item", by itself: each brings and transforms half of its input, each multiplies half of the
// tile's elements, and pairs meet only where their sums are added.  With an item to a pair (up to eight) the loads of the whole reduction are in flight at once, and the
// chain has one wait for memory; with more (512 channels), a pair asks for its next item's input and filter before it multiplies.
//
// A launch that does nothing takes 1.7 us in a row of launches, this one 4.3 to 6.5 with an item to a pair, 9.5 at 512 channels, where
// the transform of an item is on every SIMD's way four times (2.4 us of vector instructions).  8 channels per workgroup, twice the compute units with half the filter each:
// no faster there (9.3), nor elsewhere.
#include "row_form.h"

#include <algorithm>

namespace wc {

namespace {

struct FewArgs {
  const void* x; const void* U; const void* bias; void* y;
  int N, D, H, W, C, K;           // x (N, D, H, W, C), C rounded up to 8
  int oD, oH, oW;
  int pd, ph, pw, kd;
  int bn, bh, bw, n_h, n_w;       // box: output planes, rows, tiles of a row; boxes per plane
  int lw, irow, n_img;            // LDS rows of a row of tiles and of a plane of the box; N oD planes
  FastDiv f_lw, f_irow, f_bw, f_bh, f_d;
  int n_box, n_wg, per_xcd;
  int steps, items, shares;       // channel blocks, channel blocks times planes of taps, the wavefront pairs that share them
  int x_bytes, u_bytes;
  int x_row, tail;                // elements from a pixel of x to the next: C, or `tail` (below 8) fewer
  const void* w; long long w_k, w_c;      // the filter itself where U is null: elements from an output channel and an input channel to the next
};

// How a workgroup comes by its filter: as row_filter_kernel left it, or itself from 3x3 taps in a row, in the order of memory or against it.  kByBlock: the
// taps of 8 channels in a row as well, at a multiple of 16 bytes
enum FewFilter { kTransformed, kByBlock, kTaps, kTapsBack };

template <typename T> struct MfmaFew;
template <> struct MfmaFew<half_t> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <> struct MfmaFew<bf16_t> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};

// Partial sums of an element in LDS: [channel][tile], the rows of sixteen tiles 20 words apart: free of conflicts both ways (stores: four channels that are
// four rows apart, sixteen tiles each; reads: sixteen channels of four tiles)
constexpr int kPartRow = 20, kPart = 16 * kPartRow;

// FW, for 3x3 layers whose filter is new to every call (training, the functions): a launch of its own for the transform costs the host 3 us and the
// chain as much, where all such a layer takes is 4 to 9.  A lane's fragments are 8 channels of an output channel: 144 bytes of w
// where U is 288, and some 250 vector instructions an item.  The numbers are row_filter_kernel's.  us of a call, two launches | one, fp16:
// N=24 96 -> 96, 9x7 9.5 | 6.5, N=1 96 -> 64, 28x28 9.8 | 6.4, 256 -> 256, 14x14 11.2 | 10.8, 512 -> 512, 7x7 20.1 | 18.1 (where not: row_few_filter_pays).
//
// SLOTS: rows of LDS for a box's input.  RC: row taps whose filter fragments are in registers at a time.  ANY: as in conv_row.hip
// ONE: no pair has more than one item.  7x7 with more: two sets of 12 fragments of input leave 2 of 14 row taps room (all seven of a half spilled 7 to 11
// registers; us so | two at a time: N=1 512 -> 160, 7x7 25.5 | 21.4, 160 -> 160, 28x28 11.9 | 9.9, N=4 250 -> 512, 7x7 15.4 | 13.5, N=2 384 -> 96, 14x14
// 19.7 | 17.0; the other shapes' fastest of the four 29.9, 14.9, 18.2, 24.0)
template <typename T, int KH, int SLOTS, int RC, int THREADS, bool ONE, bool ANY, int FW>
__global__ __launch_bounds__(THREADS) void row_few_kernel(FewArgs a) {
  constexpr int KP = row_pieces(KH), R = KH * KP, OUT = row_outputs_of(KH), UN = SLOTS / 32, TS = SLOTS * kRowPitch, BUF = 6 * TS;
  static_assert(BUF >= 6 * kPart * 4 && R % RC == 0 && SLOTS % 32 == 0, "partial sums in the place of the input, whole turns");
  extern __shared__ unsigned char lds_all[];
  const int wg = xcd_remap(blockIdx.x, a.per_xcd);
  if (wg >= a.n_wg) return;
  const int kg = wg / a.n_box, box = wg - kg * a.n_box;       // a filter's workgroups lie on one XCD
  const int b_w = box % a.n_w, q_ = box / a.n_w;
  const int i0 = q_ / a.n_h * a.bn, h0 = q_ % a.n_h * a.bh, w0 = b_w * a.bw;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), share = wave >> 1, tg = wave & 1;
  unsigned char* const lds = lds_all + share * BUF;           // of the pair
  const __amdgpu_buffer_rsrc_t xdesc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.x), 0, a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t udesc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.U), 0, a.u_bytes, 0x00020000);

  // ---- input: units of (row of a tile, 8 channels), half of them to each wavefront of the pair
  const int chunk = lane & 3, slot0 = tg * (SLOTS / 2) + (lane >> 2);
  int base[UN], plane[UN];
  unsigned in[UN];                // bit j: pixel j is inside the image's rows and columns
#pragma unroll
  for (int i = 0; i < UN; ++i) {
    int s = slot0 + i * 16;
    const int im = fast_div(s, a.f_irow); s -= im * a.irow;
    const int zh = fast_div(s, a.f_lw), iw = s - zh * a.lw;
    const int img = i0 + im, n = fast_div(img, a.f_d), h = h0 + zh - a.ph, w = (w0 + iw) * OUT - a.pw;
    plane[i] = img - n * a.oD - a.pd;
    const bool ok = im < a.bn && img < a.n_img && zh < a.bh + KH - 1 && (unsigned)h < (unsigned)a.H;
    base[i] = (((n * a.D + plane[i]) * a.H + h) * a.W + w) * (ANY ? a.x_row : a.C) * 2 + chunk * 16;
    in[i] = 0;
#pragma unroll
    for (int j = 0; j < 6; ++j) in[i] |= ok && (unsigned)(w + j) < (unsigned)a.W ? 1u << j : 0u;
  }
  const int pixel = (ANY ? a.x_row : a.C) * 2, plane_bytes = a.H * a.W * pixel;
  u32x4 xr[ONE ? 1 : 2][UN][6];
  auto load_x = [&](auto to_c, int item) {
    constexpr int to = decltype(to_c)::value;
    const int rd = item / a.steps, step = item - rd * a.steps;
    const bool there = step * 32 + chunk * 8 < a.C;
    // the lanes of the last eight channels start `tail` channels before and shift (store_v)
    const int back = ANY && step * 32 + chunk * 8 == a.C - 8 ? a.tail * 2 : 0;
#pragma unroll
    for (int i = 0; i < UN; ++i) {
      const bool ok = there && (unsigned)(plane[i] + rd) < (unsigned)a.D;
      const int from = base[i] + rd * plane_bytes + step * 64 - back;
#pragma unroll
      for (int j = 0; j < 6; ++j) xr[to][i][j] = __builtin_amdgcn_raw_buffer_load_b128(xdesc, ok && (in[i] >> j & 1) ? from + j * pixel : (int)kOutside, 0, 0);
    }
  };
  auto store_v = [&](auto from_c, int item) {
    constexpr int from = decltype(from_c)::value;
    const int step = item % a.steps;
    const int by = ANY && step * 32 + chunk * 8 == a.C - 8 ? a.tail : 0;
#pragma unroll
    for (int i = 0; i < UN; ++i) {
      u32x4 (&x)[6] = xr[from][i];
      if constexpr (ANY) {
#pragma unroll
        for (int j = 0; j < 6; ++j) x[j] = shift_channels(x[j], by);
      }
#pragma unroll
      for (int word = 0; word < 4; ++word) {
        Pack<T, 2> two[6];
#pragma unroll
        for (int j = 0; j < 6; ++j) {
          const unsigned v = x[j][word];
          two[j] = __builtin_bit_cast(Pack<T, 2>, v);
        }
        row_input_channel(two, 0);
        row_input_channel(two, 1);
#pragma unroll
        for (int t = 0; t < 6; ++t) x[t][word] = __builtin_bit_cast(unsigned, two[t]);
      }
#pragma unroll
      for (int t = 0; t < 6; ++t) *reinterpret_cast<u32x4*>(lds + v_offset(slot0 + i * 16, chunk) + t * TS) = x[t];
    }
  };

  // ---- filter: rows 16 (kg % 2) .. + 16 of the block's fragments; a lane's chunk of 8 channels is in the fragment of its half
  const int kb = kg >> 1, kp = kg & 1, u_base = kb * (a.steps * a.kd * R * 2) * 6144;
  const int u_lane = (lane >> 5) * 6144 + (((lane >> 4) & 1) * 32 + kp * 16 + (lane & 15)) * 16 + tg * 3072;
  // R == RC: two sets, the next item's comes while this one's is multiplied
  constexpr int SETS = R == RC && !ONE && FW == kTransformed ? 2 : 1;
  u32x4 uf[SETS][RC][3];
  auto load_u = [&](auto to_c, int item, int part) {
    constexpr int to = decltype(to_c)::value % SETS;
    const int rd = item / a.steps, step = item - rd * a.steps;
    const int at = u_base + ((step * a.kd + rd) * R + part * RC) * 2 * 6144;
#pragma unroll
    for (int r = 0; r < RC; ++r)
#pragma unroll
      for (int t = 0; t < 3; ++t) uf[to][r][t] = __builtin_amdgcn_raw_buffer_load_b128(udesc, u_lane + t * 1024, at + r * 2 * 6144, 0);
  };

  // ---- the same from the filter itself: its taps on their way, and what becomes of them
  static_assert(FW == kTransformed || (KH == 3 && RC == R && !ANY), "three rows of three taps, whole chunks of channels");
  constexpr int WL = FW == kByBlock ? 9 : FW == kTransformed ? 1 : 8;
  u32x4 wr[WL];
  unsigned short last[FW == kTaps || FW == kTapsBack ? 8 : 1];
  const int w_m = kp * 16 + (lane & 15), w_row = min(kb * 32 + ((w_m >> 2) & 1) * 16 + (w_m >> 3) * 4 + (w_m & 3), a.K - 1);     // (rows beyond K are not stored)
  auto load_w = [&](int item) {
    const int c = item * 32 + (lane >> 4) * 8;
    const bool there = c < a.C;
    const T* const p = static_cast<const T*>(a.w) + w_row * a.w_k + (there ? c : 0) * a.w_c;
    if constexpr (FW == kByBlock) {
#pragma unroll
      for (int i = 0; i < 9; ++i) wr[i] = *reinterpret_cast<const u32x4*>(p + i * 8);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const T* const q = p + e * a.w_c - (FW == kTapsBack ? 8 : 0);
        __builtin_memcpy(&wr[e], q, 16);
        __builtin_memcpy(&last[e], q + 8, 2);
      }
    }
    if (!there) {                       // a last block of fewer channels: zeros, as x has them
#pragma unroll
      for (int i = 0; i < WL; ++i) wr[i] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (unsigned short& l : last) l = 0;
    }
  };
  auto make_u = [&]() {
    auto tap = [&](int e, int t) -> float {
      if (FW == kTapsBack) t = 8 - t;
      const int at = FW == kByBlock ? e * 9 + t : t;
      if (FW != kByBlock && t == 8) return static_cast<float>(__builtin_bit_cast(T, last[FW == kByBlock ? 0 : e]));
      const unsigned two = wr[FW == kByBlock ? at / 8 : e][at % 8 / 2];
      return static_cast<float>(__builtin_bit_cast(Pack<T, 2>, two).v[at % 2]);
    };
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int word = 0; word < 4; ++word) {
        Pack<T, 2> o[3];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float g0 = tap(word * 2 + e, r * 3), g1 = tap(word * 2 + e, r * 3 + 1), g2 = tap(word * 2 + e, r * 3 + 2);
          const RowPair pair = row_filter_pair(g0, g1, g2, 0.f, 0.f, tg == 0 ? kA : kB, tg == 0 ? kA2 : kB2, tg == 0 ? kRowFa : kRowFb);
          const T plus = static_cast<T>(pair.plus), minus = static_cast<T>(pair.minus);
          o[0].v[e] = tg == 0 ? static_cast<T>(g0) : plus;
          o[1].v[e] = tg == 0 ? plus : minus;
          o[2].v[e] = tg == 0 ? minus : static_cast<T>(g2);
        }
#pragma unroll
        for (int t = 0; t < 3; ++t) uf[0][r][t][word] = __builtin_bit_cast(unsigned, o[t]);
      }
  };

  // this lane's tile
  int vo;
  {
    int i = lane & 15;
    if (i >= a.bn * a.bh * a.bw) i = 0;
    const int q1 = fast_div(i, a.f_bw), q2 = fast_div(q1, a.f_bh);
    vo = q2 * a.irow + (q1 - q2 * a.bh) * a.lw + i - q1 * a.bw;
  }

  f32x4 acc[3];
#pragma unroll
  for (int t = 0; t < 3; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  load_x(ic<0>{}, share);
  if constexpr (FW == kTransformed) load_u(ic<0>{}, share, 0);
  else load_w(share);
  if constexpr (!ONE) {
    if (share + a.shares < a.items) load_x(ic<1>{}, share + a.shares);
  }
  // every pair goes as many rounds: the barriers are the workgroup's
  auto round = [&](auto cur_c, int item) {
    constexpr int cur = decltype(cur_c)::value;
    const bool mine = ONE || item < a.items, more = !ONE && item + a.shares < a.items;
    if (mine) {
      store_v(cur_c, item);
      if constexpr (SETS == 2) {
        if (more) load_u(ic<1 - cur>{}, item + a.shares, 0);
      }
      if constexpr (FW != kTransformed) {
        make_u();
        if (more) load_w(item + a.shares);
      }
    }
    __syncthreads();
    if (mine) {
#pragma unroll
      for (int part = 0; part < R / RC; ++part) {
        if (part > 0) load_u(ic<0>{}, item, part);
#pragma unroll
        for (int r = part * RC; r < part * RC + RC; ++r) {
          const unsigned char* const v = lds + v_offset(vo + r / KP * a.lw + r % KP, lane >> 4) + tg * 3 * TS;
#pragma unroll
          for (int t = 0; t < 3; ++t) acc[t] = MfmaFew<T>::run(uf[cur % SETS][r % RC][t], *reinterpret_cast<const u32x4*>(v + t * TS), acc[t]);
        }
      }
      if constexpr (!ONE) {
        if constexpr (SETS == 1 && FW == kTransformed) {
          if (more) load_u(ic<0>{}, item + a.shares, 0);
        }
        if (item + 2 * a.shares < a.items) load_x(cur_c, item + 2 * a.shares);
      }
    }
    __syncthreads();
  };
  if constexpr (ONE) {
    round(ic<0>{}, share);
  } else {
    for (int first = 0; first < a.items; first += 2 * a.shares) {
      round(ic<0>{}, first + share);
      if (first + a.shares < a.items) round(ic<1>{}, first + share + a.shares);
    }
  }
  {
    float* const part = reinterpret_cast<float*>(lds) + tg * 3 * kPart + (lane >> 4) * 4 * kPartRow + (lane & 15);
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) part[t * kPart + e * kPartRow] = acc[t][e];
  }
  __syncthreads();

  // ---- the shares' sums and the output transform: a quarter of the tiles to a wavefront, lane = channel + 16 tile
  const int waves = a.shares * 2, c = lane & 15;
  // rows 8 i + 4 h .. + 4 of the block's 32 are channels 16 h + 4 i .. + 4 (row_filter_kernel)
  const int row = ((c >> 2) & 1) * 8 + (c >> 3) * 4 + (c & 3), k = kb * 32 + (c >> 3) * 16 + kp * 8 + (c & 7);
  for (int w4 = wave; w4 < 4; w4 += waves) {
    const int tile = w4 * 4 + (lane >> 4);
    const float* part = reinterpret_cast<const float*>(lds_all) + row * kPartRow + tile;
    float m[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < a.shares; ++s, part += BUF / 4) {
#pragma unroll
      for (int t = 0; t < 6; ++t) m[t] += part[t * kPart];
    }
    const int q1 = fast_div(tile, a.f_bw), q2 = fast_div(q1, a.f_bh);
    const int img = i0 + q2, h = h0 + q1 - q2 * a.bh, w = (w0 + tile - q1 * a.bw) * OUT;
    if (q2 >= a.bn || img >= a.n_img || h >= a.oH || k >= a.K) continue;
    const float bias = a.bias ? static_cast<float>(static_cast<const T*>(a.bias)[k]) : 0.f;
    const RowOutputs<OUT> out = row_outputs<OUT>(m[0], m[1] + m[2], m[1] - m[2], m[5], m[3] + m[4], m[3] - m[4], bias);
    T* const yp = static_cast<T*>(a.y) + (((size_t)img * a.oH + h) * a.oW + w) * a.K + k;
#pragma unroll
    for (int j = 0; j < OUT; ++j)
      if (w + j < a.oW) yp[(size_t)j * a.K] = static_cast<T>(out.o[j]);
  }
}

// LDS rows of a box and the pairs of wavefronts of a workgroup at most, by the kernel's extent
constexpr int few_slots(int kh) { return kh == 7 ? 64 : 32; }
constexpr int few_shares(int kh, bool one) { return one && kh != 7 ? 8 : 4; }
// Workgroups along the output channels: of a last block of 32, the first sixteen rows are channels 0 to 7 and 16 to 23
int few_groups(int K) { return K / 32 * 2 + (K % 32 > 8 ? 2 : K % 32 > 0 ? 1 : 0); }

// Pairs of wavefronts that share out `items`
int few_pairs(int items, int kh) {
  return ceil_div(items, ceil_div(items, few_shares(kh, items <= few_shares(kh, true))));
}

RowBox few_box(int planes, int oH, int nW, int kh) { return choose_box(planes, 1, oH, nW, 1, kh, 16, few_slots(kh)); }

}  // namespace

// The workgroups of the launch where all are on the chip at once, at most three to a CU; else 0.  Of 600 layers drawn over 1 to 32 images (3-D: 8), 32 to 512 channels (128) and 7 to 56
// rows, at most 2000 of these workgroups, the launch takes 0.80 of the time of the other shapes' choice in the mean so, 1.02 of it where a few are
// left for a second round; the faster of the two for each would be 0.80 as well.  us, other shapes | this, fp16 and bf16, launches in a row: N=1 512 -> 512, 7x7 12.2 | 9.5, 256 -> 256,
// 14x14 9.5 | 6.3, N=4 9.8 | 6.5, N=8 (two rounds) 9.8 | 11.2, N=1 160 -> 160, 28x28 9.4 | 5.5, N=4 64 -> 96, 24x24 6.6 | 4.3, N=4 384 -> 288, 12x12 11.7 | 8.6,
// 5x5 N=9 160 -> 96, 10x10 10.0 | 5.8, 7x7 N=2 119 -> 391, 15x13 13.0 | 8.9, 3-D N=1 64 -> 64, 4x14x14 8.1 | 5.6; more to a CU: N=25 32 -> 64, 31x31 6.0 | 7.4.
int row_few_workgroups(long long planes, int oH, int nW, int kd, int kh, int K, int C, bool padded, RowBox* box) {
  const int groups = few_groups(K), items = ceil_div(C, 32) * kd;
  const bool one = items <= few_shares(kh, true), any = C % 8 != 0 && !padded;
  const int pairs = few_pairs(items, kh);
  // the wavefronts that the registers let a CU have, and the workgroups of LDS
  const int waves = !one ? 8 : kh == 7 ? (any ? 12 : 16) : any ? 16 : kh == 5 ? 20 : 24;
  const int resident = std::max(1, std::min({3, 160 * 1024 / (pairs * 6 * few_slots(kh) * kRowPitch), waves / (2 * pairs)}));
  const long long most = (long long)resident * kCus;
  // a box holds sixteen tiles at most, which spares most layers the search for it (a plan of N=64 256 -> 256, 14x14 4.2 us with it, 3.8 without)
  if (ceil_div_ll(planes * oH * nW, 16) * groups > most) return 0;
  *box = few_box((int)planes, oH, nW, kh);
  const long long workgroups = box->boxes * groups;
  return workgroups <= most ? (int)workgroups : 0;
}

// How the kernel can take the filter as it is (kTransformed: not)
static FewFilter few_filter(const wc_conv_desc* d, const void* w, const int64_t s[5]) {
  if (d->kernel[0] != 1 || d->kernel[1] != 3 || d->kernel[2] != 3 || d->C % 8 || (s[4] != 1 && s[4] != -1) || s[3] != 3 * s[4] || (reinterpret_cast<uintptr_t>(w) & 1)) return kTransformed;
  if (s[4] == 1 && s[1] == 9 && s[0] % 8 == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0) return kByBlock;
  // Sixteen loads of scattered channels an item instead of nine: ahead where the reduction has an item to a pair (input gradients, us of a call, two launches | one, 256 -> 256,
  // 14x14 13.2 | 11.9, N=24 96 -> 96, 9x7 11.9 | 8.7), behind with more (512 -> 512, 7x7 20.2 | 20.4, N=2 416 -> 224, 19x17 16.8 | 17.5) and with planes of
  // taps (128 -> 128, 3x9x9 14.6 | 17.2, forward 15.8 | 26.6)
  if (ceil_div(d->C, 32) > few_shares(3, true)) return kTransformed;
  return s[4] == 1 ? kTaps : kTapsBack;
}
bool row_few_takes_filter(const wc_conv_desc* d, const void* w, const int64_t s[5]) { return few_filter(d, w, s) != kTransformed; }

// Every workgroup transforms the filter that it takes, every box of a channel group anew, and a CU does so one item after the other: one launch is the
// faster call where a CU has at most eight items of it.  Of 93 layers, us of a call, two launches | one (the GPU's part of it): three items, up to two workgroups a CU 9.7 | 8.8 (8.1 | 8.4),
// three 10.0 | 11.8 (9.0 | 11.4); four 9.8 | 9.6 and 10.8 | 13.6; five, one 9.8 | 7.8, two 11.1 | 12.8; eight, one 10.7 | 9.8; one and two items are ahead with three
// workgroups a CU as well, 9.8 | 6.9 and 9.8 | 8.2.
// With more than an item to a pair the time goes by C and that of the two launches by the filter, C K.  Of 106 layers: 288 -> 256 12.0 | 12.7, 320 12.7 | 12.4, 384 -> 256
// 14.3 | 14.8, 320 15.0 | 14.8, 448 -> 224 15.2 | 16.1, 384 16.8 | 16.4, 512 -> 128 14.5 | 18.2, 320 18.0 | 18.7, 512 19.9 | 18.6, 640 -> 384 21.1 | 22.0, 512 22.3 | 21.8, 768 -> 448
// 24.9 | 25.7, 640 26.9 | 25.8, 1024 -> 64 21.6 | 33.1, 640 32.8 | 32.6.
bool row_few_filter_pays(const wc_conv_desc* d, int workgroups) {
  const int items = ceil_div(d->C, 32);
  if (items > few_shares(3, true)) return d->K >= 320 && 4 * d->K >= 3 * d->C;
  return ceil_div(workgroups, kCus) * items <= 8;
}

// Images n_images from x on; x as row_conv takes it.  box: the plan's, whose search took a call 0.2 to 0.4 us of the host; null: the images are not
// the plan's.  U null: the filter is w
int row_few_conv(const wc_conv_desc* d, const void* x, int x_row, int n_images, const RowBox* box, const void* U, const void* w, const int64_t* w_strides, const void* bias, void* y,
                 void* stream) {
  FewArgs a{};
  const int kh = d->kernel[1];
  const FewFilter how = U ? kTransformed : few_filter(d, w, w_strides);
  WC_CHECK_ARG(U || how != kTransformed, "row form, few tiles: neither a transformed filter nor one that the kernel takes");
  a.w = w;
  if (!U) { a.w_k = w_strides[0]; a.w_c = w_strides[1]; }
  a.x = x; a.U = U; a.bias = bias; a.y = y;
  a.N = n_images; a.D = d->in[0]; a.H = d->in[1]; a.W = d->in[2]; a.C = wc_padded_channels8(d->C); a.K = d->K;
  a.x_row = x_row; a.tail = a.C - x_row;
  a.pd = d->pad[0]; a.ph = d->pad[1]; a.pw = d->pad[2]; a.kd = d->kernel[0];
  a.oD = a.D + 2 * a.pd - a.kd + 1; a.oH = a.H + 2 * a.ph - kh + 1; a.oW = a.W + 2 * a.pw - kh + 1;
  a.n_img = a.N * a.oD;
  const RowBox b = box ? *box : few_box(a.n_img, a.oH, ceil_div(a.oW, row_outputs_of(kh)), kh);
  a.bn = b.bn; a.bh = b.bh; a.bw = b.bw; a.n_h = b.n_h; a.n_w = b.n_w;
  a.lw = b.bw + row_pieces(kh) - 1; a.irow = b.irow;
  a.f_lw = make_fast_div(a.lw); a.f_irow = make_fast_div(a.irow); a.f_bw = make_fast_div(a.bw); a.f_bh = make_fast_div(a.bh); a.f_d = make_fast_div(a.oD);
  a.n_box = (int)b.boxes;
  a.n_wg = a.n_box * few_groups(a.K);
  a.per_xcd = ceil_div(a.n_wg, kXcds);
  a.steps = ceil_div(a.C, 32); a.items = a.steps * a.kd;
  const bool one = a.items <= few_shares(kh, true);
  a.shares = few_pairs(a.items, kh);
  a.x_bytes = (int)((long long)a.N * a.D * a.H * a.W * x_row * 2);
  a.u_bytes = (int)(row_u_elems(d) * 2);
  return dispatch_dtype(d->dtype, [&](auto t) -> int {
    using T = decltype(t);
    if constexpr (sizeof(T) == 2) {
      auto launch = [&](auto kh_c, auto one_c) -> int {
        constexpr bool ONE = decltype(one_c)::value != 0;
        constexpr int KH = decltype(kh_c)::value, SLOTS = few_slots(KH), RC = KH == 7 && !ONE ? 2 : KH;
        constexpr int SHARES = few_shares(KH, ONE), THREADS = 128 * SHARES;
        auto fn = a.tail ? &row_few_kernel<T, KH, SLOTS, RC, THREADS, ONE, true, kTransformed> : &row_few_kernel<T, KH, SLOTS, RC, THREADS, ONE, false, kTransformed>;
        if constexpr (KH == 3) {
          if (how == kByBlock) fn = &row_few_kernel<T, KH, SLOTS, RC, THREADS, ONE, false, kByBlock>;
          if constexpr (ONE) {                // scattered taps have an item to a pair (few_filter)
            if (how == kTaps) fn = &row_few_kernel<T, KH, SLOTS, RC, THREADS, ONE, false, kTaps>;
            else if (how == kTapsBack) fn = &row_few_kernel<T, KH, SLOTS, RC, THREADS, ONE, false, kTapsBack>;
          }
        }
        constexpr int bytes = 6 * SLOTS * kRowPitch;          // of a pair
        if (const int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), SHARES * bytes)) return rc;
        hipLaunchKernelGGL(fn, dim3(a.per_xcd * kXcds), dim3(128 * a.shares), a.shares * bytes, as_stream(stream), a);
        WC_CHECK_LAUNCH("row_few_kernel");
        return WC_OK;
      };
      auto go = [&](auto kh_c) -> int { return one ? launch(kh_c, ic<1>{}) : launch(kh_c, ic<0>{}); };
      if (kh == 3) return go(ic<3>{});
      if (kh == 5) return go(ic<5>{});
      return go(ic<7>{});
    }
    return fail(WC_ERR_UNSUPPORTED, "row form: 16-bit types");
  });
}

}  // namespace wc
