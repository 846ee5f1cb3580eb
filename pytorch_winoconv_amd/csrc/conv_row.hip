// One-kernel convolution on the tile F(4, 3) along the width axis only ("row form"): 16-bit types, stride 1, 3x3 and 3x3x3
// kernels.  5x5 kernels run on F(2, 5), 7x7 kernels on two of F(3, 4) side by side, which have the same six points and so the
// same V: below, 4 w is 2 w or 3 w and A^T has as many rows.
//
//   y[o_d, o_h, 4 w + i] = sum_t A^T[i][t]  sum_(r_d, r_h) sum_c  U[r][t][k][c]  V[o_d + r_d, o_h + r_h, w][t][c]
//   V[., w][t] = sum_j B^T[t][j] x[., 4 w + j],      U[r][t] = sum_j G[t][j] w[r, j]
//
// The three-kernel path writes V and M to memory and reads them back (2.25 times the input and the output each way for
// F(4x4, 3x3), 4 times for F(2x2, 3x3)), which is what bounds it: at N=64, 256 -> 256 channels, 56x56 its three kernels
// move 1.13 GB at 5 TB/s.  Here one axis is transformed and the other axes' taps stay in the reduction: half the
// multiplications of the plain sum (the 2-D tile saves three quarters of them), but V lives in LDS, the products in
// accumulators, and x, U and y are all the memory traffic there is.  The sum over taps and channels is taken in fp32
// before the output transform, so only V and U are rounded to the storage type.
#include "row_form.h"

#include <algorithm>

namespace wc {

namespace {

struct RowArgs {
  const void* x; const void* U; const void* bias; void* y;
  int N, D, H, W, C, K;           // x (N, D, H, W, C), C rounded up to 8; y (N, oD, oH, oW, K)
  int oD, oH, oW, nW;             // nW tiles of 4 (5x5: 2) outputs per row
  int pd, ph, pw;
  int bn, bd, bh, bw;             // output box of a workgroup: images, planes, rows, tiles of a row
  FastDiv f_bw, f_bh, f_bd, f_prow, f_irow;
  int prow, irow;                 // LDS rows of a plane and of an image of the box's input (tile rows, with the halo and padding)
  int n_d, n_h, n_w;              // boxes per axis
  int n_kb, n_box, per_xcd;       // channel blocks, boxes
  int box_fast;                   // 1: neighbouring workgroups share a channel block, 0: a box
  int steps, local_steps;         // ceil(C / 32), and the share of one of the CS groups of wavefronts that split the channels
  int x_bytes, u_bytes;
  int lw;                         // tiles of a row of the box's input (7 taps: one more than bw)
  FastDiv f_lw;
  int x_row, tail;                // elements from a pixel of x to the next: C, or `tail` (below 8) fewer
};

// What the NI items of a step carry beside their products: the transform of 8 UN channels, over the first two thirds of the
// items, and for each unit six moves (an element to LDS, the next load of its register) behind its last channel
template <int UN, int NI>
struct RowItems {
  // one unit: the middle of the step, so that its loads, issued in the last quarter, have the first one to arrive
  static constexpr int from = UN == 1 ? NI / 4 : 0, to = UN == 1 ? 3 * NI / 4 : 2 * NI / 3;
  static constexpr int first_channel(int item) {
    const int n = item < from ? 0 : ((item - from) * 8 * UN + to - from - 1) / (to - from);
    return n < 8 * UN ? n : 8 * UN;
  }
  static constexpr int channels(int item) { return first_channel(item + 1) - first_channel(item); }
  static constexpr int window = UN == 1 ? NI - to : UN > 2 ? NI / 6 : NI / 3;
  static constexpr int at(int v) { return from + (v / 6 + 1) * (to - from) / UN + v % 6 * window / 6; }
  static constexpr int first_move(int item) { int n = 0; while (n < 6 * UN && at(n) < item) ++n; return n; }
  static constexpr int moves(int item) { return first_move(item + 1) - first_move(item); }
  static constexpr bool ok() {
    if (at(6 * UN - 1) >= NI) return false;
    for (int v = 0; v < 6 * UN; ++v)
      if (first_channel(at(v)) < (v / 6 + 1) * 8) return false;       // moved before its unit is transformed
    return true;
  }
};

template <int KG, int TB, int S, int CS>
constexpr int row_lds_bytes() {
  const int v = CS * 2 * 6 * S * kRowPitch, ex = 2 * KG * 3 * TB * 8 * 256, part = (CS - 1) * 2 * KG * 3 * TB * 16 * 256;
  return v > ex ? (v > part ? v : part) : (ex > part ? ex : part);
}

// ANY: rows of x or y that are no multiple of 16 bytes.  The last eight channels of x are loaded as they lie, ending with the last one, and
// shifted into their places, zeros behind them, in the step that takes them: a copy of x with padded rows cost, us, C a multiple of 8 | two
// channels fewer, copied | this: N=16 96 -> 64, 56x56 10.8 | 21.5 | 11.9, 320 -> 64 22.6 | 40.4 | 23.7, N=8 256 -> 128, 28x28 11.0 | 15.9 | 12.1, N=2 96 -> 96,
// 28x28 7.8 | 10.2 | 8.4.  Of y's rows the last stores are cut: N=4 64 -> 464, 86x86 28, 466 channels 42 element by element, now 29.  STAY: a workgroup per CU that goes from box to box
template <typename T, int KD, int KH, int KG, int TB, int S, int CS, bool STAY, bool ANY>
__global__ __launch_bounds__(128 * KG * CS) __attribute__((amdgpu_waves_per_eu(2, TB == 2 ? 2 : 3)))
void row_conv_kernel(RowArgs a) {
  using Frag = typename MfmaRow<T>::Frag;
  constexpr int KP = row_pieces(KH), R = KD * KH * KP, Q = 2 * R, NI = 3 * Q, THREADS = 128 * KG, UN = S * 4 / THREADS;
  constexpr int TS = S * kRowPitch, BUF = 6 * TS, OUT = row_outputs_of(KH);
  constexpr int UD = Q % 3 == 0 ? 3 : Q % 5 == 0 ? 5 : 4, VD = 3;      // depth of the rings of filter and input fragments
  static_assert(RowItems<UN, NI>::ok(), "items of a step");
  static_assert(S * 4 % THREADS == 0 && Q % UD == 0, "whole units per thread, whole turns of the ring");
  extern __shared__ unsigned char lds_all[];
  static_assert(!STAY || CS == 1, "shares end after their box");
  // this XCD's boxes from the workgroup's own on; STAY: every (workgroups of the XCD)-th
  int place = blockIdx.x / kXcds;
  const int place0 = blockIdx.x % kXcds * a.per_xcd, places = min(a.per_xcd, a.n_kb * a.n_box - place0);
  if (place >= places) return;
  int kb, n0, d0, h0, w0;
  auto go_to_box = [&]() {
    const int wg = place0 + place;
    int box;
    if (a.box_fast) { kb = wg / a.n_box; box = wg - kb * a.n_box; }
    else { box = wg / a.n_kb; kb = wg - box * a.n_kb; }
    const int b_w = box % a.n_w;
    int q_ = box / a.n_w;
    const int b_h = q_ % a.n_h; q_ /= a.n_h;
    const int b_d = q_ % a.n_d;
    n0 = q_ / a.n_d * a.bn; d0 = b_d * a.bd; h0 = b_h * a.bh; w0 = b_w * a.bw;
  };
  go_to_box();
  const int sd = a.bd + KD - 1, sh = a.bh + KH - 1, lw = KP == 1 ? a.bw : a.lw;

  const int lane = threadIdx.x & 63, wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cs = wave_all / (2 * KG), wave = wave_all - cs * 2 * KG, tid = wave * 64 + lane;
  const int tg = wave / KG, kg = wave % KG;
  unsigned char* const lds = lds_all + cs * 2 * BUF;
  const int step0 = cs * a.local_steps;                 // the channel blocks of this share: step0 .. + local_steps, as far as they exist
  const __amdgpu_buffer_rsrc_t xdesc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.x), 0, a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t udesc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.U), 0, a.u_bytes, 0x00020000);

  // ---- filter fragments: a ring of three groups (row tap, half of a channel block) of three elements
  const int n_groups = a.steps * Q, k_blocks = (a.K + 31) / 32;
  const int u_lane = lane * 16 + tg * 3072;
  int u_base = 0;
  u32x4 uf[UD][3];
  auto load_u = [&](int slot, int group, int t) {
    uf[slot][t] = __builtin_amdgcn_raw_buffer_load_b128(udesc, u_lane + t * 1024, u_base + min(step0 * Q + group, n_groups - 1) * 6144, 0);
  };

  // ---- input: units of (row of a tile, 8 channels)
  int xo[UN][6];
  u32x4 xr[UN][6];
  auto find_x = [&]() {
#pragma unroll
    for (int i = 0; i < UN; ++i) {
      const int u = tid + i * THREADS, g = u & 3;
      int s = u >> 2;
      const int in = fast_div(s, a.f_irow); s -= in * a.irow;
      const int zd = fast_div(s, a.f_prow); s -= zd * a.prow;
      const int zh = fast_div(s, KP == 1 ? a.f_bw : a.f_lw), iw = s - zh * lw;
      const int n = n0 + in, d = d0 + zd - a.pd, h = h0 + zh - a.ph, w = (w0 + iw) * OUT - a.pw;
      const bool ok = in < a.bn && zd < sd && zh < sh && n < a.N && (unsigned)d < (unsigned)a.D && (unsigned)h < (unsigned)a.H;
      const int base = (((n * a.D + d) * a.H + h) * a.W + w) * (ANY ? a.x_row : a.C) * 2 + g * 16;
#pragma unroll
      for (int j = 0; j < 6; ++j) xo[i][j] = ok && (unsigned)(w + j) < (unsigned)a.W ? base + j * (ANY ? a.x_row : a.C) * 2 : (int)kOutside;
    }
  };
  find_x();
  // the channel block is in the scalar offset (ANY: the last one in the lane's, which shifts it); beyond the last channel of the last block
  // lanes load zeros (cut_x)
  auto load_x = [&](int i, int j, int step) {
    const int block = ANY && step0 + step >= a.steps - 1 ? 0 : min(step0 + step, a.steps - 1);
    xr[i][j] = __builtin_amdgcn_raw_buffer_load_b128(xdesc, xo[i][j], block * 64, 0);
  };
  auto cut_x = [&](int step) {
    if (step0 + step >= a.steps - 1 && (tid & 3) * 8 + (step0 + step) * 32 >= a.C) {
#pragma unroll
      for (int i = 0; i < UN; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j) xo[i][j] = (int)kOutside;
    }
    if constexpr (ANY) {                 // once a box; the lanes of the last eight channels start `tail` channels before (outside stays outside)
      if (step0 + step == a.steps - 1) {
        const unsigned by = (a.steps - 1) * 64 - ((tid & 3) * 8 + (a.steps - 1) * 32 == a.C - 8 ? a.tail * 2 : 0);
#pragma unroll
        for (int i = 0; i < UN; ++i)
#pragma unroll
          for (int j = 0; j < 6; ++j) xo[i][j] = (int)((unsigned)xo[i][j] + by);
      }
    }
  };
  auto shift_x = [&](int step) {
    if constexpr (ANY) {
      if (a.tail == 0 || step0 + step != a.steps - 1) return;
      const int by = (tid & 3) * 8 + (a.steps - 1) * 32 == a.C - 8 ? a.tail : 0;
#pragma unroll
      for (int i = 0; i < UN; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j) xr[i][j] = shift_channels(xr[i][j], by);
    }
  };
  // one of a unit's eight channels at a time, in place: the six inputs of xr become the six elements of the tile
  auto transform_channel = [&](auto i_c, auto e_c) {
    constexpr int i = decltype(i_c)::value, word = decltype(e_c)::value / 2, e = decltype(e_c)::value % 2;
    Pack<T, 2> x[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      const unsigned two = xr[i][j][word];
      x[j] = __builtin_bit_cast(Pack<T, 2>, two);
    }
    row_input_channel(x, e);
#pragma unroll
    for (int t = 0; t < 6; ++t) xr[i][t][word] = __builtin_bit_cast(unsigned, x[t]);
  };
  const int vst = v_offset(tid >> 2, tid & 3);       // THREADS / 4 rows further on, the chunk has the same position
  auto store_v = [&](int i, int t, int buf) {
    *reinterpret_cast<u32x4*>(lds + buf * BUF + vst + i * (THREADS / 4) * kRowPitch + t * TS) = xr[i][t];
  };

  auto tile_of = [&](int i, int& iw, int& ih, int& id, int& in) {
    const int q1 = fast_div(i, a.f_bw), q2 = fast_div(q1, a.f_bh);
    iw = i - q1 * a.bw; ih = q1 - q2 * a.bh;
    in = fast_div(q2, a.f_bd); id = q2 - in * a.bd;
  };

  // ---- LDS address of this lane's tile in each 32-tile block
  int vo[TB];            // in rows
#pragma unroll
  for (int b = 0; b < TB; ++b) {
    int i = b * 32 + (lane & 31);
    if (i >= a.bn * a.bd * a.bh * a.bw) i = 0;
    int iw, ih, id, in;
    tile_of(i, iw, ih, id, in);
    vo[b] = in * a.irow + id * a.prow + ih * lw + iw;
  }

  f32x16 acc[3][TB];
  cut_x(0);
#pragma unroll
  for (int i = 0; i < UN; ++i)
#pragma unroll
    for (int j = 0; j < 6; ++j) load_x(i, j, 0);
  for (;;) {                             // a box (not STAY: the only one); its first input is under way
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[t][b][e] = 0.f;
    u_base = min(kb * KG + kg, k_blocks - 1) * n_groups * 6144;
    cut_x(1);
    // Loads return in order and the compiler counts them over both ways into the loop: the order of the loads here is that of
    // a step, the input of step 1 ahead of the filter's later groups, or every step would wait for its last loads.
    auto load_u_groups = [&](int from, int to) {
#pragma unroll
      for (int i = from; i < to; ++i) load_u(i / 3, i / 3, i % 3);
    };
    load_u_groups(0, UD * 3 / 2);
    shift_x(0);
    static_for<0, 8 * UN>([&](auto h_c) { transform_channel(ic<decltype(h_c)::value / 8>{}, ic<decltype(h_c)::value % 8>{}); });
#pragma unroll
    for (int i = 0; i < UN; ++i) {
#pragma unroll
      for (int t = 0; t < 6; ++t) store_v(i, t, 0);
#pragma unroll
      for (int j = 0; j < 6; ++j) load_x(i, j, 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    load_u_groups(UD * 3 / 2, UD * 3 - 1);           // the last one: in item 0
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();

    for (int step = 0; step < a.local_steps; ++step) {
      const int cur = (step & 1) * BUF + tg * 3 * TS;
      if constexpr (R > 3) {               // keeps the compiler from holding the addresses of all taps in registers
#pragma unroll
        for (int b = 0; b < TB; ++b) asm volatile("" : "+v"(vo[b]));
      }
      cut_x(step + 2);
      shift_x(step + 1);
      u32x4 vf[VD][TB];
      auto load_v = [&](int item) {                  // element item % 3 of group item / 3
        const int q = item / 3, r = (q >> 1) / KP, off = (r / KH) * a.prow + r % KH * lw + (q >> 1) % KP;
#pragma unroll
        for (int b = 0; b < TB; ++b)
          vf[item % VD][b] = *reinterpret_cast<const u32x4*>(lds + cur + v_offset(vo[b] + off, (lane >> 5) + (q & 1) * 2) + item % 3 * TS);
      };
      // A step is a stream of items, one element of one group each.  The loads that refill the rings, the transform of the
      // next step's input, its stores to LDS and the loads of the step after are dealt out over the items and, in an item,
      // over its MFMAs: a wavefront issues in order, and what stands between two MFMAs beyond the 32 cycles of the first
      // leaves the matrix core idle.
#pragma unroll
      for (int i = 0; i < VD - 1; ++i) load_v(i);
      static_for<0, NI>([&](auto item_c) {
        constexpr int item = decltype(item_c)::value, q = item / 3, t = item % 3, last = (item + NI - 1) % NI;
        constexpr int channels = RowItems<UN, NI>::channels(item), moves = RowItems<UN, NI>::moves(item);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (item + VD - 1 < NI) load_v(item + VD - 1);
#pragma unroll
        for (int b = 0; b < TB; ++b)
          acc[t][b] = MfmaRow<T>::run(__builtin_bit_cast(Frag, uf[q % UD][t]), __builtin_bit_cast(Frag, vf[item % VD][b]), acc[t][b]);
        // the ring slot of the item before: its fragment of UD groups later
        load_u(last / 3 % UD, step * Q + last / 3 + UD - (item == 0 ? Q : 0), last % 3);
        static_for<0, channels>([&](auto n_c) {
          constexpr int h = RowItems<UN, NI>::first_channel(item) + decltype(n_c)::value;
          transform_channel(ic<h / 8>{}, ic<h % 8>{});
        });
        static_for<0, moves>([&](auto n_c) {
          constexpr int v = RowItems<UN, NI>::first_move(item) + decltype(n_c)::value;
          store_v(v / 6, v % 6, (step + 1) & 1);
          load_x(v / 6, v % 6, step + 2);
        });
        __builtin_amdgcn_sched_group_barrier(0x100, TB, 0);
#pragma unroll
        for (int g = 0; g < TB; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, (14 * channels + 3 + TB - 1) / TB, 0);
          __builtin_amdgcn_sched_group_barrier(0x200, (moves + TB - 1) / TB, 0);
          __builtin_amdgcn_sched_group_barrier(0x20, (moves + TB) / TB, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
    }

    if constexpr (CS > 1) {                // the shares' sums come together in the first share's registers
      f32x4* part = reinterpret_cast<f32x4*>(lds_all) + lane;
      constexpr int NV = 3 * TB * 4;
      if (cs > 0) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          const f32x16& c = acc[v / 4 % 3][v / 12];
          f32x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = c[v % 4 * 4 + e];
          part[(((cs - 1) * 2 * KG + wave) * NV + v) * 64] = o;
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      if (cs == 0) {
#pragma unroll
        for (int o = 0; o < CS - 1; ++o)
#pragma unroll
          for (int v = 0; v < NV; ++v) {
            const f32x4 p = part[((o * 2 * KG + wave) * NV + v) * 64];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[v / 4 % 3][v / 12][v % 4 * 4 + e] += p[e];
          }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      if (cs > 0) {                        // the barrier of the output transform below
        __builtin_amdgcn_s_barrier();
        return;
      }
    }

    // ---- output transform.  Elements 0 to 2 (points 0, a, -a) are with the first half of the wavefronts, 3 to 5 (1/a,
    // -1/a, infinity) with the second; each half finishes one half of the outputs (two blocks: a block each; one block: half
    // of its channels each) and hands three sums of the other half over through LDS.
    // Each wavefront reduces its three elements to (x, s, d): the element at 0 or infinity, and sum and difference of the pair.
    const int at_kb = kb, at_n = n0, at_d = d0, at_h = h0, at_w = w0;
    bool more = false;
    if constexpr (STAY) {                  // the next box's input comes while this one is written out
      place += gridDim.x / kXcds;
      more = place < places;
      if (more) {
        go_to_box();
        find_x();
        cut_x(0);
#pragma unroll
        for (int i = 0; i < UN; ++i)
#pragma unroll
          for (int j = 0; j < 6; ++j) load_x(i, j, 0);
      }
    }
    constexpr int NC = TB;              // chunks of 8 accumulator registers a wavefront finishes
    auto finish = [&](auto tg_c) {
      constexpr int TG = decltype(tg_c)::value, X = TG == 0 ? 0 : 2, P0 = TG == 0 ? 1 : 0;
      // chunk c of a half: tile block, first register
      auto tile_block = [](int half, int c) { return (half * TB + c) / 2; };
      auto first = [](int half, int c) { return (half * TB + c) % 2 * 8; };
      auto reg = [&](int t, int half, int c, int e) -> float { return acc[t][tile_block(half, c)][first(half, c) + e]; };
      f32x4* ex = reinterpret_cast<f32x4*>(lds) + (size_t)(TG * KG + kg) * 6 * NC * 64 + lane;
      const f32x4* other = reinterpret_cast<const f32x4*>(lds) + (size_t)((1 - TG) * KG + kg) * 6 * NC * 64 + lane;
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i4 = 0; i4 < 2; ++i4) {
          f32x4 x, s, d;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float p = reg(P0, 1 - TG, c, i4 * 4 + e), m = reg(P0 + 1, 1 - TG, c, i4 * 4 + e);
            x[e] = reg(X, 1 - TG, c, i4 * 4 + e); s[e] = p + m; d[e] = p - m;
          }
          ex[((c * 2 + i4) * 3 + 0) * 64] = x; ex[((c * 2 + i4) * 3 + 1) * 64] = s; ex[((c * 2 + i4) * 3 + 2) * 64] = d;
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int k0 = (at_kb * KG + kg) * 32 + (lane >> 5) * 16 + first(TG, c);
        const int ti = tile_block(TG, c) * 32 + (lane & 31);
        int iw, ih, id, in;
        tile_of(ti, iw, ih, id, in);
        const int n = at_n + in, od = at_d + id, oh = at_h + ih, ow = (at_w + iw) * OUT;
        const bool ok = ti < a.bn * a.bd * a.bh * a.bw && n < a.N && od < a.oD && oh < a.oH && k0 < a.K;
        T* const yp = static_cast<T*>(a.y) + ((((size_t)n * a.oD + od) * a.oH + oh) * a.oW + ow) * a.K + k0;
        const T* const bp = static_cast<const T*>(a.bias);
        Pack<T, 8> bv, o[OUT];
#pragma unroll
        for (int e = 0; e < 8; ++e) bv.v[e] = T(0);
        if (bp) {
          if constexpr (!ANY) {
            __builtin_memcpy(&bv, bp + min(k0, a.K - 8), 16);
          } else if (k0 + 8 <= a.K) {
            __builtin_memcpy(&bv, bp + k0, 16);
          } else {
#pragma unroll
            for (int e = 0; e < 7; ++e)
              if (k0 + e < a.K) bv.v[e] = bp[k0 + e];
          }
        }
#pragma unroll
        for (int i4 = 0; i4 < 2; ++i4) {
          f32x4 g[3];
#pragma unroll
          for (int j = 0; j < 3; ++j) g[j] = other[((c * 2 + i4) * 3 + j) * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = i4 * 4 + e;
            const float p = reg(P0, TG, c, i), m = reg(P0 + 1, TG, c, i), x = reg(X, TG, c, i), b = static_cast<float>(bv.v[i]);
            const float m0 = TG == 0 ? x : g[0][e], mi = TG == 0 ? g[0][e] : x;
            const float sa = TG == 0 ? p + m : g[1][e], sb = TG == 0 ? g[1][e] : p + m;
            const float da = TG == 0 ? p - m : g[2][e], db = TG == 0 ? g[2][e] : p - m;
            const RowOutputs<OUT> out = row_outputs<OUT>(m0, sa, da, mi, sb, db, b);
#pragma unroll
            for (int j = 0; j < OUT; ++j) o[j].v[i] = static_cast<T>(out.o[j]);
          }
        }
#pragma unroll
        for (int i = 0; i < OUT; ++i) {
          T* const dst = yp + (size_t)i * a.K;
          const bool in_row = ok && ow + i < a.oW;
          if constexpr (!ANY) {
            if (in_row) *reinterpret_cast<u32x4*>(dst) = __builtin_bit_cast(u32x4, o[i]);
          } else {
            if (in_row && k0 + 8 <= a.K) {
              __builtin_memcpy(dst, &o[i], 16);          // rows of y start at any multiple of the element size
            } else if (in_row) {
              store_some(dst, __builtin_bit_cast(u32x4, o[i]), a.K - k0);
            }
          }
        }
      }
    };
    if (tg == 0) finish(ic<0>{});
    else finish(ic<1>{});
    if (!more) return;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();          // the sums handed over have been read: LDS is free for the next box
  }
}

// ---- U[k / 32][channel block][row tap][half][element][lane][8]: the order in which the wavefronts read it.  Lane l holds
// row l % 32 of a 32 x 16 fragment, channels 8 (l / 32) .. + 8 of the half; row 8 i + 4 h + j of a block is output channel
// 16 h + 4 i + j, which puts 16 consecutive channels of a tile into the accumulators of a lane.
struct RowFilterArgs {
  const void* w; void* U;
  long long s[5];
  int K, C, kd, kh, steps;
  long long total;
};

// The taps of a row are compile-time: counted at run time they cost a call that transforms 512 x 512 channels of 3x3 0.8 of 23 us
template <typename T, int KW>
__global__ __launch_bounds__(256) void row_filter_kernel(RowFilterArgs a) {
  constexpr int P = row_pieces(KW), G = KW == 7 ? 4 : KW;      // 7 taps: 0 to 2 and 3 to 6, as four each
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.total) return;
  const int R = a.kd * a.kh * P;
  const int e2 = (int)(idx & 3) * 2;
  const int lane = (int)(idx >> 2) & 63;
  long long q = idx >> 8;
  const int half = (int)(q & 1); q >>= 1;
  const int r = (int)(q % R); q /= R;
  const int step = (int)(q % a.steps);
  const int kb = (int)(q / a.steps);
  const int m = lane & 31;
  const int k = kb * 32 + ((m >> 2) & 1) * 16 + (m >> 3) * 4 + (m & 3);
  const int c = step * 32 + half * 16 + (lane >> 5) * 8 + e2;
  const int piece = r % P, rr = r / P, rd = rr / a.kh, rh = rr - rd * a.kh;
  Pack<T, 2> out[6];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    float g[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    if (k < a.K && c + e < a.C) {
      const T* p = static_cast<const T*>(a.w) + k * a.s[0] + (c + e) * a.s[1] + rd * a.s[2] + rh * a.s[3] + piece * 3 * a.s[4];
#pragma unroll
      for (int j = 0; j < G; ++j)
        if (KW != 7 || j < 3 + piece) g[j] = static_cast<float>(p[j * a.s[4]]);
    }
    const RowPair a2 = row_filter_pair(g[0], g[1], g[2], g[3], g[4], kA, kA2, kRowFa), b2 = row_filter_pair(g[0], g[1], g[2], g[3], g[4], kB, kB2, kRowFb);
    out[0].v[e] = static_cast<T>(g[0]);
    out[1].v[e] = static_cast<T>(a2.plus);
    out[2].v[e] = static_cast<T>(a2.minus);
    out[3].v[e] = static_cast<T>(b2.plus);
    out[4].v[e] = static_cast<T>(b2.minus);
    out[5].v[e] = static_cast<T>(g[G - 1]);
  }
  T* dst = static_cast<T*>(a.U) + ((idx >> 8) * 6) * 512 + lane * 8 + e2;
#pragma unroll
  for (int t = 0; t < 6; ++t) *reinterpret_cast<Pack<T, 2>*>(dst + t * 512) = out[t];
}

}  // namespace

// Box of a workgroup: at most `tiles` tiles whose input rows, with the halo of the taps, fill at most `slots` rows of LDS;
// the fewest boxes over the output, and among those the fewest rows.  Fragment reads take the tiles of a box in order, which
// is free of bank conflicts where their rows are consecutive modulo 16 (the period of v_offset).  Planes and images are padded
// to row counts that continue the count of their tiles across the halo modulo 8, which leaves reads whose sixteen lanes
// cross an image or a plane 8 rows off: two cycles.  So do the lanes of a block that has fewer than 32 tiles, which all read
// tile 0.  Cycles for the conflict-free number of them, per pass over the taps: N=64, 56x56 (4 images of 8 rows x 2 tiles) 24
// for 12, 14x14 (14 rows x 4 tiles) 18 for 12, 28x28 15 for 12, 16x56x56 (4 planes of 14 rows x 1 tile) 72 for 36, N=1 7x7 6 for
// 6; counted by SQ_LDS_BANK_CONFLICT at N=64 256 -> 256, 56x56: 14.45 M of 36.1 M cycles of the LDS.
RowBox choose_box(int N, int oD, int oH, int nW, int kd, int kh, int tiles, int slots) {
  RowBox best{};
  long long best_rows = 0;
  auto padded = [](int rows, int like) { return rows + ((like - rows) & 7); };
  for (int bw = 1; bw <= tiles && bw <= nW; ++bw)
    for (int bd = 1; bd * bw <= tiles && bd <= oD; ++bd)
      for (int bh = 1; bh * bd * bw <= tiles && bh <= oH; ++bh) {
        RowBox b;
        const int plane = (bw + row_pieces(kh) - 1) * (bh + kh - 1);
        b.prow = bd > 1 ? padded(plane, bw * bh) : plane;
        const int image = (bd + kd - 2) * b.prow + plane, image_p = padded(image, bd * bh * bw);
        if (image > slots) break;
        const int bn = std::min(std::min(tiles / (bw * bd * bh), (slots - image) / image_p + 1), N);
        b.irow = image_p;
        b.bn = bn; b.bd = bd; b.bh = bh; b.bw = bw;
        b.n_n = ceil_div(N, bn); b.n_d = ceil_div(oD, bd); b.n_h = ceil_div(oH, bh); b.n_w = ceil_div(nW, bw);
        b.boxes = (long long)b.n_n * b.n_d * b.n_h * b.n_w;
        const long long rows = b.boxes * (image * bn * 16 - bw);      // wide boxes: neighbouring tiles share two of their six pixels
        if (!best.boxes || b.boxes < best.boxes || (b.boxes == best.boxes && rows < best_rows)) { best = b; best_rows = rows; }
      }
  return best;
}

namespace {

// The shapes of workgroup, by what fills the chip.  Measured, fp16, us (wide, a workgroup per box | half | small | split):
//   wide   eight wavefronts, 64 tiles x 128 channels, one workgroup per CU: every byte of V is used for 128 channels
//   half   four, 64 tiles x 64 channels, two per CU: the transform of one runs beside the products of the other, finer rounds
//   small  four, 32 tiles x 64 channels: more workgroups, shorter steps
//   split  eight, 32 tiles x 32 channels, the channel blocks shared out over four pairs of wavefronts
// N=64: 256 -> 256 channels, 56x56 188 | 190 | 231, 14x14 22 | 17 | 20; 128 -> 128, 28x28 17.2 | 18.0 | 22.5, 56x56
// 68 | 60 | 74; N=16, 256 -> 256, 14x14 21 | 15 | 12.4 | 10.6; N=1, 512 -> 512, 7x7 33 | 22 | 19 | 12.  (Layers of up to 128 input
// channels come here in 3-D or with tile 4; with tile 2 the one-kernel F(2x2, 3x3) form takes most of them, see row_preferred.)
enum RowShape { kRowWide, kRowHalf, kRowSmall, kRowSplit };
// tall_planes: output planes, images in 2-D, that go to tall boxes; the rest is rest_n images of rest_d planes.  few: the workgroups
// where all goes in boxes of few tiles instead (conv_row_few.hip), of few_box, else 0
struct RowPlan { RowShape shape; RowBox box, few_box; long long wide_groups; int tall_planes, rest_n, rest_d, few; double us; };

//
// How long a launch of each takes, in units of a full round of the wide shape, fitted to 330 layers drawn over 1 to 64 images, 32 to 512 channels and
// 7 to 112 rows (3-D: 1 to 8, 32 to 128, 14 to 56; three boxes in four are no whole rounds), each timed in every shape.  Steps of a line are
// where a CU's workgroups change their number: half boxes are two to a CU (one in 3-D, whose boxes take all of its LDS), small ones three.
// Over 300 layers drawn anew the choice takes 1.6 % longer than the fastest shape of each in the mean, with a line through the origin for
// half boxes, and small ones up to one a CU only, 3.2 %.  fp16, us, wide | half | small: 280 half boxes of 7 steps 25.2 | 25.9 |
// 21.0, 252 of 7 steps 22.5 | 16.7 | 21.4; 3-D, 280 of 2 steps 18.0 | 26.2 | 20.6, 160 17.7 | 25.2 | 27.9 (two rounds of half boxes, one of wide
// ones).  Half boxes of 5x5 filters, one a CU, against two small ones, of 4 and more steps: 0.43 to 0.50 of a unit in 29 layers of 130 to 256 half
// boxes, the faster in each (0.58, fitted to boxes of any number, took small ones from 7 steps on): 4 steps 12.6 | 14.7, 6 16.5 | 19.5, 7 17.7 | 21.8
// (195 boxes) and 18.6 | 23.8 (231), 8 19.3 | 24.3.
struct RowModel { double wide, wide_round, half, half_two, half_more, half_at, half_step, small_two, small_three, small_more; };
constexpr RowModel kRow3x3{0.86, 0.92, 0.60, 0.97, 1.27, 1.0, 0.12, 1.6, 2.1, 0.82}, kRow5x5{0.82, 0.80, 0.46, 0.75, 1.15, 0.85, 0.10, 1.25, 1.7, 0.68},
    kRow3d{0.78, 0.72, 0.53, 1.06, 0.0, 0.0, 0.0, 1.2, 1.7, 0.60};

RowPlan make_row_shape(int N, int oD, int oH, int nW, int kd, int kh, int K, int steps) {
  RowPlan p{};
  const RowBox wide = choose_box(N, oD, oH, nW, kd, kh, 64, 128), half = kd == 1 ? choose_box(N, oD, oH, nW, kd, kh, 64, 64) : wide;
  const RowBox small = choose_box(N, oD, oH, nW, kd, kh, 32, 64);
  const long long n_wide = wide.boxes * ceil_div(K, 128), n_half = half.boxes * ceil_div(K, 64), n_small = small.boxes * ceil_div(K, 64);
  auto rounds = [](long long n) { return (double)((n + kCus - 1) / kCus); };
  auto take = [&](RowShape shape, const RowBox& box, double us) {
    if (p.us == 0.0 || us < p.us) { p.shape = shape; p.box = box; p.us = us; }
  };
  p.wide_groups = n_wide;
  if (kh == 7) {
    // Seven rows' halo leaves 64 tiles all of a wide workgroup's LDS, 32 a third of a CU's (kRowSmall) or, with the channels in
    // two shares, two thirds (kRowSplit), which alone in a round is the fastest.  Else whole rounds of each, of 470 layers drawn over 1 to 64 images, 24
    // to 512 channels and 7 to 112 rows, each timed in every shape: 0.15 % over the fastest in the mean (0.16 and 0.14 % on the halves that the
    // lines were and were not fitted to; 0.2 % measured on 200 others), a line without rounds for small boxes and split ones for K <= 32 alone 1.4 %.  fp16, us, wide | small | split:
    // N=51 96 -> 192, 23x25 67 | 71 | 121, N=26 296 -> 54, 32x38 78 | 105 | 110, N=32 43 -> 29, 28x73 41 | 31 | 37, N=5 501 -> 150, 58x25 126 | 117 | 75, N=6
    // 100 -> 150, 45x61 46 | 52 | 53, N=32 128 -> 128, 112x112 421 | 600 | 802, N=1 512 -> 512, 14x14 117 | 55 | 33.
    const long long n_split = small.boxes * ceil_div(K, 32);
    if (steps < 2 || n_split > kCus) {
      take(kRowWide, wide, rounds(n_wide) * (std::min(10.5, 7 + 3.5 * n_wide / kCus) * steps + 6));
      take(kRowSmall, small, rounds(n_small) * (3.6 * steps + 2));
    }
    if (steps >= 2) take(kRowSplit, small, rounds(n_split) * (2.3 * steps + 6));
    return p;
  }
  const double us_small = 0.4 * steps * kd * kh + 4, unit = ((kd == 1 ? 0.82 * kh : 6.9) * steps + 7) / 0.92;
  if (steps >= 4) {
    const RowBox split = choose_box(N, oD, oH, nW, kd, kh, 32, 32);
    if (split.boxes * ceil_div(K, 32) <= kCus) { take(kRowSplit, split, us_small); return p; }
  }
  if (n_small <= kCus) { take(kRowSmall, small, us_small); return p; }
  const RowModel& m = kd == 3 ? kRow3d : kh == 5 ? kRow5x5 : kRow3x3;
  // (seven whole rounds of 3-D boxes, N=8 128 -> 128, 16x56x56, took 0.84 of a unit each)
  take(kRowWide, wide, unit * (n_wide <= kCus ? m.wide : (kd == 3 && n_wide > 4 * kCus ? 0.86 : m.wide_round) * rounds(n_wide)));
  take(kRowHalf, half, unit * (n_half <= kCus ? m.half : kd == 3 ? m.half * rounds(n_half) : n_half <= 2 * kCus ? m.half_two
                               : std::max(m.half_more, m.half_at * n_half / (2.0 * kCus) + m.half_step)));
  take(kRowSmall, small, us_small * (n_small <= 2 * kCus ? m.small_two : n_small <= 3 * kCus ? m.small_three : m.small_more * n_small / kCus));
  return p;
}

// The first `tall_planes` of a batch in tall boxes (conv_row_tall.hip), the rest in the shape above.  A tall box takes the CU
// that has it 2.1 us per 16 channels and plane of taps and 10.5 beside them, so a batch is worth cutting where its last round
// would be nearly empty: N=64 256 -> 256 channels, 56x56 has 784 boxes, three rounds and sixteen boxes; 61 images fill the
// three and the other three images take 12 us.  A 3-D batch is cut within its last image (N=8 128 -> 128, 16x56x56, 756 of 784 boxes
// hold 123 of 128 planes, 3 rounds, the other 5 planes 20 us; seven images and one were 3 rounds of 686 boxes and 37 us).  The
// model's constants are measured ones (fp16, us, this shape alone in whole rounds | a box: 512 -> 512, 28x28 157 | 78 for 32 half
// blocks, 256 -> 256, 56x56 175 | 44 for 16).
//
// copied: x comes with channels padded to a multiple of 8
RowPlan make_row_plan(int N, int oD, int oH, int nW, int kd, int kh, int K, int C, bool copied) {
  const int steps = ceil_div(C, 32);
  RowPlan best = make_row_shape(N, oD, oH, nW, kd, kh, K, steps);
  best.rest_n = N; best.rest_d = oD;
  best.few = row_few_workgroups((long long)N * oD, oH, nW, kd, kh, K, C, copied, &best.few_box);
  if (kh != 3 || best.few) return best;
  const double box_us = 2.1 * 2 * steps * kd + 10.5;
  // Tall boxes read padded rows.  What their copy takes between two layers that differ by it alone, over 109 layers: tall boxes and the others are
  // chosen with 0.1 % lost in the mean (at 3 us and 9 TB/s 0.4 %: N=31 175 -> 232, 66x25 52 us, 47 in wide boxes).  Where x is copied in any case
  // (channel-first) the other boxes find the copy in L2 and are ahead by less of it: without a price the same mean, but N=27 105 -> 144, 83x37 48 | 56 us.
  const double bytes = N * (double)oD * oH * nW * 4 * C * 4, copy_us = C % 8 == 0 ? 0 : copied ? 3 + bytes / 9e6 : 5 + bytes / 7e6;
  const long long per_group = (long long)ceil_div(oH, 4) * ceil_div(K, 128), planes = (long long)N * oD;
  const long long boxes = ceil_div_ll(planes * nW, 32) * per_group;
  const long long groups = boxes / kCus * kCus / per_group;       // groups of 32 columns in whole rounds
  long long cut = std::min(groups * 32 / nW, planes - 1);
  if (planes - cut > oD) cut = cut / oD * oD;                     // the rest: whole images, or planes of the last one
  const double wide_groups = best.wide_groups;
  for (const long long n : {planes, cut}) {
    if (n < 1) continue;
    RowPlan p{};
    const long long rest = planes - n;
    if (rest > 0) {
      const int rest_n = (int)ceil_div_ll(rest, oD), rest_d = rest_n > 1 ? oD : (int)rest;
      p = make_row_shape(rest_n, rest_d, oH, nW, kd, kh, K, steps);
      p.rest_n = rest_n; p.rest_d = rest_d;
    }
    const long long rounds = ceil_div_ll(ceil_div_ll(n * nW, 32) * per_group, kCus);
    p.us += rounds * box_us + (rest > 0 ? 2 : 0) + copy_us;
    p.tall_planes = (int)n;
    if (p.us < best.us) best = p;
  }
  best.wide_groups = (long long)wide_groups;
  return best;
}

// The search over boxes takes some microseconds: the last plans of a host thread are kept.
RowPlan row_plan(int N, int oD, int oH, int nW, int kd, int kh, int K, int C, bool copied = false) {
  struct Entry { int key[9]; RowPlan plan; };
  thread_local Entry cache[64] = {};
  const int key[9] = {N, oD, oH, nW, kd, kh, K, C, copied};
  unsigned h = 2166136261u;
  for (int v : key) h = (h ^ (unsigned)v) * 16777619u;
  Entry& e = cache[(h ^ (h >> 15)) % 64];
  if (!std::equal(key, key + 9, e.key)) {
    e.plan = make_row_plan(N, oD, oH, nW, kd, kh, K, C, copied);
    std::copy(key, key + 9, e.key);
  }
  return e.plan;
}

// Filters that overflow an XCD's 4 MB of L2: its workgroups work on one channel block at a time
bool filter_fits_l2(const RowArgs& a) { return a.u_bytes <= (3 << 20); }

template <typename T, int KD, int KH, int KG, int TB, int S, int CS = 1, bool STAY = false>
int launch_row(const RowArgs& args, const RowBox& b, void* stream) {
  RowArgs a = args;
  a.bn = b.bn; a.bd = b.bd; a.bh = b.bh; a.bw = b.bw; a.lw = b.bw + row_pieces(KH) - 1; a.prow = b.prow; a.irow = b.irow;
  a.f_bw = make_fast_div(b.bw); a.f_bh = make_fast_div(b.bh); a.f_bd = make_fast_div(b.bd);
  a.f_lw = make_fast_div(a.lw); a.f_prow = make_fast_div(b.prow); a.f_irow = make_fast_div(b.irow);
  a.n_d = b.n_d; a.n_h = b.n_h; a.n_w = b.n_w;
  a.n_box = (int)b.boxes;
  a.local_steps = ceil_div(a.steps, CS);
  a.n_kb = ceil_div(a.K, 32 * KG);
  a.box_fast = !filter_fits_l2(a);
  a.per_xcd = ceil_div(a.n_kb * a.n_box, kXcds);
  constexpr int bytes = row_lds_bytes<KG, TB, S, CS>();
  const bool whole = a.tail == 0 && a.K % 8 == 0 && (reinterpret_cast<uintptr_t>(a.y) & 15) == 0;
  auto fn = whole ? row_conv_kernel<T, KD, KH, KG, TB, S, CS, STAY, false> : row_conv_kernel<T, KD, KH, KG, TB, S, CS, STAY, true>;
  int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), bytes);
  if (rc) return rc;
  hipLaunchKernelGGL(fn, dim3(STAY ? std::min(a.per_xcd * kXcds, kCus) : a.per_xcd * kXcds), dim3(128 * KG * CS), bytes, as_stream(stream), a);
  WC_CHECK_LAUNCH("row_conv_kernel");
  return WC_OK;
}

}  // namespace

bool row_conv_fits(const wc_conv_desc* d) {
  if (d->dtype == WC_F32 || d->stride != 1 || d->whole_kernel) return false;
  const int kd = d->kernel[0], kh = d->kernel[1], kw = d->kernel[2];
  if (!((kd == 1 && kh == 3 && kw == 3) || (kd == 3 && kh == 3 && kw == 3) || (kd == 1 && (kh == 5 || kh == 7) && kw == kh && d->ndim == 2))) return false;
  const int cp = wc_padded_channels8(d->C);
  for (int q = 0; q < 3; ++q)
    if (d->in[q] + 2 * d->pad[q] < d->kernel[q]) return false;
  const long long out = (long long)d->N * (d->in[0] + 2 * d->pad[0] - kd + 1) * (d->in[1] + 2 * d->pad[1] - kh + 1) *
                        (d->in[2] + 2 * d->pad[2] - kw + 1);
  return (long long)d->N * d->in[0] * d->in[1] * d->in[2] * cp * 2 < (1ll << 30) && out < (1ll << 31) &&
         row_u_elems(d) * 2 < (1ull << 30);
}

size_t row_u_elems(const wc_conv_desc* d) {
  return (size_t)ceil_div(d->K, 32) * ceil_div(d->C, 32) * d->kernel[0] * d->kernel[1] * row_pieces(d->kernel[1]) * 2 * 6 * 512;
}

int row_filter(const wc_conv_desc* d, const void* w, const int64_t w_strides[5], void* U, void* stream) {
  WC_CHECK_ARG(w && w_strides && U, "row form filter: null pointer");
  RowFilterArgs a;
  a.w = w; a.U = U;
  for (int i = 0; i < 5; ++i) a.s[i] = w_strides[i];
  a.K = d->K; a.C = d->C; a.kd = d->kernel[0]; a.kh = d->kernel[1]; a.steps = ceil_div(d->C, 32);
  a.total = (long long)ceil_div(d->K, 32) * a.steps * a.kd * a.kh * row_pieces(d->kernel[2]) * 2 * 256;
  const unsigned blocks = (unsigned)ceil_div_ll(a.total, 256);
  auto launch = [&](auto kw) {
    const auto fn = d->dtype == WC_F16 ? &row_filter_kernel<half_t, decltype(kw)::value> : &row_filter_kernel<bf16_t, decltype(kw)::value>;
    hipLaunchKernelGGL(fn, dim3(blocks), dim3(256), 0, as_stream(stream), a);
  };
  if (d->kernel[2] == 7) launch(ic<7>{});
  else if (d->kernel[2] == 5) launch(ic<5>{});
  else launch(ic<3>{});
  WC_CHECK_LAUNCH("row_filter_kernel");
  return WC_OK;
}

// 7x7 layers nearly always (row_no_slower_7x7): two of F(3, 4) a row are 28 products per output where pieces sharing a transformed input take 36 on F(2x2, 2x2)
// and 25 on F(3x3, 3x3) (tile 4 in fp16), and the error is smaller than either's (bf16 3.9e-3 | 4.5e-3, fp16 4.8e-4 | 1.5e-3).  us,
// row | other, bf16: N=32 128 -> 128, 112x112 408 | 565, N=16 256 -> 256, 56x56 228 | 319, 64 -> 64 26 | 45, 512 -> 512, 14x14
// 108 | 144, N=6 100 -> 150, 45x61 47 | 72, N=1 128 -> 128, 56x56 12 | 30, 32 -> 32, 14x14 7.5 | 15; fp16 with tile 4: 415 | 520,
// 235 | 248, 26 | 40, 108 | 135, 46 | 63, 12 | 24, 7.4 | 12.8.
//
// 5x5 layers: F(2, 5) needs 15 products per output where the plan it replaces, two- or three-tap pieces sharing one
// transformed input, needs 20 on F(2x2, 2x2) and 11 on F(3x3, 3x3) (tile 4 in fp16), without V and M in memory, and is as
// exact as the first (2-norm against fp64, bf16 5.2e-3 | 5.4e-3) and 2.5 times as the second (fp16 6.5e-4 | 1.7e-3).  us, row | other, bf16:
// N=32 128 -> 128, 112x112 246 | 407, N=16 256 -> 256, 56x56 127 | 200, 64 -> 64 15 | 37, 512 -> 512, 14x14 60 | 71, N=6
// 100 -> 150, 45x61 36 | 53, N=1 128 -> 128, 56x56 9 | 22, 64 -> 64, 28x28 7 | 16, 32 -> 32, 14x14 7 | 13; fp16 with tile 4: 248 | 365,
// 131 | 134, 14 | 33, 57 | 62, 35 | 43, 9 | 17, 7 | 13, 7 | 12.  Over more than 256 channels it would replace stacked pieces.  Those of tile
// 2 are slower (us, pieces | row, N=64 512 -> 512, 28x28 649 | 456) but more exact, bf16 4.8e-3 | 5.2e-3, fp16 6.0e-4 | 6.5e-4 over 288 channels (the points are the
// best there are for F(2, 5)), and stay; those of tile 4 are four times less exact (fp16 2.8e-3).
// Layers of 33 to 40 output channels keep the other plan, though it is slower (N=2 64 -> 40, 15x14 7 | 15): no measurement puts a
// line there, tests/test_gpu_row.py and test_gpu_row_5x5_7x7.py take them for 5x5 layers beside the row form.
static bool row_preferred_5x5(const wc_conv_desc* d) {
  if (d->m == 2 && wc_padded_channels(d->C) > 256) return false;
  // fp16 with tile 4: the stacked pieces of F(4x4, .) multiply 9 times per output where F(2, 5) does 15 and are the faster ones where their
  // product runs on whole rounds of persistent tiles and has the output channels to pay for four transformed inputs.  us, row | pieces:
  // 512 -> 512 N=64 56x56 1718 | 1579, 28x28 463 | 416, N=8 56x56 251 | 228, N=64 20x20 260 | 228, 1024 -> 1024 N=32 28x28 922 | 659, 384 -> 768
  // N=64 28x28 523 | 444, 288 -> 512 N=16 56x56 273 | 265, 320 -> 512 N=32 40x40 300 | 303; rounds or tiles short: 512 -> 512 N=24 28x28 199 | 207, N=64 14x14
  // 126 | 175, N=8 60x60 268 | 313, 1024 -> 1024 N=64 14x14 490 | 515; 256 output channels: 512 -> 256 N=32 56x56 461 | 599.
  if (d->m == 4 && d->dtype == WC_F16 && wc_padded_channels(d->C) > 256 && d->K >= 512) {
    const int oH = d->in[1] + 2 * d->pad[1] - 4, oW = d->in[2] + 2 * d->pad[2] - 4;
    if (persistent_pays(36, (long long)d->N * ceil_div(oH, 4) * ceil_div(oW, 4), 4 * wc_padded_channels(d->C), d->K, wc_padded_channels8(d->K), d->dtype)) return false;
  }
  return d->K <= 32 || d->K > 40;
}

// 7x7 layers of fp16 with tile 4 over up to 256 channels: whether the row form takes no longer than the pieces that share one transformed
// input on F(3x3, 3x3), which run on 512 x 128 tiles.  The row form's boxes of 64 tiles take 10.5 us a step of 32 channels and 4
// beside them with all CUs at work, less in a last round that is nearly empty; the pieces, whose error is three times as large, are ahead where
// that round is and theirs is not.  us, row | pieces (this model of both): 256 -> 256, 112x112 N=2 155 | 137 (151 | 139), N=3 164 | 202 (166 | 180), N=4 245 | 227
// (241 | 222), N=8 422 | 404 (422 | 402), N=12 616 | 626 (604 | 624), N=16 801 | 826 (785 | 804); 256 -> 512, N=8 803 | 765 (785 | 764); 256 -> 256, 80x80
// N=8 247 | 229 (241 | 232), 100x100 349 | 367 (345 | 364), 56x56 N=32 421 | 470 (433 | 465), 28x28 N=64 224 | 298 (250 | 304), 14x14 71 | 132; 224 -> 224,
// 112x112 N=8 375 | 365 (372 | 368); 160 -> 256, 100x100 N=5 161 | 152 (158 | 156); 128 -> 128, 112x112 N=32 424 | 528 (410 | 563).
static bool row_no_slower_7x7(const wc_conv_desc* d, const RowPlan& p) {
  if ((p.shape == kRowSplit && p.box.boxes * ceil_div(d->K, 32) <= kCus) || !(d->K % 128 == 0 || d->K % 128 >= 96)) return true;
  const int oH = d->in[1] + 2 * d->pad[1] - 6, oW = d->in[2] + 2 * d->pad[2] - 6, steps = ceil_div(d->C, 32);
  auto rounds = [](long long n, double start, double share) { return n / kCus + (n % kCus ? start + share * (n % kCus) / kCus : 0.0); };
  const long long rows = (long long)d->N * (ceil_div(oH, 3) + 2) * (ceil_div(oW, 3) + 2), tiles = 25 * ceil_div_ll(rows, 512) * ceil_div(d->K, 128);
  const double pieces = 1.02 * (tiles >= 2 * kCus ? rounds(tiles, 0.4, 0.6) : 1.25 * tiles / kCus) * (8 * steps + 8 + 8.0 * 256 / d->K);
  const long long full = p.wide_groups / kCus, rest = p.wide_groups % kCus;
  return full * (10.5 * steps + 4) + (rest ? (7 + 3.5 * rest / kCus) * steps + 4 : 0) <= pieces;
}

// Against the other forms, us (row | other), channels -> channels on P output pixels:
//  * Where tile 2 is asked for (the modules in 3-D and in bfloat16): always.  The row form takes 9/8 (3-D: 27/16) times the products of
//    the F(2, 3) tiles and none of their traffic.  fp16, 3-D: 32 -> 32 on 401408 60 | 107, 64 -> 64 on 50176 14 | 36, 128 -> 128 on 401408
//    229 | 426, 192 -> 192 on 50176 85 | 121, 256 -> 256 on 200704 421 | 555, on 6272 30 | 35, on 3136 22 | 31, 384 -> 384 on
//    50176 237 | 281, 512 -> 512 on 50176 425 | 476, on 12544 114 | 128, on 196 19 | 24; bf16 as fp16.  The exception, 512 -> 512
//    on 16 clips of 2x7x7 (a row of 7 outputs fills two tiles of 4) 44 | 35, stays here for its error: against fp64 in the 2-norm
//    fp16 6.3e-4 | 8.5e-4, bf16 5.1e-3 | 6.8e-3.  bf16, 2-D: 256 -> 256 on 200704 182 | 374, 512 -> 512 on 50176 187 | 225.
//  * Where tile 4 is asked for, whose larger error the caller accepts (fp16 4e-3, bf16 3e-2; 3-D 2x4x4 5e-3, 4e-2), the faster
//    one.  Up to one and a half rounds of the chip the row form's single launch decides (2-D: 512 on 12544 47 | 54, bf16 48 | 53;
//    256 on 12544 17 | 30; 512 on 49 12 | 17; 3-D: 512 on 196 19 | 41, on 6272 70 | 69).  Beyond, F(4x4, 3x3) needs half the products
//    and F(2x4x4, 3x3x3) a third, and they overtake with the channels.  Per pixel they take about 1500 (C + K) + C K units in 2-D,
//    512 (C + K) + C K in 3-D, and the row form 10.5 and 3.6 of them per product of padded channels.  2-D, fp16 (bf16): 256 -> 256
//    on 200704 188 | 219 (182 | 217), 384 on 50176 108 | 111 (112 | 107), 512 on 50176 178 | 140 (187 | 141), 300 -> 200 76 | 67
//    (78 | 64).  3-D, fp16: 128 on 401408 229 | 539, 256 on 200704 421 | 580, 384 on 50176 237 | 260, 512 on 50176 425 | 349,
//    on 25088 212 | 204, on 12544 114 | 114.
//  * Never where the one-kernel F(2x2, 3x3) form runs (conv_thin.hip), though it is up to a third slower on its larger layers
//    (128 -> 128 on 50176 pixels 17 | 25): that form rounds no products either, and its error is the smaller one (fp16 6.2e-4 |
//    6.1e-4, bf16 5.0e-3 | 4.2e-3).
bool row_preferred(const wc_conv_desc* d) {
  wc_plan plan;
  wc_conv_desc e = *d;
  e.stacked = 0; e.direct = 0; e.row = 0;
  if (wc_plan_conv(&e, &plan) == WC_OK && thin_conv_fits(&e, &plan)) return false;
  if (d->kernel[1] == 7) {
    if (d->m != 4 || d->dtype != WC_F16 || wc_padded_channels(d->C) > 256) return true;
    const int oH = d->in[1] + 2 * d->pad[1] - 6, oW = d->in[2] + 2 * d->pad[2] - 6;
    return row_no_slower_7x7(d, row_plan(d->N, 1, oH, ceil_div(oW, 3), 1, 7, d->K, d->C));
  }
  if (d->kernel[1] == 5) return row_preferred_5x5(d);
  if (d->m != 4) return true;
  const int kd = d->kernel[0], oD = d->in[0] + 2 * d->pad[0] - kd + 1, oH = d->in[1] + 2 * d->pad[1] - 2, oW = d->in[2] + 2 * d->pad[2] - 2;
  if (row_plan(d->N, oD, oH, ceil_div(oW, 4), kd, 3, d->K, d->C).wide_groups <= 3 * kCus / 2) return true;
  const double C = d->C, K = d->K, products = (double)wc_padded_channels(d->C) * (ceil_div(d->K, 64) * 64.0);
  return kd == 1 ? 10.5 * products < 1500.0 * (C + K) + C * K : 3.6 * products < 512.0 * (C + K) + C * K;
}

// Whether x has to come with its channels padded to a multiple of 8: tall boxes, whose input goes straight to LDS, and rows of less than 16 bytes
bool row_reads_padded(const wc_conv_desc* d) {
  if (d->C % 8 == 0) return false;
  const int force = test_gemm_config(), kd = d->kernel[0], kh = d->kernel[1];
  if (d->C < 8 || (force == 21 && kh == 3)) return true;
  if (kh != 3 || (force >= 16 && force <= 19) || force == 30) return false;
  return row_plan(d->N, d->in[0] + 2 * d->pad[0] - kd + 1, d->in[1] + 2 * d->pad[1] - 2, ceil_div(d->in[2] + 2 * d->pad[2] - 2, 4), kd, kh, d->K,
                  d->C).tall_planes > 0;
}

static bool takes_few(const RowPlan& plan) {
  const int force = test_gemm_config();
  return force == 30 || (plan.few > 0 && force != 21 && (force < 16 || force > 19));
}

// Whether the layer's one kernel takes this filter as it is, so that nothing has to be transformed before it
bool row_takes_filter(const wc_conv_desc* d, const void* w, const int64_t w_strides[5]) {
  if (!row_conv_fits(d) || d->kernel[1] != 3 || !row_few_takes_filter(d, w, w_strides)) return false;
  const RowPlan plan = row_plan(d->N, d->in[0] + 2 * d->pad[0] - d->kernel[0] + 1, d->in[1] + 2 * d->pad[1] - 2, ceil_div(d->in[2] + 2 * d->pad[2] - 2, 4), d->kernel[0], 3,
                                d->K, d->C);
  return takes_few(plan) && (test_gemm_config() == 30 || row_few_filter_pays(d, plan.few));
}

// x (N, D, H, W, x_row) channel-last: x_row is C, where row_reads_padded allows it, or C rounded up to 8 (zeros beyond C).  Rows of whole 16
// bytes start at a multiple of 16; others, of which a pass's first image starts anywhere, at any element;
// images first_image .. + n_images of the batch.  U null: the filter is w, which row_takes_filter
int row_conv(const wc_conv_desc* d, const void* x, int x_row, int first_image, int n_images, const void* U, const void* bias, void* y, void* stream,
             const void* w, const int64_t* w_strides) {
  WC_CHECK_ARG(row_conv_fits(d), "row form: 16-bit, stride 1, kernels 3x3, 3x3x3, 5x5 and 7x7");
  WC_CHECK_ARG(((x_row % 8 == 0 ? reinterpret_cast<uintptr_t>(x) : 0) | reinterpret_cast<uintptr_t>(U)) % 16 == 0, "row form: x and U must be 16-byte aligned");
  RowArgs a{};
  a.x = x; a.U = U; a.bias = bias; a.y = y;
  a.N = n_images; a.D = d->in[0]; a.H = d->in[1]; a.W = d->in[2]; a.C = wc_padded_channels8(d->C); a.K = d->K;
  a.x_row = x_row; a.tail = a.C - x_row;
  a.pd = d->pad[0]; a.ph = d->pad[1]; a.pw = d->pad[2];
  a.oD = a.D + 2 * a.pd - d->kernel[0] + 1; a.oH = a.H + 2 * a.ph - d->kernel[1] + 1; a.oW = a.W + 2 * a.pw - d->kernel[2] + 1;
  a.nW = ceil_div(a.oW, row_outputs_of(d->kernel[1]));
  a.steps = ceil_div(a.C, 32);
  a.x_bytes = (int)((long long)a.N * a.D * a.H * a.W * a.x_row * 2);
  a.u_bytes = (int)(row_u_elems(d) * 2);
  const int force = test_gemm_config();
  // the shapes are the whole batch's, so that the passes of a batch add in the order of the batch in one pass
  RowPlan plan = row_plan(d->N, a.oD, a.oH, a.nW, d->kernel[0], d->kernel[1], a.K, d->C, x_row != d->C);
  if (force >= 16 && force <= 19) { plan.shape = (RowShape)(force - 16); plan.tall_planes = 0; plan.rest_n = -1; }
  if (force == 21 && d->kernel[1] == 3) plan.tall_planes = d->N * a.oD;
  const int tall = std::min(std::max(plan.tall_planes - first_image * a.oD, 0), n_images * a.oD);
  if (takes_few(plan)) return row_few_conv(d, x, x_row, n_images, plan.few > 0 && n_images == d->N ? &plan.few_box : nullptr, U, w, w_strides, bias, y, stream);
  WC_CHECK_ARG(U, "row form: no transformed filter");
  if (tall > 0) {
    WC_CHECK_ARG(a.tail == 0, "row form: tall boxes of %d channels", x_row);
    const int rc = tall_row_conv(d, x, tall, U, bias, y, stream);
    if (rc || tall == n_images * a.oD) return rc;
    // the rest: the images from there on, of the first of them (the only one then) the planes from there on
    const int images = tall / a.oD, first_d = tall - images * a.oD;
    a.x = static_cast<const unsigned char*>(x) + (long long)images * a.D * a.H * a.W * a.x_row * 2;
    a.y = static_cast<unsigned char*>(y) + (long long)tall * a.oH * a.oW * a.K * 2;
    a.N -= images;
    a.oD -= first_d; a.pd -= first_d;
    a.x_bytes = (int)((long long)a.N * a.D * a.H * a.W * a.x_row * 2);
  }
  return dispatch_dtype(d->dtype, [&](auto t) -> int {
    using T = decltype(t);
    if constexpr (sizeof(T) == 2) {
      auto go = [&](auto kd, auto kh) -> int {
        constexpr int KD = decltype(kd)::value, KH = decltype(kh)::value;
        RowPlan p = plan;
        if (a.N != p.rest_n || a.oD != p.rest_d) {
          const int tiles = p.shape <= kRowHalf ? 64 : 32, slots = KH == 7 ? (tiles == 64 ? 128 : 64) : p.shape == kRowWide ? 128 : p.shape == kRowSplit ? 32 : p.shape == kRowHalf && KD > 1 ? 128 : 64;
          p.box = choose_box(a.N, a.oD, a.oH, a.nW, KD, KH, tiles, slots);
        }
        if constexpr (KH == 7) {
          if (p.shape == kRowSplit) return launch_row<T, KD, KH, 1, 1, 64, 2>(a, p.box, stream);
          if (p.shape == kRowSmall) return launch_row<T, KD, KH, 2, 1, 64>(a, p.box, stream);
          return launch_row<T, KD, KH, 4, 2, 128>(a, p.box, stream);
        } else {
          switch (p.shape) {
            case kRowWide:
              // More boxes than CUs: a workgroup per CU that asks for its next box's input before it writes a box out, which
              // hides that input's way from memory behind the write-out and saves the start of a workgroup.  Measured, fp16, us,
              // a workgroup per box | this: N=64 256 -> 256, 56x56 196 | 185, 128 -> 128, 56x56 71 | 66, 256 -> 256, 28x28 53.3 |
              // 52.0, N=8 128 -> 128, 16x56x56 242 | 239.  Filters beyond an XCD's L2 (box_fast): 512 -> 512, N=16 28x28 48.1 |
              // 49.3.  (Not with the deeper ring of 5x5 kernels, whose registers do not hold the next box beside it.)
              if constexpr (KH == 3) {
                if (filter_fits_l2(a) && ceil_div(a.K, 128) * p.box.boxes > kCus) return launch_row<T, KD, KH, 4, 2, 128, 1, true>(a, p.box, stream);
              }
              return launch_row<T, KD, KH, 4, 2, 128>(a, p.box, stream);
            case kRowHalf: return launch_row<T, KD, KH, 2, 2, KD == 1 ? 64 : 128>(a, p.box, stream);
            case kRowSmall: return launch_row<T, KD, KH, 2, 1, 64>(a, p.box, stream);
            default: return launch_row<T, KD, KH, 1, 1, 32, 4>(a, p.box, stream);
          }
        }
      };
      if (d->kernel[1] == 7) return go(ic<1>{}, ic<7>{});
      if (d->kernel[1] == 5) return go(ic<1>{}, ic<5>{});
      if (d->kernel[0] == 1) return go(ic<1>{}, ic<3>{});
      return go(ic<3>{}, ic<3>{});
    }
    return fail(WC_ERR_UNSUPPORTED, "row form: 16-bit types");
  });
}

}  // namespace wc
