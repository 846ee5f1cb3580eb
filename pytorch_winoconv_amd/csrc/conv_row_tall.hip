// The row form (conv_row.hip) on tall boxes: 32 tiles of a row times four rows times 128 output channels per workgroup, one
// workgroup of eight wavefronts per CU that goes from box to box.
//
// What bounds the wide workgroups of conv_row.hip (64 tiles) is what comes from L2 beside the products: 144 KB of filter for
// 72 products of 32x32x16 per SIMD, 75 KB/us and CU with the input, and every fragment of V is read once per product.  Here a
// filter fragment meets twice the tiles, and the four rows of a wavefront slide over six rows of V, so that a fragment of V
// read once meets up to three taps: six reads for twelve products.  The products of a half block of channels (16) then take
// 24 ns each with all 256 CUs busy, what the matrix cores sustain with changing operands, against 29 with the wide
// workgroup's reads and loads; with the transform and the input from memory 29 (wide: 34).
//
// The 192 accumulators of a wavefront leave 64 registers.  So x does not pass through them: LDS-DMA brings it as it is (ldsX),
// each wavefront its own rows, which need no barrier, and the transform takes it from there in words of two channels, a third
// of the work beside the products of each element.  Tap planes (3-D) lengthen the reduction: x is transformed again for each.
// A box also needs 10.5 us for its output transform and the way back into the products: the registers allow the four parts
// of the exchange no overlap, all CUs write 33 MB at the same time, and the first filter fragments wait behind that.
//
// Measured, fp16, us, wide | tall with its last round cut off (make_row_plan): N=64 256 -> 256 channels, 56x56 199 | 162 (195 | 170 with x from memory),
// 512 -> 512, 28x28 184 | 157, 256 -> 256, 28x28 51.5 | 45, N=32 256 -> 384, 56x56 139 | 128, N=8 128 -> 128, 16x56x56 236 | 230.
#include "row_form.h"

#include <algorithm>

namespace wc {

namespace {

struct TallArgs {
  const void* x; const void* U; const void* bias; void* y;
  int N, D, H, W, C, K;           // x (N, D, H, W, C), y (N, oD, oH, oW, K)
  int oD, oH, oW, nW;             // nW tiles of 4 outputs per row
  int pd, ph, pw, kd;
  int n_col;                      // columns: tiles of a row of every plane of every image, N oD nW
  FastDiv f_w, f_d;               // by nW, by oD
  int n_cg, n_hb, n_kb;           // groups of 32 columns, of four rows, of 128 channels
  int n_box, per_xcd, box_fast;   // n_cg n_hb; box_fast 1: neighbouring workgroups share a channel block, 0: a box
  int cblocks;                    // ceil(C / 32)
  int x_bytes, u_bytes;
};

constexpr int TB = 4, ROWS = TB + 2;
constexpr int kVBuf = 6 * ROWS * 1024;             // six elements of six rows of 32 tiles, 16 channels
constexpr int kRawWave = 3 * 3 * 1024;             // three rows of 8 tiles, six pixels each, 32 channels
constexpr int kExWave = 6 * 1024;                  // what a wavefront hands over at a time in the output transform

// Where the transform of a half block of input stands in the 18 positions of a half step: three units of three positions
// (read, first channel, second channel and store; in half 0 the unit's next loads as well).  Loads return in order, so the
// first filter fragments behind a wavefront's input loads wait for memory: the two wavefronts of a SIMD (one of each half of
// the elements) load in different parts of the step, and one multiplies while the other waits.
struct TallBeside {
  static constexpr int read(int half, int u) { return half == 0 ? 4 * u : 4 + 4 * u; }
  static constexpr int filter_loads(int from, int to) {       // issued at positions from .. to - 1 of the two halves: three each behind 5, 11, 17
    int n = 0;
    for (int p = from; p < to; ++p) n += p % ROWS == ROWS - 1 ? 3 : 0;
    return n;
  }
  // issued between the last load of unit u in half 0 and its read in half 1 (position 17's filter fragments are behind its loads)
  static constexpr int after_loads(int u) {
    return filter_loads(read(0, u) + 3, 3 * ROWS + read(1, u)) + 3 * (2 - u);
  }
};

// The lane, computed on the spot: where the registers are full a kept one is spilled
__device__ __forceinline__ int lane_id() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(l));
  return l;
}

// KT: rows of y that are no multiple of 16 bytes, or a y or bias that starts elsewhere than at one (a view into another tensor)
template <typename T, int UR, bool KT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void tall_row_kernel(TallArgs a) {
  using Frag = typename MfmaRow<T>::Frag;
  __shared__ __attribute__((aligned(1024))) unsigned char ldsV[kVBuf + std::max(kVBuf, 8 * kExWave)];
  __shared__ __attribute__((aligned(1024))) unsigned char ldsX[8 * kRawWave];
  int place = blockIdx.x / kXcds;
  const int place0 = blockIdx.x % kXcds * a.per_xcd, places = min(a.per_xcd, a.n_kb * a.n_box - place0);
  if (place >= places) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tg = wave >> 2, kg = wave & 3;
  int kb, c0, h0;
  auto go_to_box = [&]() {
    const int wg = place0 + place;
    int box;
    if (a.box_fast) { kb = wg / a.n_box; box = wg - kb * a.n_box; }
    else { box = wg / a.n_kb; kb = wg - box * a.n_kb; }
    const int cg = box / a.n_hb;
    c0 = cg * 32; h0 = (box - cg * a.n_hb) * TB;
  };
  const __amdgpu_buffer_rsrc_t xdesc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.x), 0, a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t udesc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.U), 0, a.u_bytes, 0x00020000);

  // ---- input: this wavefront brings 8 tiles (its columns) of three rows into its own part of ldsX and transforms them.
  // A load: two of the six pixels of the 8 tiles, 32 channels: lane = pixel * 32 + tile * 4 + chunk of 16 bytes; tiles 4 to 7
  // have their two halves of 16 channels exchanged, so that the reads of a half meet every bank once.
  const int C2 = a.C * 2;
  int xbase = 0, xrow = 0;         // byte offset of this lane's first pixel in row 0 of the wavefront's three, tap plane 0; that row
  unsigned long long xin_w[3], xin_d[3];
  unsigned long long in_c = 0;
  auto find_x = [&]() {
    const int l = lane_id(), l_tile = (l >> 2) & 7, l_chunk = (l & 3) ^ ((l >> 3) & 2), l_px = l >> 5;
    in_c = __ballot((a.cblocks - 1) * 32 + l_chunk * 8 < a.C);
    const int col = c0 + kg * 8 + l_tile;
    const int q = fast_div(col, a.f_w), iw = col - q * a.nW;
    const int n = fast_div(q, a.f_d), d = q - n * a.oD - a.pd;
    const int w = iw * 4 - a.pw + l_px;
    xrow = h0 + tg * 3 - a.ph;
    xbase = (((n * a.D + d) * a.H + xrow) * a.W + w) * C2 + l_chunk * 16;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      xin_w[p] = __ballot(col < a.n_col && (unsigned)(w + 2 * p) < (unsigned)a.W);
      xin_d[p] = __ballot((unsigned)(d + p) < (unsigned)a.D);
    }
  };
  int x_rd = 0, x_cb = 0;          // the step that is loaded
  unsigned char* const raw = ldsX + wave * kRawWave;
  auto load_x = [&](auto u_c, auto p_c) {
    constexpr int u = decltype(u_c)::value, p = decltype(p_c)::value;
    unsigned long long in = xin_w[p] & (x_rd == 0 ? xin_d[0] : x_rd == 1 ? xin_d[1] : xin_d[2]);
    if (x_cb == a.cblocks - 1) in &= in_c;
    if ((unsigned)(xrow + u) >= (unsigned)a.H) in = 0;
    const int off = xbase + ((x_rd * a.H + u) * a.W + 2 * p) * C2 + x_cb * 64;
    int voff;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(voff) : "v"((int)kOutside), "v"(off), "s"(in));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xdesc, (__attribute__((address_space(3))) void*)(raw + u * 3072 + p * 1024), 16, voff, 0, 0, 0);
  };
  // half of the channels of a unit: lane = tile * 8 + word of two channels
  const int t_tile = lane >> 3, t_word = lane & 7;
  const int raw_at = wave * kRawWave + t_tile * 64 + ((t_tile >> 2) & 1) * 32 + t_word * 4;      // half 0; half 1: ^ 32
  const int v_to = tg * 3 * 1024 + (t_word >> 2) * 512 + ((kg * 8 + t_tile) ^ ((t_word >> 2) * 8)) * 16 + (t_word & 3) * 4;
  Pack<T, 2> xw[6];
  auto read_raw = [&](auto u_c, int half) {
    constexpr int u = decltype(u_c)::value;
    int flip = half * 32;
    asm volatile("" : "+s"(flip));         // one instruction each time instead of a second address kept in a register
    const unsigned char* const from = ldsX + (raw_at ^ flip);
#pragma unroll
    for (int j = 0; j < 6; ++j) xw[j] = *reinterpret_cast<const Pack<T, 2>*>(from + u * 3072 + j * 512);
  };
  auto store_v = [&](auto u_c, int half) {
    constexpr int u = decltype(u_c)::value;
#pragma unroll
    for (int t = 0; t < 6; ++t) *reinterpret_cast<Pack<T, 2>*>(ldsV + half * kVBuf + v_to + (t * ROWS + u) * 1024) = xw[t];
  };

  // ---- filter fragments: groups (element, half of a channel block) of three row taps
  const int R = a.kd * 3, n_groups = a.cblocks * R * 2, k_blocks = (a.K + 31) / 32;
  const int u_lane = lane * 16 + tg * 3072;
  u32x4 uf[UR][3];
  auto u_of = [&](int kb_, int rd, int cb) { return min(kb_ * 4 + kg, k_blocks - 1) * n_groups * 6144 + (cb * R + rd * 3) * 12288; };
  auto load_u = [&](int slot, int base, int half, int e, int r) {
    uf[slot][r] = __builtin_amdgcn_raw_buffer_load_b128(udesc, u_lane + e * 1024, base + (r * 2 + half) * 6144, 0);
  };
  const int v_from = tg * 3 * ROWS * 1024 + (lane >> 5) * 512 + ((lane & 31) ^ ((lane >> 5) * 8)) * 16;

  go_to_box();
  find_x();
  static_for<0, 9>([&](auto i) { load_x(ic<decltype(i)::value / 3>{}, ic<decltype(i)::value % 3>{}); });
  int u_base = u_of(kb, 0, 0);
  auto fill_u = [&]() {
#pragma unroll
    for (int g = 0; g < UR; ++g)
#pragma unroll
      for (int r = 0; r < 3; ++r) load_u(g, u_base, g / 3, g % 3, r);
  };

  // the first half block; the first one of every later box is transformed beside the last products of the box before
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  static_for<0, 3>([&](auto u) {
    read_raw(u, 0);
    row_input_channel(xw, 0);
    row_input_channel(xw, 1);
    store_v(u, 0);
  });
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  f32x16 acc[3][TB];
  for (;;) {
    // the ring is filled anew for each box: kept over the output transform it would not leave that its registers
    fill_u();
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[t][b][e] = 0.f;
    const int at_kb = kb, at_c = c0, at_h = h0;
    bool more = true;
    int rd = 0, cb = 0;
    for (;;) {
      // the step after this one: of this box, or the first of the next one
      const bool last = cb == a.cblocks - 1 && rd == a.kd - 1;
      if (last) {
        place += gridDim.x / kXcds;
        more = place < places;
        if (more) { go_to_box(); find_x(); }
        x_rd = 0; x_cb = 0;
      } else {
        x_cb = cb + 1; x_rd = rd;
        if (x_cb == a.cblocks) { x_cb = 0; ++x_rd; }
      }
      const int u_next = u_of(kb, x_rd, x_cb);
      // One half of a channel block (16 channels): three elements; for each the six rows of V pass by and meet the taps
      // whose output rows the wavefront has.  Beside it a third of the transform of the half block that follows.
      auto half_step = [&](auto half_c) {
        constexpr int half = decltype(half_c)::value, NP = 3 * ROWS;
        u32x4 vf[3];
        auto load_v = [&](int pos) { vf[pos % 3] = *reinterpret_cast<const u32x4*>(ldsV + half * kVBuf + v_from + pos * 1024); };
        load_v(0);
        load_v(1);
        static_for<0, NP>([&](auto pos_c) {
          constexpr int pos = decltype(pos_c)::value, u = pos / ROWS, n = pos % ROWS, g = half * 3 + u;
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (pos + 2 < NP) load_v(pos + 2);
          static_for<0, 3>([&](auto u_c) {
            constexpr int tu = decltype(u_c)::value, at = TallBeside::read(half, tu);
            if constexpr (pos == at) {
              // half 1: the loads of this unit were issued in the half before; those issued after them may be in flight
              if constexpr (half == 1) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(TallBeside::after_loads(tu)) : "memory");
              read_raw(u_c, 1 - half);
            }
          });
          static_for<0, 3>([&](auto r_c) {
            constexpr int r = 2 - decltype(r_c)::value, b = n - r;
            if constexpr (b >= 0 && b < TB)
              acc[u][b] = MfmaRow<T>::run(__builtin_bit_cast(Frag, uf[g % UR][r]), __builtin_bit_cast(Frag, vf[pos % 3]), acc[u][b]);
          });
          static_for<0, 3>([&](auto u_c) {
            constexpr int tu = decltype(u_c)::value, at = TallBeside::read(half, tu);
            if constexpr (pos == at + 2) row_input_channel(xw, 0);
            if constexpr (pos == at + 3) {
              row_input_channel(xw, 1);
              store_v(u_c, 1 - half);
            }
            if constexpr (half == 0 && pos == at + 3) static_for<0, 3>([&](auto p_c) { load_x(u_c, p_c); });
          });
          if constexpr (n == ROWS - 1) {
            __builtin_amdgcn_sched_barrier(0);
            constexpr int gn = g + UR;
#pragma unroll
            for (int r = 0; r < 3; ++r) load_u(g % UR, gn < 6 ? u_base : u_next, gn % 6 / 3, gn % 3, r);
          }
          __builtin_amdgcn_sched_barrier(0);
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
      };
      half_step(ic<0>{});
      half_step(ic<1>{});
      u_base = u_next; rd = x_rd; cb = x_cb;
      if (last) break;
    }
    // A box's last fragments are loaded for nothing, but the waits for x have counted them (TallBeside::after_loads): they are
    // used here, so that they stay.  (The bias, whose registers they have, waits for them anyway.)
#pragma unroll
    for (int g = 0; g < UR; ++g)
#pragma unroll
      for (int r = 0; r < 3; ++r) asm volatile("" :: "v"(uf[g][r]));

    // ---- output transform: elements 0 to 2 (points 0, a, -a) are with the first four wavefronts, 3 to 5 (1/a, -1/a, infinity)
    // with the others; each half finishes two of the four rows and hands three sums of the other two over through LDS
    const __amdgpu_buffer_rsrc_t bdesc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.bias), 0, a.bias ? a.K * 2 : 0, 0x00020000);
    auto finish = [&](auto tg_c) {
      constexpr int TG = decltype(tg_c)::value, X = TG == 0 ? 0 : 2, P0 = TG == 0 ? 1 : 0;
      // before anything is stored: loads wait for the stores ahead of them
      u32x4 bias[2];
      {
        const int k0 = ((at_kb * 4 + kg) * 32 + (lane_id() >> 5) * 16) * 2;
        if constexpr (!KT) {
          bias[0] = __builtin_amdgcn_raw_buffer_load_b128(bdesc, k0, 0, 0);
          bias[1] = __builtin_amdgcn_raw_buffer_load_b128(bdesc, k0 + 16, 0, 0);
        } else {
#pragma unroll
          for (int e = 0; e < 16; e += 2) {
            const unsigned lo = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(bdesc, k0 + e * 2, 0, 0);
            const unsigned hi = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(bdesc, k0 + e * 2 + 2, 0, 0);
            bias[e / 8][e % 8 / 2] = lo | hi << 16;
          }
        }
      }
      static_for<0, TB>([&](auto c_c) {
        constexpr int c = decltype(c_c)::value, mine = TG * 2 + c / 2, theirs = (1 - TG) * 2 + c / 2, first = c % 2 * 8;
        // each part computes its own addresses: the registers are full, and a value that is kept from part to part is spilled
        const int l = lane_id();
        __builtin_amdgcn_sched_barrier(0);
        f32x4* const ex = reinterpret_cast<f32x4*>(ldsV + kVBuf + wave * kExWave) + l;
        const f32x4* const other = reinterpret_cast<const f32x4*>(ldsV + kVBuf + (wave ^ 4) * kExWave) + l;
#pragma unroll
        for (int i4 = 0; i4 < 2; ++i4) {
          f32x4 x, s, d;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float p = acc[P0][theirs][first + i4 * 4 + e], m = acc[P0 + 1][theirs][first + i4 * 4 + e];
            x[e] = acc[X][theirs][first + i4 * 4 + e]; s[e] = p + m; d[e] = p - m;
          }
          ex[(i4 * 3 + 0) * 64] = x; ex[(i4 * 3 + 1) * 64] = s; ex[(i4 * 3 + 2) * 64] = d;
        }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        const int k0 = (at_kb * 4 + kg) * 32 + (l >> 5) * 16 + first;
        Pack<T, 8> o[4];
#pragma unroll
        for (int i4 = 0; i4 < 2; ++i4) {
          f32x4 g[3];
#pragma unroll
          for (int j = 0; j < 3; ++j) g[j] = other[(i4 * 3 + j) * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = i4 * 4 + e;
            unsigned two = bias[first / 8][i / 2];
            asm volatile("" : "+v"(two));          // converted here, not all of them ahead of time
            const float bv = static_cast<float>(__builtin_bit_cast(Pack<T, 2>, two).v[e % 2]);
            const float p = acc[P0][mine][first + i], m = acc[P0 + 1][mine][first + i], x = acc[X][mine][first + i];
            const RowOutputs<4> out = TG == 0 ? row_outputs<4>(x, p + m, p - m, g[0][e], g[1][e], g[2][e], bv)
                                           : row_outputs<4>(g[0][e], g[1][e], g[2][e], x, p + m, p - m, bv);
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j].v[i] = static_cast<T>(out.o[j]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();      // read: free for the next part
        const int col = at_c + (l & 31), q = fast_div(col, a.f_w), iw = col - q * a.nW;
        const bool ok = col < a.n_col && at_h + mine < a.oH && k0 < a.K;
        T* const yp = static_cast<T*>(a.y) + (((size_t)q * a.oH + at_h + mine) * a.oW + iw * 4) * a.K + k0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          T* const dst = yp + (size_t)i * a.K;
          const bool in_row = ok && iw * 4 + i < a.oW;
          if constexpr (!KT) {
            if (in_row) *reinterpret_cast<u32x4*>(dst) = __builtin_bit_cast(u32x4, o[i]);
          } else {
            if (in_row && k0 + 8 <= a.K) {
              __builtin_memcpy(dst, &o[i], 16);          // rows of y start at any multiple of the element size
            } else if (in_row) {
              store_some(dst, __builtin_bit_cast(u32x4, o[i]), a.K - k0);
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    if (tg == 0) finish(ic<0>{});
    else finish(ic<1>{});
    if (!more) return;
  }
}

// Filters that overflow an XCD's 4 MB of L2: its workgroups work on one channel block at a time
constexpr int kFilterInL2 = 3 << 20;

}  // namespace

// the first n_planes output planes (2-D: images) from x on
int tall_row_conv(const wc_conv_desc* d, const void* x, int n_planes, const void* U, const void* bias, void* y, void* stream) {
  TallArgs a{};
  a.x = x; a.U = U; a.bias = bias; a.y = y;
  a.D = d->in[0]; a.H = d->in[1]; a.W = d->in[2]; a.C = wc_padded_channels8(d->C); a.K = d->K;
  a.pd = d->pad[0]; a.ph = d->pad[1]; a.pw = d->pad[2]; a.kd = d->kernel[0];
  a.oD = a.D + 2 * a.pd - a.kd + 1; a.oH = a.H + 2 * a.ph - 2; a.oW = a.W + 2 * a.pw - 2;
  a.N = ceil_div(n_planes, a.oD);
  a.nW = ceil_div(a.oW, 4);
  a.n_col = n_planes * a.nW;
  a.f_w = make_fast_div(a.nW); a.f_d = make_fast_div(a.oD);
  a.n_cg = ceil_div(a.n_col, 32); a.n_hb = ceil_div(a.oH, TB); a.n_kb = ceil_div(a.K, 128);
  a.n_box = a.n_cg * a.n_hb;
  a.cblocks = ceil_div(a.C, 32);
  a.x_bytes = (int)((long long)a.N * a.D * a.H * a.W * a.C * 2);
  a.u_bytes = (int)(row_u_elems(d) * 2);
  a.box_fast = a.u_bytes > kFilterInL2;
  a.per_xcd = ceil_div(a.n_kb * a.n_box, kXcds);
  const bool whole = a.K % 8 == 0 && ((reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(bias)) & 15) == 0;
  // one workgroup per CU, and at most one per box
  const int grid = std::min(a.per_xcd * kXcds, kCus);
  return dispatch_dtype(d->dtype, [&](auto t) -> int {
    using T = decltype(t);
    if constexpr (sizeof(T) == 2) {
      if (whole) hipLaunchKernelGGL((tall_row_kernel<T, 2, false>), dim3(grid), dim3(512), 0, as_stream(stream), a);
      else hipLaunchKernelGGL((tall_row_kernel<T, 2, true>), dim3(grid), dim3(512), 0, as_stream(stream), a);
      WC_CHECK_LAUNCH("tall_row_kernel");
      return WC_OK;
    }
    return fail(WC_ERR_UNSUPPORTED, "row form: 16-bit types");
  });
}

}  // namespace wc
