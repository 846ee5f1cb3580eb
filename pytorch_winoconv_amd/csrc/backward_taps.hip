// Weight gradient of 3x3 and 3x3x3 layers at stride 1 in a 16-bit type, taken directly ("tap form"):
//
//   dw[rd, rh, rw][k][c] = sum over the output pixels p of  dy[p][k]  x[p + (rd, rh, rw)][c]
//
// Images, planes and rows are laid one after the other with the padding kept in, as a line of positions
// L = ((n oD + d) Hp + h) Wp + w, Hp = oH + 2, Wp = oW + 2.  dy is zero at the two last rows and columns, so tap (rh, rw)
// reads x at L + rh Wp + rw, whatever row or image that crosses into.  A workgroup takes a run of positions, one depth
// tap, 128 (or 64) output and 64 input channels with all nine taps: x passes once through a ring of LDS rows (a position
// each), 64 positions at a time, and dy through two stages.  The operands need eight consecutive positions of one channel,
// which ds_read_b64_tr_b16 delivers; a wavefront holds one kernel row: it reads twelve positions and shifts the taps
// 1 and 2 out of them in registers, five LDS reads of 8 bytes for six products instead of ten.
//
// The transform domain multiplies less (8 products per pixel of a 3x3x3 filter against 27) but moves V and dM through
// memory: N=8 128 -> 128, 16x56x56, fp16, 797 us of which 760 are that traffic; here 368 us, 0.95 PFLOP/s (a library
// matrix product reaches 1.1 on this card) with x and dy through registers (taps_kernel) and 318 by LDS-DMA (taps_dma_kernel), sums
// included.  Through registers 114 vector instructions stand beside the 24 products of a wavefront's step, most of them for
// addresses; by LDS-DMA under forty, and a step takes 1.9 us for the 1.73 that its products take at the rate the matrix cores sustain with
// changing operands.  Both | registers: N=64 64 -> 64, 56x56 33 | 42, 256 -> 256, 28x28 77 | 85, 128 -> 128, 28x28 37.5 | 40, N=8 64 -> 64, 8x28x28
// 32.5 | 39.  Beside its steps a launch moves its partial sums, 59 MB each way where 200 workgroups share 0.6 MB of dw.  Variants that were
// slower: dy turned channel by channel in LDS and read 16 bytes at a time 424 us, four wavefronts of all nine taps 439; operands
// read a group ahead changed nothing (377).  Operands are exact, sums fp32.
#include "column_sums.h"
#include "lds_dma.h"
#include "wc_transform.h"

#include <algorithm>

namespace wc {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c, half_t) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c, bf16_t) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

constexpr int kStep = 64;                 // positions per step
constexpr int kMirror = 32;               // ring rows repeated behind its end: a fragment reads 20 rows without a wrap
// LDS bytes per position.  A transposing read takes 4 rows x 64 bytes at a time: a pitch of 64 modulo 128 puts them into
// different banks
constexpr int kXPitch = 64 * 2 + 64;
template <int KG> constexpr int kDyPitch = KG * 128 + 64;

struct TapsArgs {
  const void* x; const void* dy; float* part;
  float* bias;                     // column sums of dy, a row of 64 KG per workgroup in order (part, depth tap, input and output channels); null: none
  int D, H, W, C, K;               // x (N, D, H, W, C), dy (N, oD, oH, oW, K)
  int oD, oH, oW, pd, ph, pw;
  long long x_elems, dy_elems;
  int Hp, Wp;                      // oH + 2, oW + 2
  FastDiv f_wp, f_hp, f_od;
  int total;                       // positions
  int part_steps;                  // steps of 64 positions per part
  int halo, ring;                  // positions of x beyond a step's own (a multiple of 64), rows of the ring: halo + 128
  int n_kd, n_k, n_c, tiles, n_wg, per_xcd;
};

template <int KG> constexpr int taps_tile_floats() { return KG * 6 * 24 * 64 * 4; }
template <int KG> constexpr int taps_lds(int ring) { return 2 * kStep * kDyPitch<KG> + (ring + kMirror) * kXPitch; }

// The products of 16 positions: x from `xb` on (rows XP bytes apart), two blocks of 32 output channels of dy
template <typename T, int XP, int DP>
__device__ __forceinline__ void taps_products(f32x16 (&acc)[3][2], const unsigned char* xb, const unsigned char* d0, const unsigned char* d1) {
  typedef s16x4 __attribute__((address_space(3))) * LdsVec;
  auto read_tr = [](const unsigned char* p) { return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsVec)(p))); };
  const u32x2 e0 = read_tr(xb), e1 = read_tr(xb + 4 * XP), e2 = read_tr(xb + 8 * XP);
  u32x4 df[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const unsigned char* const d = i ? d1 : d0;
    const u32x2 lo = read_tr(d), hi = read_tr(d + 4 * DP);
    df[i] = u32x4{lo[0], lo[1], hi[0], hi[1]};
  }
  const u32x4 x0 = {e0[0], e0[1], e1[0], e1[1]}, x2 = {e0[1], e1[0], e1[1], e2[0]};
  const u32x4 x1 = {__builtin_amdgcn_alignbit(e0[1], e0[0], 16), __builtin_amdgcn_alignbit(e1[0], e0[1], 16),
                    __builtin_amdgcn_alignbit(e1[1], e1[0], 16), __builtin_amdgcn_alignbit(e2[0], e1[1], 16)};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    acc[0][i] = mfma(x0, df[i], acc[0][i], T{});
    acc[1][i] = mfma(x1, df[i], acc[1][i], T{});
    acc[2][i] = mfma(x2, df[i], acc[2][i], T{});
  }
}

// Partial sums in the order of the accumulators: 1 KB per store
__device__ __forceinline__ void taps_store(const f32x16 (&acc)[3][2], float* out) {
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 o = {acc[t][i][4 * q], acc[t][i][4 * q + 1], acc[t][i][4 * q + 2], acc[t][i][4 * q + 3]};
        *reinterpret_cast<f32x4*>(out + ((t * 2 + i) * 4 + q) * 256) = o;
      }
}

template <typename T, int KG>
__global__ __launch_bounds__(384 * KG) __attribute__((amdgpu_waves_per_eu(3, 3)))
void taps_kernel(TapsArgs a) {
  constexpr int THREADS = 384 * KG, ND = kStep * KG * 8, NX = kStep * 8, NU = (ND + NX + THREADS - 1) / THREADS;
  constexpr int DP = kDyPitch<KG>, XP = kXPitch;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  unsigned char* const lds_x = lds + 2 * kStep * DP;
  const int wg = xcd_remap(blockIdx.x, a.per_xcd);
  if (wg >= a.n_wg) return;
  const int part = wg / a.tiles;                  // tiles of a part are neighbours: they share dy and x in an XCD's L2
  int tile = wg - part * a.tiles;
  const int ct = tile % a.n_c; tile /= a.n_c;
  const int kt = tile % a.n_k, kd = tile / a.n_k;
  const int k0 = kt * 64 * KG, c0 = ct * 64;
  const int holder = kd * a.n_c + ct;               // of those with this part's rows of dy
  const int q0 = part * a.part_steps * kStep, q_end = min(a.total, q0 + a.part_steps * kStep);
  const int steps = (q_end - q0 + kStep - 1) / kStep;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / 6, kh = wave % 6 / 2, cb = wave & 1;

  const T* const xp = static_cast<const T*>(a.x) + c0;
  const T* const dp = static_cast<const T*>(a.dy) + k0;
  const u32x4 zero = {0u, 0u, 0u, 0u};
  // position -> 16 bytes of x (8 channels from c on) or of dy; zeros where there is none
  auto place = [&](int pos, int& plane, int& h, int& w) {
    const int row = fast_div(pos, a.f_wp);
    w = pos - row * a.Wp;
    plane = fast_div(row, a.f_hp);
    h = row - plane * a.Hp;
  };
  // rows start at any multiple of the element size; beyond the last channel of a position come the next one's, in columns
  // that nobody writes out, and beyond the last position the tensor ends
  auto load16 = [&](const T* p, const T* end, bool ok) {
    u32x4 v = zero;
    if (ok) {
      if (p + 8 <= end) {
        __builtin_memcpy(&v, p, 16);
      } else {
        Pack<T, 8> o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o.v[e] = p + e < end ? p[e] : T(0);
        v = __builtin_bit_cast(u32x4, o);
      }
    }
    return v;
  };
  auto load_x = [&](int pos, int c) {
    int plane, h, w;
    place(pos, plane, h, w);
    const int n = fast_div(plane, a.f_od), d = plane - n * a.oD + kd - a.pd;
    h -= a.ph; w -= a.pw;
    const bool ok = pos < a.total && c0 + c < a.C && (unsigned)d < (unsigned)a.D && (unsigned)h < (unsigned)a.H && (unsigned)w < (unsigned)a.W;
    return load16(xp + ((((long long)n * a.D + d) * a.H + h) * a.W + w) * a.C + c, static_cast<const T*>(a.x) + a.x_elems, ok);
  };
  auto load_dy = [&](int pos, int k) {
    int plane, h, w;
    place(pos, plane, h, w);
    const bool ok = pos < q_end && k0 + k < a.K && h < a.oH && w < a.oW;
    return load16(dp + (((long long)plane * a.oH + h) * a.oW + w) * a.K + k, static_cast<const T*>(a.dy) + a.dy_elems, ok);
  };

  u32x4 reg[NU];
  auto load = [&](int step) {                       // dy of a step, and the 64 positions of x it is the first to reach
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + i * THREADS;
      if (u < ND) reg[i] = load_dy(q0 + step * kStep + u / (8 * KG), u % (8 * KG) * 8);
      else if (u < ND + NX) reg[i] = load_x(q0 + step * kStep + a.halo + (u - ND) / 8, (u - ND) % 8 * 8);
    }
  };
  auto put_x = [&](int slot, int v, u32x4 value) {  // v: unit of 64 rows from ring row `slot` on
    unsigned char* const p = lds_x + (slot + v / 8) * XP + v % 8 * 16;
    *reinterpret_cast<u32x4*>(p) = value;
    if (slot == 0 && v / 8 < kMirror) *reinterpret_cast<u32x4*>(p + a.ring * XP) = value;
  };
  auto store = [&](int step, int slot) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + i * THREADS;
      if (u < ND) *reinterpret_cast<u32x4*>(lds + ((step & 1) * kStep + u / (8 * KG)) * DP + u % (8 * KG) * 16) = reg[i];
      else if (u < ND + NX) put_x(slot, u - ND, reg[i]);
    }
  };

  f32x16 acc[3][2];
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[t][i][e] = 0.f;

  load(0);
  for (int j = 0; j < a.halo; j += kStep)
#pragma unroll
    for (int v0 = 0; v0 < NX; v0 += THREADS) {
      const int v = tid + v0;
      if (v < NX) put_x(j, v, load_x(q0 + j + v / 8, v % 8 * 8));
    }
  store(0, a.halo);
  __syncthreads();

  // a lane's address in a fragment of 16 positions x 32 channels: group b of 16 lanes reads rows 8 (b / 2) .. + 3, columns
  // 16 (b % 2) .. + 15
  const int frag_row = 8 * (lane >> 5) + ((lane & 15) >> 2), frag_col = ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
  const int x_lane = frag_row * XP + cb * 64 + frag_col, d_lane = frag_row * DP + kg * 128 + frag_col;

  int slot = 0;                                     // ring row of the step's first position
  const int turns = 6 * KG * a.n_kd * a.n_c;
  int turn = wave + 6 * KG * holder;                    // steps until this wavefront adds one's rows of dy up
  float colsum[2] = {0.f, 0.f};
  for (int step = 0; step < steps; ++step) {
    const bool more = step + 1 < steps;
    if (more) load(step + 1);
    const int row = slot + kh * a.Wp;
    const unsigned char* const db = lds + (step & 1) * kStep * DP + d_lane;
    if (turn == 0) {
      if (a.bias) add_rows<T, KG * 64, DP, false>(lds + (step & 1) * kStep * DP, kStep, lane, colsum);
      turn = turns;
    }
    --turn;
#pragma unroll
    for (int kk = 0; kk < kStep / 16; ++kk) {
      const int r = row + kk * 16 >= a.ring ? row + kk * 16 - a.ring : row + kk * 16;
      const unsigned char* const xb = lds_x + r * XP + x_lane;
      taps_products<T, XP, DP>(acc, xb, db + kk * 16 * DP, db + kk * 16 * DP + 64);
    }
    if (more) {
      int to = slot + a.halo + kStep;               // ring = halo + 128: rows that no wavefront reads any more
      if (to >= a.ring) to -= a.ring;
      store(step + 1, to);
    }
    slot += kStep;
    if (slot >= a.ring) slot -= a.ring;
    __syncthreads();
  }

  if (a.bias) store_sums<6 * KG, KG * 64>(colsum, reinterpret_cast<float*>(lds), wave, lane, a.bias + (((long long)part * a.n_kd * a.n_c + holder) * a.n_k + kt) * 64 * KG);
  taps_store(acc, a.part + (long long)wg * taps_tile_floats<KG>() + wave * 24 * 256 + lane * 4);
}

// The same with x and dy brought to LDS by LDS-DMA, two steps ahead: channels in multiples of 8, 16-byte aligned tensors.  Where
// the rows of a step lie is worked out once per position, by two wavefronts in turn, a step before it is needed, and read from a
// table in LDS; positions outside the image are offsets outside the descriptor's range, which bring zeros.  Rows are not
// padded: their 64-byte pieces are exchanged by the row instead (LDS-DMA writes rows one after the other), x in every other two rows,
// dy of 128 channels by the row modulo 4.
template <int KG> constexpr int taps_dma_lds(int ring) { return 3 * kStep * KG * 128 + (ring + kMirror) * 128 + 4 * 2 * kStep * 4; }

template <typename T, int KG>
__global__ __launch_bounds__(384 * KG) __attribute__((amdgpu_waves_per_eu(3, 3)))
void taps_dma_kernel(TapsArgs a) {
  constexpr int NW = 6 * KG, ND = 8 * KG, NL = (ND + 8 + NW - 1) / NW;      // loads of 1 KB: ND of dy and 8 of x per step
  constexpr int DP = KG * 128, XP = 128, DY_STAGE = kStep * DP, DROWS = 8 / KG;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  unsigned char* const lds_x = lds + 3 * DY_STAGE;
  unsigned* const table = reinterpret_cast<unsigned*>(lds_x + (a.ring + kMirror) * XP);      // of step s: (s & 3) * 128, dy, then x
  const int wg = xcd_remap(blockIdx.x, a.per_xcd);
  if (wg >= a.n_wg) return;
  const int part = wg / a.tiles;
  int tile = wg - part * a.tiles;
  const int ct = tile % a.n_c; tile /= a.n_c;
  const int kt = tile % a.n_k, kd = tile / a.n_k;
  const int k0 = kt * 64 * KG, c0 = ct * 64;
  const int holder = kd * a.n_c + ct;               // of those with this part's rows of dy
  const int q0 = part * a.part_steps * kStep, q_end = min(a.total, q0 + a.part_steps * kStep);
  const int steps = (q_end - q0 + kStep - 1) / kStep;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int kg = wave / 6, kh = wave % 6 / 2, cb = wave & 1;

  // offsets count from the plane of dy and the image of x that the part begins in
  const int plane0 = fast_div(fast_div(q0, a.f_wp), a.f_hp), n0 = fast_div(plane0, a.f_od);
  const long long dy_start = ((long long)plane0 * a.oH * a.oW * a.K + k0) * 2, x_start = ((long long)n0 * a.D * a.H * a.W * a.C + c0) * 2;
  const u32x4 dyd = dma_descriptor(static_cast<const unsigned char*>(a.dy) + dy_start, a.dy_elems * 2 - dy_start);
  const u32x4 xd = dma_descriptor(static_cast<const unsigned char*>(a.x) + x_start, a.x_elems * 2 - x_start);
  auto place = [&](int pos, int& plane, int& h, int& w) {
    const int row = fast_div(pos, a.f_wp);
    w = pos - row * a.Wp;
    plane = fast_div(row, a.f_hp);
    h = row - plane * a.Hp;
  };
  auto dy_offset = [&](int pos) {
    int plane, h, w;
    place(pos, plane, h, w);
    const bool ok = pos < q_end && h < a.oH && w < a.oW;
    return ok ? (unsigned)(((plane - plane0) * a.oH + h) * a.oW + w) * (unsigned)a.K * 2u : kOutside;
  };
  auto x_offset = [&](int pos) {
    int plane, h, w;
    place(pos, plane, h, w);
    const int n = fast_div(plane, a.f_od), d = plane - n * a.oD + kd - a.pd;
    h -= a.ph; w -= a.pw;
    const bool ok = pos < a.total && (unsigned)d < (unsigned)a.D && (unsigned)h < (unsigned)a.H && (unsigned)w < (unsigned)a.W;
    return ok ? (unsigned)((((n - n0) * a.D + d) * a.H + h) * a.W + w) * (unsigned)a.C * 2u : kOutside;
  };
  auto fill = [&](int step, int which) {            // by one wavefront: the rows of dy (0) or x (1) of a step
    table[(step & 3) * 2 * kStep + which * kStep + lane] = which ? x_offset(q0 + step * kStep + a.halo + lane) : dy_offset(q0 + step * kStep + lane);
  };
  // a lane's 16 bytes of a row, wherever the exchange puts them; channels that are not there lie outside
  const int dy_chunk = KG == 2 ? (lane & 15) ^ ((lane >> 4) * 4) : (lane & 7) ^ ((lane >> 4) & 1) * 4, x_chunk = (lane & 7) ^ ((lane >> 4) & 1) * 4;
  const unsigned dy_out = k0 + dy_chunk * 8 < a.K ? 0u : kOutside, x_out = c0 + x_chunk * 8 < a.C ? 0u : kOutside;
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds, ldsx0 = lds0 + 3 * DY_STAGE;
  auto load_x = [&](unsigned row_off, int slot, int v) {         // eight rows from ring row slot + 8 v on
    const unsigned off = (row_off + x_chunk * 16) | x_out;
    dma16(xd, off, ldsx0 + slot * XP + v * 1024);
    if (slot == 0 && v * 8 < kMirror) dma16(xd, off, ldsx0 + a.ring * XP + v * 1024);
  };
  auto issue = [&](int step, int stage, int slot) {
    const unsigned* const t = table + (step & 3) * 2 * kStep;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int u = wave + i * NW;
      if (u < ND) dma16(dyd, (t[u * DROWS + lane / (8 * KG)] + dy_chunk * 16) | dy_out, lds0 + stage * DY_STAGE + u * 1024);
      else if (u < ND + 8) load_x(t[kStep + (u - ND) * 8 + lane / 8], slot, u - ND);
    }
  };

  f32x16 acc[3][2];
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[t][i][e] = 0.f;

  if (wave < 6) fill(wave >> 1, wave & 1);
  for (int v = wave; v < a.halo / 8; v += NW) load_x(x_offset(q0 + v * 8 + lane / 8), v / 8 * 64, v % 8);
  __syncthreads();
  issue(0, 0, a.halo);
  if (steps > 1) issue(1, 1, a.halo + kStep);

  const int frag_row = 8 * (lane >> 5) + ((lane & 15) >> 2), frag_col = ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
  const int x_lane = frag_row * XP + ((cb * 64 + frag_col) ^ (((kh * a.Wp + frag_row) >> 1) & 1) * 64);
  const int d_swap = KG == 2 ? (frag_row & 3) * 64 : ((frag_row >> 1) & 1) * 64;
  const int d_lane0 = frag_row * DP + ((kg * 128 + frag_col) ^ d_swap), d_lane1 = frag_row * DP + ((kg * 128 + 64 + frag_col) ^ d_swap);

  int slot = 0, to = a.halo + 2 * kStep, stage = 0, filler = 0;      // ring rows of the step's first position and of the loads two steps on
  const int turns = NW * a.n_kd * a.n_c;
  int turn = wave + NW * holder;                    // steps until this wavefront adds one's rows of dy up
  float colsum[2] = {0.f, 0.f};
  for (int step = 0; step < steps; ++step) {
    // this step's loads are there (the next step's, at least two per wavefront, may be on their way), for all, and all are done
    // with the last step's rows and the table's
    if (step + 1 < steps) asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int next = stage == 0 ? 2 : stage - 1;
    if (step + 2 < steps) issue(step + 2, next, to);
    if (step + 3 < steps && (wave >> 1) == filler) fill(step + 3, wave & 1);
    filler = filler == NW / 2 - 1 ? 0 : filler + 1;
    const int row = slot + kh * a.Wp;
    const unsigned char* const db = lds + stage * DY_STAGE;
    if (turn == 0) {
      if (a.bias) add_rows<T, KG * 64, DP, true>(lds + stage * DY_STAGE, kStep, lane, colsum);
      turn = turns;
    }
    --turn;
#pragma unroll
    for (int kk = 0; kk < kStep / 16; ++kk) {
      const int r = row + kk * 16 >= a.ring ? row + kk * 16 - a.ring : row + kk * 16;
      taps_products<T, XP, DP>(acc, lds_x + r * XP + x_lane, db + kk * 16 * DP + d_lane0, db + kk * 16 * DP + d_lane1);
    }
    slot += kStep;
    if (slot >= a.ring) slot -= a.ring;
    to += kStep;
    if (to >= a.ring) to -= a.ring;
    stage = stage == 2 ? 0 : stage + 1;
  }
  if (a.bias) store_sums<6 * KG, KG * 64>(colsum, reinterpret_cast<float*>(lds), wave, lane, a.bias + (((long long)part * a.n_kd * a.n_c + holder) * a.n_k + kt) * 64 * KG);
  taps_store(acc, a.part + (long long)wg * taps_tile_floats<KG>() + wave * 24 * 256 + lane * 4);
}

// dw <- the sum of the parts, in a fixed order.  A workgroup owns one accumulator quarter (64 lanes x 4 input channels) of
// one tile; its wavefronts share out the parts.
struct TapsSumArgs {
  const float* part;
  void* dw;
  long long s[5];
  int S, tiles, n_k, n_c, K, C, f32;
  int blocks;                      // beyond them: the bias gradient's
  ColumnSums bias;
};
template <typename T, int KG>
__global__ __launch_bounds__(256) void taps_sum_kernel(TapsSumArgs a) {
  __shared__ f32x4 sums[3][64];
  static_assert(sizeof(sums) >= 256 * 4, "sum_columns takes as much");
  const int lane = threadIdx.x & 63, group = threadIdx.x >> 6;
  int b = blockIdx.x;
  if (b >= a.blocks) return sum_columns<T>(a.bias, b - a.blocks, reinterpret_cast<float*>(sums));
  const int q = b & 3, i = (b >> 2) & 1, kw = (b >> 3) % 3, wave = b / 24 % (6 * KG);
  int tile = b / (24 * 6 * KG);
  const float* src = a.part + (long long)b * 256 + lane * 4;
  const long long stride = (long long)a.tiles * taps_tile_floats<KG>();
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int p = group; p < a.S; p += 4) sum += *reinterpret_cast<const f32x4*>(src + p * stride);
  if (group) sums[group - 1][lane] = sum;
  __syncthreads();
  if (group) return;
#pragma unroll
  for (int j = 0; j < 3; ++j) sum += sums[j][lane];
  const int ct = tile % a.n_c; tile /= a.n_c;
  const int kt = tile % a.n_k, kd = tile / a.n_k;
  const int k = kt * 64 * KG + wave / 6 * 64 + i * 32 + (lane & 31), c = ct * 64 + (wave & 1) * 32 + 8 * q + 4 * (lane >> 5);
  if (k >= a.K) return;
  const long long dst = k * a.s[0] + c * a.s[1] + kd * a.s[2] + wave % 6 / 2 * a.s[3] + kw * a.s[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (c + e < a.C) store_as<T>(a.dw, dst + e * a.s[1], sum[e], a.f32);
}

struct TapsPlan { int kg, halo, ring, total, steps, parts, part_steps, tiles; };

// Parts of the line of positions.  A workgroup takes 1.45 us per step (1.9 with the whole chip at work; 1.0 for 64 output
// channels: two of those on a CU only share its LDS, one each is the most that pays), and its sums are written and read back, 0.29 MB per 128 x 64 channels: the
// fewest microseconds for the slowest workgroup and that traffic.  Measured fp16, us over parts: N=64 128 -> 128, 28x28
// 128: 39.6, 76: 37.2, 64: 38.5, 32: 53.5; 64 -> 64, 56x56 204: 34.4, 153: 37.7, 64: 66; 256 -> 256, 14x14 32: 43, 22: 41, 10: 55; N=8 64 -> 64, 28x28 128:
// 17.5, 64: 14.2, 43: 13.6; N=8 128 -> 128, 16x56x56 42: 342, 28: 374, 19: 511.
int taps_parts(int steps, int tiles, int kg) {
  int best = 1;
  double best_t = 1e30;
  for (int s = 1; s == 1 || s * tiles <= kCus; ++s) {
    const int per = ceil_div(steps, s), parts = ceil_div(steps, per);
    const double fill = (double)parts * tiles / kCus;
    const double step_us = kg == 2 ? (fill > 0.5 ? 1.45 + 0.9 * (fill - 0.5) : 1.45) : 1.0;
    const double t = per * step_us + parts * tiles * (kg * 0.147) / 4.0;
    if (t < best_t * (1.0 - 1e-9)) { best = s; best_t = t; }
  }
  return best;
}

bool taps_plan(const wc_conv_desc* d, const int out[3], TapsPlan* p) {
  if (d->dtype == WC_F32 || d->stride != 1 || d->whole_kernel) return false;
  if (d->kernel[1] != 3 || d->kernel[2] != 3 || (d->kernel[0] != 3 && d->kernel[0] != 1)) return false;
  const long long Wp = out[2] + 2, total = (long long)d->N * out[0] * (out[1] + 2) * Wp;
  if (Wp > 1024 || total >= (1ll << 31) - 4096) return false;       // positions stay ints, with a run's halo beyond the end
  p->kg = ceil_div(d->K, 64) == 1 || ceil_div(d->K, 64) == 3 ? 1 : 2;
  p->halo = (int)(2 * Wp + 2 + kStep - 1) / kStep * kStep;
  p->ring = p->halo + 2 * kStep;
  if ((p->kg == 2 ? taps_lds<2>(p->ring) : taps_lds<1>(p->ring)) > 160 * 1024) return false;
  p->total = (int)total;
  p->steps = ceil_div(p->total, kStep);
  p->tiles = d->kernel[0] * ceil_div(d->K, 64 * p->kg) * ceil_div(d->C, 64);
  const int S = taps_parts(p->steps, p->tiles, p->kg);
  p->part_steps = ceil_div(p->steps, std::min(S, p->steps));
  p->parts = ceil_div(p->steps, p->part_steps);
  // the last part is cut off at `total`, but the kernel takes its full length first: up to 64 * parts positions more
  return (long long)p->parts * p->part_steps * kStep < (1ll << 31);
}

template <typename T, int KG>
int launch_taps(const wc_conv_desc* d, const int out[3], const TapsPlan& p, const void* x, const void* dy, const GradOut& to, float* part, void* stream) {
  TapsArgs a;
  a.x = x; a.dy = dy; a.part = part; a.bias = to.db ? to.db_part : nullptr;
  a.D = d->in[0]; a.H = d->in[1]; a.W = d->in[2]; a.C = d->C; a.K = d->K;
  a.oD = out[0]; a.oH = out[1]; a.oW = out[2]; a.pd = d->pad[0]; a.ph = d->pad[1]; a.pw = d->pad[2];
  a.x_elems = (long long)d->N * a.D * a.H * a.W * a.C; a.dy_elems = (long long)d->N * a.oD * a.oH * a.oW * a.K;
  a.Hp = a.oH + 2; a.Wp = a.oW + 2;
  a.f_wp = make_fast_div(a.Wp); a.f_hp = make_fast_div(a.Hp); a.f_od = make_fast_div(a.oD);
  a.total = p.total; a.part_steps = p.part_steps; a.halo = p.halo; a.ring = p.ring;
  a.n_kd = d->kernel[0]; a.n_k = ceil_div(a.K, 64 * KG); a.n_c = ceil_div(a.C, 64); a.tiles = p.tiles;
  a.n_wg = p.tiles * p.parts; a.per_xcd = ceil_div(a.n_wg, kXcds);
  // x and dy by LDS-DMA where rows are whole 16 bytes and 31-bit offsets reach what a part reads
  const long long planes = ((p.part_steps + 4ll) * kStep + p.halo) / ((long long)a.Hp * a.Wp) + 2;
  const int dma_ring = p.halo + 3 * kStep, dma_lds = taps_dma_lds<KG>(dma_ring);
  const bool dma = a.C % 8 == 0 && a.K % 8 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(dy)) & 15) == 0 &&
                   planes * a.oH * a.oW * a.K * 2 < (1ll << 31) && (planes / a.oD + 2) * a.D * a.H * a.W * a.C * 2 < (1ll << 31) && dma_lds <= 160 * 1024;
  if (dma) a.ring = dma_ring;
  const auto fn = dma ? &taps_dma_kernel<T, KG> : &taps_kernel<T, KG>;
  const int lds = dma ? dma_lds : taps_lds<KG>(p.ring);
  if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds)) return rc;
  hipLaunchKernelGGL(fn, dim3((unsigned)(a.per_xcd * kXcds)), dim3(384 * KG), lds, as_stream(stream), a);
  WC_CHECK_LAUNCH("taps_kernel");
  TapsSumArgs b;
  b.part = part; b.dw = to.dw; b.f32 = to.dw_f32;
  for (int i = 0; i < 5; ++i) b.s[i] = to.s[i];
  b.S = p.parts; b.tiles = p.tiles; b.n_k = a.n_k; b.n_c = a.n_c; b.K = a.K; b.C = a.C;
  b.blocks = p.tiles * 144 * KG;
  b.bias = {a.bias, to.db, p.parts * a.n_kd * a.n_c, a.n_k * 64 * KG, a.K, to.db_f32};
  hipLaunchKernelGGL((taps_sum_kernel<T, KG>), dim3((unsigned)(b.blocks + (to.db ? ceil_div(a.K, 16) : 0))), dim3(256), 0, as_stream(stream), b);
  WC_CHECK_LAUNCH("taps_sum_kernel");
  return WC_OK;
}

}  // namespace

// Against the transform domain, fp16, us (taps | F(2,3), in 2-D also F(4,3) tiles): N=8 128 -> 128, 16x56x56 318 | 779; 64 -> 64,
// 8x28x28 33 | 82; N=64 128 -> 128, 28x28 38 | 66 | 53; N=64 256 -> 256, 14x14 42 | 52 | 49; N=8 256 -> 256, 28x28 35 | 41 | 39; N=1 128 -> 128,
// 28x28 15 | 20 | 21.  F(4,3) multiplies a quarter as much and its traffic grows with C + K, the products here with C K (padded to
// tiles), so it is ahead on large wide layers, counted in steps of 64 positions and tiles of 128 x 64 channels: 512 -> 512, 56x56 N=32
// (54000) 426 | 529 | 375, 28x28 N=64 (29000) 236 | 283 | 236, N=16 (7200) 86 | 96 | 110; 384 -> 384, 28x28 N=64 (16000) 146 | 212 | 143, 14x14 (4600) 62 | 85 |
// 78; 1024 -> 1024, 14x14 N=64 (33000) 284 | 262 | 266, 7x7 (10400) 129 | 134 | 136; 256 -> 256, 56x56 N=64 (27000) 226 | 405 | 268; 72 -> 72, 56x56 (6700) 66 | 133 | 77.
// Channels that are no multiples of 8 go through registers (us, F(4,3) | taps: 100 -> 150, N=64 28x28 53 | 56; against F(2,3) alone
// still ahead: 50 -> 64, N=32 56x56 32 | 71; 3 -> 64, N=64 112x112 106 | 334).  Small problems are launches and latency: two of them
// here, six there (512 -> 512, N=1 7x7 28 | 39 | 48).
bool taps_gradient_fits(const wc_conv_desc* d, const int out[3], size_t* workspace_bytes, size_t* bias_bytes) {
  TapsPlan p;
  if (test_gemm_config() == 20 || !taps_plan(d, out, &p)) return false;
  if (d->ndim == 2 && d->m == 4 && (long long)p.steps * p.tiles > (d->C % 8 == 0 && d->K % 8 == 0 ? 12000 : 2560)) {
    const long long padded = (long long)ceil_div(d->K, 64 * p.kg) * 64 * p.kg * ceil_div(d->C, 64) * 64;
    if (padded > 256 * 256 || padded * 5 > 8ll * d->C * d->K) return false;
  }
  *bias_bytes = (size_t)p.parts * p.tiles * 64 * p.kg * 4;
  *workspace_bytes = (size_t)p.parts * p.tiles * (p.kg == 2 ? taps_tile_floats<2>() : taps_tile_floats<1>()) * 4;
  return true;
}

int taps_gradient(const wc_conv_desc* d, const int out[3], const void* x, const void* dy, const GradOut& to, float* part, void* stream) {
  TapsPlan p;
  WC_CHECK_ARG(taps_plan(d, out, &p), "tap form of the weight gradient: 16-bit, 3x3 or 3x3x3, stride 1");
  return dispatch_dtype(d->dtype, [&](auto t) -> int {
    using T = decltype(t);
    if constexpr (sizeof(T) == 2) {
      return p.kg == 2 ? launch_taps<T, 2>(d, out, p, x, dy, to, part, stream)
                       : launch_taps<T, 1>(d, out, p, x, dy, to, part, stream);
    }
    return fail(WC_ERR_UNSUPPORTED, "tap form of the weight gradient: 16-bit types");
  });
}

}  // namespace wc
