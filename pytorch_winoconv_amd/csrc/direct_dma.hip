// The direct form of 16-bit types: y (pixels x K) = pixels of x under the taps (pixels x kh kw C) times U (K, kh kw C), a product
// whose first operand is x itself, and up to four such products in one launch (the parity classes of a strided layer's input
// gradient; workgroup b works on class b % n, so that the classes, whose reductions differ, share out every XCD).
//
// The register-staged kernel (gemm_kernel<..., DIRECT>, gemm.hip) has one stage of 32 channels in flight beside the one it
// multiplies, and walks the taps one after the other over all channels: a pixel's next use is megabytes of other pixels away,
// and x, read 2.25 times at stride 2, came 2.2 times from beyond L2.  Here
//  - LDS-DMA brings the operands (no registers, no VALU stores): two stages are in flight while a third is multiplied, with one
//    barrier per stage and exact counts of what may still be on its way.  Pixels outside the image are loads outside the
//    descriptor's range, which bring zeros; bit masks per row say which taps those are, so a tap costs a wavefront four
//    instructions per load;
//  - taps that read the same pixels (equal modulo the stride) follow each other for each block of 32 channels, so that all
//    readings but the first come from L2 (fetched 1.04 times, N=41 128 channels, 112x112 at stride 2).
// Rows of 64 bytes in LDS with their 16-byte chunks swizzled by the row, as in gemm_kernel (LDS-DMA writes 16 whole rows per
// instruction; each lane fetches the chunk that belongs where it writes).  Four wavefronts; a stage of the 256 x 128 tile is 24 KB
// and 16 products of 32x32x16 per SIMD, and takes a CU 0.50 us whether one or two workgroups share it (the products alone
// 0.38, what the matrix cores sustain); a launch has 7 us beside its stages.
//
// Measured, us, fp16, register-staged | this, x in rotation: stride 2, 3x3 128 -> 128, 112x112 N=8 27 | 18, N=16 32 | 28, N=32
// 57 | 44, N=64 111 | 87; N=1 56x56 12.3 | 9.5; N=2 256 -> 512, 15x17 20 | 14.4; N=64 256 -> 512, 28x28 51 | 43; 1x1 64 -> 256 56x56 N=64 20.7 | 12.8; input
// gradients (classes turned, class_of_block) N=32 128 <- 128, 112x112 86 | 51, 128 <- 256, 56x56 42 | 29, N=64 256 <- 512, 28x28 75 | 54.
#include "lds_dma.h"
#include "wc_transform.h"

#include <algorithm>

namespace wc {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct MfmaD;
template <> struct MfmaD<half_t> {
  using Frag = f16x8;
  __device__ static __forceinline__ f32x16 run(Frag a, Frag b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};
template <> struct MfmaD<bf16_t> {
  using Frag = bf16x8;
  __device__ static __forceinline__ f32x16 run(Frag a, Frag b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};

// acc += a b in place.  The builtin's result may be another register than its addend, and with two stages of a loop's body the compiler
// chose so, and copied every accumulator back.  It does not know these as matrix instructions, and waits for none of their results: nothing
// but them may touch the accumulators up to mfma16_done (tests/test_wide_tile_code.py looks the built code through for that).
template <typename T>
__device__ __forceinline__ void mfma16(f32x4& acc, typename MfmaD<T>::Frag a, typename MfmaD<T>::Frag b) {
  if constexpr (std::is_same_v<T, half_t>)
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// The wait, of eight passes at most, that a row of accumulators goes through before it is read
__device__ __forceinline__ void mfma16_done(f32x4 (&a)[8]) {
  asm volatile("s_nop 15" : "+a"(a[0]), "+a"(a[1]), "+a"(a[2]), "+a"(a[3]), "+a"(a[4]), "+a"(a[5]), "+a"(a[6]), "+a"(a[7]));
}

struct DirectDmaArgs {
  const void* x; const void* bias; void* y;
  long long x_bytes;
  int H, W, C, K, cblocks, stride;
  int tiles_k, n_blocks, per_xcd, n_classes;
  int o_step, o_H, o_W;           // as in gemm_direct_conv; o_step 0: rows one after the other
  struct Class {
    const void* U;
    int P, tiles_p, kh, kw, oH, oW, pad_h, pad_w, o_y0, o_x0, u_bytes;
    FastDiv f_image, f_row;       // by oH oW, by oW
  } cls[4];
};

__device__ __forceinline__ int row_swizzle(int r) { return (((r >> 1) ^ (r >> 3)) & 1) | (((r >> 2) & 1) << 1); }

constexpr int kWideStages = 4;

constexpr int direct_dma_lds(int BM, int BN, int S) {
  const int stages = S * (BM + BN) * 64, out = BM * (BN + 8) * 2;
  return stages > out ? stages : out;
}

// What a workgroup brings to LDS: stage after stage of BM pixels and BN output channels x 32 channels, each wavefront LA and LB loads of 16
// rows of 64 bytes.
//
// Offsets are from the first pixel (inside the image or not) of the first image row that the tile reads: they fit 31 bits (the
// host has checked it) and are not negative.  Taps outside the image have a set bit in out_y or out_x, and bit 31 puts a
// load out of the descriptor's range: it brings zeros.
template <int LA, int LB, int RING>
struct DirectOperands {
  static constexpr int BM = LA * 64, STAGE = (LA + LB) * 4096;
  u32x4 xd, ud;
  unsigned out_y[LA], out_x[LA], base[LA], uoff[LB], xoff[LA], uo, lds0;
  int nk, left, sload;                              // stages, those still to load and the ring's place for the next
  int tap_y, tap_x, phase_y, phase_x, cb, wave;

  __device__ __forceinline__ DirectOperands(const DirectDmaArgs& a, const DirectDmaArgs::Class& c, int p0, int k0, int w, int lane, const unsigned char* lds)
      : wave(w) {
    const int per = c.oH * c.oW, b0 = fast_div(p0, c.f_image), oy0 = fast_div(p0 - b0 * per, c.f_row);
    const long long row0 = (long long)b0 * a.H + min(oy0 * a.stride, a.H) - c.pad_h;
    const long long start = (row0 * a.W - c.pad_w) * a.C * 2;
    xd = dma_descriptor(static_cast<const unsigned char*>(a.x) + start, a.x_bytes - start);
    ud = dma_descriptor(c.U, c.u_bytes);
    auto outside = [](int first, int size, int taps) {             // bit t: first + t is not in 0 .. size - 1
      const int lo = min(max(-first, 0), taps), hi = min(max(size - first, 0), taps);
      return ~(unsigned)(((1ull << hi) - 1) & ~((1ull << lo) - 1));
    };
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      const int row = (wave * LA + i) * 16 + (lane >> 2), p = min(p0 + row, c.P - 1);
      const int b = fast_div(p, c.f_image), rem = p - b * per, oy = fast_div(rem, c.f_row), ox = rem - oy * c.oW;
      out_y[i] = p0 + row < c.P ? outside(oy * a.stride - c.pad_h, a.H, c.kh) : ~0u;
      out_x[i] = outside(ox * a.stride - c.pad_w, a.W, c.kw);
      base[i] = (unsigned)((((long long)b * a.H + oy * a.stride - c.pad_h - row0) * a.W + ox * a.stride) * a.C * 2) + ((lane & 3) ^ row_swizzle(row)) * 16;
    }
    const int u_row = c.kh * c.kw * a.C * 2;
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int row = (wave * LB + i) * 16 + (lane >> 2);
      uoff[i] = k0 + row < a.K ? (k0 + row) * u_row + ((lane & 3) ^ row_swizzle(row)) * 16 : kOutside;
    }
    nk = left = c.kh * c.kw * a.cblocks;
    lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)lds;
    sload = tap_y = tap_x = phase_y = phase_x = cb = 0;
    offsets(a, c);
  }
  __device__ __forceinline__ void offsets(const DirectDmaArgs& a, const DirectDmaArgs::Class& c) {
    const unsigned xo = (unsigned)((tap_y * a.W + tap_x) * a.cblocks + cb) * 64;
#pragma unroll
    for (int i = 0; i < LA; ++i) xoff[i] = (((out_y[i] << (31 - tap_y)) | (out_x[i] << (31 - tap_x))) & 0x80000000u) | (base[i] + xo);
    uo = (unsigned)((tap_y * c.kw + tap_x) * a.cblocks + cb) * 64;
  }
  __device__ __forceinline__ void issue_part(int i) {          // load i of LA + LB
    const unsigned to = lds0 + sload * STAGE;
    if (i < LA) {
      u32x4 xs = xd;
      if (left <= 0) xs[2] = 0;                    // beyond the last stage: loads that reach no memory, for the counts
      dma16(xs, xoff[i], to + (wave * LA + i) * 1024);
    } else {
      u32x4 us = ud;
      if (left <= 0) us[2] = 0;
      dma16(us, uoff[i - LA] + uo, to + BM * 64 + (wave * LB + i - LA) * 1024);
    }
  }
  __device__ __forceinline__ void issue() {
#pragma unroll
    for (int i = 0; i < LA + LB; ++i) issue_part(i);
  }
  // BRANCHES: most taps need the first two lines only, which is faster between short stages (us, 1 x 192 -> 32, 29x29 stride 2 12.7 | 11.1, N=25 128 ->
  // 224, 34x34 15.0 | 13.4); without, a step is one block of code for the scheduler
  template <bool BRANCHES>
  __device__ __forceinline__ void advance(const DirectDmaArgs& a, const DirectDmaArgs::Class& c) {
    --left;
    sload = sload == RING - 1 ? 0 : sload + 1;
    if constexpr (BRANCHES) {
      tap_x += a.stride;
      if (tap_x >= c.kw) {
        tap_x = phase_x;
        tap_y += a.stride;
        if (tap_y >= c.kh) {
          tap_y = phase_y;
          if (++cb == a.cblocks) {
            cb = 0;
            if (++phase_x == min(a.stride, c.kw)) { phase_x = 0; tap_y = ++phase_y; }
            tap_x = phase_x;
          }
        }
      }
      offsets(a, c);
      return;
    }
    const int nx = tap_x + a.stride;
    const bool row_done = nx >= c.kw;
    const int ny = tap_y + (row_done ? a.stride : 0);
    const bool taps_done = ny >= c.kh;
    cb += taps_done ? 1 : 0;
    const bool phase_done = cb == a.cblocks;
    phase_x += phase_done ? 1 : 0;
    const bool phases_done = phase_x == min(a.stride, c.kw);
    cb = phase_done ? 0 : cb;
    phase_x = phases_done ? 0 : phase_x;
    phase_y += phases_done ? 1 : 0;
    tap_x = row_done ? phase_x : nx;
    tap_y = taps_done ? phase_y : ny;
    offsets(a, c);
  }
};

// Rows of a tile from LDS (pitch BN + 8) to y
template <typename T, int BM, int BN>
__device__ __forceinline__ void direct_rows_out(const DirectDmaArgs& a, const DirectDmaArgs::Class& c, const T* cs, int p0, int k0, int tid) {
  constexpr int CS = BN + 8, CPRO = BN / 8, RPPO = 256 / CPRO;
  const int per = c.oH * c.oW, orow = tid / CPRO, ocol = tid % CPRO * 8;
  if (k0 + ocol >= a.K) return;
#pragma unroll 4
  for (int r = 0; r < BM / RPPO; ++r) {
    const int row = orow + r * RPPO, p = p0 + row;
    if (p >= c.P) break;
    long long to = p;
    if (a.o_step) {
      const int b = fast_div(p, c.f_image), rem = p - b * per, oy = fast_div(rem, c.f_row), ox = rem - oy * c.oW;
      to = ((long long)b * a.o_H + oy * a.o_step + c.o_y0) * a.o_W + ox * a.o_step + c.o_x0;
    }
    *reinterpret_cast<u32x4*>(static_cast<T*>(a.y) + to * a.K + k0 + ocol) = *reinterpret_cast<const u32x4*>(cs + row * CS + ocol);
  }
}

template <typename T, int WM, int WN, int NWK, int S, int SUB>
__global__ __launch_bounds__(256, WM * WN >= 6 ? 2 : WM * WN >= 4 ? 3 : 4) void direct_dma_kernel(DirectDmaArgs a) {
  using MF = MfmaD<T>;
  constexpr int NWP = 4 / NWK, BM = 32 * NWP * WM, BN = 32 * NWK * WN;
  constexpr int LA = BM / 64, LB = BN / 64;        // loads of 16 rows of 64 bytes that each of the four wavefronts makes per stage
  constexpr int STAGE = (BM + BN) * 64;            // bytes
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[];

  int blk = xcd_remap(blockIdx.x, a.per_xcd);
  if (blk >= a.n_blocks) return;
  const DirectDmaArgs::Class c = a.cls[class_of_block(blk, a.n_classes, a.per_xcd)];
  blk /= a.n_classes;
  if (blk >= c.tiles_p * a.tiles_k) return;
  const int k0 = blk % a.tiles_k * BN, p0 = blk / a.tiles_k * BM;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  DirectOperands<LA, LB, S * SUB> in(a, c, p0, k0, wave, lane, lds_raw);
  const int nk = in.nk;
  const int wp = wave / NWK, wk = wave % NWK, l32 = lane & 31, lhi = lane >> 5;
  const int fz = row_swizzle(l32);
  const int xa = (wp * WM * 32 + l32) * 64, wa = (BM + wk * WN * 32 + l32) * 64;
  f32x16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

#pragma unroll
  for (int s = 0; s < (S - 1) * SUB; ++s) { in.issue(); in.template advance<true>(a, c); }
  int cur = 0;
  for (int kt = 0; kt < nk; kt += SUB) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((LA + LB) * (S - 2) * SUB) : "memory");
    typename MF::Frag xf[2][WM], wf[2][WN];
    auto fload = [&](int kk) {
      const unsigned char* const st = lds_raw + cur * STAGE + (kk >> 1) * STAGE;
      const int ko = (((kk & 1) * 2 + lhi) ^ fz) * 16;
#pragma unroll
      for (int i = 0; i < WM; ++i) xf[kk & 1][i] = *reinterpret_cast<const typename MF::Frag*>(st + xa + i * 2048 + ko);
#pragma unroll
      for (int j = 0; j < WN; ++j) wf[kk & 1][j] = *reinterpret_cast<const typename MF::Frag*>(st + wa + j * 2048 + ko);
    };
    fload(0);
#pragma unroll
    for (int kk = 0; kk < 2 * SUB; ++kk) {
      if ((kk & 1) == 0) in.issue();
      if (kk + 1 < 2 * SUB) fload(kk + 1);
      __builtin_amdgcn_sched_barrier(0);
      if ((kk & 1) == 0) in.template advance<true>(a, c);
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) acc[i][j] = MF::run(wf[kk & 1][j], xf[kk & 1][i], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = cur == (S - 1) * SUB ? 0 : cur + SUB;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // out through LDS, so that stores are whole rows
  constexpr int CS = BN + 8;
  T* const cs = reinterpret_cast<T*>(lds_raw);
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float bv[4] = {0.f, 0.f, 0.f, 0.f};
      const int kl = (wk * WN + j) * 32 + 8 * q + 4 * lhi;
      if (a.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (k0 + kl + e < a.K) bv[e] = static_cast<float>(static_cast<const T*>(a.bias)[k0 + kl + e]);
      }
#pragma unroll
      for (int i = 0; i < WM; ++i) {
        Pack<T, 4> o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(acc[i][j][4 * q + e] + bv[e]);
        *reinterpret_cast<Pack<T, 4>*>(cs + ((wp * WM + i) * 32 + l32) * CS + kl) = o;
      }
    }
  __syncthreads();
  direct_rows_out<T, BM, BN>(a, c, cs, p0, k0, tid);
}

// The same product on tiles of 64 WM pixels x 128 channels, one workgroup to a CU, four wavefronts of 16 WM x 128 on 16x16x32 products: for
// problems of a few more than one round of 256 x 128 tiles, whose last tiles double the work of the CUs that have them.
//
// A wavefront is alone on its SIMD, so nothing may wait: the fragments of a stage are read while the one before is multiplied (the only way that
// 4 WM + 32 registers of operands are free again in time is two sets of them, hence two stages a turn of the loop), and a stage's loads are
// spread over its rows of products (all at once, at its start, they hold the wavefront up until the last is taken: 40.2 | 36.6 us at N=8).
// Of a stage of 448 x 128, 0.74 us, products and their fragment reads alone take 0.48 and the loads alone 0.47 (78 KB/us into each
// CU from L2): they overlap by half, and 36 stages are 27 us of the 47 below: x from memory, first loads and write-out are the rest.  fp16, x in rotation, 256 x 128 | here: N=32 128 -> 128, 112x112 stride 2 52 | 49 us (50.5 | 50.3 with more between the calls), N=22 47.5 | 37.3, N=44 256 -> 256, 56x56 75 | 59.
template <typename T, int WM>
__global__ __launch_bounds__(256, 1) void direct_wide_kernel(DirectDmaArgs a) {
  using MF = MfmaD<T>;
  constexpr int BM = 64 * WM, BN = 128, S = kWideStages, L = WM + 2, STAGE = (BM + BN) * 64, WN = 8;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[];

  int blk = xcd_remap(blockIdx.x, a.per_xcd);
  if (blk >= a.n_blocks) return;
  const DirectDmaArgs::Class c = a.cls[0];
  const int k0 = blk % a.tiles_k * BN, p0 = blk / a.tiles_k * BM;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  DirectOperands<WM, 2, S> in(a, c, p0, k0, wave, lane, lds_raw);
  const int nk = in.nk;

  const int l16 = lane & 15, quad = lane >> 4, ko = (quad ^ row_swizzle(l16)) * 16;
  const int xa = (wave * WM * 16 + l16) * 64 + ko, wa = (BM + l16) * 64 + ko;
  f32x4 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  typename MF::Frag xf[2][WM], wf[2][WN];
  int cur = 0;                                      // the ring's place of the next stage to read
  auto fload = [&](auto to) {
    constexpr int B = decltype(to)::value;
    const unsigned char* const st = lds_raw + cur * STAGE;
#pragma unroll
    for (int j = 0; j < WN; ++j) wf[B][j] = *reinterpret_cast<const typename MF::Frag*>(st + wa + j * 1024);
#pragma unroll
    for (int i = 0; i < WM; ++i) xf[B][i] = *reinterpret_cast<const typename MF::Frag*>(st + xa + i * 1024);
    cur = cur == S - 1 ? 0 : cur + 1;
  };

#pragma unroll
  for (int s = 0; s < S; ++s) { in.issue(); in.template advance<false>(a, c); }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(L * (S - 1)) : "memory");
  fload(ic<0>{});
  // Stage kt is in registers; kt + 1 must have landed (two more may be on their way), and everyone has read kt, whose place takes kt + S
  auto step = [&](auto from) {
    constexpr int B = decltype(from)::value;
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(L * (S - 2)) : "memory");
    const unsigned char* const st = lds_raw + cur * STAGE;
    cur = cur == S - 1 ? 0 : cur + 1;
#pragma unroll
    for (int i = 0; i < WM; ++i) {                  // a row of products; the next stage's fragments come beside the first ones
      xf[1 - B][i] = *reinterpret_cast<const typename MF::Frag*>(st + xa + i * 1024);
      if (i < 4) {
        wf[1 - B][2 * i] = *reinterpret_cast<const typename MF::Frag*>(st + wa + 2 * i * 1024);
        wf[1 - B][2 * i + 1] = *reinterpret_cast<const typename MF::Frag*>(st + wa + (2 * i + 1) * 1024);
      }
#pragma unroll
      for (int j = 0; j < WN; ++j) mfma16<T>(acc[i][j], wf[B][j], xf[B][i]);
      __builtin_amdgcn_sched_barrier(0);
      in.issue_part(i);
      if (i < 2) in.issue_part(WM + i);
      if (i == WM - 1) in.template advance<false>(a, c);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int kt = 0;
  do {                                              // an odd count gets a stage of zeros
    step(ic<0>{});
    step(ic<1>{});
    kt += 2;
  } while (kt < nk);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int i = 0; i < WM; ++i) mfma16_done(acc[i]);

  constexpr int CS = BN + 8;
  T* const cs = reinterpret_cast<T*>(lds_raw);
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
    const int kl = j * 16 + 4 * quad;
    if (a.bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (k0 + kl + e < a.K) bv[e] = static_cast<float>(static_cast<const T*>(a.bias)[k0 + kl + e]);
    }
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      Pack<T, 4> o;
      asm volatile("" : "+a"(acc[i][j]));           // read when it is its turn: together they do not fit beside themselves
#pragma unroll
      for (int e = 0; e < 4; ++e) o.v[e] = static_cast<T>(acc[i][j][e] + bv[e]);
      *reinterpret_cast<Pack<T, 4>*>(cs + ((wave * WM + i) * 16 + l16) * CS + kl) = o;
    }
  }
  __syncthreads();
  direct_rows_out<T, BM, BN>(a, c, cs, p0, k0, tid);
}

// The bytes from the first image row that n consecutive output pixels read to the end of the last
long long tile_span(long long n, int H, int W, int C, int kh, int stride, int oH, int oW) {
  const long long rows = (n / oW + 2) * stride + (n / ((long long)oH * oW) + 1) * std::max(0, H - (oH - 1) * stride) +
                         std::max(0, (oH - 1) * stride - H) + kh;
  return rows * W * C * 2;
}

}  // namespace

bool direct_dma_fits(const DirectClass* classes, int n, int H, int W, int C, int K, int stride) {
  for (int i = 0; i < n; ++i) {
    const DirectClass& d = classes[i];
    if (tile_span(256, H, W, C, d.kh, stride, d.oH, d.oW) >= (1ll << 31) || (long long)K * d.kh * d.kw * C * 2 >= (1ll << 31) || d.kh > 32 || d.kw > 32) return false;
  }
  return true;
}

template <typename T>
static int launch_direct_dma(DirectDmaArgs a, const DirectClass* classes, int N, int tile, void* stream) {
  auto start = [&](auto bm, auto bn, auto fn, int lds) -> int {
    constexpr int BM = decltype(bm)::value, BN = decltype(bn)::value;
    int most = 0;
    for (int i = 0; i < a.n_classes; ++i) {
      const DirectClass& d = classes[i];
      const long long P = (long long)N * d.oH * d.oW;
      a.cls[i] = {d.U, (int)P, ceil_div((int)P, BM), d.kh, d.kw, d.oH, d.oW, d.pad_h, d.pad_w, d.o_y0, d.o_x0,
                  (int)((long long)a.K * d.kh * d.kw * a.C * 2), make_fast_div(d.oH * d.oW), make_fast_div(d.oW)};
      most = std::max(most, a.cls[i].tiles_p);
    }
    a.tiles_k = ceil_div(a.K, BN);
    const long long blocks = (long long)most * a.tiles_k * a.n_classes;
    WC_CHECK_ARG(blocks < (1ll << 30), "direct_dma: problem too large");
    a.n_blocks = (int)blocks;
    a.per_xcd = ceil_div((int)blocks, kXcds);
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds)) return rc;
    hipLaunchKernelGGL(fn, dim3((unsigned)(a.per_xcd * kXcds)), dim3(256), lds, as_stream(stream), a);
    WC_CHECK_LAUNCH("direct_dma_kernel");
    return WC_OK;
  };
  auto launch = [&](auto wm, auto wn, auto nwk, auto s, auto sub) -> int {
    constexpr int WM = decltype(wm)::value, WN = decltype(wn)::value, NWK = decltype(nwk)::value, S = decltype(s)::value, SUB = decltype(sub)::value;
    constexpr int BM = 32 * (4 / NWK) * WM, BN = 32 * NWK * WN;
    return start(ic<BM>{}, ic<BN>{}, &direct_dma_kernel<T, WM, WN, NWK, S, SUB>, direct_dma_lds(BM, BN, S * SUB));
  };
  auto wide = [&](auto wm) -> int {
    constexpr int WM = decltype(wm)::value;
    return start(ic<64 * WM>{}, ic<128>{}, &direct_wide_kernel<T, WM>, direct_dma_lds(64 * WM, 128, kWideStages));
  };
  switch (tile) {
    case 5: return wide(ic<5>{});                                             // 320 x 128 .. 448 x 128
    case 6: return wide(ic<6>{});
    case 7: return wide(ic<7>{});
    case 0: return launch(ic<4>{}, ic<2>{}, ic<2>{}, ic<3>{}, ic<1>{});      // 256 x 128
    case 1: return launch(ic<2>{}, ic<2>{}, ic<2>{}, ic<3>{}, ic<1>{});      // 128 x 128
    case 2: return launch(ic<2>{}, ic<2>{}, ic<1>{}, ic<3>{}, ic<1>{});      // 256 x 64
    case 3: return launch(ic<2>{}, ic<1>{}, ic<2>{}, ic<4>{}, ic<1>{});      // 128 x 64
    default: return launch(ic<1>{}, ic<1>{}, ic<2>{}, ic<3>{}, ic<2>{});     // 64 x 64, 64 channels between barriers
  }
}

// P: pixels of all classes.  us, fp16, 256x128 | 128x128 | 64x64 tile (256x64 | 128x64 | 64x64 for 64 channels):
//   forward, 256x128 tiles in all: 392 44 | 54 | 67, 294 41 | 40 | 52, 196 27.4 | 28 | 37 and 43 | 45 | 65, 98 24 | 18 | 22, 74 24 | 17.6 | 18; 128x128
//   tiles in all: 79 14.4 | 10.4, 50 27 | 15;   64 channels, 256x64 tiles in all: 391 14.9 | 15.8 | 15.6, 98 11.3 | 8.7 | 9.1
//   classes, rounds of 256x128 tiles and input channels (those of dy), 256x128 | 128x128: 0.7 18.4 | 16.0 (128), 25.9 | 22.2 (256), 45 | 37 (512); 1.0
//   20.2 | 19.1, 28.5 | 28.1, 49 | 51; 1.5 22.0 | 19.9, 30.9 | 28.9, 54 | 61; 2.2 33 | 28, 49 | 41, 86 | 73; 3.3 35.2 | 34.7, 53.7 | 54.4, 95 | 99; 5.5 50.2
//   | 50.1, 81 | 84, 142 | 153; 128x128 | 64x64 in tiles of 128x128: 196 22 | 22 and 20 | 23, 28 34 | 25;   64 channels, 256x64 | 128x64: 0.7 rounds 13.2 | 14.5, 5.5 37 | 44
//   forward, rounds of 256x128 tiles and stages of a tile, x in rotation, 256x128 | 320, 384 or 448 x 128: 1.05 27.0 | 23.8 (18), 47.5 | 37.3 (36), 75 | 59 (72);
//   1.45 30.5 | 28.3, 50 | 44, 80 | 69; 1.7 32.4 | 32.9, 52.7 | 49.9, 85 | 78; 2.2 48 | 49, 76 | 72, 124 | 115; 2.7 50 | 55, 79.6 | 82.9, 129 | 133; 3.3
//   62 | 63, 100 | 97, 163 | 154; 4.4 (three rounds of the middle one) 79 | 81, 129 | 129, 213 | 205; reductions of 9 stages lose or draw
// The large tile, two to a CU, wherever most CUs have one, and where a few more than one or two rounds of them would be left, as many rows more in
// a tile as make whole rounds; classes, whose tiles are of four lengths, share out better in smaller
// ones unless the reduction is long and the large tiles are there at once, or many.
static int choose_tile(long long P, int C, int K, int taps, bool classes, bool wide_fits) {
  const int force = test_gemm_config();
  if (force >= 22 && force <= (wide_fits ? 29 : 26)) return force - 22;
  auto tiles = [&](int bm, int bn) { return ceil_div_ll(P, bm) * ceil_div(K, bn); };
  if (K <= 64) {
    const long long t = tiles(256, 64);
    return t > 2 * kCus ? 3 : t >= kCus ? 2 : 4;
  }
  const long long big = tiles(256, 128), mid = tiles(128, 128);
  if (classes) {
    const bool full = K % 128 == 0 || K % 128 > 64;
    if (full && ((C >= 512 && big >= kCus && big <= 2 * kCus) || (C >= 256 && big >= 3 * kCus))) return 0;
    return mid >= 3 * kCus / 4 ? 1 : 4;
  }
  const int stages = taps * C / 32;
  if (wide_fits)
    for (int wm = 5; wm <= 7; ++wm) {
      const long long rounds = ceil_div_ll(tiles(64 * wm, 128), kCus);
      if (rounds > 2 || big <= rounds * kCus) continue;
      if (rounds == 1 ? stages >= (wm < 7 ? 18 : 36) : wm != 6 && stages >= 36) return wm;
      break;
    }
  return big >= 3 * kCus / 4 ? 0 : mid >= kCus / 2 ? 1 : 4;
}

int direct_dma(const void* x, const DirectClass* classes, int n, const void* bias, void* y, int N, int H, int W, int C, int K, int stride,
               int dtype, void* stream, int o_step, int o_H, int o_W) {
  long long P = 0;
  for (int i = 0; i < n; ++i) P += (long long)N * classes[i].oH * classes[i].oW;
  const DirectClass& first = classes[0];
  const bool wide_fits = n == 1 && tile_span(448, H, W, C, first.kh, stride, first.oH, first.oW) < (1ll << 31);
  const int tile = choose_tile(P, C, K, first.kh * first.kw, n > 1, wide_fits);
  for (int i = 0; i < n; ++i)
    WC_CHECK_ARG(classes[i].U && classes[i].oH > 0 && classes[i].oW > 0 && (long long)N * classes[i].oH * classes[i].oW < (1ll << 31), "direct_dma: problem too large");
  DirectDmaArgs a{};
  a.x = x; a.bias = bias; a.y = y; a.x_bytes = (long long)N * H * W * C * 2;
  a.H = H; a.W = W; a.C = C; a.K = K; a.cblocks = C / 32; a.stride = stride; a.n_classes = n;
  a.o_step = o_step; a.o_H = o_H; a.o_W = o_W;
  return dtype == WC_F16 ? launch_direct_dma<half_t>(a, classes, N, tile, stream) : launch_direct_dma<bf16_t>(a, classes, N, tile, stream);
}

}  // namespace wc
