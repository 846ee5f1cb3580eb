// Batched product with the reduction along the rows of both operands:
//
//   D[t][s] (na x nb, fp32) = sum over rows p of part s of  A[t][p][0..na) (x) B[t][p][0..nb)
//
// This is the contraction over the tiles in the weight gradient (dU = dM^T V per transform
// element): both operands are stored the way the forward kernels write them, rows = tiles,
// channels contiguous, and nothing is transposed in memory.  The reference has no counterpart
// (its backward pass was never written: src/back/utils.cu:15-24).
//
// A stage holds BK rows of each operand exactly as they lie in memory (16-byte loads and LDS
// stores of whole rows).  The MFMA operands need 8 consecutive reduction elements per lane, which
// in this layout are a column: for 16-bit types ds_read_b64_tr_b16 delivers exactly that (16 lanes
// read 4 rows x 32 bytes, and lane j receives column j of the 4 x 16 block), for fp32 the operand
// of v_mfma_f32_32x32x2_f32 is a single element and a plain 4-byte read of a row does.  LDS rows
// are padded by 32 bytes so that the 4 rows of a transposing read fall into different banks.
//
// The reduction is split into S parts of Pq rows (few outputs, a long reduction: the parts are
// what fills the chip); the caller adds the parts.  Workgroup = 4 wavefronts (2 x 2), each owning
// W x W blocks of 32 x 32.  V feeds the MFMA "A" side, so a lane ends up with 4 consecutive
// columns of D and stores them as one 16-byte write.
#include "column_sums.h"
#include "lds_dma.h"
#include "split_bf16.h"
#include "wc_transform.h"

#include <algorithm>

namespace wc {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef short short8v __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t Chunk16 __attribute__((ext_vector_type(4)));

struct GemmTnArgs {
  const void* A;             // (T, P, lda)
  const void* B;             // (T, P, ldb)
  float* D;                  // (T, S, na, ldd)
  long long P;
  int lda, ldb, na, nb, ldd;
  int S, Pq;
  int tiles_a, tiles_b;
  int n_blocks, per_xcd;
  // GATHER (the weight gradient of a convolution taken directly, one batch per tap): A is dy (P = N oH oW rows, the
  // same for every batch), B is x itself, and row p = (b, oy, ox) of batch t = (ky, kx) is the pixel
  // (stride oy + ky - pad_h, stride ox + kx - pad_w) of image b, zeros outside the image
  int H, W, oH, oW, conv_stride, pad_h, pad_w, kw;
  FastDiv div_per, div_oW;
  long long b_elems;         // of x
  // the taps of a part as neighbours, which read the same rows of dy and mostly the same of x, where these are more than L2
  // holds; 0: the parts of a tap, which do not meet at the same lines (us, fp16, stride 2, taps | parts: N=32 128 -> 128, 112x112, 128 MB
  // in all, 60 | 90, N=64 64 -> 64, 56x56, 32 MB 38 | 44; N=16 96 -> 96, 50x50, 10 MB 27.5 | 26.5, N=8 128 -> 128, 56x56, 8 MB 27 | 23)
  int n_taps;
  float* sums;               // column sums of A, a row of tiles_a times the tile's columns per (s, t, tile of B); null: none
  int T;
};

__device__ __forceinline__ floatx16 mfma16(short8v a, short8v b, floatx16 c, half_t) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}
__device__ __forceinline__ floatx16 mfma16(short8v a, short8v b, floatx16 c, bf16_t) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <typename T, int W, int BK, bool GATHER = false>
__global__ __launch_bounds__(256, 2) void gemm_tn_kernel(GemmTnArgs g) {
  constexpr int BT = 64 * W;                       // tile extent on both output axes
  constexpr int EPC = 16 / sizeof(T);              // elements per 16-byte chunk
  constexpr int PITCH = BT + 32 / sizeof(T);       // LDS row, elements
  constexpr int CPR = BT / EPC;                    // chunks per row
  constexpr int RPP = 256 / CPR;                   // rows per load pass
  constexpr int NL = BK / RPP;                     // load passes per operand
  constexpr int STAGE = 2 * BK * PITCH;            // A rows, then B rows
  static_assert(RPP * CPR == 256 && NL * RPP == BK && NL >= 1, "tile shape");

  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  T* lds = reinterpret_cast<T*>(lds_raw);

  const int blk = xcd_remap(blockIdx.x, g.per_xcd);
  if (blk >= g.n_blocks) return;
  const int tb = blk % g.tiles_b;
  const int ta = (blk / g.tiles_b) % g.tiles_a;
  const int ts = blk / (g.tiles_b * g.tiles_a);
  const int s = GATHER && g.n_taps ? ts / g.n_taps : ts % g.S;
  const int t = GATHER && g.n_taps ? ts % g.n_taps : ts / g.S;
  const int a0 = ta * BT, b0 = tb * BT;
  const long long p_begin = (long long)s * g.Pq;
  const long long p_end = min(g.P, p_begin + g.Pq);
  const int nk = p_end > p_begin ? (int)((p_end - p_begin + BK - 1) / BK) : 0;

  const T* Ap = static_cast<const T*>(g.A) + (GATHER ? 0 : (long long)t * g.P * g.lda);
  const T* Bp = static_cast<const T*>(g.B) + (GATHER ? 0 : (long long)t * g.P * g.ldb);
  const int tap_y = GATHER ? t / g.kw : 0, tap_x = GATHER ? t - tap_y * g.kw : 0;

  const int tid = threadIdx.x;
  const int lrow = tid / CPR, lcol = (tid % CPR) * EPC;
  const bool a_in = a0 + lcol < g.lda, b_in = b0 + lcol < g.ldb;   // ld is a multiple of 8: whole chunks

  Chunk16 ra[NL], rb[NL];
  auto gload = [&](int kt) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const long long p = p_begin + (long long)kt * BK + lrow + i * RPP;
      const Chunk16 zero = {0u, 0u, 0u, 0u};
      ra[i] = (p < p_end && a_in) ? *reinterpret_cast<const Chunk16*>(Ap + p * g.lda + a0 + lcol) : zero;
      if constexpr (GATHER) {
        const int pi = (int)min(p, g.P - 1);
        const int b = fast_div(pi, g.div_per), rem = pi - b * (g.oH * g.oW);
        const int oy = fast_div(rem, g.div_oW), ox = rem - oy * g.oW;
        const int iy = oy * g.conv_stride + tap_y - g.pad_h, ix = ox * g.conv_stride + tap_x - g.pad_w;
        const bool inside = (unsigned)iy < (unsigned)g.H && (unsigned)ix < (unsigned)g.W;
        rb[i] = (p < p_end && b_in && inside)
                    ? *reinterpret_cast<const Chunk16*>(Bp + (((long long)b * g.H + iy) * g.W + ix) * g.ldb + b0 + lcol) : zero;
      } else {
        rb[i] = (p < p_end && b_in) ? *reinterpret_cast<const Chunk16*>(Bp + p * g.ldb + b0 + lcol) : zero;
      }
    }
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int off = buf * STAGE + (lrow + i * RPP) * PITCH + lcol;
      *reinterpret_cast<Chunk16*>(lds + off) = ra[i];
      *reinterpret_cast<Chunk16*>(lds + off + BK * PITCH) = rb[i];
    }
  };

  const int lane = tid & 63, wave = tid >> 6;
  const int wa = wave >> 1, wb = wave & 1;
  const int l32 = lane & 31, lhi = lane >> 5;

  floatx16 acc[W][W];
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // offset of a lane's fragment source inside a stage, for block 0 of its wavefront and step 0
  int fa, fb;
  if constexpr (sizeof(T) == 2) {
    // 16-lane group b reads rows 8*lhi + (0..3), columns 16*(b&1) + (0..15); lane s of the group
    // supplies the 4 elements at row s/4, columns 4*(s%4)..+3 and receives column s of the block
    const int b = lane >> 4, sl = lane & 15;
    const int row = 8 * lhi + (sl >> 2), col = 16 * (b & 1) + 4 * (sl & 3);
    fa = row * PITCH + wa * W * 32 + col;
    fb = BK * PITCH + row * PITCH + wb * W * 32 + col;
  } else {
    fa = lhi * PITCH + wa * W * 32 + l32;
    fb = BK * PITCH + lhi * PITCH + wb * W * 32 + l32;
  }

  if (nk > 0) {
    gload(0);
    lstore(0);
  }
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) gload(kt + 1);
    const T* st = lds + cur * STAGE;
    if constexpr (sizeof(T) == 2) {
      typedef short4v __attribute__((address_space(3))) * LdsVec;
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk) {
        short8v af[W], bf[W];
#pragma unroll
        for (int i = 0; i < W; ++i) {
          const T* src = st + fa + kk * 16 * PITCH + i * 32;
          const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsVec)(src));
          const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsVec)(src + 4 * PITCH));
          af[i] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
#pragma unroll
        for (int j = 0; j < W; ++j) {
          const T* src = st + fb + kk * 16 * PITCH + j * 32;
          const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsVec)(src));
          const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsVec)(src + 4 * PITCH));
          bf[j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
#pragma unroll
        for (int i = 0; i < W; ++i)
#pragma unroll
          for (int j = 0; j < W; ++j) acc[i][j] = mfma16(bf[j], af[i], acc[i][j], T{});
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < BK / 2; ++kk) {
        float af[W], bf[W];
#pragma unroll
        for (int i = 0; i < W; ++i) af[i] = st[fa + kk * 2 * PITCH + i * 32];
#pragma unroll
        for (int j = 0; j < W; ++j) bf[j] = st[fb + kk * 2 * PITCH + j * 32];
#pragma unroll
        for (int i = 0; i < W; ++i)
#pragma unroll
          for (int j = 0; j < W; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(bf[j], af[i], acc[i][j], 0, 0, 0);
      }
    }
    if (kt + 1 < nk) lstore(cur ^ 1);
    __syncthreads();
  }

  // accumulator (i, j), register 4q + e: row a0 + 32 (W wa + i) + l32, column b0 + 32 (W wb + j) + 8q + 4 lhi + e
  float* Dt = g.D + ((long long)t * g.S + s) * g.na * g.ldd;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    const int row = a0 + (wa * W + i) * 32 + l32;
    if (row >= g.na) continue;
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = b0 + (wb * W + j) * 32 + 8 * q + 4 * lhi;
        if (col < g.ldd) {
          floatx4 o = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
          *reinterpret_cast<floatx4*>(Dt + (long long)row * g.ldd + col) = o;
        }
      }
  }
}

// 16-bit types with both operands brought to LDS by LDS-DMA, three stages of 32 rows ahead.  Rows are not padded: their 64-byte
// pieces are exchanged by the row instead, so that the 4 rows of a transposing read fall into different banks.  Rows past the
// part's end and pixels outside the image are offsets outside the descriptor's range, which bring zeros.  GATHER: where the
// rows of x lie is worked out for 64 rows at a time by one wavefront and read from a table in LDS.
// gemm_tn_kernel waits for each of its loads, which stand behind branches, a stage after it asked for them.  us, whole gradients in fp16, through
// registers | by LDS-DMA: N=64 256 -> 512, 28x28 at stride 2 67 | 55, 1x1 64 -> 256, 56x56 54 | 40, F(4,3) of 512 -> 512, 56x56 N=32 372 | 339; N=32 128 ->
// 128, 112x112 at stride 2 85 | 90, bound by the same rows of x and dy from beyond L2 for every tap, and 60 with the taps as neighbours (n_taps).
constexpr int kTnRows = 32, kTnStages = 4;
template <int W> constexpr int tn_dma_lds() { return kTnStages * 2 * kTnRows * W * 128 + 4 * 64 * 4; }

template <typename T, int W, bool GATHER>
__global__ __launch_bounds__(256, 2) void gemm_tn_dma_kernel(GemmTnArgs g) {
  constexpr int BT = 64 * W, PITCH = BT * 2, HALF = kTnRows * PITCH, STAGE = 2 * HALF;     // bytes: A's rows, then B's
  constexpr int L = W, RPI = 8 / W;                // loads of 1 KB of each operand per wavefront and stage, rows per load
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[];
  unsigned* const table = reinterpret_cast<unsigned*>(lds_raw + kTnStages * STAGE);        // rows 64 j .. 64 j + 63 of the part at (j & 3) * 64

  const int blk = xcd_remap(blockIdx.x, g.per_xcd);
  if (blk >= g.n_blocks) return;
  const int tb = blk % g.tiles_b;
  const int ta = (blk / g.tiles_b) % g.tiles_a;
  const int ts = blk / (g.tiles_b * g.tiles_a);
  const int s = GATHER && g.n_taps ? ts / g.n_taps : ts % g.S;
  const int t = GATHER && g.n_taps ? ts % g.n_taps : ts / g.S;
  const int a0 = ta * BT, b0 = tb * BT;
  const long long p_begin = (long long)s * g.Pq;
  const int rows = (int)max(min(g.P - p_begin, (long long)g.Pq), 0ll);
  const int nk = (rows + kTnRows - 1) / kTnRows;

  const T* const Ap = static_cast<const T*>(g.A) + ((GATHER ? 0 : (long long)t * g.P) + p_begin) * g.lda + a0;
  const Chunk16 ad = dma_descriptor(Ap, ((long long)rows * g.lda - a0) * 2);
  const int image0 = GATHER ? fast_div((int)min(p_begin, g.P - 1), g.div_per) : 0;
  const long long b_start = GATHER ? (long long)image0 * g.H * g.W * g.ldb + b0 : ((long long)t * g.P + p_begin) * g.ldb + b0;
  const T* const Bp = static_cast<const T*>(g.B) + b_start;
  const Chunk16 bd = dma_descriptor(Bp, (GATHER ? g.b_elems - b_start : (long long)rows * g.ldb - b0) * 2);
  const int tap_y = GATHER ? t / g.kw : 0, tap_x = GATHER ? t - tap_y * g.kw : 0;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  auto fill = [&](int j) {                         // by one wavefront
    const int row = j * 64 + lane, pi = (int)min(p_begin + row, g.P - 1);
    const int b = fast_div(pi, g.div_per), rem = pi - b * (g.oH * g.oW);
    const int oy = fast_div(rem, g.div_oW), ox = rem - oy * g.oW;
    const int iy = oy * g.conv_stride + tap_y - g.pad_h, ix = ox * g.conv_stride + tap_x - g.pad_w;
    const bool inside = row < rows && (unsigned)iy < (unsigned)g.H && (unsigned)ix < (unsigned)g.W;
    table[(j & 3) * 64 + lane] = inside ? (unsigned)(((b - image0) * g.H + iy) * g.W + ix) * (unsigned)g.ldb * 2u : kOutside;
  };
  // a lane's 16 bytes of a row, wherever the exchange puts them; columns that are not there lie outside
  const int lrow = lane / (8 * W), chunk = W == 2 ? (lane & 15) ^ (lrow & 3) * 4 : (lane & 7) ^ ((lrow >> 1) & 1) * 4;
  const unsigned a_out = a0 + chunk * 8 < g.lda ? 0u : kOutside, b_out = b0 + chunk * 8 < g.ldb ? 0u : kOutside;
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds_raw;
  auto issue = [&](int kt) {
    const unsigned to = lds0 + (kt % kTnStages) * STAGE + wave * L * 1024;
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int row = kt * kTnRows + (wave * L + i) * RPI + lrow;
      dma16(ad, ((unsigned)row * (unsigned)g.lda * 2u + chunk * 16) | a_out, to + i * 1024);
      const unsigned off = GATHER ? table[row & 255] : (unsigned)row * (unsigned)g.ldb * 2u;
      dma16(bd, (off + chunk * 16) | b_out, to + HALF + i * 1024);
    }
  };

  const int wa = wave >> 1, wb = wave & 1, l32 = lane & 31, lhi = lane >> 5;
  floatx16 acc[W][W];
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // 16-lane group b reads rows 8 lhi + (0..3), columns 16 (b & 1) + (0..15), as in gemm_tn_kernel
  int fa[W], fb[W];
  {
    const int sl = lane & 15, row = 8 * lhi + (sl >> 2), col = ((lane >> 4) & 1) * 32 + (sl & 3) * 8;
    const int swap = W == 2 ? (row & 3) * 64 : ((row >> 1) & 1) * 64;
#pragma unroll
    for (int i = 0; i < W; ++i) {
      fa[i] = row * PITCH + ((((wa * W + i) * 64) + col) ^ swap);
      fb[i] = HALF + row * PITCH + ((((wb * W + i) * 64) + col) ^ swap);
    }
  }

  if constexpr (GATHER) {
    if (wave < 2) fill(wave);
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < kTnStages - 1; ++k)
    if (k < nk) issue(k);
  const int holder = t * g.tiles_b + tb, turns = 4 * g.T * g.tiles_b;      // holders of these rows of A
  int turn = wave + 4 * holder;                    // stages until this wavefront adds one's rows up
  float colsum[2] = {0.f, 0.f};
  for (int kt = 0; kt < nk; ++kt) {
    if (kt + 2 < nk) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(4 * L) : "memory");
    else if (kt + 1 < nk) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(2 * L) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (kt + kTnStages - 1 < nk) issue(kt + kTnStages - 1);
    if constexpr (GATHER) {
      // rows of the stages four and five on: the next step reads the first of them
      if ((kt & 1) == 0 && kt + 4 < nk && wave == ((kt >> 1) & 3)) fill((kt >> 1) + 2);
    }
    const unsigned char* const st = lds_raw + (kt % kTnStages) * STAGE;
    if (turn == 0) {
      if (g.sums) add_rows<T, BT, PITCH, true>(st, kTnRows, lane, colsum);
      turn = turns;
    }
    --turn;
    typedef short4v __attribute__((address_space(3))) * LdsVec;
    auto read = [&](const unsigned char* src) {
      const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsVec)(src));
      const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsVec)(src + 4 * PITCH));
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
#pragma unroll
    for (int kk = 0; kk < kTnRows / 16; ++kk) {
      short8v af[W], bf[W];
#pragma unroll
      for (int i = 0; i < W; ++i) af[i] = read(st + kk * 16 * PITCH + fa[i]);
#pragma unroll
      for (int j = 0; j < W; ++j) bf[j] = read(st + kk * 16 * PITCH + fb[j]);
#pragma unroll
      for (int i = 0; i < W; ++i)
#pragma unroll
        for (int j = 0; j < W; ++j) acc[i][j] = mfma16(bf[j], af[i], acc[i][j], T{});
    }
  }

  if (g.sums) store_sums<4, BT>(colsum, reinterpret_cast<float*>(lds_raw), wave, lane, g.sums + (((long long)s * g.T * g.tiles_b + holder) * g.tiles_a + ta) * BT);
  float* const Dt = g.D + ((long long)t * g.S + s) * g.na * g.ldd;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    const int row = a0 + (wa * W + i) * 32 + l32;
    if (row >= g.na) continue;
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = b0 + (wb * W + j) * 32 + 8 * q + 4 * lhi;
        if (col < g.ldd) {
          floatx4 o = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
          *reinterpret_cast<floatx4*>(Dt + (long long)row * g.ldd + col) = o;
        }
      }
  }
}

// fp32 on the bf16 matrix cores, each operand in three parts (split_bf16.h): a stage of 16 rows is split on its way to LDS, three
// planes of rows of bf16 that the transposing reads take like 16-bit rows, two stages ahead of the products in registers.
// The caller chooses it where its error is the smaller one (see wc_conv_backward_weight).  Six products of 32x32x16 take 0.4 of the time of the eight
// of 32x32x2 they replace, and the rest of a stage is splitting.  Whole gradients on F(4,3), us, fp32 instructions | so: N=16 128 -> 128, 56x56
// 92 | 74, N=32 256 -> 256, 56x56 388 | 324, N=8 256 -> 256, 28x28 64 | 53, N=4 512 -> 512, 14x14 58 | 54, N=64 64 -> 64, 56x56 133 | 129.
template <int W> constexpr int tn_split_lds() { return 2 * 2 * 3 * 16 * (W * 128 + 32); }

template <int W>
__global__ __launch_bounds__(256, 2) void gemm_tn_split_kernel(GemmTnArgs g) {
  constexpr int BT = 64 * W, BK = 16, PITCH = BT * 2 + 32, PLANE = BK * PITCH, HALF = 3 * PLANE, STAGE = 2 * HALF;      // bytes
  constexpr int CPR = BT / 4, RPP = 256 / CPR, NL = BK / RPP;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[];
  const int blk = xcd_remap(blockIdx.x, g.per_xcd);
  if (blk >= g.n_blocks) return;
  const int tb = blk % g.tiles_b;
  const int ta = (blk / g.tiles_b) % g.tiles_a;
  const int ts = blk / (g.tiles_b * g.tiles_a);
  const int s = ts % g.S, t = ts / g.S;
  const int a0 = ta * BT, b0 = tb * BT;
  const long long p_begin = (long long)s * g.Pq;
  const int rows = (int)max(min(g.P - p_begin, (long long)g.Pq), 0ll);
  const int nk = (rows + BK - 1) / BK;
  // rows past the part's end and columns past the row's lie outside the descriptors: zeros
  const float* const Ap = static_cast<const float*>(g.A) + ((long long)t * g.P + p_begin) * g.lda + a0;
  const float* const Bp = static_cast<const float*>(g.B) + ((long long)t * g.P + p_begin) * g.ldb + b0;
  const __amdgpu_buffer_rsrc_t ad = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Ap), 0, (int)max(((long long)rows * g.lda - a0) * 4, 0ll), 0x00020000);
  const __amdgpu_buffer_rsrc_t bd = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Bp), 0, (int)max(((long long)rows * g.ldb - b0) * 4, 0ll), 0x00020000);

  const int tid = threadIdx.x, lrow = tid / CPR, lcol = tid % CPR * 4;
  const unsigned a_out = a0 + lcol < g.lda ? 0u : kOutside, b_out = b0 + lcol < g.ldb ? 0u : kOutside;
  Chunk16 ra[2][NL], rb[2][NL];
  auto gload = [&](auto set_c, int kt) {
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const unsigned row = kt * BK + lrow + i * RPP;
      ra[set][i] = __builtin_amdgcn_raw_buffer_load_b128(ad, (int)(((row * (unsigned)g.lda + lcol) * 4) | a_out), 0, 0);
      rb[set][i] = __builtin_amdgcn_raw_buffer_load_b128(bd, (int)(((row * (unsigned)g.ldb + lcol) * 4) | b_out), 0, 0);
    }
  };
  auto lstore = [&](auto set_c, int buf) {
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const Split p = split_bf16(half ? rb[decltype(set_c)::value][i] : ra[decltype(set_c)::value][i]);
        unsigned char* const to = lds_raw + buf * STAGE + half * HALF + (lrow + i * RPP) * PITCH + lcol * 2;
        *reinterpret_cast<u2*>(to) = u2{p.h[0], p.h[1]};
        *reinterpret_cast<u2*>(to + PLANE) = u2{p.m[0], p.m[1]};
        *reinterpret_cast<u2*>(to + 2 * PLANE) = u2{p.l[0], p.l[1]};
      }
  };

  const int lane = tid & 63, wave = tid >> 6, wa = wave >> 1, wb = wave & 1, l32 = lane & 31, lhi = lane >> 5;
  floatx16 acc[W][W];
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  // as in gemm_tn_kernel
  const int sl = lane & 15, frag = (8 * lhi + (sl >> 2)) * PITCH + ((lane >> 4) & 1) * 32 + (sl & 3) * 8;
  const int fa = frag + wa * W * 64, fb = HALF + frag + wb * W * 64;

  auto stage = [&](int kt, auto set_c) {
    constexpr int set = decltype(set_c)::value;      // kt % 2
    gload(set_c, kt + 2);                            // beyond the part: zeros
    const unsigned char* const st = lds_raw + set * STAGE;
    typedef short4v __attribute__((address_space(3))) * LdsVec;
    auto read = [&](const unsigned char* src) {
      const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsVec)(src));
      const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsVec)(src + 4 * PITCH));
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    short8v af[3][W], bf[3][W];
#pragma unroll
    for (int q : {2, 0, 1}) {
#pragma unroll
      for (int i = 0; i < W; ++i) af[q][i] = read(st + q * PLANE + fa + i * 64);
#pragma unroll
      for (int j = 0; j < W; ++j) bf[q][j] = read(st + q * PLANE + fb + j * 64);
    }
    static_for<0, 6>([&](auto q_c) {                 // the small products first, as in gemm_kernel
      constexpr int q = decltype(q_c)::value, qa = q == 1 ? 2 : q == 2 || q == 4 ? 1 : 0, qb = q == 0 ? 2 : q == 2 || q == 3 ? 1 : 0;
#pragma unroll
      for (int i = 0; i < W; ++i)
#pragma unroll
        for (int j = 0; j < W; ++j) acc[i][j] = mfma16(bf[qb][j], af[qa][i], acc[i][j], bf16_t{});
    });
    lstore(ic<1 - set>{}, 1 - set);
    __syncthreads();
  };
  gload(ic<0>{}, 0);
  gload(ic<1>{}, 1);
  lstore(ic<0>{}, 0);
  __syncthreads();
  // The bf16 instructions cut their sums off instead of rounding them, which a long sum of one sign shows: every 64 stages the
  // accumulators go into rounded sums (2-norm against fp64, x and dy without negative values, fp32 instructions | one sum | so:
  // N=64 256 -> 256, 56x56 2.7e-7 | 5.9e-7 | 1.4e-7, 512 -> 512 5.9e-7 | 3.0e-6 | 1.5e-7; normal ones 8.3e-6 | 7.8e-6 | 5.6e-6).
  floatx16 sum[W][W] = {};
  for (int from = 0; from < nk; from += 64) {
    const int to = min(from + 64, nk);
    for (int kt = from; kt < to; kt += 2) {          // a stage beyond the last adds zeros
      stage(kt, ic<0>{});
      stage(kt + 1, ic<1>{});
    }
#pragma unroll
    for (int i = 0; i < W; ++i)
#pragma unroll
      for (int j = 0; j < W; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          sum[i][j][e] += acc[i][j][e];
          acc[i][j][e] = 0.f;
        }
  }
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j) acc[i][j] = sum[i][j];

  // sums that an infinity has made no number, again on the fp32 instructions (as in gemm_kernel)
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j) {
      bool number = true;
#pragma unroll
      for (int e = 0; e < 16; e += 2) number = number && !__builtin_isunordered(acc[i][j][e], acc[i][j][e + 1]);
      if (__all(number)) continue;
      const int ca = (wa * W + i) * 32 + l32, cb = (wb * W + j) * 32 + l32;
      const unsigned oa = a0 + ca < g.lda ? 0u : kOutside, ob = b0 + cb < g.ldb ? 0u : kOutside;
      floatx16 again = {};
#pragma unroll 4
      for (int row = 0; row < rows; row += 2) {        // a row beyond the part: zeros
        const unsigned r = row + lhi;
        const uint32_t av = __builtin_amdgcn_raw_buffer_load_b32(ad, (int)(((r * (unsigned)g.lda + ca) * 4) | oa), 0, 0);
        const uint32_t bv = __builtin_amdgcn_raw_buffer_load_b32(bd, (int)(((r * (unsigned)g.ldb + cb) * 4) | ob), 0, 0);
        again = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(bv), __uint_as_float(av), again, 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (acc[i][j][e] != acc[i][j][e]) acc[i][j][e] = again[e];
    }

  float* const Dt = g.D + ((long long)t * g.S + s) * g.na * g.ldd;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    const int row = a0 + (wa * W + i) * 32 + l32;
    if (row >= g.na) continue;
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = b0 + (wb * W + j) * 32 + 8 * q + 4 * lhi;
        if (col < g.ldd) {
          floatx4 o = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
          *reinterpret_cast<floatx4*>(Dt + (long long)row * g.ldd + col) = o;
        }
      }
  }
}

template <typename T, int W, bool GATHER = false>
int launch_tn(GemmTnArgs g, int T_, bool split, void* stream, bool* summed) {
  constexpr int BT = 64 * W;
  constexpr int BK = sizeof(T) == 2 ? 64 : 16;     // reduction rows per stage (64: measured 5 % faster than 32)
  constexpr size_t lds = (size_t)2 * 2 * BK * (BT + 32 / sizeof(T)) * sizeof(T);
  g.tiles_a = ceil_div(g.na, BT);
  g.tiles_b = ceil_div(g.nb, BT);
  const long long blocks = (long long)g.tiles_a * g.tiles_b * g.S * T_;
  WC_CHECK_ARG(blocks < (1ll << 30), "batched_gemm_tn: problem too large");
  g.n_blocks = (int)blocks;
  g.per_xcd = ceil_div((int)blocks, kXcds);
  if constexpr (sizeof(T) == 2) {
    // by LDS-DMA where 31-bit offsets reach what a part reads, which its last stages overrun by up to 255 rows
    const long long images = GATHER ? (long long)(g.Pq - 1) / ((long long)g.oH * g.oW) + 2 : 0;
    const long long reach = (g.Pq + 256ll) * std::max(g.lda, GATHER ? 0 : g.ldb) * 2;
    if (((reinterpret_cast<uintptr_t>(g.A) | reinterpret_cast<uintptr_t>(g.B)) & 15) == 0 && reach < (1ll << 31) &&
        images * g.H * g.W * g.ldb * 2 < (1ll << 31) && g.P < (1ll << 31)) {
      if (summed) *summed = g.sums != nullptr;
      const auto fn = &gemm_tn_dma_kernel<T, W, GATHER>;
      constexpr int dma_lds = tn_dma_lds<W>();
      if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), dma_lds)) return rc;
      hipLaunchKernelGGL(fn, dim3((unsigned)(g.per_xcd * kXcds)), dim3(256), dma_lds, as_stream(stream), g);
      WC_CHECK_LAUNCH("gemm_tn_dma_kernel");
      return WC_OK;
    }
  }
  if constexpr (sizeof(T) == 4 && !GATHER) {
    if (split && (g.Pq + 64ll) * std::max(g.lda, g.ldb) * 4 < (1ll << 31)) {
      const auto fn = &gemm_tn_split_kernel<W>;
      constexpr int split_lds = tn_split_lds<W>();
      if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), split_lds)) return rc;
      hipLaunchKernelGGL(fn, dim3((unsigned)(g.per_xcd * kXcds)), dim3(256), split_lds, as_stream(stream), g);
      WC_CHECK_LAUNCH("gemm_tn_split_kernel");
      return WC_OK;
    }
  }
  if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&gemm_tn_kernel<T, W, BK, GATHER>), lds)) return rc;
  hipLaunchKernelGGL((gemm_tn_kernel<T, W, BK, GATHER>), dim3((unsigned)(g.per_xcd * kXcds)), dim3(256), lds, as_stream(stream), g);
  WC_CHECK_LAUNCH("gemm_tn_kernel");
  return WC_OK;
}

}  // namespace

int tn_sum_width(int na, int nb) { return ceil_div(na, na > 64 && nb > 64 ? 128 : 64) * (na > 64 && nb > 64 ? 128 : 64); }
int tn_sum_rows(int T_, int na, int nb, int S) { return S * T_ * ceil_div(nb, na > 64 && nb > 64 ? 128 : 64); }

int batched_gemm_tn(const void* A, const void* B, float* D, int T_, long long P, int lda, int ldb, int na, int nb,
                    int ldd, int S, int Pq, bool split, int dtype, void* stream, float* a_sums, bool* summed) {
  WC_CHECK_ARG(A && B && D, "batched_gemm_tn: null pointer");
  WC_CHECK_ARG(T_ > 0 && P > 0 && na > 0 && nb > 0 && S > 0 && Pq > 0, "batched_gemm_tn: empty problem");
  WC_CHECK_ARG(lda % 8 == 0 && ldb % 8 == 0 && ldd % 4 == 0 && lda >= na && ldb >= nb && ldd >= nb,
               "batched_gemm_tn: row strides %d, %d, %d", lda, ldb, ldd);
  WC_CHECK_ARG((long long)S * Pq >= P, "batched_gemm_tn: %d parts of %d rows do not cover %lld rows", S, Pq, P);
  GemmTnArgs g;
  g.A = A; g.B = B; g.D = D; g.P = P;
  g.lda = lda; g.ldb = ldb; g.na = na; g.nb = nb; g.ldd = ldd;
  g.S = S; g.Pq = Pq;
  g.H = g.W = g.oH = g.oW = g.conv_stride = g.pad_h = g.pad_w = g.kw = 0;
  g.div_per = g.div_oW = make_fast_div(1); g.b_elems = 0; g.n_taps = 0;
  g.sums = a_sums; g.T = T_;
  const bool big = na > 64 && nb > 64;
  return dispatch_dtype(dtype, [&](auto t) {
    using TT = decltype(t);
    return big ? launch_tn<TT, 2>(g, T_, split, stream, summed) : launch_tn<TT, 1>(g, T_, split, stream, summed);
  });
}

// dW[(ky, kx)][s] (K x C, fp32) = sum over the output pixels p = (b, oy, ox) of part s of dy[p][0..K) (x)
// x[b][stride oy + ky - pad_h][stride ox + kx - pad_w][0..C): the weight gradient taken directly, one batch per tap,
// x gathered row by row (zeros outside the image).  dy (N oH oW, K) and x (N, H, W, C) as they lie in memory.
int gemm_tn_conv(const void* dy, const void* x, float* D, int N, int H, int W, int C, int K, int kh, int kw, int stride,
                 int pad_h, int pad_w, int oH, int oW, int S, int Pq, int dtype, void* stream, float* dy_sums, bool* summed) {
  WC_CHECK_ARG(dy && x && D, "gemm_tn_conv: null pointer");
  WC_CHECK_ARG(C % 8 == 0 && K % 8 == 0 && S > 0 && Pq > 0, "gemm_tn_conv: C %d, K %d (multiples of 8)", C, K);
  const long long P = (long long)N * oH * oW;
  WC_CHECK_ARG(P > 0 && P < (1ll << 31) && (long long)S * Pq >= P, "gemm_tn_conv: %d parts of %d rows and %lld rows", S, Pq, P);
  GemmTnArgs g;
  g.A = dy; g.B = x; g.D = D; g.P = P;
  g.lda = K; g.ldb = C; g.na = K; g.nb = C; g.ldd = C;
  g.S = S; g.Pq = Pq;
  g.H = H; g.W = W; g.oH = oH; g.oW = oW; g.conv_stride = stride; g.pad_h = pad_h; g.pad_w = pad_w; g.kw = kw;
  g.div_per = make_fast_div(oH * oW); g.div_oW = make_fast_div(oW);
  g.b_elems = (long long)N * H * W * C; 
  const long long bytes = (g.b_elems + P * K) * (dtype == WC_F32 ? 4 : 2);
  g.n_taps = bytes > (16 << 20) ? kh * kw : 0;
  g.sums = dy_sums; g.T = kh * kw;
  const bool big = K > 64 && C > 64;
  return dispatch_dtype(dtype, [&](auto t) {
    using TT = decltype(t);
    return big ? launch_tn<TT, 2, true>(g, kh * kw, false, stream, summed) : launch_tn<TT, 1, true>(g, kh * kw, false, stream, summed);
  });
}

}  // namespace wc
