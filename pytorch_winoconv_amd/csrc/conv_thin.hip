// One-kernel F(2x2, 3x3) convolution for thin layers: fp16 / bf16 with at most 128 input channels, fp32 with at
// most 64, and any storage type with at most 4 (tiny_conv3x3_kernel, further down).
//
// Same arithmetic as the three-kernel path (input transform of src/split_kernel.cu:60-120, the
// batched product of src/base_conv_launchers.cu:353-367, output transform of
// src/split_kernel.cu:126-203), without V and M in HBM.  With few channels the product has so
// little arithmetic per byte that the transform-domain buffers (4x the input and 4x the output
// for this tile) are all the cost; here x is read once and y written once.
//
// What makes it fit: U of one wavefront's 16 output channels (16 elements x 16 x Cp) stays in
// registers for the life of the workgroup, so LDS only carries the transformed input of the
// 16 tiles in flight.  A workgroup (4 wavefronts, 16 output channels each) walks over blocks of
// 16 tiles: every thread loads the 4 x 4 window of one tile for a few channels, transforms it
// (fp16: packed fp16 adds; bf16: fp32) and stores the 16 elements to LDS in the storage type; after
// one barrier every wavefront multiplies all 16 elements by its part of U on v_mfma_f32_16x16x32
// (U as the row operand, so a lane ends up with 4 consecutive output channels of one tile).  The
// width half of the output transform happens in the MFMA accumulators (A^T has only 0 and +-1:
// a product is added into the accumulators it belongs to), the height half in fp32 registers.  The
// window of the next block is requested before the products of this one, and LDS is
// double-buffered, so there is one barrier per block.  With 128 channels U would take the whole
// register file: thin_rows_kernel gives a wavefront one row of the elements.
// Launches with few blocks of tiles use workgroups of half the size (32 output channels), and U reaches the
// registers through LDS: see thin_conv3x3_kernel.
#include "wc_transform.h"
#include <algorithm>

namespace wc {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

namespace {

template <typename T> struct Mfma16;
template <> struct Mfma16<half_t> {
  using Frag = half8;
  __device__ static __forceinline__ floatx4 run(Frag a, Frag b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma16<bf16_t> {
  using Frag = bf16x8;
  __device__ static __forceinline__ floatx4 run(Frag a, Frag b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
// fp32: a lane's 16-byte fragment holds four consecutive channels and feeds four v_mfma_f32_16x16x4_f32, each
// of which pairs channel e of the four lane groups' fragments (both operands are cut the same way, so every
// channel of a 16-channel step meets its partner exactly once).
template <> struct Mfma16<float> {
  using Frag = floatx4;
  __device__ static __forceinline__ floatx4 run(Frag a, Frag b, floatx4 c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
    return c;
  }
};

// The accumulator scheme below is written for these matrices.
static_assert(Mats<KIND_23>::at(0, 0) == 1 && Mats<KIND_23>::at(0, 1) == 1 && Mats<KIND_23>::at(0, 2) == 1 &&
              Mats<KIND_23>::at(0, 3) == 0 && Mats<KIND_23>::at(1, 0) == 0 && Mats<KIND_23>::at(1, 1) == 1 &&
              Mats<KIND_23>::at(1, 2) == -1 && Mats<KIND_23>::at(1, 3) == -1, "A^T of F(2,3)");

constexpr int kThinTiles = 16;      // tiles per block
constexpr int kThinK = 64;          // output channels per workgroup

// Rows of U and V that fill a line of LDS (thin_rows_kernel), and the threads and the LDS of a workgroup: of those, a wavefront per row of
// elements and 32 output channels, and V of two blocks of tiles with what the rows hand over behind it
template <typename T, int CP> constexpr bool kThinRows = CP * sizeof(T) == 256;
template <typename T, int CP, int KSUB> constexpr int kThinThreads = (kThinRows<T, CP> ? 128 : 64) * KSUB;
template <typename T, int CP, int KSUB>
constexpr int kThinLds = 2 * 16 * kThinTiles * CP * (int)sizeof(T) + (kThinRows<T, CP> ? KSUB * 8 * 1024 : 0);

struct ThinArgs {
  const void* x;
  const void* U;
  const void* bias;
  void* y;
  int H, W, C, K, Cp;
  int oH, oW, nH, nW;
  int pad1, pad2;
  int P;          // tiles of the whole batch
  int n_blocks;   // ceil(P / 16)
  int per_xcd;    // gridDim.x / 8
  int x_bytes;    // size of x, below 1 GiB
  int y_bytes;    // size of y, below 2 GiB
  int row_bytes;  // W * C * sizeof(T)
  int k_whole;    // K is a multiple of 4: a lane's 4 output channels go out in one store
  FastDiv div_nW, div_nH;
};

// Store of one lane's share of an output tile: tile p, output channels ko .. ko + 4, both output rows and the OBN output columns
// from ob0 on in out[oa][ob], bias bv added.  Stores go through a buffer descriptor and are issued unconditionally: a
// position outside (oH, oW), a tile beyond the last or a lane without work (`live` false) gets an offset beyond
// the buffer and is dropped by the hardware.  No branch around the stores matters for speed: loads and stores
// share one in-order counter, and only with straight-line code can the wait for the next block's window leave
// this block's stores in flight.
template <typename T, bool KW, int OBN>
__device__ __forceinline__ void store_tile(const ThinArgs& a, __amdgpu_buffer_rsrc_t ydesc, int p, int ko, bool live,
                                           const float (&bv)[4], const floatx4 (&out)[2][OBN], int ob0 = 0) {
  const int q = fast_div(p, a.div_nW);
  const int tw = p - q * a.nW;
  const int b = fast_div(q, a.div_nH);
  const int th = q - b * a.nH;
  const unsigned o00 = (((unsigned)b * a.oH + 2 * th) * a.oW + 2 * tw + ob0) * a.K + ko;   // in elements
  const bool h1 = 2 * th + 1 < a.oH;
#pragma unroll
  for (int oa = 0; oa < 2; ++oa) {
#pragma unroll
    for (int ob = 0; ob < OBN; ++ob) {
      const floatx4 s4 = out[oa][ob];
      const bool inside = live && (oa == 0 || h1) && 2 * tw + ob0 + ob < a.oW;
      const unsigned off = o00 + (oa * a.oW + ob) * a.K;
      Pack<T, 4> o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o.v[r] = static_cast<T>(s4[r] + bv[r]);
      if constexpr (KW) {
        const unsigned byte_off = inside ? off * (unsigned)sizeof(T) : kOutside;
        if constexpr (sizeof(T) == 4) {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, o), ydesc, byte_off, 0, 0);
        } else {
          typedef unsigned u2 __attribute__((ext_vector_type(2)));
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, o), ydesc, byte_off, 0, 0);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const unsigned byte_off = inside && ko + r < a.K ? (off + r) * (unsigned)sizeof(T) : kOutside;
          if constexpr (sizeof(T) == 4)
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, o.v[r]), ydesc, byte_off, 0, 0);
          else
            __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, o.v[r]), ydesc, byte_off, 0, 0);
        }
      }
    }
  }
}

// The bias of a lane's four output channels, loaded once per kernel.
template <typename T>
__device__ __forceinline__ void load_bias(const ThinArgs& a, int ko, float (&bv)[4]) {
  const T* bias = static_cast<const T*>(a.bias);
#pragma unroll
  for (int r = 0; r < 4; ++r) bv[r] = bias && ko + r < a.K ? static_cast<float>(bias[ko + r]) : 0.f;
}

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
struct TwoFloats {                  // (a vector of two costs moves of register pairs)
  float lo, hi;
  __device__ __forceinline__ TwoFloats operator+(TwoFloats o) const { return {lo + o.lo, hi + o.hi}; }
  __device__ __forceinline__ TwoFloats operator-(TwoFloats o) const { return {lo - o.lo, hi - o.hi}; }
};

// B^T of F(2,3) on four elements, STRIDE apart
template <int STRIDE, typename V>
__device__ __forceinline__ void bt23(V* d) {
  const V d0 = d[0], d1 = d[STRIDE], d2 = d[2 * STRIDE], d3 = d[3 * STRIDE];
  d[0] = d0 - d2;
  d[STRIDE] = d1 + d2;
  d[2 * STRIDE] = d2 - d1;
  d[3 * STRIDE] = d1 - d3;
}
// the whole block: along its lines, then its columns
template <typename V>
__device__ __forceinline__ void transform(V (&d)[16]) {
#pragma unroll
  for (int l = 0; l < 4; ++l) bt23<1>(d + 4 * l);
#pragma unroll
  for (int l = 0; l < 4; ++l) bt23<4>(d + l);
}
static_assert(Mats<KIND_23>::bt(0, 0) == 1 && Mats<KIND_23>::bt(0, 2) == -1 && Mats<KIND_23>::bt(1, 1) == 1 &&
              Mats<KIND_23>::bt(1, 2) == 1 && Mats<KIND_23>::bt(2, 1) == -1 && Mats<KIND_23>::bt(2, 2) == 1 &&
              Mats<KIND_23>::bt(3, 1) == 1 && Mats<KIND_23>::bt(3, 3) == -1, "B^T of F(2,3)");

// KW: K is a multiple of 4, a lane's 4 output channels go out in one store (a compile-time choice: a branch
// around the stores, even a uniform one, makes the compiler wait for all memory operations at the loop top).
// KSUB: groups of 16 output channels per workgroup, 4 or 2.  With 2 a workgroup has half the wavefronts, half of
// U to fetch and half the products, and the launch has twice the workgroups: for layers whose blocks of tiles
// would leave more than half of the CUs idle (a workgroup with one block spends most of its time fetching U and,
// in fp32, multiplying).
template <typename T, int CP, bool KW, int KSUB>
__global__ __launch_bounds__(64 * KSUB) __attribute__((amdgpu_waves_per_eu(KSUB / 2, KSUB / 2))) void thin_conv3x3_kernel(ThinArgs a) {
  static_assert(CP * sizeof(T) <= 128, "a wavefront holds U of all 16 elements");
  constexpr bool PLAIN = sizeof(T) == 4;             // one accumulator per element, width transform in VALU (measured: no gain for 16-bit types)
  constexpr int EPF = 16 / sizeof(T);                // channels per 16-byte fragment
  constexpr int NT = 64 * KSUB;
  constexpr int NROW = 4;                 // element rows
  constexpr int VEC = kThinTiles * CP / NT;   // channels per thread in the transform
  constexpr int CVECS = CP / VEC;
  constexpr int KS = CP / (4 * EPF);      // fragment steps along the channels (four lane groups x EPF channels each)
  // Bytes per (element, tile) row in LDS: no padding; the 16-byte chunks of a row are permuted by the row instead.
  // A fragment read takes one chunk from each of 16 consecutive rows; the LDS of this part delivers 16-byte reads
  // at 256 bytes per clock only if those 16 chunks fall into 16 different 16-byte columns of a 256-byte line
  // (rows padded by 16 bytes, which are conflict-free for 128-byte wide LDS, measured half that rate).  With R rows
  // per 256 bytes, chunk c of row r sits at position c ^ ((r / R) mod chunks per row).
  constexpr int PITCH = CP * sizeof(T);
  constexpr int CPRW = PITCH / 16;             // chunks per row: 4 or 8
  constexpr int RPL = 16 / CPRW;               // rows per 256-byte line
  static_assert(CPRW == 4 || CPRW == 8, "rows of 64 or 128 bytes");
  static_assert(VEC * sizeof(T) <= 16, "a thread's channels stay inside one chunk");
  constexpr int BUF = 16 * kThinTiles * PITCH;
  using MF = Mfma16<T>;
  using Frag = typename MF::Frag;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kbase = (blockIdx.y * KSUB + wave) * 16;

  // transform role: tile pl of the block, channels c .. c + VEC.  x is read through a buffer descriptor:
  // one 32-bit offset per load, and a window element outside the image is an offset beyond the
  // buffer, which reads as zero.
  const int pl = tid / CVECS;
  const int c = (tid % CVECS) * VEC;
  const bool c_ok = c < a.C;
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.x), 0, a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ydesc = __builtin_amdgcn_make_buffer_rsrc(a.y, 0, a.y_bytes, 0x00020000);
  Pack<T, VEC> raw[16];

  // Offset of a window element = row part + column part.  A row outside the image contributes
  // 2^31 and a column outside 2^30: with x below 1 GiB every sum that contains one of them lies
  // beyond the buffer, so no per-element select is needed.
  auto load_window = [&](int blk) {
    const int p = blk * kThinTiles + pl;
    const bool valid = p < a.P && c_ok;
    const int q = fast_div(p, a.div_nW);
    const int tw = p - q * a.nW;
    const int b = fast_div(q, a.div_nH);
    const int th = q - b * a.nH;
    const int y0 = 2 * th - a.pad1, x0 = 2 * tw - a.pad2;
    const unsigned row0 = (unsigned)(b * a.H + y0) * (unsigned)a.row_bytes;
    const unsigned col0 = (unsigned)(x0 * a.C + c) * (unsigned)sizeof(T);
    unsigned rowoff[4], coloff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      rowoff[i] = valid && (unsigned)(y0 + i) < (unsigned)a.H ? row0 + i * a.row_bytes : 0x80000000u;
      coloff[i] = (unsigned)(x0 + i) < (unsigned)a.W ? col0 + i * a.C * (unsigned)sizeof(T) : 0x40000000u;
    }
#pragma unroll
    for (int i1 = 0; i1 < 4; ++i1)
#pragma unroll
      for (int i2 = 0; i2 < 4; ++i2) raw[i1 * 4 + i2] = buffer_load_pack<T, VEC>(rsrc, rowoff[i1] + coloff[i2]);
  };

  const int nwg = gridDim.x;
  int blk = xcd_remap(blockIdx.x, a.per_xcd);
  if (blk < a.n_blocks) load_window(blk);   // in flight while U arrives

  // this wavefront's part of U: row operand, lane = output channel kbase + lane % 16, 8 channels
  // from 8 * (lane / 16).  Rows beyond K repeat row K - 1: a row of U only reaches the same row of the
  // product, and those rows are never stored.
  // Memory is read in whole rows (consecutive lanes take consecutive 16 bytes) and the fragments go to the lanes
  // that need them through this wavefront's own slice of LDS, which nothing else uses yet: a load whose
  // neighbouring lanes address different rows, as the operand layout would have it, measured 3.8 times slower per
  // byte with every line in L2, and for a workgroup with one block of tiles that load is most of the kernel.
  Frag u[NROW * 4][KS];
  {
    constexpr int NW = NT / 64;
    constexpr int SLICE = 2 * BUF / NW;                // bytes of LDS per wavefront
    constexpr int EPR = SLICE / (16 * PITCH);          // elements per round: 16 rows of U each
    constexpr int NEL = NROW * 4;
    static_assert(EPR >= 1 && NEL % EPR == 0 && KS == PITCH / 64, "staging of U");
    unsigned char* slice = lds + wave * SLICE;
    const unsigned char* Ub = static_cast<const unsigned char*>(a.U);
    uint4v tmp[NEL][KS];
    int srow[KS], scol[KS];
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const int off = (i * 64 + lane) * 16;            // byte of the 16-row block
      srow[i] = off / PITCH;
      scol[i] = off % PITCH;
    }
    static_for<0, NEL>([&](auto t_) {
      constexpr int t = decltype(t_)::value;
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        const long long row = (long long)t * a.K + min(kbase + srow[i], a.K - 1);
        tmp[t][i] = *reinterpret_cast<const uint4v*>(Ub + row * PITCH + scol[i]);
      }
    });
    const int fswz = ((lane & 15) / RPL) & (CPRW - 1);
    static_for<0, NEL / EPR>([&](auto r_) {
      constexpr int rd = decltype(r_)::value;
      static_for<0, EPR>([&](auto e_) {
        constexpr int e = decltype(e_)::value;
#pragma unroll
        for (int i = 0; i < KS; ++i)
          *reinterpret_cast<uint4v*>(slice + (e * 16 + srow[i]) * PITCH +
                                     (((scol[i] >> 4) ^ ((srow[i] / RPL) & (CPRW - 1))) << 4)) = tmp[rd * EPR + e][i];
      });
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      static_for<0, EPR>([&](auto e_) {
        constexpr int e = decltype(e_)::value;
        static_for<0, KS>([&](auto s_) {
          constexpr int s2 = decltype(s_)::value;
          u[rd * EPR + e][s2] = *reinterpret_cast<const Frag*>(slice + (e * 16 + (lane & 15)) * PITCH +
                                                              ((((lane >> 4) + 4 * s2) ^ fswz) << 4));
        });
      });
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    });
  }

  // U and the bias have arrived before the loop starts: a wait for them inside the loop would also wait, on
  // every pass, for the window loads of the next block, which are younger (loads return in order).
  float bv[4];
  load_bias<T>(a, kbase + 4 * (lane >> 4), bv);
#pragma unroll
  for (int t = 0; t < NROW * 4; ++t)
#pragma unroll
    for (int s2 = 0; s2 < KS; ++s2) asm volatile("" : "+v"(u[t][s2]));
#pragma unroll
  for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(bv[r]));
  __syncthreads();   // the first block's V goes where other wavefronts staged their U

  for (int it = 0; blk < a.n_blocks; blk += nwg, ++it) {
    unsigned char* buf = lds + (it & 1) * BUF;
    // Input transform, two channels at a time.  fp16 adds pairs of channels
    // in fp16 like the reference's kernels (calculation_kernels.cu:786-806 computes in T); bf16,
    // which has no packed add, goes through fp32.
    // all channels of this thread lie in one chunk
    const int cb = c * (int)sizeof(T);
    T* vdst = reinterpret_cast<T*>(buf + pl * PITCH + ((((cb >> 4) ^ ((pl / RPL) & (CPRW - 1))) << 4) | (cb & 15)));
    static_for<0, VEC / 2>([&](auto h_) {
      constexpr int h = decltype(h_)::value;
      if constexpr (std::is_same<T, half_t>::value) {
        half2v d[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) d[e] = half2v{raw[e].v[2 * h], raw[e].v[2 * h + 1]};
        transform(d);
#pragma unroll
        for (int e = 0; e < 16; ++e)
          *reinterpret_cast<half2v*>(vdst + e * (kThinTiles * PITCH / (int)sizeof(T)) + 2 * h) = d[e];
      } else {
        typedef float float2v __attribute__((ext_vector_type(2)));
        float2v d[16];
#pragma unroll
        for (int e = 0; e < 16; ++e)
          d[e] = float2v{static_cast<float>(raw[e].v[2 * h]), static_cast<float>(raw[e].v[2 * h + 1])};
        transform(d);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float o[2] = {d[e][0], d[e][1]};
          store_pack<T, 2>(vdst + e * (kThinTiles * PITCH / (int)sizeof(T)) + 2 * h, o);
        }
      }
    });
    __syncthreads();
    if (blk + nwg < a.n_blocks) load_window(blk + nwg);

    // The products M[i][j] = U[i][j] V[i][j] over the channels, and the width half of the output transform,
    // zw[i][0] = M[i][0] + M[i][1] + M[i][2], zw[i][1] = M[i][1] - M[i][2] - M[i][3].  16-bit types do the sums in
    // the accumulators (z0 takes j = 0, 1, 2; zp takes j = 1 and zn j = 2, 3, so that no operand needs its sign
    // changed): 24 MFMAs per channel step instead of 16, 12 accumulators instead of 16, no VALU work - their
    // MFMAs are cheap and registers are what is short.  fp32, whose MFMAs are sixteen times slower and bound the
    // kernel, keeps one accumulator per element and adds in VALU.  Consecutive MFMAs write different accumulators.
    floatx4 zw[NROW][2];
    const unsigned char* vrow = buf + (lane & 15) * PITCH;
    const int vswz = ((lane & 15) / RPL) & (CPRW - 1);
    if constexpr (PLAIN) {
      floatx4 mm[NROW][4];
#pragma unroll
      for (int i = 0; i < NROW; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) mm[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
      static_for<0, KS>([&](auto s_) {
        constexpr int s = decltype(s_)::value;
        static_for<0, 4>([&](auto j_) {
          constexpr int j = decltype(j_)::value;
          Frag v[NROW];
          static_for<0, NROW>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            v[i] = *reinterpret_cast<const Frag*>(vrow + (i * 4 + j) * kThinTiles * PITCH + ((((lane >> 4) + 4 * s) ^ vswz) << 4));
          });
          static_for<0, NROW>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            mm[i][j] = MF::run(u[i * 4 + j][s], v[i], mm[i][j]);
          });
        });
      });
#pragma unroll
      for (int i = 0; i < NROW; ++i) {
        zw[i][0] = mm[i][0] + mm[i][1] + mm[i][2];
        zw[i][1] = mm[i][1] - mm[i][2] - mm[i][3];
      }
    } else {
      floatx4 z0[NROW], zp[NROW], zn[NROW];
#pragma unroll
      for (int i = 0; i < NROW; ++i) z0[i] = zp[i] = zn[i] = floatx4{0.f, 0.f, 0.f, 0.f};
      static_for<0, KS>([&](auto s_) {
        constexpr int s = decltype(s_)::value;
        static_for<0, 4>([&](auto j_) {
          constexpr int j = decltype(j_)::value;
          Frag v[NROW];
          static_for<0, NROW>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            v[i] = *reinterpret_cast<const Frag*>(vrow + (i * 4 + j) * kThinTiles * PITCH + ((((lane >> 4) + 4 * s) ^ vswz) << 4));
          });
          static_for<0, NROW>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            if constexpr (j <= 2) z0[i] = MF::run(u[i * 4 + j][s], v[i], z0[i]);
          });
          static_for<0, NROW>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            if constexpr (j == 1) zp[i] = MF::run(u[i * 4 + j][s], v[i], zp[i]);
            if constexpr (j >= 2) zn[i] = MF::run(u[i * 4 + j][s], v[i], zn[i]);
          });
        });
      });
#pragma unroll
      for (int i = 0; i < NROW; ++i) {
        zw[i][0] = z0[i];
        zw[i][1] = zp[i] - zn[i];
      }
    }

    // Height half of the output transform: out[0][b] = zw[0][b] + zw[1][b] + zw[2][b], out[1][b] = zw[1][b] -
    // zw[2][b] - zw[3][b].
    floatx4 out[2][2];
#pragma unroll
    for (int ob = 0; ob < 2; ++ob) {
      out[0][ob] = zw[0][ob] + zw[1][ob] + zw[2][ob];
      out[1][ob] = zw[1][ob] - zw[2][ob] - zw[3][ob];
    }

    // lane = tile lane % 16, output channels ko .. ko + 4
    const int p = blk * kThinTiles + (lane & 15);
    const int ko = kbase + 4 * (lane >> 4);
    store_tile<T, KW, 2>(a, ydesc, p, ko, p < a.P && ko < a.K, bv, out);
  }
}

// The same for rows of U and V of 256 bytes: 128 channels of a 16-bit type, 64 of fp32.  U of 16 output channels and all
// elements would be twice the register file, so a wavefront has one row of elements and 32 output channels (KB groups of 16), and the
// rows meet in LDS.  One workgroup is all a CU's LDS holds, so nothing else runs while its wavefronts wait for each other: the
// transform of the next block, the loads of the one after and the output of the one before are dealt out over a block's
// products, and a block has one barrier that waits for LDS and one that waits for nothing.
//
// Two rows of elements and 16 output channels a wavefront, each phase of a block behind the last one, took 73 us (2.6 a block) where this
// takes 57 (fp16 N=64 128 -> 128, 56x56; 28x28 25.5 | 21.4; bf16 77 | 63; fp32 N=64 64 -> 64, 56x56 79 | 69.5).  The dealing out
// alone is 70: fragments of V fed one product and a half, LDS 256 KB of reads a block.  What is left of 1.8 us a block: taken out one at a
// time, the loads are 0.4 of it (64 KB through L1, the same from a footprint of 4 KB), products 0.4, the hand-over and the output 0.3.
// Of a thin_conv3x3_kernel with 128-byte rows two run on a CU, side by side, and the same order of its work was slower (64 channels 23.0 | 23.8).
template <typename T, int CP, bool KW, int KSUB>
__global__ __launch_bounds__((kThinThreads<T, CP, KSUB>)) __attribute__((amdgpu_waves_per_eu(KSUB / 2, KSUB / 2))) void thin_rows_kernel(ThinArgs a) {
  constexpr bool PLAIN = sizeof(T) == 4;             // one accumulator per element, width transform in VALU (measured: no gain for 16-bit types)
  constexpr int EPF = 16 / sizeof(T);                // channels per 16-byte fragment
  constexpr int NT = kThinThreads<T, CP, KSUB>, NW = NT / 64;
  constexpr int KB = KSUB * 4 / NW;                  // groups of 16 output channels per wavefront, of one row of elements
  constexpr int VEC = kThinTiles * CP / NT;   // channels per thread in the transform
  constexpr int CVECS = CP / VEC;
  constexpr int KS = CP / (4 * EPF);      // fragment steps along the channels (four lane groups x EPF channels each)
  // rows of an (element, tile) in LDS as in thin_conv3x3_kernel: chunk c of row r at position c ^ r
  static_assert(CP * sizeof(T) == 256, "a row is a line of LDS");
  constexpr int PITCH = CP * sizeof(T);
  static_assert(VEC * sizeof(T) >= 4 && VEC * sizeof(T) <= 16, "a thread's channels stay inside one chunk");
  constexpr int ELEM = kThinTiles * PITCH, BUF = 16 * ELEM;
  using MF = Mfma16<T>;
  using Frag = typename MF::Frag;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = wave & 3;                              // this wavefront's row of elements
  const int kbase = (blockIdx.y * KSUB + (wave >> 2) * KB) * 16;

  // transform role: tile pl of the block, channels c .. c + VEC.  x is read through a buffer descriptor:
  // one 32-bit offset per load, and a window element outside the image is an offset beyond the
  // buffer, which reads as zero.
  const int pl = tid / CVECS;
  const int c = (tid % CVECS) * VEC;
  const bool c_ok = c < a.C;
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.x), 0, a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ydesc = __builtin_amdgcn_make_buffer_rsrc(a.y, 0, a.y_bytes, 0x00020000);
  using Words = Pack<uint32_t, VEC * (int)sizeof(T) / 4>;
  Words raw[16];

  // Offset of a window element = row part + column part.  A row outside the image contributes
  // 2^31 and a column outside 2^30: with x below 1 GiB every sum that contains one of them lies
  // beyond the buffer, so no per-element select is needed.
  unsigned rowoff[4], coloff[4];
  auto find_window = [&](int blk) {
    const int p = blk * kThinTiles + pl;
    const bool valid = (p < a.P) & c_ok;
    const int q = fast_div(p, a.div_nW);
    const int tw = p - q * a.nW;
    const int b = fast_div(q, a.div_nH);
    const int th = q - b * a.nH;
    const int y0 = 2 * th - a.pad1, x0 = 2 * tw - a.pad2;
    const unsigned row0 = (unsigned)(b * a.H + y0) * (unsigned)a.row_bytes;
    const unsigned col0 = (unsigned)(x0 * a.C + c) * (unsigned)sizeof(T);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      rowoff[i] = valid & ((unsigned)(y0 + i) < (unsigned)a.H) ? row0 + i * a.row_bytes : 0x80000000u;
      coloff[i] = (unsigned)(x0 + i) < (unsigned)a.W ? col0 + i * a.C * (unsigned)sizeof(T) : 0x40000000u;
    }
  };
  auto load_element = [&](int e) { raw[e] = __builtin_bit_cast(Words, buffer_load_pack<T, VEC>(rsrc, rowoff[e >> 2] + coloff[e & 3])); };
  auto load_window = [&](int blk) {
    find_window(blk);
#pragma unroll
    for (int e = 0; e < 16; ++e) load_element(e);
  };

  const int nwg = gridDim.x;
  int blk = xcd_remap(blockIdx.x, a.per_xcd);
  if (blk < a.n_blocks) load_window(blk);   // in flight while U arrives

  // this wavefront's part of U: row operand, lane = output channel kbase + lane % 16, 8 channels
  // from 8 * (lane / 16).  Rows beyond K repeat row K - 1: a row of U only reaches the same row of the
  // product, and those rows are never stored.
  // Memory is read in whole rows (consecutive lanes take consecutive 16 bytes) and the fragments go to the lanes
  // that need them through this wavefront's own slice of LDS, which nothing else uses yet: a load whose
  // neighbouring lanes address different rows, as the operand layout would have it, measured 3.8 times slower per
  // byte with every line in L2, and for a workgroup with one block of tiles that load is most of the kernel.
  constexpr int NEL = 4 * KB;                          // blocks of 16 rows of U: element t / KB of the row, channels 16 (t % KB)
  Frag u[NEL][KS];
  {
    constexpr int SLICE = 2 * BUF / NW;                // bytes of LDS per wavefront
    constexpr int EPR = SLICE / (16 * PITCH) < NEL ? SLICE / (16 * PITCH) : NEL;          // blocks per round: 16 rows of U each
    static_assert(EPR >= 1 && NEL % EPR == 0 && KS == PITCH / 64, "staging of U");
    unsigned char* slice = lds + wave * SLICE;
    const unsigned char* Ub = static_cast<const unsigned char*>(a.U);
    uint4v tmp[NEL][KS];
    int srow[KS], scol[KS];
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const int off = (i * 64 + lane) * 16;            // byte of the 16-row block
      srow[i] = off / PITCH;
      scol[i] = off % PITCH;
    }
    static_for<0, NEL>([&](auto t_) {
      constexpr int t = decltype(t_)::value;
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        const long long r = (long long)(row * 4 + t / KB) * a.K + min(kbase + t % KB * 16 + srow[i], a.K - 1);
        tmp[t][i] = *reinterpret_cast<const uint4v*>(Ub + r * PITCH + scol[i]);
      }
    });
    const int fswz = lane & 15;
    static_for<0, NEL / EPR>([&](auto r_) {
      constexpr int rd = decltype(r_)::value;
      static_for<0, EPR>([&](auto e_) {
        constexpr int e = decltype(e_)::value;
#pragma unroll
        for (int i = 0; i < KS; ++i)
          *reinterpret_cast<uint4v*>(slice + (e * 16 + srow[i]) * PITCH +
                                     (((scol[i] >> 4) ^ (srow[i] & 15)) << 4)) = tmp[rd * EPR + e][i];
      });
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      static_for<0, EPR>([&](auto e_) {
        constexpr int e = decltype(e_)::value;
        static_for<0, KS>([&](auto s_) {
          constexpr int s2 = decltype(s_)::value;
          u[rd * EPR + e][s2] = *reinterpret_cast<const Frag*>(slice + (e * 16 + (lane & 15)) * PITCH +
                                                              ((((lane >> 4) + 4 * s2) ^ fswz) << 4));
        });
      });
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    });
  }

  // What this lane finishes: four output channels (`quad` of the workgroup's) of a tile, in one output column.  Neighbouring
  // lanes have neighbouring channels, so that stores are 128 bytes (64 of 32 output channels) at a time.
  constexpr int QUADS = 4 * KSUB;
  static_assert(2 * kThinTiles * QUADS == NT, "a column of a quad for every thread");
  const int quad = lane % QUADS, ob = wave & 1, my_tile = (wave >> 1) * (64 / QUADS) + lane / QUADS;
  const int ko = blockIdx.y * KSUB * 16 + quad * 4;

  // U and the bias have arrived before the loop starts: a wait for them inside the loop would also wait, on
  // every pass, for the window loads of the next block, which are younger (loads return in order).
  float bv[4];
  load_bias<T>(a, ko, bv);
#pragma unroll
  for (int t = 0; t < NEL; ++t)
#pragma unroll
    for (int s2 = 0; s2 < KS; ++s2) asm volatile("" : "+v"(u[t][s2]));
#pragma unroll
  for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(bv[r]));
  __syncthreads();   // the first block's V goes where other wavefronts staged their U

  // Input transform in units: B^T on a line of two channels' windows, or on a column, whose results go back to where the window was.
  // fp16 adds pairs of channels in fp16 like the reference's kernels (calculation_kernels.cu:786-806 computes in T); bf16,
  // which has no packed add, goes through fp32.
  using Two = std::conditional_t<std::is_same<T, half_t>::value, half2v, TwoFloats>;
  constexpr int UNITS = 4 * VEC;               // per pair of channels four lines, then four columns
  Two d[16];
  auto transform_unit = [&](auto u_) {
    constexpr int u = decltype(u_)::value, h = u / 8, l = u % 4;
    if constexpr (u % 8 < 4) {
#pragma unroll
      for (int e = 4 * l; e < 4 * l + 4; ++e) {
        if constexpr (std::is_same<T, half_t>::value) d[e] = __builtin_bit_cast(half2v, raw[e].v[h]);
        else if constexpr (sizeof(T) == 2) d[e] = TwoFloats{__builtin_bit_cast(float, raw[e].v[h] << 16), __builtin_bit_cast(float, raw[e].v[h] & 0xffff0000u)};
        else d[e] = TwoFloats{__builtin_bit_cast(float, raw[e].v[2 * h]), __builtin_bit_cast(float, raw[e].v[2 * h + 1])};
      }
      bt23<1>(d + 4 * l);
    } else {
      bt23<4>(d + l);
#pragma unroll
      for (int e = l; e < 16; e += 4) {
        if constexpr (std::is_same<T, half_t>::value) {
          raw[e].v[h] = __builtin_bit_cast(uint32_t, d[e]);
        } else if constexpr (sizeof(T) == 2) {
          const Pack<T, 2> two = {{static_cast<T>(d[e].lo), static_cast<T>(d[e].hi)}};
          raw[e].v[h] = __builtin_bit_cast(uint32_t, two);
        } else {
          raw[e].v[2 * h] = __builtin_bit_cast(uint32_t, d[e].lo);
          raw[e].v[2 * h + 1] = __builtin_bit_cast(uint32_t, d[e].hi);
        }
      }
    }
  };
  // all channels of this thread lie in one chunk
  const int cb = c * (int)sizeof(T);
  unsigned char* const vdst = lds + pl * PITCH + ((((cb >> 4) ^ pl) << 4) | (cb & 15));
  auto store_element = [&](int e, int buf) {
    typedef uint32_t vec __attribute__((ext_vector_type(VEC * sizeof(T) / 4)));
    *reinterpret_cast<vec*>(vdst + buf + e * ELEM) = __builtin_bit_cast(vec, raw[e]);
  };
  auto meet = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
  };

  // The height half of the output transform takes the four rows of elements, which are four wavefronts': each leaves its
  // zw[0 .. 1] of KB groups of 16 channels in LDS behind V, 1 KB each, and a block later all finish what these add up to.
  // A lane leaves the channels 4 (lane / 16) .. + 4 of tile lane % 16; the tiles of a quad are exchanged by the quad's number, which
  // lets the lanes of a tile read from different banks.
  constexpr int LEFT = 2 * KB * 1024;           // bytes of a wavefront
  unsigned char* const leave = lds + 2 * BUF + wave * LEFT + (lane >> 4) * 256;
  const unsigned char* const take =
      lds + 2 * BUF + quad / 4 / KB * 4 * LEFT + quad / 4 % KB * 2048 + ob * 1024 + quad % 4 * 256 + ((my_tile ^ quad) & 15) * 16;
  auto finish = [&](bool live, int blk) {
    floatx4 z[4], out[2][1];
#pragma unroll
    for (int i = 0; i < 4; ++i) z[i] = *reinterpret_cast<const floatx4*>(take + i * LEFT);
    out[0][0] = z[0] + z[1] + z[2];
    out[1][0] = z[1] - (z[2] + z[3]);
    asm volatile("" : "+v"(out[0][0]), "+v"(out[1][0]));       // read before the barrier that comes
    const int p = max(blk, 0) * kThinTiles + my_tile;
    store_tile<T, KW, 1>(a, ydesc, p, ko, live & (p < a.P) & (ko < a.K), bv, out, ob);
  };

  // of a fragment of the first channel step; that of step s lies 4 s chunks on, which the permutation makes an exclusive or
  int vrow = (lane & 15) * PITCH + row * 4 * ELEM + (((lane >> 4) ^ (lane & 15)) << 4);

  // A block: the products M[i][j] = U[i][j] V[i][j] over the channels, and the width half of the output transform,
  // zw[i][0] = M[i][0] + M[i][1] + M[i][2], zw[i][1] = M[i][1] - M[i][2] - M[i][3].  16-bit types do the sums in
  // the accumulators (z0 takes j = 0, 1, 2; zp takes j = 1 and zn j = 2, 3, so that no operand needs its sign
  // changed): 24 MFMAs per channel step instead of 16, 12 accumulators instead of 16, no VALU work - their
  // MFMAs are cheap and registers are what is short.  fp32, whose MFMAs are sixteen times slower and bound the
  // kernel, keeps one accumulator per element and adds in VALU.  Consecutive MFMAs write different accumulators.
  //
  // The products are a stream of items, one step of channels of one element each.  The transform of the
  // next block, its way to LDS and the loads of the block after are dealt out over the items (MORE: there is a next block).
  auto block = [&](auto more_, int it) {
    constexpr bool MORE = decltype(more_)::value != 0;
    // Fragments two items ahead; the transform from the first quarter on, of bf16, whose numbers take twice the registers, in the last three
    // eighths, before which its loads are not waited for either (us, from 1/4 | 5/8: fp16 57.1 | 60.8, fp32 69.5 | 69.6, bf16 spilling 72 | 62.7)
    constexpr int NI = KS * 4, VD = 3, FROM = std::is_same<T, bf16_t>::value ? NI * 5 / 8 : NI / 4, MEET = 2;
    const int cur = (it & 1) * BUF, next = BUF - cur;
    asm volatile("" : "+v"(vrow));                // addresses are worked out again: registers are short
    floatx4 acc[PLAIN ? 4 : 3][KB];          // PLAIN: M; else z0, zp, zn
#pragma unroll
    for (int j = 0; j < (PLAIN ? 4 : 3); ++j)
#pragma unroll
      for (int k = 0; k < KB; ++k) acc[j][k] = floatx4{0.f, 0.f, 0.f, 0.f};
    Frag vf[VD];
    auto load_v = [&](int item) { vf[item % VD] = *reinterpret_cast<const Frag*>(lds + ((vrow ^ (item / 4 * 64)) + cur) + item % 4 * ELEM); };
#pragma unroll
    for (int i = 0; i < VD - 1; ++i) load_v(i);
    static_for<0, NI>([&](auto item_) {
      constexpr int item = decltype(item_)::value, s = item / 4, j = item % 4;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (item + VD - 1 < NI) load_v(item + VD - 1);
#pragma unroll
      for (int k = 0; k < KB; ++k) {
        if constexpr (PLAIN) acc[j][k] = MF::run(u[j * KB + k][s], vf[item % VD], acc[j][k]);
        else if constexpr (j <= 2) acc[0][k] = MF::run(u[j * KB + k][s], vf[item % VD], acc[0][k]);
      }
#pragma unroll
      for (int k = 0; k < KB; ++k)
        if constexpr (!PLAIN && j >= 1) acc[j == 1 ? 1 : 2][k] = MF::run(u[j * KB + k][s], vf[item % VD], acc[j == 1 ? 1 : 2][k]);
      if constexpr (item == MEET - 1) finish(it > 0, blk - nwg);
      if constexpr (item == MEET) __builtin_amdgcn_s_barrier();             // all have read what the last block left: its place may be written
      if constexpr (MORE) {
        constexpr auto first = [](int i) { return i <= FROM ? 0 : (i - FROM) * UNITS / (NI - FROM); };
        static_assert(first(MEET) <= UNITS - 4, "written behind the barrier");
        static_for<first(item), first(item + 1)>([&](auto u_) {
          constexpr int unit = decltype(u_)::value;
          if constexpr (unit == UNITS - 4) find_window(blk + 2 * nwg);
          transform_unit(u_);
          if constexpr (unit >= UNITS - 4) {
#pragma unroll
            for (int e = unit % 4; e < 16; e += 4) {
              store_element(e, next);
              load_element(e);
            }
          }
        });
      }
    });
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      floatx4 zw[2] = {acc[0][k], acc[1][k] - acc[2][k]};
      if constexpr (PLAIN) {
        zw[0] = acc[0][k] + acc[1][k] + acc[2][k];
        zw[1] -= acc[3][k];
      }
      const int quad_left = (wave >> 2) * 4 * KB + 4 * k + (lane >> 4);
#pragma unroll
      for (int b = 0; b < 2; ++b) *reinterpret_cast<floatx4*>(leave + (2 * k + b) * 1024 + ((lane ^ quad_left) & 15) * 16) = zw[b];
    }
    meet();
  };

  if (blk >= a.n_blocks) return;
  static_for<0, UNITS>([&](auto u_) { transform_unit(u_); });
#pragma unroll
  for (int e = 0; e < 16; ++e) store_element(e, 0);
  if (blk + nwg < a.n_blocks) load_window(blk + nwg);
  meet();
  int it = 0;
  for (; blk + nwg < a.n_blocks; blk += nwg, ++it) block(ic<1>{}, it);
  block(ic<0>{}, it);
  finish(true, blk);
}

// The same for at most 4 input channels (first layers: grey or RGB images), any storage type.  Padding 3
// channels to the 32 of the batched GEMM makes V ten times the input, and M is 4x the output whatever
// the channel count, so the three-kernel path spends its time on buffers; here the product runs on
// v_mfma_f32_16x16x4_f32 in fp32 with a reduction of exactly 4 channels, U (16 elements x 16 output
// channels x 4) is 16 registers per lane, and a block is 64 tiles: a thread transforms one channel of
// one tile, a wavefront multiplies four column blocks of 16 tiles.
template <typename T, bool KW>
__global__ __launch_bounds__(256) void tiny_conv3x3_kernel(ThinArgs a) {
  constexpr int TILES = 64;
  constexpr int BUF = 16 * TILES * 4;     // floats per buffer, [element][tile][channel]
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  float* ldsf = reinterpret_cast<float*>(lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kbase = blockIdx.y * kThinK + wave * 16;
  const int pl = tid >> 2, c = tid & 3;
  const bool c_ok = c < a.C;
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.x), 0, a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ydesc = __builtin_amdgcn_make_buffer_rsrc(a.y, 0, a.y_bytes, 0x00020000);
  Pack<T, 1> raw[16];

  auto load_window = [&](int blk) {      // offsets as in thin_conv3x3_kernel
    const int p = blk * TILES + pl;
    const bool valid = p < a.P && c_ok;
    const int q = fast_div(p, a.div_nW);
    const int tw = p - q * a.nW;
    const int b = fast_div(q, a.div_nH);
    const int th = q - b * a.nH;
    const int y0 = 2 * th - a.pad1, x0 = 2 * tw - a.pad2;
    const unsigned row0 = (unsigned)(b * a.H + y0) * (unsigned)a.row_bytes;
    const unsigned col0 = (unsigned)(x0 * a.C + c) * (unsigned)sizeof(T);
    unsigned rowoff[4], coloff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      rowoff[i] = valid && (unsigned)(y0 + i) < (unsigned)a.H ? row0 + i * a.row_bytes : 0x80000000u;
      coloff[i] = (unsigned)(x0 + i) < (unsigned)a.W ? col0 + i * a.C * (unsigned)sizeof(T) : 0x40000000u;
    }
#pragma unroll
    for (int i1 = 0; i1 < 4; ++i1)
#pragma unroll
      for (int i2 = 0; i2 < 4; ++i2) raw[i1 * 4 + i2] = buffer_load_pack<T, 1>(rsrc, rowoff[i1] + coloff[i2]);
  };

  const int nwg = gridDim.x;
  int blk = xcd_remap(blockIdx.x, a.per_xcd);
  if (blk < a.n_blocks) load_window(blk);

  // U as the row operand: lane = output channel kbase + lane % 16, input channel lane / 16 (U's rows are
  // Cp long, channels beyond C hold zeros)
  float u[16];
  {
    const int ko = min(kbase + (lane & 15), a.K - 1);
    const T* U = static_cast<const T*>(a.U) + (long long)ko * a.Cp + (lane >> 4);
#pragma unroll
    for (int t = 0; t < 16; ++t) u[t] = static_cast<float>(U[(long long)t * a.K * a.Cp]);
  }

  float bv[4];
  load_bias<T>(a, kbase + 4 * (lane >> 4), bv);
#pragma unroll
  for (int t = 0; t < 16; ++t) asm volatile("" : "+v"(u[t]));
#pragma unroll
  for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(bv[r]));

  for (int it = 0; blk < a.n_blocks; blk += nwg, ++it) {
    float* buf = ldsf + (it & 1) * BUF;
    {
      float d[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) d[e] = static_cast<float>(raw[e].v[0]);
      transform(d);
#pragma unroll
      for (int e = 0; e < 16; ++e) buf[(e * TILES + pl) * 4 + c] = d[e];
    }
    __syncthreads();
    if (blk + nwg < a.n_blocks) load_window(blk + nwg);

#pragma unroll 1
    for (int cb = 0; cb < TILES / 16; ++cb) {
      floatx4 z0[4], zp[4], zn[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) z0[i] = zp[i] = zn[i] = floatx4{0.f, 0.f, 0.f, 0.f};
      const float* vcol = buf + (cb * 16 + (lane & 15)) * 4 + (lane >> 4);
      static_for<0, 4>([&](auto j_) {
        constexpr int j = decltype(j_)::value;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = vcol[(i * 4 + j) * TILES * 4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if constexpr (j <= 2) z0[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(u[i * 4 + j], v[i], z0[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (j == 1) zp[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(u[i * 4 + j], v[i], zp[i], 0, 0, 0);
          if constexpr (j >= 2) zn[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(u[i * 4 + j], v[i], zn[i], 0, 0, 0);
        }
      });
      floatx4 out[2][2];
#pragma unroll
      for (int ob = 0; ob < 2; ++ob) {
        floatx4 z[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) z[i] = ob == 0 ? z0[i] : zp[i] - zn[i];
        out[0][ob] = z[0] + z[1] + z[2];
        out[1][ob] = z[1] - z[2] - z[3];
      }
      const int p = blk * TILES + cb * 16 + (lane & 15);
      const int ko = kbase + 4 * (lane >> 4);
      store_tile<T, KW, 2>(a, ydesc, p, ko, p < a.P && ko < a.K, bv, out);
    }
  }
}

template <typename T>
int launch_tiny(ThinArgs a, int k_groups, void* stream) {
  constexpr int lds = 2 * 16 * 64 * 4 * 4;
  a.n_blocks = ceil_div(a.P, 64);
  int wgs = std::min(a.n_blocks, std::max(kXcds, 1024 / k_groups / kXcds * kXcds));
  a.per_xcd = ceil_div(wgs, kXcds);
  if (a.k_whole)
    hipLaunchKernelGGL((tiny_conv3x3_kernel<T, true>), dim3((unsigned)(a.per_xcd * kXcds), (unsigned)k_groups), dim3(256), lds,
                       as_stream(stream), a);
  else
    hipLaunchKernelGGL((tiny_conv3x3_kernel<T, false>), dim3((unsigned)(a.per_xcd * kXcds), (unsigned)k_groups), dim3(256), lds,
                       as_stream(stream), a);
  WC_CHECK_LAUNCH("tiny_conv3x3_kernel");
  return WC_OK;
}

template <typename T, int CP, int KSUB>
int launch_thin_groups(ThinArgs a, void* stream) {
  constexpr int lds = kThinLds<T, CP, KSUB>, threads = kThinThreads<T, CP, KSUB>;
  const int k_groups = ceil_div(a.K, 16 * KSUB);
  // workgroups that stay resident (registers and LDS): two per CU, one of thin_rows_kernel;
  // shared among the groups of output channels, in whole multiples of the 8 XCDs
  int wgs = std::min(a.n_blocks, std::max(kXcds, (kThinRows<T, CP> ? 256 : 512) / k_groups / kXcds * kXcds));
  a.per_xcd = ceil_div(wgs, kXcds);
  void (*fn)(ThinArgs);
  if constexpr (kThinRows<T, CP>) fn = a.k_whole ? &thin_rows_kernel<T, CP, true, KSUB> : &thin_rows_kernel<T, CP, false, KSUB>;
  else fn = a.k_whole ? &thin_conv3x3_kernel<T, CP, true, KSUB> : &thin_conv3x3_kernel<T, CP, false, KSUB>;
  if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds)) return rc;
  hipLaunchKernelGGL(fn, dim3((unsigned)(a.per_xcd * kXcds), (unsigned)k_groups), dim3(threads), lds, as_stream(stream), a);
  WC_CHECK_LAUNCH("thin_conv3x3_kernel");
  return WC_OK;
}

template <typename T, int CP>
int launch_thin(ThinArgs a, void* stream) {
  // half-size workgroups while the full-size ones would fill at most half of the CUs (a thread's channels must be all inside C or all outside)
  constexpr int vec2 = kThinTiles * CP / kThinThreads<T, CP, 2>;
  const int forced = test_gemm_config();            // wc_test_gemm_override: 8 = full size, 9 = half size
  const bool half = forced == 9 || (forced != 8 && (long long)a.n_blocks * ceil_div(a.K, kThinK) * 2 <= kCus);
  if (half && a.C % vec2 == 0) return launch_thin_groups<T, CP, 2>(a, stream);
  return launch_thin_groups<T, CP, 4>(a, stream);
}

}  // namespace

bool thin_conv_fits(const wc_conv_desc* d, const wc_plan* plan) {
  if (d->ndim != 2 || d->whole_kernel) return false;
  if (plan->n_pieces != 1 || plan->tap_step != 1 || plan->m[0] != 1 || plan->m[1] != 2 || plan->m[2] != 2) return false;
  const wc_piece& pc = plan->piece[0];
  if (pc.r[0] != 1 || pc.r[1] != 3 || pc.r[2] != 3) return false;
  const long long es = d->dtype == WC_F32 ? 4 : 2;
  if ((long long)d->N * d->in[1] * d->in[2] * d->C * es >= (1ll << 30)) return false;   // 32-bit offsets into x, two spare bits
  int out[3], grid[3];
  if (wc_conv_out_dims(d, out, grid) != WC_OK) return false;
  if ((long long)d->N * out[1] * out[2] * d->K * es >= (1ll << 31)) return false;      // and into y
  if (d->C <= 4) return d->K <= 8 * kThinK;          // tiny_conv3x3_kernel, any storage type
  const int Cp = wc_padded_channels(d->C);
  if (d->dtype == WC_F32) {
    // fp32: U of 32 channels fits four wavefronts, of 64 channels eight (the products run on fp32 MFMA)
    if (Cp > 64 || d->C % 2 != 0) return false;
    return d->K <= (Cp == 64 ? 4 : 8) * kThinK;
  }
  if (Cp > 128 || (Cp == 96) || d->C % (Cp == 32 ? 2 : 4) != 0) return false;
  return d->K <= (Cp == 128 ? 4 : 8) * kThinK;   // measured: no gain beyond (K = 512 at 128 channels: 0.97x)
}

int thin_conv_forward(const wc_conv_desc* d, const wc_plan* plan, const void* x, const void* U, const void* bias,
                      void* y, void* stream) {
  WC_CHECK_ARG(thin_conv_fits(d, plan), "thin_conv_forward: problem outside the kernel's range");
  int out[3], grid[3];
  int rc = wc_conv_out_dims(d, out, grid);
  if (rc) return rc;
  const int Cp = wc_padded_channels(d->C);
  const long long P = (long long)d->N * grid[1] * grid[2];
  WC_CHECK_ARG(P < (1ll << 31) - kThinTiles, "thin_conv_forward: too many tiles");
  WC_CHECK_ARG((reinterpret_cast<uintptr_t>(x) & 7) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(U) & 15) == 0,
               "thin_conv_forward: x must be 8-byte aligned, y and U 16-byte aligned");
  const int es = d->dtype == WC_F32 ? 4 : 2;
  ThinArgs a;
  a.x = x; a.U = U; a.bias = bias; a.y = y;
  a.H = d->in[1]; a.W = d->in[2]; a.C = d->C; a.K = d->K; a.Cp = Cp;
  a.oH = out[1]; a.oW = out[2]; a.nH = grid[1]; a.nW = grid[2];
  a.pad1 = d->pad[1]; a.pad2 = d->pad[2];
  a.P = (int)P;
  a.n_blocks = (int)ceil_div_ll(P, kThinTiles);
  a.per_xcd = 0;
  a.x_bytes = (int)((long long)d->N * d->in[1] * d->in[2] * d->C * es);
  a.y_bytes = (int)((long long)d->N * out[1] * out[2] * d->K * es);
  a.k_whole = d->K % 4 == 0;
  a.row_bytes = d->in[2] * d->C * es;
  a.div_nW = make_fast_div(a.nW);
  a.div_nH = make_fast_div(a.nH);
  const int k_groups = ceil_div(d->K, kThinK);
  if (d->C <= 4) return dispatch_dtype(d->dtype, [&](auto t) -> int { return launch_tiny<decltype(t)>(a, k_groups, stream); });
  return dispatch_dtype(d->dtype, [&](auto t) -> int {
    using T = decltype(t);
    if constexpr (sizeof(T) == 2) {
      if (Cp == 128) return launch_thin<T, 128>(a, stream);
      return Cp == 64 ? launch_thin<T, 64>(a, stream) : launch_thin<T, 32>(a, stream);
    } else {
      return Cp == 64 ? launch_thin<T, 64>(a, stream) : launch_thin<T, 32>(a, stream);
    }
  });
}

}  // namespace wc
