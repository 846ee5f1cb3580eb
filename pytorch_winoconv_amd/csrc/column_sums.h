// Column sums of dy (the bias gradient) beside a weight gradient, whose kernels have dy's rows in LDS: the wavefronts that hold the
// same rows take turns, stage by stage, at adding one stage's rows up, so no launch and no second read of dy is left of it.
//
// A bias gradient of its own reads dy again and is two launches.  us of a layer's weight and bias gradient, two calls | one, fp16:
// N=64 128 -> 128, 28x28 46.6 | 40.4; N=8 128 -> 128, 16x56x56 356 | 338; stride 2, N=32 128 -> 256, 56x56 41.2 | 35.3.  Sums are fp32, in a fixed order.
#pragma once
#include "wc_common.h"

namespace wc {

// s += the lane's columns of `rows` rows (a multiple of 8) at `st`, COLS 16-bit columns each, PITCH bytes apart.  64 columns: the wavefront's
// halves take every other row.  SWAP: the rows' 64-byte pieces are exchanged as LDS-DMA leaves them (row & 3, of 64 columns (row >> 1) & 1).
template <typename T, int COLS, int PITCH, bool SWAP>
__device__ __forceinline__ void add_rows(const unsigned char* st, int rows, int lane, float (&s)[2]) {
  static_assert(COLS == 64 || COLS == 128, "one or two 16-bit columns a lane");
  const unsigned char* const p = COLS == 128 ? st + lane * 4 : st + (lane >> 5) * PITCH;
  const int col = COLS == 128 ? 0 : (lane & 31) * 4;
  for (int r0 = 0; r0 < rows; r0 += 8) {
    Pack<T, 2> v[COLS / 16];
#pragma unroll
    for (int i = 0; i < COLS / 16; ++i) {
      const int r = i * 128 / COLS;                 // and, of 64 columns, the row after it, of the same piece
      const unsigned char* const q = SWAP ? st + ((COLS == 128 ? lane * 4 : col) ^ (COLS == 128 ? (r & 3) * 64 : ((r >> 1) & 1) * 64)) + (COLS == 128 ? 0 : (lane >> 5) * PITCH)
                                          : p + col;
      v[i] = *reinterpret_cast<const Pack<T, 2>*>(q + (r0 + r) * PITCH);
    }
#pragma unroll
    for (int i = 0; i < COLS / 16; ++i) {
      s[0] += static_cast<float>(v[i].v[0]);
      s[1] += static_cast<float>(v[i].v[1]);
    }
  }
}

// out[0 .. COLS) = the sums of a workgroup's NW wavefronts, through LDS that nobody uses any more (all threads call it)
template <int NW, int COLS>
__device__ __forceinline__ void store_sums(float (&s)[2], float* lds, int wave, int lane, float* out) {
  if constexpr (COLS == 64) {
#pragma unroll
    for (int e = 0; e < 2; ++e) s[e] += __shfl_xor(s[e], 32);
  }
  __syncthreads();
  if (COLS == 128 || lane < 32) *reinterpret_cast<float2*>(lds + wave * COLS + lane * 2) = float2{s[0], s[1]};
  __syncthreads();
  const int c = wave * 64 + lane;
  if (c >= COLS) return;
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) t += lds[w * COLS + c];
  out[c] = t;
}

// A result of the parameter's type: T, or fp32 where the parameter is (without T's rounding)
template <typename T>
__device__ __forceinline__ void store_as(void* p, long long i, float v, bool f32) {
  if (f32) static_cast<float*>(p)[i] = v;
  else static_cast<T*>(p)[i] = static_cast<T>(v);
}

// db[16 b .. 16 b + 15] = the sums of `rows` rows of `ld` floats, by a workgroup of 256
struct ColumnSums {
  const float* part;       // null: none
  void* db;
  int rows, ld, K, f32;
};
template <typename T>
__device__ __forceinline__ void sum_columns(const ColumnSums& a, int b, float* lds) {
  const int c = threadIdx.x & 15, group = threadIdx.x >> 4, k = b * 16 + c;
  float t = 0.f;
  if (k < a.K) {
#pragma unroll 8
    for (int r = group; r < a.rows; r += 16) t += a.part[(long long)r * a.ld + k];
  }
  lds[threadIdx.x] = t;
  __syncthreads();
  if (group || k >= a.K) return;
  for (int j = 1; j < 16; ++j) t += lds[j * 16 + c];
  store_as<T>(a.db, k, t, a.f32);
}

// The same from rows of a pass over dy of its own, in the order of bias_parts_kernel (bias_gradient.hip): 64 runs of rows, then halves
template <typename T>
__device__ __forceinline__ void sum_columns_halves(const ColumnSums& a, int b, float* lds) {
  const int c = threadIdx.x & 15, group = threadIdx.x >> 4, k = b * 16 + c;
  float t[4] = {0.f, 0.f, 0.f, 0.f};
  if (k < a.K) {
    for (int r = group; r < a.rows; r += 64) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (r + 16 * j < a.rows) t[j] += a.part[(long long)(r + 16 * j) * a.ld + k];
    }
  }
  float s = (t[0] + t[2]) + (t[1] + t[3]);
  for (int half = 8; half > 0; half >>= 1) {
    lds[threadIdx.x] = s;
    __syncthreads();
    if (group < half) s += lds[threadIdx.x + half * 16];
    __syncthreads();
  }
  if (group == 0 && k < a.K) store_as<T>(a.db, k, s, a.f32);
}

// Sums over runs of dy's rows by workgroups of 256, `blocks` runs times `col_tiles`: a thread adds `vec` columns up, `cols` of them side by side
struct RowSums {
  const void* dy;
  float* part;             // (blocks, K)
  long long rows, rows_per_block;
  int K, vec, cols, groups, blocks, col_tiles;
};
RowSums row_sums_of(const void* dy, float* part, long long rows, int K, int dtype);

template <typename T, int VEC>
__device__ __forceinline__ void sum_rows(const RowSums& a, int block, int tile, float* lds) {
  constexpr int PITCH = VEC + (VEC > 1);
  const int group = threadIdx.x / a.cols, col = threadIdx.x - group * a.cols;
  const int k = (tile * a.cols + col) * VEC;
  const long long begin = block * a.rows_per_block, end = min(a.rows, begin + a.rows_per_block);
  float s[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) s[e] = 0.f;
  if (group < a.groups && k < a.K) {
    const T* p = static_cast<const T*>(a.dy) + (begin + group) * a.K + k;
    const long long step = (long long)a.groups * a.K;
    long long r = begin + group;
    for (; r + 3 * a.groups < end; r += 4 * a.groups, p += 4 * step) {
      Pack<T, VEC> v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const Pack<T, VEC>*>(p + i * step);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < VEC; ++e) s[e] += static_cast<float>(v[i].v[e]);
    }
    for (; r < end; r += a.groups, p += step) {
      const Pack<T, VEC> v = *reinterpret_cast<const Pack<T, VEC>*>(p);
#pragma unroll
      for (int e = 0; e < VEC; ++e) s[e] += static_cast<float>(v.v[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < VEC; ++e) lds[threadIdx.x * PITCH + e] = s[e];
  __syncthreads();
  for (int i = threadIdx.x; i < a.cols * VEC; i += 256) {
    const int c = i / VEC, e = i - c * VEC;
    const int kk = (tile * a.cols + c) * VEC + e;
    if (kk >= a.K) continue;
    float t = 0.f;
    for (int g = 0; g < a.groups; ++g) t += lds[(g * a.cols + c) * PITCH + e];
    a.part[(long long)block * a.K + kk] = t;
  }
}

// whatever the width of a thread's loads; lds: 256 (16 / sizeof(T) + 1) floats
template <typename T>
__device__ __forceinline__ void sum_rows_any(const RowSums& a, int block, int tile, float* lds) {
  if (sizeof(T) == 2 && a.vec == 8) sum_rows<T, 16 / sizeof(T)>(a, block, tile, lds);
  else if (a.vec == 4) sum_rows<T, 4>(a, block, tile, lds);
  else if (a.vec == 2) sum_rows<T, 2>(a, block, tile, lds);
  else sum_rows<T, 1>(a, block, tile, lds);
}

}  // namespace wc
