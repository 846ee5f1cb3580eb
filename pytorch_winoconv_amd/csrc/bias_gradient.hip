// Bias gradient: db[k] = sum over the rows p of dy[p][k], dy (P, K) channel-last as the convolution wrote y.  The reference
// has no backward pass (src/back/utils.cu:15-24).
//
// One read of dy bounds it.  A workgroup takes a run of rows, a thread 16 bytes of a row (less where rows are no multiple of that)
// with fp32 sums in registers, neighbouring threads neighbouring bytes; the threads of a channel meet in LDS, the workgroups'
// sums in a second kernel, all in a fixed order.  Measured, us, torch's sum | this: fp16 N=8 128 channels, 16x56x56 (103 MB)
// 49 | 22 (4.7 TB/s), N=64 128 channels, 28x28 19 | 6.6, bf16 N=32 256 channels, 28x28 25 | 6.5, fp32 N=8 256 channels, 56x56
// 24 | 7.8, N=1 512 channels, 7x7 (two launches) 5.8 | 5.6.
#include "column_sums.h"

#include <algorithm>

namespace wc {

namespace {

constexpr int kBiasThreads = 256;

struct BiasPlan { int vec, cols, col_tiles, groups, blocks; long long rows_per_block; };

// vec: elements of a thread's load.  cols: loads side by side in a workgroup, groups: its rows in flight.
BiasPlan bias_plan(long long P, int K, int dtype, bool aligned) {
  BiasPlan p;
  const int es = dtype == WC_F32 ? 4 : 2;
  p.vec = aligned ? 16 / es : 1;
  while (K % p.vec) p.vec /= 2;
  const int n = K / p.vec;
  p.cols = std::min(n, kBiasThreads);
  p.col_tiles = ceil_div(n, p.cols);
  p.groups = kBiasThreads / p.cols;
  // 64 KB a workgroup, and at most two rounds of the eight that a CU holds: below that a workgroup is mostly its own start
  const long long blocks = std::max(1ll, std::min(4096ll / p.col_tiles, P * K * es / 65536));
  p.rows_per_block = ceil_div_ll(P, blocks);
  p.blocks = (int)ceil_div_ll(P, p.rows_per_block);
  return p;
}

template <typename T, int VEC>
__global__ __launch_bounds__(kBiasThreads) void bias_rows_kernel(RowSums a) {
  __shared__ float sums[kBiasThreads * (VEC + (VEC > 1))];
  sum_rows<T, VEC>(a, blockIdx.x, blockIdx.y, sums);
}

// db[k] = sum over the workgroups' rows; 16 channels a workgroup, 64 threads to a channel's sums
template <typename T>
__global__ __launch_bounds__(1024) void bias_parts_kernel(const float* __restrict__ part, void* __restrict__ db, int blocks, int K, bool f32) {
  __shared__ float sums[64][16];
  const int c = threadIdx.x & 15, group = threadIdx.x >> 4, k = blockIdx.x * 16 + c;
  float s = 0.f;
  if (k < K) {
#pragma unroll 4
    for (int b = group; b < blocks; b += 64) s += part[(long long)b * K + k];
  }
  sums[group][c] = s;
  __syncthreads();
  for (int half = 32; half > 0; half >>= 1) {
    if (group < half) sums[group][c] += sums[group + half][c];
    __syncthreads();
  }
  if (group == 0 && k < K) store_as<T>(db, k, sums[0][c], f32);
}

}  // namespace

// (the number of workgroups is the larger where a thread reads 16 bytes)
size_t bias_part_bytes(long long rows, int K, int dtype) {
  return (size_t)std::max(bias_plan(rows, K, dtype, true).blocks, bias_plan(rows, K, dtype, false).blocks) * K * 4;
}

RowSums row_sums_of(const void* dy, float* part, long long rows, int K, int dtype) {
  const BiasPlan p = bias_plan(rows, K, dtype, (reinterpret_cast<uintptr_t>(dy) & 15) == 0);
  return {dy, part, rows, p.rows_per_block, K, p.vec, p.cols, p.groups, p.blocks, p.col_tiles};
}

int bias_sums(const void* dy, void* db, long long rows, int K, int dtype, bool f32, float* part, void* stream) {
  const RowSums a = row_sums_of(dy, part, rows, K, dtype);
  return dispatch_dtype(dtype, [&](auto t) -> int {
    using T = decltype(t);
    constexpr int FULL = 16 / sizeof(T);
    auto fn = a.vec == FULL ? &bias_rows_kernel<T, FULL> : a.vec == 4 ? &bias_rows_kernel<T, 4> : a.vec == 2 ? &bias_rows_kernel<T, 2>
                                                                                             : &bias_rows_kernel<T, 1>;
    hipLaunchKernelGGL(fn, dim3((unsigned)a.blocks, (unsigned)a.col_tiles), dim3(kBiasThreads), 0, as_stream(stream), a);
    WC_CHECK_LAUNCH("bias_rows_kernel");
    hipLaunchKernelGGL(bias_parts_kernel<T>, dim3((unsigned)ceil_div(K, 16)), dim3(1024), 0, as_stream(stream), part,
                       db, a.blocks, K, f32);
    WC_CHECK_LAUNCH("bias_parts_kernel");
    return WC_OK;
  });
}

}  // namespace wc

using namespace wc;

extern "C" {

int wc_bias_gradient_workspace_bytes(long long rows, int K, int dtype, size_t* bytes) {
  WC_CHECK_ARG(bytes != nullptr, "wc_bias_gradient_workspace_bytes: null output");
  WC_CHECK_ARG(rows > 0 && K > 0 && (dtype == WC_F32 || dtype == WC_F16 || dtype == WC_BF16), "rows %lld, K %d, dtype %d", rows, K, dtype);
  *bytes = bias_part_bytes(rows, K, dtype);
  return WC_OK;
}

int wc_bias_gradient(const void* dy, void* db, long long rows, int K, int dtype, void* workspace, size_t workspace_bytes, void* stream) {
  size_t need = 0;
  if (int rc = wc_bias_gradient_workspace_bytes(rows, K, dtype, &need)) return rc;
  WC_CHECK_ARG(dy && db, "wc_bias_gradient: null pointer");
  if (!workspace || workspace_bytes < need)
    return fail(WC_ERR_WORKSPACE, "wc_bias_gradient: workspace of %zu bytes, %zu needed", workspace ? workspace_bytes : (size_t)0, need);
  if ((reinterpret_cast<uintptr_t>(workspace) & 15) != 0) return fail(WC_ERR_WORKSPACE, "wc_bias_gradient: workspace must be 16-byte aligned");
  return bias_sums(dy, db, rows, K, dtype, false, static_cast<float*>(workspace), stream);
}

}  // extern "C"
