// Sums of per-workgroup partials over the workgroups, in a fixed order.
#pragma once

#include "pkda_common.h"

namespace pkda {
namespace {  // one copy per translation unit

// out[i] = sum over p in [0, count) of part[p * stride + i], i in [0, n).
struct ColumnSum {
  const float* part;
  void* out;
  int count, stride, n;
  int out_dtype;
  int blocks;  // workgroups that take it: ceil(n / COLS)
};

// A workgroup takes COLS adjacent columns.  The partials of a column are summed
// in 256 classes -- class c takes c, c + 256, ... in order -- and the classes in
// a halving tree, so a chain is count / 256 additions long.  Thread (slot,
// column) holds the classes slot, slot + SLOTS, ... in registers: their loads go
// out together, and the COLS threads of a slot read adjacent words.  It takes the
// tree down to one sum a slot, LDS the rest.  Two sums share a launch; the
// second may be empty.
//
// With many columns the partials' bytes bound it, with few the loads'
// latency, so the width follows n:
//   n >= 8192  whole 128-byte lines, 1,024 threads: 512 x 12,288 partials
//              (25 MB, the convolution's dw) in 7.1 us; 256 threads 10.1
//   n >= 2048  64-byte pieces, 256 threads, which find room beside another
//              stream's workgroups where 1,024 wait: 512 x 2,048 (the gate's
//              ddt_bias) 106 us beside the preconditioner's last pass against
//              118, and that pass 155 -> 150 us
//   else       32-byte pieces, four times the workgroups on the same partials:
//              1,024 x 128 (the gated norm's dweight) in 4.2 us
// The forms before it took one workgroup per column, a line fetched per word
// (190 us for the gate's two sums), or two launches of few workgroups (18.8 us
// for the norm's dweight, 15.8 for the convolution's dw).
template <int COLS, int THREADS>
__global__ __launch_bounds__(THREADS) void column_sums_kernel(ColumnSum a, ColumnSum b) {
  constexpr int SLOTS = THREADS / COLS, CLASSES = 256, K = CLASSES / SLOTS;
  __shared__ float s[THREADS];
  const bool first = (int)blockIdx.x < a.blocks;
  const ColumnSum& j = first ? a : b;
  const int col = threadIdx.x % COLS, slot = threadIdx.x / COLS;
  const int i = (blockIdx.x - (first ? 0 : a.blocks)) * COLS + col;
  float acc[K];
#pragma unroll
  for (int c = 0; c < K; ++c) acc[c] = 0.f;
  if (i < j.n) {
    const float* __restrict__ p = j.part + i;
    int q = slot;
#pragma unroll 2
    for (; q - slot + CLASSES <= j.count; q += CLASSES)  // whole rounds
#pragma unroll
      for (int c = 0; c < K; ++c) acc[c] += p[(int64_t)(q + c * SLOTS) * j.stride];
    if (q - slot < j.count) {  // the last round: rows past the end read the last one and add 0
#pragma unroll
      for (int c = 0; c < K; ++c) {
        const float x = p[(int64_t)min(q + c * SLOTS, j.count - 1) * j.stride];
        acc[c] += q + c * SLOTS < j.count ? x : 0.f;
      }
    }
  }
#pragma unroll
  for (int off = K / 2; off > 0; off >>= 1)
#pragma unroll
    for (int c = 0; c < off; ++c) acc[c] += acc[c + off];
  s[threadIdx.x] = acc[0];
  __syncthreads();
#pragma unroll
  for (int off = SLOTS / 2; off > 0; off >>= 1) {
    if (slot < off) s[threadIdx.x] += s[threadIdx.x + off * COLS];
    __syncthreads();
  }
  if (slot == 0 && i < j.n) {
    if (j.out_dtype == PKDA_BF16) static_cast<bf16_t*>(j.out)[i] = f32_to_bf16(s[col]);
    else static_cast<float*>(j.out)[i] = s[col];
  }
}

inline ColumnSum column_sum(const float* part, int count, int stride, int n, void* out, int out_dtype = PKDA_F32) {
  return {part, out, count, stride, n, out_dtype, 0};
}

inline int launch_column_sums(ColumnSum a, ColumnSum b, hipStream_t s, const char* what) {
  const int n = a.n > b.n ? a.n : b.n;
  if (n <= 0) return 0;
  const int cols = n >= 8192 ? 32 : n >= 2048 ? 16 : 8;
  a.blocks = (a.n + cols - 1) / cols;
  b.blocks = (b.n + cols - 1) / cols;
  const dim3 grid((unsigned)(a.blocks + b.blocks));
  if (cols == 32) hipLaunchKernelGGL((column_sums_kernel<32, 1024>), grid, dim3(1024), 0, s, a, b);
  else if (cols == 16) hipLaunchKernelGGL((column_sums_kernel<16, 256>), grid, dim3(256), 0, s, a, b);
  else hipLaunchKernelGGL((column_sums_kernel<8, 256>), grid, dim3(256), 0, s, a, b);
  return launch_status(what);
}

}  // namespace
}  // namespace pkda
