// Reduction of the bias gradient behind fa_bias_grad_reduce, and the bias tensor's copy with padded rows (fa_pad_bias_rows).  The dK/dV kernel writes the gradient of an attn_bias tensor
// per (batch, head); a bias that was broadcast over the batch and/or the heads wants the sum over the entries that shared
// it.  One pass: every thread owns 8 consecutive keys of one output row, adds the slices in a fixed order (batch outer,
// head inner) in fp32 and rounds once.  HBM-bound: each input element is read once, each output element written once.  With the batch's
// lengths (cu_q, cu_k) only what the dK/dV kernel writes is read - the rows and keys a sequence has, under a causal mask up to the
// diagonal - so the slices need no clearing: training steps of 8 x 16 heads x 660 .. 1100, d = 64 502 -> 404 us, 8 x 12 x 900, d = 32 254 -> 227.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "fa_params.h"

namespace fa {

namespace {

template <typename T, bool kVecStore>
__global__ void __launch_bounds__(256) bias_grad_reduce_kernel(const T* __restrict__ in, T* __restrict__ out, int nb, int nh,
                                                               int rows, int cols, int64_t in_bs, int64_t in_hs,
                                                               int64_t in_rs, int64_t out_bs, int64_t out_hs, int64_t out_rs,
                                                               int sum_batch, int sum_heads, const BiasGradLens l) {
  typedef Elem<T> E;
  const int cpr = (cols + 7) >> 3;  // chunks of 8 keys per row (the input rows are padded to whole chunks)
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)rows * cpr) return;
  const int row = (int)(i / cpr), ch = (int)(i % cpr);
  const int ho = blockIdx.y, bo = blockIdx.z;
  const int b0 = sum_batch ? 0 : bo, b1 = sum_batch ? nb : bo + 1;
  const int h0 = sum_heads ? 0 : ho, h1 = sum_heads ? nh : ho + 1;
  float acc[8];
#pragma unroll
  for (int j = 0; j < 8; j++) acc[j] = 0.f;
  const T* const src = in + (int64_t)row * in_rs + ch * 8;
  for (int b = b0; b < b1; b++) {
    int n = cols;  // keys of this row that hold a gradient
    if (l.cu_q) {
      int begin, Lq, Lk;
      n = 0;
      if (seq_extent(l.cu_q, b, l.total_q, l.max_sq, &begin, &Lq) && seq_extent(l.cu_k, b, l.total_k, l.max_sk, &begin, &Lk) && row < Lq)
        n = l.causal && row + 1 < Lk ? row + 1 : Lk;
      if (ch * 8 >= n) continue;
    }
    for (int h = h0; h < h1; h++) {
      const typename E::vec8 v = *reinterpret_cast<const typename E::vec8*>(src + (int64_t)b * in_bs + (int64_t)h * in_hs);
#pragma unroll
      for (int j = 0; j < 8; j++) acc[j] += ch * 8 + j < n ? (float)v[j] : 0.f;
    }
  }
  T* const dst = out + (int64_t)bo * out_bs + (int64_t)ho * out_hs + (int64_t)row * out_rs + ch * 8;
  if (kVecStore && ch * 8 + 8 <= cols) {
    typename E::vec8 r;
#pragma unroll
    for (int j = 0; j < 8; j++) r[j] = (T)acc[j];
    *reinterpret_cast<typename E::vec8*>(dst) = r;
  } else {
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (ch * 8 + j < cols) dst[j] = (T)acc[j];
  }
}

// A bias tensor's rows copied to rows of whole 16-byte chunks, zeros behind the last key, for tensors whose rows the attention kernels cannot
// read as they are (odd lengths, other strides).  HBM-bound: a thread moves one chunk, read whole where its eight keys are there and lie
// together (a row of odd length starts at any even address: an unaligned 16-byte load; eight 2-byte loads took 85 us for 8 x 12 x 901
// x 901), a workgroup the chunks of four rows (8 rows 69, 4 rows 66, 2 rows 74).  us of a clearing and a strided copy / this: 8 x 701 x 701
// 8.0 / 6.2, 16 x 1100 x 1100 22.9 / 14.5, 12 x 2047 x 2047 52.6 / 40.4 (5.0 TB/s moved), 8 x 16 x 1101 x 1101 169 / 125.
// (Groups of rows in a loop over a bounded grid, see pad_bias_grid.)
__global__ void __launch_bounds__(256) pad_bias_rows_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst, int nh, int64_t rows,
                                                            int64_t cols, int cpr, int64_t row_groups, int64_t groups, int64_t s_bs,
                                                            int64_t s_hs, int64_t s_rs, int64_t s_ks) {
  for (int64_t g = blockIdx.x; g < groups; g += gridDim.x) {
    const int64_t bh = g / row_groups, r0 = (g - bh * row_groups) * kPadBiasRows;
    const int nrows = (int)(rows - r0 < kPadBiasRows ? rows - r0 : kPadBiasRows);
    const uint16_t* const s = src + bh / nh * s_bs + bh % nh * s_hs + r0 * s_rs;
    uint16_t* const d = dst + (bh * rows + r0) * cpr * 8;
    const unsigned n = (unsigned)nrows * (unsigned)cpr;
    for (unsigned t = threadIdx.x; t < n; t += 256) {
      const unsigned i = t / (unsigned)cpr;
      const int64_t col0 = (int64_t)(t - i * (unsigned)cpr) * 8;
      union { uint16_t e[8]; uint4 v; } c;
      const uint16_t* const from = s + i * s_rs + col0 * s_ks;
      if (s_ks == 1 && col0 + 8 <= cols) {
        __builtin_memcpy(c.e, from, 16);
      } else {
#pragma unroll
        for (int j = 0; j < 8; j++) {
          c.e[j] = 0;
          if (col0 + j < cols) c.e[j] = from[j * s_ks];
        }
      }
      *reinterpret_cast<uint4*>(d + (int64_t)t * 8) = c.v;
    }
  }
}

}  // namespace

hipError_t launch_pad_bias_rows(const void* src, void* dst, int nb, int nh, int64_t rows, int64_t cols, int64_t s_bs, int64_t s_hs, int64_t s_rs,
                                int64_t s_ks, hipStream_t stream) {
  if (nb == 0 || nh == 0 || rows == 0 || cols == 0) return hipSuccess;
  const PadBiasGrid g = pad_bias_grid(nb, nh, rows);
  hipLaunchKernelGGL(pad_bias_rows_kernel, dim3(g.blocks), dim3(256), 0, stream, reinterpret_cast<const uint16_t*>(src),
                     reinterpret_cast<uint16_t*>(dst), nh, rows, cols, (int)((cols + 7) >> 3), g.row_groups, g.groups, s_bs, s_hs, s_rs, s_ks);
  return hipGetLastError();
}

hipError_t launch_bias_grad_reduce(const void* in, void* out, int dtype, int nb, int nh, int rows, int cols, int64_t in_bs,
                                   int64_t in_hs, int64_t in_rs, int sum_batch, int sum_heads, int64_t out_bs, int64_t out_hs,
                                   int64_t out_rs, const BiasGradLens& lens, bool vec_store, hipStream_t stream) {
  if (nb == 0 || nh == 0 || rows == 0 || cols == 0) return hipSuccess;
  const int64_t n = (int64_t)rows * ((cols + 7) >> 3);
  const dim3 grid((unsigned)((n + 255) / 256), (unsigned)(sum_heads ? 1 : nh), (unsigned)(sum_batch ? 1 : nb));
#define FA_BGR(T, V)                                                                                                   \
  hipLaunchKernelGGL((bias_grad_reduce_kernel<T, V>), grid, dim3(256), 0, stream, reinterpret_cast<const T*>(in),      \
                     reinterpret_cast<T*>(out), nb, nh, rows, cols, in_bs, in_hs, in_rs, out_bs, out_hs, out_rs, sum_batch, \
                     sum_heads, lens)
  if (dtype == 0) {
    if (vec_store) FA_BGR(_Float16, true); else FA_BGR(_Float16, false);
  } else {
    if (vec_store) FA_BGR(__bf16, true); else FA_BGR(__bf16, false);
  }
#undef FA_BGR
  return hipGetLastError();
}

}  // namespace fa
