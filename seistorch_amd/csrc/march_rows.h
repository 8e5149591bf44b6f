// Kernels and helpers shared by the files that launch marching kernels: the
// receivers' cells in the rows of their depths, unit order, fills and copies.
#pragma once

#include "common.h"
#include "march.h"
#include "tiles.h"

#include <algorithm>

namespace {

using namespace seis::march;
using seis::tiles::kXcds;

__global__ __launch_bounds__(256) void k_fill_i32(int32_t* __restrict__ p, int64_t n, int32_t v) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = v;
}

// Receiver t's cell in the (slots, B, nx) rows; with head/next, the receivers
// of one cell are chained for the adjoint's sources.
__global__ __launch_bounds__(256) void k_row_cells(const int64_t* __restrict__ rec, int64_t R,
                                                   int64_t plane, int nx, int B,
                                                   const int32_t* __restrict__ row_slot,
                                                   int64_t* __restrict__ cell,
                                                   int32_t* __restrict__ head,
                                                   int32_t* __restrict__ next) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= R) return;
  const int64_t b = rec[t] / plane, i = rec[t] - b * plane;
  const int64_t c = ((int64_t)row_slot[i / nx] * B + b) * nx + i % nx;
  if (cell) cell[t] = c;
  if (head) next[t] = atomicExch(head + c, (int32_t)t);
}

// XCD-aware block order, as tiles.h: each XCD takes a contiguous range.
__device__ __forceinline__ int xcd_block(int per) {
  const int w = blockIdx.x;
  return (w % kXcds) * per + w / kXcds;
}

__device__ __forceinline__ bool march_unit(const Split& sp, int B, int blk, int& strip, int& seg,
                                           int& b) {
  const int64_t unit = (int64_t)blk * kWavesPerBlock +
                       __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int64_t row = unit / sp.group, row2 = row / sp.strips;
  strip = (int)(row - row2 * sp.strips);
  seg = (int)(row2 % sp.segs);
  b = (int)(row2 / sp.segs) * sp.group + (int)(unit - row * sp.group);
  return b < B;
}

template <typename P>
__device__ __forceinline__ Const<P> launch_params() {
  return (Const<P>)__builtin_amdgcn_kernarg_segment_ptr();
}

__global__ __launch_bounds__(256) void k_zero(float* __restrict__ p, int64_t n) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0.0f;
}

__global__ __launch_bounds__(256) void k_copy(const float* __restrict__ a, float* __restrict__ b,
                                              int64_t n) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) b[t] = a[t];
}

inline unsigned blocks_of(int64_t n) { return (unsigned)((n + 255) / 256); }

inline int zero(float* p, int64_t n, hipStream_t s) {
  k_zero<<<blocks_of(n), 256, 0, s>>>(p, n);
  SEIS_CHECK_LAUNCH();
  return 0;
}

inline int64_t pad64(int64_t n) { return (n + 63) / 64 * 64; }

inline int aux_blocks(int64_t n) { return (int)std::min<int64_t>((n + kThreads - 1) / kThreads, 512); }

inline int64_t split_blocks(const Split& sp, int64_t B) {
  const int64_t units = (int64_t)sp.strips * sp.segs * sp.group * ((B + sp.group - 1) / sp.group);
  return (units + kWavesPerBlock - 1) / kWavesPerBlock;
}

}  // namespace
