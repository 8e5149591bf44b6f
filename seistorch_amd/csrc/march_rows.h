// Kernels and helpers shared by the files that launch marching kernels: the
// receivers' cells in the rows of their depths, unit order, fills and copies.
#pragma once

#include "common.h"
#include "march.h"
#include "tiles.h"

#include <algorithm>

namespace {

using namespace seis::march;
using seis::Grid;
using seis::TimeConsts;
using seis::tiles::kXcds;

__global__ __launch_bounds__(256) void k_fill_i32(int32_t* __restrict__ p, int64_t n, int32_t v) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = v;
}

// Marked rows numbered from the top, their count in row_slot[nz]; one wave.
__global__ __launch_bounds__(64) void k_number_rows(int32_t* __restrict__ row_slot, int nz) {
  int base = 0;
  for (int z0 = 0; z0 < nz; z0 += 64) {
    const int z = z0 + (int)threadIdx.x;
    const bool on = z < nz && row_slot[z] >= 0;
    const unsigned long long m = __ballot(on);
    if (on) row_slot[z] = base + __popcll(m & ((1ull << threadIdx.x) - 1));
    base += __popcll(m);
  }
  if (threadIdx.x == 0) row_slot[nz] = base;
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

inline int aux_blocks(int64_t n) {
  return (int)std::min<int64_t>((n + kThreads - 1) / kThreads, 512);
}

inline int64_t split_blocks(const Split& sp, int64_t B) {
  const int64_t units = (int64_t)sp.strips * sp.segs * sp.group * ((B + sp.group - 1) / sp.group);
  return (units + kWavesPerBlock - 1) / kWavesPerBlock;
}

// c^2, A and B of the damped update, once per loop (d null: none).
__global__ __launch_bounds__(256) void k_coefs(const float* __restrict__ vp,
                                               const float* __restrict__ d, int64_t plane,
                                               TimeConsts k, float* __restrict__ c2,
                                               float* __restrict__ A, float* __restrict__ Bc) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= plane) return;
  const float c = vp[i], dd = d ? d[i] : 0.0f;
  c2[i] = c * c;
  A[i] = 1.0f / (k.idt2 + dd * k.idt);
  Bc[i] = k.idt2 - dd * k.idt;
}

// Adjoint sources of the next launch's levels in the receivers' rows, filled by
// blocks after a march's.
struct Sources {
  float* rows;           // (levels, row_cells) of the next launch
  const int32_t *head, *next;
  int64_t R, row_cells;
  const float* rgrad;    // row of the first level; the next level's precedes it
  int levels, blocks;
};

__device__ __forceinline__ void fill_sources(const Sources& so, int block) {
  for (int64_t c = (int64_t)block * kThreads + threadIdx.x; c < so.row_cells;
       c += (int64_t)so.blocks * kThreads) {
    const int32_t h = so.head[c];
    for (int lev = 0; lev < so.levels; ++lev) {
      const float* rg = so.rgrad - (int64_t)lev * so.R;
      float s = 0.0f;
      for (int32_t t = h; t >= 0; t = so.next[t]) s += rg[t];
      so.rows[lev * so.row_cells + c] = s;
    }
  }
}

__global__ __launch_bounds__(kThreads) void k_sources(Sources so) { fill_sources(so, blockIdx.x); }

// Shots whose waves run side by side on the same strips.  Eight share the
// coefficient rows in L2 while neighbouring segments still find each other's
// halo rows in the last-level cache: 64 shots of 900 x 2500, 10^9 cell updates
// per second of the adjoint with groups of 1 / 4 / 8 / 16 / 64: 335 / 393 /
// 399 / 375 / 343; of the forward 887 / 922 / 937 / 921 / 836.
constexpr int kShotGroup = 8;

constexpr int kMaxT = kMaxSteps;
// Steps of the next launch when `left` remain to the next boundary: the remainder
// first, so that the launch that ends at the boundary takes all max_t steps (and can
// write both fields of a snapshot).  With fewer left, the last launch may be a single
// step, and the pair's first field is copied.
inline int next_steps(int64_t left, int max_t) {
  const int64_t r = left % max_t;
  if (r == 0) return max_t;
  return r >= 2 ? 2 : 1;
}

inline int widest(int64_t nx) { return nx % 4 == 0 ? 4 : nx % 2 == 0 ? 2 : 1; }

struct Plan {
  int vx_f, vx_a, rows_f, rows_a, t_f, t_a;
};

// Launch shape; 0 = automatic.  Four steps per launch at every size (two were
// slower throughout).  Wide lanes on long segments recompute least, narrow
// lanes on short segments give the most waves: the lines are where the better
// one changed in microseconds per step, forward / adjoint, (cells per lane,
// rows): 164 x 164 x 1 shot (1, 4) 3.6 / 5.4, (1, 8) 3.8 / 6.7; 300 x 500 x 8
// (1, 8) 4.4 / 9.0, (1, 12) 4.7 / 8.8, (2, 8) 4.5 / 9.1; 900 x 2500 x 2 (1, 16)
// 7.6 / 14.4, (2, 16) 7.5 / 15.5; x 8 (4, 16) 23.6 and (2, 12) 57 of the adjoint
// against (4, 16) 60; x 64 (4, 32) 143 / 279, (2, 32) 156 / 284, (4, 16) 148 /
// 318.
// n cells of all shots, `wide` the widest lanes that divide the grid.
inline Plan make_plan(int64_t n, int wide, int32_t steps, int32_t vec_x, int32_t rows) {
  Plan p;
  p.t_f = p.t_a = steps ? steps : 4;
  if (n < 300000) { p.vx_f = p.vx_a = 1; p.rows_f = p.rows_a = 4; }
  else if (n < 3000000) { p.vx_f = p.vx_a = 1; p.rows_f = 8; p.rows_a = 12; }
  else if (n < 8000000) { p.vx_f = 2; p.vx_a = 1; p.rows_f = p.rows_a = 16; }
  else if (n < 40000000) { p.vx_f = 4; p.vx_a = 2; p.rows_f = p.rows_a = 16; }
  else { p.vx_f = p.vx_a = 4; p.rows_f = p.rows_a = 32; }
  p.vx_f = std::min(p.vx_f, wide);
  p.vx_a = std::min(p.vx_a, wide);
  if (vec_x) p.vx_f = p.vx_a = vec_x;
  if (rows) p.rows_f = p.rows_a = rows;
  return p;
}

}  // namespace
