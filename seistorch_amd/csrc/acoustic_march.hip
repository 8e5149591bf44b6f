// The acoustic loops on the marching kernels (march.h): T time steps per
// launch, records and adjoint sources through rows of the receivers' depths,
// rings and snapshots written and read by the launches themselves.
#include "common.h"
#include "march.h"
#include "seistorch_amd.h"
#include "tiles.h"

#include <algorithm>
#include <vector>

using seis::Grid;
using seis::TimeConsts;
using namespace seis::march;
using seis::tiles::kXcds;

namespace {

// c^2, A and B of the damped update, once per loop.
__global__ __launch_bounds__(256) void k_coefs(const float* __restrict__ vp,
                                               const float* __restrict__ d, int64_t plane,
                                               TimeConsts k, float* __restrict__ c2,
                                               float* __restrict__ A, float* __restrict__ Bc) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= plane) return;
  const float c = vp[i], dd = d[i];
  c2[i] = c * c;
  A[i] = 1.0f / (k.idt2 + dd * k.idt);
  Bc[i] = k.idt2 - dd * k.idt;
}

// row_slot[z] = 0 for every row that holds a receiver of any shot (-1 before).
__global__ __launch_bounds__(256) void k_mark_rows(const int64_t* __restrict__ rec, int64_t R,
                                                   int64_t plane, int nx,
                                                   int32_t* __restrict__ row_slot) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < R) row_slot[(rec[t] % plane) / nx] = 0;
}

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

// Work beside the march of one launch: the records of the previous launch's
// levels, or the adjoint sources of the next one's.
struct Gather {
  const float* rows;     // (levels, row_cells) of the previous launch
  const int64_t* cell;
  int64_t R, row_cells;
  float* rec;            // row of the first of those levels
  int levels, blocks;    // blocks of 256 threads, after the march's
};

struct Sources {
  float* rows;           // (levels, row_cells) of the next launch
  const int32_t *head, *next;
  int64_t R, row_cells;
  const float* rgrad;    // row of the first level; the next level's precedes it
  int levels, blocks;
};

__device__ __forceinline__ void gather_records(const Gather& ga, int block) {
  const int64_t n = ga.R * ga.levels;
  for (int64_t i = (int64_t)block * kThreads + threadIdx.x; i < n;
       i += (int64_t)ga.blocks * kThreads) {
    const int64_t lev = i / ga.R, t = i - lev * ga.R;
    ga.rec[i] = ga.rows[lev * ga.row_cells + ga.cell[t]];
  }
}

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

__global__ __launch_bounds__(kThreads) void k_gather(Gather ga) { gather_records(ga, blockIdx.x); }
__global__ __launch_bounds__(kThreads) void k_sources(Sources so) { fill_sources(so, blockIdx.x); }

// XCD-aware unit order, as tiles.h: each XCD takes a contiguous range.
__device__ __forceinline__ bool march_unit(const Split& sp, int B, int per, int& strip, int& seg,
                                           int& b) {
  const int w = blockIdx.x;
  const int64_t blk = (int64_t)(w % kXcds) * per + w / kXcds;
  const int64_t unit =
      blk * kWavesPerBlock + __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int64_t row = unit / sp.group, row2 = row / sp.strips;
  strip = (int)(row - row2 * sp.strips);
  seg = (int)(row2 % sp.segs);
  b = (int)(row2 / sp.segs) * sp.group + (int)(unit - row * sp.group);
  return b < B;
}

// The kernels take one struct, so that its constant-memory copy is at the
// start of the kernel's arguments.
struct FwdLaunch {
  FwdParams p;
  Gather ga;
  int per;
};

struct AdjLaunch {
  AdjParams p;
  Sources so;
  int per;
};

template <typename P>
__device__ __forceinline__ Const<P> launch_params() {
  return (Const<P>)__builtin_amdgcn_kernarg_segment_ptr();
}

template <int T, int VX>
__global__ __launch_bounds__(kThreads) void k_march_fwd(FwdLaunch a) {
  if ((int)blockIdx.x >= a.per * kXcds) {
    gather_records(a.ga, (int)blockIdx.x - a.per * kXcds);
    return;
  }
  int strip, seg, b;
  if (!march_unit(a.p.sp, a.p.B, a.per, strip, seg, b)) return;
  march_forward<T, VX>(a.p, launch_params<FwdParams>(), b, strip, seg);
}

template <int T, int VX>
__global__ __launch_bounds__(kThreads) void k_march_adj(AdjLaunch a) {
  if ((int)blockIdx.x >= a.per * kXcds) {
    fill_sources(a.so, (int)blockIdx.x - a.per * kXcds);
    return;
  }
  int strip, seg, b;
  if (!march_unit(a.p.sp, a.p.B, a.per, strip, seg, b)) return;
  march_adjoint<T, VX>(a.p, launch_params<AdjParams>(), b, strip, seg);
}

// grad = 2c * (sum over shots of the gradient planes) on the undamped
// interior, 0 elsewhere (and everywhere when nothing was accumulated).
__global__ __launch_bounds__(256) void k_march_grad(const float* __restrict__ vp,
                                                    const float* __restrict__ gpart, int n,
                                                    float* __restrict__ grad, Grid g) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.plane) return;
  const int z = (int)(i / g.nx), x = (int)(i - (int64_t)z * g.nx);
  float s = 0.0f;
  if (seis::interior(z, x, g))
    for (int b = 0; b < n; ++b) s += gpart[b * g.plane + i];
  grad[i] = 2.0f * vp[i] * s;
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

int zero(float* p, int64_t n, hipStream_t s) {
  k_zero<<<blocks_of(n), 256, 0, s>>>(p, n);
  SEIS_CHECK_LAUNCH();
  return 0;
}

// Shots whose waves run side by side on the same strips.  Eight share the
// coefficient rows in L2 while neighbouring segments still find each other's
// halo rows in the last-level cache: 64 shots of 900 x 2500, 10^9 cell updates
// per second of the adjoint with groups of 1 / 4 / 8 / 16 / 64: 335 / 393 /
// 399 / 375 / 343; of the forward 887 / 922 / 937 / 921 / 836.
constexpr int kShotGroup = 8;

#define SEIS_MARCH_CASES(F) \
  F(1, 1) F(1, 2) F(1, 4) F(2, 1) F(2, 2) F(2, 4) F(4, 1) F(4, 2) F(4, 4)

int launch_fwd(int T, int VX, const Coefs& cf, const FwdLevels& f, const int32_t* src, int B,
               const Grid& g, const TimeConsts& k, int rows, const Gather& ga, hipStream_t s) {
  const Split sp = make_split(g, T, VX, rows, std::min(B, kShotGroup));
  const int64_t units = (int64_t)sp.strips * sp.segs * sp.group * ((B + sp.group - 1) / sp.group);
  const int64_t blocks = (units + kWavesPerBlock - 1) / kWavesPerBlock;
  const int per = (int)((blocks + kXcds - 1) / kXcds);
  const unsigned grid = (unsigned)(per * kXcds + ga.blocks);
  const FwdLaunch a{{cf, f, src, B, sp, g, k}, ga, per};
  switch (T * 8 + VX) {
#define SEIS_F(T_, V_)                                                                      \
  case T_ * 8 + V_:                                                                         \
    k_march_fwd<T_, V_><<<grid, kThreads, 0, s>>>(a);                                       \
    break;
    SEIS_MARCH_CASES(SEIS_F)
#undef SEIS_F
    default:
      seis::set_error("unsupported march shape (%d steps, vec_x %d)", T, VX);
      return 1;
  }
  SEIS_CHECK_LAUNCH();
  return 0;
}

int launch_adj(int T, int VX, const Coefs& cf, const AdjLevels& f, const int32_t* src, int B,
               const Grid& g, const TimeConsts& k, int rows, bool rebuild_last, const Sources& so,
               hipStream_t s) {
  const Split sp = make_split(g, T, VX, rows, std::min(B, kShotGroup));
  const int64_t units = (int64_t)sp.strips * sp.segs * sp.group * ((B + sp.group - 1) / sp.group);
  const int64_t blocks = (units + kWavesPerBlock - 1) / kWavesPerBlock;
  const int per = (int)((blocks + kXcds - 1) / kXcds);
  const unsigned grid = (unsigned)(per * kXcds + so.blocks);
  const AdjLaunch a{{cf, f, src, B, sp, g, k, rebuild_last}, so, per};
  switch (T * 8 + VX) {
#define SEIS_F(T_, V_)                                                                      \
  case T_ * 8 + V_:                                                                         \
    k_march_adj<T_, V_><<<grid, kThreads, 0, s>>>(a);                                       \
    break;
    SEIS_MARCH_CASES(SEIS_F)
#undef SEIS_F
    default:
      seis::set_error("unsupported march shape (%d steps, vec_x %d)", T, VX);
      return 1;
  }
  SEIS_CHECK_LAUNCH();
  return 0;
}

constexpr int kMaxT = kMaxSteps;
// ring floats of one time level: those of a launch's levels are one buffer,
// whose offsets stay below kRowOut bytes
constexpr int64_t kMaxRing = (int64_t)1 << 25;

// Steps of the next launch when `left` remain to the next boundary: the
// remainder first, so that the launch that ends at the boundary takes at
// least two steps (and can write both fields of a snapshot) unless left == 1.
inline int next_steps(int64_t left, int max_t) {
  const int64_t r = left % max_t;
  if (r == 0) return max_t;
  return r >= 2 ? 2 : 1;
}

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
Plan make_plan(int64_t B, int64_t nz, int64_t nx, int32_t steps, int32_t vec_x, int32_t rows) {
  Plan p;
  p.t_f = p.t_a = steps ? steps : 4;
  const int64_t n = B * nz * nx;
  const int wide = nx % 4 == 0 ? 4 : nx % 2 == 0 ? 2 : 1;
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

inline int64_t pad64(int64_t n) { return (n + 63) / 64 * 64; }

// Workspace (in floats): coefficient planes, two sets of receiver rows, the
// receivers' cells (forward) or chains (adjoint).
struct Work {
  float *c2, *A, *Bc, *rows[2];
  int64_t* cell;
  int32_t *head, *next;
  int64_t row_cells, total;
};

Work carve(float* base, int64_t B, int64_t nz, int64_t nx, int64_t slots, int64_t R,
           bool adjoint) {
  Work w;
  const int64_t plane = pad64(nz * nx);
  w.row_cells = slots * B * nx;
  const int64_t rows = pad64(kMaxT * w.row_cells);
  int64_t o = 0;
  auto take = [&](int64_t n) { const int64_t at = o; o += pad64(n); return base + at; };
  w.c2 = take(plane); w.A = take(plane); w.Bc = take(plane);
  w.rows[0] = take(rows); w.rows[1] = take(rows);
  w.cell = nullptr; w.head = w.next = nullptr;
  if (adjoint) {
    w.head = reinterpret_cast<int32_t*>(take(w.row_cells));
    w.next = reinterpret_cast<int32_t*>(take(R));
  } else {
    w.cell = reinterpret_cast<int64_t*>(take(2 * R));
  }
  w.total = o;
  return w;
}

int aux_blocks(int64_t n) { return (int)std::min<int64_t>((n + kThreads - 1) / kThreads, 512); }

int check_march(int64_t B, int64_t nz, int64_t nx, float dt, float h, int64_t nt, int64_t R,
                int32_t npml, int32_t slots, const int32_t* row_slot, int32_t steps,
                int32_t vec_x, int32_t rows) {
  SEIS_CHECK_ARG(B >= 1 && B <= 65535, "batch size %lld outside [1, 65535]", (long long)B);
  SEIS_CHECK_ARG(nz >= 1 && nx >= 1 && nz * nx <= kMaxCells, "grid %lld x %lld too large",
                 (long long)nz, (long long)nx);
  SEIS_CHECK_ARG(dt > 0.0f && h > 0.0f, "dt and h must be positive (dt=%g, h=%g)", dt, h);
  SEIS_CHECK_ARG(nt >= 1 && R >= 0 && R < (int64_t)1 << 31, "nt %lld, R %lld", (long long)nt,
                 (long long)R);
  SEIS_CHECK_ARG(npml >= 0, "npml %d", npml);
  SEIS_CHECK_ARG(slots >= 0 && slots <= nz && (R == 0 || (slots > 0 && row_slot)),
                 "receivers need their rows (slots %d)", slots);
  SEIS_CHECK_ARG(steps == 0 || steps == 1 || steps == 2 || steps == 4, "steps %d not 1, 2 or 4",
                 steps);
  SEIS_CHECK_ARG(vec_x == 0 || vec_x == 1 || vec_x == 2 || vec_x == 4, "vec_x %d not 1, 2 or 4",
                 vec_x);
  SEIS_CHECK_ARG(vec_x == 0 || nx % vec_x == 0, "vec_x %d does not divide nx = %lld", vec_x,
                 (long long)nx);
  SEIS_CHECK_ARG(rows >= 0 && rows <= 1 << 20, "rows %d", rows);
  SEIS_CHECK_ARG(B * 2 * (nz + nx) <= kMaxRing, "too many shots for the ring (%lld)",
                 (long long)B);
  return 0;
}

}  // namespace

extern "C" {

int seis_receiver_rows(const int64_t* rec_flat, int64_t R, int64_t nz, int64_t nx,
                       int32_t* row_slot, void* stream) {
  SEIS_CHECK_ARG(row_slot && (R == 0 || rec_flat) && R >= 0, "bad arguments");
  SEIS_CHECK_ARG(nz >= 1 && nx >= 1 && nz * nx < (int64_t)1 << 31, "grid %lld x %lld",
                 (long long)nz, (long long)nx);
  hipStream_t s = (hipStream_t)stream;
  k_fill_i32<<<blocks_of(nz), 256, 0, s>>>(row_slot, nz, -1);
  SEIS_CHECK_LAUNCH();
  if (R > 0) {
    k_mark_rows<<<blocks_of(R), 256, 0, s>>>(rec_flat, R, nz * nx, (int)nx, row_slot);
    SEIS_CHECK_LAUNCH();
  }
  k_number_rows<<<1, 64, 0, s>>>(row_slot, (int)nz);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int64_t seis_acoustic_march_workspace(int64_t B, int64_t nz, int64_t nx, int32_t slots, int64_t R,
                                      int32_t adjoint) {
  return carve(nullptr, B, nz, nx, slots, R, adjoint != 0).total;
}

int seis_acoustic_march_forward(const float* vp, const float* d, const float* wavelet, int64_t nt,
                                const int32_t* src_zx, const int64_t* rec_flat, int64_t R,
                                const int32_t* row_slot, int32_t slots, float* rec_out,
                                float* ring, float* snaps, int32_t snap_every, float* work,
                                float* const* fields, int32_t* final_fields, int64_t B, int64_t nz,
                                int64_t nx, float dt, float h, int32_t npml, int32_t multiple,
                                int32_t steps, int32_t vec_x, int32_t rows, void* stream) {
  if (int e = check_march(B, nz, nx, dt, h, nt, R, npml, slots, row_slot, steps, vec_x, rows))
    return e;
  SEIS_CHECK_ARG(vp && d && wavelet && src_zx && work && fields && final_fields,
                 "null pointer argument");
  SEIS_CHECK_ARG(R == 0 || (rec_flat && rec_out), "bad receiver arguments");
  for (int i = 0; i < 4; ++i) {
    SEIS_CHECK_ARG(fields[i], "null field buffer");
    for (int j = 0; j < i; ++j)
      SEIS_CHECK_ARG(fields[i] != fields[j], "the four field buffers must be distinct");
  }
  SEIS_CHECK_ARG(!snaps || snap_every > 0, "snapshots need snap_every > 0");
  const int64_t ring_len = ring ? seis_ring_len(nz, nx, npml, multiple) : 0;
  SEIS_CHECK_ARG(!ring || ring_len > 0, "grid %lld x %lld has no interior inside npml=%d",
                 (long long)nz, (long long)nx, npml);
  const Grid g = seis::make_grid(nz, nx, npml, multiple != 0);
  const TimeConsts k = seis::make_consts(dt, h);
  const Plan p = make_plan(B, nz, nx, steps, vec_x, rows);
  const Work w = carve(work, B, nz, nx, slots, R, false);
  hipStream_t s = (hipStream_t)stream;
  const int64_t field = B * g.plane;
  k_coefs<<<blocks_of(g.plane), 256, 0, s>>>(vp, d, g.plane, k, w.c2, w.A, w.Bc);
  SEIS_CHECK_LAUNCH();
  if (R > 0) {
    k_row_cells<<<blocks_of(R), 256, 0, s>>>(rec_flat, R, g.plane, g.nx, (int)B, row_slot, w.cell,
                                             nullptr, nullptr);
    SEIS_CHECK_LAUNCH();
  }
  const Coefs cf{w.c2, w.A, w.Bc};
  // cur = u^n, prev = u^{n-1}; either may be a snapshot's slot, then its
  // buffer joins the free ones
  float* cur = fields[0];
  float* prev = fields[1];
  std::vector<float*> free_bufs{fields[2], fields[3]};
  auto is_buf = [&](float* q) {
    return q == fields[0] || q == fields[1] || q == fields[2] || q == fields[3];
  };
  auto take = [&]() { float* q = free_bufs.back(); free_bufs.pop_back(); return q; };
  if (int e = zero(cur, field, s)) return e;
  if (int e = zero(prev, field, s)) return e;
  const int64_t last_snap = snaps ? seis_snapshot_count(nt, snap_every) * snap_every : 0;
  Gather ga{nullptr, w.cell, R, w.row_cells, nullptr, 0, 0};
  int parity = 0;
  int64_t n = 0;
  while (n < nt) {
    // launches end where a snapshot pair (u^m, u^{m+1}) is the newest pair
    int64_t stop = nt, m = 0;
    if (last_snap > 0 && n <= last_snap) {
      m = std::max<int64_t>(1, (n - 1 + snap_every) / snap_every) * snap_every;
      stop = m + 1;
    }
    const int T = next_steps(stop - n, p.t_f);
    const bool snap = m > 0 && n + T == stop;
    float* slot = snap ? snaps + (m / snap_every - 1) * 2 * field : nullptr;
    FwdLevels f{};
    f.u = cur; f.up = prev;
    f.o1 = snap ? slot + field : take();
    f.o0 = T == 1 ? nullptr : (snap ? slot : take());
    f.w = wavelet + n;
    f.ring_levels = ring ? (int)std::min<int64_t>(T, nt - 1 - n) : 0;
    f.ring = f.ring_levels > 0 ? ring + n * B * ring_len : nullptr;
    f.ring_len = ring_len;
    f.ring_step = B * ring_len;
    f.rows = R > 0 ? w.rows[parity] : nullptr;
    f.row_slot = row_slot;
    f.slots = slots;
    SEIS_PROF(SEIS_KERNEL_ACOUSTIC_MARCH_FWD, s);
    if (int e = launch_fwd(T, p.vx_f, cf, f, src_zx, (int)B, g, k, p.rows_f, ga, s)) return e;
    SEIS_PROF(SEIS_KERNEL_ACOUSTIC_MARCH_FWD, s);
    if (T == 1 && snap) {  // u^m was not written by this launch
      k_copy<<<blocks_of(field), 256, 0, s>>>(cur, slot, field);
      SEIS_CHECK_LAUNCH();
    }
    if (is_buf(prev)) free_bufs.push_back(prev);
    if (T == 1) {
      prev = cur;
    } else {
      if (is_buf(cur)) free_bufs.push_back(cur);
      prev = f.o0;
    }
    cur = f.o1;
    if (R > 0) {
      ga.rows = w.rows[parity];
      ga.rec = rec_out + n * R;
      ga.levels = T;
      ga.blocks = aux_blocks(R * T);
      parity ^= 1;
    }
    n += T;
  }
  if (ga.blocks > 0) {
    k_gather<<<ga.blocks, kThreads, 0, s>>>(ga);
    SEIS_CHECK_LAUNCH();
  }
  // the last pair is never a snapshot's (m <= nt - 2), except u^{nt-1} when
  // one step follows the last snapshot: then it goes to a buffer of its own
  if (!is_buf(prev)) {
    float* q = take();
    k_copy<<<blocks_of(field), 256, 0, s>>>(prev, q, field);
    SEIS_CHECK_LAUNCH();
    prev = q;
  }
  for (int i = 0; i < 4; ++i) {
    if (fields[i] == cur) final_fields[0] = i;
    if (fields[i] == prev) final_fields[1] = i;
  }
  return 0;
}

int seis_acoustic_march_backward(const float* vp, const float* d, const float* wavelet, int64_t nt,
                                 const int32_t* src_zx, const int64_t* rec_flat, int64_t R,
                                 const int32_t* row_slot, int32_t slots, const float* rec_grad,
                                 const float* ring, const float* snaps, int32_t snap_every,
                                 float* work, float* const* u, float* const* mu, float* grad_part,
                                 float* grad, int64_t B, int64_t nz, int64_t nx, float dt, float h,
                                 int32_t npml, int32_t multiple, int32_t steps, int32_t vec_x,
                                 int32_t rows, void* stream) {
  if (int e = check_march(B, nz, nx, dt, h, nt, R, npml, slots, row_slot, steps, vec_x, rows))
    return e;
  SEIS_CHECK_ARG(vp && d && wavelet && src_zx && work && u && mu && grad_part && grad,
                 "null pointer argument");
  SEIS_CHECK_ARG(R == 0 || (rec_flat && rec_grad), "bad receiver arguments");
  for (int i = 0; i < 4; ++i) {
    SEIS_CHECK_ARG(u[i] && mu[i], "null field buffer");
    for (int j = 0; j < i; ++j)
      SEIS_CHECK_ARG(u[i] != u[j] && mu[i] != mu[j], "the field buffers must be distinct");
  }
  const int64_t ring_len = seis_ring_len(nz, nx, npml, multiple);
  SEIS_CHECK_ARG(ring_len > 0, "grid %lld x %lld has no interior inside npml=%d", (long long)nz,
                 (long long)nx, npml);
  SEIS_CHECK_ARG(nx - 2 * npml - 1 >= 4 && nz - (multiple ? 1 : 2) * npml - 1 >= kMaxT,
                 "interior of %lld x %lld too small", (long long)nz, (long long)nx);
  SEIS_CHECK_ARG(ring || nt <= 2, "ring storage is required for nt > 2");
  SEIS_CHECK_ARG(!snaps || snap_every > 0, "snapshots need snap_every > 0");
  const Grid g = seis::make_grid(nz, nx, npml, multiple != 0);
  const TimeConsts k = seis::make_consts(dt, h);
  const Plan p = make_plan(B, nz, nx, steps, vec_x, rows);
  const Work w = carve(work, B, nz, nx, slots, R, true);
  hipStream_t s = (hipStream_t)stream;
  const int64_t field = B * g.plane;
  k_coefs<<<blocks_of(g.plane), 256, 0, s>>>(vp, d, g.plane, k, w.c2, w.A, w.Bc);
  SEIS_CHECK_LAUNCH();
  if (R > 0) {
    k_fill_i32<<<blocks_of(w.row_cells), 256, 0, s>>>(w.head, w.row_cells, -1);
    SEIS_CHECK_LAUNCH();
    k_row_cells<<<blocks_of(R), 256, 0, s>>>(rec_flat, R, g.plane, g.nx, (int)B, row_slot, nullptr,
                                             w.head, w.next);
    SEIS_CHECK_LAUNCH();
  }
  const Coefs cf{w.c2, w.A, w.Bc};
  if (int e = zero(mu[0], field, s)) return e;
  if (int e = zero(mu[1], field, s)) return e;
  const float* X = u[1];  // u^{k-1}
  const float* Y = u[0];  // u^k
  const float* M1 = mu[0];
  const float* M2 = mu[1];
  std::vector<float*> ufree{u[2], u[3]}, mfree{mu[2], mu[3]};
  auto owned = [](float* const* set, const float* q) -> float* {
    for (int i = 0; i < 4; ++i)
      if (set[i] == q) return set[i];
    return nullptr;
  };
  auto take = [](std::vector<float*>& v) { float* q = v.back(); v.pop_back(); return q; };
  auto release = [&](std::vector<float*>& v, float* const* set, const float* q) {
    if (float* o = owned(set, q)) v.push_back(o);
  };
  const int64_t last_snap = snaps ? seis_snapshot_count(nt, snap_every) * snap_every : 0;
  // launches end where the next pair comes from a snapshot: after iteration
  // k = m + 2 the fields (u^{m+1}, u^m) are taken from storage.  Iteration 1
  // adds nothing (u^0 = 0) and its mu is not read, so the loop ends at k = 2.
  auto steps_at = [&](int64_t kk, int64_t& m) -> int {
    int64_t left = kk - 1;
    m = 0;
    if (last_snap > 0 && kk >= snap_every + 2) {
      m = std::min(last_snap, (kk - 2) / snap_every * snap_every);
      left = kk - 2 - m + 1;
    }
    return next_steps(left, p.t_a);
  };
  auto sources = [&](int64_t kk, int T, float* out) {
    return Sources{out, w.head, w.next, R, w.row_cells, rec_grad + (kk - 1) * R, T,
                   aux_blocks(w.row_cells)};
  };
  int parity = 0;
  int64_t kk = nt;
  bool first = true;
  if (kk >= 2 && R > 0) {
    int64_t m;
    const int T = steps_at(kk, m);
    const Sources so = sources(kk, T, w.rows[0]);
    k_sources<<<so.blocks, kThreads, 0, s>>>(so);
    SEIS_CHECK_LAUNCH();
  }
  while (kk >= 2) {
    int64_t m, m2;
    const int T = steps_at(kk, m);
    const int64_t kn = kk - T;
    Sources so{};
    if (R > 0 && kn >= 2) so = sources(kn, steps_at(kn, m2), w.rows[parity ^ 1]);
    AdjLevels f{};
    f.x = X; f.y = Y; f.m1 = M1; f.m2 = M2;
    f.ox = take(ufree);
    f.om1 = take(mfree);
    f.oy = T > 1 ? take(ufree) : nullptr;
    f.om2 = T > 1 ? take(mfree) : nullptr;
    f.gpart = grad_part;
    f.first = first;
    f.w = wavelet + (kk - 1);
    f.ring = ring ? ring + (kk - 3) * B * ring_len : nullptr;
    f.ring_len = ring_len;
    f.ring_step = B * ring_len;
    f.rows = R > 0 ? w.rows[parity] : nullptr;
    f.row_slot = row_slot;
    f.slots = slots;
    SEIS_PROF(SEIS_KERNEL_ACOUSTIC_MARCH_ADJ, s);
    if (int e = launch_adj(T, p.vx_a, cf, f, src_zx, (int)B, g, k, p.rows_a, kn + 1 >= 3, so, s))
      return e;
    SEIS_PROF(SEIS_KERNEL_ACOUSTIC_MARCH_ADJ, s);
    first = false;
    release(ufree, u, Y);
    release(mfree, mu, M2);
    if (T > 1) {
      release(ufree, u, X);
      release(mfree, mu, M1);
      Y = f.oy; M2 = f.om2;
    } else {
      Y = X; M2 = M1;
    }
    X = f.ox;
    M1 = f.om1;
    kk = kn;
    parity ^= 1;
    if (m > 0 && kk == m + 1) {  // (u^{k-1}, u^k) = (u^m, u^{m+1}) from storage
      release(ufree, u, X);
      release(ufree, u, Y);
      const float* slot = snaps + (m / snap_every - 1) * 2 * field;
      X = slot;
      Y = slot + field;
    }
  }
  k_march_grad<<<blocks_of(g.plane), 256, 0, s>>>(vp, grad_part, first ? 0 : (int)B, grad, g);
  SEIS_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
