// The acoustic loops on the marching kernels (march.h): T time steps per
// launch, records and adjoint sources through rows of the receivers' depths,
// rings and snapshots written and read by the launches themselves.
#include "common.h"
#include "march.h"
#include "march_rows.h"
#include "seistorch_amd.h"
#include "tiles.h"

#include <algorithm>
#include <vector>

using seis::Grid;
using seis::TimeConsts;
using namespace seis::march;
using seis::tiles::kXcds;

namespace {

// row_slot[z] = 0 for every row that holds a receiver of any shot (-1 before).
__global__ __launch_bounds__(256) void k_mark_rows(const int64_t* __restrict__ rec, int64_t R,
                                                   int64_t plane, int nx,
                                                   int32_t* __restrict__ row_slot) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < R) row_slot[(rec[t] % plane) / nx] = 0;
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

__device__ __forceinline__ void gather_records(const Gather& ga, int block) {
  const int64_t n = ga.R * ga.levels;
  for (int64_t i = (int64_t)block * kThreads + threadIdx.x; i < n;
       i += (int64_t)ga.blocks * kThreads) {
    const int64_t lev = i / ga.R, t = i - lev * ga.R;
    ga.rec[i] = ga.rows[lev * ga.row_cells + ga.cell[t]];
  }
}

__global__ __launch_bounds__(kThreads) void k_gather(Gather ga) { gather_records(ga, blockIdx.x); }
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

template <int T, int VX>
__global__ __launch_bounds__(kThreads) void k_march_fwd(FwdLaunch a) {
  if ((int)blockIdx.x >= a.per * kXcds) {
    gather_records(a.ga, (int)blockIdx.x - a.per * kXcds);
    return;
  }
  int strip, seg, b;
  if (!march_unit(a.p.sp, a.p.B, xcd_block(a.per), strip, seg, b)) return;
  march_forward<T, VX>(a.p, launch_params<FwdParams>(), b, strip, seg);
}

template <int T, int VX>
__global__ __launch_bounds__(kThreads) void k_march_adj(AdjLaunch a) {
  if ((int)blockIdx.x >= a.per * kXcds) {
    fill_sources(a.so, (int)blockIdx.x - a.per * kXcds);
    return;
  }
  int strip, seg, b;
  if (!march_unit(a.p.sp, a.p.B, xcd_block(a.per), strip, seg, b)) return;
  march_adjoint<T, VX>(a.p, launch_params<AdjParams>(), b, strip, seg);
}

// Several problems in one launch: a table of their parameters in device
// memory, blocks numbered through all of them.
struct FwdItem {
  FwdParams p;
  Gather aux;
  int T, block0, aux0;  // steps of this launch (0: records only), first blocks
};

struct AdjItem {
  AdjParams p;
  Sources aux;
  int T, block0, aux0;
};

template <typename Item>
struct BatchLaunch {
  const Item* items;
  int n, blocks, per, aux_blocks;
};

// The last item whose first block (march or auxiliary) is at most blk: items
// without blocks of the kind start where the next one does.
template <typename Item>
__device__ __forceinline__ Const<Item> find_item(const BatchLaunch<Item>& a, int blk, bool aux) {
  const Const<Item> c = (Const<Item>)a.items;
  int lo = 0, hi = a.n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if ((aux ? c[mid].aux0 : c[mid].block0) <= blk) lo = mid;
    else hi = mid - 1;
  }
  return c + lo;
}

template <typename V>
__device__ __forceinline__ V read_const(Const<V> c) {
  V v;
  __builtin_memcpy(&v, (const V*)c, sizeof(V));
  return v;
}

template <int VX>
__global__ __launch_bounds__(kThreads) void k_march_fwd_batch(BatchLaunch<FwdItem> a) {
  if ((int)blockIdx.x >= a.per * kXcds) {
    const int blk = (int)blockIdx.x - a.per * kXcds;
    const Const<FwdItem> it = find_item(a, blk, true);
    gather_records(read_const(&it->aux), blk - it->aux0);
    return;
  }
  const int blk = xcd_block(a.per);
  if (blk >= a.blocks) return;
  const Const<FwdItem> it = find_item(a, blk, false);
  const FwdParams p = read_const(&it->p);
  int strip, seg, b;
  if (!march_unit(p.sp, p.B, blk - it->block0, strip, seg, b)) return;
  switch (it->T) {
    case 4: march_forward<4, VX>(p, &it->p, b, strip, seg); break;
    case 2: march_forward<2, VX>(p, &it->p, b, strip, seg); break;
    default: march_forward<1, VX>(p, &it->p, b, strip, seg); break;
  }
}

template <int VX>
__global__ __launch_bounds__(kThreads) void k_march_adj_batch(BatchLaunch<AdjItem> a) {
  if ((int)blockIdx.x >= a.per * kXcds) {
    const int blk = (int)blockIdx.x - a.per * kXcds;
    const Const<AdjItem> it = find_item(a, blk, true);
    fill_sources(read_const(&it->aux), blk - it->aux0);
    return;
  }
  const int blk = xcd_block(a.per);
  if (blk >= a.blocks) return;
  const Const<AdjItem> it = find_item(a, blk, false);
  const AdjParams p = read_const(&it->p);
  int strip, seg, b;
  if (!march_unit(p.sp, p.B, blk - it->block0, strip, seg, b)) return;
  switch (it->T) {
    case 4: march_adjoint<4, VX>(p, &it->p, b, strip, seg); break;
    case 2: march_adjoint<2, VX>(p, &it->p, b, strip, seg); break;
    default: march_adjoint<1, VX>(p, &it->p, b, strip, seg); break;
  }
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

// ring floats of one time level: those of a launch's levels are one buffer,
// whose offsets stay below kRowOut bytes
constexpr int64_t kMaxRing = (int64_t)1 << 25;

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

// A lane (of up to four cells) may hold one of the ring's columns only.
int check_ring(int64_t nz, int64_t nx, int32_t npml, int64_t ring_len) {
  SEIS_CHECK_ARG(ring_len > 0, "grid %lld x %lld has no interior inside npml=%d", (long long)nz,
                 (long long)nx, npml);
  SEIS_CHECK_ARG(nx - 2 * npml - 1 >= 4, "interior of %lld x %lld too small", (long long)nz,
                 (long long)nx);
  return 0;
}

// One problem's operands.
struct Problem {
  const float *vp, *d, *wavelet;
  int64_t nt;
  const int32_t* src;
  const int64_t* rec_flat;
  int64_t R;
  const int32_t* row_slot;
  int slots;
  int64_t B;
  Grid g;
  TimeConsts k;
  int64_t ring_len;
  float* snaps;
  int32_t snap_every;
  Work w;

  int64_t field() const { return B * g.plane; }
  int64_t last_snap() const {
    return snaps ? seis_snapshot_count(nt, snap_every) * snap_every : 0;
  }
  Coefs coefs() const { return {w.c2, w.A, w.Bc}; }
};

// The forward loop of a problem, launch by launch.
struct FwdRun {
  Problem p;
  float* ring;
  float* rec;
  float* fields[4];
  // cur = u^n, prev = u^{n-1}; either may be a snapshot's slot, then its
  // buffer joins the free ones
  float *cur, *prev;
  std::vector<float*> free_bufs;
  int64_t n = 0;
  int parity = 0;
  Gather ga;  // records of the previous launch's levels

  FwdRun(const Problem& q, float* ring_, float* rec_, float* const* f)
      : p(q), ring(ring_), rec(rec_), fields{f[0], f[1], f[2], f[3]}, cur(f[0]), prev(f[1]),
        free_bufs{f[2], f[3]}, ga{nullptr, q.w.cell, q.R, q.w.row_cells, nullptr, 0, 0} {}

  bool is_buf(const float* q) const {
    return q == fields[0] || q == fields[1] || q == fields[2] || q == fields[3];
  }
  float* take() {
    float* q = free_bufs.back();
    free_bufs.pop_back();
    return q;
  }
  bool done() const { return n >= p.nt; }

  // The next launch: its steps and levels; to (if any) receives a copy of from
  // after it.
  int next(int max_t, FwdLevels& f, const float*& from, float*& to) {
    // launches end where a snapshot pair (u^m, u^{m+1}) is the newest pair
    int64_t stop = p.nt, m = 0;
    const int64_t last_snap = p.last_snap(), K = p.snap_every;
    if (last_snap > 0 && n <= last_snap) {
      m = std::max<int64_t>(1, (n - 1 + K) / K) * K;
      stop = m + 1;
    }
    const int T = next_steps(stop - n, max_t);
    const bool snap = m > 0 && n + T == stop;
    float* slot = snap ? p.snaps + (m / K - 1) * 2 * p.field() : nullptr;
    f = FwdLevels{};
    f.u = cur; f.up = prev;
    f.o1 = snap ? slot + p.field() : take();
    f.o0 = T == 1 ? nullptr : (snap ? slot : take());
    f.w = p.wavelet + n;
    f.ring_levels = ring ? (int)std::min<int64_t>(T, p.nt - 1 - n) : 0;
    f.ring = f.ring_levels > 0 ? ring + n * p.B * p.ring_len : nullptr;
    f.ring_len = p.ring_len;
    f.ring_step = p.B * p.ring_len;
    f.rows = p.R > 0 ? p.w.rows[parity] : nullptr;
    f.row_slot = p.row_slot;
    f.slots = p.slots;
    from = T == 1 ? cur : nullptr;  // u^m was not written by this launch
    to = T == 1 && snap ? slot : nullptr;
    if (is_buf(prev)) free_bufs.push_back(prev);
    if (T == 1) {
      prev = cur;
    } else {
      if (is_buf(cur)) free_bufs.push_back(cur);
      prev = f.o0;
    }
    cur = f.o1;
    return T;
  }

  // After the launch of T steps: what the next one gathers.
  void advance(int T) {
    if (p.R > 0) {
      ga.rows = p.w.rows[parity];
      ga.rec = rec + n * p.R;
      ga.levels = T;
      ga.blocks = aux_blocks(p.R * T);
      parity ^= 1;
    }
    n += T;
  }

  // The last pair is never a snapshot's (m <= nt - 2), except u^{nt-1} when
  // one step follows the last snapshot: then it is copied to a free buffer.
  bool finish(const float*& from, float*& to) {
    if (is_buf(prev)) return false;
    from = prev;
    to = prev = take();
    return true;
  }

  void final_fields(int32_t* o) const {
    for (int i = 0; i < 4; ++i) {
      if (fields[i] == cur) o[0] = i;
      if (fields[i] == prev) o[1] = i;
    }
  }
};

// The adjoint loop of a problem, launch by launch.  Launches end where the
// next pair comes from a snapshot: after iteration k = m + 2 the fields
// (u^{m+1}, u^m) are taken from storage.  Iteration 1 adds nothing (u^0 = 0)
// and its mu is not read, so the loop ends at k = 2.
struct AdjRun {
  Problem p;
  const float* ring;
  const float* rgrad;
  float *u[4], *mu[4], *gpart;
  const float *X, *Y, *M1, *M2;  // u^{k-1}, u^k, mu^{k+1}, mu^{k+2}
  std::vector<float*> ufree, mfree;
  int64_t kk;
  int parity = 0;
  bool first = true;

  AdjRun(const Problem& q, const float* ring_, const float* rgrad_, float* const* u_,
         float* const* mu_, float* gpart_)
      : p(q), ring(ring_), rgrad(rgrad_), u{u_[0], u_[1], u_[2], u_[3]},
        mu{mu_[0], mu_[1], mu_[2], mu_[3]}, gpart(gpart_), X(u_[1]), Y(u_[0]), M1(mu_[0]),
        M2(mu_[1]), ufree{u_[2], u_[3]}, mfree{mu_[2], mu_[3]}, kk(q.nt) {}

  static void release(std::vector<float*>& v, float* const (&set)[4], const float* q) {
    for (int i = 0; i < 4; ++i)
      if (set[i] == q) v.push_back(set[i]);
  }
  static float* take(std::vector<float*>& v) {
    float* q = v.back();
    v.pop_back();
    return q;
  }
  bool done() const { return kk < 2; }

  int steps_at(int64_t k, int max_t, int64_t& m) const {
    int64_t left = k - 1;
    const int64_t last_snap = p.last_snap(), K = p.snap_every;
    m = 0;
    if (last_snap > 0 && k >= K + 2) {
      m = std::min(last_snap, (k - 2) / K * K);
      left = k - 2 - m + 1;
    }
    return next_steps(left, max_t);
  }

  // Adjoint sources of the launch that begins at iteration k (none: no blocks).
  Sources sources(int64_t k, int max_t, int set) const {
    Sources so{};
    int64_t m;
    if (p.R > 0 && k >= 2)
      so = Sources{p.w.rows[set], p.w.head, p.w.next, p.R, p.w.row_cells, rgrad + (k - 1) * p.R,
                   steps_at(k, max_t, m), aux_blocks(p.w.row_cells)};
    return so;
  }

  // The next launch, and the sources it prepares for the one after it.
  int next(int max_t, AdjLevels& f, Sources& so, bool& rebuild_last) {
    int64_t m;
    const int T = steps_at(kk, max_t, m);
    const int64_t kn = kk - T;
    so = sources(kn, max_t, parity ^ 1);
    f = AdjLevels{};
    f.x = X; f.y = Y; f.m1 = M1; f.m2 = M2;
    f.ox = take(ufree);
    f.om1 = take(mfree);
    f.oy = T > 1 ? take(ufree) : nullptr;
    f.om2 = T > 1 ? take(mfree) : nullptr;
    f.gpart = gpart;
    f.first = first;
    f.w = p.wavelet + (kk - 1);
    f.ring = ring ? ring + (kk - 3) * p.B * p.ring_len : nullptr;
    f.ring_len = p.ring_len;
    f.ring_step = p.B * p.ring_len;
    f.rows = p.R > 0 ? p.w.rows[parity] : nullptr;
    f.row_slot = p.row_slot;
    f.slots = p.slots;
    rebuild_last = kn + 1 >= 3;
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
      const float* slot = p.snaps + (m / p.snap_every - 1) * 2 * p.field();
      X = slot;
      Y = slot + p.field();
    }
    return T;
  }
};

int copy(const float* a, float* b, int64_t n, hipStream_t s) {
  k_copy<<<blocks_of(n), 256, 0, s>>>(a, b, n);
  SEIS_CHECK_LAUNCH();
  return 0;
}

// The coefficient planes and the receivers' cells (forward) or chains.
int prepare(const Problem& p, bool adjoint, hipStream_t s) {
  k_coefs<<<blocks_of(p.g.plane), 256, 0, s>>>(p.vp, p.d, p.g.plane, p.k, p.w.c2, p.w.A, p.w.Bc);
  SEIS_CHECK_LAUNCH();
  if (p.R == 0) return 0;
  if (adjoint) {
    k_fill_i32<<<blocks_of(p.w.row_cells), 256, 0, s>>>(p.w.head, p.w.row_cells, -1);
    SEIS_CHECK_LAUNCH();
  }
  k_row_cells<<<blocks_of(p.R), 256, 0, s>>>(p.rec_flat, p.R, p.g.plane, p.g.nx, (int)p.B,
                                             p.row_slot, p.w.cell, p.w.head, p.w.next);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int final_grad(const AdjRun& r, float* grad, hipStream_t s) {
  k_march_grad<<<blocks_of(r.p.g.plane), 256, 0, s>>>(r.p.vp, r.gpart, r.first ? 0 : (int)r.p.B,
                                                      grad, r.p.g);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int check_adjoint(int64_t nz, int64_t nx, int64_t nt, int32_t npml, int32_t multiple,
                  int64_t ring_len, const float* ring) {
  if (int e = check_ring(nz, nx, npml, ring_len)) return e;
  SEIS_CHECK_ARG(nz - (multiple ? 1 : 2) * npml - 1 >= kMaxT,
                 "interior of %lld x %lld too small", (long long)nz, (long long)nx);
  SEIS_CHECK_ARG(ring || nt <= 2, "ring storage is required for nt > 2");
  return 0;
}

int check_fields(float* const* f) {
  for (int i = 0; i < 4; ++i) {
    SEIS_CHECK_ARG(f[i], "null field buffer");
    for (int j = 0; j < i; ++j)
      SEIS_CHECK_ARG(f[i] != f[j], "the four field buffers must be distinct");
  }
  return 0;
}

// ---- batches

// Launches of a batch: items [first, first + n) of the table, and copies after.
struct Round {
  size_t first;
  int n, blocks, aux_blocks, vx;
};

struct CopyAfter {
  size_t round;
  const float* from;
  float* to;
  int64_t n;
};

// An upper bound of one problem's launches: every stretch between two
// snapshots takes its remainder in at most two, and one or two more carry the
// first sources or the last records.
int64_t max_items(int64_t nt, int32_t snap_every) {
  return nt / kMaxT + 2 * (seis_snapshot_count(nt, snap_every) + 1) + 3;
}

template <typename Item>
void add_item(std::vector<Item>& items, Round& r, Item it, int64_t blocks) {
  it.block0 = r.blocks;
  it.aux0 = r.aux_blocks;
  r.blocks += (int)blocks;
  r.aux_blocks += it.aux.blocks;
  ++r.n;
  items.push_back(it);
}

template <typename Item, typename K>
int launch_round(K k, const Item* table, const Round& r, hipStream_t s) {
  const int per = (r.blocks + kXcds - 1) / kXcds;
  const BatchLaunch<Item> a{table + r.first, r.n, r.blocks, per, r.aux_blocks};
  const unsigned grid = (unsigned)(per * kXcds + r.aux_blocks);
  if (grid == 0) return 0;
  k<<<grid, kThreads, 0, s>>>(a);
  SEIS_CHECK_LAUNCH();
  return 0;
}

template <typename Item>
int upload(const std::vector<Item>& items, Item* table, hipStream_t s) {
  // from pageable memory: the copy has left it when the call returns
  SEIS_CHECK_HIP(hipMemcpyAsync(table, items.data(), items.size() * sizeof(Item),
                                hipMemcpyHostToDevice, s));
  return 0;
}

constexpr int kShapeCols = 6;  // nz, nx, B, nt, R, slots
constexpr int64_t kMaxProblems = (int64_t)1 << 20;

struct Batch {
  std::vector<Problem> p;
  std::vector<int64_t> out, ring, field;  // offsets
  int wide = 4;
  int64_t items = 0, floats = 0, fields = 0;
};

// The problems of a batch, laid out one after another in the arenas; work may
// be null (sizes only).
int make_batch(Batch& b, int64_t n, const int64_t* shape, const float* dt_h, const float* vp,
               const float* d, const float* wavelet, const int32_t* src, const int64_t* rec_flat,
               const int32_t* row_slot, bool rings, float* snaps, int32_t snap_every, float* work,
               int32_t npml, bool adjoint, int32_t vec_x, int32_t rows) {
  SEIS_CHECK_ARG(n >= 1 && n <= kMaxProblems && shape && dt_h, "bad batch of %lld", (long long)n);
  SEIS_CHECK_ARG(snap_every >= 0, "snap_every %d", snap_every);
  int64_t model = 0, wav = 0, so = 0, ro = 0, oo = 0, ri = 0, sn = 0, fo = 0, sl = 0;
  for (int64_t i = 0; i < n; ++i) {
    const int64_t* q = shape + i * kShapeCols;
    const int64_t nz = q[0], nx = q[1], B = q[2], nt = q[3], R = q[4];
    if (int e = check_march(B, nz, nx, dt_h[2 * i], dt_h[2 * i + 1], nt, R, npml, (int)q[5],
                            row_slot ? row_slot : reinterpret_cast<const int32_t*>(shape), 0,
                            vec_x, rows))
      return e;
    Problem p{};
    p.vp = vp + model; p.d = d + model; p.wavelet = wavelet + wav;
    p.nt = nt;
    p.src = src + 2 * so;
    p.rec_flat = rec_flat + ro;
    p.R = R;
    p.row_slot = row_slot + sl;
    p.slots = (int)q[5];
    p.B = B;
    p.g = seis::make_grid(nz, nx, npml, false);
    p.k = seis::make_consts(dt_h[2 * i], dt_h[2 * i + 1]);
    p.ring_len = rings ? seis_ring_len(nz, nx, npml, 0) : 0;
    if (rings)
      if (int e = check_ring(nz, nx, npml, p.ring_len)) return e;
    p.snaps = snaps ? snaps + sn : nullptr;
    p.snap_every = snap_every;
    p.w = carve(work ? work + b.floats : nullptr, B, nz, nx, q[5], R, adjoint);
    b.p.push_back(p);
    b.out.push_back(oo);
    b.ring.push_back(ri);
    b.field.push_back(fo);
    b.wide = std::min(b.wide, widest(nx));
    b.items += max_items(nt, snap_every);
    b.floats += p.w.total;
    model += nz * nx; wav += nt; so += B; ro += R; oo += nt * R; sl += nz + 1;
    ri += nt > 1 ? (nt - 1) * B * p.ring_len : 0;
    sn += seis_snapshot_count(nt, snap_every) * 2 * B * nz * nx;
    fo += B * nz * nx;
  }
  b.fields = fo;
  return 0;
}

// The plan for all cells of a launch, but with longer segments: next to each
// other's units the problems fill the chip with fewer.  ms, forward / adjoint, with
// segments of 16 and 24 rows: 16 problems of 31 10^6 cells 23.2 / 47.2 and 23.1 /
// 45.3, 12 of 18 10^6 12.6 / 26.8 and 12.5 / 25.8, 4 of 7 10^6 4.4 / 9.7 and 4.1 /
// 9.5.  What bounds them is the issue of vector instructions (about 25 per cell and
// step, a quarter of the lanes idle in the strips' halos); with one and two steps
// per launch the step kernels of the first took 36 / 86.
Plan batch_plan(int64_t cells, int wide, int32_t vec_x, int32_t rows) {
  Plan p = make_plan(cells, wide, 0, vec_x, rows);
  if (!rows && cells >= 3000000) p.rows_f = p.rows_a = 24;
  return p;
}

template <typename Item>
Item* table_of(const Batch& b, float* work) {
  return reinterpret_cast<Item*>(work + b.floats);
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
  if (int e = check_fields(fields)) return e;
  SEIS_CHECK_ARG(!snaps || snap_every > 0, "snapshots need snap_every > 0");
  const int64_t ring_len = ring ? seis_ring_len(nz, nx, npml, multiple) : 0;
  if (ring)
    if (int e = check_ring(nz, nx, npml, ring_len)) return e;
  const Grid g = seis::make_grid(nz, nx, npml, multiple != 0);
  const TimeConsts k = seis::make_consts(dt, h);
  const Plan p = make_plan(B * nz * nx, widest(nx), steps, vec_x, rows);
  hipStream_t s = (hipStream_t)stream;
  const Problem q{vp, d, wavelet, nt, src_zx, rec_flat, R, row_slot, slots, B, g, k, ring_len,
                  snaps, snap_every, carve(work, B, nz, nx, slots, R, false)};
  if (int e = prepare(q, false, s)) return e;
  FwdRun run(q, ring, rec_out, fields);
  if (int e = zero(run.cur, q.field(), s)) return e;
  if (int e = zero(run.prev, q.field(), s)) return e;
  const float* from;
  float* to;
  while (!run.done()) {
    FwdLevels f;
    const int T = run.next(p.t_f, f, from, to);
    SEIS_PROF(SEIS_KERNEL_ACOUSTIC_MARCH_FWD, s);
    if (int e = launch_fwd(T, p.vx_f, q.coefs(), f, src_zx, (int)B, g, k, p.rows_f, run.ga, s))
      return e;
    SEIS_PROF(SEIS_KERNEL_ACOUSTIC_MARCH_FWD, s);
    if (to)
      if (int e = copy(from, to, q.field(), s)) return e;
    run.advance(T);
  }
  if (run.ga.blocks > 0) {
    k_gather<<<run.ga.blocks, kThreads, 0, s>>>(run.ga);
    SEIS_CHECK_LAUNCH();
  }
  if (run.finish(from, to))
    if (int e = copy(from, to, q.field(), s)) return e;
  run.final_fields(final_fields);
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
  if (int e = check_fields(u)) return e;
  if (int e = check_fields(mu)) return e;
  const int64_t ring_len = seis_ring_len(nz, nx, npml, multiple);
  if (int e = check_adjoint(nz, nx, nt, npml, multiple, ring_len, ring)) return e;
  SEIS_CHECK_ARG(!snaps || snap_every > 0, "snapshots need snap_every > 0");
  const Grid g = seis::make_grid(nz, nx, npml, multiple != 0);
  const TimeConsts k = seis::make_consts(dt, h);
  const Plan p = make_plan(B * nz * nx, widest(nx), steps, vec_x, rows);
  hipStream_t s = (hipStream_t)stream;
  const Problem q{vp, d, wavelet, nt, src_zx, rec_flat, R, row_slot, slots, B, g, k, ring_len,
                  const_cast<float*>(snaps), snap_every, carve(work, B, nz, nx, slots, R, true)};
  if (int e = prepare(q, true, s)) return e;
  AdjRun run(q, ring, rec_grad, u, mu, grad_part);
  if (int e = zero(mu[0], q.field(), s)) return e;
  if (int e = zero(mu[1], q.field(), s)) return e;
  const Sources s0 = run.sources(nt, p.t_a, 0);
  if (s0.blocks > 0) {
    k_sources<<<s0.blocks, kThreads, 0, s>>>(s0);
    SEIS_CHECK_LAUNCH();
  }
  while (!run.done()) {
    AdjLevels f;
    Sources so;
    bool last;
    const int T = run.next(p.t_a, f, so, last);
    SEIS_PROF(SEIS_KERNEL_ACOUSTIC_MARCH_ADJ, s);
    if (int e = launch_adj(T, p.vx_a, q.coefs(), f, src_zx, (int)B, g, k, p.rows_a, last, so, s))
      return e;
    SEIS_PROF(SEIS_KERNEL_ACOUSTIC_MARCH_ADJ, s);
  }
  return final_grad(run, grad, s);
}

int64_t seis_acoustic_march_batch_workspace(int64_t n, const int64_t* shape, int32_t snap_every,
                                            int32_t adjoint) {
  if (n < 1 || n > kMaxProblems || !shape) {
    seis::set_error("bad batch of %lld", (long long)n);
    return -1;
  }
  Batch b;
  std::vector<float> ones(2 * (size_t)n, 1.0f);
  if (make_batch(b, n, shape, ones.data(), nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                 false, nullptr, snap_every, nullptr, 0, adjoint != 0, 0, 0))
    return -1;
  const size_t item = adjoint ? sizeof(AdjItem) : sizeof(FwdItem);
  return b.floats + b.items * (int64_t)((item + 3) / 4);
}

int seis_acoustic_march_batch_forward(int64_t n, const int64_t* shape, const float* dt_h,
                                      const float* vp, const float* d, const float* wavelet,
                                      const int32_t* src_zx, const int64_t* rec_flat,
                                      const int32_t* row_slot, float* rec_out, float* ring,
                                      float* snaps, int32_t snap_every, float* work,
                                      float* const* fields, int32_t npml, int32_t vec_x,
                                      int32_t rows, void* stream) {
  SEIS_CHECK_ARG(vp && d && wavelet && src_zx && work && fields, "null pointer argument");
  SEIS_CHECK_ARG(!snaps || snap_every > 0, "snapshots need snap_every > 0");
  Batch b;
  if (int e = make_batch(b, n, shape, dt_h, vp, d, wavelet, src_zx, rec_flat, row_slot,
                         ring != nullptr, snaps, snap_every, work, npml, false, vec_x, rows))
    return e;
  if (int e = check_fields(fields)) return e;
  hipStream_t s = (hipStream_t)stream;
  std::vector<FwdRun> runs;
  for (int64_t i = 0; i < n; ++i) {
    const Problem& q = b.p[i];
    SEIS_CHECK_ARG(q.R == 0 || (rec_flat && rec_out && row_slot), "bad receiver arguments");
    float* f[4];
    for (int j = 0; j < 4; ++j) f[j] = fields[j] + b.field[i];
    float* rg = ring ? ring + b.ring[i] : nullptr;
    // played once for the buffers of the last pair, which then become the
    // first two: the caller finds u^nt and u^{nt-1} in fields[0] and fields[1]
    FwdRun dry(q, rg, rec_out, f);
    const float* from;
    float* to;
    while (!dry.done()) {
      FwdLevels lv;
      dry.advance(dry.next(make_plan(1, 1, 0, vec_x, rows).t_f, lv, from, to));
    }
    (void)dry.finish(from, to);
    int32_t at[2] = {0, 1};
    dry.final_fields(at);
    float* g[4];
    for (int j = 0, other = 2; j < 4; ++j)
      g[j] = f[j == at[0] ? 0 : j == at[1] ? 1 : other++];
    runs.emplace_back(q, rg, rec_out ? rec_out + b.out[i] : nullptr, g);
    if (int e = prepare(q, false, s)) return e;
    if (int e = zero(runs.back().cur, q.field(), s)) return e;
    if (int e = zero(runs.back().prev, q.field(), s)) return e;
  }
  std::vector<FwdItem> items;
  std::vector<Round> rounds;
  std::vector<CopyAfter> copies;
  for (bool more = true; more;) {
    int64_t cells = 0;
    for (const FwdRun& r : runs) cells += r.done() ? 0 : r.p.field();
    const Plan p = batch_plan(cells, b.wide, vec_x, rows);
    Round rd{items.size(), 0, 0, 0, p.vx_f};
    more = false;
    for (FwdRun& r : runs) {
      if (r.done() && r.ga.blocks == 0) continue;
      more = true;
      FwdItem it{};
      it.aux = r.ga;
      r.ga.blocks = 0;
      int64_t blocks = 0;
      if (!r.done()) {
        const float* from;
        float* to;
        FwdLevels f;
        it.T = r.next(p.t_f, f, from, to);
        const Split sp = make_split(r.p.g, it.T, p.vx_f, p.rows_f,
                                    (int)std::min<int64_t>(r.p.B, kShotGroup));
        it.p = FwdParams{r.p.coefs(), f, r.p.src, (int)r.p.B, sp, r.p.g, r.p.k};
        blocks = split_blocks(sp, r.p.B);
        if (to) copies.push_back({rounds.size(), from, to, r.p.field()});
        r.advance(it.T);
        if (r.done() && r.finish(from, to))
          copies.push_back({rounds.size(), from, to, r.p.field()});
      }
      add_item(items, rd, it, blocks);
    }
    if (more) rounds.push_back(rd);
  }
  SEIS_CHECK_ARG((int64_t)items.size() <= b.items, "batch table of %lld items", (long long)b.items);
  FwdItem* table = table_of<FwdItem>(b, work);
  if (int e = upload(items, table, s)) return e;
  size_t c = 0;
  for (size_t i = 0; i < rounds.size(); ++i) {
    const Round& r = rounds[i];
    auto* k = r.vx == 4 ? k_march_fwd_batch<4> : r.vx == 2 ? k_march_fwd_batch<2>
                                                           : k_march_fwd_batch<1>;
    SEIS_PROF(SEIS_KERNEL_BATCH_FWD, s);
    if (int e = launch_round(k, table, r, s)) return e;
    SEIS_PROF(SEIS_KERNEL_BATCH_FWD, s);
    for (; c < copies.size() && copies[c].round == i; ++c)
      if (int e = copy(copies[c].from, copies[c].to, copies[c].n, s)) return e;
  }
  return 0;
}

int seis_acoustic_march_batch_backward(int64_t n, const int64_t* shape, const float* dt_h,
                                       const float* vp, const float* d, const float* wavelet,
                                       const int32_t* src_zx, const int64_t* rec_flat,
                                       const int32_t* row_slot, const float* rec_grad,
                                       const float* ring, const float* snaps, int32_t snap_every,
                                       float* work, float* const* u, float* const* mu,
                                       float* grad_part, float* grad, int32_t npml, int32_t vec_x,
                                       int32_t rows, void* stream) {
  SEIS_CHECK_ARG(vp && d && wavelet && src_zx && work && u && mu && grad_part && grad,
                 "null pointer argument");
  SEIS_CHECK_ARG(!snaps || snap_every > 0, "snapshots need snap_every > 0");
  Batch b;
  if (int e = make_batch(b, n, shape, dt_h, vp, d, wavelet, src_zx, rec_flat, row_slot, true,
                         const_cast<float*>(snaps), snap_every, work, npml, true, vec_x,
                         rows))
    return e;
  if (int e = check_fields(u)) return e;
  if (int e = check_fields(mu)) return e;
  hipStream_t s = (hipStream_t)stream;
  if (int e = zero(mu[0], b.fields, s)) return e;
  if (int e = zero(mu[1], b.fields, s)) return e;
  std::vector<AdjRun> runs;
  for (int64_t i = 0; i < n; ++i) {
    const Problem& q = b.p[i];
    SEIS_CHECK_ARG(q.R == 0 || (rec_flat && rec_grad && row_slot), "bad receiver arguments");
    if (int e = check_adjoint(q.g.nz, q.g.nx, q.nt, npml, 0, q.ring_len, ring)) return e;
    float *fu[4], *fm[4];
    for (int j = 0; j < 4; ++j) {
      fu[j] = u[j] + b.field[i];
      fm[j] = mu[j] + b.field[i];
    }
    runs.emplace_back(q, ring ? ring + b.ring[i] : nullptr,
                      rec_grad ? rec_grad + b.out[i] : nullptr, fu, fm, grad_part + b.field[i]);
    if (int e = prepare(q, true, s)) return e;
  }
  std::vector<AdjItem> items;
  std::vector<Round> rounds;
  const int t_a = make_plan(1, 1, 0, vec_x, rows).t_a;
  Round rd{0, 0, 0, 0, 1};  // the first launches' sources
  for (const AdjRun& r : runs) {
    AdjItem it{};
    it.aux = r.sources(r.p.nt, t_a, 0);
    if (it.aux.blocks > 0) add_item(items, rd, it, 0);
  }
  rounds.push_back(rd);
  for (;;) {
    int64_t cells = 0;
    for (const AdjRun& r : runs) cells += r.done() ? 0 : r.p.field();
    if (cells == 0) break;
    const Plan p = batch_plan(cells, b.wide, vec_x, rows);
    rd = Round{items.size(), 0, 0, 0, p.vx_a};
    for (AdjRun& r : runs) {
      if (r.done()) continue;
      AdjItem it{};
      AdjLevels f;
      bool last;
      it.T = r.next(p.t_a, f, it.aux, last);
      const Split sp = make_split(r.p.g, it.T, p.vx_a, p.rows_a,
                                  (int)std::min<int64_t>(r.p.B, kShotGroup));
      it.p = AdjParams{r.p.coefs(), f, r.p.src, (int)r.p.B, sp, r.p.g, r.p.k, last};
      add_item(items, rd, it, split_blocks(sp, r.p.B));
    }
    rounds.push_back(rd);
  }
  SEIS_CHECK_ARG((int64_t)items.size() <= b.items, "batch table of %lld items", (long long)b.items);
  AdjItem* table = table_of<AdjItem>(b, work);
  if (!items.empty())
    if (int e = upload(items, table, s)) return e;
  for (const Round& r : rounds) {
    auto* k = r.vx == 4 ? k_march_adj_batch<4> : r.vx == 2 ? k_march_adj_batch<2>
                                                           : k_march_adj_batch<1>;
    SEIS_PROF(SEIS_KERNEL_BATCH_BWD, s);
    if (int e = launch_round(k, table, r, s)) return e;
    SEIS_PROF(SEIS_KERNEL_BATCH_BWD, s);
  }
  for (int64_t i = 0, model = 0; i < n; ++i) {
    if (int e = final_grad(runs[i], grad + model, s)) return e;
    model += runs[i].p.g.plane;
  }
  return 0;
}

}  // extern "C"
