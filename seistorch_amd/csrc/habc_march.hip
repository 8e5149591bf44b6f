// The HABC loops with up to four time steps per launch away from the edges: the
// marching waves of march.h on the core of the grid, the steps of habc_strips.h on
// the frame around it.
#include "common.h"
#include "habc_strips.h"
#include "march.h"
#include "march_rows.h"
#include "seistorch_amd.h"
#include "tiles.h"

#include <algorithm>
#include <vector>

namespace {

// The strip ranges alone, a frame's step of the marching loops: the rebuilt field over
// uc (SAME) or into uo.  (Kernels of their own: with uo among the arguments of
// k_habc_adj_deep, one step took 2 to 2.5 % longer, 35.1 us for 34.3 at 500 x 2400 x 2.)
template <int S, bool SAME>
__global__ __launch_bounds__(256) void k_frame_adj(
    const float* __restrict__ vp, const float* __restrict__ bw, const float* __restrict__ y1,
    const float* __restrict__ y2, float* __restrict__ out, const float* __restrict__ um,
    float* __restrict__ uc, float* __restrict__ uo, float* __restrict__ gpart,
    const int32_t* __restrict__ src, const float* __restrict__ wn, int recon, int B, HabcCtx hc,
    seis::TimeConsts k, Deep dp, Frame f, int ngf, int G, TileMap tb, int ngb, TileMap ts) {
  if constexpr (SAME)
    (void)habc_adj_strip_block<S, true>((int)blockIdx.x, vp, bw, y1, y2, out, um, uc,
                                        gpart, src, wn, recon, B, hc, k, dp, f, ngf, G, tb, ngb,
                                        ts);
  else
    (void)habc_adj_strip_block<S, false>((int)blockIdx.x, vp, bw, y1, y2, out, um,
                                         TwoFields{uc, uo}, gpart, src, wn, recon, B, hc, k, dp,
                                         f, ngf, G, tb, ngb, ts);
}

// k_habc_post without the receivers in `skip`, after a frame's step of the marching
// loops.
__global__ __launch_bounds__(256) void k_frame_post(
    const float* __restrict__ vp, const float* __restrict__ um, float* __restrict__ uc,
    float* __restrict__ lam, float* __restrict__ gpart, const int64_t* __restrict__ rec,
    const float* __restrict__ rgrad, int64_t R, const float* __restrict__ ring_slot,
    int64_t ring_len, int recon, int B, int S, Grid g, seis::TimeConsts k, Deep skip) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < R) {
    const int64_t f = rec[t];
    const float sk = rgrad[t];
    const int64_t b = f / g.plane;
    const int i = (int)(f - b * g.plane);
    const int z = i / g.nx, x = i - z * g.nx;
    if (in_deep(z, x, skip)) return;
    atomicAdd(lam + f, sk);
    if (seis::interior(z, x, g)) {
      const float Lu = lap5(um + b * g.plane, z, x, i, g, k.ih2);
      atomicAdd(gpart + (b / S) * g.plane + i, 2.0f * vp[i] * (1.0f / k.idt2) * Lu * sk);
    }
    return;
  }
  t -= R;
  if (recon != 0 && t < (int64_t)B * ring_len) {
    const int64_t b = t / ring_len;
    const int64_t j = t - b * ring_len;
    uc[b * g.plane + seis::ring_cell(j, g)] = recon == 1 ? ring_slot[t] : 0.0f;
  }
}

template <int S>
constexpr auto* k_frame_adj_in = &k_frame_adj<S, true>;
template <int S>
constexpr auto* k_frame_adj_out = &k_frame_adj<S, false>;

// ---- four time steps per launch away from the boundary

// Core: the cells at least kW + 3 + kMaxT from every edge.  Within kMaxT cells of
// it the step is the undamped one, so the marching waves of march.h take up to
// kMaxT steps of Core in one launch from the fields at its start alone.  The frame
// around Core takes its steps one by one, step t of T also on the T - t outermost
// cells of Core, which the frame's next steps read and the march leaves to itself.
// (With one step per launch everywhere the fields cross HBM once per step, which
// is what bounded it: 16 shots of 900 x 2500, 105 us forward, 261 adjoint per step
// with the records and rings, now 70 and 167: 34 and 72 of them the march, most of the
// rest the frame's steps, bound by their loads' latency and long set-up per cell.)
constexpr int kCoreMargin = kW + 3 + kMaxT;

inline Deep core_of(int64_t nz, int64_t nx) {
  const int v = widest(nx);
  return Deep{kCoreMargin, (int)nz - kCoreMargin, (kCoreMargin + v - 1) / v * v,
              ((int)nx - kCoreMargin) / v * v};
}

inline Deep shrunk(const Deep& c, int e) { return Deep{c.z0 + e, c.z1 - e, c.x0 + e, c.x1 - e}; }

// What a launch's adjoint sources reach of Core: a source in the frame kMaxT - 1
// cells away is in Core's last level.
inline Deep reach_of(const Deep& core) { return shrunk(core, 1 - kMaxT); }

// row_slot[z] = 0 for every row that holds a receiver in `in` (-1 before).
__global__ __launch_bounds__(256) void k_core_rows(const int64_t* __restrict__ rec, int64_t R,
                                                   int64_t plane, int nx, Deep in,
                                                   int32_t* __restrict__ row_slot) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= R) return;
  const int i = (int)(rec[t] % plane), z = i / nx;
  if (in_deep(z, i - z * nx, in)) row_slot[z] = 0;
}

// Cells of the receivers in `part` in the (slots, B, nx) rows, -1 for the others; with
// head/next, the receivers of one cell are chained for the adjoint's sources.
__global__ __launch_bounds__(256) void k_core_cells(const int64_t* __restrict__ rec, int64_t R,
                                                    int64_t plane, int nx, int B, Deep part,
                                                    const int32_t* __restrict__ row_slot,
                                                    int64_t* __restrict__ cell,
                                                    int32_t* __restrict__ head,
                                                    int32_t* __restrict__ next) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= R) return;
  const int64_t b = rec[t] / plane;
  const int i = (int)(rec[t] - b * plane), z = i / nx, x = i - z * nx;
  const bool in = in_deep(z, x, part) && row_slot && row_slot[z] >= 0;
  const int64_t c = in ? ((int64_t)row_slot[z] * B + b) * nx + x : -1;
  if (cell) cell[t] = c;
  if (head && in) next[t] = atomicExch(head + c, (int32_t)t);
}

struct CoreFwd {
  FwdParams p;
  int per;
};

struct CoreAdj {
  AdjParams p;
  int per;
};

template <int T, int VX>
__global__ __launch_bounds__(kThreads) void k_core_fwd(CoreFwd a) {
  int strip, seg, b;
  if (!march_unit(a.p.sp, a.p.B, xcd_block(a.per), strip, seg, b)) return;
  march_forward_strip<T, VX, false>(a.p, launch_params<FwdParams>(), b, strip, seg);
}

template <int T, int VX>
__global__ __launch_bounds__(kThreads) void k_core_adj(CoreAdj a) {
  int strip, seg, b;
  if (!march_unit(a.p.sp, a.p.B, xcd_block(a.per), strip, seg, b)) return;
  march_adjoint_strip<T, VX, kDeep>(a.p, launch_params<AdjParams>(), b, strip, seg);
}

#define SEIS_CORE_LAUNCH(K, T, VX, a, s)                                            \
  switch (T * 8 + VX) {                                                             \
    case 9: K<1, 1><<<a.per * kXcds, kThreads, 0, s>>>(a); break;                   \
    case 10: K<1, 2><<<a.per * kXcds, kThreads, 0, s>>>(a); break;                  \
    case 12: K<1, 4><<<a.per * kXcds, kThreads, 0, s>>>(a); break;                  \
    case 17: K<2, 1><<<a.per * kXcds, kThreads, 0, s>>>(a); break;                  \
    case 18: K<2, 2><<<a.per * kXcds, kThreads, 0, s>>>(a); break;                  \
    case 20: K<2, 4><<<a.per * kXcds, kThreads, 0, s>>>(a); break;                  \
    case 33: K<4, 1><<<a.per * kXcds, kThreads, 0, s>>>(a); break;                  \
    case 34: K<4, 2><<<a.per * kXcds, kThreads, 0, s>>>(a); break;                  \
    default: K<4, 4><<<a.per * kXcds, kThreads, 0, s>>>(a); break;                  \
  }                                                                                 \
  SEIS_CHECK_LAUNCH();

// Records and rings of a launch's levels: receivers in Core from the rows, the
// others and the rings from the levels' fields.
struct CoreKeep {
  const float* lev[kMaxT];
  const float* rows;
  const int64_t* cell;
  const int64_t* rec;
  int64_t R, row_cells, ring_len;
  float* out;   // records of the first level
  float* ring;  // ring slot of the first level
  int ring_levels, B;
};

__global__ __launch_bounds__(256) void k_core_keep(CoreKeep a, Grid g) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int l = blockIdx.y;
  const float* u = a.lev[l];
  if (t < a.R) {
    const int64_t c = a.cell[t];
    a.out[l * a.R + t] = c >= 0 ? a.rows[l * a.row_cells + c] : u[a.rec[t]];
    return;
  }
  t -= a.R;
  if (l < a.ring_levels && t < (int64_t)a.B * a.ring_len) {
    const int64_t b = t / a.ring_len;
    const int64_t j = t - b * a.ring_len;
    a.ring[l * a.B * a.ring_len + t] = u[b * g.plane + seis::ring_cell(j, g)];
  }
}

// grad: on Core 2c A0 times the march's sums over the shots' planes, elsewhere the
// frame's sums over the shot groups'.
__global__ __launch_bounds__(256) void k_core_grad(const float* __restrict__ vp,
                                                   const float* __restrict__ gcore, int nb,
                                                   const float* __restrict__ gpart, int G,
                                                   float* __restrict__ out, Deep core, Grid g,
                                                   seis::TimeConsts k) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.plane) return;
  const int z = (int)(t / g.nx), x = (int)(t - (int64_t)z * g.nx);
  float s = 0.0f;
  if (in_deep(z, x, core)) {
    for (int b = 0; b < nb; ++b) s += gcore[b * g.plane + t];
    s = 2.0f * vp[t] * (1.0f / k.idt2) * s;
  } else {
    for (int q = 0; q < G; ++q) s += gpart[(int64_t)q * g.plane + t];
  }
  out[t] = s;
}

struct CoreWork {
  float *c2, *A, *Bc, *rows;
  int64_t* cell;
  int32_t *head, *next;
  int64_t row_cells, total;
};

CoreWork carve_core(float* base, int64_t B, int64_t nz, int64_t nx, int64_t slots, int64_t R) {
  CoreWork w;
  int64_t o = 0;
  auto take = [&](int64_t n) { const int64_t at = o; o += pad64(n); return base + at; };
  w.row_cells = slots * B * nx;
  w.c2 = take(nz * nx); w.A = take(nz * nx); w.Bc = take(nz * nx);
  w.rows = take(kMaxT * w.row_cells);
  w.cell = reinterpret_cast<int64_t*>(take(2 * R));
  w.head = reinterpret_cast<int32_t*>(take(w.row_cells));
  w.next = reinterpret_cast<int32_t*>(take(R));
  w.total = o;
  return w;
}


int check_core(int64_t nz, int64_t nx, int64_t R, int32_t slots, const int32_t* row_slot,
               int32_t vec_x, int32_t rows) {
  const Deep c = core_of(nz, nx);
  SEIS_CHECK_ARG(nz * nx <= kMaxCells && c.z1 - c.z0 >= 4 * kMaxT && c.x1 - c.x0 >= 4 * kMaxT,
                 "grid %lld x %lld has too few cells away from its edges", (long long)nz,
                 (long long)nx);
  SEIS_CHECK_ARG(slots >= 0 && slots <= nz && (slots == 0 || (row_slot && R > 0)) &&
                     R < (int64_t)1 << 31,
                 "receivers need their rows (slots %d)", slots);
  SEIS_CHECK_ARG(vec_x == 0 || ((vec_x == 1 || vec_x == 2 || vec_x == 4) && nx % vec_x == 0),
                 "vec_x %d for nx = %lld", vec_x, (long long)nx);
  SEIS_CHECK_ARG(rows >= 0 && rows <= 1 << 20, "rows %d", rows);
  return 0;
}

}  // namespace

extern "C" {

// Core needs a few cells beyond what a launch's frame steps take of it.
int32_t seis_habc_march_fits(int64_t nz, int64_t nx) {
  const Deep c = core_of(nz, nx);
  return nz * nx <= kMaxCells && c.z1 - c.z0 >= 4 * kMaxT && c.x1 - c.x0 >= 4 * kMaxT;
}

int seis_habc_core_rows(const int64_t* rec_flat, int64_t R, int64_t nz, int64_t nx,
                        int32_t* row_slot, void* stream) {
  SEIS_CHECK_ARG(row_slot && (R == 0 || rec_flat) && R >= 0, "bad arguments");
  SEIS_CHECK_ARG(nz >= 1 && nx >= 1 && nz * nx < (int64_t)1 << 31, "grid %lld x %lld",
                 (long long)nz, (long long)nx);
  hipStream_t s = (hipStream_t)stream;
  k_fill_i32<<<blocks_of(nz), 256, 0, s>>>(row_slot, nz, -1);
  SEIS_CHECK_LAUNCH();
  if (R > 0) {
    k_core_rows<<<blocks_of(R), 256, 0, s>>>(rec_flat, R, nz * nx, (int)nx,
                                             reach_of(core_of(nz, nx)), row_slot);
    SEIS_CHECK_LAUNCH();
  }
  k_number_rows<<<1, 64, 0, s>>>(row_slot, (int)nz);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int64_t seis_habc_march_workspace(int64_t B, int64_t nz, int64_t nx, int32_t slots, int64_t R) {
  return carve_core(nullptr, B, nz, nx, slots, R).total;
}

int seis_habc_march_forward(const float* vp, const float* b, const float* wavelet, int64_t nt,
                            const int32_t* src_zx, const int64_t* rec_flat, int64_t R,
                            const int32_t* row_slot, int32_t slots, float* rec_out, float* ring,
                            float* snaps, int32_t snap_every, float* work, float* const* fields,
                            int32_t* final_fields, int64_t B, int64_t nz, int64_t nx, float dt,
                            float h, int32_t npml, int32_t multiple, int32_t shots_per_group,
                            int32_t vec_x, int32_t rows, void* stream) {
  if (int e = habc_check(B, nz, nx, dt, h, shots_per_group)) return e;
  if (int e = check_core(nz, nx, R, slots, row_slot, vec_x, rows)) return e;
  SEIS_CHECK_ARG(vp && b && wavelet && src_zx && work && fields && final_fields,
                 "null pointer argument");
  SEIS_CHECK_ARG(nt >= 1 && R >= 0 && (R == 0 || (rec_flat && rec_out)), "bad receiver arguments");
  for (int i = 0; i < 5; ++i) SEIS_CHECK_ARG(fields[i], "null field buffer");
  const int64_t ring_len = ring ? seis_ring_len(nz, nx, npml, multiple) : 0;
  SEIS_CHECK_ARG(!ring || ring_len > 0, "grid has no interior inside npml=%d", npml);
  SEIS_CHECK_ARG(!snaps || snap_every > 0, "snapshots need snap_every > 0");
  const HabcCtx hc{seis::make_grid(nz, nx, npml, multiple != 0), multiple ? 1 : 0, dt, h};
  const Grid& g = hc.g;
  const int S = shots_per_group, G = (int)((B + S - 1) / S);
  const int ngf = frame_groups(nz, nx, G, S);
  const Deep core = core_of(nz, nx);
  const Plan pl = make_plan(B * (core.z1 - core.z0) * (core.x1 - core.x0), widest(nx), 0, vec_x,
                            rows);
  const seis::TimeConsts k = seis::make_consts(dt, h);
  const CoreWork w = carve_core(work, B, nz, nx, slots, R);
  hipStream_t s = (hipStream_t)stream;
  const int64_t field = B * g.plane;
  k_coefs<<<blocks_of(g.plane), 256, 0, s>>>(vp, nullptr, g.plane, k, w.c2, w.A, w.Bc);
  SEIS_CHECK_LAUNCH();
  if (R > 0) {
    k_core_cells<<<blocks_of(R), 256, 0, s>>>(rec_flat, R, g.plane, g.nx, (int)B, core,
                                              slots ? row_slot : nullptr, w.cell, nullptr,
                                              nullptr);
    SEIS_CHECK_LAUNCH();
  }
  float *cur = fields[0], *prev = fields[1];
  std::vector<float*> free_bufs{fields[2], fields[3], fields[4]};
  auto take = [&]() { float* q = free_bufs.back(); free_bufs.pop_back(); return q; };
  for (float* q : {cur, prev}) {
    k_habc_fill<<<nblk(field), 256, 0, s>>>(q, field);
    SEIS_CHECK_LAUNCH();
  }
  const int64_t last_snap = snaps ? seis_snapshot_count(nt, snap_every) * snap_every : 0;
  for (int64_t n = 0; n < nt;) {
    int64_t stop = nt, m = 0;
    if (last_snap > 0 && n <= last_snap) {
      m = std::max<int64_t>(1, (n - 1 + snap_every) / snap_every) * snap_every;
      stop = m + 1;
    }
    const int T = next_steps(stop - n, kMaxT);
    // fields of the levels: the frame's are whole only around Core, the march's
    // (the last two) on Core; the second of four takes u^{n-1}'s place
    float* lev[kMaxT + 2] = {prev, cur};  // lev[t + 1] = u^{n+t}
    float* spare = nullptr;
    if (T == 4) {
      spare = take();
      lev[2] = spare;
      lev[3] = prev;
    }
    if (T >= 2) lev[T] = take();
    lev[T + 1] = take();
    CoreFwd a{};
    a.p.cf = Coefs{w.c2, w.A, w.Bc};
    a.p.f.u = cur; a.p.f.up = prev;
    a.p.f.o1 = lev[T + 1];
    a.p.f.o0 = T >= 2 ? lev[T] : nullptr;
    a.p.f.w = wavelet + n;
    a.p.f.rows = slots ? w.rows : nullptr;
    a.p.f.row_slot = row_slot;
    a.p.f.slots = slots;
    a.p.src = src_zx;
    a.p.B = (int)B;
    a.p.sp = make_split(Region{core.z0, core.z1, core.x0, core.x1}, T, pl.vx_f, pl.rows_f,
                        (int)std::min<int64_t>(B, kShotGroup));
    a.p.g = g;
    a.p.k = k;
    a.per = (int)((split_blocks(a.p.sp, B) + kXcds - 1) / kXcds);
    SEIS_PROF(SEIS_KERNEL_HABC_FWD, s);
    SEIS_CORE_LAUNCH(k_core_fwd, T, pl.vx_f, a, s);
    for (int t = 1; t <= T; ++t) {
      const Deep dp = shrunk(core, T - t);
      const Frame fr = make_frame(g, dp, (G + ngf - 1) / ngf);
      SEIS_HABC_LAUNCH_V(k_habc_fwd_deep, S, 1, dim3(fr.per * kXcds), s, vp, lev[t], lev[t - 1],
                         lev[t + 1], src_zx, wavelet + n + t - 1, (int)B, hc, k, dp,
                         (TileMap{0, 0, 0, 0}), b, fr, ngf, G);
    }
    SEIS_PROF(SEIS_KERNEL_HABC_FWD, s);
    CoreKeep kp{};
    for (int t = 1; t <= T; ++t) kp.lev[t - 1] = lev[t + 1];
    kp.rows = w.rows; kp.cell = w.cell; kp.rec = rec_flat;
    kp.R = R; kp.row_cells = w.row_cells; kp.ring_len = ring_len;
    kp.out = R ? rec_out + n * R : nullptr;
    kp.ring_levels = ring ? (int)std::min<int64_t>(T, nt - 1 - n) : 0;
    kp.ring = kp.ring_levels > 0 ? ring + n * B * ring_len : nullptr;
    kp.B = (int)B;
    const int64_t items = R + (kp.ring_levels > 0 ? B * ring_len : 0);
    if (items > 0) {
      k_core_keep<<<dim3(nblk(items), T), 256, 0, s>>>(kp, g);
      SEIS_CHECK_LAUNCH();
    }
    if (spare) free_bufs.push_back(spare);
    free_bufs.push_back(prev);
    if (T >= 2) free_bufs.push_back(cur);
    prev = T >= 2 ? lev[T] : cur;
    cur = lev[T + 1];
    n += T;
    if (m > 0 && n == stop) {
      float* sp = snaps + (m / snap_every - 1) * 2 * field;
      k_habc_copy2<<<nblk(field), 256, 0, s>>>(prev, sp, cur, sp + field, field);
      SEIS_CHECK_LAUNCH();
    }
  }
  for (int i = 0; i < 5; ++i) {
    if (fields[i] == cur) final_fields[0] = i;
    if (fields[i] == prev) final_fields[1] = i;
  }
  return 0;
}

int seis_habc_march_backward(const float* vp, const float* b, const float* wavelet, int64_t nt,
                             const int32_t* src_zx, const int64_t* rec_flat, int64_t R,
                             const int32_t* row_slot, int32_t slots, const float* rec_grad,
                             const float* ring, const float* snaps, int32_t snap_every,
                             float* work, float* const* u, float* const* lam, float* grad_core,
                             float* grad_part, float* grad, int64_t B, int64_t nz, int64_t nx,
                             float dt, float h, int32_t npml, int32_t multiple,
                             int32_t shots_per_group, int32_t vec_x, int32_t rows, void* stream) {
  if (int e = habc_check(B, nz, nx, dt, h, shots_per_group)) return e;
  if (int e = check_core(nz, nx, R, slots, row_slot, vec_x, rows)) return e;
  SEIS_CHECK_ARG(vp && b && wavelet && src_zx && work && u && lam && grad_core && grad_part &&
                     grad,
                 "null pointer argument");
  SEIS_CHECK_ARG(nt >= 1 && R >= 0 && (R == 0 || (rec_flat && rec_grad)),
                 "bad receiver arguments");
  for (int i = 0; i < 5; ++i) SEIS_CHECK_ARG(lam[i] && (i == 4 || u[i]), "null field buffer");
  const int64_t ring_len = seis_ring_len(nz, nx, npml, multiple);
  SEIS_CHECK_ARG(ring_len > 0, "grid has no interior inside npml=%d", npml);
  SEIS_CHECK_ARG(ring || nt <= 2, "ring storage is required for nt > 2");
  SEIS_CHECK_ARG(!snaps || snap_every > 0, "snapshots need snap_every > 0");
  const HabcCtx hc{seis::make_grid(nz, nx, npml, multiple != 0), multiple ? 1 : 0, dt, h};
  const Grid& g = hc.g;
  const int S = shots_per_group, G = (int)((B + S - 1) / S);
  const int ngf = frame_groups(nz, nx, G, S), ngb = even_share(G, std::min(4, 2 * ngf));
  const Deep core = core_of(nz, nx);
  const Plan pl = make_plan(B * (core.z1 - core.z0) * (core.x1 - core.x0), widest(nx), 0, vec_x,
                            rows);
  const seis::TimeConsts k = seis::make_consts(dt, h);
  const CoreWork w = carve_core(work, B, nz, nx, slots, R);
  hipStream_t s = (hipStream_t)stream;
  const int64_t field = B * g.plane;
  k_coefs<<<blocks_of(g.plane), 256, 0, s>>>(vp, nullptr, g.plane, k, w.c2, w.A, w.Bc);
  SEIS_CHECK_LAUNCH();
  if (slots > 0) {
    k_fill_i32<<<blocks_of(w.row_cells), 256, 0, s>>>(w.head, w.row_cells, -1);
    SEIS_CHECK_LAUNCH();
    k_core_cells<<<blocks_of(R), 256, 0, s>>>(rec_flat, R, g.plane, g.nx, (int)B,
                                              reach_of(core), row_slot, nullptr, w.head, w.next);
    SEIS_CHECK_LAUNCH();
  }
  float *X = u[1], *Y = u[0];      // u^{k-1}, u^k
  float *M1 = lam[0], *M2 = lam[1];  // lambda^{k+1}, lambda^{k+2}
  std::vector<float*> ufree{u[2], u[3]}, lfree{lam[2], lam[3], lam[4]};
  auto take = [](std::vector<float*>& v) { float* q = v.back(); v.pop_back(); return q; };
  for (float* q : {M1, M2}) {
    k_habc_fill<<<nblk(field), 256, 0, s>>>(q, field);
    SEIS_CHECK_LAUNCH();
  }
  k_habc_fill<<<nblk((int64_t)G * g.plane), 256, 0, s>>>(grad_part, (int64_t)G * g.plane);
  SEIS_CHECK_LAUNCH();
  const int64_t last_snap = snaps ? seis_snapshot_count(nt, snap_every) * snap_every : 0;
  bool first = true;
  // iteration 1 adds nothing (u^0 = 0)
  for (int64_t kk = nt; kk >= 2;) {
    int64_t left = kk - 1, m = 0;
    if (last_snap > 0 && kk >= snap_every + 2) {
      m = std::min<int64_t>(last_snap, (kk - 2) / snap_every * snap_every);
      left = kk - 2 - m + 1;
    }
    const int T = next_steps(left, kMaxT);
    // L[t + 1] = lambda^{kk+1-t}, U[t + 1] = u^{kk-1-t}; the frame's first levels of
    // four take the place of fields that the march has read
    float* L[kMaxT + 2] = {M2, M1};
    float* U[kMaxT + 2] = {Y, X};
    float* spare = nullptr;
    if (T == 4) {
      spare = take(lfree);
      L[2] = spare;
      L[3] = M2;
      U[2] = Y;
      U[3] = X;
    }
    if (T >= 2) {
      L[T] = take(lfree);
      U[T] = take(ufree);
    }
    L[T + 1] = take(lfree);
    U[T + 1] = take(ufree);
    CoreAdj a{};
    a.p.cf = Coefs{w.c2, w.A, w.Bc};
    a.p.f.x = X; a.p.f.y = Y; a.p.f.m1 = M1; a.p.f.m2 = M2;
    a.p.f.ox = U[T + 1];
    a.p.f.om1 = L[T + 1];
    a.p.f.oy = T >= 2 ? U[T] : nullptr;
    a.p.f.om2 = T >= 2 ? L[T] : nullptr;
    a.p.f.gpart = grad_core;
    a.p.f.first = first;
    a.p.f.w = wavelet + (kk - 1);
    a.p.f.rows = slots ? w.rows : nullptr;
    a.p.f.row_slot = row_slot;
    a.p.f.slots = slots;
    a.p.src = src_zx;
    a.p.B = (int)B;
    a.p.sp = make_split(Region{core.z0, core.z1, core.x0, core.x1}, T, pl.vx_a, pl.rows_a,
                        (int)std::min<int64_t>(B, kShotGroup));
    a.p.g = g;
    a.p.k = k;
    a.p.rebuild_last = true;
    a.per = (int)((split_blocks(a.p.sp, B) + kXcds - 1) / kXcds);
    if (slots > 0) {
      const Sources so{w.rows, w.head, w.next, R, w.row_cells, rec_grad + (kk - 1) * R, T,
                       aux_blocks(w.row_cells)};
      k_sources<<<so.blocks, kThreads, 0, s>>>(so);
      SEIS_CHECK_LAUNCH();
    }
    SEIS_PROF(SEIS_KERNEL_HABC_BWD, s);
    SEIS_CORE_LAUNCH(k_core_adj, T, pl.vx_a, a, s);
    first = false;
    for (int t = 1; t <= T; ++t) {
      const int64_t kt = kk - t + 1;
      const int recon = kt >= 3 ? 1 : 2;
      const Deep dp = shrunk(core, T - t);
      const Frame fr = make_frame(g, dp, (G + ngf - 1) / ngf, true);
      const TileMap tmb = band_tiles(g, dp, kBandVX, (G + ngb - 1) / ngb);
      const TileMap tms = side_tiles(g, dp, (G + ngb - 1) / ngb);
      const dim3 grid((fr.per + tmb.per + tms.per) * kXcds);
      if (U[t - 1] == U[t + 1])
        SEIS_HABC_LAUNCH(k_frame_adj_in, S, grid, s, vp, b, L[t], L[t - 1], L[t + 1], U[t],
                         U[t - 1], nullptr, grad_part, src_zx, wavelet + (kt - 1), recon, (int)B,
                         hc, k, dp, fr, ngf, G, tmb, ngb, tms);
      else
        SEIS_HABC_LAUNCH(k_frame_adj_out, S, grid, s, vp, b, L[t], L[t - 1], L[t + 1], U[t],
                         U[t - 1], U[t + 1], grad_part, src_zx, wavelet + (kt - 1), recon, (int)B,
                         hc, k, dp, fr, ngf, G, tmb, ngb, tms);
      const int64_t items = R + B * ring_len;
      const float* slot = recon == 1 ? ring + (kt - 3) * B * ring_len : nullptr;
      k_frame_post<<<nblk(items), 256, 0, s>>>(vp, U[t], U[t + 1], L[t + 1], grad_part, rec_flat,
                                               R ? rec_grad + (kt - 1) * R : nullptr, R, slot,
                                               ring_len, recon, (int)B, S, g, k, dp);
      SEIS_CHECK_LAUNCH();
    }
    SEIS_PROF(SEIS_KERNEL_HABC_BWD, s);
    if (spare) lfree.push_back(spare);
    lfree.push_back(M2);
    ufree.push_back(Y);
    if (T >= 2) {
      lfree.push_back(M1);
      ufree.push_back(X);
    }
    M2 = T >= 2 ? L[T] : M1;
    Y = T >= 2 ? U[T] : X;
    M1 = L[T + 1];
    X = U[T + 1];
    kk -= T;
    if (m > 0 && kk == m + 1) {  // (u^{k-1}, u^k) = (u^m, u^{m+1}) from storage
      const float* sp = snaps + (m / snap_every - 1) * 2 * field;
      k_habc_copy2<<<nblk(field), 256, 0, s>>>(sp, X, sp + field, Y, field);
      SEIS_CHECK_LAUNCH();
    }
  }
  k_core_grad<<<nblk(g.plane), 256, 0, s>>>(vp, grad_core, first ? 0 : (int)B, grad_part, G, grad,
                                            core, g, k);
  SEIS_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
