// The elastic forward loop on time-skewed marching waves: up to three time
// steps per launch, all five fields crossing HBM once for them.
//
// Layout as march.h: one wave owns a strip of columns and marches down a segment
// of rows of one shot; all rows in flight live in registers, x-neighbours come
// from the adjacent lanes.  At march row z, level t = 1..T (state n + t) takes row
// r = z - t: the stresses of r (which need vz of r + 1 and vx of r - 1, r, a level
// below), vz of r (tzz of r - 1, r, txz of r) and vx of r - 1 (txz of r - 1, r).
// With vx one row behind, the next level finds what it needs in the same march row,
// so that a level costs one row and one cell of halo.  Every value has the operands
// and order of the one-step kernels (k_el_T, k_el_V) and is bit-identical.
#include "common.h"
#include "march.h"
#include "march_rows.h"
#include "seistorch_amd.h"
#include "tiles.h"

#include <algorithm>
#include <vector>

using seis::Grid;

namespace {

enum { kL2M = 0, kLam, kMc, kRc, kAinv, kBm, kNumCoef };
enum { kVx = 0, kVz, kTxx, kTzz, kTxz, kNumFields };

constexpr int kElMaxT = 3;

struct ElParams {
  const float* coef;  // kNumCoef planes
  const float* in[kNumFields];
  float* out[kNumFields];
  const float* w;  // wavelet samples from n on
  const int32_t* src;  // (B, 2)
  int src_mask, rec_mask;  // fields with sources, with receivers
  float* ring;  // slot of state n + 1 (5 x B x ring_len), or null
  int64_t ring_len, ring_step;
  int ring_levels;
  float* rows;  // receiver rows of the T levels, (T, 5, slots, B, nx), or null
  const int32_t* row_slot;
  int slots, B;
  float dti;
  Split sp;
  Grid g;
};

// Level t's values of field f on row r: into the receivers' row and the ring row.
template <int VX>
__device__ __forceinline__ void keep_row(Const<ElParams> p, int b, const Lane& l, int t, int f,
                                         int r, const float (&V)[VX]) {
  const int npml = p->g.npml, ztop = p->g.ztop, nx = p->g.nx;
  const int zbot = p->g.nz - 1 - npml, xr = nx - 1 - npml;
  if (t <= p->ring_levels && (r == ztop || r == zbot)) {
    float* q = p->ring + (t - 1) * p->ring_step + ((int64_t)f * p->B + b) * p->ring_len +
               (r == zbot && ztop >= 0 ? nx - 2 * npml - 2 : 0) - npml - 1;
#pragma unroll
    for (int e = 0; e < VX; ++e)
      if (l.x0 + e > npml && l.x0 + e < xr) q[l.x0 + e] = V[e];
  }
  if (p->rows && ((p->rec_mask >> f) & 1)) {
    const int slot = scalar_at(p->row_slot, r);
    if (slot >= 0) {
      float* q = p->rows +
                 ((((int64_t)(t - 1) * kNumFields + f) * p->slots + slot) * p->B + b) * nx + l.x0;
#pragma unroll
      for (int e = 0; e < VX; ++e) q[e] = V[e];
    }
  }
}

// A source row, a ring row or a receivers' row: adds level t's source sample to
// the fields from f0 on (r is their row) and keeps what is wanted of them.
template <int N, int VX>
__device__ __forceinline__ void el_special(Const<ElParams> p0, int b, const Lane& l, int t, int f0,
                                           int r, int z0, int z1, float (&V)[N][VX]) {
  const Const<ElParams> p = cold(p0);
  const int sz = scalar_at(p->src, 2 * b), sx = scalar_at(p->src, 2 * b + 1);
  if (r == sz) {
    const float w = scalar_at(p->w, t - 1);
#pragma unroll
    for (int i = 0; i < N; ++i)
      if ((p->src_mask >> (f0 + i)) & 1) {
#pragma unroll
        for (int e = 0; e < VX; ++e)
          if (l.x0 + e == sx) V[i][e] += w;
      }
  }
  if (r < z0 || r >= z1 || !l.inner) return;
#pragma unroll
  for (int i = 0; i < N; ++i) keep_row<VX>(p, b, l, t, f0 + i, r, V[i]);
}

// EDGE: the strip (its halo included) reaches the grid's border, where the
// differences end.  RINGCOLS: it holds one of the ring's columns.
template <int T, int VX, bool EDGE, bool RINGCOLS>
__device__ __forceinline__ void el_march_strip(const ElParams& p, Const<ElParams> pc, int b,
                                               int strip, int seg) {
  constexpr int kAhead = kRowsAhead;
  const Lane l = make_lane<T, VX>(strip, p.sp, p.g.nx);
  const int64_t plane = p.g.plane, off = (int64_t)b * plane;
  const int nz = p.g.nz;
  const int z0 = seg * p.sp.rows, z1 = min(z0 + p.sp.rows, nz);  // owned rows
  const int zs = z0 - T;
  Buf I[kNumFields], O[kNumFields];
#pragma unroll
  for (int f = 0; f < kNumFields; ++f) {
    I[f] = make_buf(p.in[f] + off, plane);
    O[f] = make_buf(p.out[f] + off, plane);
  }
  // the coefficients as one buffer; rows outside the grid (whose values reach no
  // cell inside it) may read another plane's
  const Buf CF = make_buf(p.coef, kNumCoef * plane);
  const uint32_t pitch = (uint32_t)p.g.nx * 4u, cplane = (uint32_t)plane * 4u;
  const float dti = p.dti;
  const int sz = scalar_at(p.src, 2 * b);
  const int rt = p.ring ? p.g.ztop : -1, rb = p.ring ? nz - 1 - p.g.npml : -1;
  const int32_t* row_slot = p.rows ? p.row_slot : nullptr;
  bool xl0[VX], xr0[VX];  // EDGE: there is a left / right neighbour
#pragma unroll
  for (int e = 0; e < VX; ++e) {
    xl0[e] = !EDGE || l.x0 + e > 0;
    xr0[e] = !EDGE || l.x0 + e < p.g.nx - 1;
  }
  // the lane's ring column (at most one): offset of its row 0 in a field's ring
  const uint32_t rlen = (uint32_t)p.ring_len * 4u, rstep = (uint32_t)p.ring_step * 4u;
  const Buf RG = RINGCOLS ? make_buf(p.ring + (int64_t)b * p.ring_len,
                                     (p.ring_levels - 1) * p.ring_step +
                                         (int64_t)(kNumFields - 1) * p.B * p.ring_len + p.ring_len)
                          : CF;
  uint32_t rcol = kLaneOut;
  int re = 0;
  const int rlo = max(z0, p.g.ztop + 1), rn = max(min(z1, nz - 1 - p.g.npml) - rlo, 0);
  const int rlev = p.ring_levels;
  if constexpr (RINGCOLS) {
    const int npml = p.g.npml, xr = p.g.nx - 1 - npml, nxi = p.g.nx - 2 * npml - 2;
    const int ztop = p.g.ztop, zbot = nz - 1 - npml;
#pragma unroll
    for (int e = 0; e < VX; ++e) {
      const int x = l.x0 + e;
      if (l.inner && (x == npml || x == xr)) {
        re = e;
        rcol = 4u * (uint32_t)((ztop >= 0 ? 2 * nxi : nxi) + (x == xr ? zbot - ztop - 1 : 0) -
                               (ztop + 1));
      }
    }
  }
  auto ring_column = [&](int t, int f, int r, const float (&V)[VX]) {
    float v[1] = {V[0]};
#pragma unroll
    for (int e = 1; e < VX; ++e) v[0] = re == e ? V[e] : v[0];
    const uint32_t ro = row_offset(r, rlo, t <= rlev ? rn : 0, 4u);
    if (ro != kRowOut) buf_store<1>(RG, rcol + ro + (t - 1) * rstep + f * (uint32_t)p.B * rlen, v);
  };
  uint32_t marked = 0;  // bit t - 1: row z - t needs el_special
  int next_slot = row_slot ? scalar_at(row_slot, min(max(zs, 0), nz - 1)) : -1;
  // row z - k at index (z - zs - k) mod 4; level t's fields (stresses without the
  // level's source, as stage V takes them)
  float W[T][2][4][VX], S[T + 1][3][4][VX], c[kNumCoef][4][VX];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int e = 0; e < VX; ++e) {
#pragma unroll
      for (int t = 0; t < T; ++t) W[t][0][q][e] = W[t][1][q][e] = 0.0f;
#pragma unroll
      for (int t = 0; t <= T; ++t) S[t][0][q][e] = S[t][1][q][e] = S[t][2][q][e] = 0.0f;
#pragma unroll
      for (int k = 0; k < kNumCoef; ++k) c[k][q][e] = 0.0f;
    }
  // loads run kAhead rows ahead: set i holds what march row z consumes (row z of
  // vz, row z - 1 of the others and of the coefficients), z = i mod kAhead
  float nF[kAhead][kNumFields][VX], nC[kAhead][kNumCoef][VX];
  uint32_t zo = l.in + (uint32_t)zs * pitch;
  auto fetch = [&](int i) {
#pragma unroll
    for (int f = 0; f < kNumFields; ++f) buf_load<VX>(I[f], f == kVz ? zo : zo - pitch, nF[i][f]);
#pragma unroll
    for (int k = 0; k < kNumCoef; ++k) buf_load<VX>(CF, zo - pitch + k * cplane, nC[i][k]);
    zo += pitch;
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch(i);
  for (int z4 = zs; z4 < z1 + T + 1; z4 += 4) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int z = z4 + q, qa = q % kAhead;
#pragma unroll
      for (int e = 0; e < VX; ++e) {
        W[0][1][q][e] = nF[qa][kVz][e];
        W[0][0][(q + 3) & 3][e] = nF[qa][kVx][e];
#pragma unroll
        for (int i = 0; i < 3; ++i) S[0][i][(q + 3) & 3][e] = nF[qa][kTxx + i][e];
#pragma unroll
        for (int k = 0; k < kNumCoef; ++k) c[k][(q + 3) & 3][e] = nC[qa][k][e];
      }
      fetch(qa);
      const int slot = next_slot;
      if (row_slot) next_slot = scalar_at(row_slot, min(max(z + 1, 0), nz - 1));
#pragma unroll
      for (int t = 1; t <= T; ++t) {
        const int r = z - t, s = (q - t) & 3, su = (q - t - 1) & 3, sd = (q - t + 1) & 3;
        const float(&vx0)[VX] = W[t - 1][0][s];
        const float(&vxu)[VX] = W[t - 1][0][su];
        const float(&vz0)[VX] = W[t - 1][1][s];
        const float(&vzd)[VX] = W[t - 1][1][sd];
        const bool zl = !EDGE || r > 0, zr = !EDGE || r < nz - 1, zru = !EDGE || r - 1 < nz - 1;
        // the stresses of row r from the state below, its sources included
        float P[3][VX];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int e = 0; e < VX; ++e) P[i][e] = S[t - 1][i][s][e];
        if (t > 1 && __builtin_expect(r == sz, 0)) {
          const Const<ElParams> k = cold(pc);
          const int sx = scalar_at(k->src, 2 * b + 1);
          const float w = scalar_at(k->w, t - 2);
#pragma unroll
          for (int i = 0; i < 3; ++i)
            if ((k->src_mask >> (kTxx + i)) & 1) {
#pragma unroll
              for (int e = 0; e < VX; ++e)
                if (l.x0 + e == sx) P[i][e] += w;
            }
        }
        const float vxl = from_left(vx0[VX - 1]), vzr = from_right(vz0[0]);
        float N[3][VX];
#pragma unroll
        for (int e = 0; e < VX; ++e) {
          const float a = c[kAinv][s][e], bm = c[kBm][s][e];
          const float l2m = c[kL2M][s][e], lam = c[kLam][s][e], mc = c[kMc][s][e];
          const float dxv = vx0[e] - (e == 0 ? vxl : vx0[e == 0 ? 0 : e - 1]);
          const float dxz = (e == VX - 1 ? vzr : vz0[e == VX - 1 ? e : e + 1]) - vz0[e];
          const float vx_x = xl0[e] ? dxv : 0.0f;
          const float vz_z = zr ? vzd[e] - vz0[e] : 0.0f;
          const float vx_z = zl ? vx0[e] - vxu[e] : 0.0f;
          const float vz_x = xr0[e] ? dxz : 0.0f;
          N[0][e] = a * (dti * (l2m * vx_x + lam * vz_z) + bm * P[0][e]);
          N[1][e] = a * (dti * (l2m * vz_z + lam * vx_x) + bm * P[1][e]);
          N[2][e] = a * (mc * (vz_x + vx_z) + bm * P[2][e]);
        }
        const float(&txxu)[VX] = S[t][0][su];
        const float(&tzzu)[VX] = S[t][1][su];
        const float(&txzu)[VX] = S[t][2][su];
        const float txzl = from_left(N[2][VX - 1]), txxr = from_right(txxu[0]);
        float Vz[1][VX], Vx[1][VX];
#pragma unroll
        for (int e = 0; e < VX; ++e) {
          const float dxt = N[2][e] - (e == 0 ? txzl : N[2][e == 0 ? 0 : e - 1]);
          const float dxx = (e == VX - 1 ? txxr : txxu[e == VX - 1 ? e : e + 1]) - txxu[e];
          const float txz_x = xl0[e] ? dxt : 0.0f;
          const float tzz_z = zl ? N[1][e] - tzzu[e] : 0.0f;
          const float txx_x = xr0[e] ? dxx : 0.0f;
          const float txz_z = zru ? N[2][e] - txzu[e] : 0.0f;
          Vz[0][e] = c[kAinv][s][e] *
                     (c[kRc][s][e] * (txz_x + tzz_z) + c[kBm][s][e] * vz0[e]);
          Vx[0][e] = c[kAinv][su][e] *
                     (c[kRc][su][e] * (txx_x + txz_z) + c[kBm][su][e] * vxu[e]);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int e = 0; e < VX; ++e) S[t][i][s][e] = N[i][e];
        if (__builtin_expect((marked >> (t - 1)) & 1u, 0)) {
          el_special<1, VX>(pc, b, l, t, kVz, r, z0, z1, Vz);
          el_special<3, VX>(pc, b, l, t, kTxx, r, z0, z1, N);
        }
        if (__builtin_expect((marked >> t) & 1u, 0))
          el_special<1, VX>(pc, b, l, t, kVx, r - 1, z0, z1, Vx);
        if constexpr (RINGCOLS) {
          ring_column(t, kVz, r, Vz[0]);
#pragma unroll
          for (int i = 0; i < 3; ++i) ring_column(t, kTxx + i, r, N[i]);
          ring_column(t, kVx, r - 1, Vx[0]);
        }
        if (t < T) {
#pragma unroll
          for (int e = 0; e < VX; ++e) {
            W[t < T ? t : 0][1][s][e] = Vz[0][e];
            W[t < T ? t : 0][0][su][e] = Vx[0][e];
          }
        } else {
          const uint32_t ro = l.out + row_offset(r, z0, z1 - z0, pitch);
          buf_store<VX>(O[kVz], ro, Vz[0]);
#pragma unroll
          for (int i = 0; i < 3; ++i) buf_store<VX>(O[kTxx + i], ro, N[i]);
          buf_store<VX>(O[kVx], l.out + row_offset(r - 1, z0, z1 - z0, pitch), Vx[0]);
        }
      }
      marked = (marked << 1) | (z == sz || z == rt || z == rb || slot >= 0 ? 1u : 0u);
    }
  }
}

template <int T, int VX>
__device__ __forceinline__ void el_march(const ElParams& p, Const<ElParams> pc, int b, int strip,
                                         int seg) {
  const int xa = strip * out_cols(T, VX), xb = xa + out_cols(T, VX);
  const int xl = p.g.npml, xr = p.g.nx - 1 - p.g.npml, halo = halo_lanes(T, VX) * VX;
  const int z0 = seg * p.sp.rows, z1 = min(z0 + p.sp.rows, p.g.nz);
  const bool cols = p.ring && ((xa <= xl && xl < xb) || (xa <= xr && xr < xb));
  const bool edge = xa <= halo || xb + halo >= p.g.nx || z0 <= T || z1 + T + 1 >= p.g.nz;
  if (cols) el_march_strip<T, VX, true, true>(p, pc, b, strip, seg);
  else if (edge) el_march_strip<T, VX, true, false>(p, pc, b, strip, seg);
  else el_march_strip<T, VX, false, false>(p, pc, b, strip, seg);
}

// Records of the previous launch's levels, as blocks after the march's.
struct ElGather {
  const float* rows;
  const int64_t* cell;
  const int32_t* field;  // per channel
  int64_t R, row_cells;  // row_cells: of one field
  float* rec;
  int nch, levels, blocks;
};

__device__ __forceinline__ void el_gather(const ElGather& ga, int block) {
  const int64_t per = ga.R * ga.nch, n = per * ga.levels;
  for (int64_t i = (int64_t)block * kThreads + threadIdx.x; i < n;
       i += (int64_t)ga.blocks * kThreads) {
    const int64_t lev = i / per, t = i - lev * per, r = t / ga.nch;
    const int f = ga.field[t - r * ga.nch];
    ga.rec[i] = ga.rows[(lev * kNumFields + f) * ga.row_cells + ga.cell[r]];
  }
}

__global__ __launch_bounds__(kThreads) void k_el_gather(ElGather ga) {
  el_gather(ga, blockIdx.x);
}

struct ElLaunch {
  ElParams p;
  ElGather ga;
  int per;
};

template <int T, int VX>
__global__ __launch_bounds__(kThreads) void k_el_march(ElLaunch a) {
  if ((int)blockIdx.x >= a.per * kXcds) {
    el_gather(a.ga, (int)blockIdx.x - a.per * kXcds);
    return;
  }
  int strip, seg, b;
  if (!march_unit(a.p.sp, a.p.B, xcd_block(a.per), strip, seg, b)) return;
  el_march<T, VX>(a.p, launch_params<ElParams>(), b, strip, seg);
}

int launch_el(int T, int VX, const ElParams& p, const ElGather& ga, hipStream_t s) {
  const int64_t blocks = split_blocks(p.sp, p.B);
  const int per = (int)((blocks + kXcds - 1) / kXcds);
  const unsigned grid = (unsigned)(per * kXcds + ga.blocks);
  const ElLaunch a{p, ga, per};
  switch (T * 8 + VX) {
#define SEIS_F(T_, V_)                                    \
  case T_ * 8 + V_:                                       \
    k_el_march<T_, V_><<<grid, kThreads, 0, s>>>(a);      \
    break;
    SEIS_F(1, 1) SEIS_F(1, 2) SEIS_F(2, 1) SEIS_F(2, 2) SEIS_F(3, 1) SEIS_F(3, 2)
#undef SEIS_F
    default:
      seis::set_error("unsupported march shape (%d steps, vec_x %d)", T, VX);
      return 1;
  }
  SEIS_CHECK_LAUNCH();
  return 0;
}

struct ElWork {
  float* rows[2];
  int64_t* cell;
  int64_t row_cells, total;
};

ElWork carve_el(float* base, int64_t B, int64_t nx, int64_t slots, int64_t R) {
  ElWork w;
  w.row_cells = slots * B * nx;
  const int64_t rows = pad64(kElMaxT * kNumFields * w.row_cells);
  w.rows[0] = base;
  w.rows[1] = base + rows;
  w.cell = reinterpret_cast<int64_t*>(base + 2 * rows);
  w.total = 2 * rows + pad64(2 * R);
  return w;
}

// Launch shape; 0 = automatic.  Three steps per launch at every size (two were
// slower throughout; four would need the coefficients of five rows).  Short segments
// give the most waves, long ones recompute least.  us per step with segments of 4 / 8 /
// 12 / 16 rows, one cell per lane:
//   0.03 10^6 cells, 164 x 164 x 1 shot 5.0 / 6.3 / 7.2 / 8.0; 0.6, 300 x 500 x 4 6.9 / 7.3 /
//   8.2 / 9.1;
//   0.9, 800 x 1100 x 1 8.6 / 8.0 / 8.4 / 9.2; 300 x 500 x 6 7.8 / 7.6 / 8.3 / 9.1; 1.2, 300 x
//   500 x 8 10.3 / 8.2 / 9.1 / 9.1; 1.3, 700 x 900 x 2 10.3 / 8.9 / 9.7 / 9.2;
//   1.5, 500 x 601 x 5 12.2 / 10.9 / 10.9 / 10.4; 1.6, 451 x 877 x 4 13.4 / 11.9 / 11.8 / 10.9;
//   1.8, 600 x 1000 x 3 12.9 / 10.1 / 11.1 / 10.6; 1200 x 1500 x 1 13.0 / 11.3 / 10.7 / 10.1; 300
//   x 500 x 12 16.5 / 12.3 / 11.3 / 12.4; 1.7, 164 x 164 x 64 14.2 / 9.7 / 9.7 / 10.7;
//   2.4, 300 x 500 x 16 16.9 / 12.6 / 11.5 / 12.6; 2.7, 900 x 1500 x 2 17.4 / 13.2 / 12.3 / 11.8;
//   4.0, 500 x 1000 x 8 24 / 17.3 / 16.6 / 17.5; 4.3, 900 x 1200 x 4 26 / 18.7 / 17.4 / 16.5;
// and with 12 / 32 rows, 32 with two cells per lane: 4.9, 1300 x 1900 x 2 23.3 / 22.6, 27.5;
// 5.8, 800 x 900 x 8 22.9 / 24.4, 25.4; 7.2, 1200 x 1501 x 4 39.8 / 34.4; 700 x 1900 x 8 50.1,
// 46.9 (32 rows); 900 x 2500 x 16 171, 154.  The last two are bound by HBM (40 bytes per
// cell and launch, 29 us per step at the rate of a large copy for 700 x 1900 x 8) and by
// the issue of vector instructions; one step per launch, with launches for sources and
// records, took 21 us at 451 x 877 x 4 and 116 us at 700 x 1900 x 8.
struct ElShape {
  int vx, rows;
};

ElShape el_shape(int64_t n, int64_t nx, int32_t vec_x, int32_t rows) {
  ElShape s{1, 32};
  if (n < 750000) s.rows = 4;
  else if (n < 1400000) s.rows = 8;
  else if (n < 2000000) s.rows = 16;
  else if (n < 5000000) s.rows = 12;
  else if (nx % 2 == 0) s.vx = 2;
  if (vec_x) s.vx = vec_x;
  if (rows) s.rows = rows;
  return s;
}

// A launch's offsets in bytes stay below kRowOut (rings of its levels) and below
// kLaneOut (the coefficient planes).
constexpr int64_t kElCells = (int64_t)1 << 26;
constexpr int64_t kElRing = (int64_t)1 << 25;

}  // namespace

extern "C" {

int64_t seis_elastic_march_workspace(int64_t B, int64_t nx, int32_t slots, int64_t R) {
  return carve_el(nullptr, B, nx, slots, R).total;
}

int seis_elastic_march_forward(const float* coef, const float* wavelet, int64_t nt,
                               const int32_t* src_zx, int32_t src_mask, const int64_t* rec_flat,
                               int64_t R, const int32_t* rec_field, int32_t rec_mask, int32_t nch,
                               const int32_t* row_slot, int32_t slots, float* rec_out, float* ring,
                               float* snaps, int32_t snap_every, float* work,
                               float* const* fields, float* const* scratch, int64_t B, int64_t nz,
                               int64_t nx, float dt, float h, int32_t npml, int32_t multiple,
                               int32_t steps, int32_t vec_x, int32_t rows, void* stream) {
  SEIS_CHECK_ARG(B >= 1 && B <= 65535, "batch size %lld outside [1, 65535]", (long long)B);
  SEIS_CHECK_ARG(nz >= 2 && nx >= 2 && nz * nx <= kElCells, "grid %lld x %lld", (long long)nz,
                 (long long)nx);
  SEIS_CHECK_ARG(dt > 0.0f && h > 0.0f, "dt and h must be positive");
  SEIS_CHECK_ARG(coef && wavelet && src_zx && fields && scratch, "null pointer argument");
  for (int f = 0; f < kNumFields; ++f)
    SEIS_CHECK_ARG(fields[f] && scratch[f] && fields[f] != scratch[f], "bad field pointers");
  SEIS_CHECK_ARG(nt >= 1 && R >= 0 && R < (int64_t)1 << 31 && nch >= 1, "nt %lld, R %lld",
                 (long long)nt, (long long)R);
  SEIS_CHECK_ARG(R == 0 || (rec_flat && rec_field && rec_out && row_slot && slots > 0 && work),
                 "bad receiver arguments");
  SEIS_CHECK_ARG(npml >= 0 && slots >= 0 && slots <= nz, "npml %d, slots %d", npml, slots);
  SEIS_CHECK_ARG(steps >= 0 && steps <= kElMaxT, "steps %d outside [0, 3]", steps);
  SEIS_CHECK_ARG(vec_x >= 0 && vec_x <= 2 && (vec_x == 0 || nx % vec_x == 0),
                 "vec_x %d for nx = %lld", vec_x, (long long)nx);
  SEIS_CHECK_ARG(rows >= 0 && rows <= 1 << 20, "rows %d", rows);
  const int64_t ring_len = ring ? seis_ring_len(nz, nx, npml, multiple) : 0;
  SEIS_CHECK_ARG(!ring || ring_len > 0, "grid has no interior inside npml=%d", npml);
  SEIS_CHECK_ARG(kNumFields * B * ring_len <= kElRing, "too many shots for the ring (%lld)",
                 (long long)B);
  SEIS_CHECK_ARG(!snaps || snap_every > 0, "snapshots need snap_every > 0");
  const Grid g = seis::make_grid(nz, nx, npml, multiple != 0);
  const int64_t field = B * g.plane;
  hipStream_t s = (hipStream_t)stream;
  const int max_t = steps ? steps : kElMaxT;
  const ElShape sh = el_shape(B * nz * nx, nx, vec_x, rows);
  const int vx = sh.vx, rows_seg = sh.rows;
  const ElWork w = carve_el(work, B, nx, slots, R);
  if (R > 0) {
    k_row_cells<<<blocks_of(R), 256, 0, s>>>(rec_flat, R, g.plane, g.nx, (int)B, row_slot, w.cell,
                                             nullptr, nullptr);
    SEIS_CHECK_LAUNCH();
  }
  // launches end at snapshots; the output of each is the snapshot's slot or the
  // buffer set that leaves the last state in `fields`
  struct Step {
    int T;
    int64_t snap;  // snapshot index it writes, or -1
    bool in_fields;
  };
  std::vector<Step> plan;
  for (int64_t n = 0; n < nt;) {
    int64_t stop = nt;
    if (snaps) stop = std::min(nt, (n / snap_every + 1) * snap_every);
    const int T = (stop - n) % max_t ? (int)((stop - n) % max_t) : max_t;
    n += T;
    plan.push_back({T, snaps && n % snap_every == 0 && n <= nt - 1 ? n / snap_every - 1 : -1,
                    false});
  }
  bool set = true;
  for (size_t i = plan.size(); i-- > 0;) {
    plan[i].in_fields = set;
    set = plan[i].snap >= 0 ? true : !set;
  }
  float* cur[kNumFields];
  for (int f = 0; f < kNumFields; ++f) {
    cur[f] = set ? fields[f] : scratch[f];
    if (int e = zero(cur[f], field, s)) return e;
  }
  ElGather ga{nullptr, w.cell, rec_field, R, w.row_cells, nullptr, nch, 0, 0};
  int parity = 0;
  int64_t n = 0;
  for (const Step& st : plan) {
    ElParams p{};
    p.coef = coef;
    for (int f = 0; f < kNumFields; ++f) {
      p.in[f] = cur[f];
      p.out[f] = st.snap >= 0 ? snaps + (st.snap * kNumFields + f) * field
                 : st.in_fields ? fields[f] : scratch[f];
      cur[f] = p.out[f];
    }
    p.w = wavelet + n;
    p.src = src_zx;
    p.src_mask = src_mask;
    p.rec_mask = rec_mask;
    p.ring_levels = ring ? (int)std::min<int64_t>(st.T, nt - 1 - n) : 0;
    p.ring = p.ring_levels > 0 ? ring + n * kNumFields * B * ring_len : nullptr;
    p.ring_len = ring_len;
    p.ring_step = kNumFields * B * ring_len;
    p.rows = R > 0 ? w.rows[parity] : nullptr;
    p.row_slot = row_slot;
    p.slots = slots;
    p.B = (int)B;
    p.dti = dt * (1.0f / h);
    p.sp = make_split(g, st.T, vx, rows_seg, (int)std::min<int64_t>(B, 8));
    p.g = g;
    SEIS_PROF(SEIS_KERNEL_ELASTIC_FWD, s);
    if (int e = launch_el(st.T, vx, p, ga, s)) return e;
    SEIS_PROF(SEIS_KERNEL_ELASTIC_FWD, s);
    if (R > 0) {
      ga.rows = w.rows[parity];
      ga.rec = rec_out + n * R * nch;
      ga.levels = st.T;
      ga.blocks = aux_blocks(R * nch * st.T);
      parity ^= 1;
    }
    n += st.T;
  }
  if (ga.blocks > 0) {
    k_el_gather<<<ga.blocks, kThreads, 0, s>>>(ga);
    SEIS_CHECK_LAUNCH();
  }
  return 0;
}

}  // extern "C"
