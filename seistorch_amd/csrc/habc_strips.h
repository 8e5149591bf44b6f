// The boundary strips of the HABC step and of its adjoint, shared by the loops with
// one step per launch (habc.hip) and the marching ones (habc_march.hip): which
// strips a cell belongs to, their one-way terms, the frame around Deep.
#pragma once

#include "common.h"
#include "tiles.h"

#include <algorithm>
#include <cstddef>
#include <type_traits>

using seis::Grid;
using seis::lap_taps;
using seis::acoustic_update;
using seis::lap5;
using namespace seis::tiles;

namespace {

constexpr int kW = 50;

struct HabcCtx {
  Grid g;
  int multiple;
  float dt, h;
};

__device__ __forceinline__ bool m_top(int z, int x, const HabcCtx& c) {
  return !c.multiple && z < kW && x >= z && x <= c.g.nx - 1 - z;
}
__device__ __forceinline__ bool m_bottom(int z, int x, const HabcCtx& c) {
  const int i = c.g.nz - 1 - z;
  return z >= c.g.nz - kW && x >= i && x <= c.g.nx - 1 - i;
}
__device__ __forceinline__ bool m_left(int z, int x, const HabcCtx& c) {
  return x < kW && ((z >= x && z <= c.g.nz - 1 - x) || (c.multiple && z < kW));
}
__device__ __forceinline__ bool m_right(int z, int x, const HabcCtx& c) {
  const int i = c.g.nx - 1 - x;
  return x >= c.g.nx - kW && ((z >= i && z <= c.g.nz - 1 - i) || (c.multiple && z < kW));
}

// strip s: 0 top, 1 bottom, 2 left, 3 right
__device__ __forceinline__ int sdist(int s, int z, int x, const Grid& g) {
  return s == 0 ? z : s == 1 ? g.nz - 1 - z : s == 2 ? x : g.nx - 1 - x;
}
__device__ __forceinline__ int sstep(int s, const Grid& g) {
  return s == 0 ? g.nx : s == 1 ? -g.nx : s == 2 ? 1 : -1;
}
__device__ __forceinline__ int sedge(int s, int z, int x, const Grid& g) {
  return s == 0 ? x : s == 1 ? (g.nz - 1) * g.nx + x : s == 2 ? z * g.nx : z * g.nx + g.nx - 1;
}
__device__ __forceinline__ bool near_edge(int z, int x, const Grid& g, int margin) {
  return z < margin || z >= g.nz - margin || x < margin || x >= g.nx - margin;
}

struct OwCoef {
  float k0, k1, k2, k3, k4;
};

// one-way coefficients with the reference's FP32 order: l = 2*c*dt/dh,
// m = c**2*dt**2/(dh**2), (2-l-m), (l+2m), -m, (l-1), -l
__device__ __forceinline__ OwCoef ow_coef(float c, const HabcCtx& x) {
  const float lam = ((2.0f * c) * x.dt) / x.h;
  const float mu = ((c * c) * (x.dt * x.dt)) / (x.h * x.h);
  return OwCoef{(2.0f - lam) - mu, lam + 2.0f * mu, -mu, lam - 1.0f, -lam};
}

// blended strip value y_s at cell i (flat) for fields u, p
__device__ __forceinline__ float strip_value(int s, int z, int x, int i, const float* u,
                                             const float* p, const OwCoef& k, float b, float y,
                                             const Grid& g) {
  const int e = sstep(s, g);
  const float u2 = sdist(s, z, x, g) == kW - 1 ? u[sedge(s, z, x, g)] : u[i + 2 * e];
  const float t1 = k.k0 * u[i];
  const float t2 = k.k1 * u[i + e];
  const float t3 = k.k2 * u2;
  const float t4 = k.k3 * p[i];
  const float t5 = k.k4 * p[i + e];
  const float one = (((t1 + t2) + t3) + t4) + t5;
  return one * b + (1.0f - b) * y;
}

// Linear weights of the final assignment at a cell: value = alpha*y +
// sum_s beta_s*u1_s.
struct HabcW {
  float alpha;
  float beta[4];
};

__device__ __forceinline__ HabcW habc_weights(int z, int x, const HabcCtx& c, float b) {
  HabcW w{1.0f, {0.0f, 0.0f, 0.0f, 0.0f}};
  const Grid& g = c.g;
  if (!near_edge(z, x, g, kW)) return w;
  int last = -1;
  if (m_top(z, x, c)) last = 0;
  if (m_bottom(z, x, c)) last = 1;
  if (m_left(z, x, c)) last = 2;
  if (m_right(z, x, c)) last = 3;
  int d1 = -1, d2 = -1;
  if (!c.multiple && z < kW && x == z) { d1 = 0; d2 = 2; }
  if (!c.multiple && z < kW && x == g.nx - kW + z) { d1 = 0; d2 = 3; }
  if (z >= g.nz - kW && x == z - (g.nz - kW)) { d1 = 1; d2 = 2; }
  if (z >= g.nz - kW && x == g.nx - kW + (z - (g.nz - kW))) { d1 = 1; d2 = 3; }
  if (d1 >= 0) {
    w.alpha = 0.5f * (1.0f - b) + 0.5f * (1.0f - b);
    w.beta[d1] = 0.5f * b;
    w.beta[d2] = 0.5f * b;
  } else if (last >= 0) {
    w.alpha = 1.0f - b;
    w.beta[last] = b;
  }
  return w;
}

// Forward step for S shots per thread: out = HABC(u, p) (+ w at the source
// cells when src != nullptr).  Cells are 64 x 4 tiles in XCD-aware order.
// Cells z in [z0, z1), x in [x0, x1) handled by a vectorised launch (see
// k_habc_fwd_deep / k_habc_adj_deep); the per-cell kernels skip them.
struct Deep {
  int z0, z1, x0, x1;
};

__device__ __forceinline__ bool in_deep(int z, int x, const Deep& dp) {
  return z >= dp.z0 && z < dp.z1 && x >= dp.x0 && x < dp.x1;
}

// Most shot groups per thread of the adjoint's top and bottom bands.
constexpr int kBandGroups = 8;

// Cells per lane on the adjoint's bands: one, which divides every Deep lane
// width (Deep's column bounds are multiples of it).  Two and four cells per
// lane took 120 and 161 VGPRs in the fused kernel against 98.
constexpr int kBandVX = 1;

// Rows per thread of the vectorised adjoint on Deep in the fused kernel.  One: the deep and
// frame block ranges share one kernel, whose register count (and so the
// frame threads' occupancy) follows the larger branch; two rows per thread
// took 146 VGPRs against 91 and made the launch 20 % slower.
constexpr int kHabcRZ = 1;

// The cells outside Deep as up to four rectangles (top, bottom, left, right),
// tiled 64 x 4 each (one cell per thread) and numbered consecutively, so the
// per-cell launches only cover the strips.
struct Frame {
  int n;
  int z0[4], z1[4], x0[4], x1[4], ntx[4], ntz[4];
  int64_t t0[5];  // first global tile of each rectangle (prefix over the groups too)
  int groups, per;
};

// -> false if workgroup w (numbered within the frame's blocks) has no cell
__device__ __forceinline__ bool frame_cell(const Frame& f, int w, int& z, int& x, int& grp) {
  const int64_t t = (int64_t)(w % kXcds) * f.per + w / kXcds;
  if (t >= f.t0[f.n]) return false;
  int r = 0;
  while (r + 1 < f.n && t >= f.t0[r + 1]) ++r;
  const int64_t local = t - f.t0[r];
  const int tx = (int)(local % f.ntx[r]);
  const int tzi = (int)((local / f.ntx[r]) % f.ntz[r]);
  grp = (int)(local / ((int64_t)f.ntx[r] * f.ntz[r]));
  x = f.x0[r] + tx * kLanes + (int)(threadIdx.x % kLanes);
  z = f.z0[r] + tzi * kRowsOfThreads + (int)(threadIdx.x / kLanes);
  return x < f.x1[r] && z < f.z1[r];
}

template <int S>
__device__ __forceinline__ void habc_fwd_cell(int z, int x, int grp, const float* __restrict__ vp,
                                              const float* __restrict__ bw,
                                              const float* __restrict__ u,
                                              const float* __restrict__ p,
                                              float* __restrict__ out,
                                              const int32_t* __restrict__ src,
                                              const float* __restrict__ wn, int B,
                                              const HabcCtx& hc, const seis::TimeConsts& k,
                                              int ng = 1) {
  const Grid& g = hc.g;
  const int i = z * g.nx + x;
  const float c = vp[i];
  const float A0 = 1.0f / k.idt2;
  const float B0 = k.idt2;
  const bool edge = near_edge(z, x, g, kW);
  const float b = edge ? bw[i] : 0.0f;
  const OwCoef kc = ow_coef(c, hc);
  const bool mt = m_top(z, x, hc), mb = m_bottom(z, x, hc), ml = m_left(z, x, hc),
             mr = m_right(z, x, hc);
  int d1 = -1, d2 = -1;
  if (!hc.multiple && z < kW && x == z) { d1 = 0; d2 = 2; }
  if (!hc.multiple && z < kW && x == g.nx - kW + z) { d1 = 0; d2 = 3; }
  if (z >= g.nz - kW && x == z - (g.nz - kW)) { d1 = 1; d2 = 2; }
  if (z >= g.nz - kW && x == g.nx - kW + (z - (g.nz - kW))) { d1 = 1; d2 = 3; }
  const float w = src ? *wn : 0.0f;
  // groups grp .. grp+ng-1 of S shots
  const int b0 = grp * S, nb = min(S * ng, B - b0);
  for (int s = 0; s < nb; ++s) {
    const int bb = b0 + s;
    const int64_t off = (int64_t)bb * g.plane;
    const float* U = u + off;
    const float* P = p + off;
    const float L = lap5(U, z, x, i, g, k.ih2);
    const float y = acoustic_update(A0, B0, k.two_idt2, U[i], P[i], c * c, L);
    float v = y;
    if (edge) {
      if (mt) v = strip_value(0, z, x, i, U, P, kc, b, y, g);
      if (mb) v = strip_value(1, z, x, i, U, P, kc, b, y, g);
      if (ml) v = strip_value(2, z, x, i, U, P, kc, b, y, g);
      if (mr) v = strip_value(3, z, x, i, U, P, kc, b, y, g);
      if (d1 >= 0)
        v = 0.5f * strip_value(d1, z, x, i, U, P, kc, b, y, g) +
            0.5f * strip_value(d2, z, x, i, U, P, kc, b, y, g);
    }
    if (src && z == src[2 * bb] && x == src[2 * bb + 1]) v += w;
    out[off + i] = v;
  }
}

// The fused loop's HABC step in one launch of two block ranges: on Deep (at
// least kW cells from every edge, outside every strip) the undamped update
// only, vectorised over VX-cell lanes with the operands and order of
// k_habc_fwd's per-cell path (bit-identical); on the frame around Deep the
// per-cell step, one cell per thread.
template <int S, int VX>
__global__ __launch_bounds__(256) void k_habc_fwd_deep(const float* __restrict__ vp,
                                                       const float* __restrict__ u,
                                                       const float* __restrict__ p,
                                                       float* __restrict__ out,
                                                       const int32_t* __restrict__ src,
                                                       const float* __restrict__ wn, int B,
                                                       HabcCtx hc, seis::TimeConsts k, Deep dp,
                                                       TileMap tm, const float* __restrict__ bw,
                                                       Frame f, int ngf, int G) {
  // blocks [0, f.per*8) run the frame's cells, one cell per thread for all G
  // shot groups (the per-cell set-up once per step), the rest Deep's lane
  // vectors, so both kinds of work share the machine within one launch
  const int nf = f.per * kXcds;
  if ((int)blockIdx.x < nf) {
    int zc, xc, gc;
    if (frame_cell(f, (int)blockIdx.x, zc, xc, gc))
      habc_fwd_cell<S>(zc, xc, gc * ngf, vp, bw, u, p, out, src, wn, B, hc, k,
                       min(ngf, G - gc * ngf));
    return;
  }
  int tx, tzi, grp;
  if (!tile_of_w(tm, (int)blockIdx.x - nf, tx, tzi, grp)) return;
  const Grid& g = hc.g;
  const int x0 = dp.x0 + (tx * kLanes + (int)(threadIdx.x % kLanes)) * VX;
  const int z = dp.z0 + tzi * kRowsOfThreads + (int)(threadIdx.x / kLanes);
  if (x0 >= dp.x1 || z >= dp.z1) return;
  const int i = z * g.nx + x0;
  const float A0 = 1.0f / k.idt2;
  const float B0 = k.idt2;
  float c2[VX];
  vload<VX>(vp + i, c2);
#pragma unroll
  for (int e = 0; e < VX; ++e) c2[e] = c2[e] * c2[e];
  const float w = src ? *wn : 0.0f;
  const int b0 = grp * S, nb = min(S, B - b0);
  for (int s = 0; s < nb; ++s) {
    const int bb = b0 + s;
    const int64_t off = (int64_t)bb * g.plane;
    const float* U = u + off;
    float uu[VX], uup[VX], udn[VX], pp[VX], o[VX];
    vload<VX>(U + i, uu);
    vload<VX>(U + i - g.nx, uup);
    vload<VX>(U + i + g.nx, udn);
    vload<VX>(p + off + i, pp);
    const float ul = U[i - 1], ur = U[i + VX];
    const int sz = src ? src[2 * bb] : -1, sx = src ? src[2 * bb + 1] : -1;
#pragma unroll
    for (int e = 0; e < VX; ++e) {
      const float L = lap_taps(uup[e], e == 0 ? ul : uu[e - 1], uu[e],
                               e == VX - 1 ? ur : uu[e + 1], udn[e], k.ih2);
      float v = acoustic_update(A0, B0, k.two_idt2, uu[e], pp[e], c2[e], L);
      if (z == sz && x0 + e == sx) v += w;
      o[e] = v;
    }
    vstore<VX>(out + off + i, o);
  }
}

// One-way terms of the transposed strip blend that reach cell i: the strip
// cells n whose one-way stencil reads i, with the coefficients on u^n (c1)
// and on u^{n-1} (c2) times the blend weight beta of n.  At most 16.
__device__ __forceinline__ int oneway_terms(int z, int x, int i, const float* __restrict__ vp,
                                            const float* __restrict__ bw, const HabcCtx& hc,
                                            int* on, float* oc1, float* oc2) {
  const Grid& g = hc.g;
  int no = 0;
  for (int s = 0; s < 4; ++s) {
    const int dj = sdist(s, z, x, g);
    const int e = sstep(s, g);
    for (int m = 0; m < 3; ++m) {
      const int dn = dj - m;
      if (dn < 0 || dn > kW - 1 || (m == 2 && dn == kW - 1)) continue;
      const int n = i - m * e;
      const int nz_ = n / g.nx, nx_ = n - nz_ * g.nx;
      const float be = habc_weights(nz_, nx_, hc, bw[n]).beta[s];
      if (be == 0.0f) continue;
      const OwCoef kc = ow_coef(vp[n], hc);
      const float c1 = m == 0 ? kc.k0 : m == 1 ? kc.k1 : kc.k2;
      const float c2 = m == 0 ? kc.k3 : m == 1 ? kc.k4 : 0.0f;
      on[no] = n; oc1[no] = be * c1; oc2[no] = be * c2; ++no;
    }
    if (dj == 0) {  // the edge cell is the "+2" neighbour of the row-49 cell (roll wrap)
      const int n = i + (kW - 1) * e;
      const int nz_ = n / g.nx, nx_ = n - nz_ * g.nx;
      const float be = habc_weights(nz_, nx_, hc, bw[n]).beta[s];
      if (be != 0.0f) {
        on[no] = n; oc1[no] = be * ow_coef(vp[n], hc).k2; oc2[no] = 0.0f; ++no;
      }
    }
  }
  return no;
}

// u^k, and where the rebuilt u^{k-2} goes: over it, or into a field of its own.
struct TwoFields {
  const float* uc;
  float* uo;
};
template <bool SAME>
using Rebuild = std::conditional_t<SAME, float* __restrict__, TwoFields>;
__device__ __forceinline__ const float* u_old(const float* u) { return u; }
__device__ __forceinline__ const float* u_old(const TwoFields& u) { return u.uc; }
__device__ __forceinline__ float* u_new(float* u) { return u; }
__device__ __forceinline__ float* u_new(const TwoFields& u) { return u.uo; }

// Transpose of the step: out = H_u^T y1 + H_p^T y2 (either may be null).
// With recon/grad (fused adjoint, y1 = lambda^{k+1}, y2 = lambda^{k+2}):
// gradient 2c*A0*L(u^{k-1})*lambda^k on the interior (lambda^k without the
// adjoint source, which k_habc_post adds with its gradient share) and the
// interior rebuild of u^{k-2} from u^k (uc: SAME, over it).  recon: 0 none, 1
// rebuild, 2 zeros.
template <int S, bool SAME>
__device__ __forceinline__ void habc_adj_cell(
    int z, int x, int grp, const float* __restrict__ vp, const float* __restrict__ bw,
    const float* __restrict__ y1, const float* __restrict__ y2, float* __restrict__ out,
    const float* __restrict__ um, Rebuild<SAME> uc,
    float* __restrict__ gpart, const int32_t* __restrict__ src, const float* __restrict__ wn,
    int recon, int B, const HabcCtx& hc, const seis::TimeConsts& k, int ng = 1) {
  const Grid& g = hc.g;
  const int i = z * g.nx + x;
  const float A0 = 1.0f / k.idt2;
  const float B0 = k.idt2;
  const float c = vp[i];
  // undamped-stencil weights q(n) = c(n)^2*A0*alpha(n) at the cell and its neighbours
  const bool deep = !near_edge(z, x, g, kW + 3);
  auto qw = [&](int zz, int xx) {
    const int j = zz * g.nx + xx;
    const float cn = vp[j];
    const float al = deep ? 1.0f : habc_weights(zz, xx, hc, bw[j]).alpha;
    return (cn * cn) * A0 * al;
  };
  const float q0 = qw(z, x);
  const float qzm = z > 0 ? qw(z - 1, x) : 0.0f;
  const float qzp = z < g.nz - 1 ? qw(z + 1, x) : 0.0f;
  const float qxm = x > 0 ? qw(z, x - 1) : 0.0f;
  const float qxp = x < g.nx - 1 ? qw(z, x + 1) : 0.0f;
  const float al0 = deep ? 1.0f : habc_weights(z, x, hc, bw[i]).alpha;
  // one-way contributions: (flat offset, coefficient on y1, coefficient on y2)
  int on[16];
  float oc1[16], oc2[16];
  const int no = deep ? 0 : oneway_terms(z, x, i, vp, bw, hc, on, oc1, oc2);
  const bool in = interior(z, x, g);
  const float w = wn ? *wn : 0.0f;
  // groups grp .. grp+ng-1 of S shots, each with its own gradient partial
  for (int gi = grp; gi < grp + ng; ++gi) {
    float gacc = 0.0f;
    const int b0 = gi * S, nb = min(S, B - b0);
    for (int s = 0; s < nb; ++s) {
      const int bb = b0 + s;
      const int64_t off = (int64_t)bb * g.plane;
      float acc = 0.0f;
      if (y1) {
        const float* Y = y1 + off;
        const float Lq = lap_taps(z > 0 ? qzm * Y[i - g.nx] : 0.0f, x > 0 ? qxm * Y[i - 1] : 0.0f,
                                  q0 * Y[i], x < g.nx - 1 ? qxp * Y[i + 1] : 0.0f,
                                  z < g.nz - 1 ? qzp * Y[i + g.nx] : 0.0f, k.ih2);
        acc = (k.two_idt2 * (A0 * al0)) * Y[i] + Lq;
        for (int o = 0; o < no; ++o) acc += oc1[o] * Y[on[o]];
      }
      if (y2) {
        const float* Y = y2 + off;
        acc += -(B0 * (A0 * al0)) * Y[i];
        for (int o = 0; o < no; ++o) acc += oc2[o] * Y[on[o]];
      }
      out[off + i] = acc;
      if (in && recon >= 0 && um) {
        const float Lu = lap5(um + off, z, x, i, g, k.ih2);
        gacc += Lu * acc;
        if (recon == 1) {
          float un = u_old(uc)[off + i];
          if (z == src[2 * bb] && x == src[2 * bb + 1]) un -= w;
          u_new(uc)[off + i] = ((k.two_idt2 * um[off + i] + (c * c) * Lu) - un / A0) / B0;
        } else if (recon == 2) {
          u_new(uc)[off + i] = 0.0f;
        }
      }
    }
    if (in && um && gpart) gpart[(int64_t)gi * g.plane + i] += 2.0f * c * A0 * gacc;
  }
}

// The adjoint on the top and bottom bands: the rows outside Deep over Deep's
// columns (x0 >= kW+3 and x0+VB <= nx-kW-3).  There only the top (bottom)
// strip's one-way stencil reaches a cell: from the cells 0, 1 and 2 rows
// outward in its own column and, on the edge row, from strip row kW-1 (the
// roll wrap), and which of those four terms exist depends on the row alone.
// So a lane takes VB consecutive cells of one row, every access is a row
// vector, and each cell sums the same operands in the same order as
// habc_adj_cell (bit-identical).  TOP: the top band, else the bottom band.
template <int S, int VB, bool TOP, bool SAME>
__device__ __forceinline__ void habc_adj_band(
    int z, int x0, int grp, int ng, const float* __restrict__ vp, const float* __restrict__ bw,
    const float* __restrict__ y1, const float* __restrict__ y2, float* __restrict__ out,
    const float* __restrict__ um, Rebuild<SAME> uc,
    float* __restrict__ gpart, const int32_t* __restrict__ src, const float* __restrict__ wn,
    int recon, int B, const HabcCtx& hc, const seis::TimeConsts& k) {
  const Grid& g = hc.g;
  constexpr int st = TOP ? 0 : 1;  // the strip
  constexpr int er = TOP ? 1 : -1;  // its inward step in rows
  const int dj = TOP ? z : g.nz - 1 - z;
  const int i0 = z * g.nx + x0;
  const float A0 = 1.0f / k.idt2;
  const float B0 = k.idt2;
  // one-way term t reads row trow[t]: t = 0, 1, 2 the cells t rows outward
  // (their stencils reach this row through u, u[+e], u[+2e]), t = 3 the wrap
  bool tv[4];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const int dn = dj - m;
    tv[m] = !(dn < 0 || dn > kW - 1 || (m == 2 && dn == kW - 1));
  }
  tv[3] = dj == 0;
  const int trow[4] = {z, z - er, z - 2 * er, z + (kW - 1) * er};
  const bool hz = z > 0, hzp = z < g.nz - 1;
  auto qw = [&](int zz, int xx) {
    const int j = zz * g.nx + xx;
    const float cn = vp[j];
    return (cn * cn) * A0 * habc_weights(zz, xx, hc, bw[j]).alpha;
  };
  float q0[VB], qzm[VB], qzp[VB], qxm[VB], qxp[VB], al0[VB], c[VB];
  float oc1[4][VB], oc2[4][VB];
  bool on[4][VB];
  bool in[VB];
  bool allin = true, anyin = false;
#pragma unroll
  for (int e = 0; e < VB; ++e) {
    const int x = x0 + e;
    c[e] = vp[i0 + e];
    q0[e] = qw(z, x);
    qzm[e] = hz ? qw(z - 1, x) : 0.0f;
    qzp[e] = hzp ? qw(z + 1, x) : 0.0f;
    qxm[e] = qw(z, x - 1);
    qxp[e] = qw(z, x + 1);
    al0[e] = habc_weights(z, x, hc, bw[i0 + e]).alpha;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      on[t][e] = false;
      oc1[t][e] = 0.0f;
      oc2[t][e] = 0.0f;
      if (!tv[t]) continue;
      const int n = trow[t] * g.nx + x;
      const float be = habc_weights(trow[t], x, hc, bw[n]).beta[st];
      if (be == 0.0f) continue;
      const OwCoef kc = ow_coef(vp[n], hc);
      on[t][e] = true;
      oc1[t][e] = be * (t == 0 ? kc.k0 : t == 1 ? kc.k1 : kc.k2);
      oc2[t][e] = t == 0 ? be * kc.k3 : t == 1 ? be * kc.k4 : 0.0f;
    }
    in[e] = interior(z, x, g);
    allin = allin && in[e];
    anyin = anyin || in[e];
  }
  const float w = wn ? *wn : 0.0f;
  for (int gi = grp; gi < grp + ng; ++gi) {
    float gacc[VB];
    vzero<VB>(gacc);
    const int b0 = gi * S, nb = min(S, B - b0);
    for (int s = 0; s < nb; ++s) {
      const int bb = b0 + s;
      const int64_t off = (int64_t)bb * g.plane;
      const float* Y = y1 + off;
      const float* Y2 = y2 + off;
      float yc[VB], yzm[VB], yzp[VB], acc[VB];
      vload<VB>(Y + i0, yc);
      if (hz) vload<VB>(Y + i0 - g.nx, yzm); else vzero<VB>(yzm);
      if (hzp) vload<VB>(Y + i0 + g.nx, yzp); else vzero<VB>(yzp);
      const float yl = Y[i0 - 1], yr = Y[i0 + VB];
#pragma unroll
      for (int e = 0; e < VB; ++e) {
        const float Lq = lap_taps(hz ? qzm[e] * yzm[e] : 0.0f,
                                  qxm[e] * (e == 0 ? yl : yc[e - 1]), q0[e] * yc[e],
                                  qxp[e] * (e == VB - 1 ? yr : yc[e + 1]),
                                  hzp ? qzp[e] * yzp[e] : 0.0f, k.ih2);
        acc[e] = (k.two_idt2 * (A0 * al0[e])) * yc[e] + Lq;
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (!tv[t]) continue;
        float yt[VB];
        if (t == 0) {
#pragma unroll
          for (int e = 0; e < VB; ++e) yt[e] = yc[e];
        } else if (t == 1) {
#pragma unroll
          for (int e = 0; e < VB; ++e) yt[e] = TOP ? yzm[e] : yzp[e];
        } else {
          vload<VB>(Y + trow[t] * g.nx + x0, yt);
        }
#pragma unroll
        for (int e = 0; e < VB; ++e)
          if (on[t][e]) acc[e] += oc1[t][e] * yt[e];
      }
      float y2c[VB];
      vload<VB>(Y2 + i0, y2c);
#pragma unroll
      for (int e = 0; e < VB; ++e) acc[e] += -(B0 * (A0 * al0[e])) * y2c[e];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (!tv[t]) continue;
        float yt[VB];
        if (t == 0) {
#pragma unroll
          for (int e = 0; e < VB; ++e) yt[e] = y2c[e];
        } else {
          vload<VB>(Y2 + trow[t] * g.nx + x0, yt);
        }
#pragma unroll
        for (int e = 0; e < VB; ++e)
          if (on[t][e]) acc[e] += oc2[t][e] * yt[e];
      }
      vstore<VB>(out + off + i0, acc);
      if (anyin && recon >= 0) {
        const float* U = um + off;
        float u0[VB], uzm[VB], uzp[VB], un[VB];
        vload<VB>(U + i0, u0);
        if (hz) vload<VB>(U + i0 - g.nx, uzm); else vzero<VB>(uzm);
        if (hzp) vload<VB>(U + i0 + g.nx, uzp); else vzero<VB>(uzp);
        const float ul = U[i0 - 1], ur = U[i0 + VB];
        if (recon == 1) vload<VB>(u_old(uc) + off + i0, un);
        const int sz = src[2 * bb], sx = src[2 * bb + 1];
#pragma unroll
        for (int e = 0; e < VB; ++e) {
          if (!in[e]) continue;
          const float Lu = lap_taps(hz ? uzm[e] : 0.0f, e == 0 ? ul : u0[e - 1], u0[e],
                                    e == VB - 1 ? ur : u0[e + 1], hzp ? uzp[e] : 0.0f, k.ih2);
          gacc[e] += Lu * acc[e];
          if (recon == 1) {
            float v = un[e];
            if (z == sz && x0 + e == sx) v -= w;
            un[e] = ((k.two_idt2 * u0[e] + (c[e] * c[e]) * Lu) - v / A0) / B0;
          } else if (recon == 2) {
            un[e] = 0.0f;
          }
        }
        if (recon != 0) {
          if (allin) {
            vstore<VB>(u_new(uc) + off + i0, un);
          } else {
#pragma unroll
            for (int e = 0; e < VB; ++e)
              if (in[e]) u_new(uc)[off + i0 + e] = un[e];
          }
        }
      }
    }
    if (anyin) {
      float* gp = gpart + (int64_t)gi * g.plane + i0;
#pragma unroll
      for (int e = 0; e < VB; ++e)
        if (in[e]) gp[e] += 2.0f * c[e] * A0 * gacc[e];
    }
  }
}

// The adjoint on the left and right columns outside Deep, over Deep's rows
// (z in [kW+3, nz-kW-3)): only the left (right) strip's one-way stencil
// reaches a cell there, from the cells 0, 1 and 2 columns outward in its own
// row and, on the edge column, from strip column kW-1.  One cell per lane,
// lanes along x, so every term is a row access shifted by up to two cells;
// which terms exist depends on the column alone.  Same operands in the same
// order as habc_adj_cell (bit-identical).  LEFT: the left column, else the
// right one.
template <int S, bool LEFT, bool SAME>
__device__ __forceinline__ void habc_adj_side(
    int z, int x, int grp, int ng, const float* __restrict__ vp, const float* __restrict__ bw,
    const float* __restrict__ y1, const float* __restrict__ y2, float* __restrict__ out,
    const float* __restrict__ um, Rebuild<SAME> uc,
    float* __restrict__ gpart, const int32_t* __restrict__ src, const float* __restrict__ wn,
    int recon, int B, const HabcCtx& hc, const seis::TimeConsts& k) {
  const Grid& g = hc.g;
  constexpr int st = LEFT ? 2 : 3;  // the strip
  constexpr int ec = LEFT ? 1 : -1;  // its inward step in columns
  const int dj = LEFT ? x : g.nx - 1 - x;
  const int i = z * g.nx + x;
  const float A0 = 1.0f / k.idt2;
  const float B0 = k.idt2;
  bool tv[4];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const int dn = dj - m;
    tv[m] = !(dn < 0 || dn > kW - 1 || (m == 2 && dn == kW - 1));
  }
  tv[3] = dj == 0;
  const int toff[4] = {0, -ec, -2 * ec, (kW - 1) * ec};
  const bool hxm = x > 0, hxp = x < g.nx - 1;
  auto qw = [&](int zz, int xx) {
    const int j = zz * g.nx + xx;
    const float cn = vp[j];
    return (cn * cn) * A0 * habc_weights(zz, xx, hc, bw[j]).alpha;
  };
  const float c = vp[i];
  const float q0 = qw(z, x);
  const float qzm = qw(z - 1, x);
  const float qzp = qw(z + 1, x);
  const float qxm = hxm ? qw(z, x - 1) : 0.0f;
  const float qxp = hxp ? qw(z, x + 1) : 0.0f;
  const float al0 = habc_weights(z, x, hc, bw[i]).alpha;
  float oc1[4], oc2[4];
  bool on[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    on[t] = false;
    oc1[t] = 0.0f;
    oc2[t] = 0.0f;
    if (!tv[t]) continue;
    const int n = i + toff[t];
    const float be = habc_weights(z, x + toff[t], hc, bw[n]).beta[st];
    if (be == 0.0f) continue;
    const OwCoef kc = ow_coef(vp[n], hc);
    on[t] = true;
    oc1[t] = be * (t == 0 ? kc.k0 : t == 1 ? kc.k1 : kc.k2);
    oc2[t] = t == 0 ? be * kc.k3 : t == 1 ? be * kc.k4 : 0.0f;
  }
  const bool in = interior(z, x, g);
  const float w = wn ? *wn : 0.0f;
  for (int gi = grp; gi < grp + ng; ++gi) {
    float gacc = 0.0f;
    const int b0 = gi * S, nb = min(S, B - b0);
    for (int s = 0; s < nb; ++s) {
      const int bb = b0 + s;
      const int64_t off = (int64_t)bb * g.plane;
      const float* Y = y1 + off;
      const float* Y2 = y2 + off;
      const float yc = Y[i];
      const float yl = hxm ? Y[i - 1] : 0.0f;
      const float yr = hxp ? Y[i + 1] : 0.0f;
      const float Lq = lap_taps(qzm * Y[i - g.nx], hxm ? qxm * yl : 0.0f, q0 * yc,
                                hxp ? qxp * yr : 0.0f, qzp * Y[i + g.nx], k.ih2);
      float acc = (k.two_idt2 * (A0 * al0)) * yc + Lq;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (!on[t]) continue;
        const float yt = t == 0 ? yc : t == 1 ? (LEFT ? yl : yr) : Y[i + toff[t]];
        acc += oc1[t] * yt;
      }
      const float y2c = Y2[i];
      acc += -(B0 * (A0 * al0)) * y2c;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (!on[t]) continue;
        acc += oc2[t] * (t == 0 ? y2c : Y2[i + toff[t]]);
      }
      out[off + i] = acc;
      if (in && recon >= 0) {
        const float Lu = lap5(um + off, z, x, i, g, k.ih2);
        gacc += Lu * acc;
        if (recon == 1) {
          float un = u_old(uc)[off + i];
          if (z == src[2 * bb] && x == src[2 * bb + 1]) un -= w;
          u_new(uc)[off + i] = ((k.two_idt2 * um[off + i] + (c * c) * Lu) - un / A0) / B0;
        } else if (recon == 2) {
          u_new(uc)[off + i] = 0.0f;
        }
      }
    }
    if (in) gpart[(int64_t)gi * g.plane + i] += 2.0f * c * A0 * gacc;
  }
}

// The fused adjoint step in one launch of two block ranges.  One covers the
// rectangle Deep (z in [z0, z1), x in [x0, x1), at least kW+3
// cells from every edge, x0 and x1 multiples of VX): there no strip term
// reaches, so a lane runs a vectorised copy of the per-cell deep path of
// habc_adj_cell with the same operands in the same order (bit-identical).
// The other runs habc_adj_cell on every other cell, one cell per thread.
// Requires y1, y2, um and gpart (the fused loop's call).
// Block w of the strip ranges of the adjoint (-> false if w is past them):
// [0, f.per*8) the frame's cells (the four corners outside Deep's rows and
// columns), one cell per thread for ngf shot groups (the per-cell set-up once
// per ngf groups); the next tb.per*8 the top and bottom bands in lane vectors
// for ngb groups; the next ts.per*8 the left and right columns over Deep's
// rows, one cell per lane for ngb groups.
template <int S, bool SAME>
__device__ __forceinline__ bool habc_adj_strip_block(
    int w, const float* __restrict__ vp, const float* __restrict__ bw,
    const float* __restrict__ y1, const float* __restrict__ y2, float* __restrict__ out,
    const float* __restrict__ um, Rebuild<SAME> uc,
    float* __restrict__ gpart, const int32_t* __restrict__ src, const float* __restrict__ wn,
    int recon, int B, const HabcCtx& hc,
    const seis::TimeConsts& k, const Deep& dp, const Frame& f, int ngf, int G,
    const TileMap& tb, int ngb, const TileMap& ts) {
  const int nf = f.per * kXcds;
  const int nbnd = tb.per * kXcds;
  const int nsd = ts.per * kXcds;
  const Grid& g = hc.g;
  if (w < nf) {
    int zc, xc, gc;
    if (frame_cell(f, w, zc, xc, gc))
      habc_adj_cell<S, SAME>(zc, xc, gc * ngf, vp, bw, y1, y2, out, um, uc, gpart, src, wn,
                             recon, B, hc, k, min(ngf, G - gc * ngf));
    return true;
  }
  if (w < nf + nbnd) {
    int tx, tzi, gb;
    if (!tile_of_w(tb, w - nf, tx, tzi, gb)) return true;
    constexpr int VB = kBandVX;
    const int x0 = dp.x0 + (tx * kLanes + (int)(threadIdx.x % kLanes)) * VB;
    const int r = tzi * kRowsOfThreads + (int)(threadIdx.x / kLanes);
    const int ztop = dp.z0;  // rows [0, dp.z0) then [dp.z1, nz)
    if (x0 >= dp.x1 || r >= ztop + (g.nz - dp.z1)) return true;
    const int grp = gb * ngb, ng = min(ngb, G - grp);
    if (r < ztop)
      habc_adj_band<S, VB, true, SAME>(r, x0, grp, ng, vp, bw, y1, y2, out, um, uc, gpart,
                                       src, wn, recon, B, hc, k);
    else
      habc_adj_band<S, VB, false, SAME>(dp.z1 + (r - ztop), x0, grp, ng, vp, bw, y1, y2, out, um,
                                        uc, gpart, src, wn, recon, B, hc, k);
    return true;
  }
  if (w < nf + nbnd + nsd) {
    // side tiles: tx 0 the left column (x = lane), tx 1 the right one
    // (x = dp.x1 + lane); both are narrower than 64 cells
    int tx, tzi, gb;
    if (!tile_of_w(ts, w - nf - nbnd, tx, tzi, gb)) return true;
    const int lane = (int)(threadIdx.x % kLanes);
    const int z = dp.z0 + tzi * kRowsOfThreads + (int)(threadIdx.x / kLanes);
    const int x = tx == 0 ? lane : dp.x1 + lane;
    if (z >= dp.z1 || (tx == 0 ? x >= dp.x0 : x >= g.nx)) return true;
    const int grp = gb * ngb, ng = min(ngb, G - grp);
    if (tx == 0)
      habc_adj_side<S, true, SAME>(z, x, grp, ng, vp, bw, y1, y2, out, um, uc, gpart, src,
                                  wn, recon, B, hc, k);
    else
      habc_adj_side<S, false, SAME>(z, x, grp, ng, vp, bw, y1, y2, out, um, uc, gpart, src,
                                   wn, recon, B, hc, k);
    return true;
  }
  return false;
}

__global__ __launch_bounds__(256) void k_habc_fill(float* __restrict__ p, int64_t n) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0.0f;
}

__global__ __launch_bounds__(256) void k_habc_copy2(const float* __restrict__ a,
                                                    float* __restrict__ ao,
                                                    const float* __restrict__ b,
                                                    float* __restrict__ bo, int64_t n) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) {
    ao[t] = a[t];
    bo[t] = b[t];
  }
}

inline unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }

#define SEIS_HABC_LAUNCH(K, S, grid, s, ...)                      \
  do {                                                            \
    switch (S) {                                                  \
      case 1: K<1><<<grid, 256, 0, s>>>(__VA_ARGS__); break;     \
      case 2: K<2><<<grid, 256, 0, s>>>(__VA_ARGS__); break;     \
      case 4: K<4><<<grid, 256, 0, s>>>(__VA_ARGS__); break;     \
      default: K<8><<<grid, 256, 0, s>>>(__VA_ARGS__); break;    \
    }                                                             \
    SEIS_CHECK_LAUNCH();                                          \
  } while (0)

#define SEIS_HABC_VX(K, S_, VX_, grid, s, ...)                       \
  switch (VX_) {                                                      \
    case 1: K<S_, 1><<<grid, 256, 0, s>>>(__VA_ARGS__); break;       \
    case 2: K<S_, 2><<<grid, 256, 0, s>>>(__VA_ARGS__); break;       \
    default: K<S_, 4><<<grid, 256, 0, s>>>(__VA_ARGS__); break;      \
  }

#define SEIS_HABC_LAUNCH_V(K, S, VX, grid, s, ...)                   \
  do {                                                              \
    switch (S) {                                                    \
      case 1: SEIS_HABC_VX(K, 1, VX, grid, s, __VA_ARGS__) break;   \
      case 2: SEIS_HABC_VX(K, 2, VX, grid, s, __VA_ARGS__) break;   \
      case 4: SEIS_HABC_VX(K, 4, VX, grid, s, __VA_ARGS__) break;   \
      default: SEIS_HABC_VX(K, 8, VX, grid, s, __VA_ARGS__) break;  \
    }                                                               \
    SEIS_CHECK_LAUNCH();                                            \
  } while (0)

// The frame around dp (the whole grid if dp is empty) as rectangles of tiles;
// with corners_only, just the four corners outside dp's rows and columns (the
// bands over dp's columns go to band_tiles, the columns over dp's rows to
// side_tiles).
Frame make_frame(const Grid& g, const Deep& dp, int groups, bool corners_only = false) {
  Frame f{};
  auto add = [&](int z0, int z1, int x0, int x1) {
    if (z1 <= z0 || x1 <= x0) return;
    const int r = f.n++;
    f.z0[r] = z0; f.z1[r] = z1; f.x0[r] = x0; f.x1[r] = x1;
    f.ntx[r] = (x1 - x0 + kLanes - 1) / kLanes;
    f.ntz[r] = (z1 - z0 + kRowsOfThreads - 1) / kRowsOfThreads;
  };
  if (dp.z1 <= dp.z0 || dp.x1 <= dp.x0) {
    add(0, g.nz, 0, g.nx);
  } else if (corners_only) {
    add(0, dp.z0, 0, dp.x0);
    add(0, dp.z0, dp.x1, g.nx);
    add(dp.z1, g.nz, 0, dp.x0);
    add(dp.z1, g.nz, dp.x1, g.nx);
  } else {
    add(0, dp.z0, 0, g.nx);
    add(dp.z1, g.nz, 0, g.nx);
    add(dp.z0, dp.z1, 0, dp.x0);
    add(dp.z0, dp.z1, dp.x1, g.nx);
  }
  f.groups = groups;
  f.t0[0] = 0;
  for (int r = 0; r < f.n; ++r)
    f.t0[r + 1] = f.t0[r] + (int64_t)f.ntx[r] * f.ntz[r] * groups;
  for (int r = f.n + 1; r < 5; ++r) f.t0[r] = f.t0[f.n];
  f.per = (int)((f.t0[f.n] + kXcds - 1) / kXcds);
  return f;
}

// Tiles of the top and bottom bands of the adjoint (rows [0, dp.z0) and
// [dp.z1, nz) over dp's columns, stacked as one virtual grid of lane vectors
// of vx cells); no tiles if dp is empty.
TileMap band_tiles(const Grid& g, const Deep& dp, int vx, int groups) {
  if (dp.z1 <= dp.z0 || dp.x1 <= dp.x0) return TileMap{0, 0, 0, 0};
  const int rows = dp.z0 + (g.nz - dp.z1);
  const Grid gb{rows, dp.x1 - dp.x0, 0, (int64_t)rows * (dp.x1 - dp.x0)};
  return make_tiles(gb, vx, 1, groups);
}

// Tiles of the left and right columns of the adjoint (x in [0, dp.x0) and
// [dp.x1, nx) over dp's rows): one 64-lane tile column each (both are at
// most kW+3+3 cells wide); no tiles if dp is empty.
TileMap side_tiles(const Grid& g, const Deep& dp, int groups) {
  if (dp.z1 <= dp.z0 || dp.x1 <= dp.x0) return TileMap{0, 0, 0, 0};
  TileMap m;
  m.ntx = 2;
  m.ntz = (dp.z1 - dp.z0 + kRowsOfThreads - 1) / kRowsOfThreads;
  m.groups = groups;
  m.per = (int)(((int64_t)m.ntx * m.ntz * groups + kXcds - 1) / kXcds);
  return m;
}

// n of G groups per thread at most, evened out over the threads that this takes.
inline int even_share(int G, int n) {
  const int parts = (G + n - 1) / n;
  return (G + parts - 1) / parts;
}

// Shot groups (of S shots) per frame thread: enough threads come before sharing the
// set-up per cell, which weighs more in smaller groups.  Powers of two (three groups
// split 16 unevenly, and bands of six); three groups in one thread rather than in two
// and one.  us per step, forward / adjoint, with 1 / 2 / 4 groups per thread (threads
// with one):
//   one step per launch, S = 4: 300 x 500 x 8 (170 10^3) 16 / 44, 19 / 52; 900 x 1200 x
//   8 (445 10^3) 27.6 / 67.3, 28.7 / 70.7; 300 x 500 x 32 (680 10^3) 25.0 / 66.8, 26.1 /
//   65.7, 33 / 92; 500 x 700 x 32 (1.0 10^6) 35.2 / 103, 33.4 / 100, 40 / 105; 164 x 164 x
//   200 (1.7 10^6) 34 / 129, 36 / 126, 37 / 138; 450 x 450 x 128 (3.1 10^6) 108 / 304, 103 /
//   283, 102 / 271 (8 groups: 109 / 286); S = 2: 553 x 692 x 3 (260 10^3) 13.9 / 40.4, 14.3 /
//   42.1; 900 x 1500 x 3 (510 10^3) 20.2 / 52.0, 18.4 / 49.8;
//   the marching loops, S = 2: 900 x 1500 x 3 18.1 / 48.2, 18.3 / 50.4; 1800 x 1700 x 4 (740
//   10^3) 31.7 / 87.0, 30.7 / 86.6; 1500 x 1700 x 5 (1.0 10^6) 34.1 / 104, 34.7 / 90.7, all
//   three 31.5 / 90.1; 600 x 650 x 32 (2.1 10^6) 40 / 125, 36 / 114, 37 / 110.
// The adjoint's bands, whose set-up is longer, take twice as many: 451 x 877 x 4 37.2
// for 39.1, 300 x 500 x 8 37.7 for 38.7.
inline int frame_groups(int64_t nz, int64_t nx, int G, int S) {
  const int64_t threads = 2 * (kW + 3) * (nz + nx) * G, line = S <= 2 ? 270000 : 400000;
  const int64_t q = (threads + line / 2) / line;
  if (G == 3 && q >= 3) return 3;
  return even_share(G, q >= 8 ? 4 : q >= 2 ? 2 : 1);
}

int habc_check(int64_t B, int64_t nz, int64_t nx, float dt, float h, int S) {
  SEIS_CHECK_ARG(B >= 1 && B <= 65535, "batch size %lld outside [1, 65535]", (long long)B);
  SEIS_CHECK_ARG(nz >= 2 * kW + 2 && nx >= 2 * kW + 2,
                 "HABC needs at least %d cells per axis, got %lld x %lld", 2 * kW + 2,
                 (long long)nz, (long long)nx);
  SEIS_CHECK_ARG(nz * nx < (int64_t)1 << 31, "grid too large");
  SEIS_CHECK_ARG(dt > 0.0f && h > 0.0f, "dt and h must be positive");
  SEIS_CHECK_ARG(S == 1 || S == 2 || S == 4 || S == 8, "shots_per_group %d not in {1,2,4,8}", S);
  return 0;
}

}  // namespace
