// Time-skewed marching kernels of the constant-density acoustic loop.
//
// One wave owns a strip of columns and marches down a segment of H rows for
// one shot.  At march row z it loads row z of the incoming fields and advances
// level k = 1..T on row z-k, so T time steps are taken while each field
// crosses HBM once.  All rows in flight live in registers (three rows of every
// level); x-neighbours come from the adjacent lanes by DPP wave shifts; there
// is no LDS and no barrier.  Each level is valid one cell less far than the
// one below it, so a strip carries halo_lanes(T, VX) lanes on each side and a
// segment T rows above and below that are recomputed by its neighbours from
// the same operands in the same order: every cell's value is bit-identical to
// the one-step kernel's.
//
// Outputs go to other buffers than the inputs (neighbouring waves still read
// the inputs), so a launch takes (u^n, u^{n-1}) to (u^{n+T}, u^{n+T-1}).
#pragma once

#include "common.h"
#include "tiles.h"

namespace seis {
namespace march {

constexpr int kWave = 64;
constexpr int kWavesPerBlock = 4;
constexpr int kThreads = kWave * kWavesPerBlock;
// March rows whose loads are in flight beyond the current one (divides 4).
constexpr int kRowsAhead = 2;
constexpr int kMaxSteps = 4;

__host__ __device__ constexpr int halo_lanes(int T, int VX) { return (T + VX - 1) / VX; }
__host__ __device__ constexpr int out_cols(int T, int VX) {
  return (kWave - 2 * halo_lanes(T, VX)) * VX;
}

// The cells a launch writes: rows [z0, z1), columns [x0, x1), the columns multiples
// of the lanes' width.
struct Region {
  int z0, z1, x0, x1;
};

// Strips x segments x shots of a region, the shots in groups:
// unit = ((shot group * segs + seg) * strips + strip) * group + shot in group.
struct Split {
  int strips, segs, rows;  // rows per segment
  int group;               // shots per group
  Region reg;
};

inline Split make_split(const Region& r, int T, int VX, int rows, int group) {
  Split s;
  const int nz = r.z1 - r.z0;
  s.strips = (r.x1 - r.x0 + out_cols(T, VX) - 1) / out_cols(T, VX);
  s.segs = (nz + rows - 1) / rows;
  s.rows = (nz + s.segs - 1) / s.segs;
  s.segs = (nz + s.rows - 1) / s.rows;
  s.group = group;
  s.reg = r;
  return s;
}

inline Split make_split(const Grid& g, int T, int VX, int rows, int group) {
  return make_split(Region{0, g.nz, 0, g.nx}, T, VX, rows, group);
}

// The value of the lane to the left (lane 0: 0) / right (lane 63: 0).
__device__ __forceinline__ float from_left(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float from_right(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}

// A plane of one shot (or of the model) as a buffer: reads outside it give 0
// and writes outside it are dropped, so rows above and below the grid and
// lanes beyond its sides need no branches.  Offsets are in bytes, a row's plus
// a lane's; a plane has at most kMaxCells cells, so a row below zero wraps
// beyond the range, and kLaneOut or kRowOut in place of either (or both) stays
// beyond it.
constexpr int64_t kMaxCells = (int64_t)1 << 28;
constexpr uint32_t kLaneOut = 0x80000000u;
constexpr uint32_t kRowOut = 0x40000000u;

// Byte offset of row r if it is one of the n rows from lo on.
__device__ __forceinline__ uint32_t row_offset(int r, int lo, int n, uint32_t pitch) {
  return (uint32_t)(r - lo) < (uint32_t)n ? (uint32_t)r * pitch : kRowOut;
}

using Buf = __amdgpu_buffer_rsrc_t;

__device__ __forceinline__ Buf make_buf(const float* p, int64_t cells) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), (short)0, (int)(cells * 4),
                                           0x00020000);
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int VX>
__device__ __forceinline__ void buf_load(Buf p, uint32_t off, float (&o)[VX]) {
  if constexpr (VX == 1) {
    o[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(p, off, 0, 0));
  } else if constexpr (VX == 2) {
    const u32x2 t = __builtin_amdgcn_raw_buffer_load_b64(p, off, 0, 0);
    o[0] = __uint_as_float(t.x); o[1] = __uint_as_float(t.y);
  } else {
    const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(p, off, 0, 0);
    o[0] = __uint_as_float(t.x); o[1] = __uint_as_float(t.y);
    o[2] = __uint_as_float(t.z); o[3] = __uint_as_float(t.w);
  }
}

template <int VX>
__device__ __forceinline__ void buf_store(Buf p, uint32_t off, const float (&v)[VX]) {
  if constexpr (VX == 1) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[0]), p, off, 0, 0);
  } else if constexpr (VX == 2) {
    const u32x2 t = {__float_as_uint(v[0]), __float_as_uint(v[1])};
    __builtin_amdgcn_raw_buffer_store_b64(t, p, off, 0, 0);
  } else {
    const u32x4 t = {__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]),
                     __float_as_uint(v[3])};
    __builtin_amdgcn_raw_buffer_store_b128(t, p, off, 0, 0);
  }
}

// A lane's VX consecutive cells of a row (the grid width is a multiple of VX).
struct Lane {
  int x0;
  bool inner;        // writes (the outer lanes only supply their neighbours)
  uint32_t in, out;  // byte offset in a row for reads / writes, kLaneOut outside
};

template <int T, int VX>
__device__ __forceinline__ Lane make_lane(int strip, const Split& sp, int nx) {
  Lane l;
  constexpr int HL = halo_lanes(T, VX);
  const int lane = (int)(threadIdx.x & (kWave - 1));
  l.x0 = sp.reg.x0 + strip * out_cols(T, VX) + (lane - HL) * VX;
  const bool xin = l.x0 >= 0 && l.x0 < nx;
  l.inner = xin && lane >= HL && lane < kWave - HL && l.x0 < sp.reg.x1;
  l.in = xin ? (uint32_t)l.x0 * 4u : kLaneOut;
  l.out = l.inner ? l.in : kLaneOut;
  return l;
}

// Coefficient planes of the damped update (acoustic.py:81-84), formed once per
// loop: c^2, A = 1/(dt^-2 + d/dt), B = dt^-2 - d/dt.
struct Coefs {
  const float *c2, *A, *Bc;
};

struct FwdLevels {
  const float *u, *up;  // u^n, u^{n-1} (all shots)
  float *o1, *o0;       // u^{n+T}, u^{n+T-1} (o0 unused for T = 1)
  const float* w;       // wavelet samples from n on
  float* ring;          // ring slot of u^{n+1}, or null; the next level's follows at ring_step
  int64_t ring_len, ring_step;
  int ring_levels;      // levels (from 1) whose ring is stored
  float* rows;          // receiver rows of the T levels, (T, slots, B, nx), or null
  const int32_t* row_slot;  // per grid row: its slot, or -1
  int slots;
};

struct FwdParams {
  Coefs cf;
  FwdLevels f;
  const int32_t* src;  // (B, 2) source cells
  int B;
  Split sp;
  Grid g;
  TimeConsts k;
};

// Parameters that only rare rows and edge strips need are read from constant
// memory where they are used: `cold` hides the pointer's origin there, so that
// the compiler does not load them all ahead of the march, where they would
// push the buffer descriptors out of the scalar registers.
template <typename P>
using Const = const __attribute__((address_space(4))) P*;

template <typename P>
__device__ __forceinline__ Const<P> cold(Const<P> p) {
  asm volatile("" : "+s"(p));
  return p;
}

// A read-only value that is the same for the whole wave, through the scalar
// cache: a vector load would have to return before it could be used, and with
// it every field load issued before it.
template <typename V>
__device__ __forceinline__ V scalar_at(const V* p, int64_t i) {
  return ((const __attribute__((address_space(4))) V*)p)[i];
}

// What a source row, a ring row or a receivers' row adds to level t's row r.
template <int VX>
__device__ __forceinline__ void forward_special(Const<FwdParams> p0, int b, const Lane& l, int t,
                                                int r, int z0, int z1, float (&V)[VX]) {
  const Const<FwdParams> p = cold(p0);
  const int sz = scalar_at(p->src, 2 * b), sx = scalar_at(p->src, 2 * b + 1);
  if (r == sz) {
    const float w = scalar_at(p->f.w, t - 1);
#pragma unroll
    for (int e = 0; e < VX; ++e)
      if (l.x0 + e == sx) V[e] += w;
  }
  if (r < z0 || r >= z1 || !l.inner) return;
  const int npml = p->g.npml, ztop = p->g.ztop, nx = p->g.nx;
  const int zbot = p->g.nz - 1 - npml, xr = nx - 1 - npml;
  if (t <= p->f.ring_levels && (r == ztop || r == zbot)) {
    float* q0 = p->f.ring + (t - 1) * p->f.ring_step + (int64_t)b * p->f.ring_len +
                (r == zbot && ztop >= 0 ? nx - 2 * npml - 2 : 0) - npml - 1;
#pragma unroll
    for (int e = 0; e < VX; ++e)
      if (l.x0 + e > npml && l.x0 + e < xr) q0[l.x0 + e] = V[e];
  }
  if (p->f.rows) {
    const int slot = scalar_at(p->f.row_slot, r);
    if (slot >= 0) {
      float* q0 = p->f.rows + ((int64_t)((t - 1) * p->f.slots + slot) * p->B + b) * nx + l.x0;
#pragma unroll
      for (int e = 0; e < VX; ++e) q0[e] = V[e];
    }
  }
}

// RINGCOLS: the strip writes one of the ring's columns.
template <int T, int VX, bool RINGCOLS>
__device__ __forceinline__ void march_forward_strip(const FwdParams& p, Const<FwdParams> pc, int b,
                                                    int strip, int seg) {
  constexpr int kAhead = kRowsAhead;
  const Lane l = make_lane<T, VX>(strip, p.sp, p.g.nx);
  const int64_t plane = p.g.plane;
  const int z0 = p.sp.reg.z0 + seg * p.sp.rows, z1 = min(z0 + p.sp.rows, p.sp.reg.z1);  // owned
  const int zs = z0 - T;
  const int64_t off = (int64_t)b * plane;
  const Buf U = make_buf(p.f.u + off, plane), UP = make_buf(p.f.up + off, plane);
  const Buf O1 = make_buf(p.f.o1 + off, plane), O0 = make_buf(p.f.o0 + off, plane);
  const Buf C = make_buf(p.cf.c2, plane), CA = make_buf(p.cf.A, plane),
            CB = make_buf(p.cf.Bc, plane);
  const uint32_t pitch = (uint32_t)p.g.nx * 4u;
  const float ih2 = p.k.ih2, two_idt2 = p.k.two_idt2;
  // rows that need more than the update; bit t-1 of `marked`: row z-t
  const int sz = scalar_at(p.src, 2 * b);
  const int rt = p.f.ring ? p.g.ztop : -1, rb = p.f.ring ? p.g.nz - 1 - p.g.npml : -1;
  const int32_t* row_slot = p.f.rows ? p.f.row_slot : nullptr;
  const int nz = p.g.nz;
  // the lane's ring column (at most one): the offset of its row 0 in the rings
  // of the first level (the next level's ring follows at rstep)
  const Buf RG = RINGCOLS ? make_buf(p.f.ring + (int64_t)b * p.f.ring_len,
                                     (T - 1) * p.f.ring_step + p.f.ring_len)
                          : U;
  uint32_t rcol = kLaneOut;
  int re = 0;
  const int rlo = max(z0, p.g.ztop + 1), rn = max(min(z1, nz - 1 - p.g.npml) - rlo, 0);
  const int rlev = p.f.ring_levels;
  const uint32_t rstep = (uint32_t)p.f.ring_step * 4u;
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
  uint32_t marked = 0;
  int next_slot = row_slot ? scalar_at(row_slot, min(max(zs, 0), nz - 1)) : -1;
  float L[T][4][VX], c2[4][VX], A[4][VX], Bc[4][VX];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
#pragma unroll
    for (int e = 0; e < VX; ++e) {
#pragma unroll
      for (int t = 0; t < T; ++t) L[t][q][e] = 0.0f;
      c2[q][e] = A[q][e] = Bc[q][e] = 0.0f;
    }
  }
  // loads run kAhead rows ahead: set i holds what march row z consumes (row z
  // of u^n, row z-1 of u^{n-1} and of the coefficients), z = i mod kAhead
  float nU[kAhead][VX], nP[kAhead][VX], nc2[kAhead][VX], nA[kAhead][VX], nB[kAhead][VX];
  uint32_t zo = l.in + (uint32_t)zs * pitch;
  auto fetch = [&](int i) {
    buf_load<VX>(U, zo, nU[i]);
    buf_load<VX>(UP, zo - pitch, nP[i]);
    buf_load<VX>(C, zo - pitch, nc2[i]);
    buf_load<VX>(CA, zo - pitch, nA[i]);
    buf_load<VX>(CB, zo - pitch, nB[i]);
    zo += pitch;
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch(i);
  for (int z4 = zs; z4 < z1 + T; z4 += 4) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int z = z4 + q;
      float P[VX];
#pragma unroll
      for (int e = 0; e < VX; ++e) {
        L[0][q][e] = nU[q % kAhead][e];
        P[e] = nP[q % kAhead][e];
        c2[(q + 3) & 3][e] = nc2[q % kAhead][e];
        A[(q + 3) & 3][e] = nA[q % kAhead][e];
        Bc[(q + 3) & 3][e] = nB[q % kAhead][e];
      }
      fetch(q % kAhead);
      const int slot = next_slot;
      if (row_slot) next_slot = scalar_at(row_slot, min(max(z + 1, 0), nz - 1));
#pragma unroll
      for (int t = 1; t <= T; ++t) {
        const int r = z - t;
        const float(&um)[VX] = L[t - 1][(q - t - 1) & 3];
        const float(&u0)[VX] = L[t - 1][(q - t) & 3];
        const float(&u1)[VX] = L[t - 1][(q - t + 1) & 3];
        float V[VX];
        const float xl = from_left(u0[VX - 1]), xrr = from_right(u0[0]);
#pragma unroll
        for (int e = 0; e < VX; ++e) {
          const float left = e == 0 ? xl : u0[e == 0 ? 0 : e - 1];
          const float right = e == VX - 1 ? xrr : u0[e == VX - 1 ? e : e + 1];
          const float Lp = lap_taps(um[e], left, u0[e], right, u1[e], ih2);
          float prev;
          if (t == 1) prev = P[e];
          else prev = L[t >= 2 ? t - 2 : 0][(q - t) & 3][e];
          V[e] = acoustic_update(A[(q - t) & 3][e], Bc[(q - t) & 3][e], two_idt2, u0[e], prev,
                                 c2[(q - t) & 3][e], Lp);
        }
        if (__builtin_expect((marked >> (t - 1)) & 1u, 0))
          forward_special<VX>(pc, b, l, t, r, z0, z1, V);
        if constexpr (RINGCOLS) {
          float v[1] = {V[0]};
#pragma unroll
          for (int e = 1; e < VX; ++e) v[0] = re == e ? V[e] : v[0];
          const uint32_t ro = row_offset(r, rlo, t <= rlev ? rn : 0, 4u);
          if (ro != kRowOut) buf_store<1>(RG, rcol + ro + (t - 1) * rstep, v);
        }
        if (t < T) {
#pragma unroll
          for (int e = 0; e < VX; ++e) L[t < T ? t : 0][(q - t) & 3][e] = V[e];
        }
        if (t >= T - 1) {
          const uint32_t ro = l.out + row_offset(r, z0, z1 - z0, pitch);
          if (t == T) buf_store<VX>(O1, ro, V);
          else buf_store<VX>(O0, ro, V);
        }
      }
      marked = (marked << 1) | (z == sz || z == rt || z == rb || slot >= 0 ? 1u : 0u);
    }
  }
}

template <int T, int VX>
__device__ __forceinline__ void march_forward(const FwdParams& p, Const<FwdParams> pc, int b,
                                              int strip, int seg) {
  const int xa = strip * out_cols(T, VX), xb = xa + out_cols(T, VX);
  const int xl = p.g.npml, xr = p.g.nx - 1 - p.g.npml;
  if (p.f.ring && ((xa <= xl && xl < xb) || (xa <= xr && xr < xb)))
    march_forward_strip<T, VX, true>(p, pc, b, strip, seg);
  else
    march_forward_strip<T, VX, false>(p, pc, b, strip, seg);
}

struct AdjLevels {
  const float *x, *y;    // u^{k-1}, u^k (interior and ring cells)
  const float *m1, *m2;  // mu^{k+1}, mu^{k+2}
  float *ox, *oy;        // u^{k-1-T}, u^{k-T} (interior and ring cells, zero elsewhere)
  float *om1, *om2;      // mu^{k+1-T}, mu^{k+2-T}
  float* gpart;          // per-shot gradient planes; first: written instead of added to
  bool first;
  const float* w;        // w[k-1] is the last sample used: level t takes w[1-t]
  const float* ring;     // slot of u^{k-2}; the next level's precedes it by ring_step
  int64_t ring_len, ring_step;
  const float* rows;     // adjoint sources of the T levels, (T, slots, B, nx), or null
  const int32_t* row_slot;
  int slots;
};

// x / b for a constant b with y = 1/b rounded: one Newton step on the quotient
// (Markstein).  Rounded as the division: for the 800 divisors of 400 time steps from 0.1
// to 4 ms no mantissa of x gives another quotient.
__device__ __forceinline__ float div_const(float x, float b, float y) {
  const float q = x * y;
  return __fmaf_rn(__fmaf_rn(-b, q, x), y, q);
}

struct AdjParams {
  Coefs cf;
  AdjLevels f;
  const int32_t* src;
  int B;
  Split sp;
  Grid g;
  TimeConsts k;
  bool rebuild_last;  // the last level's u is wanted (its ring slot exists)
};

// T reverse iterations k, k-1, ..., k-T+1 of the adjoint loop: mu by the
// transposed damped step with the receivers' A*s^k added, the gradient term
// L(u^{k-1}) * mu^k (the factor 2c is applied once, after the loop), and the
// rebuilt u^{k-2} on the undamped interior with its ring from storage.
// Kinds of a strip's segment (its halo included): kFrame touches no interior
// cell (mu only), kCore holds undamped interior cells only (A and B are
// constants there and no ring cell is met), kMixed is everything else.
// kDeep is kCore for adjoint fields without the factor A, which goes to the
// Laplacian's weights instead (the sources are added as they are), as the HABC
// adjoint forms them.
enum Kind { kFrame, kMixed, kCore, kDeep };

template <int T, int VX, int KIND>
__device__ __forceinline__ void march_adjoint_strip(const AdjParams& p, Const<AdjParams> pc, int b,
                                                    int strip, int seg) {
  constexpr bool HAS_U = KIND != kFrame, EDGE = KIND == kMixed;
  constexpr bool DEEP = KIND == kDeep, CORE = KIND == kCore || DEEP;
  constexpr int kAhead = kRowsAhead;
  const Lane l = make_lane<T, VX>(strip, p.sp, p.g.nx);
  const int64_t plane = p.g.plane;
  const int z0 = p.sp.reg.z0 + seg * p.sp.rows, z1 = min(z0 + p.sp.rows, p.sp.reg.z1);
  const int zs = z0 - T;
  const int64_t off = (int64_t)b * plane;
  const Buf M1 = make_buf(p.f.m1 + off, plane), M2 = make_buf(p.f.m2 + off, plane);
  const Buf X = make_buf(p.f.x + off, plane), Y = make_buf(p.f.y + off, plane);
  const Buf OM1 = make_buf(p.f.om1 + off, plane), OM2 = make_buf(p.f.om2 + off, plane);
  const Buf OX = make_buf(p.f.ox + off, plane), OY = make_buf(p.f.oy + off, plane);
  const Buf GP = make_buf(p.f.gpart + off, plane);
  const Buf C = make_buf(p.cf.c2, plane), CA = make_buf(p.cf.A, plane),
            CB = make_buf(p.cf.Bc, plane);
  const uint32_t pitch = (uint32_t)p.g.nx * 4u;
  const int nz = p.g.nz;
  const int ztop = p.g.ztop, zbot = nz - 1 - p.g.npml, ur0 = max(ztop, 0);
  const float ih2 = p.k.ih2, two_idt2 = p.k.two_idt2;
  const float kA = 1.0f / p.k.idt2, kB = p.k.idt2;  // undamped A and B, as the forward forms them
  const float rA = 1.0f / kA, rB = 1.0f / kB;
  const float ka = two_idt2 * kA, kb = -(kB * kA);  // DEEP
  const int sz = scalar_at(p.src, 2 * b);
  const int32_t* row_slot = p.f.rows ? p.f.row_slot : nullptr;
  // rows whose u is read; owned rows whose u is written; owned rows of the
  // gradient; those that are added to (none in the first launch)
  const int un = zbot + 1 - ur0;
  const int ulo = max(z0, ur0), ulen = max(min(z1, zbot + 1) - ulo, 0);
  const int glo = max(z0, ztop + 1), glen = max(min(z1, zbot) - glo, 0);
  const int gadd = p.f.first ? 0 : glen;
  const int tl = p.rebuild_last ? T : T - 1;  // levels whose u is wanted
  // rings of levels T, T-1, .., 1 as one buffer: level t's starts at
  // rbase - t * rstep
  const uint32_t rstep = EDGE ? (uint32_t)p.f.ring_step * 4u : 0, rbase = T * rstep;
  const Buf RG = EDGE ? make_buf(p.f.ring + (int64_t)b * p.f.ring_len - (T - 1) * p.f.ring_step,
                                 (T - 1) * p.f.ring_step + p.f.ring_len)
                      : M1;
  bool xin[VX], xring[VX];
  uint32_t rcol = kLaneOut;  // the lane's ring column: offset of its row 0 in a ring
  uint32_t rrow[VX];         // the lane's cells in the top ring row
  const uint32_t rbot = ztop >= 0 ? 4u * (p.g.nx - 2 * p.g.npml - 2) : 0;  // to the bottom row
  if constexpr (EDGE) {
    const int npml = p.g.npml, xr = p.g.nx - 1 - npml;
    const int nxi = p.g.nx - 2 * npml - 2;
#pragma unroll
    for (int e = 0; e < VX; ++e) {
      const int x = l.x0 + e;
      xin[e] = x > npml && x < xr;
      xring[e] = x == npml || x == xr;
      if (xring[e])
        rcol = 4u * (uint32_t)((ztop >= 0 ? 2 * nxi : nxi) + (x == xr ? zbot - ztop - 1 : 0) -
                               (ztop + 1));
      rrow[e] = xin[e] ? 4u * (uint32_t)(x - npml - 1) : kLaneOut;
    }
  }
  // rows that hold receivers; after the fetch for march row zf, bit j: row zf-1-j
  uint32_t marked = 0;
  int next_slot = -1;
  const float* srows = p.f.rows ? p.f.rows + (int64_t)b * p.g.nx : nullptr;
  float M[T][4][VX], Q[T][4][VX], U[T][4][VX], G[4][VX];
  float c2[4][VX], A[4][VX], Bc[4][VX], cC[VX];
#pragma unroll
  for (int e = 0; e < VX; ++e) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int t = 0; t < T; ++t) M[t][q][e] = Q[t][q][e] = U[t][q][e] = 0.0f;
      G[q][e] = c2[q][e] = 0.0f;
      A[q][e] = CORE ? kA : 0.0f;
      Bc[q][e] = CORE ? kB : 0.0f;
    }
    cC[e] = 0.0f;
  }
  // loads run kAhead rows ahead: set i holds what march row z consumes (row z
  // of mu^{k+1}, c^2 and u^{k-1}, row z-1 of mu^{k+2}, u^k, A and B, row z-T
  // of the gradient, the ring columns of rows z-t), z = i mod kAhead
  float nM1[kAhead][VX], nM2[kAhead][VX], nX[kAhead][VX], nY[kAhead][VX], nc2[kAhead][VX],
      nA[kAhead][VX], nB[kAhead][VX], nG[kAhead][VX], nR[kAhead][T], nV[kAhead][VX],
      nS[kAhead][VX];
  uint32_t zo = l.in + (uint32_t)zs * pitch;
  int zf = zs;
  // level t's adjoint sources on row z-t
  auto source_row = [&](int t, int z, float(&o)[VX]) {
    const Const<AdjParams> c = cold(pc);
    const int slot = scalar_at(c->f.row_slot, min(max(z - t, 0), c->g.nz - 1));
    buf_load<VX>(make_buf(srows + (int64_t)((t - 1) * c->f.slots + max(slot, 0)) * c->B * c->g.nx,
                          c->g.nx), l.in, o);
  };
  auto fetch = [&](int i) {
    const uint32_t zp = zo - pitch;
    buf_load<VX>(M1, zo, nM1[i]);
    buf_load<VX>(C, zo, nc2[i]);
    buf_load<VX>(M2, zp, nM2[i]);
    if constexpr (!CORE) {
      buf_load<VX>(CA, zp, nA[i]);
      buf_load<VX>(CB, zp, nB[i]);
    }
    if constexpr (HAS_U) {
      if constexpr (CORE) {
        buf_load<VX>(X, zo, nX[i]);
        buf_load<VX>(Y, zp, nY[i]);
      } else {
        buf_load<VX>(X, l.in + row_offset(zf, ur0, un, pitch), nX[i]);
        buf_load<VX>(Y, l.in + row_offset(zf - 1, ur0, un, pitch), nY[i]);
      }
      buf_load<VX>(GP, l.out + row_offset(zf - T, glo, gadd, pitch), nG[i]);
    }
    if constexpr (EDGE) {
#pragma unroll
      for (int t = 1; t <= T; ++t) {
        float v[1];
        buf_load<1>(RG, rcol + row_offset(zf - t, ztop + 1, t <= tl ? zbot - ztop - 1 : 0, 4u) +
                            (rbase - t * rstep), v);
        nR[i][t - 1] = v[0];
      }
      // one of levels 1..T meets a ring row (never two: the rows are at least
      // T apart): its stored row
      const int zr = zf - ztop <= T ? ztop : zbot, tr = zf - zr;
#pragma unroll
      for (int e = 0; e < VX; ++e) nV[i][e] = 0.0f;
      if (zr >= 0 && tr >= 1 && tr <= tl) {
#pragma unroll
        for (int e = 0; e < VX; ++e) {
          float v[1];
          buf_load<1>(RG, rrow[e] + (zr == ztop ? 0 : rbot) + (rbase - tr * rstep), v);
          nV[i][e] = v[0];
        }
      }
    }
    if (srows) {
      // the adjoint sources of the first level that meets a receivers' row
      marked = (marked << 1) | (next_slot >= 0 ? 1u : 0u);
      next_slot = scalar_at(row_slot, min(max(zf, 0), nz - 1));
      const uint32_t hit = marked & ((1u << T) - 1u);
      if (__builtin_expect(hit != 0, 0)) source_row(__ffs(hit), zf, nS[i]);
    }
    zo += pitch;
    ++zf;
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch(i);

  for (int z4 = zs; z4 < z1 + T; z4 += 4) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int z = z4 + q;
      float SR[VX];
#pragma unroll
      for (int e = 0; e < VX; ++e) SR[e] = nS[q % kAhead][e];
      float PM[VX], PY[VX], gv[VX], rv[T], rw[VX];
#pragma unroll
      for (int e = 0; e < VX; ++e) {
        c2[(q + 3) & 3][e] = cC[e];
        cC[e] = nc2[q % kAhead][e];
        M[0][q][e] = nM1[q % kAhead][e];
        Q[0][q][e] = (DEEP ? cC[e] * kA : cC[e]) * M[0][q][e];
        PM[e] = nM2[q % kAhead][e];
        if constexpr (!CORE) {
          A[(q + 3) & 3][e] = nA[q % kAhead][e];
          Bc[(q + 3) & 3][e] = nB[q % kAhead][e];
        }
        if constexpr (HAS_U) {
          U[0][q][e] = nX[q % kAhead][e];
          PY[e] = nY[q % kAhead][e];
          gv[e] = nG[q % kAhead][e];
        }
      }
      if constexpr (EDGE) {
#pragma unroll
        for (int t = 0; t < T; ++t) rv[t] = nR[q % kAhead][t];
#pragma unroll
        for (int e = 0; e < VX; ++e) rw[e] = nV[q % kAhead][e];
      }
      fetch(q % kAhead);
      const uint32_t here = (marked >> kAhead) & ((1u << T) - 1u);  // bit t-1: row z-t
      const int t0 = __ffs(here);
      const int zring = z - (z - ztop <= T ? ztop : zbot);  // the level that meets a ring row
      // ---- level t on row z-t
#pragma unroll
      for (int t = 1; t <= T; ++t) {
        const int r = z - t;
        const float(&qm)[VX] = Q[t - 1][(q - t - 1) & 3];
        const float(&q0)[VX] = Q[t - 1][(q - t) & 3];
        const float(&q1)[VX] = Q[t - 1][(q - t + 1) & 3];
        const float(&ca)[VX] = c2[(q - t) & 3];
        float V[VX];
        {
          const float xl = from_left(q0[VX - 1]), xrr = from_right(q0[0]);
#pragma unroll
          for (int e = 0; e < VX; ++e) {
            const float left = e == 0 ? xl : q0[e == 0 ? 0 : e - 1];
            const float right = e == VX - 1 ? xrr : q0[e == VX - 1 ? e : e + 1];
            const float Lm = lap_taps(qm[e], left, q0[e], right, q1[e], ih2);
            float prev;
            if (t == 1) prev = PM[e];
            else prev = M[t >= 2 ? t - 2 : 0][(q - t) & 3][e];
            if constexpr (DEEP)
              V[e] = (ka * M[t - 1][(q - t) & 3][e] + Lm) + kb * prev;
            else
              V[e] = A[(q - t) & 3][e] *
                     ((two_idt2 * M[t - 1][(q - t) & 3][e] - Bc[(q - t) & 3][e] * prev) + Lm);
          }
        }
        if (__builtin_expect((here >> (t - 1)) & 1u, 0)) {
          float s[VX];
#pragma unroll
          for (int e = 0; e < VX; ++e) s[e] = SR[e];
          if (t != t0) source_row(t, z, s);  // receivers on neighbouring rows
#pragma unroll
          for (int e = 0; e < VX; ++e)
            V[e] = V[e] + (DEEP ? s[e] : A[(q - t) & 3][e] * s[e]);
        }
        if (t < T) {
#pragma unroll
          for (int e = 0; e < VX; ++e) {
            M[t < T ? t : 0][(q - t) & 3][e] = V[e];
            Q[t < T ? t : 0][(q - t) & 3][e] = (DEEP ? ca[e] * kA : ca[e]) * V[e];
          }
        }
        if (t >= T - 1) {
          const uint32_t ro = l.out + row_offset(r, z0, z1 - z0, pitch);
          if (t == T) buf_store<VX>(OM1, ro, V);
          else buf_store<VX>(OM2, ro, V);
        }
        if constexpr (HAS_U) {
          const float(&um)[VX] = U[t - 1][(q - t - 1) & 3];
          const float(&u0)[VX] = U[t - 1][(q - t) & 3];
          const float(&u1)[VX] = U[t - 1][(q - t + 1) & 3];
          const float xl = from_left(u0[VX - 1]), xrr = from_right(u0[0]);
          float un[VX], W[VX], gt[VX];
#pragma unroll
          for (int e = 0; e < VX; ++e) {
            if (t == 1) un[e] = PY[e];
            else un[e] = U[t >= 2 ? t - 2 : 0][(q - t) & 3][e];
          }
          if (__builtin_expect(r == sz, 0)) {
            const Const<AdjParams> c = cold(pc);
            const float w = scalar_at(c->f.w, 1 - t);
            const int sx = scalar_at(c->src, 2 * b + 1);
#pragma unroll
            for (int e = 0; e < VX; ++e)
              if (l.x0 + e == sx) un[e] -= w;
          }
#pragma unroll
          for (int e = 0; e < VX; ++e) {
            const float left = e == 0 ? xl : u0[e == 0 ? 0 : e - 1];
            const float right = e == VX - 1 ? xrr : u0[e == VX - 1 ? e : e + 1];
            const float Lu = lap_taps(um[e], left, u0[e], right, u1[e], ih2);
            gt[e] = Lu * V[e];
            W[e] = div_const((two_idt2 * u0[e] + ca[e] * Lu) - div_const(un[e], kA, rA), kB, rB);
            if constexpr (EDGE) {
              // columns outside the interior: the ring's stored value or nothing
              gt[e] = xin[e] ? gt[e] : 0.0f;
              W[e] = xin[e] ? W[e] : (xring[e] ? rv[t - 1] : 0.0f);
            }
          }
          if constexpr (EDGE) {
            if (t == zring) {  // a ring row
#pragma unroll
              for (int e = 0; e < VX; ++e) W[e] = rw[e];
            }
          }
#pragma unroll
          for (int e = 0; e < VX; ++e) {
            if (t == 1) G[(q - t) & 3][e] = gt[e];
            else G[(q - t) & 3][e] += gt[e];
          }
          if (t == T) {
            float go[VX];
#pragma unroll
            for (int e = 0; e < VX; ++e) go[e] = gv[e] + G[(q - t) & 3][e];
            buf_store<VX>(GP, l.out + row_offset(r, glo, glen, pitch), go);
          }
          if (t < T) {
#pragma unroll
            for (int e = 0; e < VX; ++e) U[t < T ? t : 0][(q - t) & 3][e] = W[e];
          }
          if (t >= T - 1) {
            const uint32_t ro = l.out + row_offset(r, ulo, ulen, pitch);
            if (t == T) buf_store<VX>(OX, ro, W);
            else buf_store<VX>(OY, ro, W);
          }
        }
      }
    }
  }
}

template <int T, int VX>
__device__ __forceinline__ void march_adjoint(const AdjParams& p, Const<AdjParams> pc, int b,
                                              int strip, int seg) {
  const int xa = strip * out_cols(T, VX) - halo_lanes(T, VX) * VX, xb = xa + kWave * VX;
  const int z0 = seg * p.sp.rows, z1 = min(z0 + p.sp.rows, p.g.nz);
  const int xl = p.g.npml, xr = p.g.nx - 1 - p.g.npml, zbot = p.g.nz - 1 - p.g.npml;
  // rows and columns of the strip (its halo included) against the interior's
  if (!(xb > xl + 1 && xa < xr && z1 + T - 1 > max(p.g.ztop, 0) && z0 - T < zbot))
    march_adjoint_strip<T, VX, kFrame>(p, pc, b, strip, seg);
  else if (xa <= xl || xb > xr || z0 - T <= p.g.ztop || z1 + T > zbot)
    march_adjoint_strip<T, VX, kMixed>(p, pc, b, strip, seg);
  else
    march_adjoint_strip<T, VX, kCore>(p, pc, b, strip, seg);
}

}  // namespace march
}  // namespace seis
