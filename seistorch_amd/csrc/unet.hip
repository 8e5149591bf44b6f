// Kernels of the learned gradient preconditioner (a small U-Net) for gfx950.
//
// Activations are NHWC with channels contiguous; weights and activations are
// bfloat16 (stored as raw uint16 bit patterns), accumulation is FP32 on the
// matrix cores (v_mfma_f32_16x16x32_bf16), and gradients of activations are
// kept in FP32.  A 3x3 convolution (zero padding 1, stride 1) is an implicit
// GEMM: rows = output pixels, columns = output channels, reduction index
// k = tap * Cin + ci over the 9 taps (tap = 3*(dy+1) + (dx+1)).  Weights are
// stored [Cout][9*Cin] so that one lane's 8 consecutive k are one 16-byte load.
//
// MFMA operand layout (16x16x32 bf16, one wave): lane l holds
//   A[m = l%16][k = 8*(l/16) + i], B[k = 8*(l/16) + i][n = l%16], i = 0..7,
// and the result D[m = 4*(l/16) + i][n = l%16], i = 0..3.
//
// There is no reference counterpart: the network and its training are this
// project's own (the plain-gradient FWI step of the reference,
// seistorch/fwi.py, is its fallback).
#include "common.h"
#include "seistorch_amd.h"

#include <algorithm>
#include <cstdint>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// FP32 -> bf16, round to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint16_t f2bf(float f) {
  return __builtin_bit_cast(uint16_t, (__bf16)f);
}

__device__ __forceinline__ bf16x8 load8(const uint16_t* p) {
  const uint4 v = *reinterpret_cast<const uint4*>(p);
  return __builtin_bit_cast(bf16x8, v);
}

__device__ __forceinline__ bf16x8 zero8() { return __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0)); }

constexpr float kInvSqrt2 = 0.70710678118654752f;
constexpr float kInvSqrt2Pi = 0.39894228040143268f;

// The activation and its derivative by the library's functions, forward and
// backward alike: both stand in front of a rounding to bf16 that every later layer
// builds on, and another last place of either is another rounding here and there.
__device__ __forceinline__ float gelu(float v) { return 0.5f * v * (1.0f + erff(v * kInvSqrt2)); }

__device__ __forceinline__ float gelu_grad(float v) {
  return 0.5f * (1.0f + erff(v * kInvSqrt2)) + v * kInvSqrt2Pi * expf(-0.5f * v * v);
}

// Eight bf16 values as floats and back.
__device__ __forceinline__ void unpack8(const uint16_t* p, float (&o)[8]) {
  const uint4 q = *reinterpret_cast<const uint4*>(p);
  const uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    o[2 * e] = __uint_as_float(u[e] << 16);
    o[2 * e + 1] = __uint_as_float(u[e] & 0xffff0000u);
  }
}
__device__ __forceinline__ void pack8(uint16_t* p, const float (&v)[8]) {
  bf16x8 q;
#pragma unroll
  for (int e = 0; e < 8; ++e) q[e] = (__bf16)v[e];
  *reinterpret_cast<uint4*>(p) = __builtin_bit_cast(uint4, q);
}
__device__ __forceinline__ void load8f(const float* p, float (&o)[8]) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
  o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
}

// --------------------------------------------------- asynchronous LDS tiles

// 16 bytes per lane from global memory straight into LDS at l + 16 * lane (l is
// the same for the wave); lanes that are masked off leave their bytes alone.
// The data is there after lds_arrived() and a barrier.
__device__ __forceinline__ void async16(const uint16_t* g, uint16_t* l) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) uint32_t*)g,
                                   (__attribute__((address_space(3))) uint32_t*)l, 16, 0, 0);
}
__device__ __forceinline__ void lds_arrived() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Input of a convolution: one image of C channels, or the concatenation of the
// nearest 2x upsampling of low (C1 channels, half the size) and skip (C - C1).
struct ConvInput {
  const uint16_t* x;    // the image, or skip
  const uint16_t* low;  // null: one image
  int C, C1;            // C1 = 0 for one image
};

// ---------------------------------------------------------------- conv 3x3

// Every convolution, of the network or of its data gradient, sums an output's
// products in the order k = tap * C + ci, 32 at a time, whatever the tile, so that
// the bf16 activations and gradients depend on neither launch shape nor kernel.  (A
// last-place difference before a rounding to bf16 is a different value for every
// later layer: over the network's depth two orders drift apart by as much as either
// is from the exact result, the training gradient by 1e-4 of its norm.)

// kConvAct: z = acc + bias (bf16, optional) and y = act(z) (bf16).  kConvF32: yf = acc
// (+ bias).  kConvGeluGrad: y = bf16(acc * gelu'(z)), the data gradient taken through
// the activation before it.
enum { kConvAct = 0, kConvF32 = 1, kConvGeluGrad = 2 };
constexpr int kTileW = 32;
constexpr int kWinW = kTileW + 2;
constexpr int kUnit = 8;  // bf16 per 16-byte unit

struct ConvArgs {
  ConvInput in;
  int N, H, W;
  const uint16_t* w;
  const float* bias;
  int Cout, act;
  uint16_t *z, *y;  // kConvGeluGrad reads z
  float* yf;
  int vec;  // Cout % 8 == 0 and 16-byte aligned outputs
  int tx, ty, ntile, per, lg;  // tiles in x and y, output-channel tiles, tiles per XCD
};

// A pixel's M sums, of the channels from cb on: bias, activation, stores at o.
template <int MODE, int M>
__device__ __forceinline__ void conv_out(const ConvArgs& a, int64_t o, int cb,
                                         const float (&v)[M]) {
#pragma unroll
  for (int h = 0; h < M; h += 8) {
    if (cb + h + 8 <= a.Cout && a.vec) {
      float y[8], t[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = v[h + e];
      if constexpr (MODE == kConvF32) {
        *reinterpret_cast<float4*>(a.yf + o + h) = make_float4(y[0], y[1], y[2], y[3]);
        *reinterpret_cast<float4*>(a.yf + o + h + 4) = make_float4(y[4], y[5], y[6], y[7]);
      } else if constexpr (MODE == kConvGeluGrad) {
        unpack8(a.z + o + h, t);
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] *= gelu_grad(t[e]);
        pack8(a.y + o + h, y);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = a.act ? gelu(y[e]) : y[e];
        if (a.z) pack8(a.z + o + h, y);
        pack8(a.y + o + h, t);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (cb + h + e >= a.Cout) continue;
        const float y = v[h + e];
        const int64_t q = o + h + e;
        if constexpr (MODE == kConvF32) {
          a.yf[q] = y;
        } else if constexpr (MODE == kConvGeluGrad) {
          a.y[q] = f2bf(y * gelu_grad(bf2f(a.z[q])));
        } else {
          if (a.z) a.z[q] = f2bf(y);
          a.y[q] = f2bf(a.act ? gelu(y) : y);
        }
      }
    }
  }
}

// The data gradient of a layer with 32 output channels: implicit GEMM on
// v_mfma_f32_16x16x32_bf16, weights as the first operand, so that a lane ends with
// consecutive channels of one pixel.  A block of WAVES waves computes (WAVES * RW) x
// 32 pixels x 32 channels, wave w the rows w * RW on.  The (rows + 2) x 34 pixel
// window and the 9 x 32 x 32 weights go to LDS by asynchronous loads; what hides
// their latency is the other blocks on the CU.  A wave holds the nine taps' weights
// in registers and reads each fragment of a window row once for the output rows that
// it reaches: the rows from above, so that each of them meets its taps in order.  8 x
// 256 x 384 pixels: 32 -> 32 channels through the activation 52 us, 32 -> 96 channels 109
// us (31 and 74 us of it the activations' traffic at the copy rate); k_conv3x3 takes 63 us
// for the forward of 32 -> 32.
//
// LDS holds a pixel's (or weight row's) 32 channels as four 16-byte units, unit
// u of window column c at slot u ^ ((c >> 2) & 3): 16 consecutive pixels then
// read 16 distinct quarter-rows of banks, and the swizzle is the same in every
// row, so that a lane needs one address per horizontal tap.  Weight rows are permuted,
// row j * 16 + m holding channel (m / 4) * 8 + 4 * j + m % 4, so that a lane's 8
// results are consecutive channels and leave in 16-byte stores.
template <int WAVES, int RW, int MODE>
__global__ __launch_bounds__(WAVES * 64) void k_conv3x3_grad32(ConvArgs a) {
  constexpr int kThr = WAVES * 64, kRows = WAVES * RW, kPx = (kRows + 2) * kWinW;
  constexpr int NT = 32, NF = 2, C = 32, K = 9 * C;
  constexpr int kAU = kPx * 4, kBU = 9 * NT * 4;  // 16-byte units
  constexpr int kAP = (kAU + kThr - 1) / kThr, kBP = (kBU + kThr - 1) / kThr;
  __shared__ __align__(16) uint16_t sA[kAP * kThr * kUnit];
  __shared__ __align__(16) uint16_t sB[kBP * kThr * kUnit];
  const int t = threadIdx.x, wave = t / 64, l = t % 64, m = l % 16, kq = l / 16;
  // XCD-aware order: the output-channel tiles of one pixel tile, then the next
  // pixel tile, on the same XCD
  const int unit = (int)(blockIdx.x % 8) * a.per + (int)(blockIdx.x / 8);
  const int tile = unit / a.ntile, co0 = (unit - tile * a.ntile) * NT;
  if (tile >= a.N * a.ty * a.tx) return;  // uniform over the block
  const int px0 = (tile % a.tx) * kTileW, py0 = ((tile / a.tx) % a.ty) * kRows;
  const int n = tile / (a.tx * a.ty);
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  const uint16_t* x0 = a.in.x + (((int64_t)n * a.H + py0) * a.W + px0) * C;
  // uniform: no unit lies outside the image or the channels
  const bool inside = px0 > 0 && px0 + kTileW < a.W && py0 > 0 && py0 + kRows < a.H;
  const bool whole = co0 + NT <= a.Cout;
#pragma unroll
  for (int i = 0; i < kAP; ++i) {
    const int p = (i * kThr + t) / 4, r = p / kWinW - 1, c = p % kWinW - 1;
    bool ok = true;
    if (!inside) ok = py0 + r >= 0 && py0 + r < a.H && px0 + c >= 0 && px0 + c < a.W;
    if (kAU % kThr != 0 && i == kAP - 1) ok = ok && p < kPx;
    const int cu = ((t & 3) ^ (((c + 1) >> 2) & 3)) * kUnit;
    if (ok) async16(x0 + ((int64_t)(r * a.W + c) * C + cu), &sA[(i * kThr + wave * 64) * kUnit]);
    else *reinterpret_cast<uint4*>(&sA[(i * kThr + t) * kUnit]) = zero;
  }
#pragma unroll
  for (int i = 0; i < kBP; ++i) {
    const int u = i * kThr + t, row = (u / 4) % NT, tap = u / (4 * NT);
    const int cq = (t & 3) ^ ((row >> 2) & 3), j = row / 16, mm = row % 16;
    const int co = co0 + (mm / 4) * 8 + 4 * j + mm % 4;
    bool ok = whole || co < a.Cout;
    if (kBU % kThr != 0 && i == kBP - 1) ok = ok && u < kBU;
    uint16_t* to = &sB[(i * kThr + wave * 64) * kUnit];
    if (ok) async16(a.w + (int64_t)co * K + tap * C + cq * kUnit, to);
    else *reinterpret_cast<uint4*>(&sB[u * kUnit]) = zero;
  }
  floatx4 acc[RW][2][NF];
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[r][f][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  // this lane's first fragment addresses: window column m + dx (rows and the
  // second 16 columns at constant distances), weight row m
  int xa[3];
#pragma unroll
  for (int dx = 0; dx < 3; ++dx)
    xa[dx] = ((wave * RW * kWinW + m + dx) * 4 + (kq ^ (((m + dx) >> 2) & 3))) * kUnit;
  const int wa = (m * 4 + (kq ^ ((m >> 2) & 3))) * kUnit;
  lds_arrived();
  __syncthreads();
  bf16x8 wf[9][NF];
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int j = 0; j < NF; ++j) wf[tap][j] = load8(&sB[wa + (tap * NT + j * 16) * 4 * kUnit]);
#pragma unroll
  for (int ir = 0; ir < RW + 2; ++ir) {
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) {
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const bf16x8 xf = load8(&sA[xa[dx] + (ir * kWinW + f * 16) * 4 * kUnit]);
#pragma unroll
        for (int dy = 0; dy < 3; ++dy) {
          const int r = ir - dy;
          if (r < 0 || r >= RW) continue;
#pragma unroll
          for (int j = 0; j < NF; ++j)
            acc[r][f][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[dy * 3 + dx][j], xf,
                                                                   acc[r][f][j], 0, 0, 0);
        }
      }
    }
  }
  const int cb = co0 + kq * 8;  // this lane's 8 consecutive channels
  float bv[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) bv[e] = a.bias && cb + e < a.Cout ? a.bias[cb + e] : 0.0f;
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const int yy = py0 + wave * RW + r;
    if (yy >= a.H) continue;
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      const int xx = px0 + f * 16 + m;
      if (xx >= a.W) continue;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = acc[r][f][e / 4][e % 4] + bv[e];
      conv_out<MODE, 8>(a, (((int64_t)n * a.H + yy) * a.W + xx) * a.Cout + cb, cb, v);
    }
  }
}

// The network's own convolutions and the data gradient of wider layers.  With the
// taps outside, all C channels of the window have to be at hand: a block of TH x TW
// pixels loads them once into LDS (asynchronously, C up to 512) and its waves then run
// through all of K without a barrier.  What bounds it is the latency of the weights'
// 64-byte rows from L2: 25 to 40 % of the matrix rate at 96 channels and more, 15 % at
// 32 (data gradients of 8 x 256 x 384 pixels, 64 -> 64 channels at half the size 67 us, 256 ->
// 256 at an eighth 48).  Wave (wm, wn) owns MR fragments of 16 pixels and 16 * NF output channels; the
// weights come straight from L2, two steps ahead, into registers.
//
// Pixels lie C * 2 bytes apart; the 16-byte unit u of window column c is at u ^
// ((c >> (4 - lg)) & (2^lg - 1)), 2^lg being the largest power of two in C / 8 (at
// most 16): 16 neighbouring pixels then read from all banks.

// kOne: C is 32, so that a step's 32 products are one tap.  kFar: C is beyond the
// LDS; the fragments come straight from memory (no layer of the default network).
enum { kAny = 0, kOne = 1, kFar = 2 };
template <int TH, int TW, int MR, int NF, int WM, int WN, int KIND, int MODE>
__global__ __launch_bounds__(64 * WM * WN) void k_conv3x3(ConvArgs a) {
  static_assert(TH * TW == 16 * MR * WM, "the waves cover the tile");
  constexpr int kThr = 64 * WM * WN, kWin = TW + 2, kPx = (TH + 2) * kWin, kFx = TW / 16;
  constexpr int NT = 16 * NF;  // a wave's output channels
  extern __shared__ __align__(16) uint16_t sx[];
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t / 64), l = t % 64;
  const int m = l % 16, kq = l / 16;
  const int wm = wave % WM, wn = wave / WM;
  const int C = a.in.C, K = 9 * C, nk = (K + 31) / 32, upp = C / 8, lg = a.lg;
  const int unit = (int)(blockIdx.x % 8) * a.per + (int)(blockIdx.x / 8);
  const int tile = unit / a.ntile, co0 = (unit - tile * a.ntile) * NT * WN + wn * NT;
  if (tile >= a.N * a.ty * a.tx) return;  // uniform over the block
  const int px0 = (tile % a.tx) * TW, py0 = ((tile / a.tx) % a.ty) * TH;
  const int n = tile / (a.tx * a.ty);
  // weights: lane m of fragment j holds channel co0 + (m / 4) * (NT / 4) + 4 j + m % 4
  // (rows beyond Cout repeat the last one and are not stored)
  uint32_t wp[NF];
#pragma unroll
  for (int j = 0; j < NF; ++j) {
    const int co = co0 + (m / 4) * (NT / 4) + 4 * j + m % 4;
    wp[j] = (uint32_t)(min(co, a.Cout - 1) * K + kq * 8);
  }
  auto weights = [&](int kc, uint4 (&o)[NF]) {
    const uint16_t* w = a.w + min(kc, nk - 1) * 32;
    const bool ok = KIND == kOne || kc * 32 + kq * 8 < K;
#pragma unroll
    for (int j = 0; j < NF; ++j)
      o[j] = ok ? *reinterpret_cast<const uint4*>(w + wp[j]) : make_uint4(0u, 0u, 0u, 0u);
  };
  uint4 wb[3][NF];
  weights(0, wb[0]);
  weights(1, wb[1]);
  // the window: 64 / upp pixels per wave and load
  if constexpr (KIND != kFar) {
    const int ppi = 64 / upp, pl = l / upp, ul = l - pl * upp;
    for (int p0 = wave * ppi; p0 < kPx; p0 += WM * WN * ppi) {
      const int p = p0 + pl, r = p / kWin, c = p - r * kWin;
      const int yy = py0 + r - 1, xx = px0 + c - 1;
      const int ch = (ul ^ ((c >> (4 - lg)) & ((1 << lg) - 1))) * 8;
      const bool lane = pl < ppi && p < kPx;
      const bool in = yy >= 0 && yy < a.H && xx >= 0 && xx < a.W;
      const bool lo = ch < a.in.C1;
      const int64_t q = lo ? ((int64_t)n * (a.H / 2) + yy / 2) * (a.W / 2) + xx / 2
                           : ((int64_t)n * a.H + yy) * a.W + xx;
      const uint16_t* src = lo ? a.in.low + q * a.in.C1 + ch
                               : a.in.x + q * (C - a.in.C1) + (ch - a.in.C1);
      if (lane && in) async16(src, sx + p0 * C);
      else if (lane) *reinterpret_cast<uint4*>(sx + p * C + ul * 8) = make_uint4(0u, 0u, 0u, 0u);
    }
  }
  floatx4 acc[MR][NF];
#pragma unroll
  for (int r = 0; r < MR; ++r)
#pragma unroll
    for (int j = 0; j < NF; ++j) acc[r][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  lds_arrived();
  __syncthreads();
  // this lane's tap and unit of the step: k = kc * 32 + 8 * kq = tap * C + 8 * u
  int u = kq, tap = 0;
  if (KIND != kOne)
    while (u >= upp) { u -= upp; ++tap; }
  int lx[3];  // kOne: the horizontal taps' addresses
#pragma unroll
  for (int dx = 0; dx < 3; ++dx) lx[dx] = (m + dx) * 32 + (kq ^ (((m + dx) >> 2) & 3)) * 8;
  int fo[MR];  // the fragments' distances (uniform)
#pragma unroll
  for (int r = 0; r < MR; ++r) {
    const int f = wm * MR + r;
    fo[r] = ((f / kFx) * kWin + (f % kFx) * 16) * C;
  }
  auto step = [&](uint4 (&wcur)[NF], int kc) {
    bf16x8 xf[MR];
    if constexpr (KIND == kOne) {
      const int dy = (tap * 11) >> 5, dx = tap - 3 * dy;
      const int base = (dx == 0 ? lx[0] : dx == 1 ? lx[1] : lx[2]) + dy * kWin * 32;
#pragma unroll
      for (int r = 0; r < MR; ++r) xf[r] = load8(sx + base + fo[r]);
      ++tap;
    } else {
      const int tp = min(tap, 8), dy = (tp * 11) >> 5, dx = tp - 3 * dy;
      if constexpr (KIND == kAny) {
        const int base = (dy * kWin + m + dx) * C +
                         ((u ^ (((m + dx) >> (4 - lg)) & ((1 << lg) - 1))) * 8);
#pragma unroll
        for (int r = 0; r < MR; ++r) xf[r] = load8(sx + base + fo[r]);
      } else {
#pragma unroll
        for (int r = 0; r < MR; ++r) {
          const int f = wm * MR + r, ch = u * 8;
          const int yy = py0 + f / kFx + dy - 1, xx = px0 + (f % kFx) * 16 + m + dx - 1;
          const bool lo = ch < a.in.C1;
          const int64_t q = lo ? ((int64_t)n * (a.H / 2) + yy / 2) * (a.W / 2) + xx / 2
                               : ((int64_t)n * a.H + yy) * a.W + xx;
          xf[r] = zero8();
          if (yy >= 0 && yy < a.H && xx >= 0 && xx < a.W)
            xf[r] = load8(lo ? a.in.low + q * a.in.C1 + ch
                             : a.in.x + q * (C - a.in.C1) + (ch - a.in.C1));
        }
      }
      if (kc == nk - 1) {  // products beyond K
#pragma unroll
        for (int r = 0; r < MR; ++r) xf[r] = tap > 8 ? zero8() : xf[r];
      }
      u += 4;
      while (u >= upp) { u -= upp; ++tap; }
    }
#pragma unroll
    for (int r = 0; r < MR; ++r)
#pragma unroll
      for (int j = 0; j < NF; ++j)
        acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wcur[j]),
                                                            xf[r], acc[r][j], 0, 0, 0);
  };
  for (int kc = 0; kc < nk; kc += 3) {
    weights(kc + 2, wb[2]);
    step(wb[0], kc);
    if (kc + 1 >= nk) break;
    weights(kc + 3, wb[0]);
    step(wb[1], kc + 1);
    if (kc + 2 >= nk) break;
    weights(kc + 4, wb[1]);
    step(wb[2], kc + 2);
  }
  const int cb = co0 + kq * (NT / 4);
  float bv[NT / 4];
#pragma unroll
  for (int e = 0; e < NT / 4; ++e) bv[e] = a.bias && cb + e < a.Cout ? a.bias[cb + e] : 0.0f;
#pragma unroll
  for (int r = 0; r < MR; ++r) {
    const int f = wm * MR + r, yy = py0 + f / kFx, xx = px0 + (f % kFx) * 16 + m;
    if (yy >= a.H || xx >= a.W) continue;
    float v[NT / 4];
#pragma unroll
    for (int e = 0; e < NT / 4; ++e) v[e] = acc[r][e / 4][e % 4] + bv[e];
    conv_out<MODE, NT / 4>(a, (((int64_t)n * a.H + yy) * a.W + xx) * a.Cout + cb, cb, v);
  }
}

// Weights of the data gradient: wt[ci][t][co] = w[co][8-t][ci] (taps flipped,
// channel roles swapped), so the data gradient is k_conv3x3 of the output
// gradient with wt.
__global__ __launch_bounds__(256) void k_flip_weights(const uint16_t* __restrict__ w, int Cout,
                                                      int Cin, uint16_t* __restrict__ wt) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t total = (int64_t)Cout * 9 * Cin;
  if (t >= total) return;
  const int co = (int)(t % Cout);
  const int tap = (int)((t / Cout) % 9);
  const int ci = (int)(t / ((int64_t)Cout * 9));
  wt[t] = w[((int64_t)co * 9 + (8 - tap)) * Cin + ci];
}

// Weight gradient dw[co][tap*Cin + ci] += sum_p dz[p][co] * x[p + tap][ci] and
// db[co] += sum_p dz[p][co]: a GEMM whose reduction runs over pixels.  Both
// operands lie with channels contiguous, so their fragments are read from LDS
// with the transposing ds_read_tr16_b64, which also makes the nine shifted
// windows plain row offsets.  A block of 8 waves owns CIT input x COT output
// channels and walks over 8 x 32 pixel tiles (two buffers, asynchronous loads);
// a wave owns 16 input channels, all COT output channels and the nine taps, and
// 1 / KS of the tile's rows.  The row parts are added in LDS at the end; the
// block's sums go to its own part of a workspace that k_wgrad_sum adds up, or,
// without one, into dw and db by FP32 atomics.
//
// LDS holds a pixel's CT channels as 32-byte slots (16 channels), slot s of tile
// column c at s ^ swizzle(c), so that the pixels c..c+3 and c+8..c+11 that half
// a wave reads hit distinct banks; rows repeat the pattern, so a lane's
// addresses are formed once and the rows are constant offsets.
template <int CT>
__device__ __forceinline__ int wg_slot(int p, int s) {
  if constexpr (CT == 64) return s ^ (((p >> 1) & 1) | (((p >> 3) & 1) << 1));
  if constexpr (CT == 32) return s ^ ((p >> 3) & 1);
  return s;
}

typedef short short4v __attribute__((ext_vector_type(4)));

// Element offset, in a tile row of CT channels per pixel, of what lane l reads
// for the k = 8 * (l / 16) + 4 * h .. + 3, m = l % 16 part of an MFMA operand
// that starts at column c0 with channel slot s.
template <int CT>
__device__ __forceinline__ int wg_lane(int c0, int s, int h, int l) {
  const int c = c0 + 8 * (l / 16) + 4 * h + (l % 16) / 4;
  return c * CT + wg_slot<CT>(c, s) * 16 + (l % 4) * 4;
}

__device__ __forceinline__ bf16x8 wg_frag(const uint16_t* p0, const uint16_t* p1) {
  const short4v a = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) short4v*)p0);
  const short4v b = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) short4v*)p1);
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

constexpr int kWgRows = 8;
constexpr int kWgThr = 512;
constexpr int kWgDzPx = kWgRows * kTileW, kWgXPx = (kWgRows + 2) * kWinW;

struct WgradArgs {
  ConvInput in;
  const uint16_t* dz;
  int N, H, W, Cout;
  float *dw, *db;
  float* part;  // per block (NCI * NCO * 10) sums of 16 x 16, or null
  int tx, ty, ntci, splits;
};

template <int CIT, int COT>
__global__ __launch_bounds__(kWgThr) void k_conv3x3_wgrad(WgradArgs a) {
  constexpr int NCI = CIT / 16, NCO = COT / 16, KS = 8 / NCI, RPW = kWgRows / KS;
  constexpr int kXU = kWgXPx * CIT / 8, kDU = kWgDzPx * COT / 8;  // 16-byte units
  constexpr int kXP = (kXU + kWgThr - 1) / kWgThr, kDP = (kDU + kWgThr - 1) / kWgThr;
  constexpr int kXS = kXP * kWgThr * kUnit, kDS = kDP * kWgThr * kUnit;
  __shared__ __align__(16) uint16_t lds[2 * (kXS + kDS)];
  auto sX = [&](int bf) { return lds + bf * kXS; };
  auto sD = [&](int bf) { return lds + 2 * kXS + bf * kDS; };
  const int pair = blockIdx.x / a.splits, split = blockIdx.x % a.splits;
  const int ci0 = (pair % a.ntci) * CIT, co0 = (pair / a.ntci) * COT;
  const int t = threadIdx.x, wave = t / 64, l = t % 64, m = l % 16, kq = l / 16;
  const int ci_s = wave % NCI, part = wave / NCI;
  const int C = a.in.C;
  const int ntile = a.N * a.ty * a.tx;
  const bool lo = ci0 < a.in.C1;  // uniform: C1 is a multiple of CIT
  const uint16_t* src = lo ? a.in.low + ci0 : a.in.x + (ci0 - a.in.C1);
  const int cs = lo ? a.in.C1 : C - a.in.C1, xleft = C - ci0, dleft = a.Cout - co0;
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  // this thread's units: pixel offset from the tile's first pixel (in the image
  // and in the half-size one), channel offset
  int rx[kXP], rl[kXP], cx[kXP], rd[kDP], cd[kDP];
#pragma unroll
  for (int i = 0; i < kXP; ++i) {
    const int u = i * kWgThr + t, p = u / (CIT / 8), us = u % (CIT / 8);
    const int r = p / kWinW - 1, c = p % kWinW - 1;
    rx[i] = r * a.W + c;
    rl[i] = (r >> 1) * (a.W / 2) + (c >> 1);
    cx[i] = wg_slot<CIT>(c + 1, us / 2) * 16 + (us % 2) * 8;
  }
#pragma unroll
  for (int i = 0; i < kDP; ++i) {
    const int u = i * kWgThr + t, p = u / (COT / 8), us = u % (COT / 8);
    rd[i] = (p / kTileW) * a.W + p % kTileW;
    cd[i] = wg_slot<COT>(p % kTileW, us / 2) * 16 + (us % 2) * 8;
  }
  auto fetch = [&](int tile, int bf) {
    const int px0 = (tile % a.tx) * kTileW, py0 = ((tile / a.tx) % a.ty) * kWgRows;
    const int n = tile / (a.tx * a.ty);
    const int64_t q0 = ((int64_t)n * a.H + py0) * a.W + px0;
    const uint16_t* xs =
        src + (lo ? ((int64_t)n * (a.H / 2) + py0 / 2) * (a.W / 2) + px0 / 2 : q0) * cs;
    const uint16_t* ds = a.dz + q0 * a.Cout + co0;
    // uniform: no unit lies outside the image or the channels
    const bool inside = px0 > 0 && px0 + kTileW < a.W && py0 > 0 && py0 + kWgRows < a.H &&
                        xleft >= CIT && dleft >= COT;
#pragma unroll
    for (int i = 0; i < kXP; ++i) {
      const int u = i * kWgThr + t;
      bool ok = true;
      if (!inside) {
        const int p = u / (CIT / 8), yy = py0 + p / kWinW - 1, xx = px0 + p % kWinW - 1;
        ok = yy >= 0 && yy < a.H && xx >= 0 && xx < a.W && cx[i] < xleft;
      }
      if (kXU % kWgThr != 0 && i == kXP - 1) ok = ok && u < kXU;
      if (ok)
        async16(xs + ((int64_t)(lo ? rl[i] : rx[i]) * cs + cx[i]),
                sX(bf) + (i * kWgThr + wave * 64) * kUnit);
      else *reinterpret_cast<uint4*>(sX(bf) + u * kUnit) = zero;
    }
#pragma unroll
    for (int i = 0; i < kDP; ++i) {
      const int u = i * kWgThr + t;
      bool ok = true;
      if (!inside) {
        const int p = u / (COT / 8);
        ok = py0 + p / kTileW < a.H && px0 + p % kTileW < a.W && cd[i] < dleft;
      }
      if (kDU % kWgThr != 0 && i == kDP - 1) ok = ok && u < kDU;
      if (ok)
        async16(ds + ((int64_t)rd[i] * a.Cout + cd[i]), sD(bf) + (i * kWgThr + wave * 64) * kUnit);
      else *reinterpret_cast<uint4*>(sD(bf) + u * kUnit) = zero;
    }
  };
  // this lane's addresses in the first row of its part
  int xl[3][2], dl[NCO][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      xl[k][h] = part * RPW * kWinW * CIT + wg_lane<CIT>(k, ci_s, h, l);
#pragma unroll
    for (int j = 0; j < NCO; ++j) dl[j][h] = part * RPW * kTileW * COT + wg_lane<COT>(0, j, h, l);
  }
  floatx4 acc[NCO][9], accb[NCO];
#pragma unroll
  for (int j = 0; j < NCO; ++j) {
    accb[j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < 9; ++k) acc[j][k] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  const bool bias = a.db && ci0 == 0 && ci_s == 0;
  const uint32_t one2 = 0x3f803f80u;
  const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(one2, one2, one2, one2));
  int tile = split;
  if (tile < ntile) fetch(tile, 0);
  lds_arrived();
  __syncthreads();
  for (int bf = 0; tile < ntile; tile += a.splits, bf ^= 1) {
    if (tile + a.splits < ntile) fetch(tile + a.splits, bf ^ 1);
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      bf16x8 d[NCO];
      const uint16_t* D = sD(bf) + r * kTileW * COT;
#pragma unroll
      for (int j = 0; j < NCO; ++j) d[j] = wg_frag(D + dl[j][0], D + dl[j][1]);
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        const uint16_t* X = sX(bf) + (r + k / 3) * kWinW * CIT;
        const bf16x8 x = wg_frag(X + xl[k % 3][0], X + xl[k % 3][1]);
#pragma unroll
        for (int j = 0; j < NCO; ++j)
          acc[j][k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d[j], x, acc[j][k], 0, 0, 0);
      }
      if (bias) {
#pragma unroll
        for (int j = 0; j < NCO; ++j)
          accb[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d[j], ones, accb[j], 0, 0, 0);
      }
    }
    lds_arrived();
    __syncthreads();
  }
  // the row parts of a wave's channels: added up in LDS, part by part
  float* red = reinterpret_cast<float*>(lds);
  constexpr int kRed = NCO * 10 * 4 * 64;  // floats of one wave
  static_assert(NCI * kRed * 4 <= 4 * (kXS + kDS), "the sums fit the tiles' LDS");
  for (int q = 1; q < KS; ++q) {
    if (part == q) {
#pragma unroll
      for (int j = 0; j < NCO; ++j)
#pragma unroll
        for (int k = 0; k < 10; ++k)
          *reinterpret_cast<floatx4*>(red + ci_s * kRed + ((j * 10 + k) * 64 + l) * 4) =
              k < 9 ? acc[j][k < 9 ? k : 0] : accb[j];
    }
    __syncthreads();
    if (part == 0) {
#pragma unroll
      for (int j = 0; j < NCO; ++j)
#pragma unroll
        for (int k = 0; k < 10; ++k) {
          const floatx4 v =
              *reinterpret_cast<const floatx4*>(red + ci_s * kRed + ((j * 10 + k) * 64 + l) * 4);
          if (k < 9) acc[j][k < 9 ? k : 0] += v;
          else accb[j] += v;
        }
    }
    __syncthreads();
  }
  if (part != 0) return;
  if (a.part) {
    float* o = a.part + ((int64_t)(pair * a.splits + split) * NCI + ci_s) * kRed;
#pragma unroll
    for (int j = 0; j < NCO; ++j)
#pragma unroll
      for (int k = 0; k < 10; ++k)
        *reinterpret_cast<floatx4*>(o + ((j * 10 + k) * 64 + l) * 4) =
            k < 9 ? acc[j][k < 9 ? k : 0] : accb[j];
    return;
  }
  const int K = 9 * C, ci = ci0 + ci_s * 16 + m;
#pragma unroll
  for (int j = 0; j < NCO; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int co = co0 + j * 16 + kq * 4 + i;
      if (co >= a.Cout) continue;
      if (ci < C) {
#pragma unroll
        for (int k = 0; k < 9; ++k) atomicAdd(a.dw + (int64_t)co * K + k * C + ci, acc[j][k][i]);
      }
      if (bias && m == 0) atomicAdd(a.db + co, accb[j][i]);
    }
}

// dw and db += the blocks' sums: a thread adds four sums over an eighth of the
// splits, the eighths are added in LDS in order.
__global__ __launch_bounds__(256) void k_wgrad_sum(const float* __restrict__ part, int splits,
                                                   int nci, int nco, int ntci, int pairs, int C,
                                                   int Cout, float* __restrict__ dw,
                                                   float* __restrict__ db) {
  __shared__ floatx4 red[8][32];
  const int per = nci * nco * 10 * 64;  // float4 sums of one pair
  const int item = threadIdx.x % 32, eighth = threadIdx.x / 32;
  const int64_t t = (int64_t)blockIdx.x * 32 + item;  // pairs * per is a multiple of 32
  const int pair = (int)(t / per), r = (int)(t - (int64_t)pair * per);
  floatx4 s = {0.0f, 0.0f, 0.0f, 0.0f};
  const float* p = part + (int64_t)pair * splits * per * 4 + (int64_t)r * 4;
#pragma unroll 4
  for (int q = eighth; q < splits; q += 8)
    s += *reinterpret_cast<const floatx4*>(p + (int64_t)q * per * 4);
  red[eighth][item] = s;
  __syncthreads();
  if (eighth != 0) return;
  for (int e = 1; e < 8; ++e) s += red[e][item];
  const int l = r % 64, k = (r / 64) % 10, j = (r / 640) % nco, ci_s = r / (640 * nco);
  const int ci = (pair % ntci) * nci * 16 + ci_s * 16 + l % 16;
  const int co = (pair / ntci) * nco * 16 + j * 16 + (l / 16) * 4;
  const bool bias = k == 9;
  if (bias ? !(db && ci == 0) : ci >= C) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (co + i >= Cout) continue;
    if (bias) db[co + i] += s[i];
    else dw[(int64_t)(co + i) * 9 * C + k * C + ci] += s[i];
  }
}

// k_flip_weights for several layers at once: 32 x 32 (co, ci) tiles of one tap
// through LDS, so that both sides move whole rows.
struct FlipTable {
  int n;
  int cout[SEIS_UNET_MAX_LAYERS], cin[SEIS_UNET_MAX_LAYERS];
  int first[SEIS_UNET_MAX_LAYERS + 1];  // first block of each layer
  int64_t in[SEIS_UNET_MAX_LAYERS], out[SEIS_UNET_MAX_LAYERS];
};

__global__ __launch_bounds__(256) void k_flip_layers(const uint16_t* __restrict__ w, FlipTable f,
                                                     uint16_t* __restrict__ wt) {
  __shared__ uint16_t s[32][33];
  int q = 0;
  while (q + 1 < f.n && (int)blockIdx.x >= f.first[q + 1]) ++q;
  const int cout = f.cout[q], cin = f.cin[q], tci = (cin + 31) / 32, tco = (cout + 31) / 32;
  int b = (int)blockIdx.x - f.first[q];
  const int ci0 = (b % tci) * 32;
  b /= tci;
  const int co0 = (b % tco) * 32, tap = b / tco;
  const int x = threadIdx.x % 32, y0 = threadIdx.x / 32;
  const uint16_t* W = w + f.in[q];
  uint16_t* O = wt + f.out[q];
  for (int y = y0; y < 32; y += 8)
    if (co0 + y < cout && ci0 + x < cin)
      s[y][x] = W[((int64_t)(co0 + y) * 9 + (8 - tap)) * cin + ci0 + x];
  __syncthreads();
  for (int y = y0; y < 32; y += 8)
    if (ci0 + y < cin && co0 + x < cout)
      O[((int64_t)(ci0 + y) * 9 + tap) * cout + co0 + x] = s[x][y];
}

// ----------------------------------------------------------- elementwise

// dz = dy * gelu'(z), rounded to bf16 (the operand of the next GEMMs).
__global__ __launch_bounds__(256) void k_gelu_bwd(const float* __restrict__ dy,
                                                  const uint16_t* __restrict__ z, int64_t n,
                                                  uint16_t* __restrict__ dz) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) dz[t] = f2bf(dy[t] * gelu_grad(bf2f(z[t])));
}

// The gradients of a concatenation's two parts taken through the activations
// that made them, 8 channels per thread.  low: dz = bf16((sum of the 2x2
// children of dout's first C1 channels) * gelu'(z)), (N, H/2, W/2, C1).
__global__ __launch_bounds__(256) void k_up_gelu_bwd(const float* __restrict__ dout, int N, int H,
                                                     int W, int C1, int C2,
                                                     const uint16_t* __restrict__ z,
                                                     uint16_t* __restrict__ dz) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = H / 2, Wo = W / 2, C = C1 + C2, g = C1 / 8;
  if (t >= (int64_t)N * Ho * Wo * g) return;
  const int c = (int)(t % g) * 8;
  const int64_t q = t / g;
  const int xo = (int)(q % Wo), yo = (int)((q / Wo) % Ho);
  const int n = (int)(q / ((int64_t)Wo * Ho));
  const float* b = dout + (((int64_t)n * H + 2 * yo) * W + 2 * xo) * C + c;
  float d[4][8], zz[8], v[8];
  load8f(b, d[0]);
  load8f(b + C, d[1]);
  load8f(b + (int64_t)W * C, d[2]);
  load8f(b + (int64_t)W * C + C, d[3]);
  unpack8(z + q * C1 + c, zz);
#pragma unroll
  for (int e = 0; e < 8; ++e)
    v[e] = ((d[0][e] + d[1][e]) + (d[2][e] + d[3][e])) * gelu_grad(zz[e]);
  pack8(dz + q * C1 + c, v);
}

// skip: dz = bf16((dout's channels from C1 on + a quarter of the pooled
// gradient) * gelu'(z)), (N, H, W, C2); dpool (N, H/2, W/2, C2).
__global__ __launch_bounds__(256) void k_skip_gelu_bwd(const float* __restrict__ dout,
                                                       const float* __restrict__ dpool, int N,
                                                       int H, int W, int C1, int C2,
                                                       const uint16_t* __restrict__ z,
                                                       uint16_t* __restrict__ dz) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int g = C2 / 8;
  if (t >= (int64_t)N * H * W * g) return;
  const int c = (int)(t % g) * 8;
  const int64_t q = t / g;
  const int xx = (int)(q % W), yy = (int)((q / W) % H);
  const int n = (int)(q / ((int64_t)W * H));
  float d[8], p[8], zz[8], v[8];
  load8f(dout + q * (C1 + C2) + C1 + c, d);
  load8f(dpool + (((int64_t)n * (H / 2) + yy / 2) * (W / 2) + xx / 2) * C2 + c, p);
  unpack8(z + q * C2 + c, zz);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (d[e] + 0.25f * p[e]) * gelu_grad(zz[e]);
  pack8(dz + q * C2 + c, v);
}

__global__ __launch_bounds__(256) void k_to_bf16(const float* __restrict__ x, int64_t n,
                                                 uint16_t* __restrict__ y) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) y[t] = f2bf(x[t]);
}

// 2x2 average pooling, (N, H, W, C) -> (N, H/2, W/2, C); H, W even.
__global__ __launch_bounds__(256) void k_avgpool2(const uint16_t* __restrict__ x, int N, int H,
                                                  int W, int C, uint16_t* __restrict__ y) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = H / 2, Wo = W / 2;
  if (t >= (int64_t)N * Ho * Wo * C) return;
  const int c = (int)(t % C);
  const int64_t q = t / C;
  const int xo = (int)(q % Wo);
  const int yo = (int)((q / Wo) % Ho);
  const int n = (int)(q / ((int64_t)Wo * Ho));
  const int64_t b = (((int64_t)n * H + 2 * yo) * W + 2 * xo) * C + c;
  const float s = (bf2f(x[b]) + bf2f(x[b + C])) + (bf2f(x[b + (int64_t)W * C]) +
                                                   bf2f(x[b + (int64_t)W * C + C]));
  y[t] = f2bf(0.25f * s);
}

// k_avgpool2 with 8 channels per thread (C a multiple of 8).
__global__ __launch_bounds__(256) void k_avgpool2_v(const uint16_t* __restrict__ x, int N, int H,
                                                    int W, int C, uint16_t* __restrict__ y) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = H / 2, Wo = W / 2, g = C / 8;
  if (t >= (int64_t)N * Ho * Wo * g) return;
  const int c = (int)(t % g) * 8;
  const int64_t q = t / g;
  const int xo = (int)(q % Wo), yo = (int)((q / Wo) % Ho);
  const int n = (int)(q / ((int64_t)Wo * Ho));
  const uint16_t* b = x + (((int64_t)n * H + 2 * yo) * W + 2 * xo) * C + c;
  float d[4][8], v[8];
  unpack8(b, d[0]);
  unpack8(b + C, d[1]);
  unpack8(b + (int64_t)W * C, d[2]);
  unpack8(b + (int64_t)W * C + C, d[3]);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = 0.25f * ((d[0][e] + d[1][e]) + (d[2][e] + d[3][e]));
  pack8(y + q * C + c, v);
}

// dx (N, H, W, C) = 0.25 * dy[pixel / 2] (+= dx if accumulate).
__global__ __launch_bounds__(256) void k_avgpool2_bwd(const float* __restrict__ dy, int N, int H,
                                                      int W, int C, float* __restrict__ dx,
                                                      int accumulate) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)N * H * W * C) return;
  const int c = (int)(t % C);
  const int64_t q = t / C;
  const int xx = (int)(q % W);
  const int yy = (int)((q / W) % H);
  const int n = (int)(q / ((int64_t)W * H));
  const float g = 0.25f * dy[(((int64_t)n * (H / 2) + yy / 2) * (W / 2) + xx / 2) * C + c];
  dx[t] = accumulate ? dx[t] + g : g;
}

// out (N, H, W, C1 + C2) = [nearest 2x upsampling of low (N, H/2, W/2, C1), skip].
__global__ __launch_bounds__(256) void k_up_concat(const uint16_t* __restrict__ low,
                                                   const uint16_t* __restrict__ skip, int N,
                                                   int H, int W, int C1, int C2,
                                                   uint16_t* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int C = C1 + C2;
  if (t >= (int64_t)N * H * W * C) return;
  const int c = (int)(t % C);
  const int64_t q = t / C;  // pixel
  const int xx = (int)(q % W);
  const int yy = (int)((q / W) % H);
  const int n = (int)(q / ((int64_t)W * H));
  out[t] = c < C1 ? low[(((int64_t)n * (H / 2) + yy / 2) * (W / 2) + xx / 2) * C1 + c]
                  : skip[q * C2 + (c - C1)];
}

// Gradient of k_up_concat: dlow = sum of the 2x2 children; dskip (+)= its slice.
__global__ __launch_bounds__(256) void k_up_concat_bwd_low(const float* __restrict__ dout,
                                                           int N, int H, int W, int C1, int C2,
                                                           float* __restrict__ dlow) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = H / 2, Wo = W / 2, C = C1 + C2;
  if (t >= (int64_t)N * Ho * Wo * C1) return;
  const int c = (int)(t % C1);
  const int64_t q = t / C1;
  const int xo = (int)(q % Wo);
  const int yo = (int)((q / Wo) % Ho);
  const int n = (int)(q / ((int64_t)Wo * Ho));
  const int64_t b = (((int64_t)n * H + 2 * yo) * W + 2 * xo) * C + c;
  dlow[t] = (dout[b] + dout[b + C]) + (dout[b + (int64_t)W * C] + dout[b + (int64_t)W * C + C]);
}

__global__ __launch_bounds__(256) void k_up_concat_bwd_skip(const float* __restrict__ dout,
                                                            int64_t P, int C1, int C2,
                                                            float* __restrict__ dskip,
                                                            int accumulate) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P * C2) return;
  const int64_t q = t / C2;
  const int c = (int)(t % C2);
  const float g = dout[q * (C1 + C2) + C1 + c];
  dskip[t] = accumulate ? dskip[t] + g : g;
}

// Network input: channel 0 = grad * gscale, channel 1 = (model - mshift) * mscale,
// channels 2..7 zero; (N, H, W) FP32 planes -> (N, H, W, 8) bf16.
__global__ __launch_bounds__(256) void k_pack_input(const float* __restrict__ g,
                                                    const float* __restrict__ mdl, int64_t P,
                                                    const float* __restrict__ scales,
                                                    int64_t plane, uint16_t* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P) return;
  const int64_t n = t / plane;
  const float gs = scales[3 * n], ms = scales[3 * n + 1], mm = scales[3 * n + 2];
  const uint32_t lo = (uint32_t)f2bf(g[t] * gs) | ((uint32_t)f2bf((mdl[t] - mm) * ms) << 16);
  *reinterpret_cast<uint4*>(out + t * 8) = make_uint4(lo, 0u, 0u, 0u);
}

// 1x1 head to one channel: out[p] = sum_c x[p][c] * w[c] + b (FP32).
__global__ __launch_bounds__(256) void k_head_fwd(const uint16_t* __restrict__ x, int64_t P, int C,
                                                  const float* __restrict__ w,
                                                  const float* __restrict__ b,
                                                  float* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P) return;
  float s = 0.0f;
  for (int c = 0; c < C; ++c) s += bf2f(x[t * C + c]) * w[c];
  out[t] = s + b[0];
}

// k_head_fwd with 16-byte loads (C = 8 * G); the channels in the same order, since the
// training gradient's roundings follow from the output.
template <int G>
__global__ __launch_bounds__(256) void k_head_fwd_v(const uint16_t* __restrict__ x, int64_t P,
                                                    const float* __restrict__ w,
                                                    const float* __restrict__ b,
                                                    float* __restrict__ out) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  float xv[G][8];
#pragma unroll
  for (int q = 0; q < G; ++q) unpack8(x + (p * G + q) * 8, xv[q]);
  float s = 0.0f;
#pragma unroll
  for (int q = 0; q < G; ++q)
#pragma unroll
    for (int e = 0; e < 8; ++e) s += xv[q][e] * w[q * 8 + e];
  out[p] = s + b[0];
}

// Head gradient taken through the last activation, 8 channels per thread and
// G threads per pixel: dz[p][c] = bf16(dout[p] * w[c] * gelu'(z[p][c])); dw[c]
// += sum_p dout[p] x[p][c]; db += sum_p dout[p] (summed in registers over the
// block's pixels, then in LDS, one atomic per block and channel).
template <int G>
__global__ __launch_bounds__(256) void k_head_gelu_bwd(const uint16_t* __restrict__ x,
                                                       const float* __restrict__ dout, int64_t P,
                                                       const float* __restrict__ w,
                                                       const uint16_t* __restrict__ z,
                                                       uint16_t* __restrict__ dz,
                                                       float* __restrict__ dw,
                                                       float* __restrict__ db) {
  __shared__ float red[256 / G][8 * G + 1];
  const int c = (int)(threadIdx.x % G) * 8, lp = threadIdx.x / G;
  float wv[8], sw[8] = {}, sb = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) wv[e] = w[c + e];
  for (int64_t p = (int64_t)blockIdx.x * (256 / G) + lp; p < P; p += (int64_t)gridDim.x * (256 / G)) {
    const float d = dout[p];
    float xv[8], zv[8], v[8];
    unpack8(x + p * 8 * G + c, xv);
    unpack8(z + p * 8 * G + c, zv);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = d * wv[e] * gelu_grad(zv[e]);
      sw[e] += d * xv[e];
    }
    sb += d;
    pack8(dz + p * 8 * G + c, v);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) red[lp][c + e] = sw[e];
  if (c == 0) red[lp][8 * G] = sb;
  __syncthreads();
  if (threadIdx.x <= 8 * G) {
    float s = 0.0f;
    for (int q = 0; q < 256 / G; ++q) s += red[q][threadIdx.x];
    atomicAdd(threadIdx.x < 8 * G ? dw + threadIdx.x : db, s);
  }
}

// Head gradient: dx[p][c] = dout[p] * w[c]; dw[c] += sum_p dout[p] x[p][c];
// db += sum_p dout[p].  One block per 256 pixels; thread c < C sums its channel.
__global__ __launch_bounds__(256) void k_head_bwd(const uint16_t* __restrict__ x,
                                                  const float* __restrict__ dout, int64_t P,
                                                  int C, const float* __restrict__ w,
                                                  float* __restrict__ dx, float* __restrict__ dw,
                                                  float* __restrict__ db) {
  const int64_t p0 = (int64_t)blockIdx.x * 256;
  const int64_t p1 = p0 + 256 < P ? p0 + 256 : P;
  for (int64_t e = threadIdx.x; e < (p1 - p0) * C; e += blockDim.x) {
    const int64_t p = p0 + e / C;
    const int c = (int)(e % C);
    dx[p * C + c] = dout[p] * w[c];
  }
  if (threadIdx.x < C) {
    const int c = threadIdx.x;
    float s = 0.0f;
    for (int64_t p = p0; p < p1; ++p) s += dout[p] * bf2f(x[p * C + c]);
    atomicAdd(dw + c, s);
  } else if (threadIdx.x == 255) {
    float s = 0.0f;
    for (int64_t p = p0; p < p1; ++p) s += dout[p];
    atomicAdd(db, s);
  }
}

// Masked mean squared error: loss += sum mask*(pred-target)^2 / count,
// dpred = 2*mask*(pred-target)/count.
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ pred,
                                             const float* __restrict__ target,
                                             const float* __restrict__ mask, int64_t n,
                                             float inv_count, float* __restrict__ loss,
                                             float* __restrict__ dpred) {
  __shared__ float red[256];
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  float e = 0.0f;
  if (t < n) {
    const float mk = mask ? mask[t] : 1.0f;
    const float r = mk * (pred[t] - target[t]);
    dpred[t] = 2.0f * r * inv_count;
    e = r * r * inv_count;
  }
  red[threadIdx.x] = e;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

// AdamW (decoupled weight decay) on FP32 master weights; refreshes the bf16 copy.
__global__ __launch_bounds__(256) void k_adamw(float* __restrict__ p, const float* __restrict__ g,
                                               float* __restrict__ m, float* __restrict__ v,
                                               int64_t n, float lr, float b1, float b2, float eps,
                                               float wd, float bc1, float bc2,
                                               uint16_t* __restrict__ pb) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  float w = p[t];
  w -= lr * wd * w;
  const float gt = g[t];
  const float mt = b1 * m[t] + (1.0f - b1) * gt;
  const float vt = b2 * v[t] + (1.0f - b2) * gt * gt;
  m[t] = mt;
  v[t] = vt;
  w -= lr * (mt / bc1) / (sqrtf(vt / bc2) + eps);
  p[t] = w;
  if (pb) pb[t] = f2bf(w);
}

__global__ __launch_bounds__(256) void k_fill_f32(float* __restrict__ p, int64_t n, float v) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = v;
}

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int conv_grid(ConvArgs& a, int rows, int cols, int channels) {
  a.tx = (a.W + cols - 1) / cols;
  a.ty = (a.H + rows - 1) / rows;
  a.ntile = (a.Cout + channels - 1) / channels;
  const int64_t units = (int64_t)a.N * a.ty * a.tx * a.ntile;
  SEIS_CHECK_ARG(units < ((int64_t)1 << 31) - 8, "too many tiles");
  a.per = (int)((units + 7) / 8);
  return 0;
}

template <int TH, int TW, int MR, int NF, int WM, int WN, int KIND, int MODE>
int launch_conv(ConvArgs a, hipStream_t s) {
  if (int e = conv_grid(a, TH, TW, 16 * NF * WN)) return e;
  const int lds = KIND == kFar ? 0 : (TH + 2) * (TW + 2) * a.in.C * 2;
  auto* k = k_conv3x3<TH, TW, MR, NF, WM, WN, KIND, MODE>;
  SEIS_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  k<<<(unsigned)(a.per * 8), 64 * WM * WN, lds, s>>>(a);
  SEIS_CHECK_LAUNCH();
  return 0;
}

template <int WAVES, int RW, int MODE>
int launch_grad32(ConvArgs a, hipStream_t s) {
  if (int e = conv_grid(a, WAVES * RW, kTileW, 32)) return e;
  k_conv3x3_grad32<WAVES, RW, MODE><<<(unsigned)(a.per * 8), WAVES * 64, 0, s>>>(a);
  SEIS_CHECK_LAUNCH();
  return 0;
}

template <int MODE>
int pick_conv(ConvArgs a, hipStream_t s) {
  while (a.lg < 4 && (a.in.C / 8) % (2 << a.lg) == 0) ++a.lg;
  const int C = a.in.C;
  if constexpr (MODE != kConvAct) {
    // 16 rows of 32 pixels per block, 4 where small images would leave CUs without
    // two blocks
    if (C == 32) {
      const int64_t b8 = (int64_t)a.N * ((a.H + 7) / 8) * ((a.W + kTileW - 1) / kTileW) *
                         ((a.Cout + 31) / 32);
      return b8 < 512 ? launch_grad32<4, 1, MODE>(a, s) : launch_grad32<8, 2, MODE>(a, s);
    }
  }
  // Tile and waves by what the window leaves of the LDS, the best of 14 shapes at
  // the layers of an 800 x 2400 image.  us, now and with blocks of one row of 64
  // pixels that reload their window per 32 channels: 32 -> 32 channels 159 and 200,
  // 64 -> 64 at half the size 117 and 112, 128 -> 128 at a quarter 95 and 108, 256 ->
  // 256 at an eighth 83 and 103, and with the concatenation's pass (676 MB written over
  // the four levels) before it 96 -> 32 301 and 480, 192 -> 64 264 and 295, 384 -> 128 285
  // and 314, 512 -> 256 164 and 209.
  if constexpr (MODE == kConvAct) {
    if (a.Cout <= 32 && C == 32) return launch_conv<8, 32, 4, 2, 4, 1, kOne, MODE>(a, s);
    if (C == 32) return launch_conv<4, 16, 4, 2, 1, 2, kOne, MODE>(a, s);
  }
  if (a.Cout <= 32 && C <= 128) return launch_conv<8, 32, 4, 2, 4, 1, kAny, MODE>(a, s);
  if (C <= 64) return launch_conv<4, 16, 4, 2, 1, 2, kAny, MODE>(a, s);
  if (C <= 128 || (C > 192 && C <= 256)) return launch_conv<4, 16, 4, 2, 1, 4, kAny, MODE>(a, s);
  if (C <= 192) return launch_conv<4, 32, 4, 2, 2, 2, kAny, MODE>(a, s);
  if (C <= 384) return launch_conv<4, 32, 4, 4, 2, 2, kAny, MODE>(a, s);
  if (C <= 512) return launch_conv<4, 16, 4, 4, 1, 4, kAny, MODE>(a, s);
  return launch_conv<4, 16, 4, 4, 1, 4, kFar, MODE>(a, s);
}

int conv(int mode, const ConvInput& in, int32_t N, int32_t H, int32_t W, const uint16_t* w,
         const float* bias, int32_t Cout, int32_t act, uint16_t* z, uint16_t* y, float* yf,
         hipStream_t s) {
  SEIS_CHECK_ARG(N >= 1 && H >= 1 && W >= 1, "empty image batch");
  SEIS_CHECK_ARG(in.C >= 8 && in.C % 8 == 0 && in.C <= 4096, "Cin %d must be a multiple of 8",
                 in.C);
  SEIS_CHECK_ARG(Cout >= 1 && Cout <= 4096, "Cout %d outside [1, 4096]", Cout);
  SEIS_CHECK_ARG(in.x && w && aligned16(in.x) && aligned16(w), "x and w must be 16-byte aligned");
  SEIS_CHECK_ARG((y != nullptr) != (yf != nullptr), "exactly one of y (bf16) and y_f32");
  SEIS_CHECK_ARG(y || (!z && !act), "z and act apply to the bf16 output only");
  SEIS_CHECK_ARG((int64_t)N * H <= (int64_t)1 << 24, "too many image rows");
  const int vec = Cout % 8 == 0 && aligned16(z) && aligned16(y) && aligned16(yf);
  const ConvArgs a{in, N, H, W, w, bias, Cout, act, z, y, yf, vec, 0, 0, 0, 0, 0};
  if (mode == kConvAct) return pick_conv<kConvAct>(a, s);
  if (mode == kConvF32) return pick_conv<kConvF32>(a, s);
  return pick_conv<kConvGeluGrad>(a, s);
}

int check_cat(const uint16_t* low, int32_t C1, const uint16_t* skip, int32_t C2, int32_t H,
              int32_t W) {
  SEIS_CHECK_ARG(low && skip && aligned16(low) && aligned16(skip),
                 "low and skip must be 16-byte aligned");
  SEIS_CHECK_ARG(C1 >= 64 && C1 % 64 == 0 && C2 >= 8 && C2 % 8 == 0,
                 "channel counts (%d, %d): C1 a multiple of 64, C2 of 8", C1, C2);
  SEIS_CHECK_ARG(H % 2 == 0 && W % 2 == 0, "upsampled sizes must be even");
  return 0;
}

// Tiles of a weight gradient: input and output channels per block, blocks.
struct WgradPlan {
  int cit, cot, ntci;
  int64_t pairs, splits, part;  // part: floats of the workspace
};

WgradPlan plan_wgrad(int N, int H, int W, int C, int Cout) {
  WgradPlan p;
  p.cit = C <= 16 ? 16 : C <= 32 ? 32 : 64;
  p.cot = Cout <= 32 ? 32 : 64;
  p.ntci = (C + p.cit - 1) / p.cit;
  p.pairs = (int64_t)p.ntci * ((Cout + p.cot - 1) / p.cot);
  const int64_t tiles =
      (int64_t)N * ((W + kTileW - 1) / kTileW) * ((H + kWgRows - 1) / kWgRows);
  // the LDS of one block (two for the narrow tiles) fills a CU: one round of blocks
  const int64_t blocks = p.cit * p.cot <= 1024 ? 512 : 256;
  p.splits = std::max<int64_t>(1, std::min<int64_t>(tiles, blocks / p.pairs));
  p.part = p.pairs * p.splits * (p.cit / 16) * (p.cot / 16) * 10 * 256;
  return p;
}

template <int CIT, int COT>
int launch_wgrad(WgradArgs a, const WgradPlan& p, hipStream_t s) {
  a.tx = (a.W + kTileW - 1) / kTileW;
  a.ty = (a.H + kWgRows - 1) / kWgRows;
  a.ntci = p.ntci;
  a.splits = (int)p.splits;
  k_conv3x3_wgrad<CIT, COT><<<(unsigned)(p.pairs * p.splits), kWgThr, 0, s>>>(a);
  SEIS_CHECK_LAUNCH();
  if (a.part) {
    const int64_t n = p.pairs * (CIT / 16) * (COT / 16) * 640;
    k_wgrad_sum<<<(unsigned)(n / 32), 256, 0, s>>>(a.part, a.splits, CIT / 16, COT / 16, a.ntci,
                                              (int)p.pairs, a.in.C, a.Cout, a.dw, a.db);
    SEIS_CHECK_LAUNCH();
  }
  return 0;
}

int wgrad(const ConvInput& in, const uint16_t* dz, int32_t N, int32_t H, int32_t W, int32_t Cout,
          float* dw, float* db, float* part, hipStream_t s) {
  SEIS_CHECK_ARG(N >= 1 && H >= 1 && W >= 1, "empty image batch");
  SEIS_CHECK_ARG(in.C >= 8 && Cout >= 8 && in.C <= 4096 && Cout <= 4096 && in.C % 8 == 0 &&
                     Cout % 8 == 0,
                 "channel counts (%d, %d) must be multiples of 8", in.C, Cout);
  SEIS_CHECK_ARG(in.x && dz && dw, "null pointer argument");
  SEIS_CHECK_ARG(aligned16(in.x) && aligned16(dz) && aligned16(part),
                 "x, dz and work must be 16-byte aligned");
  const WgradPlan p = plan_wgrad(N, H, W, in.C, Cout);
  const WgradArgs a{in, dz, N, H, W, Cout, dw, db, part, 0, 0, 0, 0};
  switch (p.cit + p.cot) {
    case 48: return launch_wgrad<16, 32>(a, p, s);
    case 80: return launch_wgrad<16, 64>(a, p, s);
    case 64: return launch_wgrad<32, 32>(a, p, s);
    case 96: return p.cit == 32 ? launch_wgrad<32, 64>(a, p, s) : launch_wgrad<64, 32>(a, p, s);
    default: return launch_wgrad<64, 64>(a, p, s);
  }
}

}  // namespace

extern "C" {

int seis_unet_conv3x3(const uint16_t* x, int32_t N, int32_t H, int32_t W, int32_t Cin,
                      const uint16_t* w, const float* bias, int32_t Cout, int32_t act,
                      uint16_t* z, uint16_t* y, float* y_f32, void* stream) {
  return conv(y ? kConvAct : kConvF32, {x, nullptr, Cin, 0}, N, H, W, w, bias, Cout, act, z, y,
              y_f32, (hipStream_t)stream);
}

int seis_unet_conv3x3_cat(const uint16_t* low, int32_t C1, const uint16_t* skip, int32_t C2,
                          int32_t N, int32_t H, int32_t W, const uint16_t* w, const float* bias,
                          int32_t Cout, int32_t act, uint16_t* z, uint16_t* y, void* stream) {
  if (int e = check_cat(low, C1, skip, C2, H, W)) return e;
  SEIS_CHECK_ARG(y, "null output");
  return conv(kConvAct, {skip, low, C1 + C2, C1}, N, H, W, w, bias, Cout, act, z, y, nullptr,
              (hipStream_t)stream);
}

int seis_unet_conv3x3_gelu_grad(const uint16_t* dz, int32_t N, int32_t H, int32_t W, int32_t Cout,
                                const uint16_t* wt, int32_t Cin, const uint16_t* z, uint16_t* dzp,
                                void* stream) {
  SEIS_CHECK_ARG(z && dzp && aligned16(z), "null or misaligned activation");
  return conv(kConvGeluGrad, {dz, nullptr, Cout, 0}, N, H, W, wt, nullptr, Cin, 0,
              const_cast<uint16_t*>(z), dzp, nullptr, (hipStream_t)stream);
}

int seis_unet_flip_weights(const uint16_t* w, int32_t Cout, int32_t Cin, uint16_t* wt,
                           void* stream) {
  SEIS_CHECK_ARG(w && wt && Cout >= 1 && Cin >= 1, "bad arguments");
  const int64_t n = (int64_t)Cout * 9 * Cin;
  k_flip_weights<<<blocks_for(n), 256, 0, (hipStream_t)stream>>>(w, Cout, Cin, wt);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_flip_layers(const uint16_t* w, int32_t n, const int64_t* layers, uint16_t* wt,
                          void* stream) {
  SEIS_CHECK_ARG(w && layers && wt && n >= 1 && n <= SEIS_UNET_MAX_LAYERS, "bad arguments");
  FlipTable f{};
  f.n = n;
  int64_t blocks = 0, out = 0;
  for (int q = 0; q < n; ++q) {
    const int64_t cout = layers[3 * q + 1], cin = layers[3 * q + 2];
    SEIS_CHECK_ARG(cout >= 1 && cin >= 1 && cout <= 4096 && cin <= 4096 && layers[3 * q] >= 0,
                   "layer %d: %lld x %lld", q, (long long)cout, (long long)cin);
    f.in[q] = layers[3 * q];
    f.out[q] = out;
    f.cout[q] = (int)cout;
    f.cin[q] = (int)cin;
    f.first[q] = (int)blocks;
    blocks += 9 * ((cout + 31) / 32) * ((cin + 31) / 32);
    out += cout * 9 * cin;
  }
  k_flip_layers<<<(unsigned)blocks, 256, 0, (hipStream_t)stream>>>(w, f, wt);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_conv3x3_wgrad(const uint16_t* x, const uint16_t* dz, int32_t N, int32_t H,
                            int32_t W, int32_t Cin, int32_t Cout, float* dw, float* db,
                            void* stream) {
  return wgrad({x, nullptr, Cin, 0}, dz, N, H, W, Cout, dw, db, nullptr, (hipStream_t)stream);
}

int64_t seis_unet_wgrad_workspace(int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout) {
  return N < 1 || H < 1 || W < 1 || Cin < 1 || Cout < 1 ? 0
                                                        : plan_wgrad(N, H, W, Cin, Cout).part;
}

int seis_unet_conv3x3_wgrad_ws(const uint16_t* low, int32_t C1, const uint16_t* x, int32_t C2,
                               const uint16_t* dz, int32_t N, int32_t H, int32_t W, int32_t Cout,
                               float* dw, float* db, float* work, void* stream) {
  SEIS_CHECK_ARG(work, "null workspace");
  if (!low) return wgrad({x, nullptr, C2, 0}, dz, N, H, W, Cout, dw, db, work, (hipStream_t)stream);
  if (int e = check_cat(low, C1, x, C2, H, W)) return e;
  return wgrad({x, low, C1 + C2, C1}, dz, N, H, W, Cout, dw, db, work, (hipStream_t)stream);
}

int seis_unet_gelu_bwd(const float* dy, const uint16_t* z, int64_t n, uint16_t* dz, void* stream) {
  SEIS_CHECK_ARG(dy && z && dz && n >= 0, "bad arguments");
  if (n == 0) return 0;
  k_gelu_bwd<<<blocks_for(n), 256, 0, (hipStream_t)stream>>>(dy, z, n, dz);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_to_bf16(const float* x, int64_t n, uint16_t* y, void* stream) {
  SEIS_CHECK_ARG(x && y && n >= 0, "bad arguments");
  if (n == 0) return 0;
  k_to_bf16<<<blocks_for(n), 256, 0, (hipStream_t)stream>>>(x, n, y);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_avgpool2(const uint16_t* x, int32_t N, int32_t H, int32_t W, int32_t C, uint16_t* y,
                       void* stream) {
  SEIS_CHECK_ARG(x && y && N >= 1 && C >= 1 && H >= 2 && W >= 2 && H % 2 == 0 && W % 2 == 0,
                 "avgpool2 needs even H, W");
  const int64_t n = (int64_t)N * (H / 2) * (W / 2) * C;
  if (C % 8 == 0 && aligned16(x) && aligned16(y))
    k_avgpool2_v<<<blocks_for(n / 8), 256, 0, (hipStream_t)stream>>>(x, N, H, W, C, y);
  else
    k_avgpool2<<<blocks_for(n), 256, 0, (hipStream_t)stream>>>(x, N, H, W, C, y);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_avgpool2_bwd(const float* dy, int32_t N, int32_t H, int32_t W, int32_t C, float* dx,
                           int32_t accumulate, void* stream) {
  SEIS_CHECK_ARG(dy && dx && N >= 1 && C >= 1 && H % 2 == 0 && W % 2 == 0 && H >= 2 && W >= 2,
                 "avgpool2 needs even H, W");
  const int64_t n = (int64_t)N * H * W * C;
  k_avgpool2_bwd<<<blocks_for(n), 256, 0, (hipStream_t)stream>>>(dy, N, H, W, C, dx, accumulate);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_up_concat(const uint16_t* low, const uint16_t* skip, int32_t N, int32_t H,
                        int32_t W, int32_t C1, int32_t C2, uint16_t* out, void* stream) {
  SEIS_CHECK_ARG(low && skip && out && N >= 1 && H % 2 == 0 && W % 2 == 0 && C1 >= 1 && C2 >= 1,
                 "bad arguments");
  const int64_t n = (int64_t)N * H * W * (C1 + C2);
  k_up_concat<<<blocks_for(n), 256, 0, (hipStream_t)stream>>>(low, skip, N, H, W, C1, C2, out);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_up_concat_bwd(const float* dout, int32_t N, int32_t H, int32_t W, int32_t C1,
                            int32_t C2, float* dlow, float* dskip, int32_t accumulate_skip,
                            void* stream) {
  SEIS_CHECK_ARG(dout && dlow && dskip && N >= 1 && H % 2 == 0 && W % 2 == 0, "bad arguments");
  hipStream_t s = (hipStream_t)stream;
  const int64_t nl = (int64_t)N * (H / 2) * (W / 2) * C1;
  k_up_concat_bwd_low<<<blocks_for(nl), 256, 0, s>>>(dout, N, H, W, C1, C2, dlow);
  SEIS_CHECK_LAUNCH();
  const int64_t P = (int64_t)N * H * W;
  k_up_concat_bwd_skip<<<blocks_for(P * C2), 256, 0, s>>>(dout, P, C1, C2, dskip,
                                                          accumulate_skip);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_up_gelu_bwd(const float* dout, int32_t N, int32_t H, int32_t W, int32_t C1,
                          int32_t C2, const uint16_t* z, uint16_t* dz, void* stream) {
  SEIS_CHECK_ARG(dout && z && dz && aligned16(dout) && aligned16(z) && aligned16(dz),
                 "pointers must be 16-byte aligned");
  SEIS_CHECK_ARG(N >= 1 && H >= 2 && W >= 2 && H % 2 == 0 && W % 2 == 0 && C1 >= 8 &&
                     C1 % 8 == 0 && C2 >= 0 && C2 % 8 == 0,
                 "even sizes and channel counts of 8 wanted");
  k_up_gelu_bwd<<<blocks_for((int64_t)N * (H / 2) * (W / 2) * (C1 / 8)), 256, 0,
                  (hipStream_t)stream>>>(dout, N, H, W, C1, C2, z, dz);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_skip_gelu_bwd(const float* dout, const float* dpool, int32_t N, int32_t H, int32_t W,
                            int32_t C1, int32_t C2, const uint16_t* z, uint16_t* dz,
                            void* stream) {
  SEIS_CHECK_ARG(dout && dpool && z && dz && aligned16(dout) && aligned16(dpool) && aligned16(z) &&
                     aligned16(dz),
                 "pointers must be 16-byte aligned");
  SEIS_CHECK_ARG(N >= 1 && H >= 2 && W >= 2 && H % 2 == 0 && W % 2 == 0 && C2 >= 8 &&
                     C2 % 8 == 0 && C1 >= 0 && C1 % 8 == 0,
                 "even sizes and channel counts of 8 wanted");
  k_skip_gelu_bwd<<<blocks_for((int64_t)N * H * W * (C2 / 8)), 256, 0, (hipStream_t)stream>>>(
      dout, dpool, N, H, W, C1, C2, z, dz);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_head_gelu_bwd(const uint16_t* x, const float* dout, int64_t P, const float* w,
                            const uint16_t* z, uint16_t* dz, float* dw, float* db, void* stream) {
  SEIS_CHECK_ARG(x && dout && w && z && dz && dw && db && P >= 1, "bad arguments");
  SEIS_CHECK_ARG(aligned16(x) && aligned16(z) && aligned16(dz), "pointers must be 16-byte aligned");
  const int64_t blocks = std::min<int64_t>((P + 63) / 64, 1024);
  k_head_gelu_bwd<4><<<(unsigned)blocks, 256, 0, (hipStream_t)stream>>>(x, dout, P, w, z, dz, dw,
                                                                        db);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_pack_input(const float* grad, const float* model, int32_t N, int32_t H, int32_t W,
                         const float* scales, uint16_t* out, void* stream) {
  SEIS_CHECK_ARG(grad && model && scales && out && aligned16(out), "bad arguments");
  const int64_t P = (int64_t)N * H * W;
  k_pack_input<<<blocks_for(P), 256, 0, (hipStream_t)stream>>>(grad, model, P, scales,
                                                              (int64_t)H * W, out);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_head(const uint16_t* x, int64_t P, int32_t C, const float* w, const float* b,
                   float* out, void* stream) {
  SEIS_CHECK_ARG(x && w && b && out && C >= 1, "bad arguments");
  if (C == 32 && aligned16(x))
    k_head_fwd_v<4><<<blocks_for(P), 256, 0, (hipStream_t)stream>>>(x, P, w, b, out);
  else
    k_head_fwd<<<blocks_for(P), 256, 0, (hipStream_t)stream>>>(x, P, C, w, b, out);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_head_bwd(const uint16_t* x, const float* dout, int64_t P, int32_t C, const float* w,
                       float* dx, float* dw, float* db, void* stream) {
  SEIS_CHECK_ARG(x && dout && w && dx && dw && db && C >= 1 && C <= 255, "bad arguments");
  k_head_bwd<<<blocks_for(P), 256, 0, (hipStream_t)stream>>>(x, dout, P, C, w, dx, dw, db);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_mse(const float* pred, const float* target, const float* mask, int64_t n,
                  float inv_count, float* loss, float* dpred, void* stream) {
  SEIS_CHECK_ARG(pred && target && loss && dpred && n >= 1, "bad arguments");
  hipStream_t s = (hipStream_t)stream;
  k_fill_f32<<<1, 256, 0, s>>>(loss, 1, 0.0f);
  k_mse<<<blocks_for(n), 256, 0, s>>>(pred, target, mask, n, inv_count, loss, dpred);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_adamw(float* param, const float* grad, float* m, float* v, int64_t n, float lr,
                    float beta1, float beta2, float eps, float weight_decay, int32_t step,
                    uint16_t* param_bf16, void* stream) {
  SEIS_CHECK_ARG(param && grad && m && v && n >= 1 && step >= 1, "bad arguments");
  const float bc1 = 1.0f - powf(beta1, (float)step);
  const float bc2 = 1.0f - powf(beta2, (float)step);
  k_adamw<<<blocks_for(n), 256, 0, (hipStream_t)stream>>>(param, grad, m, v, n, lr, beta1, beta2,
                                                          eps, weight_decay, bc1, bc2, param_bf16);
  SEIS_CHECK_LAUNCH();
  return 0;
}

int seis_unet_fill(float* p, int64_t n, float v, void* stream) {
  SEIS_CHECK_ARG(p && n >= 0, "bad arguments");
  if (n == 0) return 0;
  k_fill_f32<<<blocks_for(n), 256, 0, (hipStream_t)stream>>>(p, n, v);
  SEIS_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
