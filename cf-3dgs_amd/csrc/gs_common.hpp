// gs_common.hpp -- device-side building blocks shared by the rasteriser kernels.
//
// Rounding contract: every kernel is compiled with -ffp-contract=off, keeps
// HIP's correctly rounded fp32 division and square root, and spells out each
// fused multiply-add it wants.  Together with the exponential below this
// makes radii, tile rects, keys, ranges, contributor counts and the forward
// image bit-identical to the fp32 CPU restatement kept in oracle/.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/gs_raster.h"

namespace gs {

constexpr int kBX = 16;
constexpr int kBY = 16;
constexpr int kBlock = kBX * kBY;  // one 16x16 tile per 256-thread workgroup
constexpr int kWave = 64;

// ---------------------------------------------------------------------------
// Exponential of the blend: Cody & Waite reduction (Cody, Waite, "Software
// Manual for the Elementary Functions", 1980) + degree-7 Taylor polynomial,
// all steps explicit fma / rint / ldexp, which gfx950 and the host round
// identically.  Domain used by the rasteriser: x <= 0.
__device__ __forceinline__ float spec_expf(float x) {
  x = fmaxf(x, -80.0f);
  const float k = rintf(x * 1.44269502f);
  float r = fmaf(k, -0.693115234375f, x);
  r = fmaf(k, -3.19461833e-05f, r);
  float p = 1.98412701e-04f;
  p = fmaf(p, r, 1.38888892e-03f);
  p = fmaf(p, r, 8.33333377e-03f);
  p = fmaf(p, r, 4.16666679e-02f);
  p = fmaf(p, r, 1.66666672e-01f);
  p = fmaf(p, r, 0.5f);
  p = fmaf(p, r, 1.0f);
  p = fmaf(p, r, 1.0f);
  return ldexpf(p, (int)k);
}

// -0.5 (a dx^2 + c dy^2) - b dx dy with the oracle's fma placement.
__device__ __forceinline__ float blend_power(float a, float b, float c, float dx, float dy) {
  const float q = fmaf(a * dx, dx, (c * dy) * dy);
  return fmaf(-0.5f, q, -((b * dx) * dy));
}

// Saturating float -> int (NaN -> 0).
__device__ __forceinline__ int sat_i(float f) {
  if (f != f) return 0;
  if (f >= 2147483647.0f) return 2147483647;
  if (f <= -2147483648.0f) return (-2147483647 - 1);
  return (int)f;
}

// ((v + 1) * S - 1) * 0.5 evaluated in double, rounded once to float.
__device__ __forceinline__ float ndc2pix(float v, int S) {
  return (float)((((double)v + 1.0) * (double)S - 1.0) * 0.5);
}

struct f3 {
  float x, y, z;
};

__device__ __forceinline__ f3 xf43(const float* m, f3 p) {
  return {m[0] * p.x + m[4] * p.y + m[8] * p.z + m[12], m[1] * p.x + m[5] * p.y + m[9] * p.z + m[13],
          m[2] * p.x + m[6] * p.y + m[10] * p.z + m[14]};
}
__device__ __forceinline__ float xf44w(const float* m, f3 p) {
  return m[3] * p.x + m[7] * p.y + m[11] * p.z + m[15];
}

// Row-major rotation of quaternion (r, x, y, z); utils/general_utils.py:88-96.
__device__ __forceinline__ void quat_to_R(float r, float x, float y, float z, float R[9]) {
  R[0] = 1.0f - 2.0f * (y * y + z * z);
  R[1] = 2.0f * (x * y - r * z);
  R[2] = 2.0f * (x * z + r * y);
  R[3] = 2.0f * (x * y + r * z);
  R[4] = 1.0f - 2.0f * (x * x + z * z);
  R[5] = 2.0f * (y * z - r * x);
  R[6] = 2.0f * (x * z - r * y);
  R[7] = 2.0f * (y * z + r * x);
  R[8] = 1.0f - 2.0f * (x * x + y * y);
}

// d(loss)/d(r,x,y,z) given d(loss)/dR (row-major) for the polynomial above.
__device__ __forceinline__ void quat_R_grad(float r, float x, float y, float z, const float G[9], float dq[4]) {
  dq[0] = 2.0f * (-z * G[1] + y * G[2] + z * G[3] - x * G[5] - y * G[6] + x * G[7]);
  dq[1] = 2.0f * (y * G[1] + z * G[2] + y * G[3] - 2.0f * x * G[4] - r * G[5] + z * G[6] + r * G[7] -
                  2.0f * x * G[8]);
  dq[2] = 2.0f * (-2.0f * y * G[0] + x * G[1] + r * G[2] + x * G[3] + z * G[5] - r * G[6] + z * G[7] -
                  2.0f * y * G[8]);
  dq[3] = 2.0f * (-2.0f * z * G[0] - r * G[1] + x * G[2] + r * G[3] - 2.0f * z * G[4] + y * G[5] +
                  x * G[6] + y * G[7]);
}

// Pose [tx, ty, tz, qx, qy, qz, qw] -> normalised quaternion + rotation.
struct Pose {
  float R[9];
  float t[3];
  float q[4];  // (w, x, y, z), normalised
  float inv_norm;
};
__device__ __forceinline__ void make_pose(const float* p7, Pose& P) {
  const float qx = p7[3], qy = p7[4], qz = p7[5], qw = p7[6];
  const float n2 = ((qx * qx + qy * qy) + qz * qz) + qw * qw;
  P.inv_norm = 1.0f / sqrtf(n2);
  P.q[0] = qw * P.inv_norm;
  P.q[1] = qx * P.inv_norm;
  P.q[2] = qy * P.inv_norm;
  P.q[3] = qz * P.inv_norm;
  quat_to_R(P.q[0], P.q[1], P.q[2], P.q[3], P.R);
  P.t[0] = p7[0];
  P.t[1] = p7[1];
  P.t[2] = p7[2];
}
__device__ __forceinline__ f3 pose_apply(const Pose& P, f3 p) {
  return {((P.R[0] * p.x + P.R[1] * p.y) + P.R[2] * p.z) + P.t[0],
          ((P.R[3] * p.x + P.R[4] * p.y) + P.R[5] * p.z) + P.t[1],
          ((P.R[6] * p.x + P.R[7] * p.y) + P.R[8] * p.z) + P.t[2]};
}

// Real SH basis, constants of utils/sh_utils.py:26-45, polynomial of :74-100.
#define GS_SH_C0 0.28209479177387814f
#define GS_SH_C1 0.4886025119029199f
#define GS_SH_C2_0 1.0925484305920792f
#define GS_SH_C2_1 -1.0925484305920792f
#define GS_SH_C2_2 0.31539156525252005f
#define GS_SH_C2_3 -1.0925484305920792f
#define GS_SH_C2_4 0.5462742152960396f
#define GS_SH_C3_0 -0.5900435899266435f
#define GS_SH_C3_1 2.890611442640554f
#define GS_SH_C3_2 -0.4570457994644658f
#define GS_SH_C3_3 0.3731763325901154f
#define GS_SH_C3_4 -0.4570457994644658f
#define GS_SH_C3_5 1.445305721320277f
#define GS_SH_C3_6 -0.5900435899266435f

__device__ __forceinline__ void sh_basis(int deg, float x, float y, float z, float b[16]) {
  b[0] = GS_SH_C0;
  if (deg < 1) return;
  b[1] = -GS_SH_C1 * y;
  b[2] = GS_SH_C1 * z;
  b[3] = -GS_SH_C1 * x;
  if (deg < 2) return;
  const float xx = x * x, yy = y * y, zz = z * z, xy = x * y, yz = y * z, xz = x * z;
  b[4] = GS_SH_C2_0 * xy;
  b[5] = GS_SH_C2_1 * yz;
  b[6] = GS_SH_C2_2 * ((2.0f * zz - xx) - yy);
  b[7] = GS_SH_C2_3 * xz;
  b[8] = GS_SH_C2_4 * (xx - yy);
  if (deg < 3) return;
  b[9] = (GS_SH_C3_0 * y) * (3.0f * xx - yy);
  b[10] = (GS_SH_C3_1 * xy) * z;
  b[11] = (GS_SH_C3_2 * y) * ((4.0f * zz - xx) - yy);
  b[12] = (GS_SH_C3_3 * z) * ((2.0f * zz - 3.0f * xx) - 3.0f * yy);
  b[13] = (GS_SH_C3_4 * x) * ((4.0f * zz - xx) - yy);
  b[14] = (GS_SH_C3_5 * z) * (xx - yy);
  b[15] = (GS_SH_C3_6 * x) * (xx - 3.0f * yy);
}

// d(basis_k)/d(x,y,z).
__device__ __forceinline__ void sh_basis_grad(int deg, float x, float y, float z, float g[16][3]) {
#pragma unroll
  for (int k = 0; k < 16; ++k) g[k][0] = g[k][1] = g[k][2] = 0.0f;
  if (deg < 1) return;
  g[1][1] = -GS_SH_C1;
  g[2][2] = GS_SH_C1;
  g[3][0] = -GS_SH_C1;
  if (deg < 2) return;
  const float xx = x * x, yy = y * y, zz = z * z, xy = x * y, yz = y * z, xz = x * z;
  g[4][0] = GS_SH_C2_0 * y;
  g[4][1] = GS_SH_C2_0 * x;
  g[5][1] = GS_SH_C2_1 * z;
  g[5][2] = GS_SH_C2_1 * y;
  g[6][0] = -2.0f * GS_SH_C2_2 * x;
  g[6][1] = -2.0f * GS_SH_C2_2 * y;
  g[6][2] = 4.0f * GS_SH_C2_2 * z;
  g[7][0] = GS_SH_C2_3 * z;
  g[7][2] = GS_SH_C2_3 * x;
  g[8][0] = 2.0f * GS_SH_C2_4 * x;
  g[8][1] = -2.0f * GS_SH_C2_4 * y;
  if (deg < 3) return;
  g[9][0] = GS_SH_C3_0 * 6.0f * xy;
  g[9][1] = GS_SH_C3_0 * (3.0f * xx - 3.0f * yy);
  g[10][0] = GS_SH_C3_1 * yz;
  g[10][1] = GS_SH_C3_1 * xz;
  g[10][2] = GS_SH_C3_1 * xy;
  g[11][0] = GS_SH_C3_2 * (-2.0f * xy);
  g[11][1] = GS_SH_C3_2 * (4.0f * zz - xx - 3.0f * yy);
  g[11][2] = GS_SH_C3_2 * (8.0f * yz);
  g[12][0] = GS_SH_C3_3 * (-6.0f * xz);
  g[12][1] = GS_SH_C3_3 * (-6.0f * yz);
  g[12][2] = GS_SH_C3_3 * (6.0f * zz - 3.0f * xx - 3.0f * yy);
  g[13][0] = GS_SH_C3_4 * (4.0f * zz - 3.0f * xx - yy);
  g[13][1] = GS_SH_C3_4 * (-2.0f * xy);
  g[13][2] = GS_SH_C3_4 * (8.0f * xz);
  g[14][0] = GS_SH_C3_5 * (2.0f * xz);
  g[14][1] = GS_SH_C3_5 * (-2.0f * yz);
  g[14][2] = GS_SH_C3_5 * (xx - yy);
  g[15][0] = GS_SH_C3_6 * (3.0f * xx - 3.0f * yy);
  g[15][1] = GS_SH_C3_6 * (-6.0f * xy);
}

// ---------------------------------------------------------------------------
// Wave64 helpers.
// A DPP lane permutation within 16-lane rows (quad_perm, row_mirror,
// row_half_mirror: every lane has a source lane, so no lane keeps an old
// value and none needs to be zero-filled first).
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// Sum over all 64 lanes; every lane must be active.  Result is wave-uniform.
// Maximum of v over the 64 lanes of the wave (all lanes active).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const uint32_t o = (uint32_t)__shfl_xor((int)v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}

// Tile rectangle [x0, x1) x [y0, y1) of a splat at (px, py) with radius r
// (getRect of the reference rasteriser: ((p + r) + 16 - 1) / 16 for the end).
__device__ __forceinline__ void tile_rect(float px, float py, int r, int gx, int gy, int& x0, int& y0, int& x1,
                                          int& y1) {
  const float rr = (float)r;
  x0 = min(gx, max(0, sat_i((px - rr) / (float)kBX)));
  y0 = min(gy, max(0, sat_i((py - rr) / (float)kBY)));
  x1 = min(gx, max(0, sat_i((((px + rr) + (float)kBX) - 1.0f) / (float)kBX)));
  y1 = min(gy, max(0, sat_i((((py + rr) + (float)kBY) - 1.0f) / (float)kBY)));
}

// Rows of `per4` 16-byte vectors, contiguous in global memory, into LDS rows
// of `prow` floats.  A thread that then works on its own row reads
// LDS at a stride of prow words across the wave: an odd prow puts the 64
// lanes on 64 different banks (a stride of 48 puts them on 4).  The row /
// column of vector k = threadIdx.x + 256 r advance by constant steps, so no
// division per vector.  Every thread issues all of its (up to 12) loads before
// its first store, so a workgroup has its whole block in flight at once instead
// of one load-to-store round trip per vector (the SH rows of 256 Gaussians at M
// = 16 are exactly 12 vectors per thread); loads and stores are unconditional,
// clamped to the last vector, so the staging array stays in registers.  256
// threads; dst and src must not overlap.
__device__ __forceinline__ void rows_to_lds(float* __restrict__ dst, const float4* __restrict__ src, int nrows,
                                            int per4, int prow) {
  constexpr int kMax = 12;
  const int n16 = nrows * per4;
  if (n16 <= 0) return;
  float4 v[kMax];
#pragma unroll
  for (int r = 0; r < kMax; ++r) v[r] = src[min((int)threadIdx.x + r * 256, n16 - 1)];
  const int q = 256 / per4, rem = 256 - q * per4;
  const int lg = (n16 - 1) / per4, lj = (n16 - 1) - lg * per4;  // the last vector
  int k = (int)threadIdx.x, g = k / per4, j = k - g * per4;
#pragma unroll
  for (int r = 0; r < kMax; ++r) {
    const bool in = k < n16;
    float* d = dst + (in ? g : lg) * prow + 4 * (in ? j : lj);
    d[0] = v[r].x;
    d[1] = v[r].y;
    d[2] = v[r].z;
    d[3] = v[r].w;
    k += 256;
    g += q;
    j += rem;
    if (j >= per4) {
      j -= per4;
      ++g;
    }
  }
  for (; k < n16; k += 256) {
    const float4 x = src[k];
    float* d = dst + g * prow + 4 * j;
    d[0] = x.x;
    d[1] = x.y;
    d[2] = x.z;
    d[3] = x.w;
    g += q;
    j += rem;
    if (j >= per4) {
      j -= per4;
      ++g;
    }
  }
}
// Inclusive prefix sum over a workgroup of NT threads (a multiple of 64, at
// most 1024); `total` receives the workgroup sum.  Each wave scans by
// shuffles and one barrier combines the wave totals (a Hillis-Steele scan
// needs two barriers per step).  s_w (NT / 64 words of LDS) may be rewritten
// only after a later barrier.
template <int NT>
__device__ __forceinline__ uint32_t block_scan_incl(uint32_t v, uint32_t* s_w, uint32_t& total) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) s_w[w] = x;
  __syncthreads();
  uint32_t before = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const uint32_t sw = s_w[i];
    before += i < w ? sw : 0u;
    tot += sw;
  }
  total = tot;
  return x + before;
}

// One Adam element update in torch.optim.Adam's order (shared by the Adam
// kernel and the backward's fused update, so both round identically):
//   m = m + (g - m) * (1 - b1);  v = v * b2 + (1 - b2) * g * g;
//   p = p - step * m / (sqrt(v) / sqrt(bc2) + eps),  step = lr / bc1.
// The moments' update and the parameter's decrement step * m / denom, which
// does not depend on the parameter (with contraction off, p - adam_delta(..)
// is adam_one's result bit for bit).
__device__ __forceinline__ float adam_delta(float g, float& m, float& v, float b1, float b2, float eps,
                                            float inv_sqrt_bc2, float step) {
  m = fmaf(g - m, 1.0f - b1, m);
  v = fmaf(v, b2, (1.0f - b2) * g * g);
  const float denom = sqrtf(v) * inv_sqrt_bc2 + eps;
  return step * (m / denom);
}

__device__ __forceinline__ void adam_one(float& p, float g, float& m, float& v, float b1, float b2, float eps,
                                         float inv_sqrt_bc2, float step) {
  p = p - adam_delta(g, m, v, b1, b2, eps, inv_sqrt_bc2, step);
}

// 16-byte loads and stores that bypass cache retention (each byte of an
// optimiser pass is touched once).
typedef float nt4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 ld_nt(const float* p) {
  const nt4 v = __builtin_nontemporal_load(reinterpret_cast<const nt4*>(p));
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void st_nt(float* p, const float4& v) {
  const nt4 w = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(w, reinterpret_cast<nt4*>(p));
}

__device__ __forceinline__ uint64_t lanemask_lt() {
  const uint32_t lane = __lane_id();
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// Pixel (dx, dy) of thread t inside a 16 x 16 tile: wave w = t / 64 takes the
// 8 x 8 quadrant (w & 1, w >> 1), lane l the pixel (l & 7, l >> 3) in it.  A
// small splat covers more lanes of an 8 x 8 block than of a 16 x 4 strip.
__device__ __forceinline__ void tile_pixel(int t, int& dx, int& dy) {
  const int w = t >> 6, l = t & 63;
  dx = ((w & 1) << 3) + (l & 7);
  dy = ((w >> 1) << 3) + (l >> 3);
}

// The thread tile_pixel maps to pixel (dx, dy).
__device__ __forceinline__ int tile_thread(int dx, int dy) {
  return ((((dy >> 3) << 1) + (dx >> 3)) << 6) + ((dy & 7) << 3) + (dx & 7);
}

// Where a splat at (x, y) with conic (a, b, c) and opacity o can have alpha >=
// 1/255: the ellipse Q = a u^2 + 2 b u v + c v^2 <= L around its centre, (u, v)
// the pixel's offset and L = 2 ln(255 o).  On a band of rows the ellipse spans
// u in [(-b v - s(v)) / a, (-b v + s(v)) / a], s(v) = sqrt(a L - det v^2), at
// its widest where v is nearest the ellipse's own extreme, so two evaluations
// give the columns it reaches on the band.  A pixel outside is one that every
// kernel skips.
// L is padded for every rounding here and in the kernels' per-pixel power:
// 0.01 in the exponent, 1e-3 relative and absolute, and 1e-6 a c / det
// relative -- the terms a u^2 and c v^2 reach L a c / det on the ellipse and
// cancel against the cross term, so that is the scale the power rounds on.
// det is formed with its product's rounding error added back, since for a
// long thin splat a c and b^2 agree in their leading digits; past a c / det =
// 1e5 (300 times longer than wide) the power itself has no digits to spare and
// the splat counts as reaching everything.  So does one with o < 0 or NaN, a
// conic that is not positive definite or an infinite reach.  The logarithm,
// square roots and reciprocals are the 1-ulp instructions; the spans get 2e-3
// pixel and 1e-5 of the ellipse's half-width on top.
struct SplatReach {
  bool none, all;
  float bia, ia, mdet, aL, vs, V, pad;
  __device__ __forceinline__ SplatReach(float a, float b, float c, float o) {
    const float L0 = 2.0f * (0.693147182f * __builtin_amdgcn_logf(255.0f * o) + 0.01f);
    const float bb = b * b;
    const float det = fmaf(a, c, -bb) - fmaf(b, b, -bb);
    const float idet = __builtin_amdgcn_rcpf(det);
    const float L = fmaf(L0, fmaf(1e-6f * a * c, idet, 1.001f), 1e-3f);
    none = L0 <= 0.0f;
    ia = __builtin_amdgcn_rcpf(a);
    aL = a * L;
    const float cL = c * L;
    all = !(L0 > 0.0f) || !(a > 0.0f) || !(c > 0.0f) || !(a * c < 1e5f * det) || !(aL * idet < 1e30f) ||
          !(cL * idet < 1e30f);
    mdet = -det;
    bia = b * ia;
    V = __builtin_amdgcn_sqrtf(aL * idet) * 1.0001f + 2e-3f;  // half-height
    const float U = __builtin_amdgcn_sqrtf(cL * idet);        // half-width
    vs = -(b * U) * __builtin_amdgcn_rcpf(c);                 // v of the right-hand extreme
    pad = fmaf(U, 1e-5f, 2e-3f);
  }
  // columns [left, right] relative to the centre on the rows [lo, hi]; false: none
  __device__ __forceinline__ bool band(float lo, float hi, float& left, float& right) const {
    lo = fmaxf(lo, -V);
    hi = fminf(hi, V);
    const float vr = fminf(hi, fmaxf(lo, vs)), vl = fminf(hi, fmaxf(lo, -vs));
    right = fmaf(-bia, vr, __builtin_amdgcn_sqrtf(fmaxf(fmaf(mdet * vr, vr, aL), 0.0f)) * ia) + pad;
    left = fmaf(-bia, vl, -(__builtin_amdgcn_sqrtf(fmaxf(fmaf(mdet * vl, vl, aL), 0.0f)) * ia)) - pad;
    return lo <= hi;
  }
};

// Whether the splat can reach the w x h pixels whose first is (x0, y0).
__device__ __forceinline__ bool splat_reaches(float x, float y, float a, float b, float c, float o, float x0, float y0,
                                              float w, float h) {
  const SplatReach r(a, b, c, o);
  const float u = x0 - x, v = y0 - y;
  float left, right;
  const bool hit = r.band(v, v + (h - 1.0f), left, right) && left <= u + (w - 1.0f) && right >= u;
  return !r.none && (r.all || hit);
}

// The 4 x 4-pixel cells of the tile at (x0, y0) that the splat can reach: bit
// 4 cy + cx for the cell whose first pixel is (x0 + 4 cx, y0 + 4 cy).  One
// band per cell row (16 separate cell tests cost several times more).
__device__ __forceinline__ uint32_t splat_cells(float x, float y, float a, float b, float c, float o, float x0,
                                                float y0) {
  const SplatReach e(a, b, c, o);
  const float bx = x - x0, v0 = y0 - y;
  uint32_t m = 0u;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float left, right;
    const bool hit = e.band(v0 + (float)(4 * r), v0 + (float)(4 * r + 3), left, right);
    // first cell with 4 cx + 3 >= left, one past the last with 4 cx <= right
    const int c0 = (int)ceilf(fminf(fmaxf((left + bx - 3.0f) * 0.25f, 0.0f), 4.0f));
    const int c1 = (int)floorf(fminf(fmaxf((right + bx) * 0.25f, -1.0f), 3.0f)) + 1;
    const uint32_t row = (0xfu << c0) & ((1u << c1) - 1u) & 0xfu;
    m |= hit ? row << (4 * r) : 0u;
  }
  return e.none ? 0u : (e.all ? 0xffffu : m);
}

// The 8 x 8-pixel quadrants of the tile at (x0, y0) that the splat can reach:
// bit 2 qy + qx.  One band per row of quadrants.
__device__ __forceinline__ uint32_t splat_quads(float x, float y, float a, float b, float c, float o, float x0,
                                                float y0) {
  const SplatReach e(a, b, c, o);
  const float u = x0 - x, v = y0 - y;
  uint32_t m = 0u;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    float left, right;
    const bool hit = e.band(v + (float)(8 * r), v + (float)(8 * r + 7), left, right);
    const uint32_t row = (left <= u + 7.0f && right >= u ? 1u : 0u) | (left <= u + 15.0f && right >= u + 8.0f ? 2u : 0u);
    m |= hit ? row << (2 * r) : 0u;
  }
  return e.none ? 0u : (e.all ? 0xfu : m);
}

// A wave's own list of the staged splats that meet its pixels: positions j
// < limit (ascending) with bit `wv` set in s_mask[j]; returns the count
// (wave-uniform).  Needs all 64 lanes active.  NC * 64 staged entries.
template <int NC>
__device__ __forceinline__ int compact_wave_list(const uint32_t* s_mask, uint8_t* s_list, int wv, int lane, int limit) {
  int n = 0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int idx = c * 64 + lane;
    const bool hit = idx < limit && ((s_mask[idx] >> wv) & 1u);
    const uint64_t bal = __ballot(hit);
    if (hit) s_list[n + __popcll(bal & lanemask_lt())] = (uint8_t)idx;
    n += __popcll(bal);
  }
  return n;
}

// Frame f of a set whose per-frame block counts have the exclusive prefix
// `prefix`: the last f with prefix[f] <= b (frames owning no block share their
// start with the next).
__device__ __forceinline__ int frame_of_block(const uint32_t* prefix, int n, uint32_t b) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (prefix[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Block id -> logical id so that each of the 8 XCDs (dispatch is round-robin
// over XCDs) receives a contiguous run of logical work items: neighbouring
// tiles share Gaussians, so this keeps their gathers in one L2.
__device__ __forceinline__ uint32_t xcd_remap(uint32_t b, uint32_t nb) {
  const uint32_t full = nb & ~7u;
  if (b >= full) return b;
  const uint32_t per = full >> 3;
  return (b & 7u) * per + (b >> 3);
}

}  // namespace gs
