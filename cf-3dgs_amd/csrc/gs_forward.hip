// gs_forward.hip -- forward rasteriser for gfx950.
//
// Pipeline (one frame):
//   k_preprocess   per Gaussian: optional rigid pose, near cull, 3-D and EWA
//                  2-D covariance, conic, radius, tile rect, SH -> RGB; writes a
//                  48-byte splat record and a workgroup-local prefix sum of the
//                  tiles touched (SH coefficients staged through LDS so the
//                  [P,M,3] array is read with coalesced 16-byte loads)
//   k_scan_top     one workgroup: exclusive prefix of the per-workgroup sums,
//                  total -> counters[0], status -> counters[1]
//   k_duplicate    per Gaussian: (tile << 32 | depth bits, id) pairs
//   radix sort     gs_sort.hip, 8-bit LSD passes over bits [0, 32 + bits(T))
//   k_ranges       [start, end) per tile in the sorted list
//   (the depth-first schedule instead sorts the Gaussians by depth, expands
//   them into tile ids in that order (k_df_*), sorts on the tile bits alone,
//   and records the tile ranges in that sort's last pass)
//   k_blend        single-wave workgroups, each one block of a 16x16 tile's
//                  pixels: 8 x 8, or 4 x 4 with four list entries at a time
//                  per pixel where the launch is small; the wave streams the
//                  tile's list, keeps the splats whose alpha can reach 1/255
//                  on its block and stops when its pixels are saturated; a
//                  tile's waves share an XCD.
#include "gs_common.hpp"
#include "gs_internal.hpp"

#include <type_traits>
#include <vector>

namespace gs {

struct PreArgs {
  int P, M, D, W, H, gx, gy, prefiltered;
  float tanfovx, tanfovy, fx, fy, scale_mod;
  const float* view;
  const float* proj;
  const float* campos;
  const float* pose;
  const float* means;
  const float* shs;
  const float* colors;
  const float* opac;
  const float* scales;
  const float* rots;
  const float* cov_pre;
  int* radii;
  float4* splat;
  float* cov3D;
  uint32_t* tiles;
  uint32_t* local_incl;  // workgroup-local inclusive prefix of tiles
  uint32_t* block_sum;   // [nblocks] sums, then [nblocks] status flags
};

// Inclusive prefix sum over the 256 threads of a workgroup (uint32).
__device__ __forceinline__ uint32_t block_incl_scan_256(uint32_t v, uint32_t* s_tmp /*[>= 4]*/, uint32_t& total) {
  return block_scan_incl<256>(v, s_tmp, total);
}

// Workgroup bid of the nblocks of one frame's preprocess.  s_sh: [256][prow]
// staged SH coefficients (3 nc used per row).
__device__ __forceinline__ void preprocess_block(const PreArgs& a, int bid, int nblocks, float* s_sh) {
  __shared__ uint32_t s_scan[256];
  __shared__ uint32_t s_flag;
  const int base = bid * 256;
  const int i = base + threadIdx.x;
  const int nc = (a.D + 1) * (a.D + 1);
  const int stride = 3 * nc;
  const int prow = stride | 1;  // odd LDS row stride: no bank conflicts on the per-thread row reads
  if (threadIdx.x == 0) s_flag = 0;
  if (a.shs) {
    const int nloc = min(256, a.P - base);
    if (nc == a.M && (a.M & 3) == 0) {
      // contiguous rows of 3M floats, a multiple of 16 bytes when M % 4 == 0
      rows_to_lds(s_sh, reinterpret_cast<const float4*>(a.shs + (size_t)base * 3 * a.M), nloc, stride >> 2, prow);
    } else {
      for (int k = threadIdx.x; k < nloc * stride; k += 256) {
        const int g = k / stride, e = k - g * stride;
        s_sh[g * prow + e] = a.shs[(size_t)(base + g) * 3 * a.M + e];
      }
    }
  }
  __syncthreads();

  uint32_t my_tiles = 0;
  if (i < a.P) {
    a.radii[i] = 0;
    f3 p = {a.means[3 * i], a.means[3 * i + 1], a.means[3 * i + 2]};
    if (a.pose) {
      Pose ps;
      make_pose(a.pose, ps);
      p = pose_apply(ps, p);
    }
    const f3 pv = xf43(a.view, p);
    bool ok = true;
    if (pv.z <= 0.2f) {
      if (a.prefiltered) s_flag = GS_STATUS_PREFILTERED;
      ok = false;
    }
    float c3[6];
    float px = 0.f, py = 0.f, con_a = 0.f, con_b = 0.f, con_c = 0.f;
    int ir = 0;
    int x0 = 0, y0 = 0, x1 = 0, y1 = 0;
    if (ok) {
      const f3 ph = xf43(a.proj, p);
      const float pw = 1.0f / (xf44w(a.proj, p) + 0.0000001f);
      const float ndc_x = ph.x * pw, ndc_y = ph.y * pw;
      if (a.cov_pre) {
#pragma unroll
        for (int k = 0; k < 6; ++k) c3[k] = a.cov_pre[6 * i + k];
      } else {
        float R[9];
        const float4 q = reinterpret_cast<const float4*>(a.rots)[i];
        quat_to_R(q.x, q.y, q.z, q.w, R);
        const float s0 = a.scale_mod * a.scales[3 * i], s1 = a.scale_mod * a.scales[3 * i + 1],
                    s2 = a.scale_mod * a.scales[3 * i + 2];
        float L[9];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
          L[3 * r] = R[3 * r] * s0;
          L[3 * r + 1] = R[3 * r + 1] * s1;
          L[3 * r + 2] = R[3 * r + 2] * s2;
        }
#define GS_SIG(u, v) ((L[3 * (u)] * L[3 * (v)] + L[3 * (u) + 1] * L[3 * (v) + 1]) + L[3 * (u) + 2] * L[3 * (v) + 2])
        c3[0] = GS_SIG(0, 0);
        c3[1] = GS_SIG(0, 1);
        c3[2] = GS_SIG(0, 2);
        c3[3] = GS_SIG(1, 1);
        c3[4] = GS_SIG(1, 2);
        c3[5] = GS_SIG(2, 2);
#undef GS_SIG
      }
#pragma unroll
      for (int k = 0; k < 6; ++k) a.cov3D[6 * i + k] = c3[k];
      const float limx = 1.3f * a.tanfovx, limy = 1.3f * a.tanfovy;
      const float txtz = pv.x / pv.z, tytz = pv.y / pv.z;
      const float tx = fminf(limx, fmaxf(-limx, txtz)) * pv.z;
      const float ty = fminf(limy, fmaxf(-limy, tytz)) * pv.z;
      const float tz = pv.z;
      const float J00 = a.fx / tz, J02 = -(a.fx * tx) / (tz * tz);
      const float J11 = a.fy / tz, J12 = -(a.fy * ty) / (tz * tz);
      float Tm0[3], Tm1[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        Tm0[c] = J00 * a.view[c * 4 + 0] + J02 * a.view[c * 4 + 2];
        Tm1[c] = J11 * a.view[c * 4 + 1] + J12 * a.view[c * 4 + 2];
      }
      const float S[3][3] = {{c3[0], c3[1], c3[2]}, {c3[1], c3[3], c3[4]}, {c3[2], c3[4], c3[5]}};
      float MS0[3], MS1[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        MS0[c] = (Tm0[0] * S[0][c] + Tm0[1] * S[1][c]) + Tm0[2] * S[2][c];
        MS1[c] = (Tm1[0] * S[0][c] + Tm1[1] * S[1][c]) + Tm1[2] * S[2][c];
      }
      const float ca = ((MS0[0] * Tm0[0] + MS0[1] * Tm0[1]) + MS0[2] * Tm0[2]) + 0.3f;
      const float cb = (MS0[0] * Tm1[0] + MS0[1] * Tm1[1]) + MS0[2] * Tm1[2];
      const float cc = ((MS1[0] * Tm1[0] + MS1[1] * Tm1[1]) + MS1[2] * Tm1[2]) + 0.3f;
      const float det = ca * cc - cb * cb;
      if (det == 0.0f) ok = false;
      if (ok) {
        const float det_inv = 1.0f / det;
        con_a = cc * det_inv;
        con_b = -cb * det_inv;
        con_c = ca * det_inv;
        const float mid = 0.5f * (ca + cc);
        const float disc = sqrtf(fmaxf(0.1f, mid * mid - det));
        const float l1 = mid + disc, l2 = mid - disc;
        const float radius = ceilf(3.0f * sqrtf(fmaxf(l1, l2)));
        px = ndc2pix(ndc_x, a.W);
        py = ndc2pix(ndc_y, a.H);
        if (!isfinite(px) || !isfinite(py) || !isfinite(radius) || !isfinite(con_a) || !isfinite(con_b) ||
            !isfinite(con_c) || !isfinite(pv.z))
          ok = false;
        if (ok) {
          ir = sat_i(radius);
          tile_rect(px, py, ir, a.gx, a.gy, x0, y0, x1, y1);
          my_tiles = (uint32_t)(x1 - x0) * (uint32_t)(y1 - y0);
          if (my_tiles == 0) ok = false;
        }
      }
    }
    if (ok) {
      float rgb[3];
      uint32_t cbits = 0;
      if (a.shs) {
        const f3 dv = {p.x - a.campos[0], p.y - a.campos[1], p.z - a.campos[2]};
        const float len = sqrtf((dv.x * dv.x + dv.y * dv.y) + dv.z * dv.z);
        const float dx = dv.x / len, dy = dv.y / len, dz = dv.z / len;
        float b[16];
        sh_basis(a.D, dx, dy, dz, b);
        const float* sh = s_sh + threadIdx.x * prow;
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
          float acc = b[0] * sh[ch];
          for (int k = 1; k < nc; ++k) acc = acc + b[k] * sh[3 * k + ch];
          acc = acc + 0.5f;
          if (acc < 0.0f) cbits |= 1u << ch;
          rgb[ch] = fmaxf(acc, 0.0f);
        }
      } else {
        rgb[0] = a.colors[3 * i];
        rgb[1] = a.colors[3 * i + 1];
        rgb[2] = a.colors[3 * i + 2];
      }
      a.radii[i] = ir;
      a.splat[3 * i + 0] = make_float4(px, py, con_a, con_b);
      a.splat[3 * i + 1] = make_float4(con_c, a.opac[i], pv.z, __uint_as_float(cbits));
      a.splat[3 * i + 2] = make_float4(rgb[0], rgb[1], rgb[2], __int_as_float(ir));
    } else {
      my_tiles = 0;
    }
    a.tiles[i] = my_tiles;
  }
  uint32_t total;
  const uint32_t incl = block_incl_scan_256(my_tiles, s_scan, total);
  if (i < a.P) a.local_incl[i] = incl;
  if (threadIdx.x == 0) {
    a.block_sum[bid] = total;
    a.block_sum[nblocks + bid] = s_flag;
  }
}

__global__ __launch_bounds__(256) void k_preprocess(PreArgs a) {
  extern __shared__ float s_sh[];
  preprocess_block(a, blockIdx.x, gridDim.x, s_sh);
}

// Many frames' preprocess in one launch: frame f owns workgroups [prefix[f],
// prefix[f + 1]); the dynamic LDS covers the largest frame's SH rows.
__global__ __launch_bounds__(256) void k_preprocess_multi(const uint32_t* prefix, const PreArgs* args, int n) {
  extern __shared__ float s_sh[];
  const uint32_t b = blockIdx.x;
  const int f = frame_of_block(prefix, n, b);
  const PreArgs a = args[f];
  preprocess_block(a, (int)(b - prefix[f]), (int)(prefix[f + 1] - prefix[f]), s_sh);
}

// In-place exclusive prefix of n values by one workgroup of NT threads; returns
// their sum in every thread, `biggest` the largest of the thread's own values.
// Eight values a thread and round, loaded together (data is 16-byte aligned).
// One frame takes 1024 threads, a round for 2 million Gaussians; many frames
// take 256 each: 1024 had to wait for a compute unit with 16 free wave slots
// while another stream's blend ran (49 us a launch of 16 pose frames, now 6).
template <int NT>
__device__ __forceinline__ uint32_t scan_in_place(uint32_t* data, int n, uint32_t& biggest) {
  constexpr int kRun = 8;
  __shared__ uint32_t s_w[2][NT / 64];
  const int t = threadIdx.x;
  uint32_t carry = 0;
  biggest = 0;
  for (int b0 = 0, r = 0; b0 < n; b0 += NT * kRun, r ^= 1) {
    const int first = b0 + t * kRun;
    uint32_t v[kRun], sum = 0;
    if (first + kRun <= n) {
      const uint4 a = *reinterpret_cast<const uint4*>(data + first), b = *reinterpret_cast<const uint4*>(data + first + 4);
      v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
      v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    } else {
#pragma unroll
      for (int j = 0; j < kRun; ++j) v[j] = first + j < n ? data[first + j] : 0u;
    }
#pragma unroll
    for (int j = 0; j < kRun; ++j) {
      sum += v[j];
      biggest = max(biggest, v[j]);
    }
    uint32_t tot;
    uint32_t run = carry + block_scan_incl<NT>(sum, s_w[r], tot) - sum;
#pragma unroll
    for (int j = 0; j < kRun; ++j) {
      if (first + j < n) data[first + j] = run;
      run += v[j];
    }
    carry += tot;
  }
  return carry;
}

// Single workgroup: exclusive prefix of the per-workgroup tile sums (in place),
// num_rendered and the OR of the status flags.
template <int NT>
__device__ __forceinline__ void scan_top_block(uint32_t* block_sum, int nblocks, uint32_t* counters) {
  __shared__ uint32_t s_flags;
  if (threadIdx.x == 0) s_flags = 0;
  uint32_t myflags = 0, biggest;
  for (int b = threadIdx.x; b < nblocks; b += NT) myflags |= block_sum[nblocks + b];
  __syncthreads();
  if (myflags) atomicOr(&s_flags, myflags);
  const uint32_t total = scan_in_place<NT>(block_sum, nblocks, biggest);
  __syncthreads();
  if (threadIdx.x == 0) {
    counters[0] = total;
    counters[1] = s_flags;
  }
}

__global__ __launch_bounds__(1024) void k_scan_top(uint32_t* block_sum, int nblocks, uint32_t* counters) {
  scan_top_block<1024>(block_sum, nblocks, counters);
}

struct ScanTop {
  uint32_t* block_sum;
  uint32_t* counters;
  int nblocks;
};

// Workgroup f: the scan of frame f.
__global__ __launch_bounds__(256) void k_scan_top_multi(const ScanTop* st) {
  const ScanTop t = st[blockIdx.x];
  scan_top_block<256>(t.block_sum, t.nblocks, t.counters);
}

struct DupArgs {
  int P, gx, gy;
  long long capacity;
  const float4* splat;
  const uint32_t* tiles;
  const uint32_t* local_incl;
  const uint32_t* block_excl;
  uint32_t* counters;
  uint64_t* keys;
  uint32_t* vals;
};

__global__ __launch_bounds__(256) void k_duplicate(DupArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const uint32_t n = a.counters[0];
  if ((long long)n > a.capacity) {
    if (i == 0) {
      atomicOr(&a.counters[1], GS_STATUS_CAPACITY);
      atomicOr(&a.counters[3], GS_STATUS_CAPACITY);  // sticky copy
    }
    return;
  }
  if (i >= a.P) return;
  const uint32_t nt = a.tiles[i];
  if (nt == 0) return;
  uint32_t off = a.block_excl[i >> 8] + a.local_incl[i] - nt;
  const float4 s0 = a.splat[3 * i];
  const float4 s1 = a.splat[3 * i + 1];
  const float4 s2 = a.splat[3 * i + 2];
  int x0, y0, x1, y1;
  tile_rect(s0.x, s0.y, __float_as_int(s2.w), a.gx, a.gy, x0, y0, x1, y1);
  const uint64_t dbits = (uint64_t)__float_as_uint(s1.z);
  for (int y = y0; y < y1; ++y)
    for (int x = x0; x < x1; ++x) {
      a.keys[off] = ((uint64_t)(uint32_t)(y * a.gx + x) << 32) | dbits;
      a.vals[off] = (uint32_t)i;
      ++off;
    }
}

__global__ __launch_bounds__(256) void k_fill_u32(uint32_t* p, long long n, uint32_t v) {
  for (long long k = (long long)blockIdx.x * 256 + threadIdx.x; k < n; k += (long long)gridDim.x * 256) p[k] = v;
}

__global__ __launch_bounds__(256) void k_ranges(const uint64_t* keys, const uint32_t* counters, long long capacity,
                                                uint32_t* ranges) {
  const uint32_t n0 = counters[0];
  const uint32_t n = ((long long)n0 > capacity) ? 0u : n0;
  const uint32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  const uint32_t t = (uint32_t)(keys[k] >> 32);
  if (k == 0) {
    ranges[2 * t] = 0;
  } else {
    const uint32_t tp = (uint32_t)(keys[k - 1] >> 32);
    if (t != tp) {
      ranges[2 * tp + 1] = k;
      ranges[2 * t] = k;
    }
  }
  if (k == n - 1) ranges[2 * t + 1] = n;
}

// ---- depth-first binning -------------------------------------------------
// Keys for the depth sort: depth bits of visible Gaussians (positive floats
// order as their bit patterns), 0xffffffff for the rest (sorted last, and they
// touch no tile).  counters[2] = P is the sort's element count.  The tile
// rect of each visible Gaussian is packed into 8 bytes here, while the splat
// records are read in order, so the duplicate (which visits Gaussians in
// depth order, i.e. at random) reads one 8-byte record instead of the tile
// count and two 16-byte splat vectors.
// Also sets the n_ranges words of the tile ranges to [UINT_MAX, 0) per tile,
// the start the list sort's atomic min / max needs (the grid covers
// max(P, n_ranges) threads).
__device__ __forceinline__ void df_keys_block(int P, const uint32_t* tiles, const float4* splat, int gx, int gy,
                                              uint32_t* keys, uint32_t* vals, uint2* rect, uint32_t* counters,
                                              uint32_t* ranges, int n_ranges, int bid) {
  const int i = bid * 256 + threadIdx.x;
  if (i == 0) counters[2] = (uint32_t)P;
  if (i < n_ranges) ranges[i] = (i & 1) ? 0u : 0xffffffffu;
  if (i >= P) return;
  const bool vis = tiles[i] != 0u;
  keys[i] = vis ? __float_as_uint(splat[3 * i + 1].z) : 0xffffffffu;
  vals[i] = (uint32_t)i;
  if (vis) {
    const float4 s0 = splat[3 * i];
    const float4 s2 = splat[3 * i + 2];
    int x0, y0, x1, y1;
    tile_rect(s0.x, s0.y, __float_as_int(s2.w), gx, gy, x0, y0, x1, y1);
    rect[i] = make_uint2((uint32_t)x0 | ((uint32_t)y0 << 16), (uint32_t)x1 | ((uint32_t)y1 << 16));
  }
}

__global__ __launch_bounds__(256) void k_df_keys(int P, const uint32_t* tiles, const float4* splat, int gx, int gy,
                                                 uint32_t* keys, uint32_t* vals, uint2* rect, uint32_t* counters,
                                                 uint32_t* ranges, int n_ranges) {
  df_keys_block(P, tiles, splat, gx, gy, keys, vals, rect, counters, ranges, n_ranges, blockIdx.x);
}

struct DfKeysArgs {
  int P, gx, gy, n_ranges;
  const uint32_t* tiles;
  const float4* splat;
  uint32_t* keys;
  uint32_t* vals;
  uint2* rect;
  uint32_t* counters;
  uint32_t* ranges;
};

// Many frames' depth keys in one launch: frame f owns workgroups [prefix[f],
// prefix[f + 1]).
__global__ __launch_bounds__(256) void k_df_keys_multi(const uint32_t* prefix, const DfKeysArgs* args, int n) {
  const uint32_t b = blockIdx.x;
  const int f = frame_of_block(prefix, n, b);
  const DfKeysArgs a = args[f];
  df_keys_block(a.P, a.tiles, a.splat, a.gx, a.gy, a.keys, a.vals, a.rect, a.counters, a.ranges, a.n_ranges,
                (int)(b - prefix[f]));
}

// Workgroup-local inclusive prefix of the tile counts in depth order.
__device__ __forceinline__ void df_scan_block(int P, const uint32_t* dvals, const uint32_t* tiles, uint32_t* dscan,
                                              uint32_t* dblocks, int bid) {
  __shared__ uint32_t s_scan[256];
  const int k = bid * 256 + threadIdx.x;
  const uint32_t v = k < P ? tiles[dvals[k]] : 0u;
  uint32_t total;
  const uint32_t incl = block_incl_scan_256(v, s_scan, total);
  if (k < P) dscan[k] = incl;
  if (threadIdx.x == 0) dblocks[bid] = total;
}

__global__ __launch_bounds__(256) void k_df_scan(int P, const uint32_t* dvals, const uint32_t* tiles, uint32_t* dscan,
                                                 uint32_t* dblocks) {
  df_scan_block(P, dvals, tiles, dscan, dblocks, blockIdx.x);
}

// One workgroup: in-place exclusive prefix of the n block totals, and the
// largest of them in data[n].
template <int NT>
__device__ __forceinline__ void excl_scan_block(uint32_t* data, int n) {
  __shared__ uint32_t s_max;
  if (threadIdx.x == 0) s_max = 0;
  uint32_t biggest;
  scan_in_place<NT>(data, n, biggest);
  __syncthreads();
  if (biggest) atomicMax(&s_max, biggest);
  __syncthreads();
  if (threadIdx.x == 0) data[n] = s_max;
}

__global__ __launch_bounds__(1024) void k_excl_scan_1wg(uint32_t* data, int n) { excl_scan_block<1024>(data, n); }

struct DfDupArgs {
  int P, gx, gy;
  long long capacity;
  const uint2* rect;  // packed tile rect per Gaussian (k_df_keys)
  const uint32_t* tiles;
  const uint32_t* dvals;
  const uint32_t* dscan;
  const uint32_t* dblocks;  // block totals (up to kOwnPrefix blocks), else their prefix and the largest total
  uint32_t* counters;
  uint32_t* keys;  // tile ids, or tile << id_bits | id when id_bits > 0
  uint32_t* vals;  // ids (unused when id_bits > 0)
  int id_bits;
};

// Up to this many blocks of 256 Gaussians every workgroup of the duplicate forms
// the prefix of their totals itself (1024 words from L2, four a thread), which
// is as quick as the wait for a launch that does, and spares that launch.
constexpr uint32_t kOwnPrefix = 1024;

// Tile ids in depth order (sorted position k -> Gaussian dvals[k]).  Each
// Gaussian's entries form one run at its prefix offset, its rect row by row.
//
// Where no block of 256 Gaussians has more than 4096 entries, workgroup b
// expands block b.  Else the work is split by output: a workgroup takes the same
// number of consecutive entries as every other (at least 1024, and no more
// workgroups than the GPU holds at once) and finds the run its first entry lies
// in by a 64-wide search of the prefix.  Either way the runs are expanded 256 at a time,
// four entries a thread and one 16-byte store.  With the split by Gaussian
// alone the few splats that cover a whole image set the launch's length (1284
// us for 71M entries of 1 200 000 Gaussians at 1920 x 1080, now 125; 49 and 7
// for 100 000 at 480 x 270); where the blocks are even the search alone costs
// (31 us with it for 16 pose frames, 22 without).
__device__ __forceinline__ void df_duplicate_block(const DfDupArgs& a, uint32_t bid, uint32_t nblocks) {
  __shared__ uint32_t s_start[256], s_g[256], s_xy[256], s_w[256], s_k0, s_end;
  __shared__ uint32_t s_pref[kOwnPrefix], s_w4[4], s_most[4];
  const uint32_t t = threadIdx.x;
  const uint32_t n = a.counters[0];
  if ((long long)n > a.capacity) {
    if (bid == 0 && t == 0) {
      atomicOr(&a.counters[1], GS_STATUS_CAPACITY);
      atomicOr(&a.counters[3], GS_STATUS_CAPACITY);  // sticky copy
    }
    return;
  }
  const uint32_t P = (uint32_t)a.P, chunk = (n / min(nblocks, 2048u) / 1024u + 1u) * 1024u;
  const uint32_t nruns = (P + 255u) / 256u;
  const bool own = nruns <= kOwnPrefix;
  uint32_t biggest;
  if (own) {
    uint32_t v[4], sum = 0, most = 0;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      v[q] = 4u * t + q < nruns ? a.dblocks[4u * t + q] : 0u;
      sum += v[q];
      most = max(most, v[q]);
    }
    most = wave_max_u32(most);
    if ((t & 63u) == 0) s_most[t >> 6] = most;
    uint32_t total;
    uint32_t run = block_incl_scan_256(sum, s_w4, total) - sum;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      s_pref[4u * t + q] = run;
      run += v[q];
    }
    __syncthreads();
    biggest = max(max(s_most[0], s_most[1]), max(s_most[2], s_most[3]));
  } else {
    biggest = a.dblocks[nruns];
  }
  auto before = [&](uint32_t b) { return own ? s_pref[b] : a.dblocks[b]; };  // entries of the blocks before b
  const bool even = biggest <= 4096u;
  const uint32_t nchunks = even ? nruns : n / chunk + (n % chunk != 0 ? 1u : 0u);
  for (uint32_t c = bid; c < nchunks; c += nblocks) {
    uint32_t o0 = c * chunk, o1 = o0 + min(chunk, n - o0);
    if (even) {
      o0 = before(c);
      o1 = c + 1u < nruns ? before(c + 1u) : n;
      if (t == 0) s_k0 = 256u * c;
    } else if (t < 64) {
      // the last 256-run block that starts at or before o0, then its runs that
      // end there
      uint32_t lo = 0, len = nruns;
      while (len > 1) {
        const uint32_t step = (len + 63u) / 64u, k = t * step;
        const uint32_t m = (uint32_t)__popcll(__ballot(k < len && before(lo + min(k, len - 1u)) <= o0)) - 1u;
        lo += m * step;
        len = min(step, len - m * step);
      }
      const uint32_t b0 = before(lo);
      uint32_t k0 = lo * 256u;
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q) {
        const uint32_t k = lo * 256u + q * 64u + t;
        k0 += (uint32_t)__popcll(__ballot(k < P && b0 + a.dscan[min(k, P - 1u)] <= o0));
      }
      if (t == 0) s_k0 = k0;
    }
    __syncthreads();
    uint32_t pos = o0;
    for (uint32_t k0 = s_k0; pos < o1; k0 += 256) {
      const uint32_t k = k0 + t;
      uint32_t start = n, end = n, g = 0, xy = 0, w = 1;
      if (k < P) {
        g = a.dvals[k];
        end = before(k >> 8) + a.dscan[k];
        start = end - a.tiles[g];
        if (start < end) {
          const uint2 r = a.rect[g];
          xy = r.x;
          w = (r.y & 0xffffu) - (r.x & 0xffffu);
        }
      }
      s_start[t] = start;
      s_g[t] = g;
      s_xy[t] = xy;
      s_w[t] = w;
      if (t == 255) s_end = end;
      __syncthreads();
      const uint32_t lim = min(o1, s_end);
      for (uint32_t q = (pos >> 2) + t; 4u * q < lim; q += 256) {
        const uint32_t first = max(4u * q, pos), stop = min(4u * q + 4u, lim);
        // run j = last with start <= first
        uint32_t j = 0;
#pragma unroll
        for (uint32_t step = 128; step > 0; step >>= 1)
          if (s_start[j + step] <= first) j += step;
        uint32_t rw = s_w[j], id = s_g[j], p = s_xy[j];
        const uint32_t r = first - s_start[j], ry = r / rw;
        uint32_t rx = r - ry * rw, tile = ((p >> 16) + ry) * (uint32_t)a.gx + (p & 0xffffu) + rx;
        uint32_t next = j < 255u ? s_start[j + 1] : lim;
        uint32_t key[4], val[4];
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e) {
          const uint32_t o = 4u * q + e;
          key[e] = a.id_bits ? (tile << a.id_bits) | id : tile;
          val[e] = id;
          if (o < first) continue;
          ++rx;
          ++tile;
          if (rx == rw) {
            rx = 0;
            tile += (uint32_t)a.gx - rw;
          }
          if (o + 1u == next && o + 1u < stop) {
            ++j;
            rw = s_w[j];
            id = s_g[j];
            p = s_xy[j];
            rx = 0;
            tile = (p >> 16) * (uint32_t)a.gx + (p & 0xffffu);
            next = j < 255u ? s_start[j + 1] : lim;
          }
        }
        if (stop - first == 4u) {
          *reinterpret_cast<uint4*>(a.keys + 4u * q) = make_uint4(key[0], key[1], key[2], key[3]);
          if (!a.id_bits) *reinterpret_cast<uint4*>(a.vals + 4u * q) = make_uint4(val[0], val[1], val[2], val[3]);
        } else {
#pragma unroll
          for (uint32_t e = 0; e < 4; ++e) {
            const uint32_t o = 4u * q + e;
            if (o < first || o >= stop) continue;
            a.keys[o] = key[e];
            if (!a.id_bits) a.vals[o] = val[e];
          }
        }
      }
      pos = lim;
      __syncthreads();
    }
  }
}

__global__ __launch_bounds__(256) void k_df_duplicate(DfDupArgs a) { df_duplicate_block(a, blockIdx.x, gridDim.x); }

// The depth-first binning's steps between its two sorts for one frame of a
// multi-frame launch.
struct DfMid {
  DfDupArgs dup;
  uint32_t* dscan;
  uint32_t* dblocks;
  int nblocks;
};

// Many frames' workgroup-local scans of the tile counts in depth order: frame
// f owns workgroups [prefix[f], prefix[f + 1]).
__global__ __launch_bounds__(256) void k_df_scan_multi(const uint32_t* prefix, const DfMid* mid, int n) {
  const uint32_t b = blockIdx.x;
  const int f = frame_of_block(prefix, n, b);
  const DfMid m = mid[f];
  df_scan_block(m.dup.P, m.dup.dvals, m.dup.tiles, m.dscan, m.dblocks, (int)(b - prefix[f]));
}

// Workgroup f: the exclusive prefix of frame f's block totals.
__global__ __launch_bounds__(256) void k_excl_scan_multi(const DfMid* mid) {
  const DfMid m = mid[blockIdx.x];
  if (m.nblocks > (int)kOwnPrefix) excl_scan_block<256>(m.dblocks, m.nblocks);
}

// Many frames' duplicates, on the same workgroup ranges as k_df_scan_multi (a
// frame's workgroups share its chunks out among them).
__global__ __launch_bounds__(256) void k_df_duplicate_multi(const uint32_t* prefix, const DfMid* mid, int n) {
  const uint32_t b = blockIdx.x;
  const int f = frame_of_block(prefix, n, b);
  const DfDupArgs a = mid[f].dup;
  df_duplicate_block(a, b - prefix[f], prefix[f + 1] - prefix[f]);
}

struct BlendArgs {
  int W, H, gx;
  const uint32_t* ranges;
  const uint32_t* list;  // sorted entries; the Gaussian id is entry & id_mask
  uint32_t id_mask;
  const float4* splat;
  const float* bg;
  float* out_color;
  float* out_depth;
  float* out_alpha;
  float* final_T;
  uint32_t* n_contrib;
  // backward support: per-pixel state at every 256-entry batch boundary of
  // the tile's list ([ckpt][T, C0, C1, C2, D][256]), the tile's largest
  // contributor count and the pre-background sums ([C0, C1, C2, D][H*W])
  const uint32_t* ckpt_base;
  float* ckpt;
  uint32_t* tile_maxc;
  uint32_t* tile_done;
  const uint32_t* tile_order;  // the tiles, longest list first (k_tile_ckpt_scan)
  float* accum;
  // per (tile, batch) at ckpt_base[tile] + tile + batch: the entries the tile's
  // waves kept of the batch, the backward's cost estimate for that chunk
  uint32_t* bweight;
  // the backward's work items, appended as tiles finish: [0] count, then
  // (tile, chunk << 6 | cost class)
  // (these, tile_maxc and tile_done, the waves that are through with the
  // tile, are cleared by k_tile_ckpt_scan)
  uint32_t* item_log;
};

// spec_expf of four values, instruction by instruction side by side.  A wave
// issues a dependent instruction every ~10 clocks and an independent one every
// ~6, and a SIMD takes one every 2, so four chains after one another leave a
// launch of few waves waiting; the compiler's scheduler does not mix them.
__device__ __forceinline__ void spec_expf4(const float (&x)[4], float (&p)[4]) {
  float r[4], k[4];
  const float c6 = 1.38888892e-03f;
#define GS_X4(i0, i1, i2, i3) i0 "\n\t" i1 "\n\t" i2 "\n\t" i3 "\n\t"
  asm(GS_X4("v_max_f32 %4, 0xc2a00000, %12", "v_max_f32 %5, 0xc2a00000, %13", "v_max_f32 %6, 0xc2a00000, %14",
            "v_max_f32 %7, 0xc2a00000, %15")
      GS_X4("v_mul_f32 %8, 0x3fb8aa3b, %4", "v_mul_f32 %9, 0x3fb8aa3b, %5", "v_mul_f32 %10, 0x3fb8aa3b, %6",
            "v_mul_f32 %11, 0x3fb8aa3b, %7")
      GS_X4("v_rndne_f32 %8, %8", "v_rndne_f32 %9, %9", "v_rndne_f32 %10, %10", "v_rndne_f32 %11, %11")
      GS_X4("v_fmac_f32 %4, 0xbf317000, %8", "v_fmac_f32 %5, 0xbf317000, %9", "v_fmac_f32 %6, 0xbf317000, %10",
            "v_fmac_f32 %7, 0xbf317000, %11")
      GS_X4("v_fmac_f32 %4, 0xb805fdf4, %8", "v_fmac_f32 %5, 0xb805fdf4, %9", "v_fmac_f32 %6, 0xb805fdf4, %10",
            "v_fmac_f32 %7, 0xb805fdf4, %11")
      GS_X4("v_fmamk_f32 %0, %4, 0x39500d01, %16", "v_fmamk_f32 %1, %5, 0x39500d01, %16",
            "v_fmamk_f32 %2, %6, 0x39500d01, %16", "v_fmamk_f32 %3, %7, 0x39500d01, %16")
      GS_X4("v_fmaak_f32 %0, %0, %4, 0x3c088889", "v_fmaak_f32 %1, %1, %5, 0x3c088889",
            "v_fmaak_f32 %2, %2, %6, 0x3c088889", "v_fmaak_f32 %3, %3, %7, 0x3c088889")
      GS_X4("v_fmaak_f32 %0, %0, %4, 0x3d2aaaab", "v_fmaak_f32 %1, %1, %5, 0x3d2aaaab",
            "v_fmaak_f32 %2, %2, %6, 0x3d2aaaab", "v_fmaak_f32 %3, %3, %7, 0x3d2aaaab")
      GS_X4("v_fmaak_f32 %0, %0, %4, 0x3e2aaaab", "v_fmaak_f32 %1, %1, %5, 0x3e2aaaab",
            "v_fmaak_f32 %2, %2, %6, 0x3e2aaaab", "v_fmaak_f32 %3, %3, %7, 0x3e2aaaab")
      GS_X4("v_fma_f32 %0, %0, %4, 0.5", "v_fma_f32 %1, %1, %5, 0.5", "v_fma_f32 %2, %2, %6, 0.5",
            "v_fma_f32 %3, %3, %7, 0.5")
      GS_X4("v_cvt_i32_f32 %8, %8", "v_cvt_i32_f32 %9, %9", "v_cvt_i32_f32 %10, %10", "v_cvt_i32_f32 %11, %11")
      GS_X4("v_fma_f32 %0, %0, %4, 1.0", "v_fma_f32 %1, %1, %5, 1.0", "v_fma_f32 %2, %2, %6, 1.0",
            "v_fma_f32 %3, %3, %7, 1.0")
      GS_X4("v_fma_f32 %0, %0, %4, 1.0", "v_fma_f32 %1, %1, %5, 1.0", "v_fma_f32 %2, %2, %6, 1.0",
            "v_fma_f32 %3, %3, %7, 1.0")
      GS_X4("v_ldexp_f32 %0, %0, %8", "v_ldexp_f32 %1, %1, %9", "v_ldexp_f32 %2, %2, %10", "v_ldexp_f32 %3, %3, %11")
      : "=&v"(p[0]), "=&v"(p[1]), "=&v"(p[2]), "=&v"(p[3]), "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]),
        "=&v"(k[0]), "=&v"(k[1]), "=&v"(k[2]), "=&v"(k[3])
      : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(c6));
#undef GS_X4
}

// One block of 64 / E pixels of a tile by one wave: 8 x 8 pixels (E = 1) or 4 x
// 4 (4); block `part` of the tile's 4 E.
//
// Lane E p + e looks at entries e, E + e, .. of 4 E at pixel p of the block.  A
// pixel's alphas are evaluated at once -- they do not depend on each other --
// and applied in list order by its E lanes together: all carry T, each the sums
// of 4 / E of the channels r, g, b, depth.  A pixel that saturates needs no
// branch: T only falls, so an entry counts while T after it is at least 1e-4.
// A (64-pixel, entry) step costs about 42 or 56 instructions.
//
// A wave streams the tile's list on its own, 64 entries at a time, with the ids
// of window w + 2 and the splats of window w + 1 in flight while window w is
// blended, keeps the entries that reach its block (splat_reaches) and stops
// when its own pixels are opaque.  With the list staged for the whole tile, a
// batch of 256 entries took two barriers and a chain of two dependent loads,
// and the heaviest tiles' nine batches set the launch's length: 162 us at
// 500 000 Gaussians and 960 x 540, 150 at 60 000 and 479 x 270, 318 at 1 200 000
// and 1920 x 1080; now 107, 50 and 270, bound by instructions (the first and the
// last) and by the longest wave's chain (the second).
// Workgroups of one wave, so that a wave that is done leaves its place to the
// next (with eight waves a workgroup, half of the wave slots stood empty).
//
// A smaller block wastes fewer lanes (on the training scene 48% of the lanes
// of an 8 x 8 block blend, 72% of a 4 x 4 block's; on a 480 x 270 pose frame 23%
// and 45%) and makes the wave's chain shorter, but every wave reads and tests
// the whole list, ~130 instructions per 64 entries.
template <int E>
__device__ __forceinline__ void blend_block(const BlendArgs& a, uint32_t tile, int part) {
  constexpr int kBlocks = 4 * E, kCh = 4 / E, kGroup = 4 * E;
  constexpr int kBW = E == 4 ? 4 : 8, kBH = kBW;  // the block's pixels
  constexpr int kSlots = 64 + 2 * kGroup;  // 64 new entries, those left over and the last group past them
  __shared__ float4 s_geo[kSlots];   // x, y, conic a, conic b
  __shared__ float2 s_op[kSlots];    // conic c, opacity
  __shared__ float4 s_ch[kSlots];    // r, g, b, depth
  __shared__ uint32_t s_pos[kSlots]; // position in the list + 1
  const int tx = tile % a.gx, ty = tile / a.gx;
  const int lane = threadIdx.x & 63;
  const int p = lane / E, e = lane % E;
  const int bx = (part % (kBX / kBW)) * kBW, by = (part / (kBX / kBW)) * kBH;
  const int dx = bx + p % kBW, dy = by + p / kBW;
  const int px = tx * kBX + dx, py = ty * kBY + dy;
  const bool inside = px < a.W && py < a.H;
  const float pfx = (float)px, pfy = (float)py;
  const uint32_t r0 = a.ranges[2 * tile], n = a.ranges[2 * tile + 1] - r0;
  const uint32_t* list = a.list + r0;
  const uint32_t base = a.ckpt_base[tile];
  bool done = !inside;
  float T = 1.0f, C[kCh];
#pragma unroll
  for (int c = 0; c < kCh; ++c) C[c] = 0.0f;
  uint32_t last = 0;
  const float a_min = 1.0f / 255.0f, t_min = 0.0001f;
  // value v of lane k of this lane's pixel
  auto of_lane = [](float v, int k) {
    if constexpr (E == 1) return v;
    if constexpr (E == 4) return k == 0 ? dpp<0x00>(v) : (k == 1 ? dpp<0x55>(v) : (k == 2 ? dpp<0xAA>(v) : dpp<0xFF>(v)));
  };
  if (n > 0 && __ballot(inside)) {
    const uint32_t nwin = (n + 63u) / 64u;
    auto id_at = [&](uint32_t w) { return list[min(w * 64u + (uint32_t)lane, n - 1u)] & a.id_mask; };
    uint32_t id = id_at(0);
    float4 sa = a.splat[3 * id], sb = a.splat[3 * id + 1], sc = a.splat[3 * id + 2];
    id = id_at(1);
    uint32_t have = 0;   // entries in the slots
    uint32_t count = 0;  // entries kept of this 256-entry batch
    uint64_t odd = 0;    // a colour in the slots is not finite
    uint32_t w = 0;
    for (; w < nwin; ++w) {
      const float4 ea = sa, eb = sb, ec = sc;
      sa = a.splat[3 * id];
      sb = a.splat[3 * id + 1];
      sc = a.splat[3 * id + 2];
      id = id_at(w + 2);
      if ((w & 3u) == 0 && w > 0) {
        // a 256-entry boundary: the state the backward resumes from
        const uint32_t batch = w >> 2;
        if (lane == 0 && count > 0) atomicAdd(&a.bweight[base + tile + batch - 1], count);
        count = 0;
        if (inside) {
          float* ck = a.ckpt + (size_t)(base + batch - 1) * 5 * 256 + tile_thread(dx, dy);
          if (e == 0) ck[0] = T;
#pragma unroll
          for (int c = 0; c < kCh; ++c) ck[256 * (1 + kCh * e + c)] = C[c];
        }
      }
      const uint32_t pos = w * 64u + (uint32_t)lane;
      const bool hit = pos < n && splat_reaches(ea.x, ea.y, ea.z, ea.w, eb.x, eb.y, (float)(tx * kBX + bx),
                                                (float)(ty * kBY + by), (float)kBW, (float)kBH);
      const uint64_t hits = __ballot(hit);
      if (hit) {
        const uint32_t slot = have + (uint32_t)__popcll(hits & lanemask_lt());
        s_geo[slot] = ea;
        s_op[slot] = make_float2(eb.x, eb.y);
        s_ch[slot] = make_float4(ec.x, ec.y, ec.z, eb.z);
        s_pos[slot] = pos + 1u;
      }
      // a colour that is not finite must not meet a weight of zero: one of this
      // window's, or of the entries left over from the last
      odd = (have > 0 ? odd : 0ull) | __ballot(hit && !(fabsf(ec.x) + fabsf(ec.y) + fabsf(ec.z) < __builtin_inff()));
      have += (uint32_t)__popcll(hits);
      count += (uint32_t)__popcll(hits);
      const bool flush = (w & 3u) == 3u || w + 1 == nwin;
      // the slots that fill up the last group weigh nothing
      if (flush && lane < kGroup) {
        s_op[have + lane] = make_float2(0.0f, 0.0f);
        s_ch[have + lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      }
      __builtin_amdgcn_wave_barrier();
      uint32_t at = 0;
      int hit_slot = -1;  // of the lane's last contributor in this window
      for (; at + kGroup <= have || (flush && at < have); at += kGroup) {
        const float* ch = &s_ch[at].x + kCh * e;
        float pw[4], ex[4], al[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const float4 ga = s_geo[at + s * E + e];
          pw[s] = blend_power(ga.z, ga.w, s_op[at + s * E + e].x, ga.x - pfx, ga.y - pfy);
        }
        spec_expf4(pw, ex);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const float araw = fminf(0.99f, s_op[at + s * E + e].y * ex[s]);
          // an entry that is skipped, or a pixel that is done, has alpha 0
          al[s] = pw[s] > 0.0f || araw < a_min || done ? 0.0f : araw;
        }
        float wt[kGroup], Tn = T;
        bool ok = true;
#pragma unroll
        for (int i = 0; i < kGroup; ++i) {
          const float Ti = Tn * of_lane(1.0f - al[i / E], i % E);
          ok = !(Ti < t_min);
          wt[i] = ok ? of_lane(al[i / E], i % E) * Tn : 0.0f;
          Tn = Ti;
          T = ok ? Ti : T;
        }
        done = done || !ok;
        if (odd == 0) {
#pragma unroll
          for (int i = 0; i < kGroup; ++i)
#pragma unroll
            for (int c = 0; c < kCh; ++c) C[c] = fmaf(ch[4 * i + c], wt[i], C[c]);
        } else {
#pragma unroll
          for (int i = 0; i < kGroup; ++i)
#pragma unroll
            for (int c = 0; c < kCh; ++c) C[c] = wt[i] != 0.0f ? fmaf(ch[4 * i + c], wt[i], C[c]) : C[c];
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          float mine = wt[s * E];
          if constexpr (E == 4)
            mine = e == 1 ? wt[s * E + 1] : (e == 2 ? wt[s * E + 2] : (e == 3 ? wt[s * E + 3] : mine));
          hit_slot = mine != 0.0f ? (int)at + s * E + e : hit_slot;
        }
      }
      if (hit_slot >= 0) last = s_pos[hit_slot];
      if (__ballot(!done) == 0) break;
      // the entries left over wait for the next window
      have = at < have ? have - at : 0u;
      if (at > 0 && (uint32_t)lane < have) {
        const float4 g = s_geo[at + lane], c = s_ch[at + lane];
        const float2 o = s_op[at + lane];
        const uint32_t q = s_pos[at + lane];
        s_geo[lane] = g;
        s_op[lane] = o;
        s_ch[lane] = c;
        s_pos[lane] = q;
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (lane == 0 && count > 0) atomicAdd(&a.bweight[base + tile + min(w, nwin - 1) / 4], count);
  }
  // (the last contributor lies in the lane of its entry)
  if constexpr (E == 4) {
    last = max(last, (uint32_t)__shfl_xor((int)last, 1, 64));
    last = max(last, (uint32_t)__shfl_xor((int)last, 2, 64));
  }
  if (inside) {
    const int pix = py * a.W + px;
    const int HW = a.H * a.W;
#pragma unroll
    for (int c = 0; c < kCh; ++c) {
      const int ch = kCh * e + c;
      a.accum[ch * HW + pix] = C[c];
      if (ch < 3) a.out_color[ch * HW + pix] = fmaf(T, a.bg[ch], C[c]);
      else a.out_depth[pix] = C[c];
    }
    if (e == 0) {
      a.final_T[pix] = T;
      a.n_contrib[pix] = last;
      if (a.out_alpha) a.out_alpha[pix] = 1.0f - T;
    }
  }
  if (n == 0) return;
  // The last of the tile's waves to get here logs the backward's work items:
  // the list's 256-entry chunks up to the tile's last contributor, each with a
  // cost class from the entries the waves kept of it (class 0 = most).  All of
  // it goes through atomics, which are performed one after another wherever
  // the waves ran; the waits keep a wave's own in order.
  const uint32_t wlast = wave_max_u32(last);
  uint32_t turn = 0;
  if (lane == 0) {
    atomicMax(&a.tile_maxc[tile], wlast);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    turn = atomicAdd(&a.tile_done[tile], 1u);
  }
  if (__builtin_amdgcn_readfirstlane((int)turn) != kBlocks - 1) return;
  const uint32_t maxc = atomicMax(&a.tile_maxc[tile], 0u);
  for (uint32_t c = lane; c * 256u < maxc; c += 64) {
    const uint32_t kept = atomicAdd(&a.bweight[base + tile + c], 0u);
    const uint32_t cls = 63u - min(kept / (4u * kBlocks), 63u);
    const uint32_t slot = atomicAdd(&a.item_log[0], 1u);
    a.item_log[1 + 2 * slot] = tile;
    a.item_log[2 + 2 * slot] = (c << 6) | cls;
  }
}

// Workgroup b's tile (rank in the blend's order) and block.  The blocks of a
// tile read the same list and splats: they are 8 apart, so dispatch, which
// deals workgroups round-robin over the 8 XCDs, puts them on one L2.
template <int E>
__device__ __forceinline__ uint32_t blend_rank(uint32_t b, int& part) {
  part = (int)(b / 8u % (4u * E));
  return b % 8u + 8u * (b / (32u * E));
}
// Launches of at most this many tiles blend on 4 x 4 blocks, larger ones on
// 8 x 8: up to here four waves a tile leave the SIMDs half empty and the
// longest wave sets the time, which the smaller block shortens; past it the
// instructions count, of which the smaller blocks issue more.  8 x 8 / 4 x 4,
// us: 46 / 26 at 256 tiles, 100 / 50 at 510, 87 / 50 at 858, 87 / 79 and
// 100 / 77 at 1 170 - 1 450 (training scenes), but 73 / 82 at 920 and 71 / 109
// at 2 040 for sparse views; 107 / 108 at 2 040, 270 / 564 at 8 160.  (The tiles
// alone do not tell: training scenes gain from 4 x 4 blocks beyond this line,
// sparse views lose before it.  It lies where neither loses much.)
constexpr int kCellTiles = 1024;
inline unsigned blend_grid(unsigned tiles, int e) { return (tiles + 7u) / 8u * 32u * (unsigned)e; }

template <int E>
__global__ __launch_bounds__(64) void k_blend(BlendArgs a, uint32_t tiles) {
  int part;
  const uint32_t r = blend_rank<E>(blockIdx.x, part);
  if (r < tiles) blend_block<E>(a, a.tile_order[r], part);
}

// Blend of many frames in one launch: one workgroup per tile of every frame
// (each frame's tiles in its longest-first order).
template <int E>
__global__ __launch_bounds__(64) void k_blend_multi(const uint32_t* prefix, const BlendArgs* args, int n) {
  int part;
  const uint32_t r = blend_rank<E>(blockIdx.x, part);
  if (r >= prefix[n]) return;
  const int f = frame_of_block(prefix, n, r);
  const BlendArgs a = args[f];
  blend_block<E>(a, a.tile_order[r - prefix[f]], part);
}

// One workgroup: checkpoint base of every tile = exclusive prefix over tiles
// of (batches in its list - 1); ckpt_base[n_tiles] = total checkpoints.
// It also clears what the blend's waves count in: the work-item log, each
// tile's words (tile_words: last contributors, then waves done) and the kept
// entries per batch (item_log and bweight are null where no list can exist).
// Also turns the ranges of empty tiles, left at [UINT_MAX, 0) by the
// depth-first list sort, into [0, 0), and orders the tiles for the blend,
// longest list first (a counting sort on the list length in 64-entry steps,
// capped at 255 steps; the order within a step is whatever the LDS atomics
// give, which no result depends on).  A launch lasts as long as its last
// tiles: the longest lists start first, and consecutive workgroups go to
// different XCDs, so the long lists of one image region spread over the GPU.
__device__ __forceinline__ void tile_ckpt_scan_block(uint32_t* ranges, int nt, uint32_t* ckpt_base,
                                                     uint32_t* item_log, uint32_t* tile_order,
                                                     uint32_t* tile_words, uint32_t* bweight) {
  __shared__ uint32_t s[1024];
  __shared__ uint32_t s_carry;
  __shared__ uint32_t s_cls[256];
  const int t = threadIdx.x;
  if (t == 0) {
    s_carry = 0;
    if (item_log) item_log[0] = 0;
  }
  __syncthreads();
  for (int b0 = 0; b0 < nt; b0 += 1024) {
    const int b = b0 + t;
    uint32_t v = 0;
    if (b < nt) {
      uint32_t r0 = ranges[2 * b];
      const uint32_t r1 = ranges[2 * b + 1];
      if (r0 > r1) {
        r0 = r1;  // r1 = 0: an empty tile
        ranges[2 * b] = 0u;
      }
      const uint32_t len = r1 - r0;
      const uint32_t nb = (len + 255) / 256;
      v = nb > 0 ? nb - 1 : 0;
    }
    uint32_t tot;
    const uint32_t incl = block_scan_incl<1024>(v, s, tot);
    const uint32_t carry = s_carry;
    if (b < nt) ckpt_base[b] = carry + incl - v;
    __syncthreads();
    if (t == 0) s_carry = carry + tot;
    __syncthreads();
  }
  if (t == 0) ckpt_base[nt] = s_carry;
  for (int k = t; k < 2 * nt; k += 1024) tile_words[k] = 0;
  if (bweight)
    for (uint32_t k = t; k < s_carry + (uint32_t)nt; k += 1024) bweight[k] = 0;
  if (t < 256) s_cls[t] = 0;
  __syncthreads();
  auto cls_of = [&](int b) { return min((ranges[2 * b + 1] - ranges[2 * b] + 63u) / 64u, 255u); };
  for (int b = t; b < nt; b += 1024) atomicAdd(&s_cls[cls_of(b)], 1u);
  __syncthreads();
  {
    // first position of each class, longest class first
    const uint32_t v = t < 256 ? s_cls[255 - t] : 0u;
    uint32_t tot;
    const uint32_t incl = block_scan_incl<1024>(v, s, tot);
    __syncthreads();
    if (t < 256) s_cls[255 - t] = incl - v;
  }
  __syncthreads();
  for (int b = t; b < nt; b += 1024) tile_order[atomicAdd(&s_cls[cls_of(b)], 1u)] = (uint32_t)b;
}

__global__ __launch_bounds__(1024) void k_tile_ckpt_scan(uint32_t* ranges, int nt, uint32_t* ckpt_base,
                                                         uint32_t* item_log, uint32_t* tile_order,
                                                         uint32_t* tile_words, uint32_t* bweight) {
  tile_ckpt_scan_block(ranges, nt, ckpt_base, item_log, tile_order, tile_words, bweight);
}

struct CkptScan {
  uint32_t* ranges;
  uint32_t* ckpt_base;
  uint32_t* item_log;
  uint32_t* tile_order;
  uint32_t* tile_words;
  uint32_t* bweight;
  int nt;
};

// Workgroup f: the checkpoint scan of frame f.
__global__ __launch_bounds__(1024) void k_tile_ckpt_scan_multi(const CkptScan* cs) {
  const CkptScan c = cs[blockIdx.x];
  tile_ckpt_scan_block(c.ranges, c.nt, c.ckpt_base, c.item_log, c.tile_order, c.tile_words, c.bweight);
}

__global__ __launch_bounds__(256) void k_mark_visible(const float* means, int P, const float* view,
                                                      uint8_t* visible) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= P) return;
  const f3 p = {means[3 * i], means[3 * i + 1], means[3 * i + 2]};
  visible[i] = xf43(view, p).z > 0.2f ? 1 : 0;
}

}  // namespace gs

// ---------------------------------------------------------------------------
// C ABI
using namespace gs;

namespace {
inline int grid_tiles(int W, int H, int& gx, int& gy) {
  gx = (W + kBX - 1) / kBX;
  gy = (H + kBY - 1) / kBY;
  return gx * gy;
}
inline int nblocks256(long long n) { return (int)((n + 255) / 256); }
}  // namespace

extern "C" int gs_geom_layout(int P, gs_geom_layout_t* out) {
  if (P < 0 || !out) return GS_E_ARG;
  const size_t p = (size_t)P;
  size_t o = 0;
  out->splat = o;
  o = align_up(o + 48 * p, 256);
  out->cov3D = o;
  o = align_up(o + 24 * p, 256);
  out->tiles = o;
  o = align_up(o + 4 * p, 256);
  out->offsets = o;
  o = align_up(o + 4 * p, 256);
  out->scan_tmp = o;
  o = align_up(o + 8 * (size_t)nblocks256(P) + 8, 256);
  out->total = o;
  return GS_OK;
}

extern "C" int gs_binning_layout(long long capacity, int P, int width, int height, int binning,
                                 gs_binning_layout_t* out) {
  if (capacity < 0 || capacity > 0x7fffffffLL || P < 0 || width <= 0 || height <= 0 || !out) return GS_E_ARG;
  if (binning != GS_BINNING_DEPTH_FIRST && binning != GS_BINNING_SORT64) return GS_E_ARG;
  int gx, gy;
  const int nt = grid_tiles(width, height, gx, gy);
  const size_t c = (size_t)capacity;
  const bool df = binning == GS_BINNING_DEPTH_FIRST;
  const size_t kb = df ? 4 : 8;
  size_t o = 0;
  out->keys_dup = o;
  o = align_up(o + kb * c, 256);
  out->keys_alt = o;
  o = align_up(o + kb * c, 256);
  out->vals_dup = o;
  o = align_up(o + 4 * c, 256);
  out->vals_alt = o;
  o = align_up(o + 4 * c, 256);
  const size_t p = df ? (size_t)P : 0;
  out->dkeys_a = o;
  o = align_up(o + 4 * p, 256);
  out->dvals_a = o;
  o = align_up(o + 4 * p, 256);
  out->dkeys_b = o;
  o = align_up(o + 4 * p, 256);
  out->dvals_b = o;
  o = align_up(o + 4 * p, 256);
  out->dscan = o;
  o = align_up(o + 4 * p, 256);
  out->dblocks = o;
  o = align_up(o + 4 * (p / 256 + 2), 256);
  out->drect = o;
  o = align_up(o + 8 * p, 256);
  out->hist = o;
  {
    // histogram space for both sorts that share it (their tile sizes may differ)
    const size_t t_list = sort_tmp_bytes(capacity), t_depth = sort_tmp_bytes((long long)p);
    o = align_up(o + (t_list > t_depth ? t_list : t_depth), 256);
  }
  // blend checkpoints: at most capacity / 256 batch boundaries, 5 x 256 floats each
  out->ckpt = o;
  o = align_up(o + (size_t)(c / 256 + 1) * 5 * 256 * sizeof(float), 256);
  // per (tile, batch) cost estimates: tile t's batches start at ckpt_base[t] + t
  out->bweight = o;
  o = align_up(o + 4 * (c / 256 + 2 * (size_t)nt + 2), 256);
  out->items = o;
  o = align_up(o + 16 * (1 + (c / 256 + (size_t)nt + 1)), 256);
  out->item_log = o;
  o = align_up(o + 4 * (1 + 2 * (c / 256 + (size_t)nt + 1)), 256);
  out->total = o;
  // one word per list entry when the Gaussian id and the tile id fit together
  const int tb = bits_for((uint32_t)nt), idb = bits_for((uint32_t)(P > 1 ? P : 2));
  out->id_bits = (df && idb + tb <= 32) ? idb : 0;
  const int end_bit = (df ? 0 : 32) + tb;
  out->sort_passes = out->id_bits && wide_digit(tb, capacity) ? 1 : sort_passes(end_bit > 0 ? end_bit : 1);
  out->key_bytes = (int)kb;
  const bool in_b = (out->sort_passes & 1) != 0;
  out->keys_sorted = in_b ? out->keys_alt : out->keys_dup;
  out->vals_sorted = in_b ? out->vals_alt : out->vals_dup;
  if (out->id_bits) out->vals_sorted = out->keys_sorted;
  return GS_OK;
}

extern "C" int gs_image_layout(int width, int height, gs_image_layout_t* out) {
  if (width <= 0 || height <= 0 || !out) return GS_E_ARG;
  int gx, gy;
  const int nt = grid_tiles(width, height, gx, gy);
  const size_t hw = (size_t)width * height;
  size_t o = 0;
  out->ranges = o;
  o = align_up(o + 8 * (size_t)nt, 256);
  out->final_T = o;
  o = align_up(o + 4 * hw, 256);
  out->n_contrib = o;
  o = align_up(o + 4 * hw, 256);
  out->accum = o;
  o = align_up(o + 16 * hw, 256);
  out->ckpt_base = o;
  o = align_up(o + 4 * ((size_t)nt + 1), 256);
  out->tile_maxc = o;  // and behind them the count of the tile's waves that are through
  o = align_up(o + 8 * (size_t)nt, 256);
  out->tile_order = o;
  o = align_up(o + 4 * (size_t)nt, 256);
  out->total = o;
  return GS_OK;
}

static int check_frame(const gs_frame_t* f) {
  if (!f || f->width <= 0 || f->height <= 0 || !f->viewmatrix || !f->projmatrix || !f->bg) return GS_E_ARG;
  if (f->sh_degree < 0 || f->sh_degree > 3) return GS_E_ARG;
  return GS_OK;
}

// The checked preprocess arguments of one frame.
static int make_pre_args(const gs_frame_t* f, const gs_gaussians_t* g, int* radii, void* geom, size_t geom_bytes,
                         const uint32_t* counters, PreArgs& a) {
  if (check_frame(f) != GS_OK || !g || g->P < 0 || !counters) return GS_E_ARG;
  const int P = g->P;
  if (P > 0 && (!g->means3D || !g->opacities || !radii || !geom)) return GS_E_ARG;
  // (empty inputs carry no pointers, so the exactly-one-of rules apply for P > 0)
  if (P > 0 && (g->shs == nullptr) == (g->colors_precomp == nullptr)) return GS_E_ARG;
  const bool has_sr = g->scales && g->rotations;
  if (P > 0 && has_sr == (g->cov3D_precomp != nullptr)) return GS_E_ARG;
  if (g->shs && (f->sh_degree + 1) * (f->sh_degree + 1) > g->M) return GS_E_ARG;
  if (g->shs && !f->campos) return GS_E_ARG;
  gs_geom_layout_t L;
  gs_geom_layout(P, &L);
  if (geom_bytes < L.total) return GS_E_WORKSPACE;
  char* base = (char*)geom;
  a.P = P;
  a.M = g->M;
  a.D = f->sh_degree;
  a.W = f->width;
  a.H = f->height;
  grid_tiles(a.W, a.H, a.gx, a.gy);
  a.prefiltered = f->prefiltered;
  a.tanfovx = f->tanfovx;
  a.tanfovy = f->tanfovy;
  a.fx = (float)a.W / (2.0f * f->tanfovx);
  a.fy = (float)a.H / (2.0f * f->tanfovy);
  a.scale_mod = f->scale_modifier;
  a.view = f->viewmatrix;
  a.proj = f->projmatrix;
  a.campos = f->campos;
  a.pose = f->pose;
  a.means = g->means3D;
  a.shs = g->shs;
  a.colors = g->colors_precomp;
  a.opac = g->opacities;
  a.scales = g->scales;
  a.rots = g->rotations;
  a.cov_pre = g->cov3D_precomp;
  a.radii = radii;
  a.splat = (float4*)(base + L.splat);
  a.cov3D = (float*)(base + L.cov3D);
  a.tiles = (uint32_t*)(base + L.tiles);
  a.local_incl = (uint32_t*)(base + L.offsets);
  a.block_sum = (uint32_t*)(base + L.scan_tmp);
  return GS_OK;
}

// Dynamic LDS of a preprocess launch: the staged SH rows of 256 Gaussians
// (an odd row stride).
static size_t preprocess_lds(const PreArgs& a) {
  const int nc = (a.D + 1) * (a.D + 1);
  return a.shs ? (size_t)256 * ((3 * nc) | 1) * sizeof(float) : 0;
}

extern "C" int gs_preprocess(const gs_frame_t* f, const gs_gaussians_t* g, int* radii, void* geom,
                             size_t geom_bytes, uint32_t* counters, void* stream) {
  PreArgs a;
  const int rc = make_pre_args(f, g, radii, geom, geom_bytes, counters, a);
  if (rc != GS_OK) return rc;
  hipStream_t s = (hipStream_t)stream;
  const int nb = nblocks256(a.P);
  if (nb > 0) {
    const size_t shm = preprocess_lds(a);
    timing::Scope ts(timing::kPreprocess, s);
    hipLaunchKernelGGL(k_preprocess, dim3(nb), dim3(256), shm, s, a);
  }
  {
    timing::Scope ts(timing::kScan, s);
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, s, a.block_sum, nb, counters);
  }
  return hipGetLastError() == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

// Binning of one frame: everything of the forward but the blend (ranges
// cleared, depth-first or 64-bit-key binning, ranges, checkpoint bases).
// Phases of the binning: kPrepare is everything that does not read
// num_rendered (clearing the tile ranges; in the depth-first schedule also
// the depth keys, the 32-bit depth sort and the prefix of the tile counts in
// depth order), so a caller can queue it before it waits for the readback;
// kResume is the rest, after kPrepare with the same arguments.  The other
// phases split the depth-first schedule around its two sorts instead, so
// that one segmented sort can serve many frames: kKeys is the depth keys
// alone; kAfterSort everything after the depth sort; kDup the tile-count
// prefix and the duplicate (after the depth sort, before the list sort);
// kTail what follows the list sort (the checkpoint scan).
enum BinPhase { kBinAll = 0, kPrepare = 1, kResume = 2, kKeys = 3, kAfterSort = 4, kDup = 5, kTail = 6 };

static int render_binning(const gs_frame_t* f, int P, const void* geom, uint32_t* counters, long long capacity,
                          void* binning, size_t binning_bytes, void* image, size_t image_bytes, hipStream_t s,
                          int phase = kBinAll) {
  const bool pre = phase == kBinAll || phase == kPrepare, post = phase == kBinAll || phase == kResume;
  const bool split = phase == kKeys || phase == kAfterSort || phase == kDup || phase == kTail;
  if (check_frame(f) != GS_OK || P < 0 || !counters || !image) return GS_E_ARG;
  if (P > 0 && !geom) return GS_E_ARG;
  if (capacity < 0 || capacity > 0x7fffffffLL) return GS_E_ARG;
  gs_geom_layout_t LG;
  gs_binning_layout_t LB;
  gs_image_layout_t LI;
  gs_geom_layout(P, &LG);
  if (gs_binning_layout(capacity, P, f->width, f->height, f->binning, &LB) != GS_OK) return GS_E_ARG;
  gs_image_layout(f->width, f->height, &LI);
  if (binning_bytes < LB.total || image_bytes < LI.total) return GS_E_WORKSPACE;
  if (capacity > 0 && !binning) return GS_E_ARG;
  int gx, gy;
  const int nt = grid_tiles(f->width, f->height, gx, gy);
  const char* gb = (const char*)geom;
  char* bb = (char*)binning;
  char* ib = (char*)image;
  uint32_t* ranges = (uint32_t*)(ib + LI.ranges);
  const bool df = capacity > 0 && P > 0 && f->binning == GS_BINNING_DEPTH_FIRST;
  if (split && !df) return GS_E_ARG;  // only the depth-first schedule has a depth sort to split around
  // depth-first stages: keys | depth sort | tile-count prefix | duplicate | list sort | checkpoint scan
  const bool do_keys = pre || phase == kKeys, do_dsort = pre;
  const bool do_dscan = pre || phase == kAfterSort || phase == kDup;
  const bool do_dup = post || phase == kAfterSort || phase == kDup, do_lsort = post || phase == kAfterSort;
  const bool do_ckpt = post || phase == kAfterSort || phase == kTail;
  if (pre && !df)  // the depth-first schedule clears them in k_df_keys
    hipLaunchKernelGGL(k_fill_u32, dim3(std::min(nblocks256(2LL * nt), 1024)), dim3(256), 0, s, ranges, 2LL * nt,
                       0u);
  if (df) {
    if (gx > 0xffff || gy > 0xffff) return GS_E_ARG;  // tile rects are packed in 16-bit fields
    const float4* splat = (const float4*)(gb + LG.splat);
    const uint32_t* tiles = (const uint32_t*)(gb + LG.tiles);
    uint32_t* dka = (uint32_t*)(bb + LB.dkeys_a);
    uint32_t* dva = (uint32_t*)(bb + LB.dvals_a);
    const int nbp = nblocks256(P);
    hipError_t e = hipSuccess;
    int in_b = sort_passes(32) & 1;  // where the depth sort (or a segmented sort of it) leaves its result
    if (do_keys || do_dsort) {
      {
        timing::Scope ts(timing::kSort, s);
        if (do_keys)
          hipLaunchKernelGGL(k_df_keys, dim3(std::max(nbp, nblocks256(2LL * nt))), dim3(256), 0, s, P, tiles,
                             splat, gx, gy, dka, dva, (uint2*)(bb + LB.drect), counters, ranges, 2 * nt);
        if (do_dsort)
          e = sort_pairs_u32(dka, dva, (uint32_t*)(bb + LB.dkeys_b), (uint32_t*)(bb + LB.dvals_b), nullptr, P,
                             32, bb + LB.hist, s, &in_b);
      }
      if (e != hipSuccess) return GS_E_LAUNCH;
    }
    const uint32_t* dvals = (const uint32_t*)(bb + (in_b ? LB.dvals_b : LB.dvals_a));
    if (do_dscan) {
      timing::Scope ts(timing::kDuplicate, s);
      hipLaunchKernelGGL(k_df_scan, dim3(nbp), dim3(256), 0, s, P, dvals, tiles, (uint32_t*)(bb + LB.dscan),
                         (uint32_t*)(bb + LB.dblocks));
      if (nbp > (int)kOwnPrefix)
        hipLaunchKernelGGL(k_excl_scan_1wg, dim3(1), dim3(1024), 0, s, (uint32_t*)(bb + LB.dblocks), nbp);
    }
    if (do_dup) {
      timing::Scope ts(timing::kDuplicate, s);
      DfDupArgs d;
      d.P = P;
      d.gx = gx;
      d.gy = gy;
      d.capacity = capacity;
      d.rect = (const uint2*)(bb + LB.drect);
      d.tiles = tiles;
      d.dvals = dvals;
      d.dscan = (const uint32_t*)(bb + LB.dscan);
      d.dblocks = (const uint32_t*)(bb + LB.dblocks);
      d.counters = counters;
      d.keys = (uint32_t*)(bb + LB.keys_dup);
      d.vals = (uint32_t*)(bb + LB.vals_dup);
      d.id_bits = LB.id_bits;
      // a workgroup per 1024 entries where there is room for as many, up to what
      // the GPU holds at once
      const long long nchunk = (capacity + 1023) / 1024;
      hipLaunchKernelGGL(k_df_duplicate, dim3((unsigned)std::max<long long>(nbp, std::min(nchunk, 2048LL))), dim3(256), 0, s, d);
    }
    if (do_lsort) {
      timing::Scope ts(timing::kSort, s);
      const int tb = bits_for((uint32_t)nt) > 0 ? bits_for((uint32_t)nt) : 1;
      // the last pass also records the tile ranges
      if (LB.id_bits)  // one word per entry: sort on its tile bits only
        e = sort_keys_u32((uint32_t*)(bb + LB.keys_dup), (uint32_t*)(bb + LB.keys_alt), counters, capacity,
                          LB.id_bits, LB.id_bits + tb, bb + LB.hist, s, &in_b, ranges);
      else
        e = sort_pairs_u32((uint32_t*)(bb + LB.keys_dup), (uint32_t*)(bb + LB.vals_dup),
                           (uint32_t*)(bb + LB.keys_alt), (uint32_t*)(bb + LB.vals_alt), counters, capacity, tb,
                           bb + LB.hist, s, &in_b, ranges);
    }
    if (e != hipSuccess) return GS_E_LAUNCH;
  } else if (capacity > 0 && P > 0) {
    if (!post) return hipGetLastError() == hipSuccess ? GS_OK : GS_E_LAUNCH;
    DupArgs d;
    d.P = P;
    d.gx = gx;
    d.gy = gy;
    d.capacity = capacity;
    d.splat = (const float4*)(gb + LG.splat);
    d.tiles = (const uint32_t*)(gb + LG.tiles);
    d.local_incl = (const uint32_t*)(gb + LG.offsets);
    d.block_excl = (const uint32_t*)(gb + LG.scan_tmp);
    d.counters = counters;
    d.keys = (uint64_t*)(bb + LB.keys_dup);
    d.vals = (uint32_t*)(bb + LB.vals_dup);
    {
      timing::Scope ts(timing::kDuplicate, s);
      hipLaunchKernelGGL(k_duplicate, dim3(nblocks256(P)), dim3(256), 0, s, d);
    }
    const int end_bit = 32 + bits_for((uint32_t)nt);
    int in_b = 0;
    hipError_t e;
    {
      timing::Scope ts_sort(timing::kSort, s);
      e = sort_pairs_u64((uint64_t*)(bb + LB.keys_dup), (uint32_t*)(bb + LB.vals_dup), (uint64_t*)(bb + LB.keys_alt),
                         (uint32_t*)(bb + LB.vals_alt), counters, capacity, end_bit, bb + LB.hist, s, &in_b);
    }
    if (e != hipSuccess) return GS_E_LAUNCH;
    timing::Scope ts(timing::kRanges, s);
    hipLaunchKernelGGL(k_ranges, dim3(nblocks256(capacity)), dim3(256), 0, s,
                       (const uint64_t*)(bb + LB.keys_sorted), (const uint32_t*)counters, capacity, ranges);
  }
  if (post || (df && do_ckpt))
    hipLaunchKernelGGL(k_tile_ckpt_scan, dim3(1), dim3(1024), 0, s, ranges, nt, (uint32_t*)(ib + LI.ckpt_base),
                       bb ? (uint32_t*)(bb + LB.item_log) : nullptr, (uint32_t*)(ib + LI.tile_order),
                       (uint32_t*)(ib + LI.tile_maxc), bb ? (uint32_t*)(bb + LB.bweight) : nullptr);
  return hipGetLastError() == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

// Blend arguments of one frame (its workspaces as binned by render_binning).
static BlendArgs make_blend_args(const gs_frame_t* f, int P, const void* geom, long long capacity,
                                 void* binning, void* image, float* out_color, float* out_depth,
                                 float* out_alpha) {
  gs_geom_layout_t LG;
  gs_binning_layout_t LB;
  gs_image_layout_t LI;
  gs_geom_layout(P, &LG);
  gs_binning_layout(capacity, P, f->width, f->height, f->binning, &LB);
  gs_image_layout(f->width, f->height, &LI);
  int gx, gy;
  grid_tiles(f->width, f->height, gx, gy);
  const char* gb = (const char*)geom;
  char* bb = (char*)binning;
  char* ib = (char*)image;
  BlendArgs b;
  b.W = f->width;
  b.H = f->height;
  b.gx = gx;
  b.ranges = (const uint32_t*)(ib + LI.ranges);
  b.list = capacity > 0 ? (const uint32_t*)(bb + LB.vals_sorted) : nullptr;
  b.id_mask = LB.id_bits ? (1u << LB.id_bits) - 1u : 0xffffffffu;
  b.splat = (const float4*)(gb + LG.splat);
  b.bg = f->bg;
  b.out_color = out_color;
  b.out_depth = out_depth;
  b.out_alpha = out_alpha;
  b.final_T = (float*)(ib + LI.final_T);
  b.n_contrib = (uint32_t*)(ib + LI.n_contrib);
  b.ckpt_base = (const uint32_t*)(ib + LI.ckpt_base);
  b.ckpt = (float*)(bb + LB.ckpt);
  b.tile_maxc = (uint32_t*)(ib + LI.tile_maxc);
  b.tile_done = b.tile_maxc + grid_tiles(f->width, f->height, gx, gy);
  b.tile_order = (const uint32_t*)(ib + LI.tile_order);
  b.bweight = (uint32_t*)(bb + LB.bweight);
  b.item_log = (uint32_t*)(bb + LB.item_log);
  b.accum = (float*)(ib + LI.accum);
  return b;
}

extern "C" int gs_render_binning(const gs_frame_t* f, int P, const void* geom, uint32_t* counters,
                                 long long capacity, void* binning, size_t binning_bytes, void* image,
                                 size_t image_bytes, void* stream) {
  return render_binning(f, P, geom, counters, capacity, binning, binning_bytes, image, image_bytes,
                        (hipStream_t)stream);
}

static int render_blend_from(int phase, const gs_frame_t* f, int P, const void* geom, uint32_t* counters,
                             long long capacity, void* binning, size_t binning_bytes, void* image, size_t image_bytes,
                             float* out_color, float* out_depth, float* out_alpha, hipStream_t s) {
  if (!out_color || !out_depth) return GS_E_ARG;
  const int rc = render_binning(f, P, geom, counters, capacity, binning, binning_bytes, image, image_bytes, s, phase);
  if (rc != GS_OK) return rc;
  const BlendArgs b = make_blend_args(f, P, geom, capacity, binning, image, out_color, out_depth, out_alpha);
  int gx, gy;
  const int nt = grid_tiles(f->width, f->height, gx, gy);
  {
    timing::Scope ts(timing::kBlend, s);
    if (nt <= kCellTiles) hipLaunchKernelGGL(k_blend<4>, dim3(blend_grid(nt, 4)), dim3(64), 0, s, b, (uint32_t)nt);
    else hipLaunchKernelGGL(k_blend<1>, dim3(blend_grid(nt, 1)), dim3(64), 0, s, b, (uint32_t)nt);
  }
  return hipGetLastError() == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

extern "C" int gs_render(const gs_frame_t* f, int P, const void* geom, uint32_t* counters, long long capacity,
                         void* binning, size_t binning_bytes, void* image, size_t image_bytes, float* out_color,
                         float* out_depth, float* out_alpha, void* stream) {
  return render_blend_from(kBinAll, f, P, geom, counters, capacity, binning, binning_bytes, image, image_bytes,
                           out_color, out_depth, out_alpha, (hipStream_t)stream);
}

extern "C" int gs_render_prepare(const gs_frame_t* f, int P, const void* geom, uint32_t* counters, long long capacity,
                                 void* binning, size_t binning_bytes, void* image, size_t image_bytes, void* stream) {
  return render_binning(f, P, geom, counters, capacity, binning, binning_bytes, image, image_bytes,
                        (hipStream_t)stream, kPrepare);
}

extern "C" int gs_render_resume(const gs_frame_t* f, int P, const void* geom, uint32_t* counters, long long capacity,
                                void* binning, size_t binning_bytes, void* image, size_t image_bytes,
                                float* out_color, float* out_depth, float* out_alpha, void* stream) {
  return render_blend_from(kResume, f, P, geom, counters, capacity, binning, binning_bytes, image, image_bytes,
                           out_color, out_depth, out_alpha, (hipStream_t)stream);
}

// ---- the depth-first binning around a depth sort shared by many frames -----
extern "C" int gs_render_depth_keys(const gs_frame_t* f, int P, const void* geom, uint32_t* counters,
                                    long long capacity, void* binning, size_t binning_bytes, void* image,
                                    size_t image_bytes, void* stream) {
  return render_binning(f, P, geom, counters, capacity, binning, binning_bytes, image, image_bytes,
                        (hipStream_t)stream, kKeys);
}

// ---- many frames' preprocess and depth keys in three launches --------------
// Set layout: uint32 prefix[n + 1] of preprocess workgroup bounds per frame,
// uint32 prefix[n + 1] of depth-key workgroup bounds, then PreArgs[n],
// ScanTop[n] and DfKeysArgs[n], each array at a 256-byte boundary.
static size_t mpk_prefix2_offset(int n) { return align_up(sizeof(uint32_t) * (size_t)(n + 1), 256); }
static size_t mpk_pre_offset(int n) { return 2 * mpk_prefix2_offset(n); }
static size_t mpk_top_offset(int n) { return mpk_pre_offset(n) + align_up(sizeof(PreArgs) * (size_t)n, 256); }
static size_t mpk_keys_offset(int n) { return mpk_top_offset(n) + align_up(sizeof(ScanTop) * (size_t)n, 256); }

extern "C" size_t gs_multi_preprocess_keys_bytes(int n) {
  return n <= 0 ? 0 : mpk_keys_offset(n) + sizeof(DfKeysArgs) * (size_t)n;
}

extern "C" int gs_multi_preprocess_keys_build(int n, const gs_frame_t* frames, const gs_gaussians_t* gauss,
                                              int* const* radii, void* const* geom, const size_t* geom_bytes,
                                              uint32_t* const* counters, const long long* capacity,
                                              void* const* binning, const size_t* binning_bytes,
                                              void* const* image, const size_t* image_bytes, void* host_set,
                                              size_t set_bytes, unsigned* launch) {
  if (n <= 0 || !frames || !gauss || !radii || !geom || !geom_bytes || !counters || !capacity || !binning ||
      !binning_bytes || !image || !image_bytes || !host_set || !launch)
    return GS_E_ARG;
  if (set_bytes < gs_multi_preprocess_keys_bytes(n)) return GS_E_WORKSPACE;
  uint32_t* pprefix = (uint32_t*)host_set;
  uint32_t* kprefix = (uint32_t*)((char*)host_set + mpk_prefix2_offset(n));
  PreArgs* pre = (PreArgs*)((char*)host_set + mpk_pre_offset(n));
  ScanTop* top = (ScanTop*)((char*)host_set + mpk_top_offset(n));
  DfKeysArgs* keys = (DfKeysArgs*)((char*)host_set + mpk_keys_offset(n));
  unsigned long long ptotal = 0, ktotal = 0;
  size_t shm = 0;
  for (int i = 0; i < n; ++i) {
    const gs_frame_t* f = &frames[i];
    const int rc = make_pre_args(f, &gauss[i], radii[i], geom[i], geom_bytes[i], counters[i], pre[i]);
    if (rc != GS_OK) return rc;
    const int P = gauss[i].P;
    // the depth keys of the depth-first schedule, as gs_render_depth_keys
    // takes them
    if (P <= 0 || f->binning != GS_BINNING_DEPTH_FIRST || capacity[i] <= 0 || capacity[i] > 0x7fffffffLL ||
        !binning[i] || !image[i])
      return GS_E_ARG;
    gs_geom_layout_t LG;
    gs_binning_layout_t LB;
    gs_image_layout_t LI;
    gs_geom_layout(P, &LG);
    if (gs_binning_layout(capacity[i], P, f->width, f->height, f->binning, &LB) != GS_OK) return GS_E_ARG;
    gs_image_layout(f->width, f->height, &LI);
    if (binning_bytes[i] < LB.total || image_bytes[i] < LI.total) return GS_E_WORKSPACE;
    int gx, gy;
    const int nt = grid_tiles(f->width, f->height, gx, gy);
    if (gx > 0xffff || gy > 0xffff) return GS_E_ARG;  // tile rects are packed in 16-bit fields
    const int nbp = nblocks256(P);
    pprefix[i] = (uint32_t)ptotal;
    ptotal += (unsigned long long)nbp;
    kprefix[i] = (uint32_t)ktotal;
    ktotal += (unsigned long long)std::max(nbp, nblocks256(2LL * nt));
    if (ptotal > 0x7fffffffULL || ktotal > 0x7fffffffULL) return GS_E_ARG;
    shm = std::max(shm, preprocess_lds(pre[i]));
    top[i].block_sum = pre[i].block_sum;
    top[i].counters = counters[i];
    top[i].nblocks = nbp;
    const char* gb = (const char*)geom[i];
    char* bb = (char*)binning[i];
    DfKeysArgs& k = keys[i];
    k.P = P;
    k.gx = gx;
    k.gy = gy;
    k.n_ranges = 2 * nt;
    k.tiles = (const uint32_t*)(gb + LG.tiles);
    k.splat = (const float4*)(gb + LG.splat);
    k.keys = (uint32_t*)(bb + LB.dkeys_a);
    k.vals = (uint32_t*)(bb + LB.dvals_a);
    k.rect = (uint2*)(bb + LB.drect);
    k.counters = counters[i];
    k.ranges = (uint32_t*)((char*)image[i] + LI.ranges);
  }
  pprefix[n] = (uint32_t)ptotal;
  kprefix[n] = (uint32_t)ktotal;
  launch[0] = (unsigned)ptotal;
  launch[1] = (unsigned)ktotal;
  launch[2] = (unsigned)shm;
  return GS_OK;
}

extern "C" int gs_multi_preprocess_keys(int n, const void* dev_set, const unsigned* launch, void* stream) {
  if (n <= 0 || !dev_set || !launch) return GS_E_ARG;
  hipStream_t s = (hipStream_t)stream;
  const char* d = (const char*)dev_set;
  if (launch[0] > 0) {
    timing::Scope ts(timing::kPreprocess, s);
    hipLaunchKernelGGL(k_preprocess_multi, dim3(launch[0]), dim3(256), (size_t)launch[2], s, (const uint32_t*)d,
                       (const PreArgs*)(d + mpk_pre_offset(n)), n);
  }
  {
    timing::Scope ts(timing::kScan, s);
    hipLaunchKernelGGL(k_scan_top_multi, dim3(n), dim3(256), 0, s, (const ScanTop*)(d + mpk_top_offset(n)));
  }
  if (launch[1] > 0) {
    timing::Scope ts(timing::kSort, s);
    hipLaunchKernelGGL(k_df_keys_multi, dim3(launch[1]), dim3(256), 0, s,
                       (const uint32_t*)(d + mpk_prefix2_offset(n)), (const DfKeysArgs*)(d + mpk_keys_offset(n)), n);
  }
  return hipGetLastError() == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

// ---- many frames' binning steps around the list sort ----------------------
// Set layout: uint32 prefix[n + 1] of per-Gaussian workgroup bounds per frame,
// then DfMid[n] and CkptScan[n], each array at a 256-byte boundary.
// beside the workgroup count the build returns: some frame needs the launch
// that forms the block prefixes
constexpr unsigned kMidPrefixes = 1u << 31;
static size_t mbm_mid_offset(int n) { return align_up(sizeof(uint32_t) * (size_t)(n + 1), 256); }
static size_t mbm_ckpt_offset(int n) { return mbm_mid_offset(n) + align_up(sizeof(DfMid) * (size_t)n, 256); }

extern "C" size_t gs_multi_binning_steps_bytes(int n) {
  return n <= 0 ? 0 : mbm_ckpt_offset(n) + sizeof(CkptScan) * (size_t)n;
}

extern "C" int gs_multi_binning_steps_build(int n, const gs_frame_t* frames, const int* P, const void* const* geom,
                                            uint32_t* const* counters, const long long* capacity,
                                            void* const* binning, const size_t* binning_bytes, void* const* image,
                                            const size_t* image_bytes, void* host_set, size_t set_bytes,
                                            unsigned* total_blocks) {
  if (n <= 0 || !frames || !P || !geom || !counters || !capacity || !binning || !binning_bytes || !image ||
      !image_bytes || !host_set || !total_blocks)
    return GS_E_ARG;
  if (set_bytes < gs_multi_binning_steps_bytes(n)) return GS_E_WORKSPACE;
  uint32_t* prefix = (uint32_t*)host_set;
  DfMid* mid = (DfMid*)((char*)host_set + mbm_mid_offset(n));
  CkptScan* ck = (CkptScan*)((char*)host_set + mbm_ckpt_offset(n));
  unsigned long long total = 0;
  bool prefixes = false;
  for (int i = 0; i < n; ++i) {
    const gs_frame_t* f = &frames[i];
    // the depth-first schedule's split phases, as gs_render_binning_duplicate
    // and gs_render_binning_after_list_sort take them
    if (check_frame(f) != GS_OK || P[i] <= 0 || !geom[i] || !counters[i] || !binning[i] || !image[i] ||
        capacity[i] <= 0 || capacity[i] > 0x7fffffffLL || f->binning != GS_BINNING_DEPTH_FIRST)
      return GS_E_ARG;
    gs_geom_layout_t LG;
    gs_binning_layout_t LB;
    gs_image_layout_t LI;
    gs_geom_layout(P[i], &LG);
    if (gs_binning_layout(capacity[i], P[i], f->width, f->height, f->binning, &LB) != GS_OK) return GS_E_ARG;
    gs_image_layout(f->width, f->height, &LI);
    if (binning_bytes[i] < LB.total || image_bytes[i] < LI.total) return GS_E_WORKSPACE;
    int gx, gy;
    const int nt = grid_tiles(f->width, f->height, gx, gy);
    if (gx > 0xffff || gy > 0xffff) return GS_E_ARG;  // tile rects are packed in 16-bit fields
    const int nbp = nblocks256(P[i]);
    prefixes |= nbp > (int)kOwnPrefix;
    prefix[i] = (uint32_t)total;
    total += (unsigned long long)nbp;
    if (total > 0x7fffffffULL) return GS_E_ARG;
    const char* gb = (const char*)geom[i];
    char* bb = (char*)binning[i];
    char* ib = (char*)image[i];
    // where the depth sort (per frame or segmented) leaves its result
    const int in_b = sort_passes(32) & 1;
    DfDupArgs& d = mid[i].dup;
    d.P = P[i];
    d.gx = gx;
    d.gy = gy;
    d.capacity = capacity[i];
    d.rect = (const uint2*)(bb + LB.drect);
    d.tiles = (const uint32_t*)(gb + LG.tiles);
    d.dvals = (const uint32_t*)(bb + (in_b ? LB.dvals_b : LB.dvals_a));
    d.dscan = (const uint32_t*)(bb + LB.dscan);
    d.dblocks = (const uint32_t*)(bb + LB.dblocks);
    d.counters = counters[i];
    d.keys = (uint32_t*)(bb + LB.keys_dup);
    d.vals = (uint32_t*)(bb + LB.vals_dup);
    d.id_bits = LB.id_bits;
    mid[i].dscan = (uint32_t*)(bb + LB.dscan);
    mid[i].dblocks = (uint32_t*)(bb + LB.dblocks);
    mid[i].nblocks = nbp;
    ck[i].ranges = (uint32_t*)(ib + LI.ranges);
    ck[i].ckpt_base = (uint32_t*)(ib + LI.ckpt_base);
    ck[i].item_log = (uint32_t*)(bb + LB.item_log);
    ck[i].tile_words = (uint32_t*)(ib + LI.tile_maxc);
    ck[i].bweight = (uint32_t*)(bb + LB.bweight);
    ck[i].tile_order = (uint32_t*)(ib + LI.tile_order);
    ck[i].nt = nt;
  }
  prefix[n] = (uint32_t)total;
  *total_blocks = (unsigned)total | (prefixes ? kMidPrefixes : 0u);
  return GS_OK;
}

extern "C" int gs_multi_binning_duplicate(int n, const void* dev_set, unsigned total_blocks, void* stream) {
  if (n <= 0 || !dev_set) return GS_E_ARG;
  const bool prefixes = total_blocks & kMidPrefixes;
  total_blocks &= ~kMidPrefixes;
  hipStream_t s = (hipStream_t)stream;
  const uint32_t* prefix = (const uint32_t*)dev_set;
  const DfMid* mid = (const DfMid*)((const char*)dev_set + mbm_mid_offset(n));
  timing::Scope ts(timing::kDuplicate, s);
  if (total_blocks > 0) hipLaunchKernelGGL(k_df_scan_multi, dim3(total_blocks), dim3(256), 0, s, prefix, mid, n);
  if (prefixes) hipLaunchKernelGGL(k_excl_scan_multi, dim3(n), dim3(256), 0, s, mid);
  if (total_blocks > 0)
    hipLaunchKernelGGL(k_df_duplicate_multi, dim3(total_blocks), dim3(256), 0, s, prefix, mid, n);
  return hipGetLastError() == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

extern "C" int gs_multi_binning_after_list_sort(int n, const void* dev_set, void* stream) {
  if (n <= 0 || !dev_set) return GS_E_ARG;
  hipLaunchKernelGGL(k_tile_ckpt_scan_multi, dim3(n), dim3(1024), 0, (hipStream_t)stream,
                     (const CkptScan*)((const char*)dev_set + mbm_ckpt_offset(n)));
  return hipGetLastError() == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

extern "C" int gs_render_binning_after_depth_sort(const gs_frame_t* f, int P, const void* geom, uint32_t* counters,
                                                  long long capacity, void* binning, size_t binning_bytes,
                                                  void* image, size_t image_bytes, void* stream) {
  return render_binning(f, P, geom, counters, capacity, binning, binning_bytes, image, image_bytes,
                        (hipStream_t)stream, kAfterSort);
}

extern "C" int gs_render_after_depth_sort(const gs_frame_t* f, int P, const void* geom, uint32_t* counters,
                                          long long capacity, void* binning, size_t binning_bytes, void* image,
                                          size_t image_bytes, float* out_color, float* out_depth, float* out_alpha,
                                          void* stream) {
  return render_blend_from(kAfterSort, f, P, geom, counters, capacity, binning, binning_bytes, image, image_bytes,
                           out_color, out_depth, out_alpha, (hipStream_t)stream);
}

extern "C" size_t gs_multi_depth_sort_bytes(int n) { return seg_sort_desc_bytes(n, sort_passes(32)); }

extern "C" int gs_multi_depth_sort_build(int n, const gs_frame_t* frames, const int* P, const long long* capacity,
                                         void* const* binning, const size_t* binning_bytes,
                                         uint32_t* const* counters, void* host_set, size_t set_bytes,
                                         unsigned* blocks) {
  if (n <= 0 || !frames || !P || !capacity || !binning || !binning_bytes || !counters || !host_set || !blocks)
    return GS_E_ARG;
  if (set_bytes < gs_multi_depth_sort_bytes(n)) return GS_E_WORKSPACE;
  std::vector<SortSeg> segs((size_t)n);
  for (int i = 0; i < n; ++i) {
    const gs_frame_t* f = &frames[i];
    if (check_frame(f) != GS_OK || f->binning != GS_BINNING_DEPTH_FIRST || P[i] <= 0 || capacity[i] <= 0 ||
        capacity[i] > 0x7fffffffLL || P[i] > kSegMaxKeys || !binning[i] || !counters[i])
      return GS_E_ARG;
    gs_binning_layout_t LB;
    if (gs_binning_layout(capacity[i], P[i], f->width, f->height, f->binning, &LB) != GS_OK) return GS_E_ARG;
    if (binning_bytes[i] < LB.total) return GS_E_WORKSPACE;
    char* bb = (char*)binning[i];
    segs[i] = SortSeg{(uint32_t*)(bb + LB.dkeys_a), (uint32_t*)(bb + LB.dvals_a), (uint32_t*)(bb + LB.dkeys_b),
                      (uint32_t*)(bb + LB.dvals_b), nullptr, (long long)P[i], bb + LB.hist, 0, 32,
                      nullptr};
  }
  unsigned per[kSegMaxPasses];
  int passes = 0;
  if (!seg_sort_build(n, segs.data(), host_set, set_bytes, per, &passes)) return GS_E_ARG;
  *blocks = per[0];  // every frame runs all four passes
  return GS_OK;
}

extern "C" int gs_multi_depth_sort(int n, const void* dev_set, unsigned blocks, void* stream) {
  if (n <= 0 || !dev_set || blocks == 0) return GS_E_ARG;
  hipStream_t s = (hipStream_t)stream;
  timing::Scope ts(timing::kSort, s);
  const unsigned per[kSegMaxPasses] = {blocks, blocks, blocks, blocks};
  static_assert(kSegMaxPasses == 4, "the depth sort runs four 8-bit passes");
  return seg_sort_launch(n, dev_set, per, true, s) == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

extern "C" int gs_render_binning_duplicate(const gs_frame_t* f, int P, const void* geom, uint32_t* counters,
                                           long long capacity, void* binning, size_t binning_bytes, void* image,
                                           size_t image_bytes, void* stream) {
  return render_binning(f, P, geom, counters, capacity, binning, binning_bytes, image, image_bytes,
                        (hipStream_t)stream, kDup);
}

extern "C" size_t gs_multi_list_sort_bytes(int n) { return seg_sort_desc_bytes(n, kSegMaxPasses); }

extern "C" int gs_multi_list_sort_build(int n, const gs_frame_t* frames, const int* P, const long long* capacity,
                                        void* const* binning, const size_t* binning_bytes,
                                        uint32_t* const* counters, void* const* image, void* host_set,
                                        size_t set_bytes, unsigned* blocks) {
  if (n <= 0 || !frames || !P || !capacity || !binning || !binning_bytes || !counters || !image || !host_set ||
      !blocks)
    return GS_E_ARG;
  if (set_bytes < gs_multi_list_sort_bytes(n)) return GS_E_WORKSPACE;
  std::vector<SortSeg> segs((size_t)n);
  for (int i = 0; i < n; ++i) {
    const gs_frame_t* f = &frames[i];
    if (check_frame(f) != GS_OK || f->binning != GS_BINNING_DEPTH_FIRST || P[i] <= 0 || capacity[i] <= 0 ||
        capacity[i] > kSegMaxKeys || !binning[i] || !counters[i] || !image[i])
      return GS_E_ARG;
    gs_binning_layout_t LB;
    gs_image_layout_t LI;
    if (gs_binning_layout(capacity[i], P[i], f->width, f->height, f->binning, &LB) != GS_OK) return GS_E_ARG;
    if (!LB.id_bits) return GS_E_ARG;  // the shared list sort takes one-word entries only
    if (binning_bytes[i] < LB.total) return GS_E_WORKSPACE;
    gs_image_layout(f->width, f->height, &LI);
    int gx, gy;
    const int nt = grid_tiles(f->width, f->height, gx, gy);
    const int tb = bits_for((uint32_t)nt) > 0 ? bits_for((uint32_t)nt) : 1;
    char* bb = (char*)binning[i];
    segs[i] = SortSeg{(uint32_t*)(bb + LB.keys_dup), nullptr, (uint32_t*)(bb + LB.keys_alt), nullptr, counters[i],
                      capacity[i], bb + LB.hist, LB.id_bits, LB.id_bits + tb,
                      (uint32_t*)((char*)image[i] + LI.ranges)};
  }
  int passes = 0;
  return seg_sort_build(n, segs.data(), host_set, set_bytes, blocks, &passes) ? GS_OK : GS_E_ARG;
}

extern "C" int gs_multi_list_sort(int n, const void* dev_set, const unsigned* blocks, void* stream) {
  if (n <= 0 || !dev_set || !blocks || blocks[0] == 0) return GS_E_ARG;
  hipStream_t s = (hipStream_t)stream;
  timing::Scope ts(timing::kSort, s);
  return seg_sort_launch(n, dev_set, blocks, false, s) == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

extern "C" int gs_render_binning_after_list_sort(const gs_frame_t* f, int P, const void* geom, uint32_t* counters,
                                                 long long capacity, void* binning, size_t binning_bytes,
                                                 void* image, size_t image_bytes, void* stream) {
  return render_binning(f, P, geom, counters, capacity, binning, binning_bytes, image, image_bytes,
                        (hipStream_t)stream, kTail);
}

extern "C" int gs_render_after_list_sort(const gs_frame_t* f, int P, const void* geom, uint32_t* counters,
                                         long long capacity, void* binning, size_t binning_bytes, void* image,
                                         size_t image_bytes, float* out_color, float* out_depth, float* out_alpha,
                                         void* stream) {
  return render_blend_from(kTail, f, P, geom, counters, capacity, binning, binning_bytes, image, image_bytes,
                           out_color, out_depth, out_alpha, (hipStream_t)stream);
}

// ---- many frames in one blend launch --------------------------------------
// Set layout: uint32 prefix[n + 1] of tiles per frame, then BlendArgs[n] at a
// 256-byte boundary.
static size_t multi_blend_args_offset(int n) { return align_up(sizeof(uint32_t) * (size_t)(n + 1), 256); }

extern "C" size_t gs_multi_blend_bytes(int n) {
  return n <= 0 ? 0 : multi_blend_args_offset(n) + sizeof(BlendArgs) * (size_t)n;
}

extern "C" int gs_multi_blend_build(int n, const gs_frame_t* frames, const int* P, const void* const* geom,
                                    const long long* capacity, void* const* binning, void* const* image,
                                    float* const* out_color, float* const* out_depth, float* const* out_alpha,
                                    void* host_set, size_t set_bytes, unsigned* total_tiles) {
  if (n <= 0 || !frames || !P || !geom || !capacity || !binning || !image || !out_color || !out_depth || !host_set ||
      !total_tiles)
    return GS_E_ARG;
  if (set_bytes < gs_multi_blend_bytes(n)) return GS_E_WORKSPACE;
  uint32_t* prefix = (uint32_t*)host_set;
  BlendArgs* args = (BlendArgs*)((char*)host_set + multi_blend_args_offset(n));
  unsigned long long total = 0;
  for (int i = 0; i < n; ++i) {
    if (check_frame(&frames[i]) != GS_OK || P[i] < 0 || !image[i] || !out_color[i] || !out_depth[i]) return GS_E_ARG;
    if (capacity[i] < 0 || capacity[i] > 0x7fffffffLL || (P[i] > 0 && !geom[i]) || (capacity[i] > 0 && !binning[i]))
      return GS_E_ARG;
    int gx, gy;
    const int nt = grid_tiles(frames[i].width, frames[i].height, gx, gy);
    prefix[i] = (uint32_t)total;
    total += (unsigned long long)nt;
    if (total > 0x7fffffffULL) return GS_E_ARG;
    args[i] = make_blend_args(&frames[i], P[i], geom[i], capacity[i], binning[i], image[i], out_color[i],
                              out_depth[i], out_alpha ? out_alpha[i] : nullptr);
  }
  prefix[n] = (uint32_t)total;
  *total_tiles = (unsigned)total;
  return GS_OK;
}

extern "C" int gs_multi_blend(int n, const void* dev_set, unsigned total_tiles, void* stream) {
  if (n <= 0 || !dev_set || total_tiles == 0) return GS_E_ARG;
  hipStream_t s = (hipStream_t)stream;
  const uint32_t* prefix = (const uint32_t*)dev_set;
  const BlendArgs* args = (const BlendArgs*)((const char*)dev_set + multi_blend_args_offset(n));
  {
    timing::Scope ts(timing::kBlend, s);
    if (total_tiles <= (unsigned)kCellTiles)
      hipLaunchKernelGGL(k_blend_multi<4>, dim3(blend_grid(total_tiles, 4)), dim3(64), 0, s, prefix, args, n);
    else
      hipLaunchKernelGGL(k_blend_multi<1>, dim3(blend_grid(total_tiles, 1)), dim3(64), 0, s, prefix, args, n);
  }
  return hipGetLastError() == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

extern "C" int gs_mark_visible(const float* means3D, int P, const float* viewmatrix, const float* projmatrix,
                               uint8_t* visible, void* stream) {
  (void)projmatrix;
  if (P < 0 || (P > 0 && (!means3D || !viewmatrix || !visible))) return GS_E_ARG;
  if (P == 0) return GS_OK;
  hipLaunchKernelGGL(k_mark_visible, dim3(nblocks256(P)), dim3(256), 0, (hipStream_t)stream, means3D, P,
                     viewmatrix, visible);
  return hipGetLastError() == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

extern "C" const char* gs_error_string(int code) {
  switch (code) {
    case GS_OK: return "ok";
    case GS_E_ARG: return "invalid argument";
    case GS_E_WORKSPACE: return "workspace too small";
    case GS_E_LAUNCH: return "kernel launch failed";
    case GS_E_STATIC_LIMIT: return "input larger than the entry point's static scratch allows";
    case GS_E_SCRATCH: return "static scratch address lookup failed";
    default: return "unknown error";
  }
}

extern "C" int gs_abi_version(void) { return 4; }
