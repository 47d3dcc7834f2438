// gs_knn.hip -- exact mean squared distance to the 3 nearest other points
// (the quantity simple_knn's distCUDA2 returns; used for the initial scales
// at scene/gaussian_model_cf.py:194-196).
//
// The points are put in order along a Hilbert curve and searched through a
// hierarchy of bounding boxes 64 wide, all on the device (the host never sees
// the bounding box):
//   k_knn_bbox      bounding box of the points, one partial per workgroup
//   k_knn_keys      each point's place on the curve
//   radix sort      gs_sort.hip
//   k_knn_gather    points in curve order, boxes of every 16 (a leaf), 1024 and
//                   65536 consecutive points
//   k_knn_query     one wave per 64 consecutive points
// A subtree is skipped when its box is no nearer than the 3rd best so far.  The
// box distance takes the same operations in the same order as a point's, each
// of them monotonic under rounding, so it is never above the computed distance
// of a point in the box, and the result equals a brute-force search bit for
// bit.  The three best squared distances are kept sorted and summed smallest
// first, ((b0 + b1) + b2) / 3, so the value is independent of visit order.
//
// A uniform grid with a thread per point, which this replaces, adapts to the
// bounding box alone: the points of a lifted frame lie on a surface and those
// of a scene in clusters, 20 to 100 to an occupied cell, and a thread read 27
// cells of them while the wave waited for its point in the emptiest place.
#include <float.h>

#include <mutex>

#include "gs_common.hpp"
#include "gs_internal.hpp"

namespace gs {

constexpr int kKnnLeaf = 16, kKnnFan = 64;  // points of a leaf, children of a node
constexpr int kKnnParts = 256;  // workgroups of the bounding box

struct KnnLayout {
  size_t partial, keys_a, keys_b, vals_a, vals_b, sorted, hist, leaves, nodes, tops, total;
  long long n_leaf, n_node, n_top;
  int bits;  // of the curve, per axis
};

constexpr KnnLayout knn_layout(int P) {
  KnnLayout L{};
  const long long padded = ((long long)P + 63) / 64 * 64;
  L.n_leaf = padded / kKnnLeaf;
  L.n_node = (L.n_leaf + kKnnFan - 1) / kKnnFan;
  L.n_top = (L.n_node + kKnnFan - 1) / kKnnFan;
  // 3 sort passes or 4: a curve of 2^8 cells a side tells the points of a
  // surface or of a few clusters apart up to about this many of them
  L.bits = P <= (1 << 18) ? 8 : 10;
  size_t o = 0;
  L.partial = o;
  o = align_up(o + 24 * (size_t)kKnnParts, 256);
  // the gathered points take the place of three of the sort's four buffers
  // and of the fourth's size beyond; the sorted indices stay out of it
  const size_t n4 = align_up(4 * (size_t)padded, 256);
  const bool in_b = sort_passes(3 * L.bits) & 1;
  L.sorted = o;
  L.keys_a = o;
  L.keys_b = o + n4;
  const size_t spare = o + 2 * n4;
  o += 4 * n4;
  L.vals_a = in_b ? spare : o;
  L.vals_b = in_b ? o : spare;
  o += n4;
  L.hist = o;
  o = align_up(o + sort_tmp_bytes(P), 256);
  L.leaves = o;
  o = align_up(o + 32 * (size_t)L.n_leaf, 256);
  L.nodes = o;
  o = align_up(o + 32 * (size_t)L.n_node, 256);
  L.tops = o;
  o = align_up(o + 24 * (size_t)L.n_top, 256);
  L.total = o;
  return L;
}

__device__ __forceinline__ float inf_f() { return __builtin_inff(); }

// Minimum of lo[3] and maximum of hi[3] over the 16 lanes of each row.
__device__ __forceinline__ void row_box(float (&lo)[3], float (&hi)[3]) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    lo[k] = fminf(lo[k], dpp<0xB1>(lo[k]));
    lo[k] = fminf(lo[k], dpp<0x4E>(lo[k]));
    lo[k] = fminf(lo[k], dpp<0x141>(lo[k]));
    lo[k] = fminf(lo[k], dpp<0x140>(lo[k]));
    hi[k] = fmaxf(hi[k], dpp<0xB1>(hi[k]));
    hi[k] = fmaxf(hi[k], dpp<0x4E>(hi[k]));
    hi[k] = fmaxf(hi[k], dpp<0x141>(hi[k]));
    hi[k] = fmaxf(hi[k], dpp<0x140>(hi[k]));
  }
}

// The box over the whole workgroup, in every thread; s: 6 words per row of 16.
template <int NT>
__device__ __forceinline__ void block_box(float (&lo)[3], float (&hi)[3], float (*s)[6]) {
  row_box(lo, hi);
  if ((threadIdx.x & 15) == 0)
    for (int k = 0; k < 3; ++k) {
      s[threadIdx.x >> 4][k] = lo[k];
      s[threadIdx.x >> 4][3 + k] = hi[k];
    }
  __syncthreads();
  for (int r = 0; r < NT / 16; ++r)
    for (int k = 0; k < 3; ++k) {
      lo[k] = fminf(lo[k], s[r][k]);
      hi[k] = fmaxf(hi[k], s[r][3 + k]);
    }
}

// A point with a coordinate that is not finite has no neighbour and is nobody's.
__device__ __forceinline__ bool finite3(float x, float y, float z) {
  return fabsf(x) < inf_f() && fabsf(y) < inf_f() && fabsf(z) < inf_f();
}

__global__ __launch_bounds__(256) void k_knn_bbox(const float* pts, int P, float* partial) {
  __shared__ float s[16][6];
  float lo[3] = {inf_f(), inf_f(), inf_f()}, hi[3] = {-inf_f(), -inf_f(), -inf_f()};
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < P; i += (long long)gridDim.x * 256) {
    const float v[3] = {pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]};
    if (finite3(v[0], v[1], v[2]))
      for (int k = 0; k < 3; ++k) {
        lo[k] = fminf(lo[k], v[k]);
        hi[k] = fmaxf(hi[k], v[k]);
      }
  }
  block_box<256>(lo, hi, s);
  if (threadIdx.x == 0)
    for (int k = 0; k < 3; ++k) {
      partial[6 * blockIdx.x + k] = lo[k];
      partial[6 * blockIdx.x + 3 + k] = hi[k];
    }
}

// Place on the Hilbert curve through the 2^bits cells a side (J. Skilling,
// Programming the Hilbert curve, AIP Conf. Proc. 707, 2004): the axes are
// turned into the transposed index from the top bit down, Gray-coded, and
// their bits interleaved.
__device__ __forceinline__ uint32_t hilbert(uint32_t x, uint32_t y, uint32_t z, int bits) {
  uint32_t ax[3] = {x, y, z};
  for (int b = bits - 1; b > 0; --b) {
    const uint32_t low = (1u << b) - 1u;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const uint32_t t = (ax[0] ^ ax[i]) & low;
      const bool on = (ax[i] >> b) & 1u;
      ax[0] ^= on ? low : t;
      ax[i] ^= on ? 0u : t;
    }
  }
  ax[1] ^= ax[0];
  ax[2] ^= ax[1];
  uint32_t flip = 0;
  for (int b = bits - 1; b > 0; --b) flip ^= (ax[2] >> b) & 1u ? (1u << b) - 1u : 0u;
  uint32_t key = 0;
  for (int b = bits - 1; b >= 0; --b)
#pragma unroll
    for (int i = 0; i < 3; ++i) key = key << 1 | (((ax[i] ^ flip) >> b) & 1u);
  return key;
}

// floats as unsigned integers of the same order
__device__ __forceinline__ uint32_t ordered(float v) {
  const uint32_t u = __float_as_uint(v);
  return u ^ (u >> 31 ? 0xffffffffu : 0x80000000u);
}
__device__ __forceinline__ float from_ordered(uint32_t u) {
  return __uint_as_float(u ^ (u >> 31 ? 0x80000000u : 0xffffffffu));
}

__global__ __launch_bounds__(256) void k_knn_keys(const float* pts, int P, const float* partial, int parts, int bits,
                                                  uint32_t* keys, uint32_t* vals, uint32_t* tops, int n_top) {
  __shared__ float s[16][6];
  float lo[3] = {inf_f(), inf_f(), inf_f()}, hi[3] = {-inf_f(), -inf_f(), -inf_f()};
  if ((int)threadIdx.x < parts)
    for (int k = 0; k < 3; ++k) {
      lo[k] = partial[6 * threadIdx.x + k];
      hi[k] = partial[6 * threadIdx.x + 3 + k];
    }
  block_box<256>(lo, hi, s);
  // cubic cells; any scale gives a right result (0 * inf is cell 0)
  const float side = fmaxf(hi[0] - lo[0], fmaxf(hi[1] - lo[1], hi[2] - lo[2]));
  const float scale = side > 0.0f ? (float)(1 << bits) / side : 0.0f;
  const int i = blockIdx.x * 256 + threadIdx.x;
  for (int t = i; t < 6 * n_top; t += gridDim.x * 256) tops[t] = ordered(t % 6 < 3 ? inf_f() : -inf_f());
  if (i >= P) return;
  uint32_t c[3];
  for (int k = 0; k < 3; ++k) c[k] = (uint32_t)min(max(sat_i((pts[3 * (size_t)i + k] - lo[k]) * scale), 0), (1 << bits) - 1);
  keys[i] = hilbert(c[0], c[1], c[2], bits);
  vals[i] = (uint32_t)i;
}

// Workgroup b: the points of node b.  Places past the last point, and points
// with a coordinate that is not finite, are at infinity and in no box.
__global__ __launch_bounds__(1024) void k_knn_gather(const float* pts, int P, const uint32_t* vals, float4* sorted,
                                                     float4* leaves, float4* nodes, uint32_t* tops) {
  __shared__ float s[64][6];
  const uint32_t k = blockIdx.x * 1024u + threadIdx.x;
  float4 p = make_float4(inf_f(), inf_f(), inf_f(), __int_as_float(-1));
  float lo[3] = {inf_f(), inf_f(), inf_f()}, hi[3] = {-inf_f(), -inf_f(), -inf_f()};
  if (k < (uint32_t)P) {
    const uint32_t i = vals[k];
    const float v[3] = {pts[3 * (size_t)i], pts[3 * (size_t)i + 1], pts[3 * (size_t)i + 2]};
    p.w = __int_as_float((int)i);
    if (finite3(v[0], v[1], v[2])) {
      p.x = v[0];
      p.y = v[1];
      p.z = v[2];
      for (int c = 0; c < 3; ++c) lo[c] = hi[c] = v[c];
    }
  }
  if (k < ((uint32_t)P + 63u) / 64u * 64u) sorted[k] = p;
  row_box(lo, hi);
  if ((threadIdx.x & 15) == 0) {
    if (k < ((uint32_t)P + 63u) / 64u * 64u) {
      leaves[2 * (k / kKnnLeaf)] = make_float4(lo[0], lo[1], lo[2], 0.0f);
      leaves[2 * (k / kKnnLeaf) + 1] = make_float4(hi[0], hi[1], hi[2], 0.0f);
    }
    for (int c = 0; c < 3; ++c) {
      s[threadIdx.x >> 4][c] = lo[c];
      s[threadIdx.x >> 4][3 + c] = hi[c];
    }
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  for (int c = 0; c < 3; ++c) {
    lo[c] = s[threadIdx.x][c];
    hi[c] = s[threadIdx.x][3 + c];
    for (int off = 32; off > 0; off >>= 1) {
      lo[c] = fminf(lo[c], __shfl_xor(lo[c], off, 64));
      hi[c] = fmaxf(hi[c], __shfl_xor(hi[c], off, 64));
    }
  }
  if (threadIdx.x == 0) {
    nodes[2 * blockIdx.x] = make_float4(lo[0], lo[1], lo[2], 0.0f);
    nodes[2 * blockIdx.x + 1] = make_float4(hi[0], hi[1], hi[2], 0.0f);
    for (int c = 0; c < 3; ++c) {
      atomicMin(&tops[6 * (blockIdx.x / kKnnFan) + c], ordered(lo[c]));
      atomicMax(&tops[6 * (blockIdx.x / kKnnFan) + 3 + c], ordered(hi[c]));
    }
  }
}

__device__ __forceinline__ float lane_of(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Squared distance between the boxes [alo, ahi] and [blo, bhi] (a point is a
// box too), never above that of any two points in them as the search forms it.
__device__ __forceinline__ float box_d2(float alx, float aly, float alz, float ahx, float ahy, float ahz, float blx,
                                        float bly, float blz, float bhx, float bhy, float bhz) {
  const float dx = fmaxf(fmaxf(blx - ahx, alx - bhx), 0.0f), dy = fmaxf(fmaxf(bly - ahy, aly - bhy), 0.0f),
              dz = fmaxf(fmaxf(blz - ahz, alz - bhz), 0.0f);
  return (dx * dx + dy * dy) + dz * dz;
}

// One wave per 64 consecutive points of the curve, a point a lane.  Lane i
// tests the i-th child box of a node against the boxes of the wave's four
// leaves and the largest 3rd best of each; a child that passes is tested by
// every lane against its own point and 3rd best, and a leaf that passes that
// is tried point by point: its points are the same for all lanes, so they
// come through the scalar cache, and a try costs 8 instructions for the
// distance and 3 to keep the best three in order.  No lane waits for another
// one's walk, and the leaves a wave visits follow the local density.
// 129 600 points of a lifted frame: 381 us with the grid, 78 now, the longest
// wave's walk (50 leaves where the average is 19); 2 000 000 in 32 clusters: 4010
// and 534, two thirds of it instruction issue (a wave tries 39 leaves, and about
// 5 of its lanes need each).  Leaves of 8 points are no faster (91 and 551): fewer
// tries, more tests and node visits; nor is a list per row of 16 lanes.
__global__ __launch_bounds__(256) void k_knn_query(int n_group, int n_leaf, int n_node, int n_top,
                                                   const float4* __restrict__ sorted,
                                                   const float4* __restrict__ leaves,
                                                   const float4* __restrict__ nodes,
                                                   const uint32_t* __restrict__ tops, float* __restrict__ out) {
  const int g = __builtin_amdgcn_readfirstlane((int)(xcd_remap(blockIdx.x, gridDim.x) * 4u + (threadIdx.x >> 6)));
  if (g >= n_group) return;
  const int lane = threadIdx.x & 63;
  const float4 me = sorted[64 * (size_t)g + lane];
  const bool ok = me.x < inf_f();
  float b0 = FLT_MAX, b1 = FLT_MAX, b2 = FLT_MAX;
  auto consider = [&](float x, float y, float z, bool self) {
    const float ddx = me.x - x, ddy = me.y - y, ddz = me.z - z;
    float d = (ddx * ddx + ddy * ddy) + ddz * ddz;
    if (self) d = inf_f();
    // b0 <= b1 <= b2; d is not NaN for a lane whose result counts
    b2 = __builtin_amdgcn_fmed3f(b1, b2, d);
    b1 = __builtin_amdgcn_fmed3f(b0, b1, d);
    b0 = fminf(b0, d);
  };
#pragma unroll 8
  for (int j = 0; j < 64; ++j) {
    const float4 o = sorted[64 * (size_t)g + j];
    consider(o.x, o.y, o.z, j == lane);
  }
  // the wave's leaves: boxes and the bound of each, the same in all lanes
  float rl[4][3], rh[4][3], rb[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float4 l = leaves[2 * (4 * (size_t)g + r)], h = leaves[2 * (4 * (size_t)g + r) + 1];
    rl[r][0] = l.x, rl[r][1] = l.y, rl[r][2] = l.z;
    rh[r][0] = h.x, rh[r][1] = h.y, rh[r][2] = h.z;
  }
  auto bounds = [&] {
    float m = ok ? b2 : -1.0f;
    m = fmaxf(m, dpp<0xB1>(m));
    m = fmaxf(m, dpp<0x4E>(m));
    m = fmaxf(m, dpp<0x141>(m));
    m = fmaxf(m, dpp<0x140>(m));
#pragma unroll
    for (int r = 0; r < 4; ++r) rb[r] = lane_of(m, 16 * r);
  };
  auto near_wave = [&](const float4& l, const float4& h) {
    bool hit = false;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      hit |= box_d2(rl[r][0], rl[r][1], rl[r][2], rh[r][0], rh[r][1], rh[r][2], l.x, l.y, l.z, h.x, h.y, h.z) < rb[r];
    return hit;
  };
  // whether any lane's point is near child i, whose box lane i holds
  auto near_lane = [&](const float4& l, const float4& h, int i) {
    const float d = box_d2(me.x, me.y, me.z, me.x, me.y, me.z, lane_of(l.x, i), lane_of(l.y, i), lane_of(l.z, i),
                           lane_of(h.x, i), lane_of(h.y, i), lane_of(h.z, i));
    return __ballot(ok && d < b2) != 0;
  };
  auto node = [&](int c, uint64_t mask) {
    const int first = c * kKnnFan;
    const bool have = first + lane < n_leaf;
    const float4 l = leaves[2 * (size_t)(have ? first + lane : 0)], h = leaves[2 * (size_t)(have ? first + lane : 0) + 1];
    uint64_t m = __ballot(have && near_wave(l, h)) & mask;
    const bool any = m != 0;
    while (m) {
      const int i = __builtin_ctzll(m);
      m &= m - 1;
      if (!near_lane(l, h, i)) continue;
      const float4* o = sorted + (size_t)(first + i) * kKnnLeaf;
#pragma unroll
      for (int j = 0; j < kKnnLeaf; ++j) consider(o[j].x, o[j].y, o[j].z, false);
    }
    if (any) bounds();
  };
  bounds();
  // the wave's own node first, the leaves next to its own before the others
  const int own = g / 16, at = 4 * (g % 16);
  const uint64_t mine = 0xfull << at;
  const uint64_t next = (at >= 4 ? mine >> 4 : 0ull) | (at + 4 < 64 ? mine << 4 : 0ull);
  node(own, next);
  node(own, ~(mine | next));
  for (int t0 = 0; t0 < n_top; t0 += 64) {
    const bool have_t = t0 + lane < n_top;
    const uint32_t* t = tops + 6 * (size_t)(have_t ? t0 + lane : 0);
    const float4 tl = make_float4(from_ordered(t[0]), from_ordered(t[1]), from_ordered(t[2]), 0.0f);
    const float4 th = make_float4(from_ordered(t[3]), from_ordered(t[4]), from_ordered(t[5]), 0.0f);
    uint64_t mt = __ballot(have_t && near_wave(tl, th));
    while (mt) {
      const int ti = __builtin_ctzll(mt);
      mt &= mt - 1;
      if (!near_lane(tl, th, ti)) continue;
      const int c0 = (t0 + ti) * kKnnFan;
      const bool have = c0 + lane < n_node;
      const float4 l = nodes[2 * (size_t)(have ? c0 + lane : 0)], h = nodes[2 * (size_t)(have ? c0 + lane : 0) + 1];
      uint64_t m = __ballot(have && c0 + lane != own && near_wave(l, h));
      while (m) {
        const int i = __builtin_ctzll(m);
        m &= m - 1;
        if (near_lane(l, h, i)) node(c0 + i, ~0ull);
      }
    }
  }
  const int idx = __float_as_int(me.w);
  if (idx >= 0) out[idx] = ok ? ((b0 + b1) + b2) / 3.0f : inf_f();
}

// The launch sequence over a workspace laid out by knn_layout(P).
static int knn_launch(const float* points, int P, float* out, char* b, const KnnLayout& L, hipStream_t s) {
  float* partial = (float*)(b + L.partial);
  uint32_t *ka = (uint32_t*)(b + L.keys_a), *kb = (uint32_t*)(b + L.keys_b);
  uint32_t *va = (uint32_t*)(b + L.vals_a), *vb = (uint32_t*)(b + L.vals_b);
  float4* sorted = (float4*)(b + L.sorted);
  float4 *leaves = (float4*)(b + L.leaves), *nodes = (float4*)(b + L.nodes);
  uint32_t* tops = (uint32_t*)(b + L.tops);
  const int nb = (P + 255) / 256, parts = nb < kKnnParts ? nb : kKnnParts, n_group = (P + 63) / 64;
  timing::Scope ts(timing::kKnn, s);
  hipLaunchKernelGGL(k_knn_bbox, dim3(parts), dim3(256), 0, s, points, P, partial);
  hipLaunchKernelGGL(k_knn_keys, dim3(nb), dim3(256), 0, s, points, P, partial, parts, L.bits, ka, va, tops,
                     (int)L.n_top);
  int in_b;
  if (sort_pairs_u32(ka, va, kb, vb, nullptr, P, 3 * L.bits, b + L.hist, s, &in_b) != hipSuccess) return GS_E_LAUNCH;
  hipLaunchKernelGGL(k_knn_gather, dim3((unsigned)L.n_node), dim3(1024), 0, s, points, P, in_b ? vb : va, sorted,
                     leaves, nodes, tops);
  hipLaunchKernelGGL(k_knn_query, dim3((n_group + 3) / 4), dim3(256), 0, s, n_group, (int)L.n_leaf, (int)L.n_node,
                     (int)L.n_top, sorted, leaves, nodes, tops, out);
  return hipGetLastError() == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

}  // namespace gs

using namespace gs;

// Scratch of gs_knn3_meandist_static: the whole workspace of
// gs_knn3_meandist for GS_KNN_STATIC_MAX_POINTS points (about 24 MiB).  Every
// GPU the library runs on holds its own copy until the process ends.  Host
// code never passes this name to a kernel: it is a host-side stand-in, and
// the device address comes from hipGetSymbolAddress (knn_static_scratch).
static __device__ __align__(256) unsigned char scratch[knn_layout(GS_KNN_STATIC_MAX_POINTS).total];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on the current device, looked up on the
// first call on that device and kept.  nullptr when the lookup fails.
void* knn_static_scratch() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
    g_scratch_ptr[dev] = p;
  }
  return g_scratch_ptr[dev];
}
}  // namespace

extern "C" size_t gs_knn_workspace_bytes(int P) { return knn_layout(P < 0 ? 0 : P).total; }

extern "C" int gs_knn3_meandist(const float* points, int P, float* out, void* ws, size_t ws_bytes, void* stream) {
  if (P < 0 || (P > 0 && (!points || !out || !ws))) return GS_E_ARG;
  if (P == 0) return GS_OK;
  const KnnLayout L = knn_layout(P);
  if (ws_bytes < L.total) return GS_E_WORKSPACE;
  return knn_launch(points, P, out, (char*)ws, L, (hipStream_t)stream);
}

extern "C" int gs_knn3_meandist_static(const float* points, int P, float* out, void* stream) {
  if (P < 0 || (P > 0 && (!points || !out))) return GS_E_ARG;
  if (P > GS_KNN_STATIC_MAX_POINTS) return GS_E_STATIC_LIMIT;
  if (P == 0) return GS_OK;
  void* ws = knn_static_scratch();
  if (!ws) return GS_E_SCRATCH;
  return knn_launch(points, P, out, (char*)ws, knn_layout(P), (hipStream_t)stream);
}
