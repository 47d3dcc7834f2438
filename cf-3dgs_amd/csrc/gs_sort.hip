// gs_sort.hip -- stable LSD radix sort of (key, uint32 value) pairs, with
// 64-bit keys (tile << 32 | depth bits, the reference's key) or 32-bit keys
// (depth bits, or tile ids in the depth-first binning).
//
// The element count is read on the device (so the binning pipeline never
// needs the host to know num_rendered); grids are sized by capacity and
// workgroups past the count exit at once.
//
// Keys-only sorts (32-bit keys that carry their payload in the low bits)
// sort bits [start_bit, end_bit) and skip every value load and store.
//
// A sort of B bits takes ceil(B / 8) passes of near equal digits; a keys-only
// sort of 9 or 10 bits (the lists of up to 1024 tiles) takes one pass.  Per pass:
//   k_sort_upsweep  1024 or 2048 keys per workgroup (4096 with 10-bit digits and
//                   past 2^24 keys), 4 waves x 4, 8 or 16 rounds x 64 lanes, all loaded up
//                   front, counted with one LDS atomic each -> per-workgroup
//                   digit counts
//   k_sort_scan     one workgroup per digit: exclusive scan of its row, total.
//                   Sorts of up to kDirectBlocks workgroups have no such
//                   launch (kSegDirectBlocks in a segmented sort): each
//                   scatter workgroup adds the counts up itself
//   k_sort_scatter  recomputes the matches; rank = prior count of the digit in
//                   this wave + lanes below with the same digit; waves are
//                   ordered by an exclusive prefix over the 4 wave counts, so
//                   the order of equal digits is the input order (stable).
//                   The workgroup's keys are first placed in LDS in digit
//                   order, then written out by consecutive threads: each
//                   digit's run leaves as contiguous stores instead of one
//                   scattered 4-byte store per lane.
// Short sorts are bound by the chain of launches and of loads in each.  One pass
// instead of two for 510 tiles: 28 us of kernels -> 22 (137 000 entries).  Long ones
// are bound by memory: 71 million (key, value) pairs of 13 bits took 386 us a
// scatter with digits of 8 and 5 bits over 2048 keys, where a digit's run in a
// workgroup is 32 bytes and the counts as much again; with 7 and 6 bits over 4096
// keys 275, 4.1 TB/s.
// Upsweep and scatter map workgroups to key blocks XCD-aware (xcd_remap):
// dispatch deals workgroups round-robin over the 8 XCDs, and each XCD gets a
// contiguous run of blocks.  A cache line of a digit's counts covers 32
// consecutive blocks, so it is then written and read within one XCD's L2
// instead of once by each of the eight.
#include "gs_common.hpp"
#include "gs_internal.hpp"

#include <algorithm>

namespace gs {

// Lanes whose digit equals this lane's digit (only lanes with valid set).
__device__ __forceinline__ uint64_t match_digit(uint32_t d, bool valid, int bits) {
  uint64_t m = __ballot(valid);
  for (int b = 0; b < bits; ++b) {
    const bool on = (d >> b) & 1u;
    const uint64_t v = __ballot(on);
    m &= on ? v : ~v;
  }
  return m;
}

// Inclusive prefix sum over a 256-thread workgroup (thread t holds v); the
// workgroup total in `total`.  Each wave scans by shuffles, then one barrier
// combines the four wave totals (instead of a barrier pair per Hillis-Steele
// step).  s_w (4 words of LDS) may be rewritten only after a later barrier.
__device__ __forceinline__ uint32_t block_incl_scan256(uint32_t v, uint32_t* s_w, uint32_t& total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) s_w[w] = x;
  __syncthreads();
  const uint32_t w0 = s_w[0], w1 = s_w[1], w2 = s_w[2], w3 = s_w[3];
  total = (w0 + w1) + (w2 + w3);
  return x + (w > 0 ? w0 : 0u) + (w > 1 ? w1 : 0u) + (w > 2 ? w2 : 0u);
}

// The element count: *n_dev, 0 past the capacity; the capacity without n_dev.
__device__ __forceinline__ uint32_t n_eff(const uint32_t* n_dev, long long cap) {
  if (!n_dev) return (uint32_t)cap;
  const uint32_t n = *n_dev;
  return ((long long)n > cap) ? 0u : n;
}

// Workgroup `bid` of an upsweep over one key array (the kernels below pass
// their block index, or, in a segmented sort, the block index within the
// segment).
template <typename K, int ITEMS, int R>
__device__ __forceinline__ void upsweep_block(const K* __restrict__ keys, const uint32_t* n_dev, long long cap,
                                              int shift, int bits, uint32_t* hist, int nb_max, bool direct,
                                              uint32_t bid) {
  __shared__ uint32_t s_h[4][R];
  const uint32_t n = n_eff(n_dev, cap);
  constexpr uint32_t TILE = kSortThreads * ITEMS;
  const uint32_t nblk = (n + TILE - 1) / TILE;
  if (bid >= nblk) return;
  const uint32_t blk = xcd_remap(bid, nblk);  // consecutive blocks on one XCD (see the file comment)
  const uint32_t start = blk * TILE;
  for (int k = threadIdx.x; k < 4 * R; k += kSortThreads) (&s_h[0][0])[k] = 0;
  __syncthreads();
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint32_t mask = (1u << bits) - 1u;
  const uint32_t wbase = start + (uint32_t)w * (ITEMS * 64);
  // a histogram needs no ranks: one LDS atomic per key into the wave's own
  // row, with every key of the thread loaded before the first atomic.  Order
  // does not matter here, so 32-bit keys come four to a lane in 16-byte loads
  // (the key arrays are 16-byte aligned).
  if constexpr (sizeof(K) == 4 && ITEMS % 4 == 0) {
    constexpr int V = ITEMS / 4;
    uint4 kv[V];
#pragma unroll
    for (int r = 0; r < V; ++r) {
      const uint32_t idx = wbase + 4u * (uint32_t)(r * 64 + lane);
      kv[r] = idx + 3u < n ? *reinterpret_cast<const uint4*>(keys + idx)
                           : make_uint4(idx < n ? (uint32_t)keys[idx] : 0u, idx + 1u < n ? (uint32_t)keys[idx + 1] : 0u,
                                        idx + 2u < n ? (uint32_t)keys[idx + 2] : 0u, 0u);
    }
    if (bits <= 3) {
      // at most 8 bins (a short top digit): LDS atomics would pile onto a few
      // words, so each lane counts in registers, four 8-bit fields per word
      // (a lane sees at most 4 V <= 16 keys), and the wave adds the counts
      // after widening them to 16-bit fields (a wave sees at most 1024 keys)
      uint32_t lo = 0, hi = 0;
#pragma unroll
      for (int r = 0; r < V; ++r) {
        const uint32_t idx = wbase + 4u * (uint32_t)(r * 64 + lane);
        const uint32_t e[4] = {kv[r].x, kv[r].y, kv[r].z, kv[r].w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint32_t d = (e[c] >> shift) & mask;
          const uint32_t inc = idx + (uint32_t)c < n ? 1u << ((d & 3u) * 8u) : 0u;
          lo += d < 4u ? inc : 0u;
          hi += d < 4u ? 0u : inc;
        }
      }
      // 16-bit fields: w0 = bins (0, 2), w1 = (1, 3), w2 = (4, 6), w3 = (5, 7)
      uint32_t cw[4] = {lo & 0x00ff00ffu, (lo >> 8) & 0x00ff00ffu, hi & 0x00ff00ffu, (hi >> 8) & 0x00ff00ffu};
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
        for (int k = 0; k < 4; ++k) cw[k] += __shfl_xor(cw[k], off, 64);
      }
      if (lane < 8) {
        const int k = (lane >> 2) * 2 + (lane & 1);
        const uint32_t word = k == 0 ? cw[0] : (k == 1 ? cw[1] : (k == 2 ? cw[2] : cw[3]));
        const uint32_t cnt = ((lane >> 1) & 1) ? word >> 16 : word & 0xffffu;
        if ((uint32_t)lane <= mask) s_h[w][lane] = cnt;
      }
    } else if (bits <= 4) {
      // few bins (a top digit): the wave's lanes would pile onto a handful of
      // LDS words, so count each bin with a ballot instead; lane b keeps bin b
      uint32_t cnt = 0;
#pragma unroll
      for (int r = 0; r < V; ++r) {
        const uint32_t idx = wbase + 4u * (uint32_t)(r * 64 + lane);
        const uint32_t e[4] = {kv[r].x, kv[r].y, kv[r].z, kv[r].w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const bool valid = idx + (uint32_t)c < n;
          const uint32_t d = (e[c] >> shift) & mask;
          for (uint32_t b = 0; b <= mask; ++b) {
            const uint32_t m = (uint32_t)__popcll(__ballot(valid && d == b));
            if ((uint32_t)lane == b) cnt += m;
          }
        }
      }
      if ((uint32_t)lane <= mask) s_h[w][lane] = cnt;
    } else {
      // digits of 7, 6 or 5 bits leave room for 2, 4 or 8 counters of each: lanes
      // side by side add to different ones, in different banks (their adds to
      // one word follow each other: 11.4 us an upsweep of the 500 000-Gaussian
      // training scene's lists, 7.4 this way; 85 and 75 for 71M entries)
      const int room = R == 256 ? 8 - bits : 0;
      const uint32_t copy = (uint32_t)lane & ((1u << room) - 1u), at = copy << bits, skew = copy * (mask + 1u) >> room;
#pragma unroll
      for (int r = 0; r < V; ++r) {
        const uint32_t idx = wbase + 4u * (uint32_t)(r * 64 + lane);
        const uint32_t e[4] = {kv[r].x, kv[r].y, kv[r].z, kv[r].w};
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (idx + (uint32_t)c < n) atomicAdd(&s_h[w][at | (((e[c] >> shift) & mask) ^ skew)], 1u);
      }
      if (room > 0) {
        __syncthreads();
        uint32_t sum = 0;
        const int d = threadIdx.x;
        if (d <= (int)mask)
          for (uint32_t q = 0; q < 1u << room; ++q) {
            const uint32_t k = q << bits | ((uint32_t)d ^ (q * (mask + 1u) >> room));
            sum += s_h[0][k] + s_h[1][k] + s_h[2][k] + s_h[3][k];
          }
        if (d <= (int)mask || direct) hist[direct ? (size_t)blk * R + d : (size_t)d * nb_max + blk] = sum;
        return;
      }
    }
  } else {
    K kk[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const uint32_t idx = wbase + r * 64 + lane;
      kk[r] = idx < n ? keys[idx] : (K)0;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const uint32_t idx = wbase + r * 64 + lane;
      if (idx < n) atomicAdd(&s_h[w][(uint32_t)(kk[r] >> shift) & mask], 1u);
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < R; d += kSortThreads)
    hist[direct ? (size_t)blk * R + d : (size_t)d * nb_max + blk] = s_h[0][d] + s_h[1][d] + s_h[2][d] + s_h[3][d];
}

template <typename K, int ITEMS, int R>
__global__ __launch_bounds__(kSortThreads) void k_sort_upsweep(const K* __restrict__ keys, const uint32_t* n_dev,
                                                               long long cap, int shift, int bits, uint32_t* hist,
                                                               int nb_max, bool direct) {
  upsweep_block<K, ITEMS, R>(keys, n_dev, cap, shift, bits, hist, nb_max, direct, blockIdx.x);
}

// One workgroup per digit: exclusive scan over the active blocks' counts.
// Each thread takes kScanRun consecutive counts per round (all loaded before
// any is used) and scans them in registers around one workgroup scan of the
// run sums, so a row of up to 256 * kScanRun blocks costs one workgroup scan.
constexpr int kScanRun = 8;
__device__ __forceinline__ void scan_row(uint32_t* hist, uint32_t* totals, const uint32_t* n_dev, long long cap,
                                         int nb_max, int tile, int d) {
  __shared__ uint32_t s_w[4];
  const uint32_t n = n_eff(n_dev, cap);
  const int nb = (int)((n + tile - 1) / tile);
  uint32_t* row = hist + (size_t)d * nb_max;
  const int t = threadIdx.x;
  uint32_t carry = 0;
  for (int b0 = 0; b0 < nb; b0 += 256 * kScanRun) {
    const int first = b0 + t * kScanRun;
    uint32_t v[kScanRun], sum = 0;
#pragma unroll
    for (int j = 0; j < kScanRun; ++j) v[j] = first + j < nb ? row[first + j] : 0u;
#pragma unroll
    for (int j = 0; j < kScanRun; ++j) sum += v[j];
    uint32_t tot;
    const uint32_t incl = block_incl_scan256(sum, s_w, tot);
    uint32_t run = carry + incl - sum;
#pragma unroll
    for (int j = 0; j < kScanRun; ++j) {
      if (first + j < nb) row[first + j] = run;
      run += v[j];
    }
    carry += tot;
    __syncthreads();  // s_w is rewritten by the next round
  }
  if (t == 0) totals[d] = carry;
}

// The same for 10-bit digits, whose rows are short (at most 512 workgroups): a
// wave a row, four to a workgroup.
__device__ __forceinline__ void scan_row_wide(uint32_t* hist, uint32_t* totals, const uint32_t* n_dev, long long cap,
                                              int nb_max, int tile, int d) {
  const uint32_t n = n_eff(n_dev, cap);
  const int nb = (int)((n + tile - 1) / tile), lane = threadIdx.x & 63;
  uint32_t* row = hist + (size_t)d * nb_max;
  uint32_t carry = 0;
  for (int b0 = 0; b0 < nb; b0 += 64 * kScanRun) {
    const int first = b0 + lane * kScanRun;
    uint32_t v[kScanRun], sum = 0;
#pragma unroll
    for (int j = 0; j < kScanRun; ++j) v[j] = first + j < nb ? row[first + j] : 0u;
#pragma unroll
    for (int j = 0; j < kScanRun; ++j) sum += v[j];
    uint32_t x = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(x, off, 64);
      if (lane >= off) x += y;
    }
    uint32_t run = carry + x - sum;
#pragma unroll
    for (int j = 0; j < kScanRun; ++j) {
      if (first + j < nb) row[first + j] = run;
      run += v[j];
    }
    carry += __shfl(x, 63, 64);
  }
  if (lane == 0) totals[d] = carry;
}

__global__ __launch_bounds__(256) void k_sort_scan_wide(uint32_t* hist, uint32_t* totals, const uint32_t* n_dev,
                                                        long long cap, int nb_max, int tile) {
  scan_row_wide(hist, totals, n_dev, cap, nb_max, tile, (int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
}

__global__ __launch_bounds__(256) void k_sort_scan(uint32_t* hist, uint32_t* totals, const uint32_t* n_dev,
                                                   long long cap, int nb_max, int tile) {
  scan_row(hist, totals, n_dev, cap, nb_max, tile, blockIdx.x);
}

template <typename K, int ITEMS, int R, bool V>
__device__ __forceinline__ void scatter_block(const K* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
                                              K* __restrict__ keys_out, uint32_t* __restrict__ vals_out,
                                              const uint32_t* n_dev, long long cap, int shift, int bits,
                                              const uint32_t* hist, const uint32_t* totals, int nb_max,
                                              uint32_t* ranges, int tshift, bool direct, uint32_t bid) {
  static_assert(R % kSortThreads == 0, "thread t keeps digits [t DP, t DP + DP)");
  constexpr int TILE = kSortThreads * ITEMS, DP = R / kSortThreads;
  __shared__ uint32_t s_cnt[4][R];
  __shared__ uint32_t s_scan[R];
  __shared__ uint32_t s_w[4];
  __shared__ K s_key[TILE];
  __shared__ uint32_t s_val[V ? TILE : 1];  // keys-only sorts carry no values
  const uint32_t n = n_eff(n_dev, cap);
  const uint32_t nblk = (n + (uint32_t)TILE - 1) / (uint32_t)TILE;
  if (bid >= nblk) return;
  const uint32_t blk = xcd_remap(bid, nblk);  // the upsweep's mapping
  const uint32_t start = blk * (uint32_t)TILE;
  const int t = threadIdx.x;
  const int w = t >> 6, lane = t & 63;
  const uint32_t mask = (1u << bits) - 1u;
  const uint32_t wbase = start + (uint32_t)w * (ITEMS * 64);
  // the keys are on their way while the counts are read
  K key[ITEMS];
  uint32_t val[ITEMS];
  uint32_t pos[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t idx = wbase + r * 64 + lane;
    key[r] = idx < n ? keys_in[idx] : (K)0;
    if constexpr (V) val[r] = idx < n ? vals_in[idx] : 0u;
  }
  // global base of each digit for this block = exclusive scan of the digits'
  // totals + the digit's count in the blocks before
  {
    uint32_t total[DP], before[DP], sum = 0;
    bool added = false;
    if constexpr (DP == 1) {
      if (direct) {
        added = true;
        total[0] = before[0] = 0;
        for (uint32_t b0 = 0; b0 < nblk; b0 += 16) {
          uint32_t c[16];
#pragma unroll
          for (uint32_t j = 0; j < 16; ++j) c[j] = hist[(size_t)min(b0 + j, nblk - 1u) * R + t];
#pragma unroll
          for (uint32_t j = 0; j < 16; ++j) {
            total[0] += b0 + j < nblk ? c[j] : 0u;
            before[0] += b0 + j < blk ? c[j] : 0u;
          }
        }
      }
    }
    if (!added) {
#pragma unroll
      for (int i = 0; i < DP; ++i) {
        const uint32_t d = (uint32_t)(t * DP + i);
        total[i] = d <= mask ? totals[d] : 0u;
        before[i] = d <= mask ? hist[(size_t)d * nb_max + blk] : 0u;  // (a cache line of its own each)
      }
    }
#pragma unroll
    for (int i = 0; i < DP; ++i) sum += total[i];
    uint32_t tot;
    uint32_t run = block_incl_scan256(sum, s_w, tot) - sum;
#pragma unroll
    for (int i = 0; i < DP; ++i) {
      s_scan[t * DP + i] = run + before[i];
      // in a sort of one pass the digit is the tile id
      if (ranges && shift == tshift && blk == 0 && total[i] > 0) {
        ranges[2 * (t * DP + i)] = run;
        ranges[2 * (t * DP + i) + 1] = run + total[i];
      }
      run += total[i];
    }
  }
  for (int k = t; k < 4 * R; k += kSortThreads) (&s_cnt[0][0])[k] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const bool valid = wbase + r * 64 + lane < n;
    const uint32_t d = (uint32_t)(key[r] >> shift) & mask;
    const uint64_t peers = match_digit(d, valid, bits);
    const uint64_t below = peers & lanemask_lt();
    const uint32_t prior = s_cnt[w][d];
    pos[r] = prior + (uint32_t)__popcll(below);
    if (valid && below == 0) s_cnt[w][d] = prior + (uint32_t)__popcll(peers);
  }
  __syncthreads();
  // each digit's waves' local bases (exclusive scan over digits of the block
  // counts, then over waves) and the offset from local to global position
  {
    uint32_t c[DP][4], sum = 0;
#pragma unroll
    for (int i = 0; i < DP; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        c[i][k] = s_cnt[k][t * DP + i];
        sum += c[i][k];
      }
    uint32_t tot;
    uint32_t run = block_incl_scan256(sum, s_w, tot) - sum;
#pragma unroll
    for (int i = 0; i < DP; ++i) {
      s_scan[t * DP + i] -= run;  // global = s_scan[d] + local position
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        s_cnt[k][t * DP + i] = run;
        run += c[i][k];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t idx = wbase + r * 64 + lane;
    if (idx < n) {
      const uint32_t d = (uint32_t)(key[r] >> shift) & mask;
      const uint32_t lp = s_cnt[w][d] + pos[r];
      s_key[lp] = key[r];
      if constexpr (V) s_val[lp] = val[r];
    }
  }
  __syncthreads();
  const uint32_t nloc = min((uint32_t)TILE, n - start);
  for (uint32_t i = t; i < nloc; i += kSortThreads) {
    const K k = s_key[i];
    const uint32_t d = (uint32_t)(k >> shift) & mask;
    const uint32_t dst = s_scan[d] + i;
    keys_out[dst] = k;
    if constexpr (V) vals_out[dst] = s_val[i];
    if (ranges && shift != tshift) {
      // last pass of a tile-list sort: within a digit run the block's keys are
      // in final order, so a run of one tile id is contiguous here and in the
      // output; its ends give the tile's [start, end) across blocks by
      // atomic min / max (ranges start as [UINT_MAX, 0))
      const uint32_t tile = (uint32_t)(k >> tshift);
      if (i == 0 || (uint32_t)(s_key[i - 1] >> tshift) != tile) atomicMin(&ranges[2 * tile], dst);
      if (i + 1 == nloc || (uint32_t)(s_key[i + 1] >> tshift) != tile) atomicMax(&ranges[2 * tile + 1], dst + 1);
    }
  }
}

template <typename K, int ITEMS, int R, bool V>
__global__ __launch_bounds__(kSortThreads) void k_sort_scatter(const K* __restrict__ keys_in,
                                                               const uint32_t* __restrict__ vals_in,
                                                               K* __restrict__ keys_out,
                                                               uint32_t* __restrict__ vals_out,
                                                               const uint32_t* n_dev, long long cap, int shift,
                                                               int bits, const uint32_t* hist,
                                                               const uint32_t* totals, int nb_max, uint32_t* ranges,
                                                               int tshift, bool direct) {
  scatter_block<K, ITEMS, R, V>(keys_in, vals_in, keys_out, vals_out, n_dev, cap, shift, bits, hist, totals, nb_max,
                                ranges, tshift, direct, blockIdx.x);
}

// Up to this many workgroups the scatter adds the counts up itself.  At 10 (10
// 000 keys) a pass then takes 8.9 us of kernels instead of 12.9; at 98 to 127 the
// scatter's reading of every count (6.9 -> 9.5 us) costs what the scan did, but
// the host is spared 3 us for its launch.  A segmented sort, which runs in
// graphs, takes the lower limit.
constexpr int kDirectBlocks = 128, kSegDirectBlocks = 32;

template <typename K, int ITEMS, int R>
void sort_pass(const K* kin, const uint32_t* vin, K* kout, uint32_t* vout, const uint32_t* n_dev, long long capacity,
               int shift, int bits, uint32_t* hist, uint32_t* totals, int nb_max, hipStream_t s, uint32_t* ranges,
               int tshift) {
  const bool direct = R == kRadix && nb_max <= kDirectBlocks;
  hipLaunchKernelGGL((k_sort_upsweep<K, ITEMS, R>), dim3(nb_max), dim3(kSortThreads), 0, s, kin, n_dev, capacity,
                     shift, bits, hist, nb_max, direct);
  if (R == kWideRadix)
    hipLaunchKernelGGL(k_sort_scan_wide, dim3(R / 4), dim3(256), 0, s, hist, totals, n_dev, capacity, nb_max,
                       kSortThreads * ITEMS);
  else if (!direct)
    hipLaunchKernelGGL(k_sort_scan, dim3(1u << bits), dim3(256), 0, s, hist, totals, n_dev, capacity, nb_max,
                       kSortThreads * ITEMS);
  if constexpr (R == kRadix) {
    if (vin) {
      hipLaunchKernelGGL((k_sort_scatter<K, ITEMS, R, true>), dim3(nb_max), dim3(kSortThreads), 0, s, kin, vin, kout,
                         vout, n_dev, capacity, shift, bits, hist, totals, nb_max, ranges, tshift, direct);
      return;
    }
  }
  hipLaunchKernelGGL((k_sort_scatter<K, ITEMS, R, false>), dim3(nb_max), dim3(kSortThreads), 0, s, kin, vin, kout,
                     vout, n_dev, capacity, shift, bits, hist, totals, nb_max, ranges, tshift, direct);
}

// Pass p of a sort of bits [start_bit, end_bit) in `passes` near equal digits:
// its first bit and its width.
inline void pass_digit(int start_bit, int end_bit, int passes, int p, int& shift, int& bits) {
  const int total = end_bit - start_bit, base = total / passes, more = total % passes;
  shift = start_bit + p * base + (p < more ? p : more);
  bits = base + (p < more ? 1 : 0);
}

// Stable LSD sort on key bits [start_bit, end_bit); vals_a == nullptr sorts
// the keys alone.  With `ranges` (tile lists: key >> start_bit is a tile id),
// the last pass also records every tile's [start, end) into ranges, which the
// caller initialises to [UINT_MAX, 0) per tile (empty tiles keep that).
template <typename K>
hipError_t sort_pairs(K* keys_a, uint32_t* vals_a, K* keys_b, uint32_t* vals_b, const uint32_t* n_dev,
                      long long capacity, int start_bit, int end_bit, void* tmp, hipStream_t s, int* result_in_b,
                      uint32_t* ranges = nullptr) {
  const bool wide = sizeof(K) == 4 && !vals_a && wide_digit(end_bit - start_bit, capacity);
  const int passes = wide ? 1 : sort_passes(end_bit - start_bit);
  *result_in_b = passes & 1;
  if (capacity <= 0) return hipSuccess;
  const int tile = wide ? kSortThreads * kWideItems : sort_tile(capacity);
  const int nb_max = (int)((capacity + tile - 1) / tile);
  uint32_t* hist = (uint32_t*)tmp;
  uint32_t* totals = hist + align_up((size_t)(wide ? kWideRadix : kRadix) * (size_t)nb_max, 64);
  K* kin = keys_a;
  uint32_t* vin = vals_a;
  K* kout = keys_b;
  uint32_t* vout = vals_b;
  for (int p = 0; p < passes; ++p) {
    int shift, bits;
    pass_digit(start_bit, end_bit, passes, p, shift, bits);
    auto pass = tile == kSortThreads * 4 ? sort_pass<K, 4, kRadix> : sort_pass<K, 8, kRadix>;
    if (tile == kSortThreads * 16) pass = sort_pass<K, 16, kRadix>;
    if constexpr (sizeof(K) == 4)
      if (wide) pass = sort_pass<K, kWideItems, kWideRadix>;
    pass(kin, vin, kout, vout, n_dev, capacity, shift, bits, hist, totals, nb_max, s, p + 1 == passes ? ranges : nullptr,
         start_bit);
    std::swap(kin, kout);
    std::swap(vin, vout);
  }
  return hipGetLastError();
}

// ---- segmented sort ---------------------------------------------------------
// Descriptor, pass by pass: uint32 prefix[n + 1] (each segment's upsweep /
// scatter workgroups in that pass, rounded up to a multiple of 8 so that a
// segment's first block starts a round of the XCD round-robin, as a launch
// of its own does; 0 once the segment has no pass left), then one SegPass
// per segment.  The segments of a sort share their workgroups' size and digit
// array: 4096 keys and 10-bit digits if any segment takes such a digit, else
// 1024 keys (sort_tile of a capacity up to kSegMaxKeys) and 8-bit ones.
struct SegPass {
  const uint32_t* kin;
  const uint32_t* vin;
  uint32_t* kout;
  uint32_t* vout;
  const uint32_t* n_dev;
  uint32_t* hist;
  uint32_t* totals;
  uint32_t* ranges;
  long long cap;
  int nb_max;  // 0: the segment has no such pass
  int shift;
  int bits;
  int tshift;
};
constexpr int kSegItems = 4;
// beside a pass's workgroup count in blocks[p]: what the launch has to know
constexpr unsigned kSegWide = 1u << 31, kSegDirect = 1u << 30, kSegBlocks = kSegDirect - 1u;

static size_t seg_pass_bytes(int n) {
  return align_up(sizeof(uint32_t) * (size_t)(n + 1), 256) + align_up(sizeof(SegPass) * (size_t)n, 256);
}

__device__ __forceinline__ int seg_of(const uint32_t* prefix, int n, uint32_t b) {
  // the last segment whose range starts at or before b (empty ranges are skipped)
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (prefix[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

template <int ITEMS, int R>
__global__ __launch_bounds__(kSortThreads) void k_seg_upsweep(const uint32_t* prefix, const SegPass* ps, int n,
                                                              bool direct) {
  const uint32_t b = blockIdx.x;
  const int f = seg_of(prefix, n, b);
  const SegPass p = ps[f];
  upsweep_block<uint32_t, ITEMS, R>(p.kin, p.n_dev, p.cap, p.shift, p.bits, p.hist, p.nb_max, direct, b - prefix[f]);
}

// 256 workgroups per segment, one per digit.
__global__ __launch_bounds__(256) void k_seg_scan(const SegPass* ps) {
  const SegPass p = ps[blockIdx.x >> kRadixBits];
  const int d = (int)(blockIdx.x & (kRadix - 1));
  if (p.nb_max == 0 || d >> p.bits) return;
  scan_row(p.hist, p.totals, p.n_dev, p.cap, p.nb_max, kSortThreads * kSegItems, d);
}

// 256 workgroups per segment, four digits each.
__global__ __launch_bounds__(256) void k_seg_scan_wide(const SegPass* ps) {
  const SegPass p = ps[blockIdx.x / (kWideRadix / 4)];
  const int d = (int)(blockIdx.x % (kWideRadix / 4) * 4 + (threadIdx.x >> 6));
  if (p.nb_max == 0 || d >> p.bits) return;
  scan_row_wide(p.hist, p.totals, p.n_dev, p.cap, p.nb_max, kSortThreads * kWideItems, d);
}

template <int ITEMS, int R, bool V>
__global__ __launch_bounds__(kSortThreads) void k_seg_scatter(const uint32_t* prefix, const SegPass* ps, int n,
                                                              bool direct) {
  const uint32_t b = blockIdx.x;
  const int f = seg_of(prefix, n, b);
  const SegPass p = ps[f];
  scatter_block<uint32_t, ITEMS, R, V>(p.kin, p.vin, p.kout, p.vout, p.n_dev, p.cap, p.shift, p.bits, p.hist,
                                       p.totals, p.nb_max, p.ranges, p.tshift, direct, b - prefix[f]);
}

size_t seg_sort_desc_bytes(int n, int passes) {
  if (n <= 0 || passes < 1 || passes > kSegMaxPasses) return 0;
  return seg_pass_bytes(n) * (size_t)passes;
}

bool seg_sort_build(int n, const SortSeg* segs, void* host, size_t bytes, unsigned* blocks, int* passes) {
  if (n <= 0 || !segs || !host || !blocks || !passes) return false;
  int np = 0;
  const bool values = segs[0].vals_a != nullptr;
  bool wide = false;
  long long most = 0;
  for (int f = 0; f < n; ++f) {
    const SortSeg& g = segs[f];
    if (g.capacity <= 0 || g.capacity > kSegMaxKeys || !g.keys_a || !g.keys_b || !g.tmp) return false;
    if ((g.vals_a != nullptr) != values || (values && !g.vals_b)) return false;
    if (g.start_bit < 0 || g.end_bit <= g.start_bit || g.end_bit > 32) return false;
    if (((uintptr_t)g.keys_a | (uintptr_t)g.keys_b) & 15) return false;  // 16-byte key loads
    const bool gw = !values && wide_digit(g.end_bit - g.start_bit, g.capacity);
    wide |= gw;
    most = std::max(most, g.capacity);
    np = std::max(np, gw ? 1 : sort_passes(g.end_bit - g.start_bit));
  }
  if (np > kSegMaxPasses || bytes < seg_sort_desc_bytes(n, np)) return false;
  const int tile = kSortThreads * (wide ? kWideItems : kSegItems);
  const bool direct = !wide && (most + tile - 1) / tile <= kSegDirectBlocks;
  for (int p = 0; p < kSegMaxPasses; ++p) blocks[p] = 0;
  for (int p = 0; p < np; ++p) {
    char* base = (char*)host + seg_pass_bytes(n) * (size_t)p;
    uint32_t* prefix = (uint32_t*)base;
    SegPass* ps = (SegPass*)(base + align_up(sizeof(uint32_t) * (size_t)(n + 1), 256));
    unsigned long long total = 0;
    for (int f = 0; f < n; ++f) {
      const SortSeg& g = segs[f];
      const int nb_max = (int)((g.capacity + tile - 1) / tile);
      const int width = g.end_bit - g.start_bit;
      const int gp = !values && wide_digit(width, g.capacity) ? 1 : sort_passes(width);
      uint32_t* hist = (uint32_t*)g.tmp;
      SegPass& q = ps[f];
      const bool odd = p & 1;
      q.kin = odd ? g.keys_b : g.keys_a;
      q.vin = odd ? g.vals_b : g.vals_a;
      q.kout = odd ? g.keys_a : g.keys_b;
      q.vout = odd ? g.vals_a : g.vals_b;
      q.n_dev = g.n_dev;
      q.hist = hist;
      q.totals = hist + align_up((size_t)(wide ? kWideRadix : kRadix) * (size_t)nb_max, 64);  // sort_pairs' layout of tmp
      q.ranges = p + 1 == gp ? g.ranges : nullptr;
      q.cap = g.capacity;
      q.nb_max = p < gp ? nb_max : 0;
      q.shift = q.bits = 0;
      if (p < gp) pass_digit(g.start_bit, g.end_bit, gp, p, q.shift, q.bits);
      q.tshift = g.start_bit;
      prefix[f] = (uint32_t)total;
      total += p < gp ? align_up((size_t)nb_max, 8) : 0;
      if (total > kSegBlocks) return false;
    }
    prefix[n] = (uint32_t)total;
    blocks[p] = (unsigned)total | (wide ? kSegWide : 0u) | (direct ? kSegDirect : 0u);
  }
  *passes = np;
  return true;
}

template <int ITEMS, int R, bool V>
static void seg_pass_launch(int n, const uint32_t* prefix, const SegPass* q, unsigned blocks, bool direct,
                            hipStream_t s) {
  hipLaunchKernelGGL((k_seg_upsweep<ITEMS, R>), dim3(blocks), dim3(kSortThreads), 0, s, prefix, q, n, direct);
  if (R == kWideRadix)
    hipLaunchKernelGGL(k_seg_scan_wide, dim3((unsigned)n * (kWideRadix / 4)), dim3(256), 0, s, q);
  else if (!direct)
    hipLaunchKernelGGL(k_seg_scan, dim3((unsigned)n * kRadix), dim3(256), 0, s, q);
  hipLaunchKernelGGL((k_seg_scatter<ITEMS, R, V>), dim3(blocks), dim3(kSortThreads), 0, s, prefix, q, n, direct);
}

hipError_t seg_sort_launch(int n, const void* dev_desc, const unsigned* blocks, bool values, hipStream_t s) {
  for (int p = 0; p < kSegMaxPasses && blocks[p] > 0; ++p) {
    const char* base = (const char*)dev_desc + seg_pass_bytes(n) * (size_t)p;
    const uint32_t* prefix = (const uint32_t*)base;
    const SegPass* q = (const SegPass*)(base + align_up(sizeof(uint32_t) * (size_t)(n + 1), 256));
    const unsigned nb = blocks[p] & kSegBlocks;
    const bool direct = blocks[p] & kSegDirect;
    if (values) seg_pass_launch<kSegItems, kRadix, true>(n, prefix, q, nb, direct, s);
    else if (blocks[p] & kSegWide) seg_pass_launch<kWideItems, kWideRadix, false>(n, prefix, q, nb, direct, s);
    else seg_pass_launch<kSegItems, kRadix, false>(n, prefix, q, nb, direct, s);
  }
  return hipGetLastError();
}

hipError_t sort_pairs_u64(uint64_t* keys_a, uint32_t* vals_a, uint64_t* keys_b, uint32_t* vals_b,
                          const uint32_t* n_dev, long long capacity, int end_bit, void* tmp, hipStream_t s,
                          int* result_in_b) {
  return sort_pairs<uint64_t>(keys_a, vals_a, keys_b, vals_b, n_dev, capacity, 0, end_bit, tmp, s, result_in_b);
}

hipError_t sort_pairs_u32(uint32_t* keys_a, uint32_t* vals_a, uint32_t* keys_b, uint32_t* vals_b,
                          const uint32_t* n_dev, long long capacity, int end_bit, void* tmp, hipStream_t s,
                          int* result_in_b, uint32_t* ranges) {
  return sort_pairs<uint32_t>(keys_a, vals_a, keys_b, vals_b, n_dev, capacity, 0, end_bit, tmp, s, result_in_b,
                              ranges);
}

hipError_t sort_keys_u32(uint32_t* keys_a, uint32_t* keys_b, const uint32_t* n_dev, long long capacity, int start_bit,
                         int end_bit, void* tmp, hipStream_t s, int* result_in_b, uint32_t* ranges) {
  return sort_pairs<uint32_t>(keys_a, nullptr, keys_b, nullptr, n_dev, capacity, start_bit, end_bit, tmp, s,
                              result_in_b, ranges);
}

}  // namespace gs

extern "C" size_t gs_sort_tmp_bytes(long long capacity) { return gs::sort_tmp_bytes(capacity); }

extern "C" int gs_sort_pairs_u64(uint64_t* keys_a, uint32_t* vals_a, uint64_t* keys_b, uint32_t* vals_b,
                                 const uint32_t* n_dev, long long capacity, int end_bit, void* tmp,
                                 size_t tmp_bytes, int* result_in_b, void* stream) {
  if (capacity < 0 || capacity > 0x7fffffffLL || end_bit < 1 || end_bit > 64 || !n_dev || !result_in_b)
    return GS_E_ARG;
  if (capacity > 0 && (!keys_a || !vals_a || !keys_b || !vals_b || !tmp)) return GS_E_ARG;
  if (tmp_bytes < gs::sort_tmp_bytes(capacity)) return GS_E_WORKSPACE;
  const hipError_t e = gs::sort_pairs_u64(keys_a, vals_a, keys_b, vals_b, n_dev, capacity, end_bit, tmp,
                                          (hipStream_t)stream, result_in_b);
  return e == hipSuccess ? GS_OK : GS_E_LAUNCH;
}

extern "C" int gs_sort_pairs_u32(uint32_t* keys_a, uint32_t* vals_a, uint32_t* keys_b, uint32_t* vals_b,
                                 const uint32_t* n_dev, long long capacity, int end_bit, void* tmp,
                                 size_t tmp_bytes, int* result_in_b, void* stream) {
  if (capacity < 0 || capacity > 0x7fffffffLL || end_bit < 1 || end_bit > 32 || !n_dev || !result_in_b)
    return GS_E_ARG;
  if (capacity > 0 && (!keys_a || !vals_a || !keys_b || !vals_b || !tmp)) return GS_E_ARG;
  if (((uintptr_t)keys_a | (uintptr_t)keys_b) & 15) return GS_E_ARG;  // 16-byte key loads
  if (tmp_bytes < gs::sort_tmp_bytes(capacity)) return GS_E_WORKSPACE;
  const hipError_t e = gs::sort_pairs_u32(keys_a, vals_a, keys_b, vals_b, n_dev, capacity, end_bit, tmp,
                                          (hipStream_t)stream, result_in_b);
  return e == hipSuccess ? GS_OK : GS_E_LAUNCH;
}
