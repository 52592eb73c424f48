// drivers.cuh - lookup drivers shared by every index descriptor.
#pragma once

#include "device.cuh"
#include "indexes.cuh"
#include "indexes_ext.cuh"

namespace gj {

// lookup_plain_kernel is the successor of lookup_kernel
// (src/index_lookup_common.cuh:217-245): a grid-stride loop in whole waves
// (the reference rounds its loop bound to a warp multiple for the same
// reason, :235) with 64-bit indices (the reference uses int, which limits it
// to 2^31 probes).
//
// kMinWaves: waves per SIMD that the registers are cut to.  Binary search by lines fits 64
// registers without a spill (u64 keys 66 by itself: 7 waves, and one more round of workgroups
// where 8 waves take a million probes in two); the learned column layout over u32 keys fits by
// itself and is held there.  RadixSpline and Harmonia spill under the cut (405 -> 498 and 391
// -> 452 us).
template <class Dev> constexpr int kMinWaves = 1;
template <class K> inline constexpr int kMinWaves<BSearchDev<K, true>> = 8;
template <> inline constexpr int kMinWaves<LearnedDev<uint32_t, kLeafNoFallback>> = 8;
template <class Dev, class K>
__global__ __launch_bounds__(256, kMinWaves<Dev>) void lookup_plain_kernel(Dev d, const K* __restrict__ probes, uint64_t m,
                                                           uint32_t* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  d.stage(lds);
  __syncthreads();
  const uint64_t waves = (static_cast<uint64_t>(gridDim.x) * blockDim.x) / kWave;
  const uint64_t wave = (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / kWave;
  for (uint64_t base = wave * kWave; base < m; base += waves * kWave) {
    const uint64_t i = base + static_cast<uint64_t>(lane());
    const bool active = i < m;
    const K x = active ? load_stream(probes + i) : K(0);
    const uint32_t r = d.lookup(x, active, lds);
    if (active) store_stream(out + i, r);
  }
}

// Second pass of the plain driver for learned models with a few leaves routed
// to the B-tree: every probe whose result holds kFallbackMark is looked up again
// with index d.  A wave scans kMarkSlots x 64 results per step (independent,
// coalesced loads) and runs a cooperative lookup only for the slots holding a mark.
constexpr int kMarkSlots = 16;

template <class Dev, class K>
__global__ __launch_bounds__(256) void lookup_marked_kernel(Dev d, const K* __restrict__ probes, uint64_t m,
                                                            uint32_t* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  d.stage(lds);
  __syncthreads();
  const uint64_t waves = (static_cast<uint64_t>(gridDim.x) * blockDim.x) / kWave;
  const uint64_t wave = (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / kWave;
  const uint64_t span = static_cast<uint64_t>(kMarkSlots) * kWave;
  for (uint64_t base = wave * span; base < m; base += waves * span) {
    uint32_t v[kMarkSlots];
#pragma unroll
    for (int k = 0; k < kMarkSlots; ++k) {
      const uint64_t i = base + static_cast<uint64_t>(k * kWave + lane());
      v[k] = i < m ? out[i] : 0u;
    }
    uint32_t mk = 0;  // bit k: slot k holds a mark
#pragma unroll
    for (int k = 0; k < kMarkSlots; ++k) mk |= (v[k] == kFallbackMark ? 1u : 0u) << k;
    if (ballot(mk != 0) == 0) continue;  // wave-uniform
#pragma unroll 1
    for (int k = 0; k < kMarkSlots; ++k) {
      const bool marked = (mk >> k) & 1u;
      if (ballot(marked) == 0) continue;  // wave-uniform
      const uint64_t i = base + static_cast<uint64_t>(k * kWave + lane());
      const K x = marked ? probes[i] : K(0);
      const uint32_t r = d.lookup(x, marked, lds);
      if (marked) out[i] = r;
    }
  }
}

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2).  This maps the dispatch index to a logical index so that each XCD
// receives one contiguous eighth of the logical range [0, nb); workgroups from nb on keep
// their index.
__device__ __forceinline__ uint32_t xcd_logical_block(uint32_t nb) {
  if (nb % 8 != 0 || blockIdx.x >= nb) return blockIdx.x;
  return (blockIdx.x % 8) * (nb / 8) + blockIdx.x / 8;
}

// Lookup over a partitioned relation (partitioned_lookup_kernel,
// src/index_lookup_partitioning.cu:218-248): tuple t has key keys[t], and its row id
// goes to res[t], in tuple order (full-line stores); the driver then gathers the row ids
// back to probe order.  Padding tuples (key_max) are looked up too, their row ids never
// read.  The relation is `windows` windows one after the other, window w from tuple
// start[w * fan] to start[(w + 1) * fan], each in key order by partition.  Each XCD takes one
// contiguous eighth of every window, and its workgroups sweep these eighths together, a tile of
// each window in turn, so the key range in flight on an XCD (hence the index nodes and
// column lines its L2 must hold) spans a few partitions, the same ones in all the
// windows.
//
// What bounds it: fabric lines where the tuples are sparse.  Where they are dense that is not
// settled (the B-tree over 2^25 u64 keys: 8.6 L1 accesses and 0.23 fabric lines a tuple; but
// staging a run's separators in LDS, so that a tuple reads its leaf line alone, took as
// long).
template <class Dev, class K>
__global__ __launch_bounds__(256) void lookup_tuples_kernel(Dev d, const K* __restrict__ keys,
                                                            const uint64_t* __restrict__ start, uint32_t windows,
                                                            uint64_t fan, uint32_t tiles, uint32_t* __restrict__ res) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  d.stage(lds);
  __syncthreads();
  const uint32_t groups = (gridDim.x % 8 == 0) ? 8u : 1u;  // XCDs
  const uint32_t per = gridDim.x / groups;                 // workgroups per XCD
  const uint64_t g = blockIdx.x % groups;
  for (uint32_t j = blockIdx.x / groups; j < tiles; j += per) {  // this XCD's tiles, windows in turn
    const uint32_t t = windows == 1 ? j : j / windows, w = j - t * windows;
    const uint64_t first = start[w * fan], size = start[(w + 1) * fan] - first;
    const uint64_t chunk = ((size + groups - 1) / groups + kWave - 1) / kWave * kWave;
    const uint64_t lo = g * chunk, hi = lo + chunk < size ? lo + chunk : size;
    const uint64_t i = lo + static_cast<uint64_t>(t) * blockDim.x + threadIdx.x;
    if (i - lane() >= hi) continue;  // wave-uniform
    const bool active = i < hi;
    const K x = active ? load_stream(keys + first + i) : K(0);
    const uint32_t r = d.lookup(x, active, lds);
    if (active) store_stream(res + first + i, r);
  }
}

// Blockwise-sorting driver (bws_lookup, src/index_lookup_common.cuh:397-549): a workgroup
// loads a tile of probes with their positions, sorts the tile in LDS, looks it up in that
// order, so the lanes of a wave walk neighbouring index paths, and scatters the row ids back.
//
// The tile is counted, scanned and placed by the probe's coarse position in the index (the
// part of the search that reads no memory: bucket, staged separators, leaf), kBwsBins of
// them at most.  Probes of one bin stay in any order: the bins follow the column's own
// distribution and are about as many as the tile's probes, so finer order would not bring
// lanes closer.  What bounds it: LDS.  The bitonic network over whole keys (the reference
// uses CUB's block radix sort) made 66 passes over the tile, 505 us of the 829 that 2^24
// probes of 2^22 u64 keys took with binary search; now 77 of 625.
//
// Over the host link the bound is the link, and what counts is that the tiles in flight on
// an XCD, which all sweep the column from its start to its end, find each other's lines in its
// L2.  With every lane of a wave at work (all four rounds of its quads in flight) the
// queues before the link grow until the tiles have drifted apart; so (Link) only every
// 2^skip-th lane looks a probe up: one lane of a quad for a column in host memory, two where
// only the index structures are there.  2^22 probes of 2^22 keys, bitonic network -> all lanes -> now, ms:
// binary search u32 6.4 -> 10.5 -> 5.9, RadixSpline u64 11.6 -> 18.2 -> 10.7, learned u32 6.9
// -> 10.3 -> 5.9, B-tree u32 9.6 -> 9.4 -> 7.1; structures alone, B-tree u64 2.04 -> 2.86 ->
// 1.83, learned u64 0.55 -> 0.68 -> 0.44.
constexpr uint32_t kBwsBins = 2048;
constexpr int kBwsBlock = 256;

// A lookup by waves whose lanes are all at work.
template <class Dev, class K>
__device__ __forceinline__ uint32_t lookup_full(const Dev& d, K x, bool active, const uint8_t* lds) {
  if constexpr (requires { d.template lookup<true>(x, active, lds); })
    return d.template lookup<true>(x, active, lds);
  else
    return d.lookup(x, active, lds);
}

template <class Dev, class K, int TILE, bool Link>
__global__ __launch_bounds__(kBwsBlock) void lookup_bws_kernel(Dev d, const K* __restrict__ probes, uint64_t m,
                                                               uint32_t shift, uint32_t skip, uint32_t* __restrict__ out) {
  constexpr int kItems = TILE / kBwsBlock;
  constexpr int kWords = static_cast<int>(kBwsBins) / 2 / kBwsBlock;  // words of two 16-bit counts per thread
  static_assert(TILE <= 65535 && kWords == 4, "16-bit counts, 16 bytes of them per thread");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  d.stage(lds);
  const size_t ilds = (d.lds_bytes() + 15) / 16 * 16;
  K* sk = reinterpret_cast<K*>(lds + ilds);
  uint32_t* cnt = reinterpret_cast<uint32_t*>(sk + TILE);                         // counts, then offsets
  uint16_t* si = reinterpret_cast<uint16_t*>(cnt + kBwsBins / 2);
  uint32_t* wsum = reinterpret_cast<uint32_t*>(si + TILE);
  const uint32_t w = threadIdx.x / kWave;
  for (uint64_t tile = static_cast<uint64_t>(blockIdx.x) * TILE; tile < m;
       tile += static_cast<uint64_t>(gridDim.x) * TILE) {
    const uint32_t valid = m - tile < TILE ? static_cast<uint32_t>(m - tile) : static_cast<uint32_t>(TILE);
    reinterpret_cast<u32x4*>(cnt)[threadIdx.x] = u32x4{0, 0, 0, 0};
    K x[kItems];
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
      const uint32_t t = u * kBwsBlock + threadIdx.x;
      x[u] = t < valid ? load_stream(probes + tile + t) : K(0);
    }
    __syncthreads();  // counts are zero; the first tile: the index's LDS image is there
    uint32_t at[kItems];  // bin, and the rank in it above
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
      const uint32_t bin = d.coarse(x[u], lds) >> shift, half = 16 * (bin & 1);
      if (u * kBwsBlock + threadIdx.x < valid)
        at[u] = bin | ((atomicAdd(&cnt[bin / 2], 1u << half) >> half) << 16);
    }
    __syncthreads();
    u32x4 v = reinterpret_cast<u32x4*>(cnt)[threadIdx.x];
    uint32_t local = 0;
#pragma unroll
    for (int q = 0; q < kWords; ++q) {
      const uint32_t n = v[q];
      v[q] = local | ((local + (n & 0xFFFFu)) << 16);
      local += (n & 0xFFFFu) + (n >> 16);
    }
    uint32_t incl = local;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t y = __shfl_up(incl, o, kWave);
      if (lane() >= o) incl += y;
    }
    if (lane() == kWave - 1) wsum[w] = incl;
    __syncthreads();
    uint32_t before = incl - local;
#pragma unroll
    for (uint32_t q = 0; q < kBwsBlock / kWave; ++q) before += q < w ? wsum[q] : 0u;
#pragma unroll
    for (int q = 0; q < kWords; ++q) v[q] += before | (before << 16);
    reinterpret_cast<u32x4*>(cnt)[threadIdx.x] = v;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
      const uint32_t t = u * kBwsBlock + threadIdx.x;
      if (t < valid) {
        const uint32_t bin = at[u] & 0xFFFFu;
        const uint32_t p = ((cnt[bin / 2] >> (16 * (bin & 1))) & 0xFFFFu) + (at[u] >> 16);
        sk[p] = x[u];
        si[p] = static_cast<uint16_t>(t);
      }
    }
    __syncthreads();
    const uint32_t lk = Link ? skip : 0u;
    for (uint32_t base = w * (kWave >> lk); base < valid; base += kBwsBlock >> lk) {
      const uint32_t ln = static_cast<uint32_t>(lane()), t = base + (ln >> lk);
      const bool active = t < valid && (ln & ((1u << lk) - 1)) == 0;
      const K key = active ? sk[t] : K(0);
      const uint32_t r = Link ? d.lookup(key, active, lds) : lookup_full(d, key, active, lds);
      if (active) out[tile + si[t]] = r;
    }
    __syncthreads();
  }
}

}  // namespace gj
