// partition.hip - radix partitioner (gj_partition).
//
// Replaces the fast-interconnects pair gpu_contiguous_prefix_sum_int64 +
// gpu_chunked_laswwc_radix_partition_int64_int64 that run_on_stream launches
// (src/index_lookup_partitioning.cu:300-366; declarations
// src/gpu_radix_partition.cuh:8-45), whose sources are absent.  Semantics kept:
// partition p of key k is (k >> ignore_bits) & (2^radix_bits - 1); every
// partition starts on a 128-byte boundary (the reference pads partitions by
// GPU_CACHE_LINE_SIZE, src/partitioned_relation.hpp:7-10); payload = the
// tuple's position in the input.  Structure of arrays instead of Tuple{key,
// payload}.  gj_partition keeps the input order inside each partition; the
// partitioned lookup driver lets it float (the payload carries the position).
//
// Kernels (no cooperative launch, no device-wide barrier):
//   hist     one block per contiguous chunk, LDS histogram of 2^radix_bits u32 bins
//   colscan  column prefix over the blocks and the partition totals, 64 partitions a block
//   starts   one block: aligned exclusive prefix over partitions -> partition starts
//   scatter  one block per chunk (the same chunks as hist): tiles sorted by partition in
//            LDS, stable or in any order, then stored run by run; all blocks, and more where
//            the chunks are few, write the padding behind every partition
#include <algorithm>

#include "common.hpp"
#include "lookup_dispatch.hpp"

namespace gj {

constexpr int kPartTile = 4096;  // chunks are whole multiples of this many items (histogram rows are sized by it)
constexpr uint32_t kMaxRadixBits = 16;

__host__ __device__ __forceinline__ uint32_t part_align(int key_bytes) { return 128u / static_cast<uint32_t>(key_bytes); }

// The digit (k >> shift) & (fan - 1).  ignore_bits is only held below the key's width, so a
// digit may reach past the key's top bit, and the first pass of two may begin there: those
// digit bits are zero, while the shift itself takes its distance modulo 64.
struct Digit {
  uint32_t shift, mask;
  __device__ __forceinline__ Digit(uint32_t s, uint32_t fan) : shift(s & 63u), mask(s < 64u ? fan - 1u : 0u) {}
  template <class K>
  __device__ __forceinline__ uint32_t operator()(K k) const {
    return static_cast<uint32_t>(static_cast<uint64_t>(k) >> shift) & mask;
  }
};

// A store that would land past the output's capacity is not made; it is counted
// instead (never for a consistent histogram), so callers can report the loss.
__device__ __forceinline__ void drop(unsigned long long* dropped) {
  if (dropped) atomicAdd(dropped, 1ull);
}

// Segment mode of the histogram and stable scatter kernels (the second pass of a
// fan-out above 2^12): the input is cut into segs segments (segment h holds
// [start[h], start[h] + count[h]), the first pass's partitions), each segment into
// chunks of `chunk` items; block j handles chunk j - chunk0[h] of the segment h with
// chunk0[h] <= j < chunk0[h + 1], and partition p of segment h is output partition
// h * 2^bits + p.  Blocks from chunk0[segs] on have no work.  segs = 0: plain mode,
// block c handles items [c * chunk, (c + 1) * chunk), c < chunks.
struct Seg {
  const uint64_t* chunk0;  // segs + 1 entries
  const uint64_t* start;   // segs entries
  const uint64_t* count;   // segs entries
  uint32_t segs;
  uint32_t chunks;  // plain mode
};

// This block's item range and output partition base; false: the block has no work.
__device__ __forceinline__ bool seg_range(const Seg& sg, uint64_t c, uint64_t chunk, uint64_t m, uint32_t fan,
                                          uint64_t& lo, uint64_t& hi, uint64_t& pbase) {
  if (!sg.segs) {
    lo = c * chunk;
    hi = std::min<uint64_t>(m, lo + chunk);
    pbase = 0;
    return lo < m || c == 0;  // workgroups past the chunks have no work
  }
  if (c >= sg.chunk0[sg.segs]) return false;
  uint32_t a = 0, b = sg.segs;  // the segment h with chunk0[h] <= c < chunk0[h + 1]
  while (b - a > 1) {
    const uint32_t mid = (a + b) / 2;
    if (sg.chunk0[mid] <= c) a = mid; else b = mid;
  }
  lo = sg.start[a] + (c - sg.chunk0[a]) * chunk;
  hi = std::min<uint64_t>(sg.start[a] + sg.count[a], lo + chunk);
  pbase = static_cast<uint64_t>(a) * fan;
  return true;
}

// What is partitioned: the keys, or their hashes (the hash table's build; computing the hash
// where a key is read costs less than a pass that writes it and two that read it back).
template <bool Hashed, class K>
__device__ __forceinline__ K item_of(K k) {
  if constexpr (Hashed) return static_cast<K>(key_hash<K>(static_cast<uint64_t>(k)));
  return k;
}

// One block per chunk (256 or 1024 threads), four loads in flight per thread.
template <class K, bool Hashed = false>
__global__ __launch_bounds__(1024) void part_hist_kernel(const K* __restrict__ keys, uint64_t m, uint64_t chunk,
                                                         uint32_t shift, uint32_t bits, uint32_t* __restrict__ hist,
                                                         Seg sg) {
  extern __shared__ uint32_t h[];
  const uint32_t fan = 1u << bits;
  // chunk index; the scatter maps blocks the same way
  const uint64_t c = sg.segs ? static_cast<uint64_t>(blockIdx.x) : xcd_logical_block(sg.chunks);
  uint64_t lo, hi, pbase;
  if (!seg_range(sg, c, chunk, m, fan, lo, hi, pbase)) return;  // block-uniform, before any barrier
  const Digit digit(shift, fan);
  for (uint32_t p = threadIdx.x; p < fan; p += blockDim.x) h[p] = 0;
  __syncthreads();
  constexpr int kIn = 4;
  for (uint64_t i0 = lo + threadIdx.x; i0 < hi; i0 += kIn * blockDim.x) {
    K v[kIn];
#pragma unroll
    for (int u = 0; u < kIn; ++u) {
      const uint64_t i = i0 + static_cast<uint64_t>(u) * blockDim.x;
      v[u] = i < hi ? load_stream(keys + i) : K(0);
    }
#pragma unroll
    for (int u = 0; u < kIn; ++u)
      if (i0 + static_cast<uint64_t>(u) * blockDim.x < hi) atomicAdd(&h[digit(item_of<Hashed>(v[u]))], 1u);
  }
  __syncthreads();
  for (uint32_t p = threadIdx.x; p < fan; p += blockDim.x) hist[c * fan + p] = h[p];
}

// Column scan of one segment's histogram rows [r0, r1): hist[r][p] becomes the sum of the
// rows before r, count[p] the total.  A workgroup takes 64 partitions and cuts the rows
// into one span per wave: each lane sums its partition over the wave's span (a row of 64
// counts is one coalesced 256-byte read, kColIn rows in flight), the spans' sums meet in
// LDS, and a second walk over the span writes the prefixes.  (One wave per partition
// reading a row per lane touched 64 lines per load: 14.5 us for 245 rows of 1024
// partitions, now 5.)
constexpr int kColIn = 8;
constexpr uint32_t kColThreads = 1024;
__device__ __forceinline__ void scan_columns(uint32_t* __restrict__ hist, uint64_t r0, uint64_t r1, uint32_t p0,
                                             uint32_t fan, uint64_t* __restrict__ count) {
  constexpr uint32_t kWaves = kColThreads / kWave;
  __shared__ uint32_t part[kWaves][kWave];
  const uint32_t w = threadIdx.x / kWave;
  const uint32_t p = p0 + static_cast<uint32_t>(lane());
  const uint64_t per = (r1 - r0 + kWaves - 1) / kWaves;
  const uint64_t a = std::min<uint64_t>(r1, r0 + w * per), b = std::min<uint64_t>(r1, a + per);
  uint32_t sum = 0;
  for (uint64_t r = a; r < b; r += kColIn) {
    uint32_t v[kColIn];
#pragma unroll
    for (int u = 0; u < kColIn; ++u) v[u] = (r + u < b && p < fan) ? hist[(r + u) * fan + p] : 0u;
#pragma unroll
    for (int u = 0; u < kColIn; ++u) sum += v[u];
  }
  part[w][lane()] = sum;
  __syncthreads();
  uint32_t run = 0, total = 0;
#pragma unroll
  for (uint32_t v = 0; v < kWaves; ++v) {
    const uint32_t x = part[v][lane()];
    run += v < w ? x : 0u;
    total += x;
  }
  if (w == 0 && p < fan) count[p] = total;
  for (uint64_t r = a; r < b; r += kColIn) {
    uint32_t v[kColIn];
#pragma unroll
    for (int u = 0; u < kColIn; ++u) v[u] = (r + u < b && p < fan) ? hist[(r + u) * fan + p] : 0u;
#pragma unroll
    for (int u = 0; u < kColIn; ++u) {
      if (r + u < b && p < fan) hist[(r + u) * fan + p] = run;
      run += v[u];
    }
  }
}

__global__ __launch_bounds__(kColThreads) void part_colscan_kernel(uint32_t* __restrict__ hist, uint32_t blocks,
                                                                   uint32_t fan, uint64_t* __restrict__ count) {
  scan_columns(hist, 0, blocks, blockIdx.x * kWave, fan, count);
}

// The same per segment of the segmented pass (grid: segments x ceil(fan / 64)).
__global__ __launch_bounds__(kColThreads) void seg_colscan_wide_kernel(uint32_t* __restrict__ hist,
                                                                       const uint64_t* __restrict__ chunk0,
                                                                       uint32_t fan, uint64_t* __restrict__ count) {
  const uint32_t per = (fan + kWave - 1) / kWave;
  const uint32_t h = blockIdx.x / per;
  scan_columns(hist, chunk0[h], chunk0[h + 1], (blockIdx.x % per) * kWave, fan, count + static_cast<uint64_t>(h) * fan);
}

// Sum of v over the block's earlier threads (1024 threads); total: over all of them.
__device__ __forceinline__ uint64_t sum_before_1024(uint64_t v, uint64_t& total) {
  __shared__ uint64_t waves[1024 / kWave];
  uint64_t x = v;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint64_t y = __shfl_up(x, o, kWave);
    if (lane() >= o) x += y;
  }
  const uint32_t w = threadIdx.x / kWave;
  if (lane() == kWave - 1) waves[w] = x;
  __syncthreads();
  uint64_t before = x - v;
  total = 0;
#pragma unroll
  for (uint32_t q = 0; q < 1024 / kWave; ++q) {
    before += q < w ? waves[q] : 0;
    total += waves[q];
  }
  return before;
}

// start[p] = align_up(start[p-1] + count[p-1], align); one block of 1024 threads.
// Each thread owns `per` consecutive partitions and reads their counts kScanBatch at a
// time, loads first (a thread's loads do not depend on one another, so a batch is in
// flight together: at fan-out 2^16, 64 counts per thread, one at a time took 115 µs).
// start2 (optional): a second copy of start[0 .. fan).
constexpr uint32_t kScanBatch = 8;
__global__ __launch_bounds__(1024) void part_scan_starts_kernel(const uint64_t* __restrict__ count, uint32_t fan,
                                                                uint32_t align, uint64_t* __restrict__ start,
                                                                uint64_t* __restrict__ start2) {
  const uint32_t per = (fan + blockDim.x - 1) / blockDim.x;
  const uint32_t p0 = threadIdx.x * per;
  uint64_t local = 0;
  for (uint32_t q = 0; q < per; q += kScanBatch) {
    uint64_t c[kScanBatch];
#pragma unroll
    for (uint32_t u = 0; u < kScanBatch; ++u) {
      const uint32_t p = p0 + q + u;
      c[u] = (q + u < per && p < fan) ? count[p] : 0;
    }
#pragma unroll
    for (uint32_t u = 0; u < kScanBatch; ++u) local += (c[u] + align - 1) / align * align;
  }
  uint64_t total;
  uint64_t run = sum_before_1024(local, total);
  for (uint32_t q = 0; q < per; q += kScanBatch) {
    uint64_t c[kScanBatch];
#pragma unroll
    for (uint32_t u = 0; u < kScanBatch; ++u) {
      const uint32_t p = p0 + q + u;
      c[u] = (q + u < per && p < fan) ? count[p] : 0;
    }
#pragma unroll
    for (uint32_t u = 0; u < kScanBatch; ++u) {
      const uint32_t p = p0 + q + u;
      if (q + u < per && p < fan) {
        start[p] = run;
        if (start2) start2[p] = run;
      }
      run += (c[u] + align - 1) / align * align;
    }
  }
  if (threadIdx.x == 0) start[fan] = total;  // padded
}

// The same starts over many partitions (a batch of windows brings up to 2^18, where one
// block took 420 µs): block b owns the kScanSpan partitions [b * kScanSpan, ...).
// part_span_sums_kernel writes each span's padded total to sums[b];
// part_span_starts_kernel adds the totals of the spans before its own and scans its span
// through LDS (loads and stores coalesced).
constexpr uint32_t kScanThreads = 256;
constexpr uint32_t kScanSpan = kScanThreads * kScanBatch;  // 2048 partitions per block
constexpr uint32_t kOneBlockScanMax = 8192;                // up to here the one-block kernel
constexpr uint64_t kScanSumsBytes = 8192;                  // sums of up to 1024 spans (2^21 partitions)

__device__ __forceinline__ uint64_t padded_count(uint64_t c, uint32_t align) { return (c + align - 1) / align * align; }

// Sum over the block of one value per thread; every thread gets the total.
__device__ __forceinline__ uint64_t span_block_sum(uint64_t v, uint64_t* s) {
  s[threadIdx.x] = v;
  __syncthreads();
  for (uint32_t off = kScanThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) s[threadIdx.x] += s[threadIdx.x + off];
    __syncthreads();
  }
  const uint64_t t = s[0];
  __syncthreads();
  return t;
}

__global__ __launch_bounds__(kScanThreads) void part_span_sums_kernel(const uint64_t* __restrict__ count, uint32_t fan,
                                                                     uint32_t align, uint64_t* __restrict__ sums) {
  __shared__ uint64_t s[kScanThreads];
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * kScanSpan;
  uint64_t c[kScanBatch];
#pragma unroll
  for (uint32_t u = 0; u < kScanBatch; ++u) {
    const uint64_t p = base + u * kScanThreads + threadIdx.x;
    c[u] = p < fan ? count[p] : 0;
  }
  uint64_t local = 0;
#pragma unroll
  for (uint32_t u = 0; u < kScanBatch; ++u) local += padded_count(c[u], align);
  const uint64_t t = span_block_sum(local, s);
  if (threadIdx.x == 0) sums[blockIdx.x] = t;
}

__global__ __launch_bounds__(kScanThreads) void part_span_starts_kernel(const uint64_t* __restrict__ count,
                                                                       uint32_t fan, uint32_t align,
                                                                       const uint64_t* __restrict__ sums,
                                                                       uint64_t* __restrict__ start) {
  __shared__ uint64_t v[kScanSpan];
  __shared__ uint64_t s[kScanThreads];
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * kScanSpan;
  uint64_t before = 0;
  for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kScanThreads) before += sums[b];
#pragma unroll
  for (uint32_t u = 0; u < kScanBatch; ++u) {
    const uint64_t p = base + u * kScanThreads + threadIdx.x;
    v[u * kScanThreads + threadIdx.x] = p < fan ? padded_count(count[p], align) : 0;
  }
  const uint64_t off = span_block_sum(before, s);  // also orders the stores to v before the reads below
  // thread t scans v[t * kScanBatch, (t + 1) * kScanBatch)
  uint64_t local = 0;
#pragma unroll
  for (uint32_t u = 0; u < kScanBatch; ++u) local += v[threadIdx.x * kScanBatch + u];
  s[threadIdx.x] = local;
  __syncthreads();
  for (uint32_t o = 1; o < kScanThreads; o <<= 1) {  // Hillis-Steele inclusive scan
    const uint64_t y = threadIdx.x >= o ? s[threadIdx.x - o] : 0;
    __syncthreads();
    s[threadIdx.x] += y;
    __syncthreads();
  }
  uint64_t run = off + s[threadIdx.x] - local;
#pragma unroll
  for (uint32_t u = 0; u < kScanBatch; ++u) {
    const uint64_t x = v[threadIdx.x * kScanBatch + u];
    v[threadIdx.x * kScanBatch + u] = run;
    run += x;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t u = 0; u < kScanBatch; ++u) {
    const uint64_t p = base + u * kScanThreads + threadIdx.x;
    if (p < fan) start[p] = v[u * kScanThreads + threadIdx.x];
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == kScanThreads - 1) start[fan] = off + s[kScanThreads - 1];
}

// start[0 .. fan] from count[0 .. fan) (start[fan] = padded total), copied to start2 when
// given; sums: kScanSumsBytes of scratch, used above kOneBlockScanMax partitions.
inline void launch_scan_starts(const uint64_t* count, uint64_t fan, uint32_t align, uint64_t* start, uint64_t* start2,
                               uint64_t* sums, hipStream_t s) {
  if (fan <= kOneBlockScanMax) {
    hipLaunchKernelGGL(part_scan_starts_kernel, dim3(1), dim3(1024), 0, s, count, static_cast<uint32_t>(fan), align,
                       start, start2);
    GJ_HIP_CHECK(hipGetLastError());
    return;
  }
  const uint64_t spans = ceil_div(fan, kScanSpan);
  GJ_REQUIRE(spans * 8 <= kScanSumsBytes, GJ_ERR_INVALID, "too many partitions for the starts scan");
  hipLaunchKernelGGL(part_span_sums_kernel, dim3(static_cast<unsigned>(spans)), dim3(kScanThreads), 0, s, count,
                     static_cast<uint32_t>(fan), align, sums);
  GJ_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(part_span_starts_kernel, dim3(static_cast<unsigned>(spans)), dim3(kScanThreads), 0, s, count,
                     static_cast<uint32_t>(fan), align, sums, start);
  GJ_HIP_CHECK(hipGetLastError());
  if (start2) GJ_HIP_CHECK(hipMemcpyAsync(start2, start, fan * 8, hipMemcpyDeviceToDevice, s));
}

// Marks the padding slots after every partition (fewer than `align` each) with payload
// 0xFFFFFFFF and key_max: the blocks of the grid share the partitions, one slot per thread,
// kPadIn of them in flight (2^20 probes in windows of 64 at fan-out 2^10, learned: the whole
// lookup 3531 us with one, now 3277; at 2^8 1171 and 1022).
constexpr uint32_t kPadIn = 4;
template <class K>
__device__ __forceinline__ void pad_partitions(const uint64_t* __restrict__ start, const uint64_t* __restrict__ count,
                                               uint32_t fan, uint32_t align, K* __restrict__ keys,
                                               uint32_t* __restrict__ payload) {
  const uint32_t slots = (fan + gridDim.x - 1) / gridDim.x * align;  // of the block's partitions
  for (uint32_t t0 = threadIdx.x; t0 < slots; t0 += kPadIn * blockDim.x) {
    uint64_t n[kPadIn], s[kPadIn];
#pragma unroll
    for (uint32_t u = 0; u < kPadIn; ++u) {
      const uint32_t t = t0 + u * blockDim.x, p = blockIdx.x + (t / align) * gridDim.x;
      const bool mine = t < slots && p < fan;
      n[u] = mine ? count[p] : 0;
      s[u] = mine ? start[p] : 0;
    }
#pragma unroll
    for (uint32_t u = 0; u < kPadIn; ++u) {
      const uint64_t at = n[u] + (t0 + u * blockDim.x) % align;
      if (at < (n[u] + align - 1) / align * align) {
        keys[s[u] + at] = key_max<K>();
        if (payload) payload[s[u] + at] = 0xFFFFFFFFu;
      }
    }
  }
}

// Scatter.  in_payload == nullptr: payload = payload_base + input position.  A block walks
// its chunk in tiles of B x I items.  Per tile:
//   rank    Stable: each wave ranks its items among the equal digits of the wave (ballots
//           give the lanes with the same digit, a 16-bit row of counts per wave carries
//           the running rank from one 64-item slice to the next); otherwise an LDS atomic
//           add per item ranks it among the tile's equal digits in any order
//   scan    per partition: the waves' counts become exclusive prefixes, a block scan gives
//           the partition's offset in the tile, and the block's cursor moves on
//   place   keys and payloads into the tile buffer, in partition order
//   store   the tile buffer in order: neighbouring lanes store to neighbouring slots of
//           the same partition's run
// inv (optional): where every item went, in input order.
//
// What bounds it: HBM streaming (a key read, a key and a payload written) and, at large
// fan-outs, the short runs (B I / 2^bits items per partition and tile) in which the
// output is written; the next tile's items load while this one is placed and stored.  A
// scatter straight from registers (one store per lane to a random partition) and one that
// kept an open 128-byte segment per partition in LDS ran before: 10^7 u64 keys at fan-out
// 2^10, stable, 300 us a launch; this one 115.
__host__ __device__ constexpr size_t tile_lds_bytes(uint32_t fan, int key_bytes, bool payload, bool stable, int block,
                                                    int items) {
  const size_t tile = static_cast<size_t>(block) * items;
  return tile * key_bytes + (payload ? tile * 4 : 0)                            // tile keys, payloads
         + static_cast<size_t>(fan) * 8                                         // base, cur
         + static_cast<size_t>(fan) * (stable ? 2 * (block / kWave) + 2 : 4);   // rows and offsets, or counts
}

template <class K, bool Stable, bool InPayload, bool Hashed, int B, int I>
__global__ __launch_bounds__(B, 4) void part_scatter_kernel(
    const K* __restrict__ keys, const uint32_t* __restrict__ in_payload, uint32_t payload_base, uint64_t m,
    uint64_t chunk, uint32_t shift, uint32_t bits, const uint32_t* __restrict__ block_off,
    const uint64_t* __restrict__ start, const uint64_t* __restrict__ count, uint32_t align, K* __restrict__ out_keys,
    uint32_t* __restrict__ out_payload, uint32_t* __restrict__ inv, uint64_t cap,
    unsigned long long* __restrict__ dropped, Seg sg) {
  constexpr int T = B * I;
  constexpr int W = B / kWave;
  static_assert(T <= 65535, "tile offsets and ranks are 16-bit");
  constexpr int kRankItems = I / 2;  // slices ranked together (registers)
  extern __shared__ uint64_t tsm_[];
  __shared__ uint32_t wsum[W];
  const uint32_t fan = 1u << bits;
  if (align > 1) pad_partitions<K>(start, count, (sg.segs ? sg.segs : 1u) * fan, align, out_keys, out_payload);
  K* sk = reinterpret_cast<K*>(tsm_);                                // [T] tile keys, partition order
  uint32_t* sp = reinterpret_cast<uint32_t*>(sk + T);                // [T] tile payloads (with out_payload)
  uint32_t* base = sp + (out_payload ? T : 0);                       // [fan] output position of tile slot 0
  uint32_t* cur = base + fan;                                        // [fan] next output position
  uint32_t* cnt = cur + fan;                                         // [fan] counts, then tile offsets (unordered)
  uint16_t* rows = reinterpret_cast<uint16_t*>(cur + fan);           // [W][fan] (stable)
  uint16_t* off = rows + static_cast<size_t>(W) * fan;               // [fan] tile offsets (stable)
  // neighbouring chunks run on one XCD, so the partial lines that neighbouring
  // chunks write into a partition's run meet in the same L2
  const uint64_t c = sg.segs ? static_cast<uint64_t>(blockIdx.x) : xcd_logical_block(sg.chunks);  // as part_hist_kernel
  uint64_t lo, hi, pbase;
  if (!seg_range(sg, c, chunk, m, fan, lo, hi, pbase)) return;  // block-uniform, before any barrier
  const Digit digit(shift, fan);
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
  const int ln = lane();
  const uint64_t lt = (ln == 0) ? 0ull : (~0ull >> (64 - ln));  // lanes below this one
  uint16_t* mine = rows + static_cast<size_t>(w) * fan;
  for (uint32_t p = threadIdx.x; p < fan; p += B) {
    cur[p] = static_cast<uint32_t>(start[pbase + p]) + block_off[c * fan + p];
    if constexpr (!Stable) cnt[p] = 0;
  }
  auto clear_row = [&] {
    if (fan >= 8) {
      for (uint32_t p = ln * 8; p < fan; p += kWave * 8) *reinterpret_cast<u32x4*>(mine + p) = u32x4{0, 0, 0, 0};
    } else if (static_cast<uint32_t>(ln) < fan) {
      mine[ln] = 0;
    }
  };
  if constexpr (Stable) clear_row();
  __syncthreads();

  // Counts -> tile offsets; the cursors move on.  Each thread owns PER consecutive
  // partitions, whose 16-bit counts it adds two to a word.
  auto scan = [&]<int PER>() {
    const uint32_t p0 = threadIdx.x * PER;
    const bool own = p0 < fan;
    uint32_t n[PER], local = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) n[u] = 0;
    if (own) {
      if constexpr (!Stable) {
#pragma unroll
        for (int u = 0; u < PER; ++u) n[u] = cnt[p0 + u];
      } else if constexpr (PER == 1) {
#pragma unroll
        for (int v = 0; v < W; ++v) {
          const uint32_t t = rows[v * fan + p0];
          rows[v * fan + p0] = static_cast<uint16_t>(n[0]);
          n[0] += t;
        }
      } else {
        struct alignas(2 * PER) Words {
          uint32_t w[PER / 2];
        };
        Words r{};
#pragma unroll
        for (int v = 0; v < W; ++v) {
          Words* at = reinterpret_cast<Words*>(rows + v * fan + p0);
          const Words t = *at;
          *at = r;
#pragma unroll
          for (int q = 0; q < PER / 2; ++q) r.w[q] += t.w[q];  // a tile's counts sum below 2^16
        }
#pragma unroll
        for (int u = 0; u < PER; ++u) n[u] = (r.w[u / 2] >> (16 * (u & 1))) & 0xFFFFu;
      }
#pragma unroll
      for (int u = 0; u < PER; ++u) local += n[u];
    }
    uint32_t x = local;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t y = __shfl_up(x, o, kWave);
      if (ln >= o) x += y;
    }
    if (ln == kWave - 1) wsum[w] = x;
    __syncthreads();
    uint32_t run = x - local;
#pragma unroll
    for (int v = 0; v < W; ++v) run += v < w ? wsum[v] : 0u;
    if (own) {
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const uint32_t q = cur[p0 + u];
        if constexpr (Stable) off[p0 + u] = static_cast<uint16_t>(run);
        else cnt[p0 + u] = run;
        base[p0 + u] = q - run;
        cur[p0 + u] = q + n[u];
        run += n[u];
      }
    }
  };

  // The next tile's keys load while this tile is ranked, placed and stored (the barriers
  // wait for LDS operations only, so the loads stay in flight across them).
  K kn[I];
  // items of this wave in the tile that starts at t (may be none)
  auto wave_items = [&](uint64_t t) -> uint32_t {
    const uint64_t b = t + static_cast<uint64_t>(w) * (I * kWave);
    return b < hi ? static_cast<uint32_t>(std::min<uint64_t>(hi - b, I * kWave)) : 0u;
  };
  auto load_tile = [&](uint64_t t) {
    const uint32_t nn = wave_items(t);
    const K* src = keys + (t + static_cast<uint64_t>(w) * (I * kWave));
#pragma unroll
    for (int j = 0; j < I; ++j) {
      const uint32_t i = static_cast<uint32_t>(j * kWave + ln);
      kn[j] = i < nn ? load_stream(src + i) : K(0);
    }
  };
  load_tile(lo);
  for (uint64_t tile = lo; tile < hi; tile += T) {
    const uint64_t wbase = tile + static_cast<uint64_t>(w) * (I * kWave);
    const uint32_t wn = wave_items(tile);
    K k[I];
    uint32_t pay[InPayload ? I : 1], rk[I];
#pragma unroll
    for (int j = 0; j < I; ++j) {
      k[j] = item_of<Hashed>(kn[j]);
      if constexpr (InPayload) {
        const uint32_t i = static_cast<uint32_t>(j * kWave + ln);
        pay[j] = i < wn ? load_stream(in_payload + wbase + i) : 0u;
      }
    }
    if (tile + T < hi) load_tile(tile + T);  // block-uniform
    if constexpr (Stable) {
#pragma unroll
      for (int j0 = 0; j0 < I; j0 += kRankItems) {
        uint32_t d[kRankItems];
        uint32_t plo[kRankItems], phi[kRankItems];  // lanes of the slice with this lane's digit
#pragma unroll
        for (int j = 0; j < kRankItems; ++j) {
          const uint64_t valid = ballot(static_cast<uint32_t>((j0 + j) * kWave + ln) < wn);
          d[j] = digit(k[j0 + j]);
          plo[j] = static_cast<uint32_t>(valid);
          phi[j] = static_cast<uint32_t>(valid >> 32);
        }
        for (uint32_t b = 0; b < bits; ++b) {
#pragma unroll
          for (int j = 0; j < kRankItems; ++j) {
            const uint32_t one = 0u - ((d[j] >> b) & 1u);  // all ones where the digit's bit b is set
            const uint64_t set = ballot(one != 0);
            plo[j] &= ~(static_cast<uint32_t>(set) ^ one);
            phi[j] &= ~(static_cast<uint32_t>(set >> 32) ^ one);
          }
        }
#pragma unroll
        for (int j = 0; j < kRankItems; ++j) {
          const uint32_t before = static_cast<uint32_t>(__popc(plo[j] & static_cast<uint32_t>(lt)) +
                                                        __popc(phi[j] & static_cast<uint32_t>(lt >> 32)));
          const bool valid = static_cast<uint32_t>((j0 + j) * kWave + ln) < wn;
          const uint32_t at = mine[d[j]];  // every lane of the group reads the count before its first lane moves it
          rk[j0 + j] = at + before;
          if (valid && before == 0) mine[d[j]] = static_cast<uint16_t>(at + __popc(plo[j]) + __popc(phi[j]));
          __builtin_amdgcn_wave_barrier();
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < I; ++j) {
        rk[j] = 0;
        if (static_cast<uint32_t>(j * kWave + ln) < wn) rk[j] = atomicAdd(&cnt[digit(k[j])], 1u);
      }
    }
    __syncthreads();
    if (fan <= static_cast<uint32_t>(B)) scan.template operator()<1>();
    else if (fan == 2u * B) scan.template operator()<2>();
    else if (fan == 4u * B) scan.template operator()<4>();
    else scan.template operator()<8>();
    __syncthreads();
    // place
#pragma unroll
    for (int j = 0; j < I; ++j) {
      if (static_cast<uint32_t>(j * kWave + ln) < wn) {
        const uint32_t d = digit(k[j]);
        uint32_t slot;
        if constexpr (Stable) slot = off[d] + mine[d] + rk[j];
        else slot = cnt[d] + rk[j];
        if (slot < static_cast<uint32_t>(T)) {  // always true for a consistent count
          sk[slot] = k[j];
          if (out_payload) {
            if constexpr (InPayload) sp[slot] = pay[j];
            else sp[slot] = payload_base + static_cast<uint32_t>(wbase) + static_cast<uint32_t>(j * kWave + ln);
          }
        }
        if (inv) (inv + wbase)[j * kWave + ln] = base[d] + slot;
      }
    }
    if constexpr (Stable) {
      __builtin_amdgcn_wave_barrier();
      clear_row();
    }
    __syncthreads();
    if constexpr (!Stable) {  // read by the place phase, counted again from the next tile's start on
      for (uint32_t p = threadIdx.x; p < fan; p += B) cnt[p] = 0;
    }
    // store
    const uint32_t n = static_cast<uint32_t>(std::min<uint64_t>(hi - tile, T));
#pragma unroll
    for (int j = 0; j < I; ++j) {
      const uint32_t t = static_cast<uint32_t>(j * B) + threadIdx.x;
      if (t < n) {
        const K kk = sk[t];
        const uint32_t pos = base[digit(kk)] + t;
        if (pos < cap) {  // always true for a consistent histogram
          out_keys[pos] = kk;
          if (out_payload) out_payload[pos] = sp[t];
        } else {
          drop(dropped);
        }
      }
    }
    if constexpr (!Stable) __syncthreads();  // the counts are zero before the next tile adds to them
  }
}

// Chunks of the segmented pass: chunk0[h] = chunks of the segments before h (each
// segment cut into ceil(count[h] / chunk) chunks), chunk0[segs] = all chunks.  One block
// of 1024 threads, each owning `per` consecutive segments (a batch of windows brings
// thousands of segments), counts read kScanBatch at a time.
__global__ __launch_bounds__(1024) void seg_chunks_kernel(const uint64_t* __restrict__ count, uint32_t segs,
                                                          uint64_t chunk, uint64_t* __restrict__ chunk0) {
  const uint32_t per = (segs + blockDim.x - 1) / blockDim.x;
  const uint32_t h0 = threadIdx.x * per;
  uint64_t local = 0;
  for (uint32_t q = 0; q < per; q += kScanBatch) {
    uint64_t c[kScanBatch];
#pragma unroll
    for (uint32_t u = 0; u < kScanBatch; ++u) {
      const uint32_t h = h0 + q + u;
      c[u] = (q + u < per && h < segs) ? count[h] : 0;
    }
#pragma unroll
    for (uint32_t u = 0; u < kScanBatch; ++u) local += (c[u] + chunk - 1) / chunk;
  }
  uint64_t total;
  uint64_t run = sum_before_1024(local, total);
  for (uint32_t q = 0; q < per; q += kScanBatch) {
    uint64_t c[kScanBatch];
#pragma unroll
    for (uint32_t u = 0; u < kScanBatch; ++u) {
      const uint32_t h = h0 + q + u;
      c[u] = (q + u < per && h < segs) ? count[h] : 0;
    }
#pragma unroll
    for (uint32_t u = 0; u < kScanBatch; ++u) {
      const uint32_t h = h0 + q + u;
      if (q + u < per && h < segs) chunk0[h] = run;
      run += (c[u] + chunk - 1) / chunk;
    }
  }
  if (threadIdx.x == 0) chunk0[segs] = total;
}

// Segments of a batch of windows: segment h = probes [h * window, min((h + 1) * window, m)).
__global__ void seg_windows_kernel(uint64_t* __restrict__ start, uint64_t* __restrict__ count, uint32_t segs,
                                   uint64_t window, uint64_t m) {
  const uint64_t h = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (h >= segs) return;
  start[h] = h * window;
  count[h] = std::min<uint64_t>(window, m - h * window);
}

// Column scan of the segmented pass: for output partition g = h * fan + p, the
// histogram rows of segment h's chunks become exclusive prefixes and count[g] the
// total.  One thread per output partition.  A skewed first pass leaves one segment with
// most of the chunks (Zipf(1.0) probes: about 70 % of a window in segment 0, 5700
// chunks), so the rows are read kColBatch at a time, loads first: the loads do not
// depend on the running sum, and one at a time they took 730 µs per window.
constexpr int kColBatch = 16;
__global__ __launch_bounds__(256) void seg_colscan_kernel(uint32_t* __restrict__ hist, const uint64_t* __restrict__ chunk0,
                                                          uint32_t segs, uint32_t fan, uint64_t* __restrict__ count) {
  const uint64_t g = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (g >= static_cast<uint64_t>(segs) * fan) return;
  const uint64_t h = g / fan, p = g % fan;
  uint64_t run = 0;
  uint64_t j = chunk0[h];
  const uint64_t e = chunk0[h + 1];
  for (; j + kColBatch <= e; j += kColBatch) {
    uint32_t v[kColBatch];
#pragma unroll
    for (int u = 0; u < kColBatch; ++u) v[u] = hist[(j + u) * fan + p];
#pragma unroll
    for (int u = 0; u < kColBatch; ++u) {
      hist[(j + u) * fan + p] = static_cast<uint32_t>(run);
      run += v[u];
    }
  }
  for (; j < e; ++j) {
    const uint32_t v = hist[j * fan + p];
    hist[j * fan + p] = static_cast<uint32_t>(run);
    run += v;
  }
  count[g] = run;
}

namespace {

struct PartPlan {
  uint32_t fan, blocks;
  uint64_t chunk;
};

constexpr uint32_t kBlocksPerCu = 2;  // of a pass: two workgroups of 1024 threads are resident
constexpr size_t kMaxLds = 160 * 1024;

// Whole tiles per block, about kBlocksPerCu blocks per CU; each block's histogram row
// lives in scratch.
PartPlan plan(uint64_t m, uint32_t bits, int cu) {
  PartPlan p;
  p.fan = 1u << bits;
  const uint64_t want = static_cast<uint64_t>(cu) * kBlocksPerCu;
  uint64_t chunk = std::max<uint64_t>(kPartTile, ceil_div(m, want));
  chunk = ceil_div(chunk, kPartTile) * kPartTile;
  p.chunk = chunk;
  p.blocks = static_cast<uint32_t>(std::max<uint64_t>(1, ceil_div(m, chunk)));
  return p;
}

// The starts scan's span sums, then the plan's histogram rows.
uint64_t hist_bytes(uint64_t m, uint32_t bits, int cu) {
  const PartPlan p = plan(m, bits, cu);
  return kScanSumsBytes + ceil_div(static_cast<uint64_t>(p.blocks) * p.fan * 4 + 256, 256) * 256;
}

// Workgroups of the scatter: 512 threads of 8 items, 4096 items a tile (two workgroups per
// CU at fan-out 2^10).  10^7 u64 keys, whole call: at 2^10 partitions 147 us against 206
// with 2048-item tiles (shorter runs) and 149 with 8192-item ones (one workgroup per CU);
// at 2^4 87 against 88 and 113.
constexpr int kTileBlock = 512;
constexpr int kTileItems = 8;
static_assert(kTileBlock * kTileItems == kPartTile, "chunks are whole tiles");

// What a scatter launch reads and writes (see part_scatter_kernel).
template <class K>
struct Scatter {
  const K* keys;
  const uint32_t* in_payload;
  uint32_t payload_base;
  uint64_t m, chunk;
  uint32_t shift, bits;
  const uint32_t* hist;
  const uint64_t* start;
  const uint64_t* count;
  uint32_t align;
  K* out_keys;
  uint32_t* out_payload;
  uint32_t* inv;
  uint64_t cap;
  unsigned long long* dropped;
  Seg sg;
};

// Workgroups past the chunks share the padding alone: with few items and many partitions a
// thread would pad one slot after the other (5.5 k u32 items into 2^11 partitions: two
// workgroups took 51 us, now 9.6).  They are no part of the map of chunks to XCDs: counted in,
// they left the chunks of a few to the first XCDs alone (131072 u32 items into 2^12
// partitions, whole call: 33.3 us, now 31.3).
template <class K>
void launch_scatter(const Scatter<K>& a, bool stable, unsigned grid, int cu, hipStream_t s, bool hashed = false) {
  if (a.align > 1) {
    const uint64_t slots = (static_cast<uint64_t>(a.sg.segs ? a.sg.segs : 1u) << a.bits) * a.align;
    const uint64_t resident = static_cast<uint64_t>(cu) * kBlocksPerCu;
    grid = std::max(grid, static_cast<unsigned>(std::min<uint64_t>(ceil_div(slots, 2 * kTileBlock), resident)));
  }
  const size_t lds = tile_lds_bytes(1u << a.bits, sizeof(K), a.out_payload != nullptr, stable, kTileBlock, kTileItems);
  GJ_REQUIRE(lds <= kMaxLds - 1024 && (1u << a.bits) <= 8u * kTileBlock, GJ_ERR_INTERNAL,
             "partition fan-out does not fit the LDS");
  auto go = [&]<bool Stable, bool InPayload, bool Hashed = false>() {
    auto kernel = &part_scatter_kernel<K, Stable, InPayload, Hashed, kTileBlock, kTileItems>;
    if (lds > 65536)
      GJ_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kTileBlock), lds, s, a.keys, a.in_payload, a.payload_base, a.m, a.chunk,
                       a.shift, a.bits, a.hist, a.start, a.count, a.align, a.out_keys, a.out_payload, a.inv, a.cap,
                       a.dropped, a.sg);
    GJ_HIP_CHECK(hipGetLastError());
  };
  GJ_REQUIRE(!hashed || (!stable && !a.in_payload), GJ_ERR_INTERNAL, "hashes are partitioned unordered, by position");
  if (hashed) go.template operator()<false, false, true>();
  else if (stable && a.in_payload) go.template operator()<true, true>();
  else if (stable) go.template operator()<true, false>();
  else if (a.in_payload) go.template operator()<false, true>();
  else go.template operator()<false, false>();
}

// Above 2^12 partitions: a first pass on the high seg_high_bits() bits, then the
// segmented pass on the rest.
constexpr uint32_t kMaxSinglePassBits = 12;
uint32_t seg_low_bits(uint32_t bits) { return bits / 2; }
uint32_t seg_high_bits(uint32_t bits) { return bits - seg_low_bits(bits); }
uint64_t seg_max_chunks(uint64_t m, uint32_t bits) {
  return ceil_div(m, kPartTile) + (1ull << seg_high_bits(bits));
}

// Histogram region of a partitioning (the span sums, then either pass's rows).
uint64_t hist_region(uint64_t m, uint32_t bits, int cu) {
  if (bits <= kMaxSinglePassBits) return hist_bytes(m, bits, cu);
  const uint64_t seg_rows = seg_max_chunks(m, bits) * (1ull << seg_low_bits(bits)) * 4;
  return std::max<uint64_t>(hist_bytes(m, seg_high_bits(bits), cu),
                            kScanSumsBytes + ceil_div(seg_rows + 256, 256) * 256);
}

// histograms | (2 passes: first-pass keys and payloads [| segment starts, counts, chunk
// starts]) | partition starts for gj_partition
uint64_t scratch_for(uint64_t m, int key_bytes, uint32_t bits, uint32_t passes, int cu) {
  uint64_t b = hist_region(m, bits, cu);
  if (passes == 2 || bits > kMaxSinglePassBits)  // first-pass keys + payloads, each on a 256-byte boundary
    b += ceil_div((m + 32) * key_bytes, 256) * 256 + ceil_div((m + 32) * 4, 256) * 256;
  if (bits > kMaxSinglePassBits) b += 3 * ((1ull << seg_high_bits(bits)) + 2) * 8 + 256;
  b += ((1ull << bits) + 2) * 8 + 16;
  return b;
}

}  // namespace

// One partition pass with digit (k >> shift) & (2^bits - 1), stable (input order
// inside every partition) or unordered.  `align` pads partition starts (1 =
// unpadded).  Writes start[fan] and count[fan].
template <class K>
void partition_pass(const K* keys, const uint32_t* in_payload, uint32_t payload_base, uint64_t m, uint32_t shift,
                    uint32_t bits, uint32_t align, bool stable, K* out_keys, uint32_t* out_payload, uint64_t* start,
                    uint64_t* start2, uint64_t* count, uint32_t* hist, uint64_t* sums, unsigned long long* dropped,
                    int cu, hipStream_t s, bool hashed = false) {
  const PartPlan p = plan(m, bits, cu);
  const Seg sg{nullptr, nullptr, nullptr, 0, p.blocks};
  auto histogram = hashed ? &part_hist_kernel<K, true> : &part_hist_kernel<K, false>;
  hipLaunchKernelGGL(histogram, dim3(p.blocks), dim3(1024), p.fan * sizeof(uint32_t), s, keys, m, p.chunk, shift, bits,
                     hist, sg);
  GJ_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(part_colscan_kernel, dim3((p.fan + kWave - 1) / kWave), dim3(kColThreads), 0, s, hist, p.blocks,
                     p.fan, count);
  GJ_HIP_CHECK(hipGetLastError());
  launch_scan_starts(count, p.fan, align, start, start2, sums, s);
  const uint64_t cap = m + (align > 1 ? static_cast<uint64_t>(p.fan) * align : 0ull);
  launch_scatter<K>({keys, in_payload, payload_base, m, p.chunk, shift, bits, hist, start, count, align, out_keys,
                     out_payload, nullptr, cap, dropped, sg},
                    stable, p.blocks, cu, s, hashed);
}

uint64_t partition_capacity(uint64_t m, int key_bytes, uint32_t bits) {
  return m + (static_cast<uint64_t>(1) << bits) * part_align(key_bytes);
}

uint64_t partition_scratch(uint64_t m, int key_bytes, uint32_t bits, uint32_t passes) {
  return scratch_for(m, key_bytes, bits, passes, device_cu_count());
}

// The second pass above 2^12 partitions: the first pass left segment h (its partition
// on the high bits) at [start1[h], start1[h] + count1[h]) of keys / payload; each segment
// is partitioned on the low `bits` bits (digit (k >> shift) & (2^bits - 1)) into output
// partitions h * 2^bits + p, with 128-byte aligned starts.  Chunks never straddle
// segments, so every histogram row and cursor belongs to one segment.
constexpr uint64_t kSegChunk = 16384;
// Segments of this many chunks on average scan their histogram columns with a workgroup
// per 64 partitions; shorter ones take one thread per partition.
constexpr uint64_t kSegWideChunks = 32;

template <class K>
void partition_segmented(const K* keys, const uint32_t* payload, uint64_t m, uint32_t shift, uint32_t bits,
                         uint32_t segs, const uint64_t* start1, const uint64_t* count1, uint64_t* chunk0,
                         uint32_t align, bool stable, K* out_keys, uint32_t* out_payload, uint32_t* inv,
                         uint64_t* start, uint64_t* count, uint32_t* hist, uint64_t* sums,
                         unsigned long long* dropped, int cu, hipStream_t s) {
  const uint32_t fan = 1u << bits;
  const uint64_t total_fan = static_cast<uint64_t>(segs) * fan;
  // whole tiles, down to one where longer chunks would leave CUs without their two workgroups
  // (256 CUs, two windows of 262144 u32 probes at fan-out 2^12, the whole lookup: 107 -> 66 us)
  const uint64_t resident = static_cast<uint64_t>(cu) * kBlocksPerCu;
  const uint64_t chunk = std::clamp<uint64_t>(ceil_div(ceil_div(m, resident), kPartTile) * kPartTile, kPartTile, kSegChunk);
  const uint64_t blocks = ceil_div(m, chunk) + segs;  // an upper bound on the chunks
  GJ_REQUIRE(blocks < (1ull << 31), GJ_ERR_INVALID, "too many partition chunks");
  hipLaunchKernelGGL(seg_chunks_kernel, dim3(1), dim3(1024), 0, s, count1, segs, chunk, chunk0);
  GJ_HIP_CHECK(hipGetLastError());
  const Seg sg{chunk0, start1, count1, segs, 0};
  hipLaunchKernelGGL(part_hist_kernel<K>, dim3(static_cast<unsigned>(blocks)), dim3(kTileBlock),
                     fan * sizeof(uint32_t), s, keys, m, chunk, shift, bits, hist, sg);
  GJ_HIP_CHECK(hipGetLastError());
  if (ceil_div(m, chunk) >= kSegWideChunks * segs)
    hipLaunchKernelGGL(seg_colscan_wide_kernel, dim3(segs * ((fan + kWave - 1) / kWave)), dim3(kColThreads), 0, s, hist,
                       chunk0, fan, count);
  else
    hipLaunchKernelGGL(seg_colscan_kernel, dim3(static_cast<unsigned>(ceil_div(total_fan, 256))), dim3(256), 0, s, hist,
                       chunk0, segs, fan, count);
  GJ_HIP_CHECK(hipGetLastError());
  launch_scan_starts(count, total_fan, align, start, nullptr, sums, s);
  const uint64_t cap = m + (align > 1 ? total_fan * align : 0ull);
  launch_scatter<K>({keys, payload, 0u, m, chunk, shift, bits, hist, start, count, align, out_keys, out_payload, inv,
                     cap, dropped, sg},
                    stable, static_cast<unsigned>(blocks), cu, s);
}

namespace {

// A batch of windows in one partitioning: the windows are the segments of the
// segmented pass, so each window is partitioned on its own (output partition
// w * 2^bits + digit, window-major) while the batch takes one launch per kernel.  Two
// passes (or a fan-out above 2^12): a segmented pass per window on the high bits, then a
// segmented pass per (window, high digit) on the low bits.  No payloads: each pass
// records, in input order, where it put every item (inv1 for the first pass, inv2 for
// the second), which the lookup driver follows back to probe order.
uint32_t win_high_bits(uint32_t bits, uint32_t passes) {
  if (bits > kMaxSinglePassBits) return seg_high_bits(bits);
  return (passes == 2 && bits >= 2) ? (bits + 1) / 2 : 0u;  // 0: one pass
}

struct WinLayout {
  uint64_t windows, segs_b;  // windows; segments of the last pass
  uint32_t hb, lb;           // digit bits of the first pass (0: one pass) and of the last
  uint64_t o_tk, o_wstart, o_wcount, o_sa, o_ca, o_chunk0, bytes;
};

WinLayout win_layout(uint64_t m, uint64_t window, int key_bytes, uint32_t bits, uint32_t passes) {
  WinLayout L{};
  auto up = [](uint64_t v) { return ceil_div(v, 256) * 256; };
  L.windows = ceil_div(m, window);
  L.hb = win_high_bits(bits, passes);
  L.lb = bits - L.hb;
  L.segs_b = L.hb ? (L.windows << L.hb) : L.windows;
  const uint64_t tiles = ceil_div(m, static_cast<uint64_t>(kPartTile));
  const uint64_t rows_a = L.hb ? (tiles + L.windows) << L.hb : 0;
  const uint64_t rows_b = (tiles + L.segs_b) << L.lb;
  uint64_t o = kScanSumsBytes + up(std::max(rows_a, rows_b) * 4);  // span sums, histogram rows of either pass
  L.o_tk = o;
  if (L.hb) o += up((m + 32) * key_bytes);
  L.o_wstart = o;
  o += up((L.windows + 2) * 8);
  L.o_wcount = o;
  o += up((L.windows + 2) * 8);
  L.o_sa = o;
  if (L.hb) o += up((L.segs_b + 2) * 8);
  L.o_ca = o;
  if (L.hb) o += up((L.segs_b + 2) * 8);
  L.o_chunk0 = o;
  o += up((L.segs_b + 2) * 8);
  L.bytes = o;
  return L;
}

}  // namespace

uint64_t windows_capacity(uint64_t m, uint64_t window, int key_bytes, uint32_t bits) {
  return m + ceil_div(m, window) * (1ull << bits) * part_align(key_bytes);
}

uint64_t windows_tuples(uint64_t m, uint64_t window, int key_bytes, uint32_t bits) {
  return std::min<uint64_t>(windows_capacity(m, window, key_bytes, bits), m * part_align(key_bytes));
}

uint64_t windows_scratch(uint64_t m, uint64_t window, int key_bytes, uint32_t bits, uint32_t passes) {
  return win_layout(m, window, key_bytes, bits, passes).bytes;
}

bool windows_two_pass(uint32_t bits, uint32_t passes) { return win_high_bits(bits, passes) != 0; }

template <class K>
void partition_windows(const K* keys, uint64_t m, uint64_t window, uint32_t bits, uint32_t ignore, uint32_t passes,
                       K* out_keys, uint32_t* inv1, uint32_t* inv2, uint64_t* start, uint64_t* count,
                       uint8_t* scratch, unsigned long long* dropped, hipStream_t s) {
  if (m == 0) return;
  const WinLayout L = win_layout(m, window, sizeof(K), bits, passes);
  GJ_REQUIRE(inv1 && (!L.hb || inv2), GJ_ERR_INVALID, "partition_windows: missing position arrays");
  GJ_REQUIRE((L.segs_b << L.lb) < (1ull << 31), GJ_ERR_INVALID, "too many partitions in a batch of windows");
  auto* sums = reinterpret_cast<uint64_t*>(scratch);
  uint32_t* hist = reinterpret_cast<uint32_t*>(scratch + kScanSumsBytes);
  auto* wstart = reinterpret_cast<uint64_t*>(scratch + L.o_wstart);
  auto* wcount = reinterpret_cast<uint64_t*>(scratch + L.o_wcount);
  auto* chunk0 = reinterpret_cast<uint64_t*>(scratch + L.o_chunk0);
  hipLaunchKernelGGL(seg_windows_kernel, dim3(static_cast<unsigned>(ceil_div(L.windows, 256))), dim3(256), 0, s,
                     wstart, wcount, static_cast<uint32_t>(L.windows), window, m);
  GJ_HIP_CHECK(hipGetLastError());
  const uint32_t align = part_align(sizeof(K));
  const int cu = device_cu_count();
  if (!L.hb) {
    partition_segmented<K>(keys, nullptr, m, ignore, bits, static_cast<uint32_t>(L.windows), wstart, wcount, chunk0,
                           align, false, out_keys, nullptr, inv1, start, count, hist, sums, dropped, cu, s);
    return;
  }
  K* tk = reinterpret_cast<K*>(scratch + L.o_tk);
  auto* sa = reinterpret_cast<uint64_t*>(scratch + L.o_sa);
  auto* ca = reinterpret_cast<uint64_t*>(scratch + L.o_ca);
  partition_segmented<K>(keys, nullptr, m, ignore + L.lb, L.hb, static_cast<uint32_t>(L.windows), wstart, wcount,
                         chunk0, 1, false, tk, nullptr, inv1, sa, ca, hist, sums, dropped, cu, s);
  partition_segmented<K>(tk, nullptr, m, ignore, L.lb, static_cast<uint32_t>(L.segs_b), sa, ca, chunk0, align, false,
                         out_keys, nullptr, inv2, start, count, hist, sums, dropped, cu, s);
}
template void partition_windows<uint32_t>(const uint32_t*, uint64_t, uint64_t, uint32_t, uint32_t, uint32_t,
                                          uint32_t*, uint32_t*, uint32_t*, uint64_t*, uint64_t*, uint8_t*,
                                          unsigned long long*, hipStream_t);
template void partition_windows<uint64_t>(const uint64_t*, uint64_t, uint64_t, uint32_t, uint32_t, uint32_t,
                                          uint64_t*, uint32_t*, uint32_t*, uint64_t*, uint64_t*, uint8_t*,
                                          unsigned long long*, hipStream_t);

// Full partitioning into `out` (1 or 2 passes; fan-outs above 2^12 always take two, the
// second one segmented); scratch must hold partition_scratch() bytes; start must hold
// 2^bits + 1 entries (start[2^bits] = padded total).
template <class K>
void partition_keys(const K* keys, uint64_t m, uint32_t payload_base, uint32_t bits, uint32_t ignore, uint32_t passes,
                    bool stable, K* out_keys, uint32_t* out_payload, uint64_t* start, uint64_t* count, uint8_t* scratch,
                    unsigned long long* dropped, int cu, hipStream_t s, uint64_t* start2, bool hashed) {
  auto* sums = reinterpret_cast<uint64_t*>(scratch);
  uint32_t* hist = reinterpret_cast<uint32_t*>(scratch + kScanSumsBytes);
  const uint32_t align = part_align(sizeof(K));
  if (bits > kMaxSinglePassBits) {
    const uint32_t hb = seg_high_bits(bits), lb = seg_low_bits(bits);
    const uint32_t segs = 1u << hb;
    uint8_t* tmp = scratch + hist_region(m, bits, cu);
    K* tk = reinterpret_cast<K*>(tmp);
    uint32_t* tp = reinterpret_cast<uint32_t*>(tmp + ceil_div((m + 32) * sizeof(K), 256) * 256);
    uint8_t* small = tmp + ceil_div((m + 32) * sizeof(K), 256) * 256 + ceil_div((m + 32) * 4, 256) * 256;
    auto* start1 = reinterpret_cast<uint64_t*>(small);
    auto* count1 = start1 + segs + 2;
    auto* chunk0 = count1 + segs + 2;
    partition_pass<K>(keys, nullptr, payload_base, m, ignore + lb, hb, 1, stable, tk, tp, start1, nullptr, count1, hist,
                      sums, dropped, cu, s, hashed);
    partition_segmented<K>(tk, tp, m, ignore, lb, segs, start1, count1, chunk0, align, stable, out_keys, out_payload,
                           nullptr, start, count, hist, sums, dropped, cu, s);
    if (start2) GJ_HIP_CHECK(hipMemcpyAsync(start2, start, (1ull << bits) * 8, hipMemcpyDeviceToDevice, s));
    return;
  }
  if (passes == 1 || bits < 2) {
    partition_pass<K>(keys, nullptr, payload_base, m, ignore, bits, align, stable, out_keys, out_payload, start, start2,
                      count, hist, sums, dropped, cu, s, hashed);
    return;
  }
  // pass 1: the high half of the digit, unpadded, into scratch; pass 2: the full digit.
  const uint32_t b_hi = (bits + 1) / 2;
  uint8_t* tmp = scratch + hist_bytes(m, bits, cu);
  K* tk = reinterpret_cast<K*>(tmp);
  uint32_t* tp = reinterpret_cast<uint32_t*>(tmp + ceil_div((m + 32) * sizeof(K), 256) * 256);
  partition_pass<K>(keys, nullptr, payload_base, m, ignore + (bits - b_hi), b_hi, 1, stable, tk, tp, start, nullptr,
                    count, hist, sums, dropped, cu, s, hashed);
  partition_pass<K>(tk, tp, 0, m, ignore, bits, align, stable, out_keys, out_payload, start, start2, count, hist, sums,
                    dropped, cu, s);
}
template void partition_keys<uint32_t>(const uint32_t*, uint64_t, uint32_t, uint32_t, uint32_t, uint32_t, bool,
                                       uint32_t*, uint32_t*, uint64_t*, uint64_t*, uint8_t*, unsigned long long*, int,
                                       hipStream_t, uint64_t*, bool);
template void partition_keys<uint64_t>(const uint64_t*, uint64_t, uint32_t, uint32_t, uint32_t, uint32_t, bool,
                                       uint64_t*, uint32_t*, uint64_t*, uint64_t*, uint8_t*, unsigned long long*, int,
                                       hipStream_t, uint64_t*, bool);

}  // namespace gj

using namespace gj;

extern "C" {

uint64_t gj_partition_capacity(uint64_t m, int key_bytes, uint32_t radix_bits) {
  if ((key_bytes != 4 && key_bytes != 8) || radix_bits > kMaxRadixBits) return 0;
  return partition_capacity(m, key_bytes, radix_bits);
}

uint64_t gj_partition_scratch_bytes(uint64_t m, int key_bytes, const gj_partition_params* p) {
  if (!p || (key_bytes != 4 && key_bytes != 8) || p->radix_bits > kMaxRadixBits) return 0;
  uint64_t r = 0;
  const int st = guarded([&] { r = partition_scratch(m, key_bytes, p->radix_bits, p->passes == 2 ? 2 : 1); });
  return st == GJ_OK ? r : 0;
}

int gj_partition(const void* d_keys, uint64_t m, int key_bytes, const gj_partition_params* params,
                 gj_partitioned* out, void* d_scratch, uint64_t scratch_bytes, gj_stream_t stream) {
  return guarded([&] {
    GJ_REQUIRE(params && out, GJ_ERR_INVALID, "null argument");
    GJ_REQUIRE(key_bytes == 4 || key_bytes == 8, GJ_ERR_INVALID, "key_bytes must be 4 or 8");
    const uint32_t bits = params->radix_bits;
    GJ_REQUIRE(bits >= 1 && bits <= kMaxRadixBits, GJ_ERR_INVALID, "radix_bits must be in [1, 16]");
    GJ_REQUIRE(params->ignore_bits < static_cast<uint32_t>(8 * key_bytes), GJ_ERR_INVALID,
               "ignore_bits must be below the key width");
    GJ_REQUIRE(params->passes == 1 || params->passes == 2, GJ_ERR_INVALID, "passes must be 1 or 2");
    GJ_REQUIRE(m < 0xFFFFFFFFull, GJ_ERR_OVERFLOW, "partitioning needs m < 2^32 - 1 (u32 payloads)");
    GJ_REQUIRE(out->d_offsets && out->d_counts, GJ_ERR_INVALID, "null offsets / counts");
    const uint64_t cap = partition_capacity(m, key_bytes, bits);
    GJ_REQUIRE(out->capacity >= cap, GJ_ERR_INVALID, "gj_partitioned.capacity < gj_partition_capacity()");
    GJ_REQUIRE(cap < 0xFFFFFFFFull, GJ_ERR_OVERFLOW, "partitioned relation exceeds 2^32 tuples");
    const int cu = device_cu_count();
    const uint64_t need = scratch_for(m, key_bytes, bits, params->passes, cu);
    GJ_REQUIRE(d_scratch && scratch_bytes >= need, GJ_ERR_INVALID, "scratch smaller than gj_partition_scratch_bytes()");
    const hipStream_t s = S(stream);
    if (m == 0) {
      fill_bytes(out->d_offsets, 0, (1ull << bits) * 8, s);
      fill_bytes(out->d_counts, 0, (1ull << bits) * 8, s);
      return;
    }
    GJ_REQUIRE(d_keys && out->d_keys && out->d_payloads, GJ_ERR_INVALID, "null buffer");
    // partition starts (2^bits + 1 entries, the last is the padded total) live at the end of scratch
    uint8_t* sc = static_cast<uint8_t*>(d_scratch);
    uint64_t* start = reinterpret_cast<uint64_t*>(sc + need - ((1ull << bits) + 1) * 8 - 8);
    start = reinterpret_cast<uint64_t*>(reinterpret_cast<uintptr_t>(start) & ~static_cast<uintptr_t>(7));
    dispatch_key(key_bytes, [&]<class K>() {
      partition_keys<K>(static_cast<const K*>(d_keys), m, 0, bits, params->ignore_bits, params->passes, true,
                        static_cast<K*>(out->d_keys), out->d_payloads, start, out->d_counts, sc,
                        reinterpret_cast<unsigned long long*>(out->d_dropped), cu, s, out->d_offsets);
    });
  });
}

}  // extern "C"
