// lookup_dispatch.hpp - launch helpers and the internal interfaces between the
// libgj translation units.  Included only by *.hip files.
#pragma once

#include "common.hpp"
#include "drivers.cuh"
#include "index_impl.hpp"

namespace gj {

// Byte fill by a kernel (usable under stream capture, unlike hipMemsetAsync nodes).
void fill_bytes(void* d, int value, uint64_t bytes, hipStream_t s);

// Blocks of `block` threads that fit on one CU for kernel `fn` with `lds` bytes of dynamic LDS.
int blocks_per_cu(const void* fn, unsigned block, size_t lds);

inline unsigned lookup_block(const gj_lookup_params& p) {
  unsigned b = p.block_size ? p.block_size : 256u;
  GJ_REQUIRE(b % 64 == 0 && b >= 64 && b <= 256, GJ_ERR_INVALID, "block_size must be 64, 128, 192 or 256");
  return b;
}

// Blocks of a driver whose waves take steps of `per_block` items per workgroup, without a
// caller's grid_blocks: one step per wave.  The hardware then hands a workgroup's place to
// the next one as soon as it is free, where a grid of resident workgroups that each stride
// over the input ends with the slowest one and runs its waves in lockstep: 2^24 probes of
// 2^20 u32 keys (learned, column layout) 260 -> 218 us, 2^28 of 2^26 u64 keys (lines)
// 5.49 -> 5.29 ms.  Every workgroup stages the descriptor's LDS image, though, so above
// kStageStep bytes of it a wave takes one more step for each (Harmonia, 2^24 probes, one step ->
// so many -> resident workgroups that stride: 2^22 u32 keys 290 -> 264 -> 280 us, 2^20 u64 345
// -> 339 -> 367; binary search, 2^20 u32 235 -> 224 -> 243).  Never fewer workgroups than fit
// on the chip at once, if there is a step for each.
// HIP takes fewer than 2^32 threads in a launch, so beyond that many items waves take more steps.
constexpr uint64_t kStageStep = 8192;
constexpr uint64_t max_blocks(unsigned threads) { return 0xFFFFFFFFull / threads / 8 * 8; }  // whole XCD rounds
constexpr uint64_t cover_blocks(uint64_t items, uint64_t per_block, unsigned threads, size_t stage_bytes,
                                uint64_t resident) {
  const uint64_t cover = ceil_div(items, per_block);
  const uint64_t steps = 1 + stage_bytes / kStageStep;
  const uint64_t blocks = std::max<uint64_t>(ceil_div(cover, steps), std::min<uint64_t>(cover, resident));
  return std::min<uint64_t>(std::max<uint64_t>(blocks, 1), max_blocks(threads));
}
static_assert(cover_blocks(1ull << 40, 256, 256, 0, 2048) * 256 < 1ull << 32);
static_assert(cover_blocks(0xFFFFFFFFull, 64, 64, 0, 2048) * 64 < 1ull << 32);

template <class Dev, class K>
void launch_plain(const Dev& d, const K* probes, uint64_t m, uint32_t* out, const gj_lookup_params& p, hipStream_t s,
                  int cu) {
  if (m == 0) return;
  const unsigned block = lookup_block(p);
  const size_t lds = d.lds_bytes();
  const void* fn = reinterpret_cast<const void*>(&lookup_plain_kernel<Dev, K>);
  const uint64_t blocks = p.grid_blocks
                              ? std::max<uint64_t>(1, std::min<uint64_t>(p.grid_blocks, ceil_div(m, block)))
                              : cover_blocks(m, block, block, lds, static_cast<uint64_t>(blocks_per_cu(fn, block, lds)) * cu);
  hipLaunchKernelGGL((lookup_plain_kernel<Dev, K>), dim3(static_cast<unsigned>(blocks)), dim3(block), lds, s, d,
                     probes, m, out);
  GJ_HIP_CHECK(hipGetLastError());
}

// Second pass of the plain driver for learned leaves routed to the B-tree: the
// B-tree answers every probe whose result is kFallbackMark.
template <class K>
void launch_marked(const BTreeDev<K>& d, const K* probes, uint64_t m, uint32_t* out, const gj_lookup_params& p,
                   hipStream_t s, int cu) {
  if (m == 0) return;
  const unsigned block = lookup_block(p);
  const size_t lds = d.lds_bytes();
  const void* fn = reinterpret_cast<const void*>(&lookup_marked_kernel<BTreeDev<K>, K>);
  uint64_t blocks = static_cast<uint64_t>(blocks_per_cu(fn, block, lds)) * cu;
  blocks = std::min<uint64_t>(blocks, ceil_div(m, static_cast<uint64_t>(block) * kMarkSlots));
  blocks = std::max<uint64_t>(blocks, 1);
  hipLaunchKernelGGL((lookup_marked_kernel<BTreeDev<K>, K>), dim3(static_cast<unsigned>(blocks)), dim3(block), lds, s,
                     d, probes, m, out);
  GJ_HIP_CHECK(hipGetLastError());
}

// Tuples of `windows` windows of up to window_max tuples each (padding included); start:
// the starts of their partitions, `fan` a window, on the device.
template <class Dev, class K>
void launch_tuples(const Dev& d, const K* keys, const uint64_t* start, uint32_t windows, uint64_t fan,
                   uint64_t window_max, uint32_t* res, const gj_lookup_params& p, hipStream_t s, int cu) {
  if (windows == 0 || window_max == 0) return;
  const unsigned block = lookup_block(p);
  const size_t lds = d.lds_bytes();
  const void* fn = reinterpret_cast<const void*>(&lookup_tuples_kernel<Dev, K>);
  const uint64_t total = windows * window_max;
  uint64_t blocks = p.grid_blocks
                        ? std::max<uint64_t>(1, std::min<uint64_t>(p.grid_blocks, ceil_div(total, block)))
                        : cover_blocks(total, block, block, lds, static_cast<uint64_t>(blocks_per_cu(fn, block, lds)) * cu);
  if (blocks >= 8) blocks = std::min(ceil_div(blocks, 8) * 8, max_blocks(block));  // whole XCD rounds for the XCD-major chunk map
  const uint64_t groups = blocks % 8 == 0 ? 8 : 1;
  // a window's share of an XCD is rounded up to whole waves
  const uint64_t tiles = windows * ceil_div(ceil_div(window_max, groups) + kWave, block);
  GJ_REQUIRE(tiles + blocks < 0xFFFFFFFFull, GJ_ERR_INTERNAL, "too many tuple tiles");  // fewer than 2^32 tuples in all
  hipLaunchKernelGGL((lookup_tuples_kernel<Dev, K>), dim3(static_cast<unsigned>(blocks)), dim3(block), lds, s, d,
                     keys, start, windows, fan, static_cast<uint32_t>(tiles), res);
  GJ_HIP_CHECK(hipGetLastError());
}

constexpr int kBwsTile = 2048;

template <class Dev, class K>
void launch_bws(const Dev& d, const K* probes, uint64_t m, uint32_t* out, const gj_lookup_params& p, hipStream_t s,
                int cu, uint32_t skip) {
  if (m == 0) return;
  (void)lookup_block(p);  // a tile is shared by kBwsBlock threads, whatever valid block size is asked for
  const size_t lds = (d.lds_bytes() + 15) / 16 * 16 + kBwsTile * (sizeof(K) + sizeof(uint16_t)) +
                     kBwsBins * sizeof(uint16_t) + kBwsBlock / kWave * sizeof(uint32_t);
  uint32_t shift = 0;  // bins to at most kBwsBins
  while (((d.coarse_bins() - 1) >> shift) >= kBwsBins) ++shift;
  auto go = [&]<bool Link>() {
    auto kernel = &lookup_bws_kernel<Dev, K, kBwsTile, Link>;
    const void* fn = reinterpret_cast<const void*>(kernel);
    const uint64_t blocks = p.grid_blocks
                                ? std::max<uint64_t>(1, std::min<uint64_t>(p.grid_blocks, ceil_div(m, kBwsTile)))
                                : cover_blocks(m, kBwsTile, kBwsBlock, 0,
                                               static_cast<uint64_t>(blocks_per_cu(fn, kBwsBlock, lds)) * cu);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(kBwsBlock), lds, s, d, probes, m, shift, skip, out);
    GJ_HIP_CHECK(hipGetLastError());
  };
  // Up to two tiles in flight on a CU the link's queues stay short by themselves (2^22 probes, grids
  // of 512: 8.9 ms with all lanes, 9.0 with a quarter; with eight tiles on the chip a quarter of
  // the lanes takes twice as long).
  const uint64_t tiles = p.grid_blocks ? std::min<uint64_t>(p.grid_blocks, ceil_div(m, kBwsTile)) : ceil_div(m, kBwsTile);
  if (skip && tiles > 2ull * cu)
    go.template operator()<true>();
  else
    go.template operator()<false>();
}

void build_index(gj_index& ix, hipStream_t s);
template <class K> void build_btree(gj_index& ix, hipStream_t s);
template <class K> void build_extended(gj_index& ix, hipStream_t s);

// Binary search reads lines in buckets of more keys than this, and halves alone in smaller
// ones.  Lines cost instructions and registers and save dependent loads, so the line lies
// where a caller's waves are full and wait for those loads (halving -> lines, us):
//   lookups    2^22 probes, plain: buckets of 9 u32 keys 64 -> 55, of 9 u64 keys 100 -> 56
//   batches    in one persistent launch, 64 of 2000 probes: buckets of 64 u32 keys 23.6 -> 32.4, of
//              256 keys 26.8 -> 33.8; 64 of 64 to 70000: 65 u32 keys 66 -> 68, 257 keys 77 -> 68, 65 u64
//              keys 74 -> 63, 9 keys 57 -> 63.  As lookups where the launch has many (plan_lines_above):
//              8 of 2^20, 64 u32 keys 287 -> 138, 32 u64 keys 251 -> 149
//   aggregates one or two probes a wave (plain strategy, 30 M rows): buckets of 257 u32 keys 193
//              -> 206, of 409 keys 210 -> 208.  Whole waves, so agg_lines_above goes by the strategy:
//              lookup-first, 8 M rows: 17 keys 176 -> 173, 65 keys 198 -> 176, 409 keys 239 -> 184;
//              partitioned, 257 keys, 112 -> 117; lane refill and sorted by their rows: 257 keys and
//              1 M rows 12.6 -> 14.0 and 16.5 -> 17.5, 12 M 29.2 -> 28.1 and 41.7 -> 39.9, 30 M 59.5 ->
//              53.4 and 82.6 -> 83.1; lane refill in one persistent launch, 64 batches of 20000 rows
//              33.8 -> 35.6, of 300000 94.6 -> 93.6
//   tuples     as lookups, however few keys a partition has: its tuples share the lines of its keys
//              only where the keys spread evenly over the partitions (2^22 probes, windows of 2^20,
//              uniform keys of 2^18 u32 and fan-out 2^8 115 -> 119, 2^18 u64 and 2^10 138 -> 138; lognormal
//              ones 220 -> 127 and 239 -> 131, 2^22 u64 and 2^12 597 -> 224)
constexpr uint64_t kLinesLookups = 8, kLinesBatches = 128, kLinesAggregates = 512;

// Few probes over small buckets wait for the longest chain of loads, and halving's loads hit
// the L1 from the third last on: binary search of one batch goes by lines from this many
// halvings over all its probes on.  2^16 probes of 2^18 u64 keys 5.1 us, by lines 5.5; 2^17
// 8.2 and 6.7; 2^16 of 2^22 keys 9.7 and 7.2; 2^17 of 2^18 u32 keys 7.9 and 9.1.
constexpr uint64_t kLinesMinHalvings = 5ull << 18;
inline bool few_halvings(const gj_index& ix, uint64_t m) {
  return ix.kind == GJ_BINARY_SEARCH && m * ilog2_ceil(ix.sample_step) < kLinesMinHalvings;
}

// Columns shorter than a line are halved (ShortDev) in place of the window search.
template <class K>
bool short_column(const gj_index& ix) {
  const bool learned = ix.kind == GJ_LEARNED_PLR || ix.kind == GJ_LEARNED_MLP;
  return (ix.kind == GJ_RADIX_SPLINE || (learned && ix.lm_layout == GJ_LAYOUT_COLUMN)) && ix.n * sizeof(K) < 128;
}

template <class K>
ShortDev<K> short_dev(const gj_index& ix) {
  return {static_cast<const K*>(ix.d_col), ix.n};
}

// The same for all batches of a persistent launch, `probes` together.
constexpr uint64_t kLinesPlanHalvings = 5ull << 22;
inline uint64_t plan_lines_above(const gj_index& ix, uint64_t probes) {
  const bool many = ix.kind == GJ_BINARY_SEARCH && probes * ilog2_ceil(ix.sample_step) >= kLinesPlanHalvings;
  return many ? kLinesLookups : kLinesBatches;
}

// The same for a join-aggregate of `rows` fact rows in one launch.
constexpr uint64_t kLinesLookupFirst = 16, kLinesRowHalvings = 5ull << 24;
inline uint64_t agg_lines_above(const gj_index& ix, uint32_t strategy, uint64_t rows) {
  if (strategy == GJ_AGG_LOOKUP_FIRST) return kLinesLookupFirst;
  const bool many = ix.kind == GJ_BINARY_SEARCH && rows * ilog2_ceil(ix.sample_step) >= kLinesRowHalvings;
  const bool refills = strategy == GJ_AGG_LANE_REFILL || strategy == GJ_AGG_SORTED;
  return refills && many ? kLinesLookups : kLinesAggregates;
}

// Calls f(descriptor) with the device descriptor of the index (every kind).
template <class K, class F>
void with_index_dev(const gj_index& ix, F&& f, uint64_t lines_above = kLinesLookups) {
  if (short_column<K>(ix)) {
    f(short_dev<K>(ix));
    return;
  }
  switch (ix.kind) {
    case GJ_BINARY_SEARCH:
      if (ix.sample_step > lines_above)
        f(ix.bsearch_dev<K, true>());
      else
        f(ix.bsearch_dev<K, false>());
      return;
    case GJ_BTREE:
      if (ix.bt.node_bytes == 64)
        f(ix.btree_dev<K, 64>());
      else if (ix.bt.node_bytes == 256)
        f(ix.btree_dev<K, 256>());
      else
        f(ix.btree_dev<K>());
      return;
    case GJ_NO_OP: f(NoOpDev<K>{}); return;
    case GJ_HARMONIA:
      f(ix.harmonia_dev<K>());
      return;
    case GJ_RADIX_SPLINE:
      if (ix.rs_mode == kRsRadixLds)
        f(ix.rs_dev<K, kRsRadixLds>());
      else if (ix.rs_mode == kRsSamples)
        f(ix.rs_dev<K, kRsSamples>());
      else
        f(ix.rs_dev<K, kRsRadix>());
      return;
    case GJ_LEARNED_PLR:
    case GJ_LEARNED_MLP:
      if (ix.lm_layout == GJ_LAYOUT_LINES)
        f(ix.lines_dev<K>());
      else if (ix.lm_compact)
        f(ix.learned_compact_dev<K>());
      else if (ix.lm_fallback_any)
        f(ix.learned_dev<K, kLeafInline>());
      else
        f(ix.learned_dev<K, kLeafNoFallback>());
      return;
    case GJ_HASH: f(ix.hash_dev<K>()); return;
  }
  throw error(GJ_ERR_INVALID, "unknown index kind");
}

// Hash table over the column into `table` (capacity written to cap); temp: working
// memory of the partitioned build (grown as needed).
template <class K>
void build_hash_table(const gj_index& ix, dbuf& table, uint64_t& cap, dbuf& temp, hipStream_t s);
uint64_t hash_capacity(uint64_t n);

// Radix partitioner (partition.hip).  stable: input order kept inside every
// partition; otherwise the order inside a partition is arbitrary.  start2 (optional)
// receives a second copy of the 2^bits partition starts.  hashed: the keys' hashes
// (key_hash) are partitioned and written in their place.
uint64_t partition_capacity(uint64_t m, int key_bytes, uint32_t bits);
uint64_t partition_scratch(uint64_t m, int key_bytes, uint32_t bits, uint32_t passes);
// A batch of m probes cut into windows of `window`, each window partitioned on its own
// (output partition w * 2^bits + digit).  No payloads: inv1[i] is where probe i went;
// when windows_two_pass(), that is a position in the first pass's output, and
// inv2[inv1[i]] its final position (inv2 is null otherwise).  inv1 and inv2 hold m
// entries each.
uint64_t windows_capacity(uint64_t m, uint64_t window, int key_bytes, uint32_t bits);
// what of it the tuples, padding included, can take (each tuple pads one partition at most)
uint64_t windows_tuples(uint64_t m, uint64_t window, int key_bytes, uint32_t bits);
uint64_t windows_scratch(uint64_t m, uint64_t window, int key_bytes, uint32_t bits, uint32_t passes);
bool windows_two_pass(uint32_t bits, uint32_t passes);
template <class K>
void partition_windows(const K* keys, uint64_t m, uint64_t window, uint32_t bits, uint32_t ignore, uint32_t passes,
                       K* out_keys, uint32_t* inv1, uint32_t* inv2, uint64_t* start, uint64_t* count,
                       uint8_t* scratch, unsigned long long* dropped, hipStream_t s);
template <class K>
void partition_keys(const K* keys, uint64_t m, uint32_t payload_base, uint32_t bits, uint32_t ignore, uint32_t passes,
                    bool stable, K* out_keys, uint32_t* out_payload, uint64_t* start, uint64_t* count, uint8_t* scratch,
                    unsigned long long* dropped, int cu, hipStream_t s, uint64_t* start2 = nullptr,
                    bool hashed = false);

// Bytes of index-private device memory held by the extended kinds.
uint64_t extended_memory(const gj_index& ix);

// Drivers (drivers.hip)
void lookup_dispatch(const gj_index& ix, const void* probes, uint64_t m, uint32_t* out, const gj_lookup_params& p,
                     hipStream_t s);

}  // namespace gj
