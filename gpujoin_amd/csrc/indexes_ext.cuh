// indexes_ext.cuh - device descriptors of Harmonia, RadixSpline, the learned
// two-stage models and the hash table (same contract as indexes.cuh).
#pragma once

#include "device.cuh"
#include "indexes.cuh"

namespace gj {

// ---------------------------------------------------------------------------
// Harmonia (harmonia_index, src/indexes.cuh:257-307; harmonia_tree,
// src/harmonia.cuh:48-992).  Layout kept from the reference: 32 keys per node
// (fanout 33), inner keys breadth first and padded with key_max, leaf keys =
// the column, next = children[pos] + lb (src/harmonia.cuh:748-766).  Re-laid
// out for CDNA4: the build fills every node of a level but the last, so the
// reference's children[] prefix sums have a closed form,
//   children[node p of inner level l] = first[l + 1] + 33 (p - first[l]),
// which the lookup computes instead of reading a 4-byte entry per level (at
// 2^26 keys a 16.5 MiB array whose bottom-level reads miss L2); the top key
// levels sit in LDS (the reference uses 42 KiB of __constant__,
// src/harmonia.cuh:45-46); a node is searched by quads a 128-byte line at a time, a u64
// node's second line only for probes above every key of the first (the reference's early
// exit, src/harmonia.cuh:581-589).
//
// What bounds it: VALU issue while the nodes are in L2, then fabric lines.  Groups of 8, 16
// or 32 lanes with a ballot and a population count per key took about three times the
// instructions; harmonia_group_lanes is checked as before and changes nothing any more.
// 2^24 probes, groups of 8 -> quads: 2^14 u64 keys 405 -> 213 us,
// 2^20 u64 540 -> 355, 2^20 u32 391 -> 216, 2^22 u64 658 -> 477.
// ---------------------------------------------------------------------------
template <class K>
struct HarmoniaDev {
  using L = QuadLine<K, 128>;
  static constexpr int MK = 32;                                   // keys per node
  static constexpr uint32_t LK = L::kKeys;                        // keys per 128-byte line
  static constexpr uint32_t LINES = MK / LK;                      // 2 (u64) or 1 (u32)

  const K* col;
  uint64_t n;
  const K* keys;              // inner nodes x MK
  uint64_t inner_nodes;
  uint32_t depth;             // levels including the leaf level
  uint32_t lds_levels;        // top inner levels staged in LDS
  uint64_t lds_nodes;
  uint64_t first[kMaxLevels];  // first node of level l (top = 0); first[depth - 1] = inner_nodes

  __host__ __device__ size_t lds_bytes() const { return lds_nodes * MK * sizeof(K); }
  __device__ void stage(uint8_t* lds) const {
    if (lds_nodes) stage_to_lds(lds, keys, lds_bytes());
  }

  // keys of the lowest staged level below x
  __device__ __forceinline__ uint32_t coarse(K x, const uint8_t* lds) const {
    if (lds_levels == 0) return 0;
    const K* s = reinterpret_cast<const K*>(lds) + first[lds_levels - 1] * MK;
    uint32_t at = 0;
    for (uint32_t len = coarse_bins() - 1; len > 1;) {  // kernel-uniform
      const uint32_t half = len >> 1;
      at = s[at + half - 1] < x ? at + half : at;
      len -= half;
    }
    return at + (s[at] < x ? 1u : 0u);
  }
  __host__ __device__ uint32_t coarse_bins() const {
    return lds_levels ? static_cast<uint32_t>(lds_nodes - first[lds_levels - 1]) * MK + 1 : 1u;
  }

  // Keys of each lane's node below its probe; eq (leaves): the node holds the probe.
  template <bool Leaf>
  __device__ __forceinline__ uint32_t node_search(const K* base, uint32_t node, const QuadProbes<K>& q, int ql,
                                                  bool& eq) const {
    const K* lane_base = base + ql * L::kLaneKeys;
    const uint32_t line = node * LINES;  // fewer than 2^32 keys, hence lines
    L ln[kQuad];
    quad_rounds([&](auto r) { ln[r].load(lane_base, quad_bcast<r>(line)); });
    uint32_t below = quad_below(ln, q, ql);
    if constexpr (Leaf) eq = quad_holds(ln, q, ql);
    if constexpr (LINES == 2) {
      const bool more = below == LK;
      if (ballot(more) != 0) {  // wave-uniform
        const uint32_t rounds = quad_or(more ? 1u << ql : 0u);
        quad_rounds([&](auto r) {
          const uint32_t l = quad_bcast<r>(line);
          if ((rounds >> r) & 1u) ln[r].load(lane_base, l + 1);
        });
        const uint32_t rest = quad_below(ln, q, ql);
        below += more ? rest : 0u;
        if constexpr (Leaf) {
          const bool e = quad_holds(ln, q, ql);
          eq = more ? e : eq;
        }
      }
    }
    return below;
  }

  __device__ __forceinline__ uint32_t lookup(K x, bool active, const uint8_t* lds) const {
    const int ql = lane() & (kQuad - 1);
    const QuadProbes<K> q(x);
    bool live = active;
    bool eq = false;
    uint32_t pos = 0;  // fewer than 2^32 nodes
    uint32_t d = 0;
    const K* lds_keys = reinterpret_cast<const K*>(lds);
    auto step = [&](const K* from) {
      const uint32_t lb = node_search<false>(from, pos, q, ql, eq);
      const uint32_t f = static_cast<uint32_t>(first[d]), next = static_cast<uint32_t>(first[d + 1]);
      pos = live ? next + 33u * (pos - f) + lb : 0u;
    };
    for (; d < lds_levels; ++d) step(lds_keys);
    for (; d + 1 < depth; ++d) step(keys);
    const uint32_t leaf = live ? pos - static_cast<uint32_t>(inner_nodes) : 0u;
    const uint32_t lb = node_search<true>(col, leaf, q, ql, eq);
    return (live && eq) ? leaf * MK + lb : kNotFound;
  }
};

// ---------------------------------------------------------------------------
// Last-mile window search shared by RadixSpline and the learned models.
// Each lane's probe has a predicted position `pred` and a window [lo, hi) of
// the column that holds the key if it is present.  Quads read whole 128-byte
// lines (QuadLine); a quad serves its 4 probes in 4 rounds.  A round starts at
// the line holding pred and walks one line left or right until the line brackets
// the probe or leaves the window.  The search runs in phases: in each phase every
// unresolved round of every quad requests its next line before any line is
// examined, so a wave pays one memory latency per phase (one, occasionally two or
// three) rather than one per walking round.
//
// A round's line is sorted, so the owning lane only needs how many of its keys are
// below the probe (the in-line offset of the probe's lower bound) and whether the
// line holds it.  The owning lane alone holds its probe's state (line and window; a step
// to one side takes the other side's part of the window away), which keeps the registers
// per lane, and hence the waves per SIMD, where a latency-bound search needs them.
// Positions are 32-bit (n < 2^32); the column holds a line at least.
// ---------------------------------------------------------------------------
template <class K>
__device__ __forceinline__ uint32_t group_window_search(const K* col, uint64_t n, uint32_t my_pred, uint32_t my_lo,
                                                        uint32_t my_hi, K my_x, bool my_live) {
  using L = QuadLine<K, 128>;
  constexpr uint32_t LK = L::kKeys;
  const int ql = lane() & (kQuad - 1);
  const QuadProbes<K> q(my_x);
  const K* lane_base = col + ql * L::kLaneKeys;
  bool open = my_live && my_lo < my_hi;
  uint32_t line = 0, found = kNotFound;
  if (open) {
    const uint32_t p = my_pred < my_lo ? my_lo : (my_pred >= my_hi ? my_hi - 1 : my_pred);
    line = p / LK;
  }
  while (const uint64_t lanes = ballot(open)) {  // wave-uniform exit
    const uint32_t rounds = quad_or(open ? 1u << ql : 0u), base = line_at<LK>(line, n);
    L ln[kQuad];
    quad_rounds([&](auto r) { ln[r].any(); });
    quad_rounds([&](auto r) {
      const uint32_t at = quad_bcast<r>(base);
      if ((rounds >> r) & 1u) ln[r].load_keys(lane_base, at);
    });
    const uint32_t below = quad_below(ln, q, ql, lanes);
    const bool eq = quad_holds(ln, q, ql, lanes);
    if (open) {
      if (eq) {
        found = base + below;  // the line holds x at its lower-bound offset
        open = false;
      } else if (below == LK && my_hi - base > LK) {
        ++line;  // every key of the line is below x, and the window goes on to the right
        my_lo = 0xFFFFFFFFu;  // and not back to the left
      } else if (below == 0 && base > my_lo) {
        --line;  // no key of the line is below x, and the window begins further left
        my_hi = base;
      } else {
        open = false;  // x falls between two window keys (or past the window): absent
      }
    }
  }
  return found;
}

// ---------------------------------------------------------------------------
// RadixSpline (radix_spline_index, src/indexes.cuh:176-248; estimate
// src/rs.cuh:118-154).  Knots are {u64 key, f64 position} pairs, 16 bytes, like
// the reference's Coord (src/rs.cuh:38-52): the two knots around a probe are 32
// contiguous bytes, read by two 16-byte loads issued together.  The radix table
// is staged in LDS when it fits the rs_lds_bits budget (Lds = true: up to 2^13 + 2
// entries, 32 KiB, by default), else read from global memory (the reference's 18
// bits are 1 MiB).  A coarser table in LDS is possible (every 2^d-th entry of a
// 2^b-entry table is the table for b - d bits, since entry p is the first knot whose
// prefix is >= p), but it widens the knot search: at 2^26 keys, 13 bits in LDS ran
// at 18.6 G lookups/s against 23.8 for 18 bits in global memory.  The estimate is
// the reference's FP64 interpolation with an explicit fma, and the last mile is the
// line-walking window search over [est - err, est + err + 2).
// ---------------------------------------------------------------------------
struct RsKnot {
  uint64_t x;
  double y;
};
static_assert(sizeof(RsKnot) == 16, "16-byte knot");

// How a lookup finds the knots around its probe.
enum : int {
  kRsRadix = 0,     // radix table in global memory, then halving over the prefix's knots
  kRsRadixLds = 1,  // the same with the table staged in LDS
  kRsSamples = 2    // the largest key of every group of knots in LDS, then halving over the
                    // group: where the keys crowd under few prefixes, each halving being a
                    // dependent gather (2^24 probes of 2^22 lognormal keys, 6.0 halvings a key under
                    // the table, 2 in a group: 596 -> 518 us; 2^18 clustered, 3.4 and 0: 349 ->
                    // 304; with evenly spread keys the table is better: 2^24 keys 582, sampled
                    // 652)
};
constexpr uint32_t kRsSampleCount = 1024;

template <class K, int Mode = kRsRadix>
struct RadixSplineDev {
  static constexpr bool Lds = Mode == kRsRadixLds;
  const K* col;
  uint64_t n;
  const uint32_t* radix;  // radix table over the top bits of key - min_key
  uint32_t radix_count;   // entries
  const RsKnot* knots;
  K min_key, max_key;
  uint32_t shift_bits;    // prefix = (key - min_key) >> shift_bits
  uint32_t err;  // search bound (>= the builder's bound; widened at build until every key is inside)
  const K* samples;       // kRsSamples: kRsSampleCount group maxima, key_max past the last
  uint32_t group;         // knots per group
  uint32_t num_knots;

  __host__ __device__ size_t lds_bytes() const {
    if constexpr (Mode == kRsSamples) return sizeof(K) * kRsSampleCount;
    return Lds ? (static_cast<size_t>(radix_count) * 4 + 15) / 16 * 16 : 0;
  }
  __device__ void stage(uint8_t* lds) const {
    if constexpr (Lds) stage_to_lds(lds, radix, lds_bytes());
    if constexpr (Mode == kRsSamples) stage_to_lds(lds, samples, lds_bytes());
  }

  // the radix prefix, or the group of knots
  __device__ __forceinline__ uint32_t coarse(K x, const uint8_t* lds) const {
    if constexpr (Mode == kRsSamples) return samples_below(x, reinterpret_cast<const K*>(lds));
    const K c = x < min_key ? min_key : (x > max_key ? max_key : x);
    return static_cast<uint32_t>(static_cast<uint64_t>(c - min_key) >> shift_bits);
  }
  __host__ __device__ uint32_t coarse_bins() const {
    return Mode == kRsSamples ? kRsSampleCount + 1 : radix_count;
  }

  // group maxima below x
  __device__ __forceinline__ static uint32_t samples_below(K x, const K* s) {
    uint32_t b = 0;
#pragma unroll
    for (uint32_t h = kRsSampleCount / 2; h > 0; h >>= 1) b = (s[b + h - 1] < x) ? b + h : b;
    return b + (s[b] < x ? 1u : 0u);
  }

  // tab: the radix table, or the samples (LDS during lookups, the table in global memory at build)
  __device__ __forceinline__ double estimate(K x, const void* tab) const {
    if (x <= min_key) return 0.0;
    if (x >= max_key) return static_cast<double>(n - 1);
    uint32_t lower, count;  // fewer than 2^32 knots
    if constexpr (Mode == kRsSamples) {  // x < max_key, the last knot's key: some group holds it
      lower = samples_below(x, static_cast<const K*>(tab)) * group;
      count = lower + group < num_knots ? group : num_knots - lower;
    } else {
      const uint32_t* t = static_cast<const uint32_t*>(tab);
      const uint64_t prefix = static_cast<uint64_t>(x - min_key) >> shift_bits;
      lower = t[prefix];
      count = t[prefix + 1] - lower;
    }
    while (count > 0) {
      const uint32_t step = count >> 1, mid = lower + step;
      if (static_cast<K>(knots[mid].x) < x) {
        lower = mid + 1;
        count -= step + 1;
      } else {
        count = step;
      }
    }
    const RsKnot a = knots[lower - 1], b = knots[lower];
    // differences of keys fit K
    const double slope = (b.y - a.y) / static_cast<double>(static_cast<K>(b.x - a.x));
    return __builtin_fma(static_cast<double>(static_cast<K>(static_cast<uint64_t>(x) - a.x)), slope, a.y);
  }

  // [lo, hi): positions are below 2^32, so 32-bit conversions (one instruction, where a
  // 64-bit one takes a dozen in FP64) cut the same whole numbers
  __device__ __forceinline__ void window(double est, uint32_t& lo, uint32_t& hi) const {
    const double e = static_cast<double>(err);
    lo = (est < e) ? 0 : static_cast<uint32_t>(est - e);
    hi = (est + e + 2.0 > static_cast<double>(n)) ? static_cast<uint32_t>(n) : static_cast<uint32_t>(est + e + 2.0);
    if (lo > hi) lo = hi;
  }

  __device__ __forceinline__ uint32_t lookup(K x, bool active, const uint8_t* lds) const {
    uint32_t lo = 0, hi = 0, pred = 0;
    if (active) {
      const double est = estimate(x, Mode == kRsRadix ? static_cast<const void*>(radix) : lds);
      window(est, lo, hi);
      pred = static_cast<uint32_t>(est);
    }
    return group_window_search<K>(col, n, pred, lo, hi, x, active);
  }
};

// ---------------------------------------------------------------------------
// Learned two-stage position model (no reference counterpart).
//   root:  cdf = root(x), x = (key - min_key) / (max_key - min_key) in FP32;
//          linear (a*x + b), a monotone 1xH MLP with ramp units
//          clamp(w1*x + b1, 0, 1) (w1, w2 >= 0), or an error-bounded spline of
//          the column's CDF (any key distribution); leaf = floor(cdf * L)
//   leaf:  pred = start + floor(slope * dkey) in FP32, dkey = key - leaf base key
//          (the fit's intercept is folded into start); one 16-byte load.
//   window: [pred + err_lo, pred + err_hi], with err_lo/err_hi the extremes of
//          the error of every build key under this exact FP32 code, over all
//          leaves.  The window only caps the walk: a walk from any line stops
//          at the line that brackets the probe.  Leaves whose own error range
//          exceeds the bound go to the B-tree (slope = NaN).
// Keeping the leaf at 16 bytes halves the leaf table, which keeps more of it
// in L2 while the column lines stream through.
// ---------------------------------------------------------------------------
struct LeafModel {  // 16 bytes
  uint64_t base_key;  // first key routed to the leaf (0 for an empty leaf)
  uint32_t start;     // position of base_key plus the rounded intercept, clamped to [0, n]
  float slope;        // NaN: the leaf's probes are looked up in the B-tree
};
static_assert(sizeof(LeafModel) == 16, "leaf model is 16 bytes");

// Compact leaves (8 bytes) for roots that spread the keys evenly (linear or MLP
// root, every leaf within the error bound, no split leaf; 2^22 keys or more, the
// default leaf count): twice the leaves in
// the same table, so a smaller window and fewer column lines per lookup.  The
// key offset is taken from a group base shared by 2^gshift leaves (at most 512
// groups, 16 bytes each, staged in LDS) instead of the leaf's own base key:
//   pred = group.start + floor(fma(slope, f32(key - group.base_key), icpt))
// The build measures every key's error under exactly this arithmetic, so a
// leaf whose FP32 offsets lose precision only widens the bounds; if any leaf
// then exceeds the bound the build keeps the 16-byte leaves.
struct LeafCompact {  // 8 bytes
  float slope;
  float icpt;  // positions past group.start at key == group.base_key
};
static_assert(sizeof(LeafCompact) == 8, "compact leaf is 8 bytes");

struct LeafGroup {  // 16 bytes
  uint64_t base_key;  // key at start (the last key for a group past the column's end)
  uint32_t start;     // first position routed to the group's first leaf or later
  uint32_t pad;
};
static_assert(sizeof(LeafGroup) == 16, "leaf group is 16 bytes");

constexpr int kMaxHidden = 64;

struct RootModel {
  float a, b;                 // linear root
  float inv_range;            // 1 / (max_key - min_key) in FP32
  uint32_t hidden;            // > 0: MLP root
  const float* mlp;           // [w1(h), b1(h), w2(h), b2] in global memory (staged in LDS)
  uint32_t segments;          // > 0: spline root with this many segments (a power of two; the
                              // knots past the last real one repeat it)
  const uint64_t* knots;      // spline arrays in global memory (staged in LDS):
                              // key[segments + 1] u64 | cdf[segments + 1] f32 | slope[segments] f32

  __host__ __device__ size_t key_bytes() const { return ((static_cast<size_t>(segments) + 1) * 8 + 15) / 16 * 16; }
  __host__ __device__ size_t cdf_bytes() const { return ((static_cast<size_t>(segments) + 1) * 4 + 15) / 16 * 16; }
  __host__ __device__ size_t bytes() const {
    if (hidden) return ((3 * hidden + 1) * 4 + 15) / 16 * 16;
    if (segments) return key_bytes() + cdf_bytes() + (static_cast<size_t>(segments) * 4 + 15) / 16 * 16;
    return 0;
  }
  __host__ __device__ const void* params() const { return hidden ? static_cast<const void*>(mlp) : knots; }
};

// Spline root: the segment s with key[s] <= x < key[s + 1] by a branch-free
// binary search, then cdf = cdf[s] + (x - key[s]) * slope[s], kept inside
// [cdf[s], cdf[s + 1]].  Monotone in the key, so every leaf still owns a
// contiguous key range.  The knots come from an error-bounded greedy spline over
// (key, position / n), so a segment never spans a gap that the keys jump across.
__device__ __forceinline__ float spline_cdf(uint64_t x, const uint8_t* base, const RootModel& r) {
  const uint64_t* key = reinterpret_cast<const uint64_t*>(base);
  const float* cdf = reinterpret_cast<const float*>(base + r.key_bytes());
  const float* slope = reinterpret_cast<const float*>(base + r.key_bytes() + r.cdf_bytes());
  uint32_t s = 0;
  for (uint32_t step = r.segments >> 1; step > 0; step >>= 1) s = (key[s + step] <= x) ? s + step : s;
  const float d = x >= key[s] ? static_cast<float>(x - key[s]) : 0.0f;
  const float c = __builtin_fmaf(d, slope[s], cdf[s]);
  return fminf(fmaxf(c, cdf[s]), cdf[s + 1]);
}

__device__ __forceinline__ float mlp_eval(const float* p, uint32_t h, float x) {
  float f = p[3 * h];
  for (uint32_t j = 0; j < h; ++j) {
    const float a = __builtin_fmaf(p[j], x, p[h + j]);
    f = __builtin_fmaf(p[2 * h + j], fminf(fmaxf(a, 0.0f), 1.0f), f);
  }
  return f;
}

template <class K>
__device__ __forceinline__ float key_unit(K key, K min_key, float inv_range) {
  return static_cast<float>(static_cast<uint64_t>(key - min_key)) * inv_range;
}

__device__ __forceinline__ uint32_t leaf_of(float cdf, uint32_t leaves) {
  float l = cdf * static_cast<float>(leaves);
  l = l < 0.0f ? 0.0f : l;
  uint32_t li = static_cast<uint32_t>(l);
  return li >= leaves ? leaves - 1 : li;
}

// signed FP32 distance of key from the leaf's base key
template <class K>
__device__ __forceinline__ float leaf_dkey(K key, uint64_t base) {
  const uint64_t k = static_cast<uint64_t>(key);
  return k >= base ? static_cast<float>(k - base) : -static_cast<float>(base - k);
}

__device__ __forceinline__ int64_t leaf_pred(const LeafModel& m, float dkey) {
  float p = m.slope * dkey;
  p = fminf(fmaxf(p, -2.0e9f), 2.0e9f);
  return static_cast<int64_t>(m.start) + static_cast<int64_t>(floorf(p));
}

__device__ __forceinline__ int64_t compact_pred(const LeafCompact& m, const LeafGroup& g, float dkey) {
  float p = __builtin_fmaf(m.slope, dkey, m.icpt);
  p = fminf(fmaxf(p, -2.0e9f), 2.0e9f);
  return static_cast<int64_t>(g.start) + static_cast<int64_t>(floorf(p));
}

// The leaf a key is routed to by the root (whose parameters are staged at rp).
template <class K>
__device__ __forceinline__ uint32_t route_leaf(K x, const uint8_t* rp, const RootModel& root, K min_key,
                                               uint32_t leaves) {
  float cdf;
  if (root.segments) {
    cdf = spline_cdf(static_cast<uint64_t>(x), rp, root);
  } else if (root.hidden) {
    cdf = mlp_eval(reinterpret_cast<const float*>(rp), root.hidden, key_unit(x, min_key, root.inv_range));
  } else {
    cdf = __builtin_fmaf(root.a, key_unit(x, min_key, root.inv_range), root.b);
  }
  return leaf_of(cdf, leaves);
}

// How probes of leaves routed to the B-tree are answered:
//   kLeafNoFallback  no such leaf exists; the kernel carries no B-tree code
//   kLeafInline      the B-tree lookup runs inside the same kernel
//   kLeafMark        the probe's result is kFallbackMark; a second kernel of the
//                    plain driver scans the results and answers the marked probes
//                    with the B-tree, so the hot kernel keeps the no-fallback
//                    register count (used while few keys sit in fallback leaves)
constexpr int kLeafNoFallback = 0;
constexpr int kLeafInline = 1;
constexpr int kLeafMark = 2;
constexpr uint32_t kFallbackMark = 0xFFFFFFFEu;  // never a row id: n < 2^32 - 1

// A leaf whose keys no line fits within the bound is split into kSplitWays
// equal-count sub-leaves: the leaf's model holds slope = NaN and start = the
// split's index j; separator line j holds the max key of each sub-leaf (the last
// = all ones), and the number of separators below the probe picks the sub-leaf.
// A sub-leaf that is still too wide (slope = NaN) routes to the B-tree, as does a
// leaf with slope = NaN and start = kNoSplit.
constexpr uint32_t kSplitWays = 16;
constexpr uint32_t kNoSplit = 0xFFFFFFFFu;

template <class K, int Mode>
struct LearnedDev {
  static constexpr bool FB = Mode == kLeafInline;
  const K* col;
  uint64_t n;
  K min_key, max_key;
  RootModel root;
  const LeafModel* leaves;
  uint32_t num_leaves;
  int32_t err_lo, err_hi;  // window [pred + err_lo, pred + err_hi]
  uint32_t num_splits;     // split leaves
  const uint64_t* seps;    // num_splits separator lines of kSplitWays keys
  const LeafModel* subs;   // num_splits x kSplitWays sub-leaf models
  BTreeDev<K> btree;       // fallback (used when FB)

  __host__ __device__ size_t root_offset() const { return FB ? btree.lds_bytes() : 0; }
  __host__ __device__ size_t lds_bytes() const { return root_offset() + root.bytes(); }
  __device__ void stage(uint8_t* lds) const {
    if constexpr (FB) btree.stage(lds);
    if (root.bytes()) stage_to_lds(lds + root_offset(), root.params(), root.bytes());
  }

  __device__ __forceinline__ uint32_t route(K x, const uint8_t* lds) const {
    return route_leaf<K>(x, lds + root_offset(), root, min_key, num_leaves);
  }
  __device__ __forceinline__ uint32_t coarse(K x, const uint8_t* lds) const {  // the leaf
    return route(x < min_key ? min_key : (x > max_key ? max_key : x), lds);
  }
  __host__ __device__ uint32_t coarse_bins() const { return num_leaves; }

  __device__ __forceinline__ uint32_t lookup(K x, bool active, const uint8_t* lds) const {
    bool use_tree = false, split = false;
    uint64_t lo = 0, hi = 0, pred = 0;
    bool live = active && x >= min_key && x <= max_key;
    LeafModel m{};
    if (live) {
      m = leaves[route(x, lds)];
      if (__builtin_isnan(m.slope)) {
        if (m.start != kNoSplit) split = true;
        else use_tree = true;  // only with fallback leaves (Mode != kLeafNoFallback)
      }
    }
    if (num_splits && ballot(split) != 0) {  // wave-uniform
      // separators below the probe in its leaf's line (the lanes without a split read line 0)
      const uint32_t t = quad_count_less<uint64_t, 128>(seps, split ? m.start : 0u,
                                                        QuadProbes<uint64_t>(static_cast<uint64_t>(x)),
                                                        lane() & (kQuad - 1));
      if (split) {
        m = subs[static_cast<uint64_t>(m.start) * kSplitWays + (t < kSplitWays ? t : kSplitWays - 1)];
        use_tree = __builtin_isnan(m.slope);
      }
    }
    if (live) {
      if (!use_tree) {
        const int64_t p = leaf_pred(m, leaf_dkey(x, m.base_key));
        int64_t a = p + err_lo, b = p + err_hi + 1;
        a = a < 0 ? 0 : a;
        b = b > static_cast<int64_t>(n) ? static_cast<int64_t>(n) : b;
        if (a < b) {
          lo = static_cast<uint64_t>(a);
          hi = static_cast<uint64_t>(b);
          pred = static_cast<uint64_t>(p < a ? a : (p >= b ? b - 1 : p));
        }
      }
    }
    uint32_t r = group_window_search<K>(col, n, static_cast<uint32_t>(pred), static_cast<uint32_t>(lo),
                                        static_cast<uint32_t>(hi), x, live && !use_tree);
    if constexpr (Mode == kLeafInline) {
      if (ballot(use_tree) != 0) {  // wave-uniform
        const uint32_t t = btree.lookup(x, use_tree, lds);
        if (use_tree) r = t;
      }
    } else if constexpr (Mode == kLeafMark) {
      if (use_tree) r = kFallbackMark;
    }
    return r;
  }
};

// The learned index with compact leaves: no fallback and no split leaf exist.
template <class K>
struct LearnedCompactDev {
  const K* col;
  uint64_t n;
  K min_key, max_key;
  RootModel root;
  const LeafCompact* leaves;
  const LeafGroup* groups;  // num_groups entries, staged in LDS after the root
  uint32_t num_leaves, gshift, num_groups;
  int32_t err_lo, err_hi;  // window [pred + err_lo, pred + err_hi]

  __host__ __device__ size_t group_offset() const { return (root.bytes() + 15) / 16 * 16; }
  __host__ __device__ size_t lds_bytes() const {
    return group_offset() + static_cast<size_t>(num_groups) * sizeof(LeafGroup);
  }
  __device__ void stage(uint8_t* lds) const {
    if (root.bytes()) stage_to_lds(lds, root.params(), root.bytes());
    stage_to_lds(lds + group_offset(), groups, static_cast<size_t>(num_groups) * sizeof(LeafGroup));
  }
  __device__ __forceinline__ uint32_t coarse(K x, const uint8_t* lds) const {  // the leaf
    return route_leaf<K>(x < min_key ? min_key : (x > max_key ? max_key : x), lds, root, min_key, num_leaves);
  }
  __host__ __device__ uint32_t coarse_bins() const { return num_leaves; }

  __device__ __forceinline__ uint32_t lookup(K x, bool active, const uint8_t* lds) const {
    uint64_t lo = 0, hi = 0, pred = 0;
    const bool live = active && x >= min_key && x <= max_key;
    if (live) {
      const uint32_t l = route_leaf<K>(x, lds, root, min_key, num_leaves);
      const LeafCompact m = leaves[l];
      const LeafGroup g = reinterpret_cast<const LeafGroup*>(lds + group_offset())[l >> gshift];
      const int64_t p = compact_pred(m, g, leaf_dkey(x, g.base_key));
      int64_t a = p + err_lo, b = p + err_hi + 1;
      a = a < 0 ? 0 : a;
      b = b > static_cast<int64_t>(n) ? static_cast<int64_t>(n) : b;
      if (a < b) {
        lo = static_cast<uint64_t>(a);
        hi = static_cast<uint64_t>(b);
        pred = static_cast<uint64_t>(p < a ? a : (p >= b ? b - 1 : p));
      }
    }
    return group_window_search<K>(col, n, static_cast<uint32_t>(pred), static_cast<uint32_t>(lo),
                                  static_cast<uint32_t>(hi), x, live);
  }
};

// ---------------------------------------------------------------------------
// Learned index, lines layout (no reference counterpart).  The index keeps its
// own copy of the keys in 128-byte lines.  The model assigns every key a target
// line (monotone in the key); line t holds, in key order, the keys assigned to
// it, after any keys an earlier full line pushed on to it, up to CAP keys; what
// does not fit moves on to line t + 1.  So a key sits in its target line or,
// only behind a run of full lines, a few lines later, and the layout stays in
// global key order.  Each line starts with an 8-byte header {row id of its first
// key, key count}; the row id of a key is header.base + its rank in the line.
//
// Lookup: read the target line; the key is there, or absent, unless every key of
// the line is below the probe and the line is full, in which case the next line
// is read.  A probe below its target line's keys is absent (every key assigned
// to an earlier line is smaller, and no key moves backwards).
//
// Targets:
//   root only   target = umulhi(key - min_key, mult): the keys' range spread
//               linearly over the lines in fixed point (exact integer arithmetic)
//   two-stage   a root model (linear, MLP or CDF spline, staged in LDS) picks a
//               leaf; the leaf maps its key span linearly onto its own run of
//               lines: target = line0 + floor(f32(key - key0) * scale).  Leaves
//               own disjoint, ordered key ranges and line runs, so the target is
//               monotone; the build evaluates the same device code.
// ---------------------------------------------------------------------------
struct LineLeaf {  // 16 bytes
  uint64_t key0;   // first build key routed to the leaf (0 for an empty leaf)
  uint32_t line0;  // first target line of the leaf
  float scale;     // target lines per key unit over the leaf's key span
};
static_assert(sizeof(LineLeaf) == 16, "line leaf is 16 bytes");

// One descriptor serves both targets: a root-only specialisation compiled to one more
// VGPR on gfx950 (73), which costs a wave per SIMD (7 -> 6) and 3 % of the rate.
template <class K>
struct LinesDev {
  static constexpr uint32_t SLOTS = 128 / sizeof(K);  // K-sized slots per line
  static constexpr uint32_t HDR = 8 / sizeof(K);      // slots of the {base, count} header
  static constexpr uint32_t CAP = SLOTS - HDR;        // keys per line: 15 (u64), 30 (u32)
  const K* lines;  // num_lines x SLOTS
  uint64_t num_lines;
  K min_key, max_key;
  uint64_t mult;            // root only: target = umulhi(key - min_key, mult)
  RootModel root;           // two-stage: routes to a leaf
  const LineLeaf* leaves;   // nullptr: root only
  uint32_t num_leaves;

  // The root's parameters (MLP weights, spline knots) are staged in LDS.  Reading them
  // in place instead (a generic pointer that may be global) costs a third of the
  // two-stage lookup rate: flat loads make every memory wait in the kernel conservative.
  __host__ __device__ size_t lds_bytes() const { return leaves ? root.bytes() : 0; }
  __device__ void stage(uint8_t* lds) const {
    if (lds_bytes()) stage_to_lds(lds, root.params(), root.bytes());
  }

  __device__ __forceinline__ uint32_t coarse(K x, const uint8_t* lds) const {  // the leaf, or the line
    const K c = x < min_key ? min_key : (x > max_key ? max_key : x);
    if (leaves) return route_leaf<K>(c, lds, root, min_key, num_leaves);
    return static_cast<uint32_t>(__umul64hi(static_cast<uint64_t>(c - min_key), mult));
  }
  __host__ __device__ uint32_t coarse_bins() const {
    return leaves ? num_leaves : static_cast<uint32_t>(num_lines);
  }

  // rp: the root's parameters (LDS during lookups, global memory at build)
  __device__ __forceinline__ uint64_t target(K x, const uint8_t* rp) const {
    const uint64_t off = static_cast<uint64_t>(x - min_key);
    if (!leaves) return __umul64hi(off, mult);
    const LineLeaf f = leaves[route_leaf<K>(x, rp, root, min_key, num_leaves)];
    float p = leaf_dkey(x, f.key0) * f.scale;
    p = fminf(fmaxf(p, 0.0f), 2.0e9f);
    return static_cast<uint64_t>(f.line0) + static_cast<uint64_t>(floorf(p));
  }

  __device__ __forceinline__ uint32_t lookup(K x, bool active, const uint8_t* lds) const {
    const bool live = active && x >= min_key && x <= max_key;
    const uint64_t t = live ? target(x, lds) : 0;
    return group_line_walk(t, x, live);
  }

  // Quads read whole lines (QuadLine; lane 0's first piece starts with the header) and
  // serve their probes in four rounds; every open round requests its line before any line
  // is examined, so a wave pays one memory latency per step.  Slots past a line's count
  // hold key_max, which no probe exceeds, so `below` needs no count, and a line's keys are
  // all below the probe and the line is full exactly when below = CAP.
  __device__ __forceinline__ uint32_t group_line_walk(uint64_t my_line, K my_x, bool my_live) const {
    using L = QuadLine<K, 128>;
    static_assert(L::kKeys == SLOTS, "a quad line covers one line");
    const int ql = lane() & (kQuad - 1);
    const QuadProbes<K> q(my_x);
    const K* lane_base = lines + ql * L::kLaneKeys;
    bool open = my_live;
    // fewer than 2^32 lines (targets and line bases are 32-bit at build)
    uint32_t line = static_cast<uint32_t>(my_line < num_lines ? my_line : num_lines - 1);
    const uint32_t last = static_cast<uint32_t>(num_lines - 1);
    uint32_t found = kNotFound;
    while (ballot(open) != 0) {  // wave-uniform exit
      const uint32_t rounds = quad_or(open ? 1u << ql : 0u);
      L ln[kQuad];
      quad_rounds([&](auto r) { ln[r].any(); });
      quad_rounds([&](auto r) {
        const uint32_t l = quad_bcast<r>(line);
        if ((rounds >> r) & 1u) ln[r].load(lane_base, l);
      });
      uint32_t base = 0;
      quad_rounds([&](auto r) {
        const uint32_t b = quad_bcast<0>(static_cast<uint32_t>(ln[r].pc[0].k[0]));  // the header's first row id
        base = ql == r ? b : base;
#pragma unroll
        for (uint32_t h = 0; h < HDR; ++h)
          ln[r].pc[0].k[h] = ql == 0 ? key_max<K>() : ln[r].pc[0].k[h];  // the header is no key
      });
      const uint32_t below = quad_below(ln, q, ql);
      const bool eq = quad_holds(ln, q, ql);
      if (open) {
        if (below == CAP && line < last) {
          ++line;  // a full line below the probe: keys pushed on from it sit in the next line
        } else {
          // a live probe equal to the key_max fill is the column's last key, and is met in
          // its own line (behind full lines only), where the rank is its slot
          if (eq && below < CAP) found = base + below;
          open = false;
        }
      }
    }
    return found;
  }
};

// ---------------------------------------------------------------------------
// Linear-probing hash table over the column (linear_probing_hashtable,
// src/linear_probing_hashtable.cuh:14-98): capacity 2^ceil(log2(n / 0.5)),
// slot = murmur3(key) & (capacity - 1) with the finaliser of the key's width, step +1,
// empty = all-ones key.
// An entry is 16 bytes {u64 key, u32 row id, pad}.  The reference reads one entry per
// 16-byte load and steps on (ld.global.cs of a longlong2, :62), so a wave waits for its
// longest probe run, one dependent load per slot.  Here quads read whole
// 128-byte lines of 8 entries (32 bytes per lane) and serve their probes in four
// rounds, every open round requesting its line before any line is examined: a probe
// resolves within the line of its home slot unless its run passes the line's end.
// Tables below 8 slots take the entry-by-entry walk.
// ---------------------------------------------------------------------------
struct HashEntry {
  unsigned long long key;
  uint32_t value;
  uint32_t pad;
};
static_assert(sizeof(HashEntry) == 16, "16-byte entry");

template <class K>
struct HashDev {
  static constexpr uint32_t kLineEntries = 8;
  static constexpr uint32_t kEntriesPerLane = kLineEntries / kQuad;  // 2
  const HashEntry* table;
  uint64_t mask;  // capacity - 1

  __host__ __device__ size_t lds_bytes() const { return 0; }
  __device__ void stage(uint8_t*) const {}
  // the home slot's part of the table, whose order is the hashes', not the keys'
  __device__ __forceinline__ uint32_t coarse(K x, const uint8_t*) const {
    const int bits = 64 - __clzll(static_cast<long long>(mask));
    return static_cast<uint32_t>((key_hash<K>(static_cast<uint64_t>(x)) & mask) >> (bits > 11 ? bits - 11 : 0));
  }
  __host__ __device__ uint32_t coarse_bins() const { return 1u << 11; }

  __device__ __forceinline__ uint32_t lookup_entries(uint64_t k, bool live) const {
    if (!live) return kNotFound;
    uint64_t s = key_hash<K>(k) & mask;
    for (uint64_t probes = 0; probes <= mask; ++probes) {
      const u32x4 e = *reinterpret_cast<const u32x4*>(table + s);
      const uint64_t ek = (static_cast<uint64_t>(e.y) << 32) | e.x;
      if (ek == k) return e.z;
      if (ek == ~0ull) return kNotFound;
      s = (s + 1) & mask;
    }
    return kNotFound;
  }

  __device__ __forceinline__ uint32_t lookup(K x, bool active, const uint8_t*) const {
    const uint64_t k = static_cast<uint64_t>(x);
    const bool live = active && k != ~0ull;  // all-ones is the empty marker, never a stored key
    if (mask < kLineEntries - 1) return lookup_entries(k, live);  // wave-uniform
    const int ql = lane() & (kQuad - 1);
    uint64_t slot = live ? key_hash<K>(k) & mask : 0;
    uint64_t lines_left = (mask + 1) / kLineEntries;  // a table without an empty slot ends the walk
    const QuadProbes<uint64_t> q(k);
    const u32x4* lane_base = reinterpret_cast<const u32x4*>(table) + ql * kEntriesPerLane;
    bool open = live;
    uint32_t found = kNotFound;
    while (ballot(open) != 0) {  // wave-uniform exit
      const uint32_t rounds = quad_or(open ? 1u << ql : 0u);
      const uint32_t line = static_cast<uint32_t>(slot / kLineEntries);  // at most 2^33 slots
      const uint32_t off = static_cast<uint32_t>(slot) & (kLineEntries - 1);
      u32x4 e[kQuad][kEntriesPerLane];
#pragma unroll
      for (int r = 0; r < kQuad; ++r)
#pragma unroll
        for (uint32_t t = 0; t < kEntriesPerLane; ++t) e[r][t] = any_u32x4();
      quad_rounds([&](auto r) {
        const uint64_t l = quad_bcast<r>(line);
        if ((rounds >> r) & 1u) {
#pragma unroll
          for (uint32_t t = 0; t < kEntriesPerLane; ++t) e[r][t] = lane_base[l * kLineEntries + t];
        }
      });
      uint32_t flags = 0;     // bit r: round r's key is here; bit 4 + r: an empty slot from its home on
      uint32_t v[kQuad];
      quad_rounds([&](auto r) {
        const uint32_t o = quad_bcast<r>(off);
        v[r] = 0;
#pragma unroll
        for (uint32_t t = 0; t < kEntriesPerLane; ++t) {
          const uint64_t ek = (static_cast<uint64_t>(e[r][t].y) << 32) | e[r][t].x;
          // a key sits in one slot only, so a match needs no look at the home slot
          const bool m = ek == q.x[r];
          v[r] = m ? e[r][t].z : v[r];
          flags |= m ? 1u << r : 0u;
          flags |= (ek == ~0ull && static_cast<uint32_t>(ql) * kEntriesPerLane + t >= o) ? 16u << r : 0u;
        }
      });
      flags = quad_or(flags) >> ql;
      // lane r takes round r's value: one lane of the quad holds it, the others zero
      const uint32_t a = ((ql & 1) ? v[1] : v[0]) | quad_perm32<0xB1>((ql & 1) ? v[0] : v[1]);
      const uint32_t b = ((ql & 1) ? v[3] : v[2]) | quad_perm32<0xB1>((ql & 1) ? v[2] : v[3]);
      const uint32_t value = ((ql & 2) ? b : a) | quad_perm32<0x4E>((ql & 2) ? a : b);
      if (open) {
        // a present key comes before every empty slot of its run, so a match decides
        if (flags & 1u) {
          found = value;
          open = false;
        } else if ((flags & 16u) || --lines_left == 0) {
          open = false;
        } else {
          slot = ((slot | (kLineEntries - 1)) + 1) & mask;  // the next line's first entry
        }
      }
    }
    return found;
  }
};

}  // namespace gj
