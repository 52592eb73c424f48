// indexes.cuh - device-side index descriptors.
//
// Each descriptor is a small POD passed BY VALUE as a kernel argument, the
// role of the reference's device_index_t (src/indexes.cuh:18-22, 108-124).
// Every descriptor provides
//   size_t   lds_bytes() const                      bytes of LDS the lookup wants resident
//   void     stage(uint8_t* lds) const              block-cooperative fill of that LDS (no barrier)
//   uint32_t lookup(K x, bool active, const uint8_t* lds) const
//   uint32_t coarse(K x, const uint8_t* lds) const  roughly where x lies, from what needs no memory
//                                                   read: a number that ascends with x
//   uint32_t coarse_bins() const                    above every such number
// lookup() must be called by all 64 lanes of a wave together (like the
// reference's whole-warp cooperative_lookup, src/btree.cuh:598-605,
// src/harmonia.cuh:740-745); inactive lanes pass active = false and get
// kNotFound.  The result is the row id (position in the sorted column) or
// kNotFound when the key is absent.
#pragma once

#include "device.cuh"

namespace gj {

constexpr int kMaxLevels = 16;

// ---------------------------------------------------------------------------
// Cooperative search of NB-byte sorted lines (tree nodes, column lines, key lines)
// by quads.  Each lane owns one probe; a quad serves its four probes in four rounds:
// in round r its lanes fetch the line of lane r's probe, a quarter each, and each lane
// counts its own keys below that probe.  All four rounds' loads are issued
// before any compare, so a line step costs one memory latency.  The counts of the
// four rounds sit in the bytes of one register, so two quad additions sum all of them
// and lane r takes byte r.
//
// What bounds it: with every line in L2 the search is bound by VALU issue.  The form
// before this one (groups of 8 lanes, probe and node fetched through the LDS crossbar,
// one ballot, shift and population count per key) took about 230 instructions per line
// step and 64 probes; this one takes about 75.  2^24 probes, plain driver, before and
// after: B-tree over 2^20 u32 keys 449 -> 229 us, 2^20 u64 470 -> 322, 2^22 u64 557 -> 402;
// hash over 2^14 u32 keys 179 -> 159; RadixSpline over 2^16 u64 keys 382 -> 337.  Beyond
// L2 the bound is 55 G lines/s whatever the search (2^26 u64 keys: B-tree 3.12 -> 2.92 ms
// per 2^26 probes).
// ---------------------------------------------------------------------------
template <class K, int NB>
struct QuadLine {
  static constexpr int kPiece = Piece<K>::kKeys;               // keys per 16-byte piece
  static constexpr int kPieces = NB / (16 * kQuad);            // pieces per lane
  static constexpr int kLaneKeys = kPiece * kPieces;           // consecutive keys per lane
  static constexpr int kKeys = NB / static_cast<int>(sizeof(K));
  static_assert(kPieces >= 1 && kKeys < 128, "a round's count must fit its byte");
  Piece<K> pc[kPieces];

  // lane_base: the array of lines plus this lane's first key
  __device__ __forceinline__ void load(const K* lane_base, uint64_t line) {
    const K* p = lane_base + line * kKeys;
#pragma unroll
    for (int t = 0; t < kPieces; ++t) pc[t] = load_piece(p + t * kPiece);
  }
  // keys at .. at + kKeys - 1 of a column, aligned or not
  __device__ __forceinline__ void load_keys(const K* lane_base, uint32_t at) {
    const K* p = lane_base + at;
#pragma unroll
    for (int t = 0; t < kPieces; ++t) pc[t] = load_piece_any(p + t * kPiece);
  }
  // whatever the registers hold, for the rounds that then load nothing and whose count is
  // not looked at; all of a step's calls come before its loads, whose registers these are
  __device__ __forceinline__ void any() {
#pragma unroll
    for (int t = 0; t < kPieces; ++t) pc[t] = piece_of<K>(any_u32x4());
  }
  __device__ __forceinline__ uint32_t below(K x) const {
    uint32_t c = 0;
#pragma unroll
    for (int t = 0; t < kPieces; ++t)
#pragma unroll
      for (int j = 0; j < kPiece; ++j) c += pc[t].k[j] < x ? 1u : 0u;
    return c;
  }
  __device__ __forceinline__ bool holds(K x) const {
    bool e = false;
#pragma unroll
    for (int t = 0; t < kPieces; ++t)
#pragma unroll
      for (int j = 0; j < kPiece; ++j) e |= pc[t].k[j] == x;
    return e;
  }
};

// The four probes of the lane's quad.
template <class K>
struct QuadProbes {
  K x[kQuad];
  __device__ __forceinline__ explicit QuadProbes(K mine) {
    quad_rounds([&](auto r) { x[r] = quad_bcast<r>(mine); });
  }
};

// Rank of each lane's probe in the line its quad loaded for it: keys below it, and
// whether the line holds it.  lanes: those whose probe is of interest; a round that serves
// none of them in any quad is passed over: the join-aggregate's plain strategy has one or two
// live lanes a wave (12 M rows of 836139 dimension rows, learned: all rounds 91 us, now 81).
constexpr uint64_t kRoundLanes = 0x1111111111111111ull;  // the lanes that round 0 serves
template <class K, int NB>
__device__ __forceinline__ uint32_t quad_below(const QuadLine<K, NB> (&ln)[kQuad], const QuadProbes<K>& q, int ql,
                                               uint64_t lanes = ~0ull) {
  uint32_t c = 0;
#pragma unroll
  for (int r = 0; r < kQuad; ++r)
    if (lanes & (kRoundLanes << r)) c |= ln[r].below(q.x[r]) << (8 * r);
  return (quad_sum(c) >> (8 * ql)) & 0xFFu;
}
template <class K, int NB>
__device__ __forceinline__ bool quad_holds(const QuadLine<K, NB> (&ln)[kQuad], const QuadProbes<K>& q, int ql,
                                           uint64_t lanes = ~0ull) {
  uint32_t e = 0;
#pragma unroll
  for (int r = 0; r < kQuad; ++r)
    if (lanes & (kRoundLanes << r)) e |= ln[r].holds(q.x[r]) ? 1u << r : 0u;
  return (quad_or(e) >> ql) & 1u;
}

// Keys below each lane's probe in line `line` of `base` (whole lines).
template <class K, int NB>
__device__ __forceinline__ uint32_t quad_count_less(const K* base, uint32_t line, const QuadProbes<K>& q, int ql) {
  QuadLine<K, NB> ln[kQuad];
  const K* lane_base = base + ql * QuadLine<K, NB>::kLaneKeys;
  quad_rounds([&](auto r) { ln[r].load(lane_base, quad_bcast<r>(line)); });
  return quad_below(ln, q, ql);
}

// Where the keys of a column's line are read from: a partial last line is read together with
// the keys before it, as the last kKeys keys of the column (n >= kKeys).  A lane that walked
// the partial line by itself, key by key, held its wave up: 2^14 probes of 8181 keys, B-tree
// u32 6.2 us, now 4.6; learned u32 6.6, now 4.6.
template <int kKeys>
__device__ __forceinline__ uint32_t line_at(uint32_t line, uint64_t n) {
  const uint32_t last = static_cast<uint32_t>(n) - kKeys;
  return line * kKeys < last ? line * kKeys : last;
}

// Branch-free lower_bound over len keys of a column from lo on; the row id if the key before
// hi is x.
template <class K>
__device__ __forceinline__ uint32_t halve(const K* col, K x, uint64_t lo, uint64_t len, uint64_t hi) {
  const K* base = col + lo;
  while (len > 1) {
    const uint64_t half = len >> 1;
    base = (base[half] < x) ? base + half : base;
    len -= half;
  }
  const uint64_t p = static_cast<uint64_t>(base - col) + ((base[0] < x) ? 1u : 0u);
  return (p < hi && col[p] == x) ? static_cast<uint32_t>(p) : kNotFound;
}

// Position of each lane's probe in its NB-byte chunk of the column, or not found.  In a column
// shorter than a chunk each lane halves for itself: a quad's read of the padded line is so
// much code that it slows the whole lines down (2^24 probes of 2^22 u32 keys, B-tree: with it
// 292 us, now 281).  Whole: the column is no shorter (the halving, too, costs sorted tiles 5 %:
// 2^16 probes of 2^16 u32 keys 23.4 us, now 22.1).
template <class K, int NB, bool Whole = false>
__device__ __forceinline__ uint32_t quad_find_equal(const K* col, uint64_t n, uint32_t chunk, bool live, K x,
                                                    const QuadProbes<K>& q, int ql) {
  using L = QuadLine<K, NB>;
  if constexpr (!Whole)
    if (n < static_cast<uint64_t>(L::kKeys)) return live ? halve(col, x, 0, n, n) : kNotFound;  // kernel-uniform
  const uint32_t at = line_at<L::kKeys>(chunk, n);
  L ln[kQuad];
  const K* lane_base = col + ql * L::kLaneKeys;
  quad_rounds([&](auto r) { ln[r].load_keys(lane_base, quad_bcast<r>(at)); });
  const uint32_t below = quad_below(ln, q, ql);
  const bool eq = quad_holds(ln, q, ql);
  return (live && eq) ? at + below : kNotFound;
}

// ---------------------------------------------------------------------------
// Binary search (binary_search_index, src/indexes.cuh:336-375 with
// lower_bound, src/search.cuh:26-41).  One probe per lane.  The column is
// cut into 2^sample_bits equal buckets; the max key of every bucket sits in
// LDS, so the first sample_bits steps of the search never leave the CU.  Inside the
// bucket, quads read whole 128-byte lines: the first two are interpolated between the
// nearest keys known on either side (the bucket's bounds, then the first line's own edge),
// the third is the second's neighbour, and what is still open then (keys that crowd in
// their bucket) halves the rest of its range key by key.  The column may hold equal keys;
// the answer is the first of them, so a line that begins with the probe's key is a
// candidate and the search goes on to the left.
//
// What bounds it: fabric lines (about 52 G/s).  Halving alone touches log2(bucket bytes /
// 128) + 1 lines per probe, one dependent load each; in a bucket of evenly spread keys the
// first guess is off by sqrt(bucket) / 3 keys on average and the second finds the line.
// It stays for small buckets (Lines = false: two or three loads of a line that is in reach
// anyway: 2^24 probes of 2^12 u32 keys 118 us, by quads 170; with_index_dev says how small), and
// for waves whose probes all lie in about one bucket, whose lanes share their loads (sorted
// probes over 2^22 u64 keys 216 us, by quads 402).
// 2^24 uniform probes, halving alone -> by lines, us: 2^16 u64 keys 522 -> 220, 2^20 1032 ->
// 307, 2^22 2357 -> 505, 2^24 3560 -> 667; u32 2^22 1897 -> 329; behind the blockwise sort,
// 2^22 u64 1261 -> 829.
// ---------------------------------------------------------------------------
template <class K, bool Lines = true>
struct BSearchDev {
  using L = QuadLine<K, 128>;
  static constexpr uint32_t LK = L::kKeys;
  static constexpr int kGuesses = 2;  // interpolated lines (the second between the first and the bucket), then one neighbour
  const K* col;
  uint64_t n;
  const K* samples;  // 2^sample_bits bucket maxima (key_max for empty buckets)
  uint64_t step;     // keys per bucket
  uint32_t sample_bits;

  __host__ __device__ size_t lds_bytes() const { return sizeof(K) << sample_bits; }
  __device__ void stage(uint8_t* lds) const { stage_to_lds(lds, samples, lds_bytes()); }

  // the bucket
  __device__ __forceinline__ uint32_t coarse(K x, const uint8_t* lds) const {
    const K* s = reinterpret_cast<const K*>(lds);
    uint32_t b = 0;
    for (uint32_t h = (1u << sample_bits) >> 1; h > 0; h >>= 1) b = (s[b + h - 1] < x) ? b + h : b;
    return b + (s[b] < x ? 1u : 0u);
  }
  __host__ __device__ uint32_t coarse_bins() const { return (1u << sample_bits) + 1; }

  // Where x would sit between positions plo and phi, whose keys are `below` and `above` away
  // from it, if the keys between were evenly spread; any error only costs lines.
  __device__ __forceinline__ static uint32_t guess(float below, float above, uint32_t plo, uint32_t phi) {
    const float f = below * __builtin_amdgcn_rcpf(below + above);
    return plo + static_cast<uint32_t>(fminf(fmaxf(f, 0.0f), 1.0f) * static_cast<float>(phi - plo));
  }

  // Full: the wave's lanes are all at work, or about so (see narrow).
  template <bool Full = false>
  __device__ __forceinline__ uint32_t lookup(K x, bool active, const uint8_t* lds) const {
    const K* s = reinterpret_cast<const K*>(lds);
    const uint32_t nb = 1u << sample_bits, b = coarse(x, lds);
    const uint64_t lo = static_cast<uint64_t>(b) * step;
    if constexpr (!Lines) {
      if (!active || b >= nb || lo >= n) return kNotFound;
      const uint64_t hi = (lo + step < n) ? lo + step : n;
      return halve(col, x, lo, hi - lo, hi);
    } else {
      bool open = active && b < nb && lo < n;
      // x's position is in [first, last], or last + 1 where found holds it already
      uint32_t first = open ? bucket_first(b) : 0u, last = open ? bucket_last(b) : 0u;
      uint32_t found = kNotFound;
      const uint32_t b0 = __builtin_amdgcn_readfirstlane(b);
      if (ballot(open && (b > b0 + 1 || b + 1 < b0)) != 0)  // wave-uniform
        narrow<Full>(x, b, s, open, first, last, found);
      if (open) {
        const uint32_t r = halve(col, x, first, static_cast<uint64_t>(last - first) + 1, static_cast<uint64_t>(last) + 1);
        found = r != kNotFound ? r : found;
      }
      return found;
    }
  }

  // First and last position of bucket b, which begins inside the column.
  __device__ __forceinline__ uint32_t bucket_first(uint32_t b) const { return b * static_cast<uint32_t>(step); }
  __device__ __forceinline__ uint32_t bucket_last(uint32_t b) const {
    const uint32_t lo = bucket_first(b);
    return static_cast<uint32_t>(lo + step < n ? lo + step : n) - 1;
  }

  // Whole lines of bucket b by quads; what is left of it is [first, last].  The column's
  // partial last line is left to the halving.  Of the bucket's bounds only x's distances from
  // its keys are kept: the keys and positions themselves cost u64 keys a wave per SIMD (70
  // registers, now 64), which sorted probes, whose waves do not come here, paid for (2^20 of
  // them over 10^6 keys: halving alone 11.4 us, with the bounds in registers 16.4, now 11.6).
  // Rounds whose lanes have nothing left are passed over, but not in tiles sorted in LDS
  // (Full): there a wave waits for its loads, and the branches between the rounds keep their
  // work from filling the wait (2^18 probes of 2^20 u32 keys 34.9 us without them, 37.1 with;
  // unsorted 2^22 of 10^7 u64 keys 186 without, 168 with).
  template <bool Full>
  __device__ __forceinline__ void narrow(K x, uint32_t b, const K* s, bool& open, uint32_t& first, uint32_t& last,
                                         uint32_t& found) const {
    const int ql = lane() & (kQuad - 1);
    const QuadProbes<K> q(x);
    const K* lane_base = col + ql * L::kLaneKeys;
    const uint32_t whole = static_cast<uint32_t>(n / LK);  // whole lines of the column
    if (!open) b = 0;
    uint32_t line_lo = bucket_first(b) / LK, line_hi = bucket_last(b) / LK, line;
    // klo < x <= khi: the keys before the bucket (the column's first key for the first one) and at its end
    const K klo = b > 0 ? s[b - 1] : col[0];
    open = open && klo <= x;
    const float below_x = static_cast<float>(x - klo);
    line = guess(below_x, static_cast<float>(s[b] - x), b > 0 ? bucket_first(b) - 1 : 0u, bucket_last(b)) / LK;
    bool bounded = line_hi < whole;     // x is in no line behind line_hi
    bool go = open && line_lo < whole;  // lines to look at
    line_hi -= !bounded && go ? 1u : 0u;
    line = line < line_lo ? line_lo : (line > line_hi ? line_hi : line);
    for (int t = 1; t <= kGuesses + 1; ++t) {
      const uint64_t lanes = ballot(go);
      if (lanes == 0) break;  // wave-uniform
      const uint32_t rounds = quad_or(go ? 1u << ql : 0u);
      L ln[kQuad];
      quad_rounds([&](auto r) { ln[r].any(); });
      quad_rounds([&](auto r) {
        const uint32_t l = quad_bcast<r>(line);
        if ((rounds >> r) & 1u) ln[r].load(lane_base, l);
      });
      const uint64_t at_work = Full ? ~0ull : lanes;
      const uint32_t below = quad_below(ln, q, ql, at_work);
      const bool eq = quad_holds(ln, q, ql, at_work);
      asm volatile("" : "+v"(b));  // its positions are computed anew
      if (go) {
        const uint32_t base = line * LK;
        const bool right = below == LK;  // every key of the line is below x
        if (right) {
          go = line < line_hi;
          open = go || !bounded;
          line_lo = line + 1;
        } else {
          found = eq ? base + below : found;
          go = below == 0 && line > line_lo;
          open = go;
          line_hi = line - 1;
          bounded = true;
        }
        if (go) {
          line = right ? line_lo : line_hi;
          if (t < kGuesses) {  // wave-uniform
            const uint32_t at = right ? base + LK - 1 : base;  // the edge of the line on x's side
            const K edge = col[at];
            const float away = static_cast<float>(right ? x - edge : edge - x);
            line = right ? guess(away, static_cast<float>(s[b] - x), at, bucket_last(b))
                         : guess(below_x, away, b > 0 ? bucket_first(b) - 1 : 0u, at);
            line /= LK;
            line = line < line_lo ? line_lo : (line > line_hi ? line_hi : line);
          }
        }
      }
    }
    const uint32_t a = line_lo * LK, z = line_hi * LK + LK - 1;
    first = bucket_first(b);
    last = bucket_last(b);
    first = a > first ? a : first;
    last = bounded && z < last ? z : last;
  }
};

// ---------------------------------------------------------------------------
// B+-tree, re-laid out for CDNA4.  Keeps the reference's clustered-index
// semantics (btree_index over the sorted column; leaves are column chunks,
// src/btree.cuh:242-246, 504-531) with a static implicit layout:
//   * a node is NB bytes, NK = NB / sizeof(K) keys: one 128-byte line by default
//     (16 x u64 / 32 x u32), or half a line / two lines (NB = 64 / 256);
//   * the leaves are the column itself, cut into chunks of NK keys (NB bytes each);
//   * slot s of node i holds the max key of child i*NK + s (key_max past the end),
//     so the child index is the count of separators below the probe and no
//     child pointers are stored (the reference stores pointers, src/btree.cuh:58-63);
//   * levels are stored top first; the lowest level that fits the LDS budget with all
//     above it is staged in LDS and searched there by each lane for itself: about 6
//     instructions per halving, where a node's line by quads takes 75.  2^24 probes, the
//     levels above by quads -> searched: 2^20 u32 keys 229 -> 205 us, 2^20 u64 322 -> 287,
//     2^22 u64 402 -> 384.
// ---------------------------------------------------------------------------
template <class K, int NB = 128>
struct BTreeDev {
  static_assert(NB == 64 || NB == 128 || NB == 256, "B-tree nodes of 64, 128 or 256 bytes");
  static constexpr int NK = NB / static_cast<int>(sizeof(K));
  const K* col;
  uint64_t n;
  const K* nodes;  // all inner levels, top level first, NK keys per node
  uint32_t levels;
  uint32_t lds_levels;
  uint64_t level_off[kMaxLevels];      // first node of level l (top = 0)
  uint64_t level_cnt[kMaxLevels + 1];  // nodes of level l; level_cnt[levels] = column chunks

  // The lowest of the levels that fit the LDS budget is the only one staged: its slots are
  // the separators of all the nodes below it in key order, so a binary search over them
  // finds the node that the levels above would lead to.
  __host__ __device__ size_t lds_bytes() const { return lds_levels ? level_cnt[lds_levels - 1] * NB : 0; }
  __device__ void stage(uint8_t* lds) const {
    if (lds_levels) stage_to_lds(lds, nodes + level_off[lds_levels - 1] * NK, lds_bytes());
  }

  // Separators of the staged level below x, which is x's node in the next level.
  __device__ __forceinline__ uint32_t top_search(K x, const K* seps) const {
    uint32_t at = 0;
    for (uint32_t len = static_cast<uint32_t>(level_cnt[lds_levels - 1]) * NK; len > 1;) {  // kernel-uniform
      const uint32_t half = len >> 1;
      at = seps[at + half - 1] < x ? at + half : at;
      len -= half;
    }
    return at + (seps[at] < x ? 1u : 0u);
  }

  // the node below the staged level
  __device__ __forceinline__ uint32_t coarse(K x, const uint8_t* lds) const {
    return lds_levels ? top_search(x, reinterpret_cast<const K*>(lds)) : 0u;
  }
  __host__ __device__ uint32_t coarse_bins() const {
    return lds_levels ? static_cast<uint32_t>(level_cnt[lds_levels - 1]) * NK + 1 : 1u;
  }

  __device__ __forceinline__ void descend(uint32_t& node, bool& live, uint32_t c, uint32_t lvl) const {
    const uint64_t child = static_cast<uint64_t>(node) * NK + c;
    live = live && (c < static_cast<uint32_t>(NK)) && (child < level_cnt[lvl + 1]);
    node = live ? static_cast<uint32_t>(child) : 0u;
  }

  // Full: by waves whose lanes are all at work, over a column of a chunk and more.
  template <bool Full = false>
  __device__ __forceinline__ uint32_t lookup(K x, bool active, const uint8_t* lds) const {
    const int ql = lane() & (kQuad - 1);
    const QuadProbes<K> q(x);
    bool live = active;
    uint32_t node = 0;  // fewer than 2^32 / NK chunks, hence nodes of any level
    if (lds_levels) {
      node = top_search(x, reinterpret_cast<const K*>(lds));
      live = live && node < level_cnt[lds_levels];
      node = live ? node : 0u;
    }
    uint32_t lvl = lds_levels;
    for (; lvl < levels; ++lvl)
      descend(node, live, quad_count_less<K, NB>(nodes + level_off[lvl] * NK, node, q, ql), lvl);
    return quad_find_equal<K, NB, Full>(col, n, node, live, x, q, ql);
  }
};

// A column shorter than a line under an index that searches windows (or, blockwise sorted, under
// a B-tree): each lane halves for itself.  The window search holds no code for it, which slowed it down (2^23 probes of 2^22 u64
// keys, learned MLP root: with it 171 us, now 165).
template <class K>
struct ShortDev {
  const K* col;
  uint64_t n;
  __host__ __device__ size_t lds_bytes() const { return 0; }
  __device__ void stage(uint8_t*) const {}
  __device__ __forceinline__ uint32_t coarse(K, const uint8_t*) const { return 0; }
  __host__ __device__ uint32_t coarse_bins() const { return 1; }
  __device__ __forceinline__ uint32_t lookup(K x, bool active, const uint8_t*) const {
    return active ? halve(col, x, 0, n, n) : kNotFound;
  }
};

// no_op_index (src/indexes.cuh:384-406): measures probe read + row id write.
template <class K>
struct NoOpDev {
  __host__ __device__ size_t lds_bytes() const { return 0; }
  __device__ void stage(uint8_t*) const {}
  __device__ __forceinline__ uint32_t coarse(K x, const uint8_t*) const {
    return static_cast<uint32_t>(x >> (8 * sizeof(K) - 11));
  }
  __host__ __device__ uint32_t coarse_bins() const { return 1u << 11; }
  __device__ __forceinline__ uint32_t lookup(K, bool, const uint8_t*) const { return kNotFound; }
};

}  // namespace gj
