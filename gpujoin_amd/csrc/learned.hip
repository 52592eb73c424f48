// learned.hip - GPU training and calibration of the learned two-stage position
// models (no reference counterpart; they close over the same exact last-mile
// search as the reference's RadixSpline, src/indexes.cuh:205-215).
//
// Pipeline, all on the GPU over the (key, position) pairs of the sorted column:
//   1. root: linear least squares of cdf = i / n on x = unit(key)  (reduction kernel),
//            an error-bounded greedy spline of the CDF (learned_plr on skewed keys), or
//            a 1xH MLP f(x) = b2 + sum_k w2_k clamp(w1_k x + b1_k, 0, 1) whose ramps start
//            at the column's quantiles (the piecewise-linear CDF through h + 1 quantiles) and
//            are then trained with minibatch Adam by hand-written forward/backward kernels;
//            w1 and w2 are projected to >= 0 after every step, so the MLP is monotone and
//            every leaf owns a contiguous key range
//   2. routing: leaf = floor(root(x) * L); leaf start positions by a boundary kernel
//   3. leaves: per-leaf linear least squares of local position on FP32 key offsets,
//      packed into the 16-byte lookup model (intercept rounded into the start)
//   4. calibration: the error of every build key under the exact FP32 lookup code
//      gives each leaf its error range; leaves wider than the bound are routed to the
//      B-tree, and the extremes over the other leaves form the lookup window
#include <algorithm>
#include <climits>
#include <cmath>
#include <vector>

#include "common.hpp"
#include "lookup_dispatch.hpp"
#include "rs_builder.hpp"

namespace gj {

namespace {

unsigned grid_for(uint64_t work, unsigned block, unsigned cap = 65536) {
  uint64_t g = ceil_div(work, block);
  if (g == 0) g = 1;
  if (g > cap) g = cap;
  return static_cast<unsigned>(g);
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

template <class T>
__device__ __forceinline__ T wave_sum(T v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

template <class T>
__device__ __forceinline__ T wave_min(T v) {
  for (int off = 32; off > 0; off >>= 1) {
    const T o = __shfl_xor(v, off, 64);
    v = o < v ? o : v;
  }
  return v;
}
template <class T>
__device__ __forceinline__ T wave_max(T v) {
  for (int off = 32; off > 0; off >>= 1) {
    const T o = __shfl_xor(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}

// out[at .. at + count) = value, each lane its own run (called by whole waves).  Long runs
// (a gap between clusters can span a large part of the table) are written by the whole
// wave, one run after the other.
__device__ __forceinline__ void fill_runs(uint32_t* __restrict__ out, uint32_t at, uint32_t count, uint32_t value) {
  constexpr uint32_t kOwn = 32;
  uint64_t todo = ballot(count > kOwn);
  if (count <= kOwn)
    for (uint32_t k = 0; k < count; ++k) out[at + k] = value;
  while (todo) {  // wave-uniform
    const int src = __ffsll(static_cast<unsigned long long>(todo)) - 1;
    const uint32_t a = shfl32(at, src), c = shfl32(count, src), v = shfl32(value, src);
    for (uint32_t k = static_cast<uint32_t>(lane()); k < c; k += kWave) out[a + k] = v;
    todo &= todo - 1;
  }
}

__global__ void fill_words_kernel(uint32_t* __restrict__ out, uint64_t count, uint32_t value) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += stride) out[i] = value;
}
void fill_words(uint32_t* d, uint64_t count, uint32_t value, hipStream_t s) {
  hipLaunchKernelGGL(fill_words_kernel, dim3(grid_for(count, 1024)), dim3(256), 0, s, d, count, value);
  GJ_HIP_CHECK(hipGetLastError());
}

struct RootFitSums {
  double sx, sxx, st, sxt;
};

// Per-block partial sums of x, x^2, t, x*t with x = unit(key_i), t = i / n.
template <class K>
__global__ void root_sums_kernel(const K* __restrict__ col, uint64_t n, K min_key, float inv_range,
                                 RootFitSums* __restrict__ partial) {
  double sx = 0, sxx = 0, st = 0, sxt = 0;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    const double x = key_unit(col[i], min_key, inv_range);
    const double t = static_cast<double>(i) / static_cast<double>(n);
    sx += x;
    sxx += x * x;
    st += t;
    sxt += x * t;
  }
  sx = wave_sum(sx);
  sxx = wave_sum(sxx);
  st = wave_sum(st);
  sxt = wave_sum(sxt);
  __shared__ RootFitSums s[4];
  const int w = threadIdx.x / 64;
  if (lane() == 0) s[w] = {sx, sxx, st, sxt};
  __syncthreads();
  if (threadIdx.x == 0) {
    RootFitSums r{0, 0, 0, 0};
    for (int i = 0; i < static_cast<int>(blockDim.x / 64); ++i) {
      r.sx += s[i].sx;
      r.sxx += s[i].sxx;
      r.st += s[i].st;
      r.sxt += s[i].sxt;
    }
    partial[blockIdx.x] = r;
  }
}

// ---- MLP root: loss and gradient -------------------------------------------
// Samples come either from explicit arrays (x, y) or from the sorted column at
// seeded random positions (x = unit(key), y = position / n).
template <class K>
struct SampleSource {
  const float* x;
  const float* y;
  const K* col;
  uint64_t n;
  K min_key;
  float inv_range;
  uint64_t seed;
  __device__ __forceinline__ void get(uint64_t j, float& xs, float& ys) const {
    if (x) {
      xs = x[j];
      ys = y[j];
    } else {
      const uint64_t r = mix64(seed + (j + 1) * 0x9E3779B97F4A7C15ull);
      const uint64_t i = static_cast<uint64_t>((static_cast<unsigned __int128>(r) * n) >> 64);
      xs = key_unit(col[i], min_key, inv_range);
      ys = static_cast<float>(static_cast<double>(i) / static_cast<double>(n));
    }
  }
};

// grad[3H+1] += d/dp mean((f(x) - y)^2) over `count` samples; loss += mean squared error.
//
// A wave takes 64 samples at a time.  First a lane is a sample: it evaluates the network
// (the parameters are uniform, hence scalar) and leaves (x, g = dloss/df) in LDS.  Then a
// lane is a hidden unit and one of 64 / H parts of the samples: it reads the pairs back
// (the same address for all its lanes) and sums its unit's three gradients in registers,
// 64 / P additions in FP32 and the partial sums of a wave's tiles, of its parts and of the
// block's waves in FP64.
// What bounds it: with a lane per sample throughout, every one of the 3H sums is reduced
// over the wave, 6 cross-lane steps each, which outweighed the gradients themselves; and
// the blocks' atomics on one set of addresses queue up, so a block is as large as it can
// be.  65536 samples, H = 32: 24.5 -> 8.1 us; 2^22, H = 64: 303 -> 74.
constexpr int kGradBlock = 1024;

template <int H, class K>
__global__ __launch_bounds__(kGradBlock) void mlp_grad_kernel(const float* __restrict__ params, SampleSource<K> src,
                                                              uint64_t count, float* __restrict__ grad,
                                                              float* __restrict__ loss) {
  constexpr int kWaves = kGradBlock / kWave;
  constexpr int kParts = kWave / H;                // sample parts per unit
  constexpr int kPart = kWave / kParts;            // samples per part
  constexpr int kStride = kPart * 2 + 4;           // floats; the parts start on different banks
  constexpr int kOut = 3 * H + 2;                  // gradients and loss
  __shared__ __attribute__((aligned(16))) float xg[kWaves][kParts * kStride];
  __shared__ double red[kWaves][kOut];
  const int ln = lane(), w = static_cast<int>(threadIdx.x) / kWave;
  const int unit = ln % H, part = ln / H;
  const float w1 = params[unit], b1 = params[H + unit];
  const float scale = 2.0f / static_cast<float>(count);
  double gw1 = 0, gb1 = 0, gw2 = 0, gb2 = 0, l = 0;
  float* mine = xg[w] + (ln / kPart) * kStride + (ln % kPart) * 2;
  const float* theirs = xg[w] + part * kStride;
  const uint64_t waves = static_cast<uint64_t>(gridDim.x) * kWaves;
  for (uint64_t base = (static_cast<uint64_t>(blockIdx.x) * kWaves + w) * kWave; base < count; base += waves * kWave) {
    const uint64_t j = base + ln;
    float x = 0.0f, g = 0.0f;
    if (j < count) {
      float y;
      src.get(j, x, y);
      float f = params[3 * H];
#pragma unroll
      for (int k = 0; k < H; ++k) {
        const float a = __builtin_fmaf(params[k], x, params[H + k]);
        f = __builtin_fmaf(params[2 * H + k], fminf(fmaxf(a, 0.0f), 1.0f), f);
      }
      const float r = f - y;
      g = scale * r;
      l += static_cast<double>(r) * r;
      gb2 += g;
    }
    __builtin_amdgcn_wave_barrier();  // the last tile's reads come before these writes
    mine[0] = x;
    mine[1] = g;
    __builtin_amdgcn_wave_barrier();  // one wave's LDS operations complete in order
    float s1 = 0.0f, sb = 0.0f, s2 = 0.0f;
#pragma unroll
    for (int t = 0; t < kPart; t += 2) {
      const float4 v = *reinterpret_cast<const float4*>(theirs + 2 * t);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float xs = e ? v.z : v.x, gs = e ? v.w : v.y;
        const float a = __builtin_fmaf(w1, xs, b1);
        const float h = fminf(fmaxf(a, 0.0f), 1.0f);
        const bool slope = h > 0.0f && h < 1.0f;  // the ramp passes gradient only on its slope
        const float gm = slope ? gs : 0.0f, xm = slope ? xs : 0.0f;
        s2 = __builtin_fmaf(gs, h, s2);
        s1 = __builtin_fmaf(gm, xm, s1);
        sb += gm;
      }
    }
    gw1 += s1;
    gb1 += sb;
    gw2 += s2;
  }
#pragma unroll
  for (int off = H; off < kWave; off <<= 1) {
    gw1 += __shfl_xor(gw1, off, kWave);
    gb1 += __shfl_xor(gb1, off, kWave);
    gw2 += __shfl_xor(gw2, off, kWave);
  }
  gb2 = wave_sum(gb2);
  l = wave_sum(l);
  if (part == 0) {
    const double w2 = params[2 * H + unit];
    red[w][unit] = gw1 * w2;
    red[w][H + unit] = gb1 * w2;
    red[w][2 * H + unit] = gw2;
  }
  if (ln == 0) {
    red[w][3 * H] = gb2;
    red[w][3 * H + 1] = l;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kOut; i += kGradBlock) {
    double v = 0;
    for (int q = 0; q < kWaves; ++q) v += red[q][i];
    if (i < 3 * H + 1)
      atomicAdd(&grad[i], static_cast<float>(v));
    else
      atomicAdd(loss, static_cast<float>(v / static_cast<double>(count)));
  }
}

// One Adam step; w1 and w2 are projected onto >= 0 (monotone root); clears grad.
__global__ void adam_kernel(float* __restrict__ params, float* __restrict__ grad, float* __restrict__ m1,
                            float* __restrict__ m2, uint32_t h, float lr, int step) {
  const uint32_t i = threadIdx.x;
  if (i >= 3 * h + 1) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float g = grad[i];
  grad[i] = 0.0f;
  m1[i] = b1 * m1[i] + (1.0f - b1) * g;
  m2[i] = b2 * m2[i] + (1.0f - b2) * g * g;
  const float mh = m1[i] / (1.0f - powf(b1, static_cast<float>(step)));
  const float vh = m2[i] / (1.0f - powf(b2, static_cast<float>(step)));
  float p = params[i] - lr * mh / (sqrtf(vh) + eps);
  const bool nonneg = (i < h) || (i >= 2 * h && i < 3 * h);
  if (nonneg && p < 0.0f) p = 0.0f;
  params[i] = p;
}

template <class K>
void launch_mlp_grad(uint32_t h, const float* params, const SampleSource<K>& src, uint64_t count, float* grad,
                     float* loss, hipStream_t s) {
  // a block per CU at most: the blocks' sums meet in the same 3H + 2 addresses
  const unsigned blocks = grid_for(count, kGradBlock, 256);
  auto launch = [&]<int H>() {
    hipLaunchKernelGGL((mlp_grad_kernel<H, K>), dim3(blocks), dim3(kGradBlock), 0, s, params, src, count, grad, loss);
  };
  switch (h) {
    case 8: launch.template operator()<8>(); break;
    case 16: launch.template operator()<16>(); break;
    case 32: launch.template operator()<32>(); break;
    case 64: launch.template operator()<64>(); break;
    default: throw error(GJ_ERR_INVALID, "mlp hidden width must be 8, 16, 32 or 64");
  }
  GJ_HIP_CHECK(hipGetLastError());
}

// Gradient and loss are added to, so a call starts from zero.
__global__ void clear_grad_kernel(float* __restrict__ grad, uint64_t count, float* __restrict__ loss) {
  for (uint64_t i = threadIdx.x; i < count; i += blockDim.x) grad[i] = 0.0f;
  if (threadIdx.x == 0) *loss = 0.0f;
}

__global__ void mlp_forward_kernel(const float* __restrict__ params, uint32_t h, const float* __restrict__ x, uint64_t n,
                                   float* __restrict__ out) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = mlp_eval(params, h, x[i]);
}

// ---- routing, leaf fit, calibration ----------------------------------------
template <class K>
struct Router {
  K min_key;
  RootModel root;
  uint32_t leaves;
  __device__ __forceinline__ uint32_t operator()(K key) const {
    float cdf;
    if (root.segments) {
      cdf = spline_cdf(static_cast<uint64_t>(key), reinterpret_cast<const uint8_t*>(root.knots), root);
    } else {
      const float u = key_unit(key, min_key, root.inv_range);
      cdf = root.hidden ? mlp_eval(root.mlp, root.hidden, u) : __builtin_fmaf(root.a, u, root.b);
    }
    return leaf_of(cdf, leaves);
  }
};

// start[l] = first position whose bin is >= l, for bins that ascend with the position
// (start[] pre-filled with n); counts the positions whose bin is below their predecessor's
// or at or past `bins` (neither occurs under a monotone model) in *bad.  The predecessor's
// bin comes from the neighbouring lane.
template <class K, class BinOf>
__device__ __forceinline__ void bin_starts(const K* __restrict__ col, uint64_t n, uint64_t bins, BinOf&& bin_of,
                                           uint32_t* __restrict__ start, unsigned long long* bad) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  const uint64_t first = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  for (uint64_t base = first - lane(); base < n; base += stride) {
    const uint64_t i = base + lane();
    const bool active = i < n;
    const uint64_t b = active ? bin_of(col[i]) : 0;
    uint64_t before = shfl64(b, lane() == 0 ? 0 : lane() - 1) + 1;  // the first bin that starts here
    if (lane() == 0) before = i == 0 ? 0 : bin_of(col[i - 1]) + 1;
    const bool wrong = active && (b >= bins || b + 1 < before);
    if (wrong) atomicAdd(bad, 1ull);
    const bool run = active && !wrong && b + 1 > before;
    fill_runs(start, static_cast<uint32_t>(before), run ? static_cast<uint32_t>(b + 1 - before) : 0u,
              static_cast<uint32_t>(i));
  }
}

template <class K>
__global__ __launch_bounds__(256) void leaf_bounds_kernel(const K* __restrict__ col, uint64_t n, Router<K> route,
                                                          uint32_t* __restrict__ start, unsigned long long* inversions) {
  bin_starts(col, n, route.leaves, [&](K key) { return static_cast<uint64_t>(route(key)); }, start, inversions);
}

// Build-time facts of one leaf (not read by lookups).
struct LeafFit {
  uint32_t start, count;
  int32_t err_lo, err_hi;  // extremes of position - pred over the leaf's keys
};

// Leaves are fitted and calibrated a wave each: the sums, the model and the error of every
// key of the leaf under the exact lookup arithmetic in one kernel, without atomics (a
// block per leaf and a pass of two atomics per key took 146 and 92 us over 2^20 keys in 2^16
// leaves; this takes 14 us).  What bounds it: the wave's latency over its few keys, so a
// leaf of more than kBigLeaf keys, which would be a long serial chain, is put on a list
// that blocks of 1024 threads work off.
constexpr uint32_t kBigLeaf = 4096;
constexpr uint32_t kSmallLeaf = 64;  // keys per leaf, on average, up to which 16 lanes take one
constexpr int kBigBlock = 1024;

// v reduced by `pick` over the T threads (a part of a wave, a wave, or a block) that work
// on a leaf; red: T / 64 entries of LDS, unused up to a wave.
template <int T, class V, class Pick>
__device__ __forceinline__ V leaf_reduce(V v, V* red, Pick&& pick) {
  for (int off = (T < kWave ? T : kWave) / 2; off > 0; off >>= 1) v = pick(v, __shfl_xor(v, off, kWave));
  if constexpr (T > kWave) {
    __syncthreads();
    if (lane() == 0) red[threadIdx.x / kWave] = v;
    __syncthreads();
    v = red[0];
    for (int w = 1; w < T / kWave; ++w) v = pick(v, red[w]);
  }
  return v;
}
template <int T>
__device__ __forceinline__ double leaf_sum(double v, double* red) {
  return leaf_reduce<T>(v, red, [](double a, double b) { return a + b; });
}

// Least squares of local position on FP32 key offsets over the keys at [s, s + cnt).
template <int T, class K>
__device__ __forceinline__ LeafModel leaf_fit(const K* __restrict__ col, uint64_t n, uint64_t s, uint64_t cnt,
                                              uint32_t t, double* red) {
  const uint64_t base = cnt ? static_cast<uint64_t>(col[s]) : 0;
  double sd = 0, sdd = 0, sj = 0, sdj = 0;
  for (uint64_t j = t; j < cnt; j += T) {
    const double d = leaf_dkey(col[s + j], base);
    const double jj = static_cast<double>(j);
    sd += d;
    sdd += d * d;
    sj += jj;
    sdj += d * jj;
  }
  sd = leaf_sum<T>(sd, red);
  sdd = leaf_sum<T>(sdd, red);
  sj = leaf_sum<T>(sj, red);
  sdj = leaf_sum<T>(sdj, red);
  double slope = 0, icpt = 0;
  if (cnt > 1) {
    const double c = static_cast<double>(cnt);
    const double var = sdd - sd * sd / c;
    if (var > 0) slope = (sdj - sd * sj / c) / var;
    icpt = (sj - slope * sd) / c;
  }
  double st = static_cast<double>(s) + std::floor(icpt + 0.5);
  st = st < 0 ? 0 : (st > static_cast<double>(n) ? static_cast<double>(n) : st);
  LeafModel m;
  m.base_key = base;
  m.start = static_cast<uint32_t>(st);
  m.slope = static_cast<float>(slope);
  return m;
}

// Extremes of position - pred(key) over the leaf's keys, as the leaf's calibration.  An
// empty leaf has none; one wider than max_width gets an emptied range (err_hi < err_lo).
template <int T, class K, class Pred>
__device__ __forceinline__ LeafFit leaf_calibrate(const K* __restrict__ col, uint64_t s, uint64_t cnt, uint32_t t,
                                                  int64_t max_width, int* red, Pred&& pred) {
  int lo = INT_MAX, hi = INT_MIN;
  for (uint64_t j = t; j < cnt; j += T) {
    int64_t e = static_cast<int64_t>(s + j) - pred(col[s + j]);
    e = e < INT_MIN / 2 ? INT_MIN / 2 : (e > INT_MAX / 2 ? INT_MAX / 2 : e);
    lo = static_cast<int>(e) < lo ? static_cast<int>(e) : lo;
    hi = static_cast<int>(e) > hi ? static_cast<int>(e) : hi;
  }
  lo = leaf_reduce<T>(lo, red, [](int a, int b) { return a < b ? a : b; });
  hi = leaf_reduce<T>(hi, red, [](int a, int b) { return a > b ? a : b; });
  LeafFit f{static_cast<uint32_t>(s), static_cast<uint32_t>(cnt), lo, hi};
  if (cnt == 0) {
    f.err_lo = f.err_hi = 0;
  } else if (static_cast<int64_t>(hi) - lo + 1 > max_width) {
    f.err_lo = 1;
    f.err_hi = 0;
  }
  return f;
}

// What a leaf kernel does with leaf l, covering positions [s, s + cnt), with T threads.
// Fits the 16-byte model; a leaf wider than max_width goes to the B-tree (slope = NaN).
template <class K>
struct FitLeaf {
  LeafModel* out;
  template <int T>
  __device__ __forceinline__ LeafFit run(const K* col, uint64_t n, uint32_t l, uint64_t s, uint64_t cnt, uint32_t t,
                                         int64_t max_width, void* red) const {
    LeafModel m = leaf_fit<T>(col, n, s, cnt, t, static_cast<double*>(red));
    const LeafFit f = leaf_calibrate<T>(col, s, cnt, t, max_width, static_cast<int*>(red),
                                        [&](K key) { return leaf_pred(m, leaf_dkey(key, m.base_key)); });
    if (f.err_hi < f.err_lo) {
      m.slope = __builtin_nanf("");
      m.start = kNoSplit;
    }
    if (t == 0) out[l] = m;
    return f;
  }
};

// 16-byte leaf -> compact leaf over its group: start + slope * (key - base) equals
// group.start + slope * (key - group.base) + icpt for icpt = start - group.start
// + slope * (group.base - base).
template <class K>
struct CompactLeaf {
  const LeafModel* lm;
  const LeafGroup* groups;
  uint32_t gshift;
  LeafCompact* out;
  template <int T>
  __device__ __forceinline__ LeafFit run(const K* col, uint64_t, uint32_t l, uint64_t s, uint64_t cnt, uint32_t t,
                                         int64_t max_width, void* red) const {
    const LeafModel m = lm[l];
    const LeafGroup g = groups[l >> gshift];
    double icpt = static_cast<double>(static_cast<int64_t>(m.start) - static_cast<int64_t>(g.start));
    if (m.slope != 0.0f)
      icpt += static_cast<double>(m.slope) * static_cast<double>(static_cast<int64_t>(g.base_key - m.base_key));
    const LeafCompact c{m.slope, static_cast<float>(icpt)};
    if (t == 0) out[l] = c;
    return leaf_calibrate<T>(col, s, cnt, t, max_width, static_cast<int*>(red),
                             [&](K key) { return compact_pred(c, g, leaf_dkey(key, g.base_key)); });
  }
};

// Leaf l covers positions [lo[l], hi[l]); big leaves are appended to `big`.
template <int T, class K, class Op>
__global__ __launch_bounds__(256) void leaf_wave_kernel(const K* __restrict__ col, uint64_t n,
                                                        const uint32_t* __restrict__ lo, const uint32_t* __restrict__ hi,
                                                        uint32_t leaves, int64_t max_width, Op op,
                                                        LeafFit* __restrict__ fit, uint32_t* __restrict__ big_count,
                                                        uint32_t* __restrict__ big) {
  const uint32_t l = blockIdx.x * (256 / T) + threadIdx.x / T;
  if (l >= leaves) return;
  const uint64_t s = lo[l], e = hi[l];
  const uint64_t cnt = e > s ? e - s : 0;
  const uint32_t t = threadIdx.x % T;
  if (cnt > kBigLeaf) {
    if (t == 0) big[atomicAdd(big_count, 1u)] = l;
    return;
  }
  const LeafFit f = op.template run<T>(col, n, l, s, cnt, t, max_width, nullptr);
  if (t == 0) fit[l] = f;
}

template <class K, class Op>
__global__ __launch_bounds__(kBigBlock) void leaf_big_kernel(const K* __restrict__ col, uint64_t n,
                                                             const uint32_t* __restrict__ lo,
                                                             const uint32_t* __restrict__ hi, int64_t max_width, Op op,
                                                             LeafFit* __restrict__ fit,
                                                             const uint32_t* __restrict__ big_count,
                                                             const uint32_t* __restrict__ big) {
  __shared__ double red[kBigBlock / kWave];
  const uint32_t count = *big_count;
  for (uint32_t q = blockIdx.x; q < count; q += gridDim.x) {
    const uint32_t l = big[q];
    const uint64_t s = lo[l];
    const LeafFit f = op.template run<kBigBlock>(col, n, l, s, hi[l] - s, threadIdx.x, max_width, red);
    if (threadIdx.x == 0) fit[l] = f;
    __syncthreads();  // the next leaf's reductions reuse red
  }
}

// Totals over the leaves, those with an emptied range (routed to the B-tree) apart.
struct LeafStats {
  unsigned long long fb_leaves, fb_keys, wsum, wkeys;  // wsum: window widths weighted by keys
  uint32_t wmax;
  int32_t err_lo, err_hi;
  uint32_t big;  // entries of the big-leaf list
};
__global__ __launch_bounds__(kBigBlock) void leaf_stats_kernel(const LeafFit* __restrict__ fit, uint32_t leaves,
                                                         LeafStats* __restrict__ st) {
  uint64_t fbl = 0, fbk = 0, ws = 0, wk = 0;
  uint32_t wm = 0;
  int lo = 0, hi = 0;
  for (uint32_t l = blockIdx.x * blockDim.x + threadIdx.x; l < leaves; l += gridDim.x * blockDim.x) {
    const LeafFit f = fit[l];
    if (f.count == 0) continue;
    if (f.err_hi < f.err_lo) {
      ++fbl;
      fbk += f.count;
    } else {
      const uint32_t w = static_cast<uint32_t>(f.err_hi - f.err_lo + 1);
      wm = w > wm ? w : wm;
      ws += static_cast<uint64_t>(w) * f.count;
      wk += f.count;
      lo = f.err_lo < lo ? f.err_lo : lo;
      hi = f.err_hi > hi ? f.err_hi : hi;
    }
  }
  // block totals first: atomics on one address cost 10 ns each
  __shared__ LeafStats part[kBigBlock / kWave];
  LeafStats t{wave_sum(fbl), wave_sum(fbk), wave_sum(ws), wave_sum(wk), wave_max(wm), wave_min(lo), wave_max(hi), 0};
  if (lane() == 0) part[threadIdx.x / kWave] = t;
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < kBigBlock / kWave; ++w) {
    t.fb_leaves += part[w].fb_leaves;
    t.fb_keys += part[w].fb_keys;
    t.wsum += part[w].wsum;
    t.wkeys += part[w].wkeys;
    t.wmax = part[w].wmax > t.wmax ? part[w].wmax : t.wmax;
    t.err_lo = part[w].err_lo < t.err_lo ? part[w].err_lo : t.err_lo;
    t.err_hi = part[w].err_hi > t.err_hi ? part[w].err_hi : t.err_hi;
  }
  if (t.fb_leaves) {
    atomicAdd(&st->fb_leaves, t.fb_leaves);
    atomicAdd(&st->fb_keys, t.fb_keys);
  }
  if (t.wkeys) {
    atomicAdd(&st->wsum, t.wsum);
    atomicAdd(&st->wkeys, t.wkeys);
    atomicMax(&st->wmax, t.wmax);
    if (t.err_lo < 0) atomicMin(&st->err_lo, t.err_lo);
    if (t.err_hi > 0) atomicMax(&st->err_hi, t.err_hi);
  }
}

// Runs Op over the leaves and reads their totals back.
struct LeafPass {
  dbuf work;  // LeafStats | big-leaf list
  template <class K, class Op>
  LeafStats run(const K* col, uint64_t n, const uint32_t* lo, const uint32_t* hi, uint32_t leaves, int64_t max_width,
                const Op& op, LeafFit* fit, hipStream_t s) {
    const uint64_t bigs = std::min<uint64_t>(leaves, n / kBigLeaf + 1);
    work.reserve(sizeof(LeafStats) + bigs * sizeof(uint32_t));
    LeafStats* st = work.as<LeafStats>();
    uint32_t* big = reinterpret_cast<uint32_t*>(st + 1);
    fill_bytes(st, 0, sizeof(LeafStats), s);
    auto fit_with = [&]<int T>() {
      hipLaunchKernelGGL((leaf_wave_kernel<T, K, Op>), dim3(grid_for(leaves, 256 / T, 0x7FFFFFFFu)), dim3(256), 0, s, col,
                         n, lo, hi, leaves, max_width, op, fit, &st->big, big);
    };
    if (n / leaves <= kSmallLeaf)
      fit_with.template operator()<16>();
    else
      fit_with.template operator()<kWave>();
    GJ_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL((leaf_big_kernel<K, Op>), dim3(static_cast<unsigned>(std::min<uint64_t>(bigs, 256))),
                       dim3(kBigBlock), 0, s, col, n, lo, hi, max_width, op, fit, &st->big, big);
    GJ_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(leaf_stats_kernel, dim3(grid_for(leaves, kBigBlock, 32)), dim3(kBigBlock), 0, s, fit, leaves, st);
    GJ_HIP_CHECK(hipGetLastError());
    LeafStats h{};
    GJ_HIP_CHECK(hipMemcpyAsync(&h, st, sizeof(h), hipMemcpyDeviceToHost, s));
    GJ_HIP_CHECK(hipStreamSynchronize(s));
    return h;
  }
};

// Separator line of split j: sub-leaf t covers [sub_lo, sub_hi); its separator is the
// key at sub_hi - 1 (at the leaf's first position for an empty leading sub-leaf), the
// last separator is all ones, so the count of separators below a key of the split
// leaf is the index of the sub-leaf that holds it.
template <class K>
__global__ void split_sep_kernel(const K* __restrict__ col, const uint32_t* __restrict__ sub_lo,
                                 const uint32_t* __restrict__ sub_hi, const uint32_t* __restrict__ leaf_lo,
                                 uint32_t splits, uint64_t* __restrict__ sep) {
  const uint64_t g = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (g >= static_cast<uint64_t>(splits) * kSplitWays) return;
  const uint32_t t = static_cast<uint32_t>(g % kSplitWays);
  const uint32_t j = static_cast<uint32_t>(g / kSplitWays);
  if (t == kSplitWays - 1) {
    sep[g] = ~0ull;
    return;
  }
  const uint32_t h = sub_hi[g];
  const uint32_t at = h > leaf_lo[j] ? h - 1 : leaf_lo[j];
  sep[g] = static_cast<uint64_t>(col[at]);
}

// The split leaves' own models: slope = NaN, start = split index.
__global__ void split_mark_kernel(LeafModel* __restrict__ lm, const uint32_t* __restrict__ leaf_id, uint32_t splits) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= splits) return;
  LeafModel m;
  m.base_key = 0;
  m.start = j;
  m.slope = __builtin_nanf("");
  lm[leaf_id[j]] = m;
}

// Group g of the compact leaves starts at the first position routed to leaf
// g << gshift or a later leaf (start[] of leaf_bounds_kernel).
template <class K>
__global__ void compact_groups_kernel(const K* __restrict__ col, uint64_t n, const uint32_t* __restrict__ start,
                                      uint32_t groups, uint32_t gshift, LeafGroup* __restrict__ out) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= groups) return;
  const uint32_t st = start[static_cast<uint64_t>(g) << gshift];
  LeafGroup r;
  r.start = st;
  r.base_key = st < n ? static_cast<uint64_t>(col[st]) : static_cast<uint64_t>(col[n - 1]);
  r.pad = 0;
  out[g] = r;
}

// ---- lines layout ------------------------------------------------------------

// What the placement reports to the host.
struct LineStats {
  unsigned long long bad;    // keys whose target is not monotone or not below the line count
  unsigned long long carry;  // sum over lines l of the keys with a target below l that are placed at l or later
  uint32_t base_end;         // first key past the target lines
  uint32_t max_spill;        // farthest line from its first key's target
};

// first[l] = first position whose target line is >= l (first[] pre-filled with n).
template <class K>
__global__ __launch_bounds__(256) void line_first_kernel(const K* __restrict__ col, uint64_t n, LinesDev<K> d,
                                                         const uint8_t* rp, uint64_t targets,
                                                         uint32_t* __restrict__ first, LineStats* st) {
  bin_starts(col, n, targets, [&](K key) { return d.target(key, rp); }, first, &st->bad);
}

// Placement.  In key order, line l takes the keys carried over from line l - 1, then its own
// (targets of l), up to CAP; the rest moves on.  With base[l] = keys placed before line l:
//   base[l + 1] = min(first[l + 1], base[l] + CAP), hence
//   base[l] = CAP * l + min over j <= l of (first[j] - CAP * j),
// a running minimum: one pass for the minima of the blocks' spans, one that scans each span
// from the minimum before it.  Past the last target line every line takes CAP keys, so
// base[targets + k] = min(n, base[targets] + CAP * k) needs no entry.
// What bounds it: streaming.  On the host the same recurrence cost 3.0 of the 4.4 ms of a
// build over 12.3 M u64 keys (1.23 M lines), and its arrays another 0.8 ms of copies;
// the two passes take 17 us.
constexpr int kPlaceBlock = 256;
constexpr int kPlaceItems = 8;                              // consecutive lines per thread
constexpr uint64_t kPlaceTile = kPlaceBlock * kPlaceItems;  // lines per step of a block
constexpr uint64_t kPlaceBlocks = 2048;                     // each block reads the minima of all earlier ones

__device__ __forceinline__ int64_t block_min(int64_t v, int64_t* red) {
  v = wave_min(v);
  __syncthreads();
  if (lane() == 0) red[threadIdx.x / kWave] = v;
  __syncthreads();
  int64_t r = red[0];
  for (int w = 1; w < kPlaceBlock / kWave; ++w) r = red[w] < r ? red[w] : r;
  return r;
}

template <uint32_t CAP>
__global__ __launch_bounds__(kPlaceBlock) void line_span_min_kernel(const uint32_t* __restrict__ first, uint64_t entries,
                                                                    uint64_t span, int64_t* __restrict__ mins) {
  __shared__ int64_t red[kPlaceBlock / kWave];
  const uint64_t lo = blockIdx.x * span, hi = lo + span < entries ? lo + span : entries;
  int64_t m = INT64_MAX;
  for (uint64_t j = lo + threadIdx.x; j < hi; j += kPlaceBlock) {
    const int64_t f = static_cast<int64_t>(first[j]) - static_cast<int64_t>(j * CAP);
    m = f < m ? f : m;
  }
  m = block_min(m, red);
  if (threadIdx.x == 0) mins[blockIdx.x] = m;
}

// base[] continued past the target lines
struct LineBases {
  const uint32_t* base;  // targets + 1 entries
  uint64_t targets;
  uint32_t end;  // base[targets]
  uint32_t n, cap;
  __device__ __forceinline__ uint32_t operator()(uint64_t l) const {
    if (l <= targets) return base[l];
    const uint64_t b = end + (l - targets) * cap;
    return b < n ? static_cast<uint32_t>(b) : n;
  }
};

// The leaves whose lines [line0[j], line0[j + 1]) are marked as the source of a run.
struct LeafMarks {
  const uint32_t* line0;  // leaves + 1 entries; null: no marks
  uint32_t leaves;
  uint8_t* mark;
  __device__ __forceinline__ void set(uint64_t line) const {
    if (!line0) return;
    uint32_t lo = 0, len = leaves + 1;  // lo: entries of line0 that are <= line
    while (len > 0) {
      const uint32_t half = len >> 1;
      if (line0[lo + half] <= line) {
        lo += half + 1;
        len -= half + 1;
      } else {
        len = half;
      }
    }
    if (lo >= 1 && lo - 1 < leaves) mark[lo - 1] = 1;
  }
};

// How far line l (first key at position b) lies from its first key's target, the smallest
// target in the line; marks the leaf of a target that a key spills two or more lines from.
template <class K>
__device__ __forceinline__ uint32_t line_spill(const K* __restrict__ col, const LinesDev<K>& d, const uint8_t* rp,
                                               uint64_t l, uint32_t b, const LeafMarks& marks) {
  const uint64_t t = d.target(col[b], rp);
  const uint32_t spill = t < l ? static_cast<uint32_t>(l - t) : 0u;
  if (spill >= 2) marks.set(t);
  return spill;
}

// One span's contribution to the placement's totals.  Blocks store theirs and one block
// adds them up: thousands of atomics on one address cost 10 ns each (215 us of the 430 us
// that the placement's kernels took with them).
struct SpanTotals {
  unsigned long long carry;
  uint32_t max_spill, pad;
};

template <class K>
__global__ __launch_bounds__(kPlaceBlock) void line_base_kernel(const K* __restrict__ col, uint32_t n, LinesDev<K> d,
                                                                const uint8_t* rp, const uint32_t* __restrict__ first,
                                                                uint64_t entries, uint64_t span,
                                                                const int64_t* __restrict__ mins, LeafMarks marks,
                                                                uint32_t* __restrict__ base,
                                                                SpanTotals* __restrict__ totals) {
  constexpr uint32_t CAP = LinesDev<K>::CAP;
  __shared__ int64_t red[kPlaceBlock / kWave];
  const uint64_t lo = blockIdx.x * span, hi = lo + span < entries ? lo + span : entries;
  int64_t run = INT64_MAX;  // the minimum over every earlier line
  for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kPlaceBlock) run = mins[b] < run ? mins[b] : run;
  run = block_min(run, red);
  uint64_t carry = 0;
  uint32_t worst = 0;
  for (uint64_t tile = lo; tile < hi; tile += kPlaceTile) {
    const uint64_t at = tile + static_cast<uint64_t>(threadIdx.x) * kPlaceItems;
    uint32_t v[kPlaceItems + 1];
    int64_t m[kPlaceItems];  // running minimum inside the thread
    int64_t mine = INT64_MAX;
#pragma unroll
    for (int k = 0; k <= kPlaceItems; ++k) v[k] = at + k < entries ? first[at + k] : n;
#pragma unroll
    for (int k = 0; k < kPlaceItems; ++k) {
      const int64_t f = static_cast<int64_t>(v[k]) - static_cast<int64_t>((at + k) * CAP);
      mine = at + k < hi && f < mine ? f : mine;
      m[k] = mine;
    }
    // minimum over the lanes before this one, then over the waves before this one
    int64_t incl = mine;
    for (int off = 1; off < kWave; off <<= 1) {
      const int64_t o = __shfl_up(incl, off, kWave);
      if (lane() >= off && o < incl) incl = o;
    }
    int64_t before = __shfl_up(incl, 1, kWave);
    if (lane() == 0) before = INT64_MAX;
    __syncthreads();  // the last step's readers of red[]
    if (lane() == kWave - 1) red[threadIdx.x / kWave] = incl;
    __syncthreads();
    int64_t all = run;
#pragma unroll
    for (int w = 0; w < kPlaceBlock / kWave; ++w) {
      if (w < static_cast<int>(threadIdx.x / kWave)) before = red[w] < before ? red[w] : before;
      all = red[w] < all ? red[w] : all;
    }
    before = run < before ? run : before;
    run = all;
#pragma unroll
    for (int k = 0; k < kPlaceItems; ++k) {
      if (at + k < hi) {
        const int64_t mk = m[k] < before ? m[k] : before;
        const uint32_t b = static_cast<uint32_t>(mk + static_cast<int64_t>((at + k) * CAP));
        base[at + k] = b;
        carry += v[k] - b;
        // only a line behind a full one holds keys of earlier targets; an empty one none
        if (b < v[k] && at + k + 1 < entries && b < v[k + 1]) {
          const uint32_t s = line_spill(col, d, rp, at + k, b, marks);
          worst = s > worst ? s : worst;
        }
      }
    }
  }
  carry = wave_sum(carry);
  worst = wave_max(worst);
  __shared__ SpanTotals part[kPlaceBlock / kWave];
  if (lane() == 0) part[threadIdx.x / kWave] = SpanTotals{carry, worst, 0};
  __syncthreads();
  if (threadIdx.x == 0) {
    SpanTotals t = part[0];
    for (int w = 1; w < kPlaceBlock / kWave; ++w) {
      t.carry += part[w].carry;
      t.max_spill = part[w].max_spill > t.max_spill ? part[w].max_spill : t.max_spill;
    }
    totals[blockIdx.x] = t;
  }
}

// Adds the spans up (block 0) and looks at the lines past the targets, if there are any.
template <class K>
__global__ __launch_bounds__(kPlaceBlock) void line_total_kernel(const K* __restrict__ col, uint32_t n, LinesDev<K> d,
                                                                 const uint8_t* rp, const uint32_t* __restrict__ base,
                                                                 uint64_t targets, LeafMarks marks,
                                                                 const SpanTotals* __restrict__ totals, uint32_t spans,
                                                                 LineStats* st) {
  constexpr uint32_t CAP = LinesDev<K>::CAP;
  const LineBases at{base, targets, base[targets], n, CAP};
  const uint64_t tail = (static_cast<uint64_t>(n - at.end) + CAP - 1) / CAP;
  uint64_t carry = 0;
  uint32_t worst = 0;
  if (blockIdx.x == 0) {
    for (uint32_t b = threadIdx.x; b < spans; b += kPlaceBlock) {
      carry += totals[b].carry;
      worst = totals[b].max_spill > worst ? totals[b].max_spill : worst;
    }
    if (threadIdx.x == 0) st->base_end = at.end;
  }
  for (uint64_t k = static_cast<uint64_t>(blockIdx.x) * kPlaceBlock + threadIdx.x; k < tail;
       k += static_cast<uint64_t>(gridDim.x) * kPlaceBlock) {
    const uint32_t s = line_spill(col, d, rp, targets + k, at(targets + k), marks);
    worst = s > worst ? s : worst;
  }
  carry = wave_sum(carry);
  worst = wave_max(worst);
  if (lane() != 0) return;
  if (carry) atomicAdd(&st->carry, static_cast<unsigned long long>(carry));
  if (worst) atomicMax(&st->max_spill, worst);
}

// Line l holds the keys at positions [base(l), base(l + 1)), after its header.
template <class K>
__global__ void line_fill_kernel(const K* __restrict__ col, LineBases base, uint64_t lines, K* __restrict__ out) {
  using D = LinesDev<K>;
  const uint64_t slots = lines * D::SLOTS;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t g = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < slots; g += stride) {
    const uint64_t l = g / D::SLOTS;
    const uint32_t sl = static_cast<uint32_t>(g % D::SLOTS);
    const uint32_t b = base(l);
    const uint32_t cnt = base(l + 1) - b;
    K v;
    if (sl < D::HDR) {
      const uint64_t hdr = (static_cast<uint64_t>(cnt) << 32) | b;
      v = static_cast<K>(sizeof(K) == 8 ? hdr : (sl == 0 ? (hdr & 0xFFFFFFFFull) : (hdr >> 32)));
    } else {
      const uint32_t k = sl - D::HDR;
      v = k < cnt ? col[static_cast<uint64_t>(b) + k] : key_max<K>();
    }
    out[g] = v;
  }
}

// Two-stage leaves: leaf l maps its keys [start[l], start[l + 1]) linearly onto its
// lines [line0[l], line0[l + 1]).
template <class K>
__global__ void line_leaf_kernel(const K* __restrict__ col, const uint32_t* __restrict__ start,
                                 const uint32_t* __restrict__ line0, uint32_t leaves, LineLeaf* __restrict__ out) {
  const uint32_t l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= leaves) return;
  const uint32_t a = start[l], b = start[l + 1];
  LineLeaf f;
  f.line0 = line0[l];
  if (b > a) {
    const uint64_t k0 = static_cast<uint64_t>(col[a]);
    const uint64_t span = static_cast<uint64_t>(col[b - 1]) - k0;
    const uint32_t nl = line0[l + 1] - line0[l];
    f.key0 = k0;
    f.scale = static_cast<float>(static_cast<double>(nl) / (static_cast<double>(span) + 1.0));
  } else {
    f.key0 = 0;
    f.scale = 0.0f;
  }
  out[l] = f;
}

// A lines-layout build under one target model; the candidate holds its buffers
// until it is adopted by the index or dropped.
struct LinesBuild {
  dbuf lines, leaves;
  uint64_t num_lines = 0, mult = 0;
  uint32_t num_leaves = 0, max_lines = 0;
  double avg_lines = 0.0;
  RootModel root{};
  bool ok = false;
};

// Working memory of a placement: first | base | span minima | span totals | stats | marks.
struct Placement {
  dbuf buf;
  uint64_t targets = 0;
  uint32_t *first = nullptr, *base = nullptr;
  LineStats* stats = nullptr;
  uint8_t* mark = nullptr;
  LineStats h{};

  // Places the keys under target model d (d.leaves / d.mult already set; d.lines unused)
  // over `targets` target lines plus whatever tail lines the last full lines push keys
  // into, and reads the outcome back.  line0 (optional, `leaves` + 1 entries): mark[j]
  // is set for the leaves that keys spill two or more lines from.
  template <class K>
  void measure(const gj_index& ix, LinesDev<K> d, const uint8_t* rp, uint64_t lines, hipStream_t s,
               const uint32_t* line0 = nullptr, uint32_t leaves = 0) {
    constexpr uint32_t CAP = LinesDev<K>::CAP;
    const K* col = static_cast<const K*>(ix.d_col);
    const uint64_t n = ix.n, entries = lines + 1;
    targets = lines;
    auto up = [](uint64_t b) { return (b + 255) / 256 * 256; };
    const uint64_t o_base = up(entries * 4), o_min = o_base + up(entries * 4), o_tot = o_min + up(kPlaceBlocks * 8),
                   o_st = o_tot + up(kPlaceBlocks * sizeof(SpanTotals)), o_mark = o_st + up(sizeof(LineStats));
    buf.reserve(o_mark + up(line0 ? leaves : 0));
    uint8_t* p = buf.as<uint8_t>();
    first = reinterpret_cast<uint32_t*>(p);
    base = reinterpret_cast<uint32_t*>(p + o_base);
    stats = reinterpret_cast<LineStats*>(p + o_st);
    mark = line0 ? p + o_mark : nullptr;
    int64_t* mins = reinterpret_cast<int64_t*>(p + o_min);
    SpanTotals* totals = reinterpret_cast<SpanTotals*>(p + o_tot);
    const LeafMarks marks{line0, leaves, mark};
    fill_words(first, entries, static_cast<uint32_t>(n), s);
    fill_bytes(stats, 0, o_mark - o_st + (line0 ? leaves : 0), s);  // and the marks behind them
    hipLaunchKernelGGL(line_first_kernel<K>, dim3(grid_for(n, 256)), dim3(256), 0, s, col, n, d, rp, targets, first,
                       stats);
    GJ_HIP_CHECK(hipGetLastError());
    const uint64_t span = ceil_div(std::max<uint64_t>(kPlaceTile, ceil_div(entries, kPlaceBlocks)), kPlaceTile) * kPlaceTile;
    const unsigned blocks = static_cast<unsigned>(ceil_div(entries, span));
    hipLaunchKernelGGL((line_span_min_kernel<CAP>), dim3(blocks), dim3(kPlaceBlock), 0, s, first, entries, span, mins);
    GJ_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(line_base_kernel<K>, dim3(blocks), dim3(kPlaceBlock), 0, s, col, static_cast<uint32_t>(n), d, rp,
                       first, entries, span, mins, marks, base, totals);
    GJ_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(line_total_kernel<K>, dim3(64), dim3(kPlaceBlock), 0, s, col, static_cast<uint32_t>(n), d, rp,
                       base, targets, marks, totals, blocks, stats);
    GJ_HIP_CHECK(hipGetLastError());
    GJ_HIP_CHECK(hipMemcpyAsync(&h, stats, sizeof(h), hipMemcpyDeviceToHost, s));
    GJ_HIP_CHECK(hipStreamSynchronize(s));
    GJ_REQUIRE(h.bad == 0, GJ_ERR_INTERNAL, "learned lines: target model is not monotone");
  }

  // Writes the lines of the measured placement.
  template <class K>
  void emit(const gj_index& ix, LinesBuild& out, hipStream_t s) const {
    constexpr uint32_t CAP = LinesDev<K>::CAP;
    const uint64_t n = ix.n;
    // tail lines: what the last full lines push on, CAP keys at a time
    const uint64_t rest = n - h.base_end, tail = ceil_div(rest, CAP);
    double carry = static_cast<double>(h.carry);
    if (tail > 1)
      carry += static_cast<double>(tail - 1) * static_cast<double>(rest) -
               static_cast<double>(CAP) * 0.5 * static_cast<double>(tail - 1) * static_cast<double>(tail);
    out.num_lines = targets + tail;
    out.avg_lines = 1.0 + carry / static_cast<double>(n);
    out.max_lines = h.max_spill + 1;
    out.lines.alloc(out.num_lines * 128);
    const LineBases at{base, targets, h.base_end, static_cast<uint32_t>(n), CAP};
    hipLaunchKernelGGL(line_fill_kernel<K>, dim3(grid_for(out.num_lines * LinesDev<K>::SLOTS, 256)), dim3(256), 0, s,
                       static_cast<const K*>(ix.d_col), at, out.num_lines, out.lines.as<K>());
    GJ_HIP_CHECK(hipGetLastError());
    GJ_HIP_CHECK(hipStreamSynchronize(s));  // the placement's working memory may go
    out.ok = true;
  }
};

// Root-only lines: the key range spread linearly over ceil(n / line_keys) lines.
template <class K>
void lines_root_only(const gj_index& ix, uint32_t line_keys, LinesBuild& out, hipStream_t s) {
  const uint64_t targets = std::max<uint64_t>(1, ceil_div(ix.n, line_keys));
  const unsigned __int128 den = static_cast<unsigned __int128>(ix.max_key - ix.min_key) + 1;
  // mult = floor(targets * 2^64 / (range + 1)), so umulhi(range, mult) < targets; capped at
  // 2^64 - 1 for a range narrower than the line count (then target <= key - min_key)
  const unsigned __int128 q = (static_cast<unsigned __int128>(targets) << 64) / den;
  out.mult = q > static_cast<unsigned __int128>(~0ull) ? ~0ull : static_cast<uint64_t>(q);
  LinesDev<K> d{};
  d.min_key = static_cast<K>(ix.min_key);
  d.max_key = static_cast<K>(ix.max_key);
  d.mult = out.mult;
  out.num_leaves = 0;
  out.root = RootModel{};
  Placement pl;
  pl.measure<K>(ix, d, nullptr, targets, s);
  pl.emit<K>(ix, out, s);
}

// Two-stage lines: `root` routes keys to 2^bits leaves; each leaf gets lines for its
// keys at line_keys per line and maps its key span linearly onto them.
template <class K>
void lines_two_stage(const gj_index& ix, const RootModel& root, uint32_t bits, uint32_t line_keys, LinesBuild& out,
                     hipStream_t s) {
  const K* col = static_cast<const K*>(ix.d_col);
  const uint64_t n = ix.n;
  const uint32_t L = 1u << bits;
  const K kmin = static_cast<K>(ix.min_key);
  Router<K> route{kmin, root, L};
  dbuf start((static_cast<uint64_t>(L) + 1) * sizeof(uint32_t));
  std::vector<uint32_t> hs(L + 1);
  {
    fill_words(start.as<uint32_t>(), hs.size(), static_cast<uint32_t>(n), s);
    dbuf inv(sizeof(unsigned long long));
    fill_bytes(inv.p, 0, inv.bytes, s);
    hipLaunchKernelGGL(leaf_bounds_kernel<K>, dim3(grid_for(n, 256)), dim3(256), 0, s, col, n, route,
                       start.as<uint32_t>(), inv.as<unsigned long long>());
    GJ_HIP_CHECK(hipGetLastError());
    unsigned long long hinv = 0;
    GJ_HIP_CHECK(hipMemcpyAsync(&hinv, inv.p, sizeof(hinv), hipMemcpyDeviceToHost, s));
    GJ_HIP_CHECK(hipMemcpyAsync(hs.data(), start.p, hs.size() * 4, hipMemcpyDeviceToHost, s));
    GJ_HIP_CHECK(hipStreamSynchronize(s));
    GJ_REQUIRE(hinv == 0, GJ_ERR_INTERNAL, "learned lines: root model is not monotone");
  }
  // A leaf whose keys are not evenly spread over its key span overfills some of its lines,
  // and the surplus runs on through the following lines; a lookup wave walks as far as its
  // farthest probe.  So the leaves that source a run of two or more lines get twice their
  // lines (half the load where their keys crowd), and the placement is redone, up to
  // kInflateRounds times.
  constexpr int kInflateRounds = 4;
  constexpr uint32_t kMaxInflate = 16;
  std::vector<uint32_t> inflate(L, 1), line0(L + 1, 0);
  std::vector<uint8_t> mark(L);
  Placement pl;
  dbuf d_line0((static_cast<uint64_t>(L) + 1) * sizeof(uint32_t));
  out.leaves.alloc(sizeof(LineLeaf) * L);
  out.num_leaves = L;
  out.root = root;
  for (int round = 0;; ++round) {
    uint64_t lines = 0;
    for (uint32_t l = 0; l < L; ++l) {
      line0[l] = static_cast<uint32_t>(lines);
      const uint64_t c = static_cast<uint64_t>(hs[l + 1]) - hs[l];
      lines += ceil_div(c * inflate[l], line_keys);
    }
    GJ_REQUIRE(lines < 0xFFFFFFFFull, GJ_ERR_OVERFLOW, "learned lines: too many lines");
    line0[L] = static_cast<uint32_t>(lines);
    GJ_HIP_CHECK(hipMemcpyAsync(d_line0.p, line0.data(), line0.size() * 4, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(line_leaf_kernel<K>, dim3(grid_for(L, 256)), dim3(256), 0, s, col,
                       start.as<const uint32_t>(), d_line0.as<const uint32_t>(), L, out.leaves.as<LineLeaf>());
    GJ_HIP_CHECK(hipGetLastError());
    LinesDev<K> d{};
    d.min_key = kmin;
    d.max_key = static_cast<K>(ix.max_key);
    d.root = root;
    d.leaves = out.leaves.as<const LineLeaf>();
    d.num_leaves = L;
    // FP32 rounding can carry a leaf's last keys to floor(p) = its line count, the first
    // line of the next leaf (still monotone); for the last leaf that is target line `lines`
    pl.measure<K>(ix, d, reinterpret_cast<const uint8_t*>(root.params()), lines + 1, s, d_line0.as<const uint32_t>(), L);
    if (pl.h.max_spill <= 1 || round + 1 >= kInflateRounds) break;
    GJ_HIP_CHECK(hipMemcpyAsync(mark.data(), pl.mark, L, hipMemcpyDeviceToHost, s));
    GJ_HIP_CHECK(hipStreamSynchronize(s));
    bool grew = false;
    for (uint32_t j = 0; j < L; ++j) {
      if (mark[j] && inflate[j] < kMaxInflate) {
        inflate[j] *= 2;
        grew = true;
      }
    }
    if (!grew) break;
  }
  pl.emit<K>(ix, out, s);
}

// Adopts a lines build into the index: the column layout's leaves are not needed.
void adopt_lines(gj_index& ix, LinesBuild& b) {
  ix.lm_layout = GJ_LAYOUT_LINES;
  ix.lm_lines = std::move(b.lines);
  ix.lm_line_leaves = std::move(b.leaves);
  ix.lm_num_lines = b.num_lines;
  ix.lm_mult = b.mult;
  ix.lm_num_line_leaves = b.num_leaves;
  ix.lm_root = b.root;
  ix.lm_leaves.release();
  ix.lm_groups.release();
  ix.lm_seps.release();
  ix.lm_subs.release();
  ix.lm_compact = false;
  ix.lm_splits = 0;
  ix.lm_fallback_any = 0;
  ix.stats.layout = GJ_LAYOUT_LINES;
  ix.stats.lines = b.num_lines;
  ix.stats.avg_lines = b.avg_lines;
  ix.stats.max_lines = b.max_lines;
  ix.stats.leaves = b.num_leaves;
  ix.stats.root_segments = b.root.segments;
  ix.stats.fallback_leaves = 0;
  ix.stats.fallback_keys = 0;
  ix.stats.split_leaves = 0;
  ix.stats.max_window = 0;
  ix.stats.avg_window = 0.0;
  ix.stats.depth = b.num_leaves ? 2 : 1;
  ix.stats.lds_levels = 0;
}

}  // namespace

template <class K>
void build_learned(gj_index& ix, hipStream_t s) {
  const K* col = static_cast<const K*>(ix.d_col);
  const uint64_t n = ix.n;
  // default: 2^16 16-byte leaves (1 MiB, L2-resident) up to 2^26 keys, then about 1024
  // keys per leaf; twice as many compact leaves in the same bytes where the build admits them
  uint32_t bits = ix.params.learned_leaf_bits;
  if (bits == 0) bits = static_cast<uint32_t>(std::clamp(static_cast<int>(ilog2_ceil(n)) - 10, 16, 24));
  GJ_REQUIRE(bits >= 1 && bits <= 24, GJ_ERR_INVALID, "learned_leaf_bits must be in [1, 24]");
  uint32_t L = 1u << bits;  // leaves of the build in progress
  const K kmin = static_cast<K>(ix.min_key);
  const uint64_t range = ix.max_key - ix.min_key;
  RootModel root{};
  root.inv_range = range ? 1.0f / static_cast<float>(range) : 0.0f;
  std::vector<float> mlp_init;  // the MLP root's parameters before training
  ix.stats.root_trained = (ix.kind == GJ_LEARNED_MLP && !(ix.params.learned_flags & GJ_LEARNED_UNTRAINED)) ? 1u : 0u;

  // learned_plr's linear root, fitted when the first candidate that routes by it is built
  bool root_fitted = false;
  auto fit_root = [&] {
    if (ix.kind != GJ_LEARNED_PLR || root.segments || root_fitted) return;
    root_fitted = true;
    const unsigned blocks = grid_for(n, 256, 2048);
    dbuf partial(sizeof(RootFitSums) * blocks);
    hipLaunchKernelGGL(root_sums_kernel<K>, dim3(blocks), dim3(256), 0, s, col, n, kmin, root.inv_range,
                       partial.as<RootFitSums>());
    GJ_HIP_CHECK(hipGetLastError());
    std::vector<RootFitSums> h(blocks);
    GJ_HIP_CHECK(hipMemcpyAsync(h.data(), partial.p, partial.bytes, hipMemcpyDeviceToHost, s));
    GJ_HIP_CHECK(hipStreamSynchronize(s));
    RootFitSums t{0, 0, 0, 0};
    for (const auto& r : h) {
      t.sx += r.sx;
      t.sxx += r.sxx;
      t.st += r.st;
      t.sxt += r.sxt;
    }
    const double c = static_cast<double>(n);
    const double var = t.sxx - t.sx * t.sx / c;
    double a = var > 0 ? (t.sxt - t.sx * t.st / c) / var : 0.0;
    if (a < 0) a = 0;
    root.a = static_cast<float>(a);
    root.b = static_cast<float>((t.st - a * t.sx) / c);
  };
  if (ix.kind == GJ_LEARNED_MLP) {
    const uint32_t h = ix.params.mlp_hidden;
    GJ_REQUIRE(h == 8 || h == 16 || h == 32 || h == 64, GJ_ERR_INVALID, "mlp_hidden must be 8, 16, 32 or 64");
    const uint32_t np = 3 * h + 1;
    // ramp k rises from 0 at quantile k/h of the keys to 1 at quantile (k+1)/h, weight 1/h:
    // the initial root is the piecewise-linear CDF through h + 1 quantiles
    std::vector<float> q(h + 1);
    for (uint32_t k = 0; k <= h; ++k) {
      const uint64_t i = std::min<uint64_t>(n - 1, (static_cast<uint64_t>(k) * n) / h);
      K key;
      GJ_HIP_CHECK(hipMemcpyAsync(&key, col + i, sizeof(K), hipMemcpyDeviceToHost, s));
      GJ_HIP_CHECK(hipStreamSynchronize(s));
      q[k] = static_cast<float>(static_cast<uint64_t>(key - kmin)) * root.inv_range;
    }
    std::vector<float> p0(np, 0.0f);
    for (uint32_t k = 0; k < h; ++k) {
      const float w = q[k + 1] - q[k];
      p0[k] = w > 0.0f ? 1.0f / w : 0.0f;
      p0[h + k] = w > 0.0f ? -q[k] / w : (q[k] <= 0.0f ? 1.0f : 0.0f);
      p0[2 * h + k] = 1.0f / static_cast<float>(h);
    }
    p0[3 * h] = 0.0f;
    mlp_init = p0;
    ix.lm_mlp.alloc(((np * 4 + 15) / 16) * 16);
    fill_bytes(ix.lm_mlp.p, 0, ix.lm_mlp.bytes, s);
    GJ_HIP_CHECK(hipMemcpyAsync(ix.lm_mlp.p, p0.data(), np * 4, hipMemcpyHostToDevice, s));
    dbuf state(4 * 64 * 4 * 4);  // grad, m1, m2, loss
    fill_bytes(state.p, 0, state.bytes, s);
    float* grad = state.as<float>();
    float* m1 = grad + 256;
    float* m2 = grad + 512;
    float* loss = grad + 768;
    SampleSource<K> src{nullptr, nullptr, col, n, kmin, root.inv_range, ix.params.seed};
    const uint64_t batch = std::min<uint64_t>(ix.params.mlp_batch, std::max<uint64_t>(n, 1));
    const uint32_t steps = (ix.params.learned_flags & GJ_LEARNED_UNTRAINED) ? 0u : ix.params.mlp_steps;
    for (uint32_t step = 1; step <= steps; ++step) {
      src.seed = ix.params.seed + static_cast<uint64_t>(step) * 0x632BE59BD9B4E019ull;
      if (step == steps) fill_bytes(loss, 0, 16, s);
      launch_mlp_grad<K>(h, ix.lm_mlp.as<float>(), src, batch, grad, loss, s);
      hipLaunchKernelGGL(adam_kernel, dim3(1), dim3(256), 0, s, ix.lm_mlp.as<float>(), grad, m1, m2, h,
                         ix.params.mlp_lr, static_cast<int>(step));
      GJ_HIP_CHECK(hipGetLastError());
    }
    if (steps == 0) {
      // untrained root: its loss on one minibatch of the same sampler, parameters untouched
      src.seed = ix.params.seed + 0x632BE59BD9B4E019ull;
      launch_mlp_grad<K>(h, ix.lm_mlp.as<float>(), src, batch, grad, loss, s);
    }
    float hl = 0;
    GJ_HIP_CHECK(hipMemcpyAsync(&hl, loss, sizeof(float), hipMemcpyDeviceToHost, s));
    GJ_HIP_CHECK(hipStreamSynchronize(s));
    ix.stats.train_loss = hl;
    root.hidden = h;
    root.mlp = ix.lm_mlp.as<const float>();
  }

  // Spline root: GreedySplineCorridor knots over (key, position) with the error bound
  // doubled until at most `max_segs` segments remain; stored as (key, cdf = pos / n,
  // slope) with the segment count padded to a power of two by repeating the last knot.
  auto spline_root = [&](uint32_t max_segs) {
    std::vector<uint8_t> hcopy;
    const void* hk = ix.h_col;
    if (!hk) {
      hcopy.resize(n * sizeof(K));
      GJ_HIP_CHECK(hipMemcpyAsync(hcopy.data(), col, hcopy.size(), hipMemcpyDeviceToHost, s));
      GJ_HIP_CHECK(hipStreamSynchronize(s));
      hk = hcopy.data();
    }
    uint64_t err = std::max<uint64_t>(16, n / (8ull * max_segs));
    RadixSplineHost sp;
    for (;;) {
      sp = build_radix_spline(hk, n, sizeof(K), 1, static_cast<uint32_t>(std::min<uint64_t>(err, 0x7FFFFFFFull)));
      if (sp.knot_x.size() <= static_cast<size_t>(max_segs) + 1 || err >= n) break;
      err *= 2;
    }
    const uint32_t knots = static_cast<uint32_t>(sp.knot_x.size());
    uint32_t segs = 1;
    while (segs + 1 < knots) segs *= 2;
    RootModel r{};
    r.inv_range = root.inv_range;
    r.segments = segs;
    std::vector<uint8_t> h(r.bytes(), 0);
    auto* key = reinterpret_cast<uint64_t*>(h.data());
    auto* cdf = reinterpret_cast<float*>(h.data() + r.key_bytes());
    auto* slope = reinterpret_cast<float*>(h.data() + r.key_bytes() + r.cdf_bytes());
    const double inv_n = 1.0 / static_cast<double>(n);
    for (uint32_t i = 0; i <= segs; ++i) {
      const uint32_t j = std::min(i, knots - 1);
      key[i] = sp.knot_x[j];
      cdf[i] = static_cast<float>(sp.knot_y[j] * inv_n);
    }
    for (uint32_t i = 0; i < segs; ++i) {
      const uint64_t dx = key[i + 1] - key[i];
      slope[i] = dx ? static_cast<float>((static_cast<double>(cdf[i + 1]) - cdf[i]) / static_cast<double>(dx)) : 0.0f;
    }
    ix.lm_knots.alloc(h.size());
    GJ_HIP_CHECK(hipMemcpyAsync(ix.lm_knots.p, h.data(), h.size(), hipMemcpyHostToDevice, s));
    GJ_HIP_CHECK(hipStreamSynchronize(s));
    r.knots = ix.lm_knots.as<const uint64_t>();
    ix.stats.spline_points = knots;
    return r;
  };
  if (ix.kind == GJ_LEARNED_PLR && ix.params.learned_root_segments >= 2) {
    const uint32_t want = ix.params.learned_root_segments;
    GJ_REQUIRE((want & (want - 1)) == 0 && want <= 4096, GJ_ERR_INVALID,
               "learned_root_segments must be 0, 1 or a power of two <= 4096");
    root = spline_root(want);
  }

  // Lines layout: the model places the keys itself, so a present key is read from the
  // line the model names (or, behind a run of full lines, the next ones).  Candidates,
  // cheapest first: the linear root alone (no table to read), then the root routing to
  // leaves that each spread their keys over their own lines, then (learned_plr) a
  // spline root of the column's CDF routing to leaves.  The one with the fewest lines
  // per present key wins; the column layout takes over in auto mode when even that
  // reads more than 1.10 lines per key or up to more than 4 lines, or when the line
  // copy does not fit in memory.
  // A column below 16 MiB is served from L2 and the MALL, and auto keeps it without a second
  // copy of its keys.  That costs lookups (2^24 probes of 2^20 u32 keys 212 us, by lines 142:
  // one line a probe in place of leaf and key line) and saves the build of the copy; a caller
  // who wants the lines there asks for them.  Auto also keeps the column for structures placed
  // in host memory: the line copy would move every key lookup onto the host link, where
  // the column layout's model (a few MiB, cached in L2) leaves the key reads in the column.
  const uint32_t layout = ix.params.learned_layout;
  GJ_REQUIRE(layout <= GJ_LAYOUT_LINES, GJ_ERR_INVALID, "learned_layout must be 0, 1 or 2");
  constexpr uint64_t kLinesMinColumnBytes = 16ull << 20;
  if (layout == GJ_LAYOUT_LINES || (layout == GJ_LAYOUT_AUTO && n * sizeof(K) >= kLinesMinColumnBytes &&
                                    ix.params.placement != GJ_PLACE_HOST)) {
    using D = LinesDev<K>;
    const uint32_t lk = ix.params.learned_line_keys ? ix.params.learned_line_keys : (sizeof(K) == 8 ? 10u : 20u);
    GJ_REQUIRE(lk >= 1 && lk <= D::CAP, GJ_ERR_INVALID, "learned_line_keys must be in [1, keys per line]");
    const uint32_t lbits = ix.params.learned_leaf_bits
                               ? ix.params.learned_leaf_bits
                               : static_cast<uint32_t>(std::clamp(static_cast<int>(ilog2_ceil(n)) - 10, 8, 20));
    LinesBuild best;
    auto consider = [&](auto&& make) {
      LinesBuild c;
      try {
        make(c);
      } catch (const error& e) {
        if (e.status != GJ_ERR_NOMEM || layout == GJ_LAYOUT_LINES) throw;
        (void)hipGetLastError();
        return;  // auto: the line copy does not fit; try the next candidate or the column layout
      }
      // a candidate within the auto bounds beats one outside them; then fewer lines per key
      auto good = [](const LinesBuild& b) { return b.avg_lines <= 1.10 && b.max_lines <= 4; };
      if (!best.ok || (good(c) && !good(best)) || (good(c) == good(best) && c.avg_lines < best.avg_lines))
        best = std::move(c);
    };
    constexpr double kGoodLines = 1.05;  // below this, a costlier candidate cannot gain much
    const bool linear_root = root.hidden == 0 && root.segments == 0;
    if (linear_root && ix.params.learned_leaf_bits == 0)
      consider([&](LinesBuild& c) { lines_root_only<K>(ix, lk, c, s); });
    if (!best.ok || best.avg_lines > kGoodLines) {
      fit_root();
      consider([&](LinesBuild& c) { lines_two_stage<K>(ix, root, lbits, lk, c, s); });
    }
    if (ix.kind == GJ_LEARNED_PLR && linear_root && ix.params.learned_root_segments == 0 &&
        (!best.ok || best.avg_lines > kGoodLines) && n >= 4)
      consider([&](LinesBuild& c) { lines_two_stage<K>(ix, spline_root(2048), lbits, lk, c, s); });
    // Training lowers the MLP root's mean squared error, but that can leave a flat stretch
    // that routes a crowd of keys to a few leaves (lognormal keys at 2^26: 700 lines per
    // key); the quantile initialisation routes equal key counts per ramp.  So the build
    // also places the keys under the initial root, and keeps the trained one unless the
    // initial one does better.
    bool init_root = false;
    if (root.hidden && !mlp_init.empty() && !(ix.params.learned_flags & GJ_LEARNED_UNTRAINED) &&
        (!best.ok || best.avg_lines > kGoodLines || best.max_lines > 4)) {
      dbuf init_params(ix.lm_mlp.bytes);
      fill_bytes(init_params.p, 0, init_params.bytes, s);
      GJ_HIP_CHECK(hipMemcpyAsync(init_params.p, mlp_init.data(), mlp_init.size() * 4, hipMemcpyHostToDevice, s));
      RootModel r0 = root;
      r0.mlp = init_params.as<const float>();
      consider([&](LinesBuild& c) { lines_two_stage<K>(ix, r0, lbits, lk, c, s); });
      init_root = best.ok && best.root.mlp == r0.mlp;
      if (init_root) {
        // the index serves lookups with the initial parameters
        GJ_HIP_CHECK(hipMemcpyAsync(ix.lm_mlp.p, init_params.p, init_params.bytes, hipMemcpyDeviceToDevice, s));
        GJ_HIP_CHECK(hipStreamSynchronize(s));
        best.root.mlp = ix.lm_mlp.as<const float>();
      }
    }
    if (init_root) ix.stats.root_trained = 0;
    // a lookup wave walks as many lines as its farthest probe needs, so auto also bounds
    // the longest walk, not only the mean
    if (best.ok && (layout == GJ_LAYOUT_LINES || (best.avg_lines <= 1.10 && best.max_lines <= 4))) {
      if (best.root.segments == 0) {
        ix.lm_knots.release();
        ix.stats.spline_points = 0;
      }
      adopt_lines(ix, best);
      return;
    }
    GJ_REQUIRE(layout != GJ_LAYOUT_LINES, GJ_ERR_NOMEM, "learned lines: the line copy does not fit");
    ix.lm_knots.release();
    ix.stats.spline_points = 0;
  }
  ix.lm_layout = GJ_LAYOUT_COLUMN;
  ix.stats.layout = GJ_LAYOUT_COLUMN;
  fit_root();
  build_btree<K>(ix, s);  // the fallback of leaves that no window covers; the lines need none

  dbuf last_start, last_fit;  // leaf starts and fits of the last build_leaves
  // routing, leaf fits and calibration under a root; returns the build keys routed to the B-tree
  auto build_leaves = [&](const RootModel& root) -> uint64_t {
    ix.lm_compact = false;
    ix.lm_groups.release();
    Router<K> route{kmin, root, L};
    dbuf start((static_cast<uint64_t>(L) + 1 + 3) * sizeof(uint32_t));
    {
      fill_words(start.as<uint32_t>(), static_cast<uint64_t>(L) + 1, static_cast<uint32_t>(n), s);
      dbuf inv(sizeof(unsigned long long));
      fill_bytes(inv.p, 0, inv.bytes, s);
      hipLaunchKernelGGL(leaf_bounds_kernel<K>, dim3(grid_for(n, 256)), dim3(256), 0, s, col, n, route,
                         start.as<uint32_t>(), inv.as<unsigned long long>());
      GJ_HIP_CHECK(hipGetLastError());
      unsigned long long hinv = 0;
      GJ_HIP_CHECK(hipMemcpyAsync(&hinv, inv.p, sizeof(hinv), hipMemcpyDeviceToHost, s));
      GJ_HIP_CHECK(hipStreamSynchronize(s));
      GJ_REQUIRE(hinv == 0, GJ_ERR_INTERNAL, "learned index: root model is not monotone");
    }
    ix.lm_leaves.alloc(sizeof(LeafModel) * L);
    dbuf fit(sizeof(LeafFit) * L);
    const int64_t max_width = 2 * static_cast<int64_t>(ix.params.learned_max_error) + 2;
    LeafPass pass;
    LeafStats st = pass.run(col, n, start.as<const uint32_t>(), start.as<const uint32_t>() + 1, L, max_width,
                            FitLeaf<K>{ix.lm_leaves.as<LeafModel>()}, fit.as<LeafFit>(), s);
    std::vector<LeafFit> hf;  // read back only if a leaf is too wide
    if (st.fb_leaves) {
      hf.resize(L);
      GJ_HIP_CHECK(hipMemcpyAsync(hf.data(), fit.p, fit.bytes, hipMemcpyDeviceToHost, s));
      GJ_HIP_CHECK(hipStreamSynchronize(s));
    }

    // split a leaf that is too wide into kSplitWays equal-count sub-leaves, unless its
    // sub-leaves would still hold over 4 average leaves each (then no line fits them
    // either, and the extra separator read would only delay the B-tree)
    const uint64_t split_max = static_cast<uint64_t>(kSplitWays) * 4 * std::max<uint64_t>(1, ceil_div(n, L));
    std::vector<uint32_t> split_id, split_lo, split_hi, sub_lo, sub_hi;
    for (uint32_t l = 0; l < hf.size(); ++l) {
      const LeafFit& f = hf[l];
      if (f.count == 0 || f.err_hi >= f.err_lo || f.count > split_max) continue;
      st.fb_leaves -= 1;  // split leaves count through their sub-leaves
      st.fb_keys -= f.count;
      split_id.push_back(l);
      split_lo.push_back(f.start);
      split_hi.push_back(f.start + f.count);
      for (uint32_t t = 0; t < kSplitWays; ++t) {
        sub_lo.push_back(f.start + static_cast<uint32_t>((static_cast<uint64_t>(f.count) * t) / kSplitWays));
        sub_hi.push_back(f.start + static_cast<uint32_t>((static_cast<uint64_t>(f.count) * (t + 1)) / kSplitWays));
      }
    }
    const uint32_t J = static_cast<uint32_t>(split_id.size());
    ix.lm_splits = J;
    ix.lm_seps.release();
    ix.lm_subs.release();
    if (J) {
      const uint64_t S = static_cast<uint64_t>(J) * kSplitWays;
      dbuf d_id(J * 4), d_lo(J * 4), d_hi(J * 4), d_slo(S * 4), d_shi(S * 4), sfit(S * sizeof(LeafFit));
      GJ_HIP_CHECK(hipMemcpyAsync(d_id.p, split_id.data(), J * 4, hipMemcpyHostToDevice, s));
      GJ_HIP_CHECK(hipMemcpyAsync(d_lo.p, split_lo.data(), J * 4, hipMemcpyHostToDevice, s));
      GJ_HIP_CHECK(hipMemcpyAsync(d_hi.p, split_hi.data(), J * 4, hipMemcpyHostToDevice, s));
      GJ_HIP_CHECK(hipMemcpyAsync(d_slo.p, sub_lo.data(), S * 4, hipMemcpyHostToDevice, s));
      GJ_HIP_CHECK(hipMemcpyAsync(d_shi.p, sub_hi.data(), S * 4, hipMemcpyHostToDevice, s));
      ix.lm_seps.alloc(S * 8);
      ix.lm_subs.alloc(S * sizeof(LeafModel));
      hipLaunchKernelGGL(split_sep_kernel<K>, dim3(grid_for(S, 256)), dim3(256), 0, s, col, d_slo.as<const uint32_t>(),
                         d_shi.as<const uint32_t>(), d_lo.as<const uint32_t>(), J, ix.lm_seps.as<uint64_t>());
      GJ_HIP_CHECK(hipGetLastError());
      const LeafStats sub = pass.run(col, n, d_slo.as<const uint32_t>(), d_shi.as<const uint32_t>(),
                                     static_cast<uint32_t>(S), max_width, FitLeaf<K>{ix.lm_subs.as<LeafModel>()},
                                     sfit.as<LeafFit>(), s);
      st.fb_leaves += sub.fb_leaves;
      st.fb_keys += sub.fb_keys;
      st.wsum += sub.wsum;
      st.wkeys += sub.wkeys;
      st.wmax = std::max(st.wmax, sub.wmax);
      st.err_lo = std::min(st.err_lo, sub.err_lo);
      st.err_hi = std::max(st.err_hi, sub.err_hi);
      hipLaunchKernelGGL(split_mark_kernel, dim3(grid_for(J, 256)), dim3(256), 0, s, ix.lm_leaves.as<LeafModel>(),
                         d_id.as<const uint32_t>(), J);
      GJ_HIP_CHECK(hipGetLastError());
      GJ_HIP_CHECK(hipStreamSynchronize(s));  // the work lists may go
    }

    // window bounds over the (sub-)leaves that are not routed to the B-tree
    ix.lm_err_lo = st.err_lo;
    ix.lm_err_hi = st.err_hi;
    ix.lm_root = root;
    ix.stats.root_segments = root.segments;
    ix.lm_num_leaves = L;
    ix.lm_fallback_any = st.fb_leaves ? 1u : 0u;
    ix.stats.leaves = L;
    ix.stats.fallback_leaves = st.fb_leaves;
    ix.stats.fallback_keys = st.fb_keys;
    ix.stats.split_leaves = J;
    ix.stats.max_window = st.wmax;
    ix.stats.avg_window = st.wkeys ? static_cast<double>(st.wsum) / static_cast<double>(st.wkeys) : 0.0;
    ix.stats.depth = 2;
    ix.stats.lds_levels = ix.bt.lds_levels;
    last_start = std::move(start);
    last_fit = std::move(fit);
    return st.fb_keys;
  };

  // compact leaves from the last build's 16-byte leaves; false (index unchanged) when a
  // leaf's window under the compact arithmetic exceeds the bound
  auto make_compact = [&](const RootModel& root) -> bool {
    const uint32_t lbits = ilog2_ceil(L);
    const uint32_t gshift = lbits > 9 ? lbits - 9 : 0;  // at most 512 groups (8 KiB of LDS)
    const uint32_t G = L >> gshift;
    dbuf groups(sizeof(LeafGroup) * G), cl(sizeof(LeafCompact) * L);
    hipLaunchKernelGGL(compact_groups_kernel<K>, dim3(grid_for(G, 256)), dim3(256), 0, s, col, n,
                       last_start.as<const uint32_t>(), G, gshift, groups.as<LeafGroup>());
    GJ_HIP_CHECK(hipGetLastError());
    LeafPass pass;
    const LeafStats st = pass.run(col, n, last_start.as<const uint32_t>(), last_start.as<const uint32_t>() + 1, L,
                                  2 * static_cast<int64_t>(ix.params.learned_max_error) + 2,
                                  CompactLeaf<K>{ix.lm_leaves.as<const LeafModel>(), groups.as<const LeafGroup>(),
                                                 gshift, cl.as<LeafCompact>()},
                                  last_fit.as<LeafFit>(), s);
    if (st.fb_leaves) return false;
    ix.lm_leaves = std::move(cl);
    ix.lm_groups = std::move(groups);
    ix.lm_gshift = gshift;
    ix.lm_compact = true;
    ix.lm_err_lo = st.err_lo;
    ix.lm_err_hi = st.err_hi;
    ix.stats.max_window = st.wmax;
    ix.stats.avg_window = st.wkeys ? static_cast<double>(st.wsum) / static_cast<double>(st.wkeys) : 0.0;
    return true;
  };

  // With the default leaf count, a root that spreads the keys evenly gets twice the
  // leaves in compact form (the same table bytes); otherwise 16-byte leaves.  Below
  // 2^22 keys the lookups are bound by L2 hits rather than misses and the compact
  // form's LDS group table only costs occupancy, so small indexes keep 16-byte leaves.
  bool compact = false;
  if (ix.params.learned_leaf_bits == 0 && bits < 24 && root.segments == 0 && n >= (1ull << 22)) {
    L = 2u << bits;
    const uint64_t fb2 = build_leaves(root);
    compact = fb2 == 0 && ix.lm_splits == 0 && make_compact(root);
    if (!compact) L = 1u << bits;
  }
  if (!compact) {
    const uint64_t fb = build_leaves(root);
    if (ix.kind == GJ_LEARNED_PLR && ix.params.learned_root_segments == 0 && fb > 0 && n >= 4) {
      // the linear root cannot spread these keys evenly over the leaves: route by a
      // spline of the column's own CDF instead
      build_leaves(spline_root(2048));
    }
  }
}
template void build_learned<uint32_t>(gj_index&, hipStream_t);
template void build_learned<uint64_t>(gj_index&, hipStream_t);

}  // namespace gj

using namespace gj;

extern "C" {

int gj_mlp_loss_grad(const float* d_params, uint32_t hidden, const float* d_x, const float* d_y, uint64_t n,
                     float* d_grad, float* d_loss, gj_stream_t stream) {
  return guarded([&] {
    GJ_REQUIRE(d_params && d_x && d_y && d_grad && d_loss && n > 0, GJ_ERR_INVALID, "bad argument");
    const hipStream_t s = S(stream);
    hipLaunchKernelGGL(clear_grad_kernel, dim3(1), dim3(256), 0, s, d_grad, 3 * hidden + 1, d_loss);
    GJ_HIP_CHECK(hipGetLastError());
    SampleSource<uint64_t> src{d_x, d_y, nullptr, n, 0, 0.0f, 0};
    launch_mlp_grad<uint64_t>(hidden, d_params, src, n, d_grad, d_loss, s);
  });
}

int gj_mlp_forward(const float* d_params, uint32_t hidden, const float* d_x, uint64_t n, float* d_out,
                   gj_stream_t stream) {
  return guarded([&] {
    GJ_REQUIRE(d_params && d_x && d_out, GJ_ERR_INVALID, "bad argument");
    GJ_REQUIRE(hidden >= 1 && hidden <= static_cast<uint32_t>(kMaxHidden), GJ_ERR_INVALID, "bad hidden width");
    if (n == 0) return;
    hipLaunchKernelGGL(mlp_forward_kernel, dim3(grid_for(n, 256)), dim3(256), 0, S(stream), d_params, hidden, d_x, n,
                       d_out);
    GJ_HIP_CHECK(hipGetLastError());
  });
}

}  // extern "C"
