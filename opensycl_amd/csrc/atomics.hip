// Bulk atomic workloads: histogram by fetch_add(1) and strided fetch_min /
// fetch_max / fetch_add into a slot array.
//
// Reference behaviour being replaced: a user kernel in which work-item i
// applies sycl::atomic_ref<T, relaxed, device>(target[slot(i)]).fetch_<op>(v_i)
// (include/hipSYCL/sycl/libkernel/atomic_ref.hpp:143-197), which the HIP
// backend lowers to one global atomic per element
// (generic/hiplike/atomic_builtins.hpp:438-598).  Under skewed keys (Zipf)
// the hot bins serialise at the L2 / memory-side atomic units.
//
// MI355X design:
//   - strategy "privatized": every work-group keeps private counters in LDS
//     and only the group totals reach global memory.  Up to 8192 bins the
//     counters are 32-bit; above, two 16-bit counters share one 32-bit LDS
//     word (65536 bins = 128 KiB of the 160 KiB LDS).  A 16-bit counter that
//     has reached 0x8000 is drained by the one work-item that clears its top
//     bit: it adds 0x8000 to the global bin, so a field never carries into
//     its neighbour.  Up to 2^22 bins are cut into slices, one per group.
//     Group totals go straight to the bins where that takes few atomics, else
//     they are written as per-group partial histograms (coalesced, no
//     atomics) and a second kernel adds their column sums to the bins;
//   - keys are streamed with 128-bit loads, several per work-item in flight;
//   - strided fetch_min / fetch_max / fetch_add (slot = i mod num_slots):
//     the elements are the rows of a matrix whose columns always meet the
//     same slots; a work-item keeps a column's slots in registers, and the
//     group combines its rows once at the end;
//   - strategy "global": one device-scope atomic per element, the
//     reference's pattern, kept for comparison.
#include <algorithm>
#include <cmath>
#include <numeric>

#include "launch_util.hpp"

namespace acpp_impl {
namespace atomics_detail {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

enum strategy : int { strat_auto = 0, strat_privatized = 1, strat_global = 2 };

constexpr uint32_t lds_bytes_budget = 128 * 1024;

// 16-byte streaming geometry of an array: `head` scalar elements before the
// first 16-byte boundary, `nvec` aligned 16-byte chunks, then the tail.
struct geom {
  uint64_t head;
  uint64_t nvec;
  uint64_t tail_start;
  uint64_t nscalar;  // head + tail
};

template <class T>
geom make_geom(const T *p, uint64_t n) {
  constexpr uint64_t VEC = 16 / sizeof(T);
  geom g;
  g.head = ((16 - (reinterpret_cast<uintptr_t>(p) & 15)) & 15) / sizeof(T);
  if (g.head > n) g.head = n;
  g.nvec = (n - g.head) / VEC;
  g.tail_start = g.head + g.nvec * VEC;
  g.nscalar = g.head + (n - g.tail_start);
  return g;
}

__device__ __forceinline__ uint64_t scalar_index(const geom &g, uint64_t s) {
  return (s < g.head) ? s : g.tail_start + (s - g.head);
}

// --------------------------------------------------------------------------
// Histogram
// --------------------------------------------------------------------------
struct hist_params {
  const uint32_t *keys;
  geom gm;
  uint32_t *bins;
  uint32_t num_bins;
  uint32_t local_bins;   // bins of one slice (num_bins without slices)
  uint32_t slices_log2;  // SLICED: 2^slices_log2 slices of the bins
  uint32_t copies_log2;  // 32-bit counters: LDS copies of the histogram
  uint32_t chunks;       // work-groups per slice; each takes one part of the keys
  int xcd_map;           // SLICED: a chunk's slices share an XCD
  uint32_t *partials;    // NULL: the counts go straight to the bins
};

// A slice holds the bins k with (k ^ (k >> s)) mod 2^s == slice, as its
// local bins k >> s (s = slices_log2): hot neighbouring bins, and bins a power
// of two apart, fall into different slices.
__device__ __forceinline__ uint32_t slice_bin(uint32_t local, uint32_t slice, uint32_t s) {
  return (local << s) | ((local ^ slice) & ((1u << s) - 1u));
}

// 32-bit counters: the group keeps 2^copies_log2 copies of the histogram,
// word (bin << copies_log2) + copy, and work-item t counts into copy
// t mod 2^copies_log2.  Lanes that meet the same hot bin then hit adjacent
// words in different banks instead of one address.
//
// PACKED: bin b < half in the low 16 bits of word b, bin half + b in the
// high 16 bits, so the low (under skewed keys, hot) bins sit in consecutive
// words and banks; adjacent bins sharing a word put the two hottest Zipf
// bins on one address.
//
// SLICED (packed, more than 65536 bins): every group counts the keys of one
// slice of the bins and skips the others, so each key is read once per slice,
// but only once from memory: the groups of one part of the keys run on one
// XCD and meet in its L2.  Bound by the instructions per visited key (four
// keys per clock and CU).  One device atomic per key, the form before,
// serialises on hot bins and reaches 26 G keys/s on uniform ones: 2^25
// Zipf(1.1) keys into 200,000 bins 48.7 ms -> 74 us, 2^24 uniform keys
// 640 -> 46 us, 2^25 Zipf keys into 1,000,000 bins 46 ms -> 230 us.  (32-bit
// counters without a returned value, in twice the slices: 120 and 399 us.)
template <bool PACKED, bool SLICED, int UNROLL>
__global__ __launch_bounds__(1024) void histogram_kernel(hist_params p) {
  static_assert(PACKED || !SLICED, "slices use packed counters");
  extern __shared__ uint32_t lds[];
  const uint32_t my_copy = threadIdx.x & ((1u << p.copies_log2) - 1u);
  const uint32_t half = (p.local_bins + 1) / 2;
  const uint32_t s = p.slices_log2;
  const uint32_t mask = (1u << s) - 1u;
  uint32_t slice = 0, chunk = blockIdx.x;
  if constexpr (SLICED) {
    // Work-groups go to the eight XCDs in turn.
    const uint32_t i = p.xcd_map ? blockIdx.x >> 3 : blockIdx.x;
    slice = i & mask;
    chunk = p.xcd_map ? ((i >> s) << 3) + (blockIdx.x & 7u) : i >> s;
  }
  const uint32_t slice_top = SLICED ? slice << (32 - s) : 0;
  // the slice's local bins: the last one only if its bin exists
  const uint32_t slice_end =
      SLICED ? p.local_bins - (slice_bin(p.local_bins - 1, slice, s) >= p.num_bins ? 1u : 0u) : p.num_bins;
  auto bin_of = [&](uint32_t local) { return SLICED ? slice_bin(local, slice, s) : local; };
  auto add_bin = [&](uint32_t b, uint32_t v) {
    if (v && b < p.num_bins) __hip_atomic_fetch_add(&p.bins[b], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  const uint32_t words = PACKED ? half : (p.num_bins << p.copies_log2);
  for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) lds[i] = 0;
  __syncthreads();

  // The counts of a batch of keys: all LDS atomics are issued before the
  // first returned word is looked at.
  auto count = [&](const uint32_t *k, auto m_tag) {
    constexpr int M = decltype(m_tag)::value;
    if constexpr (PACKED) {
      uint32_t word[M], old[M];
      uint32_t any = 0;
#pragma unroll
      for (int j = 0; j < M; ++j) {
        // the slice in the top s bits, the local bin below
        const uint32_t l = SLICED ? __builtin_amdgcn_alignbit(k[j] ^ (k[j] >> s), k[j], s) - slice_top : k[j];
        word[j] = min(l, l - half);  // l - half wraps for the low bins
        old[j] = 0;
        if (l < slice_end) old[j] = atomicAdd(&lds[word[j]], l < half ? 1u : 0x10000u);
        any |= old[j];
      }
      if (any & 0x80008000u) {
        // A field had reached 0x8000 before the add: whoever clears its top
        // bit adds 0x8000 to the bin.  The field cannot carry before that: no
        // work-item adds more than M times without looking.
#pragma unroll
        for (int j = 0; j < M; ++j) {
          if (!(old[j] & 0x80008000u)) continue;
          const uint32_t full = atomicAnd(&lds[word[j]], 0x7fff7fffu);
          if (full & 0x8000u) add_bin(bin_of(word[j]), 0x8000u);
          if (full & 0x80000000u) add_bin(bin_of(word[j] + half), 0x8000u);
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < M; ++j)
        if (k[j] < p.num_bins) atomicAdd(&lds[(k[j] << p.copies_log2) + my_copy], 1u);
    }
  };

  const uint64_t stride = static_cast<uint64_t>(p.chunks) * blockDim.x;
  const uint64_t gtid = static_cast<uint64_t>(chunk) * blockDim.x + threadIdx.x;
  const u32x4 *kv = reinterpret_cast<const u32x4 *>(p.keys + p.gm.head);
  uint64_t c = gtid;
  for (; c + (UNROLL - 1) * stride < p.gm.nvec; c += UNROLL * stride) {
    u32x4 q[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) q[u] = SLICED ? kv[c + u * stride] : __builtin_nontemporal_load(kv + c + u * stride);
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      uint32_t k[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
      count(k, std::integral_constant<int, 4>{});
    }
  }
  for (; c < p.gm.nvec; c += stride) {
    const u32x4 q = kv[c];
    uint32_t k[4] = {q.x, q.y, q.z, q.w};
    count(k, std::integral_constant<int, 4>{});
  }
  for (uint64_t i = gtid; i < p.gm.nscalar; i += stride) {
    const uint32_t k = p.keys[scalar_index(p.gm, i)];
    count(&k, std::integral_constant<int, 1>{});
  }

  __syncthreads();
  // Groups that add to the same bins start at different ones, a wave's 64
  // always in whole lines: `count` is rounded up to 64, and callers skip what
  // lies past the end (10.4M keys into 500 bins: 15.5 us with a wave's bins
  // across lines, 13.7 us so; through partials 14.0 us).
  auto whole_waves = [](uint32_t count) { return (count + 63u) & ~63u; };
  auto rotated = [&](uint32_t i, uint32_t count) {
    const uint32_t n = whole_waves(count);
    const uint32_t first = static_cast<uint32_t>(static_cast<uint64_t>(n) * chunk / p.chunks) & ~63u;
    return i + first < n ? i + first : i + first - n;
  };
  // Many rounds of few keys: four words at a time.  One by one, the LDS latency
  // of every round counts (500 keys into 32000 bins 12.6 us, so 7.9 us; into
  // 12000 6.9 and 5.2 us).  With few rounds the groups' atomics then meet (2M
  // keys into 4000 bins 9.3 and 11.7 us).
  if (const uint32_t rounds_words = PACKED ? half : p.num_bins; !p.partials && rounds_words > 8 * blockDim.x) {
    const uint32_t rounded = whole_waves(rounds_words);
    for (uint32_t i0 = threadIdx.x; i0 < rounded; i0 += 4 * blockDim.x) {
      uint32_t w[4], v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t i = i0 + u * blockDim.x;
        w[u] = i < rounded ? rotated(i, rounds_words) : rounds_words;
        v[u] = 0;
        if (w[u] < rounds_words)
          for (uint32_t c = 0; c < (1u << p.copies_log2); ++c) v[u] += lds[(w[u] << p.copies_log2) + c];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if constexpr (PACKED) {
          if (w[u] >= rounds_words) continue;
          add_bin(bin_of(w[u]), v[u] & 0xffffu);
          add_bin(bin_of(w[u] + half), v[u] >> 16);
        } else {
          add_bin(w[u], v[u]);
        }
      }
    }
    return;
  }
  if constexpr (PACKED) {
    uint32_t *mine = p.partials + (static_cast<uint64_t>(slice) * p.chunks + chunk) * half;
    for (uint32_t i = threadIdx.x; i < whole_waves(half); i += blockDim.x) {
      if (p.partials) {
        if (i < half) mine[i] = lds[i];  // both counters of the word
      } else {
        const uint32_t w = rotated(i, half);
        if (w >= half) continue;
        const uint32_t v = lds[w];
        add_bin(bin_of(w), v & 0xffffu);
        add_bin(bin_of(w + half), v >> 16);
      }
    }
  } else {
    uint32_t *mine = p.partials + static_cast<uint64_t>(blockIdx.x) * p.num_bins;
    for (uint32_t i = threadIdx.x; i < whole_waves(p.num_bins); i += blockDim.x) {
      const uint32_t b = p.partials ? i : rotated(i, p.num_bins);
      if (b >= p.num_bins) continue;
      uint32_t v = 0;
      for (uint32_t c = 0; c < (1u << p.copies_log2); ++c) v += lds[(b << p.copies_log2) + c];
      if (p.partials)
        mine[b] = v;
      else
        add_bin(b, v);
    }
  }
}

// One device-scope atomic per key (the reference's pattern).
template <int UNROLL>
__global__ __launch_bounds__(1024) void histogram_global_kernel(const uint32_t *__restrict__ keys, geom gm,
                                                                uint32_t num_bins, uint32_t *bins) {
  auto count = [&](uint32_t k) {
    if (k < num_bins) __hip_atomic_fetch_add(&bins[k], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  const uint64_t gtid = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const u32x4 *kv = reinterpret_cast<const u32x4 *>(keys + gm.head);
  uint64_t c = gtid;
  for (; c + (UNROLL - 1) * stride < gm.nvec; c += UNROLL * stride) {
    u32x4 q[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) q[u] = __builtin_nontemporal_load(kv + c + u * stride);
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      count(q[u].x);
      count(q[u].y);
      count(q[u].z);
      count(q[u].w);
    }
  }
  for (; c < gm.nvec; c += stride) {
    const u32x4 q = kv[c];
    count(q.x);
    count(q.y);
    count(q.z);
    count(q.w);
  }
  for (uint64_t s = gtid; s < gm.nscalar; s += stride) count(keys[scalar_index(gm, s)]);
}

// bins[b] += sum over groups of the partial counts.  A work-group sums `span`
// words of every slice over its chunks (blockIdx.y takes every gridDim.y-th
// chunk, so the partials are read by many work-groups at once) and puts the
// bins' sums in order in LDS: neighbouring bins come from different slices,
// and the atomics on the bins are coalesced this way.  Integer atomics: the
// order does not matter.  PACKED partials are the words of the LDS, 16 bits
// a counter.
// Bound by the lines that the atomics touch (11 G lines/s), which is the
// bins' bytes times gridDim.y: so the spans are short, and the grid has its
// blocks in x (428,362 keys into 905,561 bins: 40.3 us with spans of 4096
// entries, 28.0 us so; 2^24 keys: 142 and 121 us).
constexpr uint32_t combine_entries = 1024;  // span << slices_log2 at most
__host__ __device__ constexpr uint32_t combine_span_log2(uint32_t slices_log2) {
  return slices_log2 <= 1 ? 8u : slices_log2 <= 5 ? 9u - slices_log2 : 4u;
}
template <bool PACKED>
__global__ __launch_bounds__(256) void histogram_combine_kernel(hist_params p) {
  __shared__ uint32_t s_low[combine_entries];
  __shared__ uint32_t s_high[PACKED ? combine_entries : 1];
  const uint32_t s = p.slices_log2;
  const uint32_t mask = (1u << s) - 1u;
  const uint32_t span_log2 = combine_span_log2(s);
  const uint32_t half = (p.local_bins + 1) / 2;
  const uint32_t words = PACKED ? half : p.num_bins;
  const uint32_t w0 = blockIdx.x << span_log2;
  const uint32_t entries = 1u << (span_log2 + s);
  for (uint32_t e = threadIdx.x; e < entries; e += blockDim.x) {
    const uint32_t slice = e >> span_log2;
    const uint32_t w = w0 + (e & ((1u << span_log2) - 1u));
    if (w >= words) continue;
    const uint32_t *src = p.partials + static_cast<uint64_t>(slice) * p.chunks * words + w;
    uint32_t low = 0, high = 0;
#pragma unroll 8
    for (uint32_t ch = blockIdx.y; ch < p.chunks; ch += gridDim.y) {
      const uint32_t v = src[static_cast<uint64_t>(ch) * words];
      low += PACKED ? v & 0xffffu : v;
      high += PACKED ? v >> 16 : 0u;
    }
    s_low[((w - w0) << s) | ((w ^ slice) & mask)] = low;
    if constexpr (PACKED) s_high[((w - w0) << s) | (((w + half) ^ slice) & mask)] = high;
  }
  __syncthreads();
  for (uint32_t e = threadIdx.x; e < entries; e += blockDim.x) {
    if (w0 + (e >> s) >= words) continue;
    const uint32_t b = (w0 << s) + e;
    if (s_low[e] && b < p.num_bins)
      __hip_atomic_fetch_add(&p.bins[b], s_low[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if constexpr (PACKED) {
      const uint32_t bh = b + (half << s);
      if (s_high[e] && bh < p.num_bins)
        __hip_atomic_fetch_add(&p.bins[bh], s_high[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// --------------------------------------------------------------------------
// Strided fetch ops: target[i % num_slots] = op(target[i % num_slots], v[i])
// --------------------------------------------------------------------------
template <int Scope, class T, class Cmp>
__device__ __forceinline__ void cas_select(T *p, T v, Cmp keep_old) {
  T old = __hip_atomic_load(p, __ATOMIC_RELAXED, Scope);
  while (!keep_old(old, v)) {
    if (__hip_atomic_compare_exchange_strong(p, &old, v, __ATOMIC_RELAXED, __ATOMIC_RELAXED, Scope))
      break;
  }
}

// identity() and apply() fold the elements of a slot before the one atomic on
// it.  A NaN stays in the fold of min and max: as the last of the folded
// elements it takes the target's place, as it does where every element has
// an atomic of its own.  (By the atomics' rule a later element would replace
// it in the fold, or the identity of a lane without elements, and the target
// would never see it.)
template <class T>
struct rmw_min {
  __device__ static T identity() { return ops::minimum<T, T>::identity(); }
  __device__ static T apply(T a, T b) {
    if constexpr (std::is_floating_point_v<T>)
      return __builtin_elementwise_minimum(a, b);  // a NaN if either is
    else
      return ops::minimum<T, T>::apply(a, b);
  }
  template <int Scope>
  __device__ static void atomic(T *p, T v) {
    if constexpr (std::is_floating_point_v<T>)
      cas_select<Scope>(p, v, [](T old, T x) { return old < x || old == x; });  // sycl::minimum rule
    else
      __hip_atomic_fetch_min(p, v, __ATOMIC_RELAXED, Scope);
  }
};

template <class T>
struct rmw_max {
  __device__ static T identity() { return ops::maximum<T, T>::identity(); }
  __device__ static T apply(T a, T b) {
    if constexpr (std::is_floating_point_v<T>)
      return __builtin_elementwise_maximum(a, b);
    else
      return ops::maximum<T, T>::apply(a, b);
  }
  template <int Scope>
  __device__ static void atomic(T *p, T v) {
    if constexpr (std::is_floating_point_v<T>)
      cas_select<Scope>(p, v, [](T old, T x) { return old > x || old == x; });
    else
      __hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, Scope);
  }
};

template <class T>
struct rmw_add {
  __device__ static T identity() { return ops::plus<T, T>::identity(); }
  __device__ static T apply(T a, T b) { return ops::wrap_add(a, b); }
  template <int Scope>
  __device__ static void atomic(T *p, T v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, Scope);
  }
};

constexpr int scope_dev = __HIP_MEMORY_SCOPE_AGENT;

// The elements after the scalar head as a matrix of 16-byte vectors whose
// rows hold a whole multiple of num_slots elements: all of a column's vectors
// meet the same VEC slots.  A work-group takes a strip of `width` columns (a
// power of two) and every row_groups-th band of blockDim.x / width rows; each
// work-item keeps its column's VEC slots in registers over all its rows, the
// group folds its rows in LDS and adds one value per slot of the strip to the
// target.
struct strip_params {
  geom gm;
  uint64_t columns;     // vectors in a row
  uint64_t row_groups;  // work-groups that share a strip
  uint32_t width_log2;
  uint64_t num_slots;
};

// Bound by the loads.  Narrow strips keep the atomics few (a group adds
// width x VEC values at most), and the rows of a strip read at least 1 KiB in
// one piece where there are rows enough.  Before, groups kept all slots in
// LDS: one device atomic per slot and group, with LDS atomics per element
// unless the slots divided the grid's stride, and device atomics per element
// for slots that do not fit the LDS: 2^26 fp32 adds into 1024 slots 50 -> 42
// us, 5000 slots 339 -> 44 us, 100,000 slots 219 -> 43 us; 2^28 into 1024
// slots 158.6 -> 157.2 us (6.8 TB/s), into 777 slots 1333 -> 160 us; 2^21
// fp32 max into 1024 slots 103 -> 11 us.
template <class T, class R, bool NT>
__global__ __launch_bounds__(1024) void strided_strip_kernel(const T *__restrict__ v, strip_params p, T *target) {
  constexpr int VEC = 16 / sizeof(T);
  constexpr int UNROLL = 4;
  extern __shared__ unsigned char lds_raw[];
  T *lds = reinterpret_cast<T *>(lds_raw);  // blockDim.x x VEC
  const uint32_t width = 1u << p.width_log2;
  const uint32_t rows = blockDim.x >> p.width_log2;
  const uint64_t strip = blockIdx.x / p.row_groups;
  const uint64_t row_group = blockIdx.x - strip * p.row_groups;
  const uint64_t first_column = strip << p.width_log2;
  const uint64_t column = first_column + (threadIdx.x & (width - 1u));
  const u32x4 *vv = reinterpret_cast<const u32x4 *>(v + p.gm.head);
  T acc[VEC];
#pragma unroll
  for (int k = 0; k < VEC; ++k) acc[k] = R::identity();
  const uint64_t stride = p.row_groups * rows * p.columns;
  uint64_t c = (row_group * rows + (threadIdx.x >> p.width_log2)) * p.columns + column;
  if (column >= p.columns || (threadIdx.x >> p.width_log2) >= rows) c = p.gm.nvec;
  auto load = [&](uint64_t i) {
    if constexpr (NT)
      return __builtin_nontemporal_load(vv + i);
    else
      return vv[i];
  };
  auto fold = [&](u32x4 q) {
    T e[VEC];
    __builtin_memcpy(e, &q, 16);
#pragma unroll
    for (int k = 0; k < VEC; ++k) acc[k] = R::apply(acc[k], e[k]);
  };
  for (; c + (UNROLL - 1) * stride < p.gm.nvec; c += UNROLL * stride) {
    u32x4 q[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) q[u] = load(c + u * stride);
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) fold(q[u]);
  }
  for (; c < p.gm.nvec; c += stride) fold(load(c));
#pragma unroll
  for (int k = 0; k < VEC; ++k) lds[threadIdx.x * VEC + k] = acc[k];
  __syncthreads();
  // Values e, e + num_slots, ... of every row of the strip meet one slot.  Only
  // slots that met an element go on to the atomics (a NaN in the target gives
  // way to any value): those of the vectors in the group's first row.
  const uint32_t values = width * VEC;
  const uint64_t first_vec = row_group * rows * p.columns + first_column;
  const uint64_t left_in_row = p.columns - first_column;
  const uint64_t left = p.gm.nvec > first_vec ? p.gm.nvec - first_vec : 0;
  const uint64_t in_row = (left < left_in_row ? left : left_in_row) * VEC;
  const uint32_t used = in_row < values ? static_cast<uint32_t>(in_row) : values;
  const uint32_t slots = p.num_slots < used ? static_cast<uint32_t>(p.num_slots) : used;
  for (uint32_t e = threadIdx.x; e < used; e += blockDim.x) {
    T x = lds[e];
    for (uint32_t r = 1; r < rows; ++r) x = R::apply(x, lds[r * values + e]);
    lds[e] = x;  // row 0's value e is read by this work-item only
  }
  __syncthreads();
  // Four to one per step: with 18 slots a chain of 57 LDS reads took 2.5 us
  // at the end of every launch.
  for (uint32_t count = used; count > slots;) {
    const uint32_t next = (count + 4 * slots - 1) / (4 * slots) * slots;  // whole periods
    for (uint32_t e = threadIdx.x; e < next; e += blockDim.x) {
      T x = lds[e];
#pragma unroll
      for (uint32_t j = 1; j < 4; ++j)
        if (e + j * next < count) x = R::apply(x, lds[e + j * next]);
      lds[e] = x;
    }
    __syncthreads();
    count = next;
  }
  for (uint32_t e = threadIdx.x; e < slots; e += blockDim.x)
    R::template atomic<scope_dev>(&target[(p.gm.head + first_column * VEC + e) % p.num_slots], lds[e]);
  // The head and the tail (fewer than 2 VEC elements).
  if (blockIdx.x == 0)
    for (uint64_t s = threadIdx.x; s < p.gm.nscalar; s += blockDim.x) {
      const uint64_t i = scalar_index(p.gm, s);
      R::template atomic<scope_dev>(&target[i % p.num_slots], v[i]);
    }
}

// The reference's pattern: one device-scope atomic per element.
template <class T, class R>
__global__ __launch_bounds__(1024) void strided_global_kernel(const T *__restrict__ v, uint64_t n,
                                                              uint32_t num_slots, T *target) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    R::template atomic<scope_dev>(&target[i % num_slots], v[i]);
}

uint32_t pick_grid(uint64_t work_items, uint32_t wg, uint64_t max_groups) {
  uint64_t g = ceil_div(work_items, wg);
  if (g < 1) g = 1;
  if (g > max_groups) g = max_groups;
  return static_cast<uint32_t>(g);
}

// More bins than max_plain_bins are counted in packed 16-bit fields, unless
// there are few keys: the partials of 32-bit counters are twice the bytes
// (2^24 keys into 32768 bins: 34.0 -> 27.6 us, into 16384 bins: 25.9 -> 22.3
// us).
constexpr uint32_t max_plain_bins = 8192;
constexpr uint32_t max_local_bins = 65536;  // packed counters of one LDS
constexpr uint32_t max_slices_log2 = 6;
constexpr uint64_t direct_keys_per_group = 4096;

// True where the groups add their counters that are not zero straight to the
// bins: few keys, or few bins.  No second launch and no partials, but atomics
// on every line of the bins by every group.  Calls with the clear of the bins,
// through partials and so: up to 2^17 keys 14.2 and 10.5 us; 2^24 keys into
// 4096 bins 22.4 and 18.8 us, 3M into 8192 14.8 and 10.4 us; 600,000 keys
// (147 groups) into 9548 bins 14.5 and 10.3 us, into 20000 bins 14.4 and
// 12.5 us, into 25000 bins 14.5 and 15.5 us; 1.5M keys (256 groups) into 9548
// bins 11.5 and 14.1 us.  In these calls the counters are plain where they fit
// the LDS: flushing packed ones takes two atomics a word (600,000 keys into
// 9548 bins: 14.4 us packed).
bool direct_flush(uint64_t n, uint32_t num_bins) {
  if (n <= (1ull << 17) || num_bins <= max_plain_bins) return true;
  return n <= 5ull << 17 && static_cast<uint64_t>(num_bins) * 4 <= lds_bytes_budget &&
         ceil_div(n, direct_keys_per_group) * num_bins <= 3ull << 20;
}

acpp_status histogram(acpp_allocation_group *g, hipStream_t stream, const uint32_t *keys,
                      uint64_t n, uint32_t *bins, uint32_t num_bins, int strat,
                      const acpp_launch_config *cfg) {
  const char *name = "acpp_histogram_u32";
  if (!g) return set_error(ACPP_ERROR_INVALID_ARGUMENT, "acpp_histogram_u32: scratch group is NULL");
  if (!bins || num_bins == 0)
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, "acpp_histogram_u32: bins is NULL or num_bins is 0");
  if (n > 0 && !keys) return set_error(ACPP_ERROR_INVALID_ARGUMENT, "acpp_histogram_u32: keys is NULL");
  if (strat < strat_auto || strat > strat_global)
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, "acpp_histogram_u32: unknown strategy");
  if (n == 0) return clear_error();
  int cus = 0;
  acpp_status st = enter_device(g, &cus);
  if (st != ACPP_SUCCESS) return st;
  const bool fits16 = static_cast<uint64_t>((num_bins + 1) / 2) * 4 <= lds_bytes_budget;
  if (strat == strat_privatized && !fits16)
    return set_error(ACPP_ERROR_UNSUPPORTED,
                     "acpp_histogram_u32: more than 65536 bins do not fit the LDS; use the global strategy");
  // More bins than one LDS holds are cut into slices, always by 1024-wide groups
  // (128 KiB of counters to clear and to flush: 2M keys into 2.5M bins 610 us
  // 64 wide).  Every slice visits
  // every key, so beyond max_slices one atomic per key is the better form.
  uint32_t slices_log2 = 0;
  while (!fits16 && slices_log2 < max_slices_log2 && ceil_div(num_bins, 1ull << slices_log2) > max_local_bins) ++slices_log2;
  const bool sliceable = !fits16 && ceil_div(num_bins, 1ull << slices_log2) <= max_local_bins;
  const int strat_given = strat;
  // A few thousand keys: every slice's counters take longer to clear and to
  // look through (1000 uniform keys into 200,000 bins 3.4 us by atomics, 10.7 us
  // in slices; 4000 Zipf keys 9.3 and 10.5 us, into 66,000 10.0 and 8.2 us; all
  // in one bin, 2000 keys 30 us and 11 us).
  const bool few_keys = n <= 2048 || (n <= 4096 && num_bins > 2 * max_local_bins);
  if (strat == strat_auto) strat = (fits16 || (sliceable && !few_keys)) ? strat_privatized : strat_global;
  const uint32_t wg_given = (cfg && cfg->work_group_size) ? cfg->work_group_size : 1024;
  if (!valid_work_group_size(wg_given))
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, "acpp_histogram_u32: bad work_group_size");
  const uint32_t wg = !fits16 && strat == strat_privatized ? 1024 : wg_given;
  const geom gm = make_geom(keys, n);

  if (strat == strat_global) {
    auto kernel = histogram_global_kernel<4>;
    int resident = 1;
    st = occupancy(kernel, static_cast<int>(wg), &resident);
    if (st != ACPP_SUCCESS) return st;
    uint64_t groups_cap = static_cast<uint64_t>(resident) * cus;
    if (cfg && cfg->groups_per_cu)
      groups_cap = std::min<uint64_t>(groups_cap, cfg->groups_per_cu * static_cast<uint64_t>(cus));
    const uint32_t grid = pick_grid(gm.nvec + gm.nscalar, wg * 4, groups_cap);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(wg), 0, stream, keys, gm, num_bins, bins);
    st = check_launch(name);
    return st == ACPP_SUCCESS ? clear_error() : st;
  }

  // Cost of a form with 2^sl slices, from rates measured on MI355X: the keys'
  // time falls with the number of groups, the time to write and read the
  // groups' partials grows with it, and their sum is least at the square
  // root.  A CU counts a key in 0.15 ns, visits one of a slice in 0.11 ns;
  // partials move at about 4 TB/s.
  const uint64_t cu_groups = static_cast<uint64_t>(cus);
  const bool groups_given = cfg && cfg->groups_per_cu;
  const bool direct = !groups_given && direct_flush(n, num_bins);
  const bool packed = num_bins > max_plain_bins && !(direct && static_cast<uint64_t>(num_bins) * 4 <= lds_bytes_budget);
  struct form {
    uint32_t slices_log2;
    uint32_t words;  // 32-bit words of a group's partial
    double groups;
    double seconds;
  };
  auto cost = [&](uint32_t sl) {
    form f;
    f.slices_log2 = sl;
    f.words = packed ? ((((num_bins - 1) >> sl) + 1) + 1) / 2 : num_bins;
    const double keys_s = static_cast<double>(n) * (sl ? (1u << sl) * 1.1e-10 : 1.5e-10);
    const double partial_s = 8.0 * f.words / 4e12;
    f.groups = std::min(static_cast<double>(cu_groups), std::sqrt(keys_s / partial_s));
    f.seconds = keys_s / f.groups + partial_s * f.groups;
    return f;
  };
  form best = cost(slices_log2);
  // Twice the slices halve the partials: better for few keys and many bins
  // (2^24 keys, 65536 bins: 35.7 -> 29.7 us; 2^23 keys: 30.3 -> 24.2 us).
  if (packed && slices_log2 < max_slices_log2 && strat_given == strat_auto) {
    const form twice = cost(slices_log2 + 1);
    if (twice.seconds < best.seconds) best = twice;
  }
  slices_log2 = best.slices_log2;
  const uint32_t slices = 1u << slices_log2;
  hist_params p;
  p.keys = keys;
  p.gm = gm;
  p.bins = bins;
  p.num_bins = num_bins;
  p.local_bins = ((num_bins - 1) >> slices_log2) + 1;
  p.slices_log2 = slices_log2;
  // Up to 8 copies of 32-bit counters within the LDS budget.
  p.copies_log2 = 0;
  while (!packed && p.copies_log2 < 3 &&
         (static_cast<uint64_t>(num_bins) << (p.copies_log2 + 1)) * 4 <= lds_bytes_budget)
    ++p.copies_log2;
  const uint32_t partial_words = best.words;
  const size_t lds = (static_cast<size_t>(partial_words) << p.copies_log2) * 4;
  auto kernel = slices > 1 ? histogram_kernel<true, true, 4>
                : packed   ? histogram_kernel<true, false, 4>
                           : histogram_kernel<false, false, 4>;
  // One group per CU by default: the kernel is bound by the CU's LDS atomic
  // rate (about two keys per clock), and a second resident group only adds
  // contention (2^28 Zipf keys, 4096 bins on MI355X: 252 us with one group
  // per CU, 302 us with two).
  uint64_t groups = cu_groups;
  if (groups_given) {
    int resident = 1;
    ACPP_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&resident, kernel, static_cast<int>(wg), lds));
    if (resident < 1) resident = 1;
    groups = std::min<uint64_t>(cfg->groups_per_cu, resident) * cu_groups;
    // Each group writes a partial histogram; keep the partials to at most 1/8
    // of the key bytes (but at least one group per CU).
    groups = std::min(groups, std::max<uint64_t>(cu_groups, (n / 8) / num_bins));
    groups = pick_grid(gm.nvec + gm.nscalar, wg * 4, groups);
  } else {
    const uint64_t part = static_cast<uint64_t>(ceil_div(n, direct_keys_per_group)) << slices_log2;
    groups = std::min(groups, part);
    // Atomics on one line are served one after the other: more than 96 groups
    // that flush few bins want more keys each (1M keys into 150 bins 7.4 us with
    // 245 groups, 5.0 us with 96; 2M into 1750 8.7 and 7.7 us).
    if (direct && !packed && groups > 96)
      groups = std::max<uint64_t>(96, std::min(groups, ceil_div(n, 3 * direct_keys_per_group)));
    if (!direct) groups = std::min(groups, static_cast<uint64_t>(best.groups) + 1);
  }
  if (slices > 1) {
    // whole chunks: every slice of a part of the keys, on one XCD if it can be
    const uint64_t per_xcd = static_cast<uint64_t>(slices) * 8;
    groups = std::max<uint64_t>(groups / slices, 1) * slices;
    if (groups > per_xcd) groups = groups / per_xcd * per_xcd;
  }
  p.xcd_map = slices > 1 && groups % (static_cast<uint64_t>(slices) * 8) == 0;
  p.chunks = static_cast<uint32_t>(groups >> slices_log2);
  const uint32_t grid = static_cast<uint32_t>(groups);
  // The sliced form can do without scratch, with one atomic per group and bin
  // instead: more than 65536 bins under stream capture, which have never held
  // the group's memory there, and any when there is none to have.  Fewer bins
  // under capture, where an allocation can fail and take the capture with it,
  // use what the cache holds (2^24 keys into 65536 bins, after an eager call: a
  // replay 61.4 us without partials, 34.0 us with them).
  p.partials = nullptr;
  if (!direct) {
    const size_t bytes = static_cast<size_t>(grid) * partial_words * sizeof(uint32_t);
    void *partials = nullptr;
    if (slices == 1) {
      st = group_obtain(g, bytes, &partials);
      if (st != ACPP_SUCCESS) return st;
    } else if (stream_is_capturing(stream)) {
      if (fits16) group_obtain_cached(g, bytes, &partials);
    } else {
      (void)group_obtain(g, bytes, &partials);
    }
    p.partials = static_cast<uint32_t *>(partials);
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(wg), lds, stream, p);
  st = check_launch(name);
  if (st != ACPP_SUCCESS) return st;
  if (!p.partials) return clear_error();
  const uint32_t x = static_cast<uint32_t>(ceil_div(partial_words, 1ull << combine_span_log2(slices_log2)));
  const uint32_t y = std::max(1u, std::min(std::min(p.chunks, 32u), 1024u / x));
  if (packed)
    hipLaunchKernelGGL(histogram_combine_kernel<true>, dim3(x, y), dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL(histogram_combine_kernel<false>, dim3(x, y), dim3(256), 0, stream, p);
  st = check_launch(name);
  return st == ACPP_SUCCESS ? clear_error() : st;
}

constexpr uint64_t min_columns = 512;
constexpr uint64_t max_columns = 8192;

template <class T, template <class> class RT>
acpp_status strided(acpp_allocation_group *g, hipStream_t stream, const T *values, uint64_t n,
                    T *target, uint32_t num_slots, int strat, const acpp_launch_config *cfg,
                    const char *name) {
  using R = RT<T>;
  if (!g) return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": scratch group is NULL");
  if (!target || num_slots == 0)
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": target is NULL or num_slots is 0");
  if (n > 0 && !values) return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": values is NULL");
  if (strat < strat_auto || strat > strat_global)
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": unknown strategy");
  if (n == 0) return clear_error();
  int cus = 0;
  acpp_status st = enter_device(g, &cus);
  if (st != ACPP_SUCCESS) return st;
  constexpr uint32_t VEC = 16 / sizeof(T);
  if (strat == strat_privatized && static_cast<uint64_t>(num_slots) * sizeof(T) > lds_bytes_budget)
    return set_error(ACPP_ERROR_UNSUPPORTED, std::string(name) + ": slots do not fit the LDS; use the global strategy");
  if (strat == strat_global) {
    const uint32_t wg = (cfg && cfg->work_group_size) ? cfg->work_group_size : 256;
    if (!valid_work_group_size(wg))
      return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": bad work_group_size");
    const uint64_t cap_groups =
        static_cast<uint64_t>(cus) * ((cfg && cfg->groups_per_cu) ? cfg->groups_per_cu : 2);
    const uint32_t grid = pick_grid(n, wg, cap_groups * 8);
    hipLaunchKernelGGL((strided_global_kernel<T, R>), dim3(grid), dim3(wg), 0, stream, values, n, num_slots, target);
  } else {
    const uint32_t wg = (cfg && cfg->work_group_size) ? cfg->work_group_size : 512;
    if (!valid_work_group_size(wg))
      return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": bad work_group_size");
    strip_params p;
    p.gm = make_geom(values, n);
    p.num_slots = num_slots;
    // The shortest row of whole vectors, repeated to min_columns at least.
    p.columns = num_slots / std::gcd<uint64_t>(VEC, num_slots);
    // Inputs that the last-level cache does not hold beside others stream past
    // it, in strips of 4 KiB a row (1 KiB cached and 4 KiB streaming: 2^28
    // fp32 into 1024 slots 169 and 157 us, 240 MB 44.6 and 39.2 us, 180 MB
    // 33.2 and 31.6 us, 130 MB 21.9 and 25.7 us).
    const bool large = n * sizeof(T) >= (160ull << 20);
    const uint32_t narrow = large ? 8 : 6;
    // Where the last strip of that row would leave more than a quarter of the
    // groups idle, the row up to max_columns with the least of it, in whole
    // cache lines (2^27 fp32 max into 18 slots: 513 columns in 3 strips 92
    // us, 1512 in 6 strips 81 us).  Less idle costs nothing, the loads are
    // bound by the memory (2^26 fp32 into 777 slots: 777 columns in 4 strips
    // 44.7 us, 6216 in 25 strips 46.8 us).
    auto idle = [&](uint64_t columns) {
      const uint64_t whole = ceil_div(columns, 1ull << narrow) << narrow;
      return static_cast<double>(whole - columns) / static_cast<double>(whole);
    };
    const uint64_t line_row = std::lcm<uint64_t>(p.columns, 8);
    const uint64_t tallest = std::min(max_columns, p.gm.nvec / (4 * ceil_div(wg, 1ull << narrow)));
    p.columns *= ceil_div(min_columns, p.columns);
    double least = idle(p.columns);
    if (least > 0.26)
      for (uint64_t c = ceil_div(min_columns, line_row) * line_row; c <= tallest && least > 1.0 / 64; c += line_row)
        if (idle(c) < least) {
          p.columns = c;
          least = idle(c);
        }
    const uint64_t used_columns = std::max<uint64_t>(1, std::min(p.columns, p.gm.nvec));
    const uint64_t rows = std::max<uint64_t>(1, ceil_div(p.gm.nvec, p.columns));
    // Strips as narrow as a wave (fewest atomics; 2^23 fp32 into 1024 slots:
    // 9.3 us, 13.3 us with 4 KiB a row), or wider when there are too few rows for all
    // work-items.
    p.width_log2 = narrow;
    while ((1u << p.width_log2) < wg && (wg >> p.width_log2) > rows) ++p.width_log2;
    while ((1u << p.width_log2) > wg) --p.width_log2;
    const uint64_t strips = ceil_div(used_columns, 1ull << p.width_log2);
    const uint64_t band_rows = wg >> p.width_log2;
    // One group per CU, but as many as keep its loads going where the groups
    // are narrower than the default: 576 work-items and six groups, 128
    // work-items where the cache holds the input and the flushes count more
    // (int32 into 67 slots: 100M 192 wide 122 us with one group, 76 with two, 72
    // with three, 26M 23, 28 and 32; 47M 64 wide 124 us with one, 67 with two,
    // 62 with six, 72 with eight.  int64: 47M 192 wide 113 us with one, 69 with
    // three, 8M 18 and 30).
    const bool groups_given = cfg && cfg->groups_per_cu;
    const uint32_t per_cu = groups_given ? cfg->groups_per_cu
                                         : std::max(1u, large ? std::min(6u, 576u / wg) : 128u / wg);
    const uint64_t cap_groups = static_cast<uint64_t>(cus) * per_cu;
    const uint64_t wanted = std::min(cap_groups, std::max<uint64_t>(1, ceil_div(p.gm.nvec, static_cast<uint64_t>(wg) * 4)));
    const uint64_t bands = std::max<uint64_t>(1, ceil_div(rows, band_rows));
    p.row_groups = std::max<uint64_t>(1, std::min(wanted / strips, bands));
    // A few strips more than CUs take two rounds of groups: then as many groups
    // to a strip as load the CUs evenly, four to a CU at most (20M fp64 into
    // 35,982 slots, 282 strips: 38.5 us with one group a strip, 28.4 with two).
    if (!groups_given && strips > static_cast<uint64_t>(cus)) {
      auto rounds = [&](uint64_t r) {
        return static_cast<double>(ceil_div(strips * r, static_cast<uint64_t>(cus))) / static_cast<double>(r);
      };
      const uint64_t most = std::min(bands, 4 * static_cast<uint64_t>(cus) / strips);
      for (uint64_t r = 2; r <= most; ++r)
        if (rounds(r) < 0.85 * rounds(p.row_groups)) p.row_groups = r;
    }
    const uint64_t grid = strips * p.row_groups;
    if (grid >= (1ull << 31))
      return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": problem too large");
    const size_t lds = static_cast<size_t>(wg) * 16;
    if (large)
      hipLaunchKernelGGL((strided_strip_kernel<T, R, true>), dim3(static_cast<uint32_t>(grid)), dim3(wg), lds, stream,
                         values, p, target);
    else
      hipLaunchKernelGGL((strided_strip_kernel<T, R, false>), dim3(static_cast<uint32_t>(grid)), dim3(wg), lds, stream,
                         values, p, target);
  }
  st = check_launch(name);
  return st == ACPP_SUCCESS ? clear_error() : st;
}

}  // namespace atomics_detail
}  // namespace acpp_impl

using namespace acpp_impl;
using namespace acpp_impl::atomics_detail;

extern "C" {

acpp_status acpp_histogram_u32(acpp_allocation_group *scratch, acpp_stream_t stream, const uint32_t *keys,
                               uint64_t n, uint32_t *bins, uint32_t num_bins, int strategy,
                               const acpp_launch_config *config) {
  return histogram(scratch, static_cast<hipStream_t>(stream), keys, n, bins, num_bins, strategy, config);
}

#define ACPP_DEFINE_STRIDED(opname, RT, tag, T)                                                           \
  acpp_status acpp_atomic_fetch_##opname##_strided_##tag(acpp_allocation_group *scratch, acpp_stream_t stream, \
                                                         const T *values, uint64_t n, T *target,          \
                                                         uint32_t num_slots, int strategy,                \
                                                         const acpp_launch_config *config) {              \
    return strided<T, RT>(scratch, static_cast<hipStream_t>(stream), values, n, target, num_slots,        \
                          strategy, config, "acpp_atomic_fetch_" #opname "_strided_" #tag);              \
  }
#define ACPP_DEFINE_STRIDED_ALL(tag, T)         \
  ACPP_DEFINE_STRIDED(add, rmw_add, tag, T)     \
  ACPP_DEFINE_STRIDED(min, rmw_min, tag, T)     \
  ACPP_DEFINE_STRIDED(max, rmw_max, tag, T)

ACPP_DEFINE_STRIDED_ALL(i32, int32_t)
ACPP_DEFINE_STRIDED_ALL(u32, uint32_t)
ACPP_DEFINE_STRIDED_ALL(i64, int64_t)
ACPP_DEFINE_STRIDED_ALL(u64, uint64_t)
ACPP_DEFINE_STRIDED_ALL(f32, float)
ACPP_DEFINE_STRIDED_ALL(f64, double)

}  // extern "C"
