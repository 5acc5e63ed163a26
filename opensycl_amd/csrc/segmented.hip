// Segmented scans and reductions: thousands of independent scans /
// reductions over [offsets[s], offsets[s+1]) in one launch.
//
// The reference has no segmented form; the nearest equivalents are one
// joint_* group algorithm call per segment
// (include/hipSYCL/sycl/libkernel/generic/hiplike/group_functions.hpp:214-287,
// 361-432) or one algorithms::inclusive_scan / reduce call per segment
// (include/hipSYCL/algorithms/numeric.hpp:226-279), each a separate launch.
//
// MI355X design:
//   - the concatenated elements are cut into equal tiles, independent of the
//     segment lengths, so log-normal segment lengths cost no load imbalance;
//   - a tile finds the segments that start in it by a search of the offsets
//     (few tiles), or from a bitmap of the starts (scans) or a table of every
//     tile's first segment (reductions) that a kernel before it wrote;
//   - scans: persistent work-groups (one wave of resident groups) draw tiles
//     from a ticket counter in order; every tile puts its segment starts in an
//     LDS bitmap and runs a segmented scan over (head flag, value) pairs:
//     (f1,v1) . (f2,v2) = (f1|f2, f2 ? v2 : v1 op v2), in registers, across
//     each wave with DPP and across waves through LDS;
//   - tiles chain through a decoupled look-back on the pair operator.  The
//     operator is not commutative, so the window is folded in tile order,
//     and a look-back stops at the nearest predecessor that contains a
//     segment start (its aggregate already discards everything before it),
//     so it is short whenever segments are shorter than a tile;
//   - scans write every element.  Reductions skip the look-back: each tile
//     writes the totals of the segments it holds whole (init for empty ones)
//     and two partial folds, and a fix-up kernel joins the partials of segments that span
//     tiles (segmented_reduce_kernel below);
//   - a plan keeps a call's scratch and parameters (acpp_segmented_plan_*).
#include <memory>
#include <mutex>
#include <new>

#include "launch_util.hpp"

namespace acpp_impl {
namespace seg_detail {

constexpr int max_waves = 16;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
// 16-byte vector accesses need dword alignment only; every segmented element
// type is 4 or 8 bytes, so any element-aligned view takes the vector path.
typedef unsigned int u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

enum : uint32_t { st_invalid = 0, st_aggregate = 1, st_prefix = 2 };

// Status tags: status_tag() in internal.hpp (epoch << 3 | head flag << 2 |
// status), shared with the scans.

__device__ __forceinline__ uint64_t ld64(const uint64_t *p) {
  return __hip_atomic_load(const_cast<uint64_t *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st64(uint64_t *p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <class W, int Bytes = sizeof(W)>
struct seg_status;

// Each tile's status has a 128-byte line of its own, so that the polls of
// all tiles in flight do not pile onto a few lines.
constexpr uint64_t seg_stride_words = 16;

template <class W>
struct seg_status<W, 4> {
  static constexpr int words = 1;
  __device__ static void publish(uint64_t *st, uint32_t tile, uint32_t epoch, uint32_t status,
                                 uint32_t f, W v) {
    const uint64_t tag = status_tag(epoch, f, status);
    st64(st + tile * seg_stride_words, (tag << 32) | __builtin_bit_cast(uint32_t, v));
  }
  __device__ static uint32_t read(const uint64_t *st, uint32_t tile, uint32_t epoch, uint32_t &f,
                                  W &v) {
    const uint64_t w = ld64(st + tile * seg_stride_words);
    const uint32_t tag = static_cast<uint32_t>(w >> 32);
    if (tag_epoch(tag) != epoch) return st_invalid;
    f = tag_head(tag);
    v = __builtin_bit_cast(W, static_cast<uint32_t>(w));
    return tag_status(tag);
  }
};

template <class W>
struct seg_status<W, 8> {
  static constexpr int words = 2;
  __device__ static void publish(uint64_t *st, uint32_t tile, uint32_t epoch, uint32_t status,
                                 uint32_t f, W v) {
    const uint64_t tag = status_tag(epoch, f, status);
    const uint64_t bits = __builtin_bit_cast(uint64_t, v);
    uint64_t *slot = st + tile * seg_stride_words;
    st64(slot, (tag << 32) | (bits & 0xffffffffu));
    st64(slot + 1, (tag << 32) | (bits >> 32));
  }
  __device__ static uint32_t read(const uint64_t *st, uint32_t tile, uint32_t epoch, uint32_t &f,
                                  W &v) {
    const uint64_t *slot = st + tile * seg_stride_words;
    const uint64_t w0 = ld64(slot);
    const uint64_t w1 = ld64(slot + 1);
    const uint32_t t0 = static_cast<uint32_t>(w0 >> 32);
    const uint32_t t1 = static_cast<uint32_t>(w1 >> 32);
    if (t0 != t1 || tag_epoch(t0) != epoch) return st_invalid;
    f = tag_head(t0);
    v = __builtin_bit_cast(W, (w1 << 32) | (w0 & 0xffffffffu));
    return tag_status(t0);
  }
};

// (f, v) pair operator, earlier . later
template <class Op, class W>
__device__ __forceinline__ void combine(uint32_t fa, W va, uint32_t &fb, W &vb) {
  vb = fb ? vb : Op::apply(va, vb);
  fb |= fa;
}

// Inclusive scan of pairs across the wave (lane order = element order).
template <class Op, class W>
__device__ __forceinline__ void wave_pair_scan(uint32_t &f, W &v) {
  const W id = Op::identity();
#define ACPP_SEG_STEP(CTRL, RM)                                  \
  {                                                              \
    const uint32_t fo = wave::dpp<CTRL, RM, 0xf>(0u, f);         \
    const W vo = wave::dpp<CTRL, RM, 0xf>(id, v);                \
    combine<Op>(fo, vo, f, v);                                   \
  }
  ACPP_SEG_STEP(wave::row_shr1, 0xf)
  ACPP_SEG_STEP(wave::row_shr2, 0xf)
  ACPP_SEG_STEP(wave::row_shr4, 0xf)
  ACPP_SEG_STEP(wave::row_shr8, 0xf)
  ACPP_SEG_STEP(wave::row_bcast15, 0xa)
  ACPP_SEG_STEP(wave::row_bcast31, 0xc)
#undef ACPP_SEG_STEP
}

// Exclusive prefixes, in element order, of a tile's per-(row, wave) pair
// totals.  s_tf / s_tv[r * nw + w] hold the totals on entry and the
// exclusive prefixes on return (P = R * nw <= 128 entries).  Called by one
// whole wave, which scans them with DPP (two entries per lane above 64);
// returns the tile aggregate, uniform across the wave.  Replaces a serial
// walk over all R * nw totals by every work-item.
template <class Op, class W>
__device__ void tile_pair_prefixes(int P, uint32_t *s_tf, W *s_tv, uint32_t &agg_f, W &agg_v) {
  const int lane = threadIdx.x & 63;
  const W id = Op::identity();
  const int per = P > 64 ? 2 : 1;
  const int a = lane * per;
  uint32_t f0 = 0, f1 = 0;
  W v0 = id, v1 = id;
  if (a < P) {
    f0 = s_tf[a];
    v0 = s_tv[a];
  }
  if (per == 2 && a + 1 < P) {
    f1 = s_tf[a + 1];
    v1 = s_tv[a + 1];
  }
  uint32_t sf = f1;  // lane total: entry a . entry a + 1
  W sv = v1;
  combine<Op>(f0, v0, sf, sv);
  wave_pair_scan<Op>(sf, sv);
  const uint32_t xf = wave::dpp<wave::wave_shr1, 0xf, 0xf>(0u, sf);
  const W xv = wave::dpp<wave::wave_shr1, 0xf, 0xf>(id, sv);
  agg_f = wave::read_lane(sf, 63);
  agg_v = wave::read_lane(sv, 63);
  if (a < P) {
    s_tf[a] = xf;
    s_tv[a] = xv;
  }
  if (per == 2 && a + 1 < P) {
    uint32_t bf = f0;
    W bv = v0;
    combine<Op>(xf, xv, bf, bv);
    s_tf[a + 1] = bf;
    s_tv[a + 1] = bv;
  }
}

// Ordered look-back by one wave: lane l polls tile (wbase - 63 + l), lane 63
// the nearest predecessor.  It stops at the nearest tile that is a prefix
// or an aggregate containing a segment start, and folds the window from
// there in tile order.  Must be called by a whole wave; result uniform.
template <class Op, class W>
__device__ void wave_pair_lookback(const uint64_t *status, uint32_t tile, uint32_t epoch,
                                   sync_header *sync, bool force_give_up, uint32_t &out_f, W &out_v) {
  using SIO = seg_status<W>;
  const int lane = threadIdx.x & 63;
  const W id = Op::identity();
  int64_t wbase = static_cast<int64_t>(tile) - 1;
  uint32_t ef = 0;  // accumulated prefix of tiles nearer than the window
  W ev = id;
  lookback_wait wait;
  wait.begin();
  bool give_up = force_give_up;  // uniform
  if (give_up && lane == 0) report_trip(sync);
  for (;;) {
    const int64_t j = wbase - (63 - lane);
    uint32_t lf = 0;
    W lv = id;
    int q;
    for (;;) {
      uint32_t st = st_prefix;  // positions before tile 0 act as an empty prefix
      lf = 0;
      lv = id;
      if (j >= 0) st = SIO::read(status, static_cast<uint32_t>(j), epoch, lf, lv);
      if (give_up) st = st_prefix;
      const bool term = (st == st_prefix) || (st == st_aggregate && lf);
      const uint64_t tm = wave::ballot(term);
      q = tm ? 63 - __builtin_clzll(tm) : -1;
      const uint64_t need = (q <= 0) ? ~0ull : (~0ull << q);  // lanes q..63
      const uint64_t bad = wave::ballot(st == st_invalid) & need;
      if (bad == 0) break;
      if (wait.failed_round()) {
        give_up = true;
        if (lane == 0) report_trip(sync);
      }
    }
    uint32_t xf = (lane >= q) ? lf : 0u;
    W xv = (lane >= q) ? lv : id;
    wave_pair_scan<Op>(xf, xv);
    uint32_t wf = wave::read_lane(xf, 63);
    W wv = wave::read_lane(xv, 63);
    // window (earlier) . accumulated (later)
    combine<Op>(wf, wv, ef, ev);
    if (q >= 0) break;
    wbase -= 64;
  }
  out_f = ef;
  out_v = ev;
}

template <class T>
struct params {
  using W = typename elem_traits<T>::work;
  const T *in;
  T *out;
  const uint64_t *offsets;  // num_segments + 1 entries
  const uint32_t *tile_seg;  // reductions: first segment of every tile (tile_table_kernel), or NULL
  const uint32_t *heads;     // scans: bit e set: a segment starts at element e; or NULL
  uint64_t head_words_total;  // 32-bit words of the bitmap
  int block_lookback;        // 1: work-group-wide look-back window
  int force_give_up;         // ACPP_VARIANT_FORCE_GIVE_UP (tests of the error path)
  uint64_t num_segments;
  uint64_t total;
  W init;
  int vec_io;
  uint32_t num_tiles;
  uint32_t epoch;
  uint32_t ticket_base;
  sync_header *sync;
  uint64_t *status;
};

__device__ __forceinline__ uint64_t clamp_off(const uint64_t *offsets, uint64_t s, uint64_t total) {
  const uint64_t o = offsets[s];
  return o < total ? o : total;
}

// The number of leading positions of [0, n) that `below` holds for, found by a
// whole wave: 64 probes a round shrink the range 65 times, so 65,536 positions
// take three dependent loads and 2^26 five.  Where `below` does not hold for a
// prefix (unsorted offsets), some value in [0, n].  The result is uniform.
template <class Below>
__device__ __forceinline__ uint64_t wave_partition_point(uint64_t n, Below below) {
  const uint64_t lane = threadIdx.x & 63;
  uint64_t lo = 0, hi = n;
  while (lo < hi) {
    const uint64_t step = (hi - lo + 64) / 65;
    const uint64_t at = lo + (lane + 1) * step - 1;
    const uint64_t c = static_cast<uint64_t>(__builtin_popcountll(wave::ballot(at < hi && below(at))));
    if (c < 64) hi = min(hi, lo + (c + 1) * step - 1);
    lo += c * step;
  }
  return lo;
}

// The number of offsets[0 .. n) below key.
__device__ __forceinline__ uint64_t wave_lower_bound(const uint64_t *offsets, uint64_t n, uint64_t key) {
  return wave_partition_point(n, [&](uint64_t i) { return offsets[i] < key; });
}

// More starts than this in 64 elements are taken for those of a run of empty segments.
constexpr uint32_t run_starts = 4096;

// Sets bit `at` of s_heads; none for no_head.  Lanes that follow one with the
// same bit leave it to that one: the starts of a run of empty segments are
// one address, and their atomics would go one after the other.
constexpr uint32_t no_head = 0xffffffffu;
__device__ __forceinline__ void mark_head(uint32_t *s_heads, uint32_t at) {
  const uint32_t before = wave::dpp<wave::wave_shr1, 0xf, 0xf>(no_head, at);
  if (at != no_head && at != before) atomicOr(&s_heads[at >> 5], 1u << (at & 31));
}

// Segments that a work-group walks one by one.  Where more start in its tile,
// most of them are empty, and it looks the tile's starts up by element instead
// (tile_starts): 30,000 empty segments in one place of 2^26 int32, 256 x 4 tiles,
// 113 us of reduce kernel walked and 63 us looked up; but two starts per element
// everywhere (2^23 int32, 1024 x 4 tiles) 111 us a call walked and 260 us
// looked up.
__host__ __device__ constexpr uint32_t max_walk_segments(uint32_t work_group) {
  return work_group > 256 ? 64u * work_group : 16384u;
}
// Calls with at most this many segments have kernels without that: a walk of
// 16 rounds is the worst that can happen to them.
__host__ __device__ constexpr uint32_t max_few_segments(uint32_t work_group) { return 16u * work_group; }

// The starts offsets[lo .. lo + count) of a tile whose first element is `base`,
// however many: one binary search finds, for each of the wave's blocks of 64
// elements, the starts in it; a second one inside the block finds each
// element's.
struct tile_starts {
  const uint64_t *starts;
  uint64_t base;
  uint32_t in_range;  // elements of the tile
  uint32_t b0, b1;    // the wave's blocks (at most 32)
  uint32_t bound;     // lane i: the starts before block b0 + i (search)

  __device__ __forceinline__ tile_starts(const uint64_t *offsets, uint64_t lo, uint64_t base_, uint32_t in_range_,
                                         uint32_t bound_ = 0)
      : starts(offsets + lo), base(base_), in_range(in_range_), bound(bound_) {
    const uint32_t waves = blockDim.x >> 6;
    const uint32_t blocks = (in_range + 63) / 64;
    const uint32_t each = (blocks + waves - 1) / waves;
    b0 = min((threadIdx.x >> 6) * each, blocks);
    b1 = min(b0 + each, blocks);
  }

  __device__ __forceinline__ void search(uint32_t count) {
    if (b1 - b0 <= 2) {  // a few rounds of the whole wave each
      bound = count;
      for (uint32_t k = 0; k <= b1 - b0; ++k) {
        const uint32_t x = static_cast<uint32_t>(wave_lower_bound(starts, count, base + (b0 + k) * 64ull));
        if ((threadIdx.x & 63) == k) bound = x;
      }
      return;
    }
    const uint64_t key = base + (b0 + (threadIdx.x & 63)) * 64ull;
    uint32_t l = 0, h = count;
    while (l < h) {
      const uint32_t mid = l + (h - l) / 2;
      if (starts[mid] < key)
        l = mid + 1;
      else
        h = mid;
    }
    bound = l;
  }

  // f(e, i, found) for the elements e of the blocks in which segments start, by
  // whole waves: found, if a segment starts at e, with the last one that does,
  // lo + i (the only one of them that can hold elements).
  template <class F>
  __device__ __forceinline__ void for_each(F f) const {
    for (uint32_t b = b0; b < b1; ++b) {
      const uint32_t first = wave::read_lane(bound, static_cast<int>(b - b0));
      const uint32_t last = wave::read_lane(bound, static_cast<int>(b - b0) + 1);
      if (last <= first) continue;
      const uint32_t e = b * 64 + (threadIdx.x & 63);
      // Runs: from one start to the next other one by searches of the whole
      // wave, up to four of them; all starts of the block by lane if more (in
      // every block, 2^20 elements in 10 million segments took 49 -> 71 us).
      uint32_t pos = first, at = 0;
      bool found = false;
      if (last - first > run_starts) {
        for (int hop = 0; hop < 4 && pos < last; ++hop) {
          const uint64_t key = starts[pos];
          const uint32_t rest = static_cast<uint32_t>(
              wave_partition_point(last - pos, [&](uint64_t i) { return starts[pos + i] <= key; }));
          pos += rest ? rest : 1;
          if (base + e == key) {
            found = e < in_range;
            at = pos - 1;
          }
        }
      }
      if (pos < last) {
        uint32_t l = first, h = last;
        while (l < h) {
          const uint32_t mid = l + (h - l) / 2;
          if (starts[mid] <= base + e)
            l = mid + 1;
          else
            h = mid;
        }
        at = l - 1;
        found = e < in_range && l > first && starts[l - 1] == base + e;
      }
      f(e, at, found);
    }
  }

  // The head bits of the blocks in which segments start.
  __device__ __forceinline__ void mark(uint32_t *s_heads) const {
    for_each([&](uint32_t e, uint32_t, bool found) {
      const uint64_t bits = wave::ballot(found);
      if ((e & 31u) == 0) s_heads[e >> 5] = static_cast<uint32_t>(bits >> (e & 32u));
    });
  }
};

// The segments whose start lies in [first, last) (all from the first one on
// when to_end): found by the work-group's first and last wave, returned to
// all through s_range.
__device__ __forceinline__ void find_segments(const uint64_t *offsets, uint64_t num_segments, uint64_t first,
                                              uint64_t last, bool to_end, uint64_t (&s_range)[2]) {
  const int w = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  if (w == 0) {
    const uint64_t lo = wave_lower_bound(offsets, num_segments, first);
    if (lane == 0) s_range[0] = lo;
  }
  if (w == static_cast<int>(blockDim.x >> 6) - 1) {
    const uint64_t hi = to_end ? num_segments : wave_lower_bound(offsets, num_segments, last);
    if (lane == 0) s_range[1] = hi;
  }
}

// tile_seg[t] = the first segment that starts at or after tile t's first
// element (num_segments for t == num_tiles).  A work-group narrows the
// offsets to those of its 256 tiles, then every work-item searches its own
// (in LDS where they fit): no step grows with a segment's length.  (One
// work-item per segment writing the segment's tiles took 17 us for 48
// segments of 250 tiles.)
constexpr uint32_t table_stage = 2048;  // offsets held in LDS
__global__ __launch_bounds__(256) void tile_table_kernel(const uint64_t *__restrict__ offsets, uint64_t num_segments,
                                                         uint64_t tile_elems, uint32_t num_tiles, uint32_t *tile_seg) {
  __shared__ uint64_t s_off[table_stage];
  __shared__ uint64_t s_range[2];
  const uint64_t t0 = static_cast<uint64_t>(blockIdx.x) * 256;
  uint64_t first = 0, count = num_segments;
  if (num_segments > table_stage) {
    find_segments(offsets, num_segments, t0 * tile_elems, (t0 + 255) * tile_elems, false, s_range);
    __syncthreads();
    first = s_range[0];
    count = s_range[1] > first ? s_range[1] - first : 0;
  }
  const bool staged = count <= table_stage;
  if (staged) {
    for (uint32_t i = threadIdx.x; i < count; i += 256) s_off[i] = offsets[first + i];
    __syncthreads();
  }
  const uint64_t t = t0 + threadIdx.x;
  if (t > num_tiles) return;
  const uint64_t key = t * tile_elems;
  uint64_t lo = 0, hi = count;
  while (lo < hi) {
    const uint64_t mid = lo + (hi - lo) / 2;
    if ((staged ? s_off[mid] : offsets[first + mid]) < key)
      lo = mid + 1;
    else
      hi = mid;
  }
  lo = t == num_tiles ? num_segments : first + lo;
  tile_seg[t] = static_cast<uint32_t>(lo);
}

// The same table written by the segments: segment s is the last to start
// before every tile boundary in (offsets[s], offsets[s + 1]].  One round trip
// where the search above takes five or more, but it reads all offsets.  A
// segment of more than serial_tiles tiles is written by 16 lanes, one of more
// than shared_tiles by the whole work-group (by the whole group from 9 tiles
// on, 120M int32 in 3977 segments took 93 us, 87 us so;
// 30M int64 in 1000 55 and 49 us).
__global__ __launch_bounds__(256) void tile_scatter_kernel(const uint64_t *__restrict__ offsets, uint64_t num_segments,
                                                           uint64_t tile_elems, uint32_t num_tiles,
                                                           uint32_t *tile_seg) {
  constexpr uint32_t serial_tiles = 4;
  constexpr uint32_t shared_tiles = 512;
  __shared__ uint32_t s_count[2];  // segments for 16 lanes, from slot 0 up; for the group, from 255 down
  __shared__ uint32_t s_seg[256];
  __shared__ uint32_t s_first[256];
  __shared__ uint32_t s_last[256];
  if (threadIdx.x < 2) s_count[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t s = blockIdx.x * 256ull + threadIdx.x;
  if (s < num_segments) {
    const uint64_t b = offsets[s] / tile_elems, e = offsets[s + 1] / tile_elems;
    const uint32_t first = static_cast<uint32_t>(min(b + 1, static_cast<uint64_t>(num_tiles)));
    const uint32_t last = static_cast<uint32_t>(min(e + 1, static_cast<uint64_t>(num_tiles)));  // exclusive
    if (last > first + serial_tiles) {
      const bool whole = last - first > shared_tiles;
      const uint32_t place = atomicAdd(&s_count[whole ? 1 : 0], 1u);
      const uint32_t slot = whole ? 255u - place : place;
      s_seg[slot] = static_cast<uint32_t>(s) + 1;
      s_first[slot] = first;
      s_last[slot] = last;
    } else {
      for (uint32_t t = first; t < last; ++t) tile_seg[t] = static_cast<uint32_t>(s) + 1;
    }
  }
  if (s == 0) {
    tile_seg[0] = 0;
    tile_seg[num_tiles] = static_cast<uint32_t>(num_segments);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x >> 4; i < s_count[0]; i += 16)
    for (uint32_t t = s_first[i] + (threadIdx.x & 15u); t < s_last[i]; t += 16) tile_seg[t] = s_seg[i];
  for (uint32_t i = 256u - s_count[1]; i < 256u; ++i)
    for (uint32_t t = s_first[i] + threadIdx.x; t < s_last[i]; t += 256) tile_seg[t] = s_seg[i];
}

// The head bitmap of the scans: bit b for every segment start b < total (the
// start of an empty segment is that of the next one that is not empty).  The
// starts and the words are merged, a word behind the starts in it, and every
// work-group takes `part` of that order, a start counting 1 and a word
// word_weight: the work does not depend on where the empty segments are (by
// words alone, 10 million in one place of 2^23 elements took 11.7 ms).  A group
// marks the words that end in its part in LDS and writes them once: the bitmap
// needs no clearing and no global atomics.  (A fill, then one global atomicOr
// per segment: 2^26 elements in 13.4 million segments took 450 us of 558.)
constexpr uint32_t word_weight = 8;
__global__ __launch_bounds__(256) void head_bitmap_kernel(const uint64_t *__restrict__ offsets, uint64_t num_segments,
                                                          uint64_t total, uint64_t head_words, uint32_t part,
                                                          uint32_t *heads) {
  extern __shared__ uint32_t s_words[];  // part / word_weight
  __shared__ uint64_t s_start[2];  // first start of the group's part, and of the next
  __shared__ uint32_t s_deep;
  const uint64_t all = num_segments + head_words * word_weight;
  const uint64_t d0 = static_cast<uint64_t>(blockIdx.x) * part;
  const uint64_t d1 = min(d0 + part, all);
  const uint32_t tid = threadIdx.x;
  auto word_of = [&](uint64_t i) { return clamp_off(offsets, i, total) >> 5; };
  if (tid < 64 || tid >= 192) {
    const uint64_t d = tid < 64 ? d0 : d1;
    const uint64_t i = wave_partition_point(num_segments, [&](uint64_t i) { return i + word_of(i) * word_weight < d; });
    if ((tid & 63) == 0) s_start[tid < 64 ? 0 : 1] = i;
  }
  for (uint32_t i = tid; i < part / word_weight; i += 256) s_words[i] = 0;
  if (tid == 0) s_deep = 0;
  __syncthreads();
  const uint64_t i0 = s_start[0], i1 = s_start[1];
  // the words before the part are those whose weight is left of d0
  const uint64_t w0 = min(head_words, (d0 > i0 ? d0 - i0 : 0) / word_weight);
  const uint64_t w1 = min(head_words, (d1 > i1 ? d1 - i1 : 0) / word_weight);
  if (w1 <= w0) return;  // a part of a run of empty segments
  const uint32_t words = static_cast<uint32_t>(min(w1 - w0, static_cast<uint64_t>(part / word_weight)));
  const uint64_t base = w0 << 5;
  const uint64_t end = min(static_cast<uint64_t>(words) << 5, total > base ? total - base : 0);
  auto mark = [&](uint64_t b) { mark_head(s_words, b - base < end ? static_cast<uint32_t>(b - base) : no_head); };
  // The first word can hold starts of the parts before, too: the last 256 of
  // them, and if those all lie in it (or at the end of the input in it),
  // whatever there is, bit by bit (below).
  if (tid < i0) {
    const uint64_t b = offsets[i0 - 1 - tid];
    mark(b);
    if (tid == 255 && min(b, total) >> 5 == w0) s_deep = 1;
  }
#pragma unroll 8
  for (uint64_t i = i0 + tid; i < i1; i += 256) mark(offsets[i]);
  __syncthreads();
  if (s_deep) {
    // From the word's first start to its next other one, by searches of a whole
    // wave, unless there are more than four or no run.
    const bool run = i0 > run_starts && min(offsets[i0 - run_starts - 1], total) >> 5 == w0;
    if (tid == 0) s_start[0] = 0;
    if (run && tid < 64) {
      uint64_t pos = wave_lower_bound(offsets, i0, base);
      for (int hop = 0; hop < 4 && pos < i0; ++hop) {
        const uint64_t key = offsets[pos];
        const uint64_t rest = wave_partition_point(i0 - pos, [&](uint64_t i) { return offsets[pos + i] <= key; });
        pos += rest ? rest : 1;
        if (tid == 0 && key >= base && key - base < 32 && key < total) atomicOr(&s_words[0], 1u << (key - base));
      }
      if (tid == 0) s_start[0] = pos;
    }
    __syncthreads();
    if (s_start[0] < i0 && tid < 32) {
      const uint64_t key = base + tid;
      uint64_t lo = 0, hi = i0;
      while (lo < hi) {
        const uint64_t mid = lo + (hi - lo) / 2;
        if (offsets[mid] < key)
          lo = mid + 1;
        else
          hi = mid;
      }
      if (lo < i0 && offsets[lo] == key && key < total) atomicOr(&s_words[0], 1u << tid);
    }
    __syncthreads();
  }
  for (uint32_t i = tid; i < words; i += 256) heads[w0 + i] = s_words[i];
}

// 32-bit words of a reduction tile's head bits, rounded up so that the values
// behind them are 16-byte aligned.
__host__ __device__ constexpr uint32_t reduce_head_words(uint32_t tile_elems) { return ((tile_elems >> 5) + 3u) & ~3u; }

// threadIdx.x through an empty asm statement: a value the compiler cannot
// move, so what is derived from it inside a loop stays inside the loop.
__device__ __forceinline__ int loop_local_thread_index() {
  int t = static_cast<int>(threadIdx.x);
  asm volatile("" : "+v"(t));
  return t;
}

// Head bits of a work-item's R row vectors from the tile's LDS bitmap, all in
// one word: bit r * VEC + k = element k of row r starts a segment.  VEC
// consecutive bits never straddle a bitmap word (VEC divides 32).
template <int R, int VEC>
__device__ __forceinline__ uint32_t row_head_bits(const uint32_t *s_heads, int tid, int B) {
  static_assert(R * VEC <= 32, "head bits of a work-item must fit one word");
  uint32_t fm = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t pos = static_cast<uint32_t>(r * B + tid) * VEC;
    fm |= ((s_heads[pos >> 5] >> (pos & 31)) & ((1u << VEC) - 1u)) << (r * VEC);
  }
  return fm;
}

// Wave scans of the (head flag, total) pairs of each row, after the
// work-item-local scans.  Lane 63 leaves the wave's row total in
// s_tf / s_tv[r * nw + w]; every work-item folds its wave-exclusive prefix
// into the row's elements up to the row's first segment start and returns
// bit r set when a segment starts in an earlier lane of row r (the elements
// then hold their full in-segment fold already).  Folding at once keeps one
// bit per row live instead of a (flag, value) pair.
template <class Op, int R, int VEC, class W>
__device__ __forceinline__ uint32_t fold_wave_prefixes(uint32_t fm, W (&v)[R][VEC], uint32_t *s_tf, W *s_tv,
                                                       int nw, int w, int lane) {
  const W id = Op::identity();
  uint32_t xcut = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t rowf = (fm >> (r * VEC)) & ((1u << VEC) - 1u);
    uint32_t tf = rowf != 0u;
    W tv = v[r][VEC - 1];
    wave_pair_scan<Op>(tf, tv);
    if (lane == 63) {
      s_tf[r * nw + w] = tf;
      s_tv[r * nw + w] = tv;
    }
    const uint32_t ef = wave::dpp<wave::wave_shr1, 0xf, 0xf>(0u, tf);
    const W ev = wave::dpp<wave::wave_shr1, 0xf, 0xf>(id, tv);
    xcut |= ef << r;
#pragma unroll
    for (int k = 0; k < VEC; ++k)
      if ((rowf & ((2u << k) - 1u)) == 0u) v[r][k] = Op::apply(ev, v[r][k]);
  }
  return xcut;
}

// MARK: the tile marks its segment starts from the offsets itself instead of
// reading the bitmap (small inputs: one launch instead of two).
// RUNS: more segments than max_few_segments.
template <class T, class Op, int R, bool MARK, bool RUNS = false>
__global__ __launch_bounds__(1024) void segmented_kernel(params<T> p) {
  using W = typename elem_traits<T>::work;
  using SIO = seg_status<W>;
  constexpr int VEC = 16 / sizeof(T);
  const int B = blockDim.x;
  const int nw = B >> 6;
  const uint64_t tile_elems = static_cast<uint64_t>(B) * R * VEC;
  const W id = Op::identity();

  extern __shared__ uint32_t s_heads[];  // tile_elems + 1 bits, in 2 x blockDim.x words
  __shared__ uint32_t s_tile;
  __shared__ uint32_t s_tf[R * max_waves];  // per (row, wave): totals, then exclusive prefixes
  __shared__ W s_tv[R * max_waves];
  __shared__ uint32_t s_aggf;
  __shared__ W s_aggv;
  __shared__ uint32_t s_lbf[max_waves];
  __shared__ W s_lbv[max_waves];
  __shared__ int s_q[max_waves];
  __shared__ int s_give_up;
  __shared__ uint64_t s_invalid[max_waves];
  __shared__ uint64_t s_range[2];  // MARK
  const uint32_t head_words = static_cast<uint32_t>((tile_elems + 1 + 31) / 32);

  // A ticket is drawn only when the work-group is ready to work on the
  // tile: every later tile's look-back waits for this tile's aggregate, so a
  // ticket held while the group is busy with another tile stalls the whole
  // chain (drawing one tile ahead made the 65,536-segment int64 scan ~3x
  // slower on MI355X).
  for (;;) {
    // The work-item's indices are re-derived in every iteration, so that the
    // per-row addresses and bit positions computed from them are too: hoisted
    // out of the loop they held ~60 VGPRs for the whole kernel and made
    // 8-row tiles spill.
    const int tid = loop_local_thread_index();
    const int w = tid >> 6;
    const int lane = tid & 63;
    __syncthreads();  // LDS of the previous tile is free again
    if (tid == 0)
      s_tile = __hip_atomic_fetch_add(&p.sync->tile_counter, 1u, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT) -
               p.ticket_base;
    __syncthreads();
    const uint32_t tile = s_tile;
    if (tile >= p.num_tiles) return;  // queue drained

    const uint64_t base = static_cast<uint64_t>(tile) * tile_elems;

    // Full tiles and the partial last tile as separate compile-time paths:
    // with no join after the loads, each row waits only for its own load.
    const bool full = p.vec_io && (base + tile_elems <= p.total);
    auto tile_body = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      // elements of the tile in range, as a 32-bit offset inside the tile
      const uint32_t in_range =
          FULL ? static_cast<uint32_t>(tile_elems) : static_cast<uint32_t>(min(p.total - base, tile_elems));
      // Head bits of elements [base, base + tile_elems] (base is a multiple
      // of 32), loaded just before the tile's data in the same block, so that
      // waiting for them does not wait for the data (loads retire in order).
      // Both loads are unconditional (addresses clamped into the bitmap) and
      // the words are masked only where they go to LDS, with opaque masks: a
      // load under a branch, or a select the compiler turned back into one,
      // made it wait for every outstanding load, the tile's data included,
      // before the head bits could go to LDS.
      uint32_t hword0 = 0, hword1 = 0, hmask0 = 0, hmask1 = 0;
      if constexpr (MARK) {
        find_segments(p.offsets, p.num_segments, base, base + in_range, false, s_range);
      } else {
        const uint64_t last = p.head_words_total - 1;
        const uint64_t i0 = (base >> 5) + tid;
        const uint64_t i1 = i0 + B;
        hword0 = p.heads[i0 < last ? i0 : last];
        hword1 = p.heads[i1 < last ? i1 : last];
        hmask0 = (static_cast<uint32_t>(tid) < head_words && i0 <= last) ? ~0u : 0u;
        hmask1 = (static_cast<uint32_t>(tid + B) < head_words && i1 <= last) ? ~0u : 0u;
        asm volatile("" : "+v"(hmask0), "+v"(hmask1));
      }
      __builtin_amdgcn_sched_barrier(0);
      W v[R][VEC];
      u32x4 q[R];
      if constexpr (FULL) {
        const u32x4_a4 *src = reinterpret_cast<const u32x4_a4 *>(p.in + base);
#pragma unroll
        for (int r = 0; r < R; ++r) q[r] = src[r * B + tid];
        // Converted at once: the copies only rename registers (4- and 8-byte
        // elements), and the loaded vectors then never live beside v.
#pragma unroll
        for (int r = 0; r < R; ++r) {
          T tmp[VEC];
          __builtin_memcpy(tmp, &q[r], 16);
#pragma unroll
          for (int k = 0; k < VEC; ++k) v[r][k] = elem_traits<T>::to_work(tmp[k]);
        }
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int k = 0; k < VEC; ++k) {
            const uint32_t li = static_cast<uint32_t>(r * B + tid) * VEC + k;
            v[r][k] = (li < in_range) ? elem_traits<T>::to_work(p.in[base + li]) : id;
          }
      }
      // Unconditional stores (2 B words of LDS; the words past head_words
      // are zero): a store under a branch made the compiler wait for the
      // tile's data as well.
      s_heads[tid] = hword0 & hmask0;
      s_heads[tid + B] = hword1 & hmask1;
      __syncthreads();
      if constexpr (MARK) {
        const uint64_t lo = s_range[0], hi = s_range[1];
        if (RUNS && hi > lo && hi - lo > max_walk_segments(B)) {
          tile_starts starts(p.offsets, lo, base, in_range);
          starts.search(static_cast<uint32_t>(hi - lo));
          starts.mark(s_heads);
        } else {
#pragma unroll 4
          for (uint64_t i = lo + tid; i < hi; i += B) {
            const uint64_t b = p.offsets[i];
            mark_head(s_heads, b >= base && b - base < in_range ? static_cast<uint32_t>(b - base) : no_head);
          }
        }
        __syncthreads();
      }

      auto head_at = [&](uint64_t pos) -> uint32_t {
        return (s_heads[pos >> 5] >> (pos & 31)) & 1u;
      };

      // Head bits of the work-item's elements, all rows in one word: bit
      // r * VEC + k = element k of row r starts a segment.
      const uint32_t fm = row_head_bits<R, VEC>(s_heads, tid, B);

      // Work-item-local segmented scan of each row vector: an element that
      // starts a segment keeps its value, the others add the running value.
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 1; k < VEC; ++k)
          v[r][k] = ((fm >> (r * VEC + k)) & 1u) ? v[r][k] : Op::apply(v[r][k - 1], v[r][k]);

      // Wave scans of the row totals; the wave-exclusive prefix is folded into
      // the row's elements at once (up to the row's first segment start), so
      // only one bit per row stays live: bit r of xcut = a segment starts in
      // an earlier lane of this wave's row r.
      const uint32_t xcut = fold_wave_prefixes<Op, R, VEC>(fm, v, s_tf, s_tv, nw, w, lane);
      __syncthreads();
      // Wave 0 turns the (row, wave) totals into exclusive prefixes and
      // publishes the tile's aggregate at once.  A tile that contains a
      // segment start publishes it as its prefix: it is final for everything
      // after the tile.
      if (w == 0) {
        uint32_t af;
        W av;
        tile_pair_prefixes<Op, W>(R * nw, s_tf, s_tv, af, av);
        if (lane == 0) {
          s_aggf = af;
          s_aggv = av;
          if (tile == 0) {
            if (p.num_tiles > 1) SIO::publish(p.status, 0, p.epoch, st_prefix, af, av);
          } else {
            SIO::publish(p.status, tile, p.epoch, af ? st_prefix : st_aggregate, af, av);
          }
        }
      }
      __syncthreads();
      // s_tf / s_tv now hold the pairs before each (row, wave) inside the
      // tile, in element order; they are read again for the results (the
      // next tile rewrites them only after the barrier at the top of the loop).
      const uint32_t agg_f = s_aggf;
      const W agg_v = s_aggv;

      // Tile prefix: ordered look-back (one wave, or the whole work-group).
      uint32_t pf = 0;
      W pv = id;
      if (tile != 0) {
        // Only elements before the tile's first segment start need the
        // prefix; a tile that begins with a segment start needs none.
        if (!head_at(0) && !p.block_lookback) {
          // One wave looks back; its first lane publishes the tile's prefix.
          if (w == 0) {
            uint32_t ef;
            W ev;
            wait_own_stores();  // the aggregate is out before the first poll
            wave_pair_lookback<Op, W>(p.status, tile, p.epoch, p.sync, p.force_give_up != 0, ef, ev);
            if (lane == 0) {
              s_lbf[0] = ef;
              s_lbv[0] = ev;
              if (!agg_f && tile + 1 < p.num_tiles) {
                uint32_t of = agg_f;
                W ov = agg_v;
                combine<Op>(ef, ev, of, ov);
                SIO::publish(p.status, tile, p.epoch, st_prefix, of, ov);
              }
            }
          }
          __syncthreads();
          pf = s_lbf[0];
          pv = s_lbv[0];
        } else if (!head_at(0)) {
          // thread t polls tile (base_t - (B - 1 - t)); thread B-1 = nearest.
          int64_t wbase = static_cast<int64_t>(tile) - 1;
          uint32_t ef = 0;  // accumulated prefix of tiles nearer than the window
          W ev = id;
          lookback_wait wait;
          wait.begin();
          bool give_up = p.force_give_up != 0;  // uniform across the work-group
          if (give_up && tid == 0) report_trip(p.sync);
          for (;;) {
            const int64_t j = wbase - (B - 1 - tid);
            uint32_t lf = 0;
            W lv = id;
            int q;
            for (;;) {
              uint32_t st = st_prefix;
              lf = 0;
              lv = id;
              if (j >= 0) st = SIO::read(p.status, static_cast<uint32_t>(j), p.epoch, lf, lv);
              if (give_up) st = st_prefix;
              const bool term = (st == st_prefix) || (st == st_aggregate && lf);
              const uint64_t tm = wave::ballot(term);
              const uint64_t im = wave::ballot(st == st_invalid);
              if (lane == 0) {
                s_q[w] = tm ? (w * 64 + 63 - __builtin_clzll(tm)) : -1;
                s_invalid[w] = im;
              }
              __syncthreads();
              q = -1;
              for (int ww = nw - 1; ww >= 0; --ww)
                if (s_q[ww] >= 0) {
                  q = s_q[ww];
                  break;
                }
              bool bad = false;
              for (int ww = 0; ww < nw; ++ww) {
                const int lo = ww * 64;
                uint64_t need;
                if (q <= lo) need = ~0ull;
                else if (q > lo + 63) need = 0;
                else need = ~0ull << (q - lo);
                bad |= (s_invalid[ww] & need) != 0;
              }
              __syncthreads();
              if (!bad) break;
              // Every work-item backs off; work-item 0's clock decides for all.
              const bool late = wait.failed_round();
              if (tid == 0) {
                s_give_up = late ? 1 : 0;
                if (late) report_trip(p.sync);
              }
              __syncthreads();
              give_up = s_give_up != 0;
            }
            // Fold window tiles [q .. B-1] in tile order.
            uint32_t xf2 = (tid >= q) ? lf : 0;
            W xv2 = (tid >= q) ? lv : id;
            wave_pair_scan<Op>(xf2, xv2);
            if (lane == 63) {
              s_lbf[w] = xf2;
              s_lbv[w] = xv2;
            }
            __syncthreads();
            uint32_t wf = 0;
            W wv = id;
            for (int ww = 0; ww < nw; ++ww) {
              uint32_t yf = s_lbf[ww];
              W yv = s_lbv[ww];
              combine<Op>(wf, wv, yf, yv);
              wf = yf;
              wv = yv;
            }
            __syncthreads();
            // window (earlier) . accumulated (later)
            combine<Op>(wf, wv, ef, ev);
            if (q >= 0) break;
            wbase -= B;
          }
          pf = ef;
          pv = ev;
          if (tid == 0 && !agg_f && tile + 1 < p.num_tiles) {
            uint32_t of = agg_f;
            W ov = agg_v;
            combine<Op>(pf, pv, of, ov);
            SIO::publish(p.status, tile, p.epoch, st_prefix, of, ov);
          }
        }
      }

      // Results: the elements already hold the fold from the start of their
      // wave's row (or of their segment); the rest is P = tile prefix . before
      // (row r, wave w), cut off by a segment start in an earlier lane or
      // among elements 0..k of the vector.
      (void)pf;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t bfr = s_tf[r * nw + w];
        const W bvr = s_tv[r * nw + w];
        const W P = bfr ? bvr : Op::apply(pv, bvr);
        const uint32_t rowf = (fm >> (r * VEC)) & ((1u << VEC) - 1u);
        const bool wcut = (xcut >> r) & 1u;
        W o[VEC];
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
          const bool cut = wcut || (rowf & ((2u << k) - 1u)) != 0u;
          o[k] = cut ? v[r][k] : Op::apply(P, v[r][k]);
        }
        if constexpr (FULL) {
          T ot[VEC];
#pragma unroll
          for (int k = 0; k < VEC; ++k) ot[k] = static_cast<T>(o[k]);
          u32x4 qv;
          __builtin_memcpy(&qv, ot, 16);
          reinterpret_cast<u32x4_a4 *>(p.out + base)[r * B + tid] = qv;
        } else {
#pragma unroll
          for (int k = 0; k < VEC; ++k) {
            const uint32_t li = static_cast<uint32_t>(r * B + tid) * VEC + k;
            if (li < in_range) p.out[base + li] = static_cast<T>(o[k]);
          }
        }
      }
    };
    if (full)
      tile_body(std::true_type{});
    else
      tile_body(std::false_type{});
  }
}

// --------------------------------------------------------------------------
// Segmented reduction without a look-back.
//
// A reduction needs only each segment's total, so tiles do not wait for
// each other.  A tile owns the segments that start in it (empty ones too; the
// last tile also those at the end).  Every tile (one work-group, launched in
// any order) runs the same in-tile (head flag, value) scan as the scan
// kernel, keeps the scanned values in LDS, and one work-item per owned
// segment then
//   - writes op(init, value at the segment's last element) if the segment
//     ends inside the tile, init if it is empty;
// while the tile stores
//   - head_part[tile]: the fold of the elements before its first segment
//     start (the whole tile if it has none: such a tile takes a plain fold);
//   - tail_part[tile], tail_seg[tile]: the fold from its last segment start
//     to the tile's end and that segment's index, when the segment continues
//     into the next tile (tail_seg = no_segment otherwise).
// A fix-up kernel then gives every segment that spans tiles tb < ... <= tl
// the total tail_part[tb] . head_part[tb+1] . ... . head_part[tl]
// (deterministic: the tree depends on the sizes only).
//
// Reading the values at the segments' ends from LDS, one work-item per
// segment, keeps the results coalesced and costs no search: a binary search
// for the segment of every last element ran in almost every step of the
// unrolled rows once segments are short (2^26 fp32 in 1.3 million segments: 186
// -> 67 us).  A tile in which at most three segments start takes plain folds
// without any scan (2^28 fp32 in 40 segments: 514 -> 180 us with the fix-up
// below, in 89,479 segments 184 -> 179 us).
// --------------------------------------------------------------------------
constexpr uint32_t no_segment = 0xffffffffu;

// Where the segments of such a run (those from a multiple of empty_run up to
// the next one) all start in one tile, the fix-up kernel writes init to its
// empty ones: empty_runs runs a work-group, so that millions of empty segments
// in one place are spread over the chip.
constexpr uint32_t empty_run = 8192;
constexpr uint32_t empty_runs = 2;
static_assert(2 * empty_run <= max_walk_segments(64) && 16 % empty_runs == 0, "a tile that does not walk its segments holds a whole run");

template <class W>
struct reduce_parts {
  W *head;
  W *tail;
  uint32_t *tail_seg;
};

using constant_u32 = const __attribute__((address_space(4))) uint32_t *;
using constant_u64 = const __attribute__((address_space(4))) uint64_t *;

// Op for folds in which some lanes or accumulators hold no element but the
// identity, to the right of others' elements too: it leaves those alone.  For
// min and max of floating-point numbers the identity is none there:
// max(NaN, -inf) is -inf, and the NaN would be lost.
template <class Op, class W>
struct skip_identity {
  static constexpr bool needed =
      std::is_floating_point_v<W> && (Op::id == ops::op_min || Op::id == ops::op_max);
  __device__ static W identity() { return Op::identity(); }
  __device__ static W apply(W a, W b) {
    if constexpr (needed)
      return b == Op::identity() ? a : Op::apply(a, b);
    else
      return Op::apply(a, b);
  }
};

// The fold of a wave's lanes, some of which may hold the identity; uniform.
// Every fold by Op is one of the folded values, so only the identity itself
// can be wrong: the longer chain of skip_identity follows then alone.
template <class Op, class W>
__device__ __forceinline__ W fold_lanes(W x) {
  W y = wave::reduce_full<Op>(x);
  if constexpr (skip_identity<Op, W>::needed) {
    if (y == Op::identity() && wave::ballot(!(x == Op::identity()))) y = wave::reduce_full<skip_identity<Op, W>>(x);
  }
  return y;
}

// RUNS: more segments than max_few_segments (a kernel of its own: with that code
// in it the other one takes 72 -> 80 us for 120M fp32 in 40 segments, 512 x 2
// tiles).
// At most 64 registers for 2 and 4 rows: two 1024-wide groups on a CU.
template <class T, class Op, int R, bool RUNS>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(R == 8 ? 4 : 8))) void segmented_reduce_kernel(params<T> p,
                                                                reduce_parts<typename elem_traits<T>::work> parts) {
  using W = typename elem_traits<T>::work;
  constexpr int VEC = 16 / sizeof(T);
  const int tid = threadIdx.x;
  const int B = blockDim.x;
  const int nw = B >> 6;
  const int w = tid >> 6;
  const int lane = tid & 63;
  const uint32_t tile_elems = static_cast<uint32_t>(B * R * VEC);
  const W id = Op::identity();

  extern __shared__ uint32_t s_heads[];     // tile_elems bits, then tile_elems values
  W *s_val = reinterpret_cast<W *>(s_heads + reduce_head_words(tile_elems));
  __shared__ uint32_t s_tf[R * max_waves];  // per (row, wave): totals, then exclusive prefixes
  __shared__ W s_tv[R * max_waves];
  __shared__ uint64_t s_range[2];
  // offsets[lo .. lo + off_cap), which are read twice, relative to the tile
  // (beyond its end: in_range + 1)
  constexpr uint32_t off_cap = 1024;
  __shared__ uint32_t s_off[off_cap];
  constexpr uint32_t max_pieces = 4;
  __shared__ W s_piece[max_pieces][max_waves];

  const uint32_t tile = blockIdx.x;
  if (tile >= p.num_tiles) return;
  const uint64_t base = static_cast<uint64_t>(tile) * tile_elems;
  const uint32_t in_range = static_cast<uint32_t>(min(p.total - base, static_cast<uint64_t>(tile_elems)));
  const bool last = tile + 1 == p.num_tiles;
  if (!p.tile_seg) find_segments(p.offsets, p.num_segments, base, base + in_range, last, s_range);

  const bool full = p.vec_io && in_range == tile_elems;
  W v[R][VEC];
  u32x4 q[R];
  if (full) {
    const u32x4_a4 *src = reinterpret_cast<const u32x4_a4 *>(p.in + base);
#pragma unroll
    for (int r = 0; r < R; ++r) q[r] = src[r * B + tid];
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        const uint32_t i = static_cast<uint32_t>(r * B + tid) * VEC + k;
        v[r][k] = (i < in_range) ? elem_traits<T>::to_work(p.in[base + i]) : id;
      }
  }
  // Scalar loads, which do not wait for the data as vector loads would (those
  // return in order); nothing writes what they read while the kernel runs.
  uint32_t lo, hi;
  if (p.tile_seg) {
    const constant_u32 table = (constant_u32)p.tile_seg;
    lo = table[tile];
    hi = table[tile + 1];
    // malformed offsets can leave entries of the table unwritten
    lo = min(lo, static_cast<uint32_t>(p.num_segments));
    hi = min(hi, static_cast<uint32_t>(p.num_segments));
  } else {
    __syncthreads();
    lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(s_range[0]));
    hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(s_range[1]));
  }
  const uint32_t owned = hi > lo ? hi - lo : 0;  // segments lo .. lo + owned - 1
  // The start of segment lo + i in the tile; in_range + 1 beyond its end.
  auto in_tile = [&](uint64_t o) -> uint32_t {
    o = min(o, p.total);
    return o <= base ? 0u : static_cast<uint32_t>(min(o - base, static_cast<uint64_t>(in_range) + 1));
  };
  auto load_off = [&](uint32_t i) { return in_tile(p.offsets[static_cast<uint64_t>(lo) + i]); };
  const bool off_in_lds = owned + 1 <= off_cap;
  // (a tile cut short by the end of the input has only the identity in some lanes)
  constexpr bool ordered = skip_identity<Op, W>::needed;
  const bool few = owned < max_pieces && (!ordered || in_range == tile_elems);
  if (!few) {
    for (uint32_t i = tid; i < (tile_elems >> 5); i += B) s_heads[i] = 0;
    if (off_in_lds)
      for (uint32_t i = tid; i <= owned; i += B) s_off[i] = load_off(i);
  }
  auto off = [&](uint32_t i) { return off_in_lds ? s_off[i] : load_off(i); };
  // Few segments start in the tile: up to max_pieces plain folds, of the
  // elements before the first start, between two starts, and after the last.
  uint32_t start[max_pieces];
  if (few) {
    const constant_u64 offsets = (constant_u64)p.offsets;
    uint64_t o[max_pieces];
#pragma unroll
    for (uint32_t j = 0; j < max_pieces; ++j) o[j] = offsets[min(static_cast<uint64_t>(lo) + j, p.num_segments)];
#pragma unroll
    for (uint32_t j = 0; j < max_pieces; ++j) start[j] = j <= owned ? in_tile(o[j]) : in_range + 1;
  }
  if (full) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      T tmp[VEC];
      __builtin_memcpy(tmp, &q[r], 16);
#pragma unroll
      for (int k = 0; k < VEC; ++k) v[r][k] = elem_traits<T>::to_work(tmp[k]);
    }
  }
  if (few) {
    auto piece_of = [&](uint32_t i) {
      uint32_t piece = 0;
#pragma unroll
      for (uint32_t j = 0; j + 1 < max_pieces; ++j) piece += (j < owned && i >= start[j]) ? 1u : 0u;
      return piece;
    };
    W acc[max_pieces];
#pragma unroll
    for (uint32_t j = 0; j < max_pieces; ++j) acc[j] = id;
    const uint32_t wave_first = __builtin_amdgcn_readfirstlane(w) * 64u * VEC;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      // a wave's 64 vectors of a row lie in one piece unless a segment starts there
      const uint32_t c = r * B * VEC + wave_first;
      const uint32_t piece = piece_of(c);
      if (piece == piece_of(c + 64 * VEC - 1)) {
        W x = v[r][0];
#pragma unroll
        for (int k = 1; k < VEC; ++k) x = Op::apply(x, v[r][k]);
#pragma unroll
        for (uint32_t j = 0; j < max_pieces; ++j)
          if (piece == j) acc[j] = Op::apply(acc[j], x);
      } else {
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
          const uint32_t mine = piece_of(c + lane * VEC + k);
#pragma unroll
          for (uint32_t j = 0; j < max_pieces; ++j) {
            if constexpr (ordered)
              acc[j] = mine == j ? Op::apply(acc[j], v[r][k]) : acc[j];
            else
              acc[j] = Op::apply(acc[j], mine == j ? v[r][k] : id);
          }
        }
      }
    }
#pragma unroll
    for (uint32_t j = 0; j < max_pieces; ++j) {
      if (j <= owned) {
        const W x = fold_lanes<Op>(acc[j]);
        if (lane == 0) s_piece[j][w] = x;
      }
    }
    __syncthreads();
    if (w == 0) {
      uint32_t tail_seg = no_segment;
#pragma unroll
      for (uint32_t j = 0; j < max_pieces; ++j) {
        if (j <= owned) {
          const W x = fold_lanes<Op>(lane < nw ? s_piece[j][lane] : id);
          if (j == 0) {
            if (lane == 0) parts.head[tile] = x;
          } else {
            const uint64_t s = static_cast<uint64_t>(lo) + j - 1;
            const uint32_t b = start[j > 0 ? j - 1 : 0], e = start[j];
            if (e > b && e > in_range) {
              tail_seg = static_cast<uint32_t>(s);
              if (lane == 0) parts.tail[tile] = x;
            } else if (lane == 0) {
              p.out[s] = static_cast<T>(e > b ? Op::apply(p.init, x) : p.init);
            }
          }
        }
      }
      if (lane == 0) parts.tail_seg[tile] = tail_seg;
    }
    return;
  }

  const bool walk = !RUNS || owned <= max_walk_segments(B);
  uint32_t bound = 0;
  __syncthreads();
  auto mark = [&](uint32_t b) { mark_head(s_heads, b < in_range ? b : no_head); };
  if (RUNS && !off_in_lds && walk) {
#pragma unroll 4
    for (uint32_t i = tid; i < owned; i += B) mark(load_off(i));
  } else if (walk) {
    for (uint32_t i = tid; i < owned; i += B) mark(off(i));
  } else {
    tile_starts starts(p.offsets, lo, base, in_range);
    starts.search(owned);
    starts.mark(s_heads);
    bound = starts.bound;
  }
  __syncthreads();

  const uint32_t fm = row_head_bits<R, VEC>(s_heads, tid, B);
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int k = 1; k < VEC; ++k)
      v[r][k] = ((fm >> (r * VEC + k)) & 1u) ? v[r][k] : Op::apply(v[r][k - 1], v[r][k]);

  const uint32_t xcut = fold_wave_prefixes<Op, R, VEC>(fm, v, s_tf, s_tv, nw, w, lane);
  __syncthreads();
  if (w == 0) {
    uint32_t af;
    W av;
    tile_pair_prefixes<Op, W>(R * nw, s_tf, s_tv, af, av);
    (void)af;
    (void)av;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    // The elements hold the fold from their wave's row start (or segment
    // start); Pv is the (row r, wave w) prefix inside the tile, cut off by
    // a segment start in an earlier lane or among elements 0..k.
    const uint32_t rowf = (fm >> (r * VEC)) & ((1u << VEC) - 1u);
    const bool wcut = (xcut >> r) & 1u;
    const W Pv = s_tv[r * nw + w];
    W o[VEC];
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
      const bool cut = wcut || (rowf & ((2u << k) - 1u)) != 0u;
      o[k] = cut ? v[r][k] : Op::apply(Pv, v[r][k]);
    }
    u32x4 qv;
    __builtin_memcpy(&qv, o, 16);
    reinterpret_cast<u32x4 *>(s_val)[r * B + tid] = qv;
  }
  __syncthreads();
  auto result = [&](uint32_t i, uint32_t b, uint32_t e) {
    const uint64_t s = static_cast<uint64_t>(lo) + i;
    if (e <= b)
      p.out[s] = static_cast<T>(p.init);
    else if (e <= in_range)
      p.out[s] = static_cast<T>(Op::apply(p.init, s_val[e - 1]));
  };
  if (RUNS && !off_in_lds) {
    // A tile that is not walked: the segments with elements, and the empty ones
    // outside of the runs that the fix-up kernel fills.
    uint32_t filled = owned, end = owned;
    if (!walk) {
      tile_starts(p.offsets, lo, base, in_range, bound).for_each([&](uint32_t, uint32_t i, bool found) {
        if (found) result(i, load_off(i), load_off(i + 1));
      });
      filled = (empty_run - lo % empty_run) % empty_run;  // from here on
      end = (hi - 1) / empty_run * empty_run - lo;        // up to here
    }
#pragma unroll 4
    for (uint32_t i = tid; i < filled; i += B) result(i, load_off(i), load_off(i + 1));
    for (uint32_t i = end + tid; i < owned; i += B) result(i, load_off(i), load_off(i + 1));
  } else {
    for (uint32_t i = tid; i < owned; i += B) result(i, off(i), off(i + 1));
  }
  if (tid == 0) {
    const uint32_t first = off(0);
    if (first > 0 && first <= in_range) parts.head[tile] = s_val[first - 1];
    const bool tail = off(owned) > in_range;
    if (tail) parts.tail[tile] = s_val[in_range - 1];
    parts.tail_seg[tile] = tail ? lo + owned - 1 : no_segment;
  }
}

// op(init, tail[tb] . head[tb+1] . ... . head[tl]) for every segment that
// continues from tile tb to tile tl > tb: one work-item per tile tb, a wave
// for a segment of more than serial_span tiles, the whole group above
// wave_span.  The work-groups past the first fix_groups fill the runs of empty
// segments.  (One work-item per segment and eight partials in flight: 18 us
// for 48 segments of 250 tiles, 3.1 ms for one segment of 65,536.)
template <class T, class Op>
__global__ __launch_bounds__(1024) void segmented_fixup_kernel(params<T> p,
                                                               reduce_parts<typename elem_traits<T>::work> parts,
                                                               uint64_t tile_elems, uint32_t fix_groups) {
  using W = typename elem_traits<T>::work;
  using Fold = skip_identity<Op, W>;
  constexpr uint32_t serial_span = 16;
  constexpr uint32_t wave_span = 1024;
  constexpr uint32_t max_list = 64;  // a group's tiles start at most 61 such segments
  __shared__ uint32_t s_count;
  __shared__ uint32_t s_tile[max_list];
  __shared__ uint32_t s_last[max_list];
  __shared__ W s_red[max_waves];
  const W id = Op::identity();
  const int w = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  if (blockIdx.x >= fix_groups) {
    const uint64_t first = (blockIdx.x - fix_groups) * static_cast<uint64_t>(empty_runs) * empty_run;
    if (threadIdx.x <= empty_runs) {
      const uint64_t s = first + threadIdx.x * empty_run;
      s_tile[threadIdx.x] =
          s < p.num_segments ? static_cast<uint32_t>(min(clamp_off(p.offsets, s, p.total) / tile_elems,
                                                         static_cast<uint64_t>(p.num_tiles - 1)))
                             : no_segment;
    }
    __syncthreads();
    constexpr uint32_t lanes = 1024 / empty_runs;  // work-items for a run
    const uint32_t j = threadIdx.x / lanes;
    if (s_tile[j] == no_segment || s_tile[j] != s_tile[j + 1]) return;
#pragma unroll 8
    for (uint32_t i = threadIdx.x % lanes; i < empty_run; i += lanes) {
      const uint64_t s = first + j * empty_run + i;
      const uint64_t b = p.offsets[s], e = p.offsets[s + 1];
      if (e <= b) p.out[s] = static_cast<T>(p.init);
    }
    return;
  }
  if (threadIdx.x == 0) s_count = 0;
  __syncthreads();
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t s = t + 1 < p.num_tiles ? parts.tail_seg[t] : no_segment;
  if (s < p.num_segments) {
    const uint64_t e = clamp_off(p.offsets, static_cast<uint64_t>(s) + 1, p.total);
    const uint32_t tl = e ? static_cast<uint32_t>((e - 1) / tile_elems) : 0;
    uint32_t slot = max_list;
    if (tl > t + serial_span) slot = atomicAdd(&s_count, 1u);
    if (slot < max_list) {
      s_tile[slot] = t;
      s_last[slot] = tl;
    } else if (tl > t) {
      W acc = parts.tail[t];
      uint32_t u = t + 1;
      for (; u + 4 <= tl + 1; u += 4) {
        W h[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) h[j] = parts.head[u + j];
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = Op::apply(acc, h[j]);
      }
      for (; u <= tl; ++u) acc = Op::apply(acc, parts.head[u]);
      p.out[s] = static_cast<T>(Op::apply(p.init, acc));
    }
  }
  __syncthreads();
  const uint32_t count = min(s_count, max_list);
  // `lanes` work-items fold head[tb + 1 .. tl], four partials in flight each.
  auto fold = [&](uint32_t tb, uint32_t tl, uint32_t me, uint32_t lanes) {
    W acc[4] = {id, id, id, id};
    uint64_t u = static_cast<uint64_t>(tb) + 1 + me;
    for (; u + 3ull * lanes <= tl; u += 4ull * lanes) {
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = Op::apply(acc[j], parts.head[u + static_cast<uint64_t>(j) * lanes]);
    }
    for (; u <= tl; u += lanes) acc[0] = Op::apply(acc[0], parts.head[u]);
    return fold_lanes<Op>(Fold::apply(Fold::apply(acc[0], acc[1]), Fold::apply(acc[2], acc[3])));
  };
  auto finish = [&](uint32_t tb, W rest) {
    p.out[parts.tail_seg[tb]] = static_cast<T>(Op::apply(p.init, Op::apply(parts.tail[tb], rest)));
  };
  for (uint32_t i = w; i < count; i += blockDim.x >> 6) {
    if (s_last[i] - s_tile[i] > wave_span) continue;
    const W x = fold(s_tile[i], s_last[i], lane, 64);
    if (lane == 0) finish(s_tile[i], x);
  }
  for (uint32_t i = 0; i < count; ++i) {
    if (s_last[i] - s_tile[i] <= wave_span) continue;
    W x = fold(s_tile[i], s_last[i], threadIdx.x, blockDim.x);
    __syncthreads();
    if (lane == 0) s_red[w] = x;
    __syncthreads();
    if (w == 0) {
      x = fold_lanes<Op>(lane < static_cast<int>(blockDim.x >> 6) ? s_red[lane] : id);
      if (lane == 0) finish(s_tile[i], x);
    }
  }
}

// --------------------------------------------------------------------------
// Host side
// --------------------------------------------------------------------------
// Default tile when the caller gives no configuration, by element count,
// element size and total bytes.  Read off timings on MI355X of every tile
// from 128 x 2 to 1024 x 8 at 2 x 10^4 .. 3 x 10^7 elements (4 and 8 bytes,
// segments of 50 and of 3000 elements and 40 segments), and above from the
// tuner's timing database:
//   scan:   n < 2^16: 256 x 2;  n < 2^20: 512 x 2 (8-byte: 1024 x 2);
//           < 12 MiB: 1024 x 2;  < 64 MiB: 1024 x 4;  n < 2^26: 512 x 8;
//           otherwise 1024 x 8
//   reduce: n < 2^16: 128 x 2;  n < 2^20: 256 x 2;  < 20 MiB: 1024 x 2;
//           < 48 MiB: 1024 x 4;  otherwise 256 x 4 (8-byte: 512 x 4), but
//           with one segment per 2^14 to 2^17 elements 1024 x 4 (the tiles are
//           then few enough for the segments to write their table: 60M int32
//           in 1000 segments 46.3 and 42.1 us, in 48 40.5 and 42.8 us, in
//           20000 42.4 and 51.6 us), and 512 x 2 from 320 MiB with at most one
//           per 2^14 (204M int32 in 300 segments 137.0 and 130.0 us, in 3977
//           140.1 and 134.7 us, in 100,000 139.0 and 158.1 us), 256 x 2 there
//           up to one per 2^12 (120M int32 in 20,000 segments 87.7 and 84.7 us,
//           300M int32 in 30,000 202.1 and 195.3 us, 150M fp64 in 15,000 207.5
//           and 199.4 us; 204M int32 in 60,000 137.3 and 142.8 us)
// 2-row scans of up to max_search_tiles tiles and reductions of as many
// tiles need one launch less, so the tiles grow with the input as long as
// they stay below that (2^20 fp32 scan: 8.5 us at 1024 x 2, 11.6 us at 512 x
// 8; 2^23 fp32 reduction: 11.9 us at 1024 x 4, 14.7 us at 1024 x 2).  Large
// scans take 8-row tiles (two 512-wide or one 1024-wide group per CU, 123
// VGPRs for int64); large reductions take 2- or 4-row tiles, which leave room for
// several groups per CU (the reduction's groups never wait for each other).
inline void default_tile(bool reduce, uint64_t total, uint64_t num_segments, int elem_bytes, uint32_t &wg,
                         int &rows) {
  const bool wide = elem_bytes == 8;
  const uint64_t mib = total * elem_bytes >> 20;
  if (total < (1ull << 20)) {
    rows = 2;
    if (total < (1ull << 16))
      wg = reduce ? 128 : 256;
    else
      wg = reduce ? 256 : (wide ? 1024 : 512);
  } else if (reduce) {
    rows = mib < 20 ? 2 : 4;
    wg = mib < 48 ? 1024 : (wide ? 512 : 256);
    const bool few = num_segments <= total >> 14;
    if (mib >= 320 && num_segments <= total >> 12) {
      wg = few ? 512 : 256;
      rows = 2;
    } else if (mib >= 48 && few && num_segments >= total >> 17) {
      wg = 1024;
    }
  } else {
    rows = mib < 12 ? 2 : mib < 64 ? 4 : 8;
    wg = (mib < 64 || total >= (1ull << 26)) ? 1024 : 512;
  }
}

// Tiles up to which a work-group finds its segments by itself: the launch of
// the kernel that does it for all tiles costs more (about 3.5 us) than the
// searches, which a few hundred resident groups overlap.
constexpr uint64_t max_search_tiles = 1024;
// Segments per tile up to which the segments write the tiles' table, and
// tiles per segment: 2^23 fp32 in 2797 segments 16.7 us written, 19.3 us
// searched; in 40 segments 20.6 and 17.5 us.
constexpr uint64_t max_scatter_segments = 16;
constexpr uint64_t max_scatter_tiles = 8;

// A segmented call with its scratch, ready to be enqueued any number of
// times (once by the calls, on every launch by a plan).
struct prepared {
  virtual ~prepared() = default;
  virtual acpp_status enqueue(hipStream_t stream) = 0;
  int device = 0;
};

template <class T, class Op>
struct call : prepared {
  using W = typename elem_traits<T>::work;
  static constexpr int VEC = 16 / sizeof(T);
  const char *name = "";
  params<T> p;
  bool reduce = false;
  bool mark = false;  // scans: segment starts are marked in the scan kernel
  uint32_t wg = 256;
  int rows = 8;
  uint32_t grid = 1;
  size_t lds = 0;
  uint64_t tile_elems = 0;
  uint32_t *table = nullptr;  // reductions
  reduce_parts<W> parts = {};
  uint32_t *heads = nullptr;  // scans
  uint64_t head_words = 0;
  void *region = nullptr;
  region_state *rs = nullptr;
  size_t region_used = 0;
  size_t region_cap = 0;
  uint32_t *trip_flag = nullptr;

  // Checks the configuration and obtains the scratch.  `stream`: where a new
  // sync region is cleared; NULL defers that to the first enqueue.
  acpp_status prepare(acpp_allocation_group *g, const hipStream_t *stream, const T *in, T *out,
                      const uint64_t *offsets, uint64_t num_segments, uint64_t total, W init, bool is_reduce,
                      const acpp_launch_config *cfg) {
    static_assert(sizeof(T) >= 4, "16-byte vector accesses at 4-byte alignment (u32x4_a4)");
    int cus = 0;
    acpp_status st = enter_device(g, &cus);
    if (st != ACPP_SUCCESS) return st;
    device = group_device(g);
    reduce = is_reduce;
    default_tile(reduce, total, num_segments, static_cast<int>(sizeof(T)), wg, rows);
    const uint32_t default_tile_rows = wg * static_cast<uint32_t>(rows);
    if (cfg && cfg->work_group_size) wg = cfg->work_group_size;
    if (!valid_work_group_size(wg))
      return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": bad work_group_size");
    // Large scans keep the default tile's size in a narrower group, up to 8
    // rows: the look-back chain grows with the tiles (14M int32 in 9471 segments,
    // 64 wide: 247 us with 4 rows, 138 us with 8; below 2^20 elements two rows
    // are better, 100,000 in 500 7.9 and 11.6 us).
    while (!reduce && total >= (1ull << 20) && rows < 8 && wg * static_cast<uint32_t>(rows) < default_tile_rows) rows *= 2;
    if (cfg && cfg->items_per_thread) rows = static_cast<int>(cfg->items_per_thread);
    if (rows != 2 && rows != 4 && rows != 8)
      return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": items_per_thread must be 2, 4 or 8");
    tile_elems = static_cast<uint64_t>(wg) * rows * VEC;
    const uint64_t num_tiles = std::max<uint64_t>(1, ceil_div(total, tile_elems));
    if (num_tiles >= (1ull << 31) || num_segments >= (1ull << 32))
      return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": problem too large");
    p.in = in;
    p.out = out;
    p.offsets = offsets;
    p.tile_seg = nullptr;
    p.heads = nullptr;
    p.head_words_total = 0;
    p.block_lookback = 0;
    p.force_give_up = 0;
    p.num_segments = num_segments;
    p.total = total;
    p.init = init;
    p.num_tiles = static_cast<uint32_t>(num_tiles);
    p.epoch = 0;
    p.ticket_base = 0;
    p.sync = nullptr;
    p.status = nullptr;
    return reduce ? prepare_reduce(g) : prepare_scan(g, stream, cus, cfg);
  }

  acpp_status prepare_reduce(acpp_allocation_group *g) {
    const uint64_t num_tiles = p.num_tiles;
    void *scratch = nullptr;
    acpp_status st = group_obtain(g, num_tiles * (2 * sizeof(W) + sizeof(uint32_t)), &scratch);
    if (st != ACPP_SUCCESS) return st;
    parts.head = static_cast<W *>(scratch);
    parts.tail = parts.head + num_tiles;
    parts.tail_seg = reinterpret_cast<uint32_t *>(parts.tail + num_tiles);
    if (num_tiles > max_search_tiles) {
      void *ts = nullptr;
      st = group_obtain(g, (num_tiles + 1) * sizeof(uint32_t), &ts);
      if (st != ACPP_SUCCESS) return st;
      table = static_cast<uint32_t *>(ts);
    }
    p.tile_seg = table;
    p.vec_io = (reinterpret_cast<uintptr_t>(p.in) & 3) == 0;
    grid = p.num_tiles;
    lds = reduce_head_words(static_cast<uint32_t>(tile_elems)) * 4 + tile_elems * sizeof(W);
    return ACPP_SUCCESS;
  }

  acpp_status prepare_scan(acpp_allocation_group *g, const hipStream_t *stream, int cus,
                           const acpp_launch_config *cfg) {
    const uint64_t num_tiles = p.num_tiles;
    acpp_status st;
    // the scan kernel stores 2 x wg words of head bits (>= the tile_elems + 1
    // bits it needs, since rows x 16-byte vector <= 32 elements)
    lds = std::max<size_t>(static_cast<size_t>((tile_elems + 1 + 31) / 32), 2 * static_cast<size_t>(wg)) * 4;
    // Small inputs (2-row tiles) mark their segment starts in the scan kernel.
    mark = rows == 2 && num_tiles <= max_search_tiles;
    if (!mark) {
      // Head bitmap over elements [0, total] plus one spare word.
      head_words = (p.total + 1 + 31) / 32 + 1;
      void *hb = nullptr;
      st = group_obtain(g, head_words * sizeof(uint32_t), &hb);
      if (st != ACPP_SUCCESS) return st;
      heads = static_cast<uint32_t *>(hb);
    }
    p.heads = heads;
    p.head_words_total = head_words;
    using SIO = seg_status<W>;
    static_assert(SIO::words <= seg_stride_words, "status slot too small");
    region_used = sizeof(sync_header) + num_tiles * seg_stride_words * sizeof(uint64_t);
    st = stream ? group_obtain_sync(g, region_used, *stream, &region, &region_cap, &rs)
                : group_obtain_sync_uncleared(g, region_used, &region, &region_cap, &rs);
    if (st != ACPP_SUCCESS) return st;
    trip_flag = host_trip_flag(device);
    p.block_lookback = (cfg && (cfg->flags & ACPP_VARIANT_BLOCK_LOOKBACK)) ? 1 : 0;
    p.force_give_up = (cfg && (cfg->flags & ACPP_VARIANT_FORCE_GIVE_UP)) ? 1 : 0;
    p.vec_io = ((reinterpret_cast<uintptr_t>(p.in) | reinterpret_cast<uintptr_t>(p.out)) & 3) == 0;
    p.sync = static_cast<sync_header *>(region);
    p.status = reinterpret_cast<uint64_t *>(static_cast<char *>(region) + sizeof(sync_header));

    // Persistent grid: one wave of resident work-groups, each drawing tiles
    // from the queue until it is empty.  With ACPP_VARIANT_TILE_PER_GROUP the
    // grid has one work-group per tile (the hardware dispatcher then keeps
    // the CUs full while groups wait in their look-back), still fed by the
    // same queue.  Every work-group draws one ticket past the last tile
    // before it exits; the ticket base counts those too.
    grid = static_cast<uint32_t>(num_tiles);
    if (cfg && (cfg->flags & ACPP_VARIANT_TILE_PER_GROUP)) return ACPP_SUCCESS;
    const uint32_t per_cu = cfg ? cfg->groups_per_cu : 0;
    return with_scan_kernel([&](auto kernel) -> acpp_status {
      int resident = 1;
      ACPP_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&resident, kernel, static_cast<int>(wg), lds));
      if (resident < 1) resident = 1;
      uint64_t cap = static_cast<uint64_t>(resident) * cus;
      if (per_cu) cap = std::min<uint64_t>(cap, static_cast<uint64_t>(per_cu) * cus);
      grid = static_cast<uint32_t>(std::min<uint64_t>(cap, num_tiles));
      return ACPP_SUCCESS;
    });
  }

  template <class F>
  acpp_status with_scan_kernel(F &&f) {
    if (mark && p.num_segments > max_few_segments(wg)) return f(segmented_kernel<T, Op, 2, true, true>);
    if (mark) return f(segmented_kernel<T, Op, 2, true>);
    if (rows == 2) return f(segmented_kernel<T, Op, 2, false>);
    if (rows == 4) return f(segmented_kernel<T, Op, 4, false>);
    return f(segmented_kernel<T, Op, 8, false>);
  }

  acpp_status enqueue(hipStream_t stream) override { return reduce ? enqueue_reduce(stream) : enqueue_scan(stream); }

  // The table of the tiles' first segments (many tiles only), one work-group
  // per tile, then the fix-up of segments that span tiles.
  acpp_status enqueue_reduce(hipStream_t stream) {
    acpp_status st;
    const uint64_t num_tiles = p.num_tiles, num_segments = p.num_segments;
    if (table) {
      if (num_segments <= max_scatter_segments * num_tiles && num_tiles <= max_scatter_tiles * num_segments)
        hipLaunchKernelGGL(tile_scatter_kernel, dim3(static_cast<uint32_t>(ceil_div(num_segments, 256))), dim3(256), 0,
                           stream, p.offsets, num_segments, tile_elems, p.num_tiles, table);
      else
        hipLaunchKernelGGL(tile_table_kernel, dim3(static_cast<uint32_t>(ceil_div(num_tiles + 1, 256))), dim3(256), 0,
                           stream, p.offsets, num_segments, tile_elems, p.num_tiles, table);
      st = check_launch(name);
      if (st != ACPP_SUCCESS) return st;
    }
    auto kernel = [&](auto runs) {
      constexpr bool RUNS = decltype(runs)::value;
      return rows == 2   ? segmented_reduce_kernel<T, Op, 2, RUNS>
             : rows == 4 ? segmented_reduce_kernel<T, Op, 4, RUNS>
                         : segmented_reduce_kernel<T, Op, 8, RUNS>;
    };
    const bool few = num_segments <= max_few_segments(wg);
    hipLaunchKernelGGL(few ? kernel(std::false_type{}) : kernel(std::true_type{}), dim3(grid), dim3(wg), lds, stream, p,
                       parts);
    st = check_launch(name);
    const bool walked = num_segments <= max_walk_segments(wg);  // whatever tiles they start in
    if (st != ACPP_SUCCESS || (num_tiles == 1 && walked)) return st;
    const uint32_t fix_groups = static_cast<uint32_t>(ceil_div(num_tiles, 1024));
    const uint64_t fill_groups = walked ? 0 : ceil_div(num_segments, static_cast<uint64_t>(empty_runs) * empty_run);
    hipLaunchKernelGGL((segmented_fixup_kernel<T, Op>), dim3(fix_groups + static_cast<uint32_t>(fill_groups)),
                       dim3(1024), 0, stream, p, parts, tile_elems, fix_groups);
    return check_launch(name);
  }

  // Parts small enough to occupy the chip, large enough that the searches do
  // not count (2^28 fp32 in 89,479 segments: 411 us with 1024 words, 404 us with
  // 4096; 2^23 in 1.7 million: 31 and 56 us), with the starts that go with
  // the words, up to one in four elements.
  acpp_status mark_heads(hipStream_t stream) {
    const uint64_t words = p.total >= (1ull << 27) ? 4096 : p.total >= (1ull << 23) ? 1024 : 256;
    const uint64_t all = p.num_segments + head_words * word_weight;
    const uint64_t even = ceil_div(ceil_div(all, ceil_div(head_words, words)), word_weight) * word_weight;
    const uint32_t part = static_cast<uint32_t>(std::min(even, 2 * words * word_weight));
    hipLaunchKernelGGL(head_bitmap_kernel, dim3(static_cast<uint32_t>(ceil_div(all, part))), dim3(256),
                       part / word_weight * 4, stream, p.offsets, p.num_segments, p.total, head_words, part, heads);
    return check_launch(name);
  }

  acpp_status enqueue_scan(hipStream_t stream) {
    region_launch rl;
    acpp_status st = begin_region_launch_flag(trip_flag, region, region_used, region_cap, rs, stream, &rl);
    if (st != ACPP_SUCCESS) return st;
    p.epoch = rl.epoch;
    p.ticket_base = rl.ticket_base;
    if (!mark) st = mark_heads(stream);
    if (st == ACPP_SUCCESS)
      st = with_scan_kernel([&](auto kernel) -> acpp_status {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(wg), lds, stream, p);
        return check_launch(name);
      });
    // every work-group draws one ticket past the last tile before it exits
    end_region_launch(rs, rl, p.num_tiles + grid, st);
    return st;
  }
};

// Validates a call and hands the prepared one to `run` (NULL when there is
// nothing to do).  `stream`: see call::prepare.
template <class T, class F>
acpp_status with_prepared(acpp_allocation_group *g, const hipStream_t *stream, const T *in, T *out,
                          const uint64_t *offsets, uint64_t num_segments, uint64_t total, T init, int op, bool reduce,
                          const acpp_launch_config *cfg, const char *name, F &&run) {
  using W = typename elem_traits<T>::work;
  if (!g) return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": scratch group is NULL");
  if (num_segments > 0 && !offsets)
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": offsets is NULL");
  if ((total > 0 && !in) || ((total > 0 || (reduce && num_segments > 0)) && !out))
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": in or out is NULL");
  if (op < ops::op_plus || op > ops::op_max)
    return set_error(ACPP_ERROR_UNSUPPORTED, std::string(name) + ": segmented forms support plus, multiply, min and max");
  if (num_segments == 0) {
    acpp_status s = run(static_cast<call<T, ops::plus<W, T>> *>(nullptr));
    return s == ACPP_SUCCESS ? clear_error() : s;
  }
  return with_op<W, T>(op, [&](auto opv) -> acpp_status {
    using Op = decltype(opv);
    if constexpr (Op::id > ops::op_max) {
      return set_error(ACPP_ERROR_UNSUPPORTED, "unsupported operator");
    } else {
      call<T, Op> c;
      c.name = name;
      acpp_status s = c.prepare(g, stream, in, out, offsets, num_segments, total, elem_traits<T>::to_work(init),
                                reduce, cfg);
      if (s == ACPP_SUCCESS) s = run(&c);
      return s == ACPP_SUCCESS ? clear_error() : s;
    }
  });
}

template <class T>
acpp_status entry(acpp_allocation_group *g, hipStream_t stream, const T *in, T *out, const uint64_t *offsets,
                  uint64_t num_segments, uint64_t total, T init, int op, bool reduce, const acpp_launch_config *cfg,
                  const char *name) {
  return with_prepared<T>(g, &stream, in, out, offsets, num_segments, total, init, op, reduce, cfg, name,
                          [&](auto *c) { return c ? c->enqueue(stream) : ACPP_SUCCESS; });
}

}  // namespace seg_detail
}  // namespace acpp_impl

using namespace acpp_impl;
using namespace acpp_impl::seg_detail;

// --------------------------------------------------------------------------
// Plans: a call whose scratch is kept.  Every launch enqueues its kernels
// directly: replaying them as a graph of as many nodes took 6 to 9 us longer
// on MI355X (2^19 fp32 scan 16.0 us as a graph, 6.8 us direct), and
// a graph has to clear the scan's sync region in every replay.
// --------------------------------------------------------------------------
struct acpp_segmented_plan {
  std::unique_ptr<prepared> call;  // empty: nothing to do
  std::mutex mutex;                // the epochs of the sync region, in launch order
  int device = 0;
};

namespace {
template <class T>
acpp_status make_plan(acpp_allocation_group *g, const T *in, T *out, const uint64_t *offsets, uint64_t num_segments,
                      uint64_t total, T init, int op, bool reduce, const acpp_launch_config *cfg, const char *name,
                      acpp_segmented_plan **plan) {
  if (!g) return set_error(ACPP_ERROR_INVALID_ARGUMENT, "scratch group is NULL");
  if (!plan) return set_error(ACPP_ERROR_INVALID_ARGUMENT, "plan output pointer is NULL");
  int cus = 0;
  acpp_status st = enter_device(g, &cus);
  if (st != ACPP_SUCCESS) return st;
  std::unique_ptr<acpp_segmented_plan> made(new (std::nothrow) acpp_segmented_plan);
  if (!made) return set_error(ACPP_ERROR_OUT_OF_MEMORY, "host allocation failed");
  made->device = group_device(g);
  st = with_prepared<T>(g, nullptr, in, out, offsets, num_segments, total, init, op, reduce, cfg, name,
                        [&](auto *c) -> acpp_status {
                          if (!c) return ACPP_SUCCESS;
                          using C = std::remove_pointer_t<decltype(c)>;
                          made->call.reset(new (std::nothrow) C(*c));
                          if (!made->call) return set_error(ACPP_ERROR_OUT_OF_MEMORY, "host allocation failed");
                          return ACPP_SUCCESS;
                        });
  if (st == ACPP_SUCCESS) *plan = made.release();
  return st;
}
}  // namespace

extern "C" {

#define ACPP_DEFINE_SEGMENTED(tag, T)                                                                 \
  acpp_status acpp_segmented_inclusive_scan_##tag(acpp_allocation_group *scratch, acpp_stream_t stream, \
                                                   const T *first, uint64_t n, T *d_first,             \
                                                   const uint64_t *offsets, uint64_t num_segments,     \
                                                   acpp_algorithm_op op,                               \
                                                   const acpp_launch_config *config) {                 \
    return entry<T>(scratch, static_cast<hipStream_t>(stream), first, d_first, offsets, num_segments,  \
                    n, T{}, op, false, config, "acpp_segmented_inclusive_scan_" #tag);                \
  }                                                                                                   \
  acpp_status acpp_segmented_reduce_##tag(acpp_allocation_group *scratch, acpp_stream_t stream,       \
                                          const T *first, uint64_t n, const uint64_t *offsets,        \
                                          uint64_t num_segments, T *out, T init,                      \
                                          acpp_algorithm_op op, const acpp_launch_config *config) {   \
    return entry<T>(scratch, static_cast<hipStream_t>(stream), first, out, offsets, num_segments, n,   \
                    init, op, true, config, "acpp_segmented_reduce_" #tag);                           \
  }                                                                                                   \
  acpp_status acpp_segmented_plan_inclusive_scan_##tag(                                                \
      acpp_allocation_group *scratch, const T *first, uint64_t n, T *d_first,                         \
      const uint64_t *offsets, uint64_t num_segments, acpp_algorithm_op op,                           \
      const acpp_launch_config *config, acpp_segmented_plan **plan) {                                 \
    return make_plan<T>(scratch, first, d_first, offsets, num_segments, n, T{}, op, false, config,    \
                        "acpp_segmented_plan_inclusive_scan_" #tag, plan);                            \
  }                                                                                                   \
  acpp_status acpp_segmented_plan_reduce_##tag(                                                        \
      acpp_allocation_group *scratch, const T *first, uint64_t n, const uint64_t *offsets,            \
      uint64_t num_segments, T *out, T init, acpp_algorithm_op op, const acpp_launch_config *config, \
      acpp_segmented_plan **plan) {                                                                   \
    return make_plan<T>(scratch, first, out, offsets, num_segments, n, init, op, true, config,        \
                        "acpp_segmented_plan_reduce_" #tag, plan);                                    \
  }

ACPP_DEFINE_SEGMENTED(i32, int32_t)
ACPP_DEFINE_SEGMENTED(i64, int64_t)
ACPP_DEFINE_SEGMENTED(f32, float)
ACPP_DEFINE_SEGMENTED(f64, double)

acpp_status acpp_segmented_plan_launch(acpp_segmented_plan *plan, acpp_stream_t stream) {
  if (!plan) return set_error(ACPP_ERROR_INVALID_ARGUMENT, "plan is NULL");
  int cur = 0;
  ACPP_CHECK_HIP(hipGetDevice(&cur));
  if (cur != plan->device) ACPP_CHECK_HIP(hipSetDevice(plan->device));
  if (!plan->call) return clear_error();
  std::lock_guard<std::mutex> lock{plan->mutex};
  acpp_status s = plan->call->enqueue(static_cast<hipStream_t>(stream));
  return s == ACPP_SUCCESS ? clear_error() : s;
}

acpp_status acpp_segmented_plan_destroy(acpp_segmented_plan *plan) {
  if (!plan) return set_error(ACPP_ERROR_INVALID_ARGUMENT, "plan is NULL");
  delete plan;
  return clear_error();
}

}  // extern "C"
