// Stream compaction: algorithms::copy_if
// (include/hipSYCL/algorithms/algorithm.hpp:178-243).
//
// Reference: an exclusive scan (generate_scan_process) of size_t flags
// pred(x[i]) ? 1 : 0, whose result processor writes x[i] to
// d_first[scan[i]] and, at the last element, the number of elements copied
// (algorithm.hpp:194-242).  An empty range writes 0 to *num_elements_copied
// and returns (algorithm.hpp:184-188).
//
// MI355X design: one launch on the decoupled look-back machinery of the scan
// (scan_common.hpp).  A tile is B work-items x R rows x one 16-byte vector;
// each work-item evaluates the predicate on its vectors into a bitmask,
// counts with popcount, the work-group ranks the selected elements with DPP
// wave scans and one LDS exchange, one wave looks back over the tile
// counts (64-bit, one 128-byte status line per tile) for the tile's output
// offset.  Meanwhile every wave compacts the selected elements of each of
// its rows into that row's own LDS segment (128 KiB of segments at the
// default 1024 x 8 tile); the segments are then stored with consecutive
// lanes on consecutive output elements (coalesced whatever the selection
// pattern).  The last tile writes the total count.
//
// The predicate is data, not a functor (a functor cannot cross the C-ABI):
// comparison with a constant, a bit-mask test, or a stencil array for any
// predicate the caller evaluates with its own kernel.
#include "launch_util.hpp"
#include "scan_common.hpp"

namespace acpp_impl {
namespace copy_if_detail {

using scan_detail::st_aggregate;
using scan_detail::st_prefix;
using scan_detail::status_stride_words;
using scan_detail::u32x4;

template <class T>
struct params {
  const T *in;
  const uint8_t *stencil;  // ACPP_PRED_STENCIL
  T *out;
  uint64_t *num_copied;     // may be NULL
  uint64_t n;
  T operand;
  T mask;
  uint32_t num_tiles;
  uint32_t epoch;
  uint32_t ticket_base;
  int force_give_up;  // ACPP_VARIANT_FORCE_GIVE_UP (tests of the error path)
  sync_header *sync;
  uint64_t *status;
};

template <int PRED, class T>
__device__ __forceinline__ bool eval(const params<T> &p, T x) {
  if constexpr (PRED == ACPP_PRED_NONZERO) return x != T(0);
  else if constexpr (PRED == ACPP_PRED_EQ) return x == p.operand;
  else if constexpr (PRED == ACPP_PRED_NE) return x != p.operand;
  else if constexpr (PRED == ACPP_PRED_LT) return x < p.operand;
  else if constexpr (PRED == ACPP_PRED_LE) return x <= p.operand;
  else if constexpr (PRED == ACPP_PRED_GT) return x > p.operand;
  else if constexpr (PRED == ACPP_PRED_GE) return x >= p.operand;
  else {
    static_assert(PRED == ACPP_PRED_MASK_EQ, "predicate on the element");
    if constexpr (std::is_integral_v<T>) return (x & p.mask) == p.operand;
    else return false;
  }
}

// The VEC stencil bytes of a data vector, loaded as one word at any address.
template <int VEC>
struct stencil_word;
template <>
struct stencil_word<2> {
  typedef uint16_t type;
};
template <>
struct stencil_word<4> {
  typedef uint32_t type;
};
template <>
struct stencil_word<8> {
  typedef uint64_t type;
};
template <>
struct stencil_word<16> {
  typedef u32x4 type;
};

// Selection bits of the tile's vectors from the stencil: bit k of fm[r] =
// element k of row r is copied (elements past the end of a partial tile read
// as 0).
template <bool FULL, int R, int VEC>
__device__ __forceinline__ void stencil_bits(const uint8_t *tile, const scan_detail::partial_tile &part,
                                             uint32_t (&fm)[R]) {
  using SW = typename stencil_word<VEC>::type;
  typedef SW SW1 __attribute__((aligned(1)));
  const int B = blockDim.x;
  const int tid = threadIdx.x;
  const SW1 *sw = reinterpret_cast<const SW1 *>(tile);
  uint32_t cut_bits = 0;
  if constexpr (!FULL) {
    if (part.count != 0 && static_cast<uint32_t>(tid) == part.tid) {
      const uint8_t *src = tile + static_cast<uint64_t>(part.row * B + part.tid) * VEC;
#pragma unroll
      for (int k = 0; k < VEC; ++k)
        if (static_cast<uint32_t>(k) < part.count && src[k] != 0) cut_bits |= 1u << k;
    }
  }
  SW bytes[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    bytes[r] = SW{};
    if (FULL || static_cast<uint32_t>(r * B + tid + 1) * VEC <= part.in_range) bytes[r] = sw[r * B + tid];
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    uint32_t words[4] = {};
    __builtin_memcpy(words, &bytes[r], sizeof(SW));
    // the words, not the bytes extracted from them, are kept until here
#pragma unroll
    for (int i = 0; i < (VEC + 3) / 4; ++i) asm volatile("" : "+v"(words[i]));
    fm[r] = 0;
#pragma unroll
    for (int k = 0; k < VEC; ++k) fm[r] |= (((words[k >> 2] >> (8 * (k & 3))) & 0xffu) != 0u ? 1u : 0u) << k;
    if (!FULL && part.cut(r, tid)) fm[r] = cut_bits;
  }
}

// Element k of a 16-byte vector of T.
template <class T>
__device__ __forceinline__ T elem(const u32x4 &q, int k) {
  T tmp[16 / sizeof(T)];
  __builtin_memcpy(tmp, &q, 16);
  return tmp[k];
}

// Selection bits of a vector from the predicate.
template <int PRED, class T>
__device__ __forceinline__ uint32_t select_bits(const params<T> &p, const u32x4 &q) {
  constexpr int VEC = 16 / sizeof(T);
  uint32_t fm = 0;
#pragma unroll
  for (int k = 0; k < VEC; ++k)
    if (eval<PRED>(p, elem<T>(q, k))) fm |= 1u << k;
  return fm;
}

// Vectors of 1- and 2-byte elements through an empty asm statement: elements
// extracted before it are not kept for uses after it.
template <class T, int R>
__device__ __forceinline__ void repack(u32x4 (&q)[R]) {
  if constexpr (sizeof(T) < 4) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      uint32_t a = q[r].x, b = q[r].y, c = q[r].z, d = q[r].w;
      asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
      q[r] = u32x4{a, b, c, d};
    }
  }
}

// Shared words of a copy_if work-group.
template <int R>
struct tile_shared {
  uint32_t tile;
  uint32_t wave[R * scan_detail::max_waves];  // per (row, wave): counts, then offsets
  uint32_t agg;
  uint64_t excl;
};

// One tile.  PRED and FULL are compile-time: a full tile has no bounds
// checks and one predicate's code, since with one work-group per CU (the
// LDS segments take 128 KiB) this phase is not overlapped with memory and
// its instruction count is on the critical path.
template <int PRED, bool FULL, class T, int R>
__device__ __forceinline__ void copy_if_tile(const params<T> &p, uint32_t tile, tile_shared<R> &sh, T *s_stage) {
  using CountOp = ops::plus<uint32_t, uint32_t>;
  using SIO = scan_detail::status_io<uint64_t>;
  constexpr int VEC = 16 / sizeof(T);
  constexpr int SEG = 64 * VEC;  // LDS room of one wave row's selection
  const int tid = threadIdx.x;
  const int B = blockDim.x;
  const int nw = B >> 6;
  const int w = tid >> 6;
  const int lane = tid & 63;
  const uint64_t tile_elems = static_cast<uint64_t>(B) * R * VEC;
  const uint64_t base = static_cast<uint64_t>(tile) * tile_elems;

  const uint32_t in_range =
      FULL ? static_cast<uint32_t>(tile_elems) : static_cast<uint32_t>(p.n > base ? min(p.n - base, tile_elems) : 0);
  const scan_detail::partial_tile part = scan_detail::partial_tile::of<T>(in_range, B);

  // The elements stay packed in their 16-byte vectors (four registers a row)
  // and are extracted where they are used: 8 rows of 8 or 16 unpacked
  // elements spill.
  u32x4 q[R];
  const scan_detail::u32x4_a1 *src = reinterpret_cast<const scan_detail::u32x4_a1 *>(p.in + base);
  if constexpr (FULL) {
#pragma unroll
    for (int r = 0; r < R; ++r) q[r] = src[r * B + tid];
  } else {
    const u32x4 cut = part.load_cut<T>(p.in + base, tid, B);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      q[r] = part.cut(r, tid) ? cut : u32x4{0, 0, 0, 0};
      if (static_cast<uint32_t>(r * B + tid + 1) * VEC <= in_range) q[r] = src[r * B + tid];
    }
    repack<T>(q);
  }
  uint32_t fm[R];
  if constexpr (PRED == ACPP_PRED_STENCIL) {
    stencil_bits<FULL, R, VEC>(p.stencil + base, part, fm);
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      fm[r] = select_bits<PRED>(p, q[r]);
      if constexpr (!FULL) {
        // only the elements in range
        const uint32_t first = static_cast<uint32_t>(r * B + tid) * VEC;
        const uint32_t cnt = in_range > first ? in_range - first : 0u;
        if (cnt < VEC) fm[r] &= (1u << cnt) - 1u;
      }
    }
  }
  // The compaction below extracts the elements again from the packed vectors
  // instead of keeping the predicate's extracted copies alive.
  repack<T>(q);
  // The same for the bits: kept as one word a row, not as lane masks, which
  // overflow the scalar registers (2^28 elements, half kept: int16 206.8 us as
  // masks, 202.3 us so; int8 137.3 and 131.0 us).
  if constexpr (sizeof(T) < 4) {
#pragma unroll
    for (int r = 0; r < R; ++r) asm volatile("" : "+v"(fm[r]));
  }
  // Ranks inside each wave row; the (row, wave) counts go to LDS.
  uint32_t wexcl[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t c = static_cast<uint32_t>(__builtin_popcount(fm[r]));
    const uint32_t incl = wave::inclusive_scan<CountOp>(c);
    wexcl[r] = incl - c;
    if (lane == 63) sh.wave[r * nw + w] = incl;
  }
  __syncthreads();
  // Wave 0 turns the (row, wave) counts into offsets and publishes the
  // tile's count before anything else, since every later tile's look-back
  // may be waiting for it.
  uint32_t agg0 = 0;
  if (w == 0) {
    agg0 = scan_detail::tile_prefixes<CountOp, uint32_t>(R * nw, sh.wave);
    if (lane == 0) {
      if (tile == 0) {
        if (p.num_tiles > 1) SIO::publish(p.status, 0, p.epoch, st_prefix, static_cast<uint64_t>(agg0));
        sh.excl = 0;
      } else {
        SIO::publish(p.status, tile, p.epoch, st_aggregate, static_cast<uint64_t>(agg0));
      }
      sh.agg = agg0;
    }
  }
  // Compaction: each wave row's selected elements go, in order, to that
  // row's own LDS segment (room for all 64 x VEC of them), at the rank
  // inside the wave row.  It needs no tile-wide offsets, so it runs while
  // wave 0 looks back; the stores below then copy segment after segment.
#pragma unroll
  for (int r = 0; r < R; ++r) {
    uint32_t pos = static_cast<uint32_t>((r * nw + w) * SEG) + wexcl[r];
    const uint32_t bits = fm[r];
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
      if (bits & (1u << k)) s_stage[pos++] = elem<T>(q[r], k);
    }
  }
  // Wave 0 looks back for the tile's output offset.
  if (w == 0 && tile != 0) {
    wait_own_stores();  // the tile's count is out before the first poll
    const uint64_t e = scan_detail::lookback<ops::plus<uint64_t, uint64_t>, uint64_t, scan_detail::lookback_slots>(
        p.status, tile, p.epoch, p.sync, p.force_give_up != 0);
    if (lane == 0) {
      if (tile + 1 < p.num_tiles) SIO::publish(p.status, tile, p.epoch, st_prefix, e + agg0);
      sh.excl = e;
    }
  }
  __syncthreads();
  // Each wave stores its own segments: a segment's elements are contiguous
  // in the output, at the offset of its (row, wave) pair, and consecutive
  // lanes take consecutive elements (coalesced stores, conflict-free LDS
  // reads).
  const uint32_t count = __builtin_amdgcn_readfirstlane(sh.agg);
  const uint64_t ex = sh.excl;
  const uint64_t tile_prefix =
      (static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(ex >> 32))) << 32) |
      __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(ex));
  if (tile + 1 == p.num_tiles && tid == 0 && p.num_copied) *p.num_copied = tile_prefix + count;
  T *dst = p.out + tile_prefix;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int seg = r * nw + w;
    const uint32_t off = sh.wave[seg];
    const uint32_t end = (seg + 1 < R * nw) ? sh.wave[seg + 1] : count;
    const T *src = s_stage + seg * SEG;
    if constexpr (sizeof(T) == 1) {
      // 4-byte stores of EPW elements: the elements before the segment's
      // first 4-byte aligned output address and those after its last whole
      // word are stored one by one (the words around them hold elements of
      // neighbouring segments); each word's source bytes are two aligned
      // LDS words shifted together.  (2-byte elements measured slower this
      // way: one store per element stays.)
      constexpr uint32_t EPW = 4 / sizeof(T);
      const uint32_t len = end - off;
      T *d = dst + off;
      const uint32_t mis = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(d) / sizeof(T)) % EPW;
      const uint32_t head = min(len, (EPW - mis) % EPW);
      if (lane < head) d[lane] = src[lane];
      const uint32_t words = (len - head) / EPW;
      uint32_t *dw = reinterpret_cast<uint32_t *>(d + head);
      const uint32_t *lds32 = reinterpret_cast<const uint32_t *>(s_stage);
      const uint32_t b0 = static_cast<uint32_t>((seg * SEG + head) * sizeof(T));  // LDS byte of word 0
      for (uint32_t j = lane; j < words; j += 64) {
        const uint32_t b = b0 + j * 4;
        const uint32_t sh = b & 3u;
        const uint32_t lo = lds32[b >> 2];
        const uint32_t hi = lds32[(b >> 2) + (sh ? 1u : 0u)];  // in the segment when sh != 0
        dw[j] = __builtin_amdgcn_alignbyte(hi, lo, sh);
      }
      const uint32_t t0 = head + words * EPW;
      if (lane < len - t0) d[t0 + lane] = src[t0 + lane];
    } else {
      for (uint32_t j = lane; j < end - off; j += 64) dst[off + j] = src[j];
    }
  }
}

template <class T, int R, int PRED>
__global__ __launch_bounds__(1024) void copy_if_kernel(params<T> p) {
  constexpr int VEC = 16 / sizeof(T);
  __shared__ tile_shared<R> sh;
  extern __shared__ unsigned char s_stage_raw[];  // R x nw segments of 64 x VEC elements (B * R * VEC)
  T *s_stage = reinterpret_cast<T *>(s_stage_raw);

  if (threadIdx.x == 0)
    sh.tile = __hip_atomic_fetch_add(&p.sync->tile_counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) -
              p.ticket_base;
  __syncthreads();
  const uint32_t tile = __builtin_amdgcn_readfirstlane(sh.tile);
  if (tile >= p.num_tiles) return;
  const uint64_t tile_elems = static_cast<uint64_t>(blockDim.x) * R * VEC;
  const uint64_t base = static_cast<uint64_t>(tile) * tile_elems;
  if (base + tile_elems <= p.n)
    copy_if_tile<PRED, true>(p, tile, sh, s_stage);
  else
    copy_if_tile<PRED, false>(p, tile, sh, s_stage);
}

__global__ void store_zero_kernel(uint64_t *p) { *p = 0; }

template <class T>
constexpr int rows() {
  return 8;
}

template <class T>
acpp_status entry(acpp_allocation_group *g, hipStream_t stream, const T *in, uint64_t n, const uint8_t *stencil,
                  T *out, int pred, T operand, T mask, uint64_t *num_copied, const acpp_launch_config *cfg,
                  const char *name) {
  constexpr int VEC = 16 / sizeof(T);
  if (!g) return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": scratch group is NULL");
  if (pred < ACPP_PRED_NONZERO || pred > ACPP_PRED_STENCIL)
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": unknown predicate");
  if (pred == ACPP_PRED_MASK_EQ && !std::is_integral_v<T>)
    return set_error(ACPP_ERROR_UNSUPPORTED, std::string(name) + ": mask predicates take integer elements");
  if (n > 0 && (!in || !out || (pred == ACPP_PRED_STENCIL && !stencil)))
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": NULL pointer argument");
  int cus = 0;
  acpp_status st = enter_device(g, &cus);
  if (st != ACPP_SUCCESS) return st;
  if (n == 0) {
    // algorithm.hpp:184-188: the count of an empty range is 0.
    // Written by a kernel: asynchronous, and allowed under stream capture.
    if (num_copied) {
      hipLaunchKernelGGL(store_zero_kernel, dim3(1), dim3(1), 0, stream, num_copied);
      st = check_launch(name);
      if (st != ACPP_SUCCESS) return st;
    }
    return clear_error();
  }
  // 1024-wide tiles, narrower for short inputs of 1- and 2-byte elements:
  // their tiles hold four or two times the elements, and a CU works through a
  // tile alone (whole calls with 256 / 512 / 1024 work-items, half kept: int8
  // 2^20 10.8 / 11.5 / 14.5 us, 2^24 20.6 / 17.7 / 18.2 us, 2^26 51.3 / 42.0 /
  // 42.2 us; int16 2^19 8.4 / 8.8 / 10.2 us, 2^22 12.7 / 11.6 / 11.9 us; int32
  // 2^21 10.4 / 9.0 / 8.8 us).
  constexpr uint64_t mid_n = sizeof(T) == 1 ? 3ull << 19 : sizeof(T) == 2 ? 3ull << 18 : 0;
  constexpr uint64_t wide_n = sizeof(T) == 1 ? 1ull << 26 : sizeof(T) == 2 ? 3ull << 21 : 0;
  const uint32_t wg = (cfg && cfg->work_group_size) ? cfg->work_group_size : n >= wide_n ? 1024 : n >= mid_n ? 512 : 256;
  if (!valid_work_group_size(wg))
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": bad work_group_size");
  if (cfg && cfg->items_per_thread && static_cast<int>(cfg->items_per_thread) != rows<T>())
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": items_per_thread must be 8 (or 0)");
  const uint64_t tile_elems = static_cast<uint64_t>(wg) * rows<T>() * VEC;
  const uint64_t num_tiles = ceil_div(n, tile_elems);
  if (num_tiles >= (1ull << 31)) return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": problem too large");

  void *region = nullptr;
  size_t cap = 0;
  region_state *rs = nullptr;
  const size_t used = sizeof(sync_header) + num_tiles * status_stride_words * sizeof(uint64_t);
  st = group_obtain_sync(g, used, stream, &region, &cap, &rs);
  if (st != ACPP_SUCCESS) return st;
  region_launch rl;
  st = begin_region_launch(g, region, used, cap, rs, stream, &rl);
  if (st != ACPP_SUCCESS) return st;
  params<T> p;
  p.in = in;
  p.stencil = stencil;
  p.out = out;
  p.num_copied = num_copied;
  p.n = n;
  p.operand = operand;
  p.mask = mask;
  p.num_tiles = static_cast<uint32_t>(num_tiles);
  p.epoch = rl.epoch;
  p.ticket_base = rl.ticket_base;
  p.force_give_up = (cfg && (cfg->flags & ACPP_VARIANT_FORCE_GIVE_UP)) ? 1 : 0;
  p.sync = static_cast<sync_header *>(region);
  p.status = reinterpret_cast<uint64_t *>(static_cast<char *>(region) + sizeof(sync_header));
  const size_t stage_bytes = static_cast<size_t>(tile_elems) * sizeof(T);  // 128 KiB at 1024 x 8
  const dim3 grid(static_cast<uint32_t>(num_tiles));
  constexpr int R = rows<T>();
  switch (pred) {
    case ACPP_PRED_NONZERO:
      hipLaunchKernelGGL((copy_if_kernel<T, R, ACPP_PRED_NONZERO>), grid, dim3(wg), stage_bytes, stream, p);
      break;
    case ACPP_PRED_EQ:
      hipLaunchKernelGGL((copy_if_kernel<T, R, ACPP_PRED_EQ>), grid, dim3(wg), stage_bytes, stream, p);
      break;
    case ACPP_PRED_NE:
      hipLaunchKernelGGL((copy_if_kernel<T, R, ACPP_PRED_NE>), grid, dim3(wg), stage_bytes, stream, p);
      break;
    case ACPP_PRED_LT:
      hipLaunchKernelGGL((copy_if_kernel<T, R, ACPP_PRED_LT>), grid, dim3(wg), stage_bytes, stream, p);
      break;
    case ACPP_PRED_LE:
      hipLaunchKernelGGL((copy_if_kernel<T, R, ACPP_PRED_LE>), grid, dim3(wg), stage_bytes, stream, p);
      break;
    case ACPP_PRED_GT:
      hipLaunchKernelGGL((copy_if_kernel<T, R, ACPP_PRED_GT>), grid, dim3(wg), stage_bytes, stream, p);
      break;
    case ACPP_PRED_GE:
      hipLaunchKernelGGL((copy_if_kernel<T, R, ACPP_PRED_GE>), grid, dim3(wg), stage_bytes, stream, p);
      break;
    case ACPP_PRED_MASK_EQ:
      // rejected above for floating-point elements
      if constexpr (std::is_integral_v<T>)
        hipLaunchKernelGGL((copy_if_kernel<T, R, ACPP_PRED_MASK_EQ>), grid, dim3(wg), stage_bytes, stream, p);
      break;
    default:
      hipLaunchKernelGGL((copy_if_kernel<T, R, ACPP_PRED_STENCIL>), grid, dim3(wg), stage_bytes, stream, p);
      break;
  }
  st = check_launch(name);
  end_region_launch(rs, rl, static_cast<uint32_t>(num_tiles), st);
  return st == ACPP_SUCCESS ? clear_error() : st;
}

}  // namespace copy_if_detail
}  // namespace acpp_impl

using namespace acpp_impl;

extern "C" {

#define ACPP_DEFINE_COPY_IF(tag, T)                                                                       \
  acpp_status acpp_copy_if_##tag(acpp_allocation_group *scratch, acpp_stream_t stream, const T *first,   \
                                 uint64_t n, T *d_first, int pred, T operand, T mask,                    \
                                 uint64_t *num_copied, const acpp_launch_config *config) {               \
    if (pred == ACPP_PRED_STENCIL)                                                                        \
      return set_error(ACPP_ERROR_INVALID_ARGUMENT, "acpp_copy_if_" #tag ": use acpp_copy_if_stencil_" #tag); \
    return copy_if_detail::entry<T>(scratch, static_cast<hipStream_t>(stream), first, n, nullptr, d_first,  \
                                    pred, operand, mask, num_copied, config, "acpp_copy_if_" #tag);        \
  }                                                                                                       \
  acpp_status acpp_copy_if_stencil_##tag(acpp_allocation_group *scratch, acpp_stream_t stream,           \
                                         const T *first, uint64_t n, const uint8_t *stencil, T *d_first, \
                                         uint64_t *num_copied, const acpp_launch_config *config) {       \
    return copy_if_detail::entry<T>(scratch, static_cast<hipStream_t>(stream), first, n, stencil, d_first,  \
                                    ACPP_PRED_STENCIL, T(0), T(0), num_copied, config,                    \
                                    "acpp_copy_if_stencil_" #tag);                                         \
  }

ACPP_DEFINE_COPY_IF(i8, int8_t)
ACPP_DEFINE_COPY_IF(u8, uint8_t)
ACPP_DEFINE_COPY_IF(i16, int16_t)
ACPP_DEFINE_COPY_IF(u16, uint16_t)
ACPP_DEFINE_COPY_IF(i32, int32_t)
ACPP_DEFINE_COPY_IF(u32, uint32_t)
ACPP_DEFINE_COPY_IF(i64, int64_t)
ACPP_DEFINE_COPY_IF(u64, uint64_t)
ACPP_DEFINE_COPY_IF(f32, float)
ACPP_DEFINE_COPY_IF(f64, double)

}  // extern "C"
