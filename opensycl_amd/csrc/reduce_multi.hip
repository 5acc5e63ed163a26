// Several sycl::reduction objects in one kernel (handler::parallel_for with
// more than one reduction, include/hipSYCL/sycl/handler.hpp:799-975; test
// tests/sycl/reduction.cpp:116-208 runs a plus and a multiplies reduction in
// one parallel_for).
//
// One launch reduces up to four inputs of the same length, each with its
// own operator and output.  Every work-group streams the inputs one after the
// other (16-byte loads, the operator switch outside the streaming loop), reduces
// each with DPP and one LDS exchange and publishes one partial per reduction; the
// last work-group to finish (fence-free ticket, as in reduce_common.hpp) folds
// all partials in a fixed order and writes the results.  A large array that
// several reductions share is read once and folded for all of them, with one
// uniform switch per operator and batch of loads (2^28 fp32 in three reductions
// 460 us one by one, 160 us so; arrays off 16-byte alignment went element by
// element: 2573 us, now 159 us).
#include "launch_util.hpp"
#include "reduce_common.hpp"

namespace acpp_impl {
namespace multi_detail {

using reduce_detail::max_waves;
using reduce_detail::partial_slot_words;
using reduce_detail::publish_partial;
using reduce_detail::wait_partial;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int max_inputs = 4;
constexpr int unroll = 4;

template <class T>
struct params {
  using W = typename elem_traits<T>::work;
  const T *in[max_inputs];
  T *out[max_inputs];
  int op[max_inputs];
  int first[max_inputs];  // the first reduction over the same array (k itself: a new array)
  int count;
  uint64_t n;
  // Per input: 0 out = op(out, fold); 1 out = fold (initialize_to_identity);
  // 2 out = op(identity[k], fold) (initialize_to_identity with a given
  // identity, which an empty range yields).
  int init_mode[max_inputs];
  W identity[max_inputs];
  uint64_t *partials; // tagged slots [count][gridDim.x] (reduce_common.hpp)
  sync_header *sync;
  uint32_t epoch;     // tag of this launch's partials (>= 1)
  int force_give_up;  // ACPP_VARIANT_FORCE_GIVE_UP (tests of the error path)
};

// Calls f(Op{}) with the operator functor for `code`.
template <class W, class F>
__device__ __forceinline__ void dispatch(int code, F &&f) {
  switch (code) {
    case ops::op_plus: f(ops::plus<W, W>{}); return;
    case ops::op_multiply: f(ops::multiply<W, W>{}); return;
    case ops::op_min: f(ops::minimum<W, W>{}); return;
    case ops::op_max: f(ops::maximum<W, W>{}); return;
    default: break;
  }
  if constexpr (std::is_integral_v<W>) {
    switch (code) {
      case ops::op_bit_and: f(ops::bit_and<W, W>{}); return;
      case ops::op_bit_or: f(ops::bit_or<W, W>{}); return;
      case ops::op_bit_xor: f(ops::bit_xor<W, W>{}); return;
      case ops::op_logical_and: f(ops::logical_and<W, W>{}); return;
      default: f(ops::logical_or<W, W>{}); return;
    }
  }
}

// The vectors of an array: aligned 16-byte chunks behind a scalar head, and
// the scalars before and behind them.
template <class T>
struct stream {
  static constexpr int VEC = 16 / sizeof(T);
  const T *in;
  uint64_t head, nvec, tail, nscalar;
  __device__ __forceinline__ stream(const T *p, uint64_t n) : in(p) {
    head = ((16 - (reinterpret_cast<uintptr_t>(p) & 15)) & 15) / sizeof(T);
    if (head > n || reinterpret_cast<uintptr_t>(p) % sizeof(T)) head = n;
    nvec = (n - head) / VEC;
    tail = head + nvec * VEC;
    nscalar = head + (n - tail);
  }
  __device__ __forceinline__ typename elem_traits<T>::work scalar(uint64_t s) const {
    return elem_traits<T>::to_work(in[s < head ? s : tail + (s - head)]);
  }
  template <bool NT>
  __device__ __forceinline__ u32x4 vec(uint64_t i) const {
    const u32x4 *src = reinterpret_cast<const u32x4 *>(in + head);
    if constexpr (NT)
      return __builtin_nontemporal_load(src + i);
    else
      return src[i];
  }
};

template <class T, class W, int VEC>
__device__ __forceinline__ void unpack(u32x4 q, W (&out)[VEC]) {
  T t[VEC];
  __builtin_memcpy(t, &q, 16);
#pragma unroll
  for (int k = 0; k < VEC; ++k) out[k] = elem_traits<T>::to_work(t[k]);
}

// Fold of one input: `unroll` independent accumulators over 16-byte loads
// (`unroll` in flight), non-temporal when NT, then the scalars.  (With one
// accumulator and a bounds check per load, one fused int32 reduction of 2^28
// elements took 175 us against 154 us for the plain reduce.)
template <class T, class Op, bool NT>
__device__ typename elem_traits<T>::work stream_fold(const T *in, uint64_t n) {
  using W = typename elem_traits<T>::work;
  constexpr int VEC = 16 / sizeof(T);
  const uint64_t gid = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  const stream<T> s(in, n);
  W acc[unroll];
#pragma unroll
  for (int u = 0; u < unroll; ++u) acc[u] = Op::identity();
  auto fold = [&](u32x4 q, W &a) {
    W t[VEC];
    unpack<T>(q, t);
#pragma unroll
    for (int k = 0; k < VEC; ++k) a = Op::apply(a, t[k]);
  };
  uint64_t i = gid;
  for (; i + (unroll - 1) * stride < s.nvec; i += unroll * stride) {
    u32x4 q[unroll];
#pragma unroll
    for (int u = 0; u < unroll; ++u) q[u] = s.template vec<NT>(i + u * stride);
#pragma unroll
    for (int u = 0; u < unroll; ++u) fold(q[u], acc[u]);
  }
  for (; i < s.nvec; i += stride) fold(s.template vec<false>(i), acc[0]);
  for (uint64_t j = gid; j < s.nscalar; j += stride) acc[0] = Op::apply(acc[0], s.scalar(j));
  W v = acc[0];
#pragma unroll
  for (int u = 1; u < unroll; ++u) v = Op::apply(v, acc[u]);
  return v;
}

// Folds of one array for every reduction m with p.first[m] == first, in the
// accumulators and the order of stream_fold.
template <class T, bool NT>
__device__ void shared_fold(const params<T> &p, int first, typename elem_traits<T>::work (&v)[max_inputs]) {
  using W = typename elem_traits<T>::work;
  constexpr int VEC = 16 / sizeof(T);
  constexpr int rows = VEC <= 4 ? unroll : 1;  // vectors unpacked at a time
  const uint64_t gid = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  const stream<T> s(p.in[first], p.n);
  bool mine[max_inputs];
  W acc[max_inputs][unroll];
#pragma unroll
  for (int m = 0; m < max_inputs; ++m) {
    mine[m] = m < p.count && p.first[m] == first;
    if (mine[m])
      dispatch<W>(p.op[m], [&](auto opv) {
#pragma unroll
        for (int u = 0; u < unroll; ++u) acc[m][u] = decltype(opv)::identity();
      });
  }
  auto each = [&](auto &&f) {
#pragma unroll
    for (int m = 0; m < max_inputs; ++m)
      if (mine[m]) dispatch<W>(p.op[m], [&](auto opv) { f(opv, acc[m]); });
  };
  uint64_t i = gid;
  for (; i + (unroll - 1) * stride < s.nvec; i += unroll * stride) {
    u32x4 q[unroll];
#pragma unroll
    for (int u = 0; u < unroll; ++u) q[u] = s.template vec<NT>(i + u * stride);
#pragma unroll
    for (int u0 = 0; u0 < unroll; u0 += rows) {
      W t[rows][VEC];
#pragma unroll
      for (int u = 0; u < rows; ++u) unpack<T>(q[u0 + u], t[u]);
      each([&](auto opv, W(&a)[unroll]) {
#pragma unroll
        for (int u = 0; u < rows; ++u)
#pragma unroll
          for (int k = 0; k < VEC; ++k) a[u0 + u] = decltype(opv)::apply(a[u0 + u], t[u][k]);
      });
    }
  }
  for (; i < s.nvec; i += stride) {
    W t[VEC];
    unpack<T>(s.template vec<false>(i), t);
    each([&](auto opv, W(&a)[unroll]) {
#pragma unroll
      for (int k = 0; k < VEC; ++k) a[0] = decltype(opv)::apply(a[0], t[k]);
    });
  }
  for (uint64_t j = gid; j < s.nscalar; j += stride) {
    const W x = s.scalar(j);
    each([&](auto opv, W(&a)[unroll]) { a[0] = decltype(opv)::apply(a[0], x); });
  }
#pragma unroll
  for (int m = 0; m < max_inputs; ++m)
    if (mine[m])
      dispatch<W>(p.op[m], [&](auto opv) {
        W x = acc[m][0];
#pragma unroll
        for (int u = 1; u < unroll; ++u) x = decltype(opv)::apply(x, acc[m][u]);
        v[m] = x;
      });
}

// Reduces every reduction's value over the work-group, one LDS exchange for
// all; `write(m, x)` runs in one work-item per reduction, in the first `waves`
// waves (one: in order).
template <class T, class F>
__device__ void group_reduce(int waves, const params<T> &p, typename elem_traits<T>::work (&v)[max_inputs],
                             typename elem_traits<T>::work (&s_waves)[max_inputs][max_waves], F &&write) {
  using W = typename elem_traits<T>::work;
  const int nw = blockDim.x >> 6;
  const int w = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int m = 0; m < max_inputs; ++m)
    if (m < p.count)
      dispatch<W>(p.op[m], [&](auto opv) {
        const W x = wave::reduce_full<decltype(opv)>(v[m]);
        if (lane == 0) s_waves[m][w] = x;
      });
  __syncthreads();
  if (w >= waves) return;
  for (int m = w; m < p.count; m += waves)
    dispatch<W>(p.op[m], [&](auto opv) {
      using Op = decltype(opv);
      const W x = wave::reduce_full<Op>(lane < nw ? s_waves[m][lane] : Op::identity());
      if (lane == 0) write(m, x);
    });
}

// Writes the result of reduction m, whose whole fold is r.
template <class T, class Op>
__device__ __forceinline__ void finish(const params<T> &p, int m, typename elem_traits<T>::work r) {
  if (p.init_mode[m] == 0) r = Op::apply(elem_traits<T>::to_work(*p.out[m]), r);
  else if (p.init_mode[m] == 2) r = Op::apply(p.identity[m], r);
  *p.out[m] = static_cast<T>(r);
}

// One reduction after the other.  The loop stays a loop: a short call spends
// its time fetching instructions (1000 int32 in two reductions 5.6 us, 6.5 us
// with the code of shared_kernel, which has a copy for each reduction).
template <class T, bool NT>
__global__ __launch_bounds__(1024) void multi_kernel(params<T> p) {
  using W = typename elem_traits<T>::work;
  __shared__ W s_waves[max_waves];
  __shared__ bool s_last;
  const bool force = p.force_give_up != 0;
  const bool alone = gridDim.x == 1 && !force;  // nothing to exchange
  for (int k = 0; k < p.count; ++k) {
    __syncthreads();  // s_waves of the previous reduction has been read
    dispatch<W>(p.op[k], [&](auto opv) {
      using Op = decltype(opv);
      W v = stream_fold<T, Op, NT>(p.in[k], p.n);
      v = reduce_detail::block_reduce<reduce_detail::plain_monoid<W, Op>>(v, s_waves);
      if (threadIdx.x == 0) {
        if (alone)
          finish<T, Op>(p, k, v);
        else
          publish_partial(p.partials, static_cast<uint64_t>(k) * gridDim.x + blockIdx.x, p.epoch, v);
      }
    });
  }
  if (alone) return;
  if (threadIdx.x == 0) s_last = reduce_detail::draw_last_ticket(p.sync);  // (the last group waits for each partial's tag)
  __syncthreads();
  if (!s_last) return;
  for (int k = 0; k < p.count; ++k) {
    __syncthreads();
    dispatch<W>(p.op[k], [&](auto opv) {
      using Op = decltype(opv);
      W r = Op::identity();
      for (uint32_t i = threadIdx.x; i < gridDim.x; i += blockDim.x)
        r = Op::apply(r, wait_partial<W>(p.partials, static_cast<uint64_t>(k) * gridDim.x + i, p.epoch, p.sync, force,
                                         Op::identity()));
      r = reduce_detail::block_reduce<reduce_detail::plain_monoid<W, Op>>(r, s_waves);
      if (threadIdx.x == 0) finish<T, Op>(p, k, r);
    });
  }
  if (threadIdx.x == 0)
    __hip_atomic_store(&p.sync->done_counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Large arrays that several reductions share are read once.
template <class T, bool NT>
__global__ __launch_bounds__(1024) void shared_kernel(params<T> p) {
  using W = typename elem_traits<T>::work;
  __shared__ W s_waves[max_inputs][max_waves];
  __shared__ bool s_last;
  W v[max_inputs];
#pragma unroll
  for (int k = 0; k < max_inputs; ++k)
    if (k < p.count && p.first[k] == k) shared_fold<T, NT>(p, k, v);
  group_reduce(blockDim.x >> 6, p, v, s_waves, [&](int m, W x) {
    publish_partial(p.partials, static_cast<uint64_t>(m) * gridDim.x + blockIdx.x, p.epoch, x);
  });
  __syncthreads();
  if (threadIdx.x == 0) {
    // (the last group waits for each partial's tag)
    s_last = reduce_detail::draw_last_ticket(p.sync);
  }
  __syncthreads();
  if (!s_last) return;
#pragma unroll
  for (int k = 0; k < max_inputs; ++k)
    if (k < p.count)
      dispatch<W>(p.op[k], [&](auto opv) {
        using Op = decltype(opv);
        W r = Op::identity();
        for (uint32_t i = threadIdx.x; i < gridDim.x; i += blockDim.x)
          r = Op::apply(r, wait_partial<W>(p.partials, static_cast<uint64_t>(k) * gridDim.x + i, p.epoch, p.sync,
                                           p.force_give_up != 0, Op::identity()));
        v[k] = r;
      });
  group_reduce(1, p, v, s_waves,
               [&](int m, W r) { dispatch<W>(p.op[m], [&](auto opv) { finish<T, decltype(opv)>(p, m, r); }); });
  if (threadIdx.x == 0)
    __hip_atomic_store(&p.sync->done_counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// n == 0: outputs with initialize_to_identity become their identity (the
// given one, or the operator's); the others keep their value.
template <class T>
__global__ void identity_kernel(params<T> p) {
  using W = typename elem_traits<T>::work;
  const int k = threadIdx.x;
  if (k < p.count && p.init_mode[k] != 0)
    dispatch<W>(p.op[k], [&](auto opv) {
      *p.out[k] = static_cast<T>(p.init_mode[k] == 2 ? p.identity[k] : decltype(opv)::identity());
    });
}

// identities: NULL, or one value per input (used where the input's
// initialize_to_identity flag is set).  init_flags: one flag per input.
template <class T>
acpp_status entry(acpp_allocation_group *g, hipStream_t stream, uint32_t count, const T *const *inputs,
                  uint64_t n, T *const *outs, const acpp_algorithm_op *op_codes, const T *identities,
                  const int *init_flags, const acpp_launch_config *cfg, const char *name) {
  using W = typename elem_traits<T>::work;
  if (!g) return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": scratch group is NULL");
  if (count < 1 || count > static_cast<uint32_t>(max_inputs))
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": count must be 1..4");
  if (!inputs || !outs || !op_codes || !init_flags)
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": NULL array argument");
  params<T> p{};
  p.count = static_cast<int>(count);
  p.n = n;
  bool any_init = false;
  for (uint32_t k = 0; k < count; ++k) {
    p.init_mode[k] = init_flags[k] ? (identities ? 2 : 1) : 0;
    p.identity[k] = identities ? elem_traits<T>::to_work(identities[k]) : W{};
    any_init = any_init || init_flags[k];
  }
  for (uint32_t k = 0; k < count; ++k) {
    const int op = op_codes[k];
    if (op < ops::op_plus || op > ops::op_logical_or)
      return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": unknown operator");
    if (std::is_floating_point_v<W> && op > ops::op_max)
      return set_error(ACPP_ERROR_UNSUPPORTED, std::string(name) + ": floating-point reductions take plus, "
                                                                   "multiply, min or max");
    if (!outs[k] || (n > 0 && !inputs[k]))
      return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": NULL input or output");
    p.in[k] = inputs[k];
    p.out[k] = outs[k];
    p.op[k] = op;
    p.first[k] = 0;
    while (p.in[p.first[k]] != p.in[k]) ++p.first[k];
  }
  uint32_t arrays = 0;  // distinct ones
  for (uint32_t k = 0; k < count; ++k) arrays += p.first[k] == static_cast<int>(k);
  int cus = 0;
  acpp_status st = enter_device(g, &cus);
  if (st != ACPP_SUCCESS) return st;
  if (n == 0) {
    // reduction_descriptor.hpp:36-53: with initialize_to_identity the output
    // is the identity; without it the output keeps its value.
    if (any_init) {
      hipLaunchKernelGGL(identity_kernel<T>, dim3(1), dim3(64), 0, stream, p);
      st = check_launch(name);
      if (st != ACPP_SUCCESS) return st;
    }
    return clear_error();
  }
  const uint32_t wg = (cfg && cfg->work_group_size) ? cfg->work_group_size : 512;
  if (!valid_work_group_size(wg))
    return set_error(ACPP_ERROR_INVALID_ARGUMENT, std::string(name) + ": bad work_group_size");
  // Non-temporal loads once the inputs are larger than the 256 MiB
  // last-level cache, as for the plain reductions.
  const bool nt = static_cast<uint64_t>(arrays) * n * sizeof(T) >= (256ull << 20);
  // Arrays that the last-level cache holds are read again sooner than folded for
  // all at once (int64 in three reductions, 32 MB 15.8 and 17.4 us, 400 MB 169
  // and 77 us; int32 in two, 4 MB 8.2 and 9.0 us, 200 MB 57 and 37 us), and the
  // fold of 1-byte elements costs more than a second read (2^28 int8 in two 82
  // and 90 us, in four 165 and 144 us).
  const bool shared = arrays < count && n * sizeof(T) >= (48ull << 20) && (sizeof(T) > 1 || count - arrays >= 2);
  auto kernel = shared ? (nt ? shared_kernel<T, true> : shared_kernel<T, false>)
                       : (nt ? multi_kernel<T, true> : multi_kernel<T, false>);
  int resident = 1;
  st = occupancy(kernel, static_cast<int>(wg), &resident);
  if (st != ACPP_SUCCESS) return st;
  const uint32_t gpc = (cfg && cfg->groups_per_cu) ? cfg->groups_per_cu : 1;
  const uint64_t cap = static_cast<uint64_t>(std::min<uint32_t>(gpc, static_cast<uint32_t>(resident))) * cus;
  constexpr int VEC = 16 / sizeof(T);
  const uint64_t needed = ceil_div(ceil_div(n, static_cast<uint64_t>(VEC)), static_cast<uint64_t>(wg) * unroll);
  const uint32_t grid = static_cast<uint32_t>(std::max<uint64_t>(1, std::min(cap, needed)));
  const size_t used = sizeof(sync_header) + static_cast<size_t>(grid) * count * partial_slot_words * sizeof(uint64_t);
  void *region = nullptr;
  size_t cap_bytes = 0;
  region_state *rs = nullptr;
  st = group_obtain_sync(g, used, stream, &region, &cap_bytes, &rs);
  if (st != ACPP_SUCCESS) return st;
  region_launch rl;
  st = begin_region_launch(g, region, used, cap_bytes, rs, stream, &rl);
  if (st != ACPP_SUCCESS) return st;
  p.sync = static_cast<sync_header *>(region);
  p.partials = reinterpret_cast<uint64_t *>(static_cast<char *>(region) + sizeof(sync_header));
  p.epoch = rl.epoch;
  p.force_give_up = (cfg && (cfg->flags & ACPP_VARIANT_FORCE_GIVE_UP)) ? 1 : 0;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(wg), 0, stream, p);
  st = check_launch(name);
  end_region_launch(rs, rl, 0, st);
  return st == ACPP_SUCCESS ? clear_error() : st;
}

}  // namespace multi_detail
}  // namespace acpp_impl

using namespace acpp_impl;

extern "C" {

#define ACPP_DEFINE_MULTI(tag, T)                                                                       \
  acpp_status acpp_reduction_multi_##tag(acpp_allocation_group *scratch, acpp_stream_t stream,         \
                                         uint32_t count, const T *const *inputs, uint64_t n,           \
                                         T *const *outs, const acpp_algorithm_op *ops,                 \
                                         int initialize_to_identity, const acpp_launch_config *config) { \
    const int flags[multi_detail::max_inputs] = {initialize_to_identity, initialize_to_identity,       \
                                                 initialize_to_identity, initialize_to_identity};      \
    return multi_detail::entry<T>(scratch, static_cast<hipStream_t>(stream), count, inputs, n, outs, ops, \
                                  nullptr, flags, config, "acpp_reduction_multi_" #tag);               \
  }                                                                                                     \
  acpp_status acpp_reduction_multi_identity_##tag(                                                     \
      acpp_allocation_group *scratch, acpp_stream_t stream, uint32_t count, const T *const *inputs,    \
      uint64_t n, T *const *outs, const acpp_algorithm_op *ops, const T *identities,                   \
      const int *initialize_to_identity, const acpp_launch_config *config) {                           \
    return multi_detail::entry<T>(scratch, static_cast<hipStream_t>(stream), count, inputs, n, outs, ops, \
                                  identities, initialize_to_identity, config,                          \
                                  "acpp_reduction_multi_identity_" #tag);                             \
  }
ACPP_DEFINE_MULTI(i8, int8_t)
ACPP_DEFINE_MULTI(u8, uint8_t)
ACPP_DEFINE_MULTI(i16, int16_t)
ACPP_DEFINE_MULTI(u16, uint16_t)
ACPP_DEFINE_MULTI(i32, int32_t)
ACPP_DEFINE_MULTI(u32, uint32_t)
ACPP_DEFINE_MULTI(i64, int64_t)
ACPP_DEFINE_MULTI(u64, uint64_t)
ACPP_DEFINE_MULTI(f32, float)
ACPP_DEFINE_MULTI(f64, double)

}  // extern "C"
