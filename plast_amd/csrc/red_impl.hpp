// red_impl.hpp — the reduction engine.
//
// A reduction problem is a Space whose last operand is the target: the target has stride 0 on
// every reduced axis. After collapsing, one of three kernel families runs:
//   rows   — the innermost axis is reduced and unit-stride: one wave64 per (row, segment), float4
//            loads, wave shuffle reduction; long rows split into segments whose partials a finalize
//            pass combines in order;
//   cols   — the innermost axis is kept and unit-stride: each lane owns four adjacent outputs (or
//            one, or a share of the flat array of narrow rows: launch_rules.hpp) and walks its chunk
//            of the reduced axis in order; chunks combine in order in a finalize pass (no atomics
//            anywhere, so results are deterministic);
//            With further reduced axes outside (a bias gradient over batch and space, say), both
//            (the columns for plain sums alone) walk the flattened reduced index: lexicographic over
//            the reduced axes, the innermost one in runs of its extent (MULTI kernels;
//            reduced_offset decodes it). The generic kernel's one lane per output took 32.6 ms for
//            config 3's B gradient (512 outputs of 131072 terms, 268 MB); config 3's training graph
//            went from 33.9 to 0.55 ms;
//   generic— any layout: one lane per output, serial walk in index order.
//
// Max/min reproduce the reference's literal fold `acc > x ? acc : x` from -FLT_MAX
// (reduce_ops.c:9, 26-30) bit for bit, including NaN (a NaN resets the fold: the result is the
// fold of what follows the last NaN) and signed zeros (ties keep the later element). Per index
// range the fold is summarised as (r, flags): r is the fold started at the range's first element,
// INDEP set when the range contains a NaN (then the range's result does not depend on what came
// before). Ranges combine in index order.
#pragma once

#include <cfloat>
#include <type_traits>

#include "common.hpp"

namespace plast {

// ------------------------------------------------------------------------- producers
// A producer turns the NIN operand values at one point of the space into the reduced value.

// A producer with kStore = true also writes its values out, at operand 0's offsets from its `dst`
// (the leading-axis kernel only; launch_reduction launches nothing and returns false for any other
// layout). Producers without the member do not store.
template <class P, class = void>
struct StoresValues : std::false_type {};
template <class P>
struct StoresValues<P, std::void_t<decltype(P::kStore)>> : std::bool_constant<P::kStore> {};
template <class P>
constexpr bool kStores = StoresValues<P>::value;

struct Load1 {
  static constexpr int NIN = 1;
  __device__ __forceinline__ float eval(const float *v) const { return v[0]; }
};

// 1 where a == e (e broadcast from the forward output), else 0: tie count of max/min backward.
struct EqualCount {
  static constexpr int NIN = 2;
  __device__ __forceinline__ float eval(const float *v) const { return v[0] == v[1] ? 1.0f : 0.0f; }
};

// dout * (z > 0 ? 1 : alpha), stored to dst as it is summed: the relu-gradient modulation of the
// fused matmul epilogues' backward (matmul_relu.cu:138-144) fused with the bias-gradient sum.
struct ReluGradStore {
  static constexpr int NIN = 2;
  static constexpr bool kStore = true;
  float alpha;
  float *dst;
  __device__ __forceinline__ float eval(const float *v) const {
    return v[0] * (v[1] > 0.0f ? 1.0f : alpha);
  }
};

// The gradient a fused leaky_relu(x + bias) node hands to its ADD, for the operands (dout, y):
// 0 + dout * (y > 0 ? 1 : alpha), the chain's leaky backward (unary_ops.c:236-258) accumulated into
// the intermediate's zeroed gradient, with its mask read from the node's output y (for alpha >= 0,
// y > 0 exactly where x + bias > 0). Summed over rows: the bias's gradient.
struct LeakyAddGrad {
  static constexpr int NIN = 2;
  float alpha;
  __device__ __forceinline__ float eval(const float *v) const {
    return 0.0f + v[0] * (v[1] > 0.0f ? 1.0f : alpha);
  }
};

// The same term for the operands (dout, y, g), summed, with g + term stored to dst (g's own
// buffer): x's gradient from the ADD's backward (kernel_macros.h:283-299) written in the pass that
// sums the bias's. A refold recomputes its terms from dout and y, which the stores leave intact.
struct LeakyAddGradStore {
  static constexpr int NIN = 3;
  static constexpr bool kStore = true;
  static constexpr bool kRefoldInputs = true;
  float alpha;
  float *dst;
  __device__ __forceinline__ float eval(const float *v) const {
    return 0.0f + v[0] * (v[1] > 0.0f ? 1.0f : alpha);
  }
  __device__ __forceinline__ float stored(const float *v, float y) const { return v[2] + y; }
};

// What a storing producer writes for the value y it sums at operands v: y itself, or, for one
// with kRefoldInputs, its own stored(v, y).
template <class P, class = void>
struct StoresOther : std::false_type {};
template <class P>
struct StoresOther<P, std::void_t<decltype(P::kRefoldInputs)>> : std::bool_constant<P::kRefoldInputs> {};
template <class P>
__device__ __forceinline__ float stored_value(const P &prod, const float *v, float y) {
  if constexpr (StoresOther<P>::value) return prod.stored(v, y);
  else return y;
}

// ------------------------------------------------------------------------- combiners

enum class Post : int { Write = 0, Mean = 1, Accum = 2 };

struct SumComb {
  using Part = float;
  using Out = float;
  static constexpr bool kExact = false;
  __device__ static Part empty() { return 0.0f; }
  // the reference's accumulator starts at 0.0f, so a lone -0 sums to +0
  __device__ static void first(Part &p, float x, int64_t) { p = 0.0f + x; }
  __device__ static void next(Part &p, float x, int64_t) { p = p + x; }
  __device__ static Part merge(Part a, Part b) { return a + b; }
  __device__ static Part shfl(Part p, int m) { return __shfl_xor(p, m); }
};

// Exact max (IS_MAX) / min fold summaries.
constexpr uint32_t kIndep = 1, kNonEmpty = 2;
struct ExtPart {
  float r;
  uint32_t flags;
};

template <bool IS_MAX>
struct ExtComb {
  using Part = ExtPart;
  using Out = float;
  static constexpr bool kExact = true;
  __device__ static float pick(float acc, float x) {
    if constexpr (IS_MAX) return acc > x ? acc : x;
    else return acc < x ? acc : x;
  }
  __device__ static float init() { return IS_MAX ? -FLT_MAX : FLT_MAX; }
  __device__ static Part empty() { return Part{0.0f, 0u}; }
  __device__ static void first(Part &p, float x, int64_t) {
    p.r = x;
    p.flags = kNonEmpty | (x != x ? kIndep : 0u);
  }
  __device__ static void next(Part &p, float x, int64_t) {
    p.r = pick(p.r, x);
    if (x != x) p.flags |= kIndep;
  }
  // a covers earlier indices than b
  __device__ static Part merge(Part a, Part b) {
    if (!(b.flags & kNonEmpty)) return a;
    if (!(a.flags & kNonEmpty) || (b.flags & kIndep)) return b;
    return Part{pick(a.r, b.r), a.flags};
  }
  // value of the reference's accumulator after folding the whole summarised range from init
  __device__ static float finish(Part p) {
    if (!(p.flags & kNonEmpty)) return init();
    if (p.flags & kIndep) return p.r;
    return pick(init(), p.r);
  }
};

// numpy argmax: first NaN if any, else first index of the maximum.
struct ArgPart {
  float v;
  int64_t i;
};
struct ArgmaxComb {
  using Part = ArgPart;
  using Out = int64_t;
  static constexpr bool kExact = false;
  __device__ static Part empty() { return Part{-__builtin_huge_valf(), INT64_MAX}; }
  // Order-free: the better of two (value, index) candidates.
  __device__ static Part merge(Part a, Part b) {
    const bool an = a.v != a.v, bn = b.v != b.v;
    if (an || bn) {
      if (an && bn) return a.i < b.i ? a : b;
      return an ? a : b;
    }
    if (a.v > b.v) return a;
    if (b.v > a.v) return b;
    return a.i < b.i ? a : b;
  }
  __device__ static void first(Part &p, float x, int64_t k) { p = Part{x, k}; }
  __device__ static void next(Part &p, float x, int64_t k) { p = merge(p, Part{x, k}); }
  __device__ static Part shfl(Part p, int m) {
    Part q;
    q.v = __shfl_xor(p.v, m);
    q.i = __shfl_xor(p.i, m);
    return q;
  }
};

// ------------------------------------------------------------------------- arguments

template <int NIN>
struct RedArgs {
  static constexpr bool kMulti = false;
  const float *in[NIN];
  void *out;
  int64_t ost[NIN][kMaxRank];  // operand strides on the kept (output) axes, innermost excluded
  int64_t tst[kMaxRank];       // target strides on the same axes
  MagicDiv dv[kMaxRank];       // extents of those axes
  int nouter;                  // number of such axes
  int64_t rst[NIN];            // operand strides along the reduced axis
  int64_t kst[NIN];            // operand strides along the kept innermost axis (cols)
  int64_t tkst;                // target stride along the kept innermost axis (cols)
  uint64_t len;                // reduced extent (all reduced axes together)
  uint64_t rows;               // rows (rows kernel) / outer count (cols kernel)
  uint64_t inner;              // kept innermost extent (cols kernel)
  uint32_t lanes;              // lanes of a wave that hold columns (cols kernel)
  uint32_t segs;               // segments per row / chunks of the reduced axis
  uint64_t seglen;
  uint32_t vec_mask;           // bit k: operand k is streamed with float4 loads (else splat)
  void *part;                  // partial summaries [segs][outputs] when segs > 1
  int post;                    // Post
  float divisor;               // Mean
};

// The same with further reduced axes outside the innermost reduced one (the MULTI kernels'). A type of
// its own: the serial refolds of every other reduction need not ask for each element whether such
// axes are there (min over the leading axis of [4096, 1024] with a zero in every column: 63 us, 72
// asking).
template <int NIN>
struct RedMultiArgs : RedArgs<NIN> {
  static constexpr bool kMulti = true;
  int nx;                      // number of those axes
  MagicDiv drun;               // extent of the innermost reduced axis
  MagicDiv dunits;             // float4 units of one run of it, the last one partial
  uint64_t vlen;               // 4 * the units of every run (what the rows kernel with VEC segments)
  MagicDiv xdv[kMaxRank];      // extents of the outer reduced axes, outermost first
  int64_t xst[NIN][kMaxRank];  // operand strides along them
};
template <int NIN, bool MULTI>
using RedArgsOf = typename std::conditional<MULTI, RedMultiArgs<NIN>, RedArgs<NIN>>::type;

// Outer-axis decode: index -> per-operand base offsets and the target offset.
template <int NIN>
__device__ __forceinline__ void decode_outer(const RedArgs<NIN> &A, uint32_t idx, int64_t *base,
                                             int64_t &tbase) {
#pragma unroll
  for (int k = 0; k < NIN; ++k) base[k] = 0;
  tbase = 0;
  for (int d = A.nouter - 1; d >= 0; --d) {
    const uint32_t nxt = A.dv[d].div(idx);
    const int64_t c = int64_t(idx - nxt * A.dv[d].d);
    idx = nxt;
#pragma unroll
    for (int k = 0; k < NIN; ++k) base[k] += c * A.ost[k][d];
    tbase += c * A.tst[d];
  }
}

template <class Comb>
__device__ __forceinline__ void store_final(void *out, int64_t off, const typename Comb::Part &p,
                                            int post, float divisor) {
  if constexpr (std::is_same<Comb, ArgmaxComb>::value) {
    static_cast<int64_t *>(out)[off] = p.i == INT64_MAX ? 0 : p.i;
  } else if constexpr (Comb::kExact) {
    static_cast<float *>(out)[off] = Comb::finish(p);
  } else {
    float *o = static_cast<float *>(out);
    if (post == int(Post::Accum)) o[off] = o[off] + p;
    else if (post == int(Post::Mean)) o[off] = p / divisor;
    else o[off] = p;
  }
}

// ------------------------------------------------------------------------- rows kernel

// Offset of the i-th reduced position in every operand: i * rst for one reduced axis, else the
// coordinates of flattened index i over the outer reduced axes and the position in the innermost
// one's run (the space has fewer than 2^32 elements there).
template <int NIN, class Args>
__device__ __forceinline__ void reduced_offset(const Args &A, uint64_t i, int64_t *off) {
  if constexpr (!Args::kMulti) {
#pragma unroll
    for (int k = 0; k < NIN; ++k) off[k] = int64_t(i) * A.rst[k];
  } else {
    uint32_t x = A.drun.div(uint32_t(i));
    const int64_t pos = int64_t(uint32_t(i) - x * A.drun.d);
#pragma unroll
    for (int k = 0; k < NIN; ++k) off[k] = pos * A.rst[k];
    for (int d = A.nx - 1; d > 0; --d) {
      const uint32_t nxt = A.xdv[d].div(x);
      const int64_t c = int64_t(x - nxt * A.xdv[d].d);
      x = nxt;
#pragma unroll
      for (int k = 0; k < NIN; ++k) off[k] += c * A.xst[k][d];
    }
#pragma unroll
    for (int k = 0; k < NIN; ++k) off[k] += int64_t(x) * A.xst[k][0];
  }
}

// The i-th term of a serial refold. A storing producer's terms are read back from where it stored
// them (only a sum over a leading axis refolds one, after its workgroup or launch has stored every
// term of the column): its inputs may have been overwritten by those stores (dc written over
// dout). One with kRefoldInputs stores something other than its terms, over none of the operands
// its terms read, and recomputes them.
template <class Prod, class Args>
__device__ __forceinline__ float value_at(const Args &A, const Prod &prod, const int64_t *base,
                                          uint64_t i) {
  constexpr int NIN = Prod::NIN;
  int64_t off[NIN];
  reduced_offset<NIN>(A, i, off);
  if constexpr (kStores<Prod> && !StoresOther<Prod>::value) {
    return prod.dst[base[0] + off[0]];
  } else {
    float v[NIN];
#pragma unroll
    for (int k = 0; k < NIN; ++k) v[k] = A.in[k][base[k] + off[k]];
    return prod.eval(v);
  }
}

template <class T>
__device__ __forceinline__ T wave_max_t(T v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    T o = __shfl_xor(v, m);
    v = o > v ? o : v;
  }
  return v;
}
__device__ __forceinline__ float wave_fmax(float v, bool is_max) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    float o = __shfl_xor(v, m);
    v = is_max ? fmaxf(v, o) : fminf(v, o);
  }
  return v;
}
__device__ __forceinline__ bool wave_any(bool b) { return __any(b); }

// Exact fold summary of [b, e) by one wave, used when the fast path saw a NaN or a zero extreme.
template <bool IS_MAX, class Prod, class Args>
__device__ ExtPart exact_range(const Args &A, const Prod &prod, const int64_t *base,
                               uint64_t b, uint64_t e, int lane) {
  // last NaN
  int64_t last_nan = -1;
  for (uint64_t i = b + lane; i < e; i += 64) {
    const float x = value_at(A, prod, base, i);
    if (x != x) last_nan = int64_t(i);
  }
  last_nan = wave_max_t(last_nan);
  const uint64_t s = last_nan >= 0 ? uint64_t(last_nan) + 1 : b;
  if (s >= e) {
    // the range ends in a NaN: the fold's value is that NaN
    return ExtPart{value_at(A, prod, base, uint64_t(last_nan)), kNonEmpty | kIndep};
  }
  float m = IS_MAX ? -__builtin_huge_valf() : __builtin_huge_valf();
  for (uint64_t i = s + lane; i < e; i += 64) {
    const float x = value_at(A, prod, base, i);
    m = IS_MAX ? fmaxf(m, x) : fminf(m, x);
  }
  m = wave_fmax(m, IS_MAX);
  float r = m;
  if (m == 0.0f) {
    // several zeros may tie: the fold keeps the last one, whose sign decides the bits
    int64_t last_zero = -1;
    for (uint64_t i = s + lane; i < e; i += 64)
      if (value_at(A, prod, base, i) == 0.0f) last_zero = int64_t(i);
    last_zero = wave_max_t(last_zero);
    r = value_at(A, prod, base, uint64_t(last_zero));
  }
  return ExtPart{r, kNonEmpty | (last_nan >= 0 ? kIndep : 0u)};
}

// A parallel-order sum that is not finite (an overflow, or inf - inf) can differ from the
// reference's serial one, whose outcome depends on the order: such an output is summed again in
// the reference's order (index order from 0.0f, one rounding per addition: reduce_ops.c:57-61).
template <class Comb>
constexpr bool kSerialSum = std::is_same<Comb, SumComb>::value;

__device__ __forceinline__ bool finite_sum(float p) { return fabsf(p) <= FLT_MAX; }

// By one lane: the serial sum of elements [0, len) at base.
template <class Prod, class Args>
__device__ float serial_sum_lane(const Args &A, const Prod &prod, const int64_t *base,
                                 uint64_t len) {
  float s = 0.0f;
  for (uint64_t i = 0; i < len; ++i) s = s + value_at(A, prod, base, i);
  return s;
}

// By a wave, for a whole row: a NaN operand makes every order's sum NaN, so the wave first looks
// for one (in parallel) and only a row without one is refolded, by lane 0; every lane returns the
// result.
template <class Prod, class Args>
__device__ float serial_sum_wave(const Args &A, const Prod &prod, const int64_t *base,
                                 uint64_t len, float p, int lane) {
  bool nan = false;
  for (uint64_t i = lane; i < len; i += 64) {
    const float x = value_at(A, prod, base, i);
    nan = nan || (x != x);
  }
  if (__any(nan)) return p;
  float r = 0.0f;
  if (lane == 0) r = serial_sum_lane(A, prod, base, len);
  return __shfl(r, 0);
}

constexpr int kRowUnroll = PLAST_ROW_UNROLL;  // float4 loads in flight per lane per operand

// The float4 unit at reduced position i (a multiple of 4) of every operand, a broadcast operand's
// value splatted. MULTI: i / 4 counts units of runs whose last unit may be partial; that one is read
// from four elements before the run's end. Returns the reduced index of the unit's first element;
// the first `skip` elements belong to the unit before.
template <int NIN, class Args>
__device__ __forceinline__ uint64_t load_unit(const Args &A, const int64_t *base, uint64_t i, f4 *x,
                                              uint32_t &skip) {
  constexpr bool MULTI = Args::kMulti;
  int64_t off[NIN];
  if constexpr (MULTI) {
    const uint32_t run = A.dunits.div(uint32_t(i / 4));
    const uint32_t at = 4 * (uint32_t(i / 4) - run * A.dunits.d);
    const uint32_t pos = at + 4 <= A.drun.d ? at : A.drun.d - 4;
    skip = at - pos;
    i = uint64_t(run) * A.drun.d + pos;
    reduced_offset<NIN>(A, i, off);
  } else {
    skip = 0;
  }
#pragma unroll
  for (int k = 0; k < NIN; ++k) {
    const float *src = A.in[k] + base[k];
    if (A.vec_mask >> k & 1u)
      x[k] = __builtin_nontemporal_load(
          reinterpret_cast<const f4u *>(src + (MULTI ? off[k] : int64_t(i))));
    else
      x[k] = f4(src[MULTI ? off[k] : 0]);
  }
  return i;
}

// The reduced index at which MULTI position i (a multiple of 4) starts.
template <int NIN>
__device__ __forceinline__ uint64_t run_index(const RedMultiArgs<NIN> &A, uint64_t i) {
  const uint32_t run = A.dunits.div(uint32_t(i / 4));
  return uint64_t(run) * A.drun.d + 4 * (uint32_t(i / 4) - run * A.dunits.d);
}

template <class Prod, class Comb, bool VEC, bool MULTI>
__global__ __launch_bounds__(kBlock) void red_rows_kernel(RedArgsOf<Prod::NIN, MULTI> A, Prod prod) {
  constexpr int NIN = Prod::NIN;
  using Part = typename Comb::Part;
  const int lane = threadIdx.x & 63;
  const uint32_t bx = blockIdx.x;
  const uint64_t task = uint64_t(bx) * (kBlock / 64) + (threadIdx.x >> 6);
  if (task >= A.rows * A.segs) return;  // whole wave exits together
  const uint32_t row = uint32_t(task / A.segs);
  const uint32_t seg = uint32_t(task - uint64_t(row) * A.segs);
  int64_t base[NIN], tbase;
  decode_outer(A, row, base, tbase);
  const uint64_t b = uint64_t(seg) * A.seglen;
  uint64_t total = A.len;
  if constexpr (VEC && MULTI) total = A.vlen;
  const uint64_t e = b + A.seglen < total ? b + A.seglen : total;
  // end of the whole float4 units; the up to three elements left are lanes 0 to 2's
  const uint64_t eu = MULTI ? e : e - (e & 3);

  Part p;
  if constexpr (Comb::kExact) {
    // fast path: plain extreme ignoring NaN, plus a NaN flag
    constexpr bool IS_MAX = std::is_same<Comb, ExtComb<true>>::value;
    float m = IS_MAX ? -__builtin_huge_valf() : __builtin_huge_valf();
    bool nan = false;
    auto take = [&](float x) {
      m = IS_MAX ? fmaxf(m, x) : fminf(m, x);
      nan = nan || (x != x);
    };
    if constexpr (VEC) {
      for (uint64_t i0 = b + uint64_t(lane) * 4; i0 < eu; i0 += 256 * kRowUnroll) {
        f4 x[kRowUnroll][NIN];
        uint64_t at[kRowUnroll];
        uint32_t skip[kRowUnroll];
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) {
          const uint64_t i = i0 + uint64_t(u) * 256;
          if (i < eu) at[u] = load_unit<NIN>(A, base, i, x[u], skip[u]);
        }
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) {
          if (i0 + uint64_t(u) * 256 >= eu) continue;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            if (MULTI && uint32_t(c) < skip[u]) continue;
            float v[NIN];
#pragma unroll
            for (int k = 0; k < NIN; ++k) v[k] = x[u][k][c];
            take(prod.eval(v));
          }
        }
      }
      if (!MULTI && eu + lane < e) take(value_at(A, prod, base, eu + lane));
    } else {
      for (uint64_t i = b + lane; i < e; i += 64) take(value_at(A, prod, base, i));
    }
    m = wave_fmax(m, IS_MAX);
    nan = wave_any(nan);
    if (!nan && m != 0.0f) {
      p = ExtPart{m, e > b ? kNonEmpty : 0u};
    } else if (e > b) {
      if constexpr (VEC && MULTI)
        p = exact_range<IS_MAX>(A, prod, base, run_index(A, b), run_index(A, e), lane);
      else
        p = exact_range<IS_MAX>(A, prod, base, b, e, lane);
    } else {
      p = Comb::empty();
    }
  } else {
    p = Comb::empty();
    Part acc[4] = {Comb::empty(), Comb::empty(), Comb::empty(), Comb::empty()};
    if constexpr (VEC) {
      for (uint64_t i0 = b + uint64_t(lane) * 4; i0 < eu; i0 += 256 * kRowUnroll) {
        f4 x[kRowUnroll][NIN];
        uint64_t at[kRowUnroll];
        uint32_t skip[kRowUnroll];
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) {
          const uint64_t i = i0 + uint64_t(u) * 256;
          if (i < eu) at[u] = load_unit<NIN>(A, base, i, x[u], skip[u]);
        }
#pragma unroll
        for (int u = 0; u < kRowUnroll; ++u) {
          if (i0 + uint64_t(u) * 256 >= eu) continue;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            if (MULTI && uint32_t(c) < skip[u]) continue;
            float v[NIN];
#pragma unroll
            for (int k = 0; k < NIN; ++k) v[k] = x[u][k][c];
            Comb::next(acc[c], prod.eval(v), int64_t(at[u] + c));
          }
        }
      }
      if (!MULTI && eu + lane < e)
        Comb::next(acc[0], value_at(A, prod, base, eu + lane), int64_t(eu + lane));
      p = Comb::merge(Comb::merge(acc[0], acc[1]), Comb::merge(acc[2], acc[3]));
    } else {
      for (uint64_t i = b + lane; i < e; i += 64) {
        Comb::next(p, value_at(A, prod, base, i), int64_t(i));
      }
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) p = Comb::merge(p, Comb::shfl(p, m));
    // every lane holds the row's sum: the check is uniform over the wave
    if constexpr (kSerialSum<Comb>)
      if (A.segs == 1 && !finite_sum(p)) p = serial_sum_wave(A, prod, base, A.len, p, lane);
  }

  if (lane != 0) return;
  if (A.segs == 1) {
    store_final<Comb>(A.out, tbase, p, A.post, A.divisor);
  } else {
    static_cast<Part *>(A.part)[task] = p;
  }
}

// Rows of at most 16 * L elements: L lanes per row, 64 / L rows per wave, so a wave reads one
// contiguous stretch of rows (a wave per row of 77 floats kept 20 of its 64 lanes on 308 bytes, and
// took 15 us for 15 MB). Each lane holds up to four float4 units of its row, all loaded before the
// first is used, and the up to three elements left. A row whose fast value could differ from the
// reference's (max/min of a NaN or a zero extreme, a non-finite sum) is redone by its own lanes, from
// the same registers: min of [1000, 100] with a zero in every row 16.9 us with a wave's rows redone
// one after the other, 4.4 with a wave per row.
template <class Prod, class Comb, int L>
__global__ __launch_bounds__(kBlock) void red_rows_short_kernel(RedArgs<Prod::NIN> A, Prod prod) {
  constexpr int NIN = Prod::NIN, U = 4;
  using Part = typename Comb::Part;
  const int lane = threadIdx.x & 63, l = lane % L;
  const uint64_t row0 = (uint64_t(blockIdx.x) * (kBlock / 64) + (threadIdx.x >> 6)) * (64 / L);
  if (row0 >= A.rows) return;  // whole wave
  const uint64_t row = row0 + lane / L;
  const bool valid = row < A.rows;
  int64_t base[NIN], tbase;
  decode_outer(A, uint32_t(valid ? row : A.rows - 1), base, tbase);
  const uint32_t len = uint32_t(A.len), units = len / 4;
  f4 x[U][NIN];
  if (units) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // a lane past the row reads its last unit: the loads take no branch
      const uint32_t q = uint32_t(l) + u * L;
      uint32_t skip;
      load_unit<NIN>(A, base, uint64_t(q < units ? q : units - 1) * 4, x[u], skip);
    }
  }
  const auto each = [&](auto &&take) {
    if (units) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t q = uint32_t(l) + u * L;
        if (q >= units) continue;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          float v[NIN];
#pragma unroll
          for (int k = 0; k < NIN; ++k) v[k] = x[u][k][c];
          take(c, prod.eval(v), int64_t(q * 4 + c));
        }
      }
    }
    for (uint32_t i = units * 4 + l; i < len; i += L)
      take(0, value_at(A, prod, base, i), int64_t(i));
  };
  Part p = Comb::empty();
  bool redo;
  if constexpr (Comb::kExact) {
    constexpr bool IS_MAX = std::is_same<Comb, ExtComb<true>>::value;
    float m = IS_MAX ? -__builtin_huge_valf() : __builtin_huge_valf();
    uint32_t nan = 0;
    each([&](int, float y, int64_t) {
      m = IS_MAX ? fmaxf(m, y) : fminf(m, y);
      nan |= y != y ? 1u : 0u;
    });
#pragma unroll
    for (int s = L / 2; s >= 1; s >>= 1) {
      const float o = __shfl_xor(m, s);
      m = IS_MAX ? fmaxf(m, o) : fminf(m, o);
      nan |= uint32_t(__shfl_xor(int(nan), s));
    }
    p = ExtPart{m, kNonEmpty};
    redo = nan != 0 || m == 0.0f;
  } else {
    Part acc[4] = {Comb::empty(), Comb::empty(), Comb::empty(), Comb::empty()};
    each([&](int c, float y, int64_t i) { Comb::next(acc[c], y, i); });
    p = Comb::merge(Comb::merge(acc[0], acc[1]), Comb::merge(acc[2], acc[3]));
#pragma unroll
    for (int s = L / 2; s >= 1; s >>= 1) p = Comb::merge(p, Comb::shfl(p, s));
    redo = false;
    if constexpr (kSerialSum<Comb>) redo = !finite_sum(p);
  }
  if (__any(redo && valid)) {  // every row of the wave at once, each by its own lanes
    if constexpr (Comb::kExact) {
      constexpr bool IS_MAX = std::is_same<Comb, ExtComb<true>>::value;
      const auto group_last = [](int v) {
#pragma unroll
        for (int s = L / 2; s >= 1; s >>= 1) {
          const int o = __shfl_xor(v, s);
          v = o > v ? o : v;
        }
        return v;
      };
      int last_nan = -1;
      each([&](int, float y, int64_t i) {
        if (y != y && int(i) > last_nan) last_nan = int(i);
      });
      last_nan = group_last(last_nan);
      // the extreme after the last NaN, and the last zero there (its index and sign)
      float m = IS_MAX ? -__builtin_huge_valf() : __builtin_huge_valf();
      int zero = -1;
      each([&](int, float y, int64_t i) {
        if (int(i) <= last_nan) return;
        m = IS_MAX ? fmaxf(m, y) : fminf(m, y);
        const int key = 2 * int(i) + int(__float_as_uint(y) >> 31);
        if (y == 0.0f && key > zero) zero = key;
      });
#pragma unroll
      for (int s = L / 2; s >= 1; s >>= 1) {
        const float o = __shfl_xor(m, s);
        m = IS_MAX ? fmaxf(m, o) : fminf(m, o);
      }
      zero = group_last(zero);
      if (redo) {
        p = ExtPart{m == 0.0f ? (zero & 1 ? -0.0f : 0.0f) : m, kNonEmpty | (last_nan >= 0 ? kIndep : 0u)};
        // a row that ends in a NaN: the fold's value is that NaN
        if (last_nan == int(len) - 1) p.r = value_at(A, prod, base, uint64_t(last_nan));
      }
    } else if constexpr (kSerialSum<Comb>) {
      uint32_t nan = 0;  // a NaN term makes every order's sum NaN
      each([&](int, float y, int64_t) { nan |= y != y ? 1u : 0u; });
#pragma unroll
      for (int s = L / 2; s >= 1; s >>= 1) nan |= uint32_t(__shfl_xor(int(nan), s));
      if (redo && !nan && l == 0) p = serial_sum_lane(A, prod, base, A.len);
    }
  }
  if (l == 0 && valid) store_final<Comb>(A.out, tbase, p, A.post, A.divisor);
}

// Combine the segments of each row in index order.
// Merge segs partials part[0], part[stride], ... in index order. The loads of a batch are issued
// before its merges: the partials come from L2 or HBM, and a serial load-merge chain would pay
// that latency once per partial (a [16384, 4096] column sum split in 64 chunks spent most of
// its time in that chain).
template <class Comb>
__device__ __forceinline__ typename Comb::Part merge_in_order(const typename Comb::Part *part,
                                                              uint64_t stride, uint32_t segs) {
  using Part = typename Comb::Part;
  constexpr uint32_t kBatch = 16;
  // whole batches of loads, the last one clamped to the final partial (loaded, not merged): a
  // partial batch of one-at-a-time loads would wait out a memory latency per partial
  Part p{};
  for (uint32_t s = 0; s < segs; s += kBatch) {
    Part q[kBatch];
#pragma unroll
    for (uint32_t i = 0; i < kBatch; ++i) {
      const uint32_t k = s + i < segs ? s + i : segs - 1;
      q[i] = part[uint64_t(k) * stride];
    }
#pragma unroll
    for (uint32_t i = 0; i < kBatch; ++i) {
      if (s + i == 0) p = q[0];
      else if (s + i < segs) p = Comb::merge(p, q[i]);
    }
  }
  return p;
}

// Any trivially copyable summary, moved `off` lanes down the wave word by word.
template <class P>
__device__ __forceinline__ P shfl_down_part(const P &p, int off) {
  static_assert(sizeof(P) % 4 == 0, "summaries are whole words");
  P q;
  const int *src = reinterpret_cast<const int *>(&p);
  int *dst = reinterpret_cast<int *>(&q);
#pragma unroll
  for (int w = 0; w < int(sizeof(P) / 4); ++w) dst[w] = __shfl_down(src[w], off);
  return q;
}

// One wave per row: lane l merges the l-th run of consecutive partials in index order, then the
// runs merge pairwise, always earlier run on the left (every combiner's merge is associative over
// ordered ranges; for sums this fixes a different, still deterministic, rounding order than one
// serial pass). A row of 4096 partials took one thread 50 us to merge serially.
template <class Prod, class Comb, class Args>
__global__ __launch_bounds__(kBlock) void red_rows_finalize(Args A, Prod prod) {
  using Part = typename Comb::Part;
  constexpr int NIN = Prod::NIN;
  const int lane = threadIdx.x & 63;
  const uint64_t row = uint64_t(blockIdx.x) * (kBlock / 64) + (threadIdx.x >> 6);
  if (row >= A.rows) return;  // whole wave
  const Part *part = static_cast<const Part *>(A.part) + row * A.segs;
  const uint32_t run = (A.segs + 63) / 64;
  const uint32_t active = (A.segs + run - 1) / run;  // lanes holding a non-empty run
  const uint32_t s0 = uint32_t(lane) * run;
  Part p = Comb::empty();
  if (uint32_t(lane) < active) {
    const uint32_t n = A.segs - s0 < run ? A.segs - s0 : run;
    p = merge_in_order<Comb>(part + s0, 1, n);
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const Part q = shfl_down_part(p, off);
    if ((lane & (2 * off - 1)) == 0 && uint32_t(lane + off) < active) p = Comb::merge(p, q);
  }
  int64_t base[NIN], tbase;
  decode_outer(A, uint32_t(row), base, tbase);
  if constexpr (kSerialSum<Comb>) {
    p = __shfl(p, 0);  // lane 0 holds the row's sum
    if (!finite_sum(p)) p = serial_sum_wave(A, prod, base, A.len, p, lane);
  }
  if (lane != 0) return;
  store_final<Comb>(A.out, tbase, p, A.post, A.divisor);
}

// ------------------------------------------------------------------------- cols kernel

template <class Prod>
constexpr int kColUnroll = Prod::NIN == 1   ? PLAST_COL_UNROLL
                           : Prod::NIN == 2 && kStores<Prod> ? PLAST_COL_UNROLL2
                                            : PLAST_COL_UNROLL3;

template <class Prod>
__device__ __forceinline__ void store_col(float *p, f4 v) {
  store_unit<PLAST_COL_NT_STORE == 1 || (PLAST_COL_NT_STORE == -1 && StoresOther<Prod>::value)>(v, p);
}

template <class Prod>
constexpr int kColMinRows = Prod::NIN >= 3 ? PLAST_COL_MIN_ROWS3 : 64;
// Float4 columns a workgroup of the small kernel owns, and the rows a lane loads per batch: producers
// of three operands take one column, those of one and storing ones of two take two, and two
// operands one over narrow rows (the gradient of a multiplied [128, 64] 4.3 us, 4.6 with two) and two
// over wide ones ([512, 4096] 5.7 us, 7.4 with one).
template <class Prod>
inline bool col_small_one(uint64_t inner) {
  return Prod::NIN >= 3 || (Prod::NIN == 2 && !kStores<Prod> && inner < 512);
}

// Fast summary of an order-sensitive fold (exact max/min): the plain extreme and a NaN flag.
struct ExtFast {
  float m;
  uint32_t nan;
};

// grid.x: (outer index, slice of 64 lanes x W columns of the kept innermost axis); grid.y: chunk
// of the reduced axis. The workgroup's four waves take interleaved rows of the chunk (wave w reads
// rows k0 + w, k0 + w + 4, ...), so each wave streams its own rows while the workgroup still
// covers one contiguous slice per row; each lane owns W adjacent columns. The four partials of a
// column combine through LDS in wave order (deterministic). Order-free combiners (sum, argmax)
// merge directly. The exact max/min fold keeps a plain extreme and a NaN flag per wave, and a
// column is refolded serially in index order only when its chunk holds a NaN or its extreme is
// zero (the cases where order decides the bits).
// ALLV (with VEC): every operand is streamed with float4 loads, so the loads take no branch on
// the operand mask (a broadcast operand's splat makes the compiler wait for each load in turn).
// RAGGED (with VEC): a row's last unit is partial, or its slices hold fewer than 64 lanes.
template <class Prod, class Comb, bool VEC, bool ALLV, bool MULTI, bool RAGGED>
__global__ __launch_bounds__(kBlock) void red_cols_kernel(RedArgsOf<Prod::NIN, MULTI> A,
                                                          Prod prod, uint32_t xblocks) {
  constexpr int NIN = Prod::NIN;
  constexpr int W = VEC ? 4 : 1;
  using Part = typename Comb::Part;
  constexpr bool kExt = Comb::kExact;
  constexpr bool IS_MAX = std::is_same<Comb, ExtComb<true>>::value;
  using Fast = typename std::conditional<kExt, ExtFast, Part>::type;
  static_assert(!(kStores<Prod> && kExt), "a storing producer visits each element once");
  static_assert(!(kStores<Prod> && MULTI), "a storing producer's sum has one reduced axis");
  __shared__ Fast sh[kBlock / 64][64 * W];

  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint32_t bx = blockIdx.x, chunk = blockIdx.y;
  const uint32_t o = bx / xblocks;
  // the lane's columns: W from jo on; a partial unit at the end of a row is read from four columns
  // before the end, and its first `skip` columns are the lane before's
  const uint32_t lanes = RAGGED ? A.lanes : 64;
  const uint64_t jo = (uint64_t(bx - o * xblocks) * lanes + lane) * W;
  const bool active = (!RAGGED || uint32_t(lane) < lanes) && jo < A.inner;  // no early return: a
  const uint64_t j = !RAGGED || jo + W <= A.inner ? jo : A.inner - W;       // barrier follows
  const int skip = RAGGED && active ? int(jo - j) : 0;
  int64_t base[NIN], lbase[NIN], tbase;
  decode_outer(A, o, base, tbase);
#pragma unroll
  for (int k = 0; k < NIN; ++k) {
    // an inactive lane loads column 0 (in bounds) and drops it: the loads take no branch
    lbase[k] = base[k];
    base[k] += int64_t(j) * A.kst[k];
    if (active) lbase[k] = base[k];
  }
  const uint64_t k0 = uint64_t(chunk) * A.seglen;
  const uint64_t k1 = k0 + A.seglen < A.len ? k0 + A.seglen : A.len;

  Fast f[W];
#pragma unroll
  for (int c = 0; c < W; ++c) {
    if constexpr (kExt) f[c] = Fast{IS_MAX ? -__builtin_huge_valf() : __builtin_huge_valf(), 0u};
    else f[c] = Comb::empty();
  }
  constexpr int kU = kColUnroll<Prod>;
  for (uint64_t r0 = k0 + wv; r0 < k1; r0 += 4 * kU) {
    float xv[kU][NIN][W];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      // a row past the chunk is clamped to its last row: loaded, not used
      const uint64_t r = r0 + 4 * u < k1 ? r0 + 4 * u : k1 - 1;
      int64_t roff[NIN];
      reduced_offset<NIN>(A, r, roff);
#pragma unroll
      for (int k = 0; k < NIN; ++k) {
        const float *src = A.in[k] + lbase[k] + roff[k];
        if constexpr (VEC) {
          const f4 v = (ALLV || (A.vec_mask >> k & 1u))
                           ? __builtin_nontemporal_load(reinterpret_cast<const f4u *>(src))
                           : f4(src[0]);
#pragma unroll
          for (int c = 0; c < W; ++c) xv[u][k][c] = v[c];
        } else {
          xv[u][k][0] = src[0];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const uint64_t r = r0 + 4 * u;
      if (!active || r >= k1) continue;
      float yv[W];
#pragma unroll
      for (int c = 0; c < W; ++c) {
        float v[NIN];
#pragma unroll
        for (int k = 0; k < NIN; ++k) v[k] = xv[u][k][c];
        const float y = prod.eval(v);
        yv[c] = stored_value(prod, v, y);
        if constexpr (kExt) {
          f[c].m = IS_MAX ? fmaxf(f[c].m, y) : fminf(f[c].m, y);
          f[c].nan |= y != y ? 1u : 0u;
        } else {
          Comb::next(f[c], y, int64_t(r));
        }
      }
      if constexpr (kStores<Prod>) {
        float *dst = prod.dst + base[0] + int64_t(r) * A.rst[0];
        if constexpr (VEC) {
          if (skip == 0) {
            store_col<Prod>(dst, f4{yv[0], yv[1], yv[2], yv[3]});
          } else {
#pragma unroll
            for (int c = 1; c < 4; ++c)
              if (c >= skip) dst[c] = yv[c];
          }
        } else {
          dst[0] = yv[0];
        }
      }
    }
  }
#pragma unroll
  for (int c = 0; c < W; ++c) sh[wv][lane * W + c] = f[c];
  __syncthreads();
  if (wv != 0 || !active) return;

#pragma unroll
  for (int c = 0; c < W; ++c) {
    const bool mine = c >= skip;
    Part p;
    if constexpr (kExt) {
      float m = sh[0][lane * W + c].m;
      uint32_t nan = sh[0][lane * W + c].nan;
#pragma unroll
      for (int w = 1; w < kBlock / 64; ++w) {
        m = IS_MAX ? fmaxf(m, sh[w][lane * W + c].m) : fminf(m, sh[w][lane * W + c].m);
        nan |= sh[w][lane * W + c].nan;
      }
      if (!nan && m != 0.0f) {
        p = ExtPart{m, kNonEmpty};
      } else {
        // the reference's fold over [k0, k1) in index order
        p = Comb::empty();
        int64_t bc[NIN];
#pragma unroll
        for (int k = 0; k < NIN; ++k) bc[k] = base[k] + int64_t(c) * A.kst[k];
        for (uint64_t r = k0; r < k1; ++r) {
          const float y = value_at(A, prod, bc, r);
          if (r == k0) Comb::first(p, y, int64_t(r));
          else Comb::next(p, y, int64_t(r));
        }
      }
    } else {
      p = sh[0][lane * W + c];
#pragma unroll
      for (int w = 1; w < kBlock / 64; ++w) p = Comb::merge(p, sh[w][lane * W + c]);
      if constexpr (kSerialSum<Comb>) {
        if (A.segs == 1 && !finite_sum(p)) {
          int64_t bc[NIN];
#pragma unroll
          for (int k = 0; k < NIN; ++k) bc[k] = base[k] + int64_t(c) * A.kst[k];
          p = serial_sum_lane(A, prod, bc, A.len);
        }
      }
    }
    if (!mine) continue;
    if (A.segs == 1) {
      store_final<Comb>(A.out, tbase + int64_t(j + c) * A.tkst, p, A.post, A.divisor);
    } else {
      const uint64_t oi = uint64_t(o) * A.inner + j + c;
      static_cast<Part *>(A.part)[uint64_t(chunk) * (A.rows * A.inner) + oi] = p;
    }
  }
}

// Small leading-axis sums in one launch (no partials leave the workgroup, so no finalize), also
// for a storing producer (the one-pass epilogue), which then sums in the same order as the plain
// sum of what it stores. A workgroup owns S4 float4 columns (4 * S4 adjacent outputs) of one outer index and walks every row
// of the reduced axis: lane (g, c) sums the rows g, g + G, g + 2G, ... (G = kBlock / S4 row groups)
// of float4 column c in order. The row groups of a wave then merge with a fixed butterfly, and the
// four waves' partials in wave order: the result is deterministic. A column whose sum is not finite
// is summed again serially in index order (the reference's order decides such sums).
// RAGGED: a row's last unit is partial (testing for it costs 5-8% where none is).
template <class Prod, int S4, bool ALLV, bool RAGGED>
__global__ __launch_bounds__(kBlock) void red_cols_small_kernel(RedArgs<Prod::NIN> A, Prod prod,
                                                                uint32_t xblocks) {
  constexpr int NIN = Prod::NIN;
  constexpr int G = kBlock / S4, kU = S4 == PLAST_COL_SMALL_S4 ? PLAST_COL_SMALL_U : PLAST_COL_SMALL_U3;
  static_assert(64 % S4 == 0, "row groups split evenly over the waves");
  __shared__ f4 sh[kBlock / 64][S4];
  const uint32_t t = threadIdx.x, c4 = t % S4, g = t / S4, lane = t & 63, wv = t >> 6;
  // XCD numbering: the workgroups of one XCD take adjacent column slices, so the slices that share
  // a cache line share that XCD's L2
  const uint32_t b = PLAST_COL_SMALL_XCD ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
  const uint32_t o = b / xblocks;
  const uint64_t j0 = uint64_t(b - o * xblocks) * (4 * S4);  // the slice's first column
  // a partial unit at the end of a row is read from four columns before the end (see red_cols_kernel)
  const bool active = j0 + 4 * c4 < A.inner;
  const uint64_t j = !RAGGED || j0 + 4 * c4 + 4 <= A.inner ? j0 + 4 * c4 : A.inner - 4;
  const int skip = RAGGED && active ? int(j0 + 4 * c4 - j) : 0;
  int64_t base0[NIN], base[NIN], lbase[NIN], tbase;
  decode_outer(A, o, base0, tbase);
#pragma unroll
  for (int k = 0; k < NIN; ++k) {
    base[k] = base0[k] + int64_t(j) * A.kst[k];
    lbase[k] = active ? base[k] : base0[k];  // an inactive lane loads column 0 and drops it
  }
  f4 f = f4(0.0f);
  for (uint64_t r0 = g; r0 < A.len; r0 += uint64_t(G) * kU) {
    f4 xv[kU][NIN];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      // rows past the end are clamped to the last row: loaded, not used (the loads take no branch)
      const uint64_t r = r0 + uint64_t(u) * G < A.len ? r0 + uint64_t(u) * G : A.len - 1;
#pragma unroll
      for (int k = 0; k < NIN; ++k) {
        const float *src = A.in[k] + lbase[k] + int64_t(r) * A.rst[k];
        xv[u][k] = (ALLV || (A.vec_mask >> k & 1u)) ? *reinterpret_cast<const f4u *>(src)
                                                    : f4(src[0]);
      }
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const uint64_t r = r0 + uint64_t(u) * G;
      if (!active || r >= A.len) continue;
      f4 yv;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float v[NIN];
#pragma unroll
        for (int k = 0; k < NIN; ++k) v[k] = xv[u][k][c];
        const float y = prod.eval(v);
        f[c] = f[c] + y;
        yv[c] = stored_value(prod, v, y);
      }
      if constexpr (kStores<Prod>) {  // a storing producer also writes each value it sums
        float *dst = prod.dst + base[0] + int64_t(r) * A.rst[0];
        if (skip == 0) {
          store_col<Prod>(dst, yv);
        } else {
#pragma unroll
          for (int c = 1; c < 4; ++c)
            if (c >= skip) dst[c] = yv[c];
        }
      }
    }
  }
  // the wave's row groups (lanes c4, c4 + S4, ...) merge pairwise with a fixed butterfly
#pragma unroll
  for (int m = S4; m < 64; m <<= 1)
#pragma unroll
    for (int c = 0; c < 4; ++c) f[c] = f[c] + __shfl_xor(f[c], m);
  if (lane < uint32_t(S4)) sh[wv][lane] = f;
  __syncthreads();
  if (t >= uint32_t(4 * S4)) return;
  // lane t finishes one output column, element t % 4 of unit t / 4: the waves' partials in wave order
  const uint64_t ju = j0 + (t & ~3u);  // the unit's first column, before a partial one moves back
  if (ju >= A.inner) return;
  const uint64_t jc = (!RAGGED || ju + 4 <= A.inner ? ju : A.inner - 4) + (t & 3u);
  if (RAGGED && jc < ju) return;
  float p = sh[0][t / 4][t % 4];
#pragma unroll
  for (int w = 1; w < kBlock / 64; ++w) p = p + sh[w][t / 4][t % 4];
  if (!finite_sum(p)) {
    int64_t bc[NIN];
#pragma unroll
    for (int k = 0; k < NIN; ++k) bc[k] = base0[k] + int64_t(jc) * A.kst[k];
    p = serial_sum_lane(A, prod, bc, A.len);
  }
  store_final<SumComb>(A.out, tbase + int64_t(jc) * A.tkst, p, A.post, A.divisor);
}

// Narrow columns: operands contiguous over [len, inner] (or constant along the reduced axis), with
// fewer columns than a wave's slice. The rows are read as one flat array: T lanes of the workgroup
// take consecutive float4 units, 4 T floats being a whole number R of rows, so the columns a lane's
// four elements fall in are the same in every step, whatever inner is, and no lane idles over a short
// row (a slice of 64 lanes keeps 3 of them on 10 columns). The workgroup's 4 T sums, R per column,
// are merged through LDS eight rows at a time, in order.
template <class Prod>
constexpr int kFlatUnroll = Prod::NIN == 1 ? 4 : 2;
struct FlatArgs {
  uint32_t T, R;
  MagicDiv dinner;
};

template <class Prod, class Comb>
__global__ __launch_bounds__(kFlatBlock) void red_cols_flat_kernel(RedArgs<Prod::NIN> A, Prod prod,
                                                                   FlatArgs F) {
  constexpr int NIN = Prod::NIN, kU = kFlatUnroll<Prod>;
  using Part = typename Comb::Part;
  constexpr bool kExt = Comb::kExact;
  constexpr bool IS_MAX = std::is_same<Comb, ExtComb<true>>::value;
  using Fast = typename std::conditional<kExt, ExtFast, Part>::type;
  __shared__ Fast sh[kFlatBlock * 4];
  const uint32_t t = threadIdx.x, o = blockIdx.x, inner = uint32_t(A.inner);
  int64_t base[NIN], tbase;
  decode_outer(A, o, base, tbase);
  const uint64_t k0 = uint64_t(blockIdx.y) * A.seglen;
  const uint64_t k1 = k0 + A.seglen < A.len ? k0 + A.seglen : A.len;
  const uint64_t nf = (k1 - k0) * inner;  // floats of the chunk
  const auto merge = [](const Fast &a, const Fast &b) {
    if constexpr (kExt) return Fast{IS_MAX ? fmaxf(a.m, b.m) : fminf(a.m, b.m), a.nan | b.nan};
    else return Comb::merge(a, b);
  };
  Fast f[4];
  uint32_t row[4];
  f4 fixed[NIN];  // the lane's columns of an operand constant along the reduced axis
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if constexpr (kExt) f[c] = Fast{IS_MAX ? -__builtin_huge_valf() : __builtin_huge_valf(), 0u};
    else f[c] = Comb::empty();
    row[c] = F.dinner.div(4 * t + c);
    const uint32_t col = 4 * t + c - row[c] * inner;
#pragma unroll
    for (int k = 0; k < NIN; ++k)
      fixed[k][c] = A.rst[k] == 0 ? A.in[k][base[k] + int64_t(col) * A.kst[k]] : 0.0f;
  }
  if (t < F.T) {
    uint64_t step = 0;
    for (uint64_t f0 = 4 * t; f0 < nf; f0 += uint64_t(4) * F.T * kU, step += kU) {
      f4 x[kU][NIN];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint64_t at = f0 + uint64_t(u) * 4 * F.T;
#pragma unroll
        for (int k = 0; k < NIN; ++k) {
          const float *src = A.in[k] + base[k] + k0 * inner;
          if (A.rst[k] == 0) {
            x[u][k] = fixed[k];
          } else if (at + 4 <= nf) {
            x[u][k] = __builtin_nontemporal_load(reinterpret_cast<const f4u *>(src + at));
          } else {
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) x[u][k][c] = at + c < nf ? src[at + c] : 0.0f;
          }
        }
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint64_t at = f0 + uint64_t(u) * 4 * F.T;
        if (at >= nf) continue;
        f4 yv;
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
          float v[NIN];
#pragma unroll
          for (int k = 0; k < NIN; ++k) v[k] = x[u][k][c];
          const float y = prod.eval(v);
          yv[c] = stored_value(prod, v, y);
          if (at + c >= nf) continue;
          if constexpr (kExt) {
            f[c].m = IS_MAX ? fmaxf(f[c].m, y) : fminf(f[c].m, y);
            f[c].nan |= y != y ? 1u : 0u;
          } else {
            Comb::next(f[c], y, int64_t(k0 + (step + u) * F.R + row[c]));
          }
        }
        if constexpr (kStores<Prod>) {
          float *dst = prod.dst + base[0] + k0 * inner + at;
          if (at + 4 <= nf) {
            store_col<Prod>(dst, yv);
          } else {
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c)
              if (at + c < nf) dst[c] = yv[c];
          }
        }
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) sh[4 * t + c] = f[c];
  }
  __syncthreads();
  // sh[r][j]: the sums of rows r, r + R, ... of column j; rows 8e .. 8e + 7 merge into row e. A round
  // leaves ceil(R / 8) * inner sums at most, R * inner being 4 T: 448, one a lane.
  for (uint32_t rows = F.R; rows > 1;) {
    const uint32_t next = (rows + 7) / 8;
    Fast g;
    if (t < next * inner) {
      const uint32_t e = F.dinner.div(t), j = t - e * inner;
      g = sh[8 * e * inner + j];
#pragma unroll
      for (uint32_t q = 1; q < 8; ++q)
        if (8 * e + q < rows) g = merge(g, sh[(8 * e + q) * inner + j]);
    }
    __syncthreads();
    if (t < next * inner) sh[t] = g;
    __syncthreads();
    rows = next;
  }
  if constexpr (kExt) {
    // Columns with a zero extreme or a NaN, all of them at once: the workgroup walks its chunk again
    // (from the caches) for the last NaN of each, the extreme after it, and the last zero after it,
    // whose sign decides the bits. One lane a column folding its chunk in order took 93 us for max of
    // [60000, 10] with a zero in every column.
    static_assert(NIN == 1, "order-sensitive folds are of one operand");
    __shared__ uint32_t last[kFlatInner], key[kFlatInner], zero[kFlatInner];
    const bool nan = t < inner && sh[t].nan;
    if (__syncthreads_or(nan || (t < inner && sh[t].m == 0.0f))) {
      const bool any_nan = __syncthreads_or(nan);
      if (t < inner) last[t] = zero[t] = 0, key[t] = IS_MAX ? 0u : ~0u;
      __syncthreads();
      // take(c, y, the row of the chunk + 1), then done(c, column) for the lane's four columns
      const auto walk = [&](auto &&take, auto &&done) {
        if (t < F.T) {
          const float *src = A.in[0] + base[0] + k0 * inner;
          uint32_t step = 0;
          for (uint64_t at = 4 * t; at < nf; at += uint64_t(4) * F.T, ++step) {
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c)
              if (at + c < nf) {
                const float v = A.rst[0] == 0 ? fixed[0][c] : src[at + c];
                take(c, prod.eval(&v), step * F.R + row[c] + 1);
              }
          }
#pragma unroll
          for (uint32_t c = 0; c < 4; ++c) done(c, 4 * t + c - row[c] * inner);
        }
        __syncthreads();
      };
      uint32_t best[4] = {};
      const auto later = [&](uint32_t *to) {
        return [&best, to](uint32_t c, uint32_t col) {
          if (best[c]) atomicMax(&to[col], best[c]);
        };
      };
      if (any_nan) {
        walk([&](uint32_t c, float y, uint32_t r) { if (y != y) best[c] = r; }, later(last));
        uint32_t from[4];
        float m[4];
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
          from[c] = t < F.T ? last[4 * t + c - row[c] * inner] : 0;
          m[c] = IS_MAX ? -__builtin_huge_valf() : __builtin_huge_valf();
        }
        // as unsigned integers ordered like the floats
        walk([&](uint32_t c, float y, uint32_t r) {
          if (r > from[c]) m[c] = IS_MAX ? fmaxf(m[c], y) : fminf(m[c], y);
        }, [&](uint32_t c, uint32_t col) {
          const uint32_t u = __float_as_uint(m[c]), o = u >> 31 ? ~u : u | 0x80000000u;
          if constexpr (IS_MAX) atomicMax(&key[col], o);
          else atomicMin(&key[col], o);
        });
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) best[c] = 0;
      walk([&](uint32_t c, float y, uint32_t r) { if (y == 0.0f) best[c] = r; }, later(zero));
      if (t < inner) {
        const uint32_t o = key[t];
        float m = nan ? __uint_as_float(o >> 31 ? o & 0x7fffffffu : ~o) : sh[t].m;
        int64_t at = base[0] + int64_t(t) * A.kst[0] + int64_t(k0) * A.rst[0];
        // (a column that ends in a NaN: the fold's value is that NaN)
        const uint32_t r = nan && last[t] == uint32_t(k1 - k0) ? last[t] : m == 0.0f ? zero[t] : 0;
        if (r) {
          const float v = A.in[0][at + int64_t(r - 1) * A.rst[0]];
          m = prod.eval(&v);
        }
        sh[t].m = m;
      }
    }
  }
  if (t >= inner) return;
  int64_t bc[NIN];
#pragma unroll
  for (int k = 0; k < NIN; ++k) bc[k] = base[k] + int64_t(t) * A.kst[k];
  Part p;
  if constexpr (kExt) {
    p = ExtPart{sh[t].m, kNonEmpty | (sh[t].nan ? kIndep : 0u)};
  } else {
    p = sh[t];
    if constexpr (kSerialSum<Comb>)
      if (A.segs == 1 && !finite_sum(p)) p = serial_sum_lane(A, prod, bc, A.len);
  }
  if (A.segs == 1) store_final<Comb>(A.out, tbase + int64_t(t) * A.tkst, p, A.post, A.divisor);
  else static_cast<Part *>(A.part)[uint64_t(blockIdx.y) * (A.rows * inner) + uint64_t(o) * inner + t] = p;
}

template <class Prod, class Comb, class Args>
__global__ __launch_bounds__(kBlock) void red_cols_finalize(Args A, Prod prod) {
  using Part = typename Comb::Part;
  constexpr int NIN = Prod::NIN;
  const uint64_t oi = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
  const uint64_t nout = A.rows * A.inner;
  if (oi >= nout) return;
  Part p = merge_in_order<Comb>(static_cast<const Part *>(A.part) + oi, nout, A.segs);
  const uint32_t o = uint32_t(oi / A.inner);
  const uint64_t j = oi - uint64_t(o) * A.inner;
  int64_t base[NIN], tbase;
  decode_outer(A, o, base, tbase);
  if constexpr (kSerialSum<Comb>) {
    if (!finite_sum(p)) {
#pragma unroll
      for (int k = 0; k < NIN; ++k) base[k] += int64_t(j) * A.kst[k];
      p = serial_sum_lane(A, prod, base, A.len);
    }
  }
  store_final<Comb>(A.out, tbase + int64_t(j) * A.tkst, p, A.post, A.divisor);
}

// The same merge with Q lanes per output, for many chunks: lane (q, o) merges the q-th run of
// consecutive chunks of output o in index order (lanes with the same q read consecutive outputs),
// then the runs merge pairwise through shuffles with the earlier run always on the left, as in
// red_rows_finalize. One batch of loads per lane instead of segs / 16 batches in sequence.
template <class Prod, class Comb, int Q, class Args>
__global__ __launch_bounds__(kBlock) void red_cols_finalize_q(Args A, Prod prod) {
  using Part = typename Comb::Part;
  constexpr int NIN = Prod::NIN;
  constexpr uint32_t OPW = 64 / Q;  // outputs per wave
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t wave = (uint64_t(blockIdx.x) * kBlock + threadIdx.x) >> 6;
  const uint32_t q = lane / OPW;
  const uint64_t nout = A.rows * A.inner;
  const uint64_t oi = wave * OPW + (lane % OPW);
  const bool valid = oi < nout;
  const uint32_t run = (A.segs + Q - 1) / Q;
  const uint32_t active = (A.segs + run - 1) / run;  // runs holding at least one chunk
  Part p = Comb::empty();
  if (valid && q < active) {
    const uint32_t s0 = q * run;
    const uint32_t n = A.segs - s0 < run ? A.segs - s0 : run;
    p = merge_in_order<Comb>(static_cast<const Part *>(A.part) + uint64_t(s0) * nout + oi, nout,
                             n);
  }
#pragma unroll
  for (uint32_t off = 1; off < uint32_t(Q); off <<= 1) {
    const Part o = shfl_down_part(p, int(off * OPW));
    if ((q & (2 * off - 1)) == 0 && q + off < active) p = Comb::merge(p, o);
  }
  if (q != 0 || !valid) return;
  const uint32_t o = uint32_t(oi / A.inner);
  const uint64_t j = oi - uint64_t(o) * A.inner;
  int64_t base[NIN], tbase;
  decode_outer(A, o, base, tbase);
  if constexpr (kSerialSum<Comb>) {
    if (!finite_sum(p)) {
#pragma unroll
      for (int k = 0; k < NIN; ++k) base[k] += int64_t(j) * A.kst[k];
      p = serial_sum_lane(A, prod, base, A.len);
    }
  }
  store_final<Comb>(A.out, tbase + int64_t(j) * A.tkst, p, A.post, A.divisor);
}

// ------------------------------------------------------------------------- generic kernel

template <int NIN>
struct GenArgs {
  const float *in[NIN];
  void *out;
  int nk, nr;                      // kept / reduced axis counts
  uint64_t kext[kMaxRank], rext[kMaxRank];
  int64_t kst[NIN + 1][kMaxRank];  // strides on kept axes (operand NIN = target)
  int64_t rst[NIN][kMaxRank];      // strides on reduced axes
  uint64_t nout, len;
  int post;
  float divisor;
};

template <class Prod, class Comb>
__global__ __launch_bounds__(kBlock) void red_generic_kernel(GenArgs<Prod::NIN> A, Prod prod) {
  constexpr int NIN = Prod::NIN;
  using Part = typename Comb::Part;
  const uint64_t stride = uint64_t(gridDim.x) * kBlock;
  for (uint64_t o = uint64_t(blockIdx.x) * kBlock + threadIdx.x; o < A.nout; o += stride) {
    int64_t base[NIN] = {};
    int64_t tbase = 0;
    uint64_t rem = o;
    for (int d = A.nk - 1; d >= 0; --d) {
      const int64_t c = int64_t(rem % A.kext[d]);
      rem /= A.kext[d];
#pragma unroll
      for (int k = 0; k < NIN; ++k) base[k] += c * A.kst[k][d];
      tbase += c * A.kst[NIN][d];
    }
    Part p = Comb::empty();
    uint64_t rc[kMaxRank] = {};
    int64_t off[NIN];
#pragma unroll
    for (int k = 0; k < NIN; ++k) off[k] = base[k];
    for (uint64_t r = 0; r < A.len; ++r) {
      float v[NIN];
#pragma unroll
      for (int k = 0; k < NIN; ++k) v[k] = A.in[k][off[k]];
      const float y = prod.eval(v);
      if (r == 0) Comb::first(p, y, int64_t(r));
      else Comb::next(p, y, int64_t(r));
      // odometer step over the reduced axes, innermost fastest
      for (int d = A.nr - 1; d >= 0; --d) {
        if (++rc[d] < A.rext[d]) {
#pragma unroll
          for (int k = 0; k < NIN; ++k) off[k] += A.rst[k][d];
          break;
        }
#pragma unroll
        for (int k = 0; k < NIN; ++k) off[k] -= int64_t(rc[d] - 1) * A.rst[k][d];
        rc[d] = 0;
      }
    }
    store_final<Comb>(A.out, tbase, p, A.post, A.divisor);
  }
}

// ------------------------------------------------------------------------- host dispatch

// Merges the chunks' partials (and, for a serial refold, reads the inputs). More than one chunk is
// planned only below PLAST_COL_BLOCKS workgroups of columns, so nout * Q lanes (at most
// PLAST_COL_BLOCKS * 256 * Q) stay far inside one launch.
template <class Prod, class Comb, class Args>
void launch_cols_finalize(const Args &A, const Prod &prod, uint64_t nout, uint64_t chunks) {
  if (PLAST_COL_FIN_Q > 1 && chunks >= 2 * PLAST_COL_FIN_Q)
    red_cols_finalize_q<Prod, Comb, PLAST_COL_FIN_Q>
        <<<ceil_div(nout * PLAST_COL_FIN_Q, kBlock), kBlock, 0, stream()>>>(A, prod);
  else
    red_cols_finalize<Prod, Comb><<<ceil_div(nout, kBlock), kBlock, 0, stream()>>>(A, prod);
}

// Reduce over every axis where operand NIN (the target) has stride 0 and extent > 1.
// `post` and `divisor` describe the epilogue; `out` is float* or int64_t* per Comb::Out.
template <class Prod, class Comb>
bool launch_reduction(const Prod &prod, const void *const *in, void *out, Space s, Post post,
                      float divisor, const char *where) {
  constexpr int NIN = Prod::NIN;
  using Part = typename Comb::Part;
  s.nops = NIN + 1;
  // An empty space: every output holds the fold of nothing (sum 0, mean 0/0, max -FLT_MAX, ...).
  if (s.numel() == 0) {
    if constexpr (kStores<Prod>) return false;
    GenArgs<NIN> G;
    memset(&G, 0, sizeof G);
    G.out = out;
    uint64_t nout = 1;
    for (int d = 0; d < s.rank; ++d) {
      if (s.st[NIN][d] == 0 && s.shape[d] != 1) continue;  // reduced axis
      G.kext[G.nk] = s.shape[d];
      G.kst[NIN][G.nk] = s.st[NIN][d];
      ++G.nk;
      nout *= s.shape[d];
    }
    if (nout == 0) return true;
    G.nout = nout;
    G.len = 0;
    G.post = int(post);
    G.divisor = divisor;
    const uint64_t gb = (nout + kBlock - 1) / kBlock;
    red_generic_kernel<Prod, Comb><<<unsigned(gb < 65536 ? gb : 65536), kBlock, 0, stream()>>>(G, prod);
    return true;
  }
  // collapse() never merges a reduced axis with a kept one: the target's stride is 0 on one and
  // not on the other.
  collapse(s);
  const int r = s.rank;
  int nred = 0, red_ax = -1;
  uint64_t nout = 1;
  for (int d = 0; d < r; ++d) {
    if (s.st[NIN][d] == 0 && s.shape[d] > 1) {
      ++nred;
      red_ax = d;
    } else {
      nout *= s.shape[d];
    }
  }
  const bool empty_space = false;

  const bool small_idx = s.numel() < (uint64_t(1) << 32) && nout < (uint64_t(1) << 32);
  // the innermost reduced axis, the other reduced axes' flattened walk in every kernel's arguments
  const auto outer_reduced = [&](RedMultiArgs<NIN> &A) {
    uint64_t len = s.shape[red_ax];
    A.drun = MagicDiv::make(uint32_t(s.shape[red_ax]));
    for (int d = 0; d < red_ax; ++d) {
      if (!(s.st[NIN][d] == 0 && s.shape[d] > 1)) continue;
      A.xdv[A.nx] = MagicDiv::make(uint32_t(s.shape[d]));
      for (int k = 0; k < NIN; ++k) A.xst[k][A.nx] = s.st[k][d];
      ++A.nx;
      len *= s.shape[d];
    }
    A.len = len;
  };
  const auto reduced = [&](int d) { return s.st[NIN][d] == 0 && s.shape[d] > 1; };
  const bool multi = nred > 1;

  // ---- rows: innermost axis reduced, unit stride for streamed operands
  // one wave per row (segment): the grid is rows * segs / 4 workgroups (rows < 2^32 segments
  // are only split when there are fewer than PLAST_ROW_WAVES rows)
  if (!kStores<Prod> && !empty_space && small_idx && nred >= 1 && red_ax == r - 1 &&
      nout <= max_blocks(kBlock) * (kBlock / 64)) {
    RedMultiArgs<NIN> A;
    memset(&A, 0, sizeof A);
    const RedArgs<NIN> &A1 = A;  // what the kernels over one reduced axis take
    for (int k = 0; k < NIN; ++k) A.in[k] = static_cast<const float *>(in[k]);
    A.out = out;
    const bool vec = !multi || s.shape[r - 1] >= 4;  // a run's partial unit is read from its end
    for (int k = 0; k < NIN; ++k) {
      A.rst[k] = s.st[k][r - 1];
      if (A.rst[k] == 1) A.vec_mask |= 1u << k;
    }
    bool unit = true;
    for (int k = 0; k < NIN; ++k) unit = unit && (A.rst[k] == 0 || A.rst[k] == 1);
    if (unit) {
      for (int d = 0; d < r - 1; ++d) {
        if (reduced(d)) continue;
        A.dv[A.nouter] = MagicDiv::make(uint32_t(s.shape[d]));
        A.tst[A.nouter] = s.st[NIN][d];
        for (int k = 0; k < NIN; ++k) A.ost[k][A.nouter] = s.st[k][d];
        ++A.nouter;
      }
      outer_reduced(A);
      A.rows = nout;
      const uint64_t units = (s.shape[r - 1] + 3) / 4;
      A.dunits = MagicDiv::make(uint32_t(units));
      A.vlen = 4 * units * (A.len / s.shape[r - 1]);
      const uint64_t span = multi && vec ? A.vlen : A.len;  // what segments divide
      // enough waves to cover the machine: split long rows when there are few of them
      uint32_t segs = 1;
      const uint64_t want_waves = multi ? PLAST_MULTI_WAVES : PLAST_ROW_WAVES;
      if (A.rows < want_waves && span >= 8192) {
        uint64_t sg = (want_waves + A.rows - 1) / A.rows;
        const uint64_t max_sg = span / 4096;
        if (sg > max_sg) sg = max_sg;
        if (sg > 65535) sg = 65535;
        segs = uint32_t(sg < 1 ? 1 : sg);
      }
      uint64_t seglen = (span + segs - 1) / segs;
      seglen = (seglen + 255) / 256 * 256;
      segs = uint32_t((span + seglen - 1) / seglen);
      A.segs = segs;
      A.seglen = seglen;
      A.post = int(post);
      A.divisor = divisor;
      if (segs > 1) {
        A.part = multi ? partials(sizeof(Part) * A.rows * segs, where)
                       : workspace(sizeof(Part) * A.rows * segs);
        if (!A.part) return false;
      }
      // short rows: 2, 8 or 32 lanes each. [50000, 77] a wave per row / 8 lanes: see the kernel. An
      // argmax walks a lane's values one after the other: rows above 16 take 8 lanes ([1024, 31] 4.2 us
      // in 2, 3.4 in 8; [65536, 17] 4.0 and 4.5), and few rows above 64 take 32 ([1024, 127] 4.2 in 8, 3.6
      // in 32, [8192, 100] 4.2 and 3.9; [8192, 45] 3.7 and 4.1).
      if (!multi && A.len <= 16 * 32) {
        const bool arg = std::is_same<Comb, ArgmaxComb>::value, few = arg && A.rows <= 8192;
        const int lanes = A.len <= (arg ? 16 : 32) ? 2 : A.len <= (few ? 64 : 128) ? 8 : 32;
        const unsigned sgrid = ceil_div(A.rows, (kBlock / 64) * (64 / lanes));
        if (lanes == 2) red_rows_short_kernel<Prod, Comb, 2><<<sgrid, kBlock, 0, stream()>>>(A1, prod);
        else if (lanes == 8) red_rows_short_kernel<Prod, Comb, 8><<<sgrid, kBlock, 0, stream()>>>(A1, prod);
        else red_rows_short_kernel<Prod, Comb, 32><<<sgrid, kBlock, 0, stream()>>>(A1, prod);
        return true;
      }
      const uint64_t waves = A.rows * segs;
      const unsigned grid = ceil_div(waves, kBlock / 64);
      if (vec && multi)
        red_rows_kernel<Prod, Comb, true, true><<<grid, kBlock, 0, stream()>>>(A, prod);
      else if (vec)
        red_rows_kernel<Prod, Comb, true, false><<<grid, kBlock, 0, stream()>>>(A1, prod);
      else
        red_rows_kernel<Prod, Comb, false, true><<<grid, kBlock, 0, stream()>>>(A, prod);
      if (segs > 1) {  // the finalize reads the partials, and the inputs for a serial refold
        const unsigned fgrid = ceil_div(A.rows, kBlock / 64);
        if (multi) red_rows_finalize<Prod, Comb><<<fgrid, kBlock, 0, stream()>>>(A, prod);
        else red_rows_finalize<Prod, Comb><<<fgrid, kBlock, 0, stream()>>>(A1, prod);
      }
      return true;
    }
  }

  // ---- cols: innermost axis kept with unit target stride (several reduced axes beside it: the
  // gradient of a broadcast operand, a sum)
  constexpr bool kMultiCols = !kStores<Prod> && std::is_same<Comb, SumComb>::value;
  if (!empty_space && small_idx && nred >= 1 && (!multi || kMultiCols) && red_ax != r - 1 &&
      s.st[NIN][r - 1] != 0) {
    RedMultiArgs<NIN> A;
    memset(&A, 0, sizeof A);
    const RedArgs<NIN> &A1 = A;  // what the kernels over one reduced axis take
    for (int k = 0; k < NIN; ++k) A.in[k] = static_cast<const float *>(in[k]);
    A.out = out;
    A.inner = s.shape[r - 1];
    A.tkst = s.st[NIN][r - 1];
    outer_reduced(A);
    bool vec = A.inner >= 4 && A.tkst == 1;
    int no = 0;
    for (int d = 0; d < r - 1; ++d) {
      if (reduced(d)) continue;
      A.dv[no] = MagicDiv::make(uint32_t(s.shape[d]));
      A.tst[no] = s.st[NIN][d];
      for (int k = 0; k < NIN; ++k) A.ost[k][no] = s.st[k][d];
      ++no;
    }
    A.nouter = no;
    constexpr bool kArg = std::is_same<Comb, ArgmaxComb>::value;
    // rows read as one flat array: operands contiguous over [len, inner] or constant along len
    bool flat = !multi && A.inner < kFlatInner;
    for (int k = 0; k < NIN; ++k) {
      A.rst[k] = s.st[k][red_ax];
      A.kst[k] = s.st[k][r - 1];
      if (A.kst[k] == 1) A.vec_mask |= 1u << k;
      else if (A.kst[k] != 0) vec = false;
      flat = flat && (A.rst[k] == 0 || (A.kst[k] == 1 && A.rst[k] == int64_t(A.inner)));
    }
    if (kStores<Prod> && A.rst[0] == 0) flat = false;
    A.rows = nout / A.inner;  // outer count
    A.post = int(post);
    A.divisor = divisor;
    const bool allv = A.vec_mask == (1u << NIN) - 1;
    const uint64_t nall = A.len * nout;
    // sums that some form takes in one launch: a capture needs no workspace for them
    const bool one_pass = std::is_same<Comb, SumComb>::value && vec && A.inner % 4 == 0 &&
                          nall <= PLAST_COL_SMALL_MAX;
    if constexpr (std::is_same<Comb, SumComb>::value) {
      // small: one launch over narrow column slices instead of chunks plus a finalize
      if (vec && !multi && nall <= PLAST_COL_SMALL_MAX &&
          col_slices(A.rows, A.len, A.inner, NIN, kStores<Prod>) && (NIN < 3 || PLAST_COL_SMALL3 != 0)) {
        const auto slices = [&](auto s4, auto every, auto ragged) {
          constexpr int S4 = decltype(s4)::value;
          const uint32_t sblocks = ceil_div(A.inner, uint64_t(4) * S4);
          const uint64_t sgrid = uint64_t(sblocks) * A.rows;
          if (sgrid > max_blocks(kBlock)) return false;
          A.segs = 1;
          red_cols_small_kernel<Prod, S4, decltype(every)::value, decltype(ragged)::value>
              <<<unsigned(sgrid), kBlock, 0, stream()>>>(A1, prod, sblocks);
          return true;
        };
        const auto with_form = [&](auto s4) {
          if (A.inner % 4 == 0)
            return allv ? slices(s4, std::true_type{}, std::false_type{}) : slices(s4, std::false_type{}, std::false_type{});
          return allv ? slices(s4, std::true_type{}, std::true_type{}) : slices(s4, std::false_type{}, std::true_type{});
        };
        bool done;
        if constexpr (NIN == 1) done = with_form(std::integral_constant<int, PLAST_COL_SMALL_S4>{});
        else if (col_small_one<Prod>(A.inner)) done = with_form(std::integral_constant<int, PLAST_COL_SMALL_S4_3>{});
        else done = with_form(std::integral_constant<int, PLAST_COL_SMALL_S4>{});
        if (done) return true;
      }
    }
    if (flat && A.rows <= max_blocks(kFlatBlock)) {
      const FlatCols f = flat_cols(A.rows, A.len, A.inner, PLAST_COL_BLOCKS);
      const ColChunks w = col_chunks(A.rows, A.len, A.inner, 1, kColMinRows<Prod>, PLAST_COL_BLOCKS);
      if (kStores<Prod> ? A.len >= 64 : flat_pays(w, f, A.rows, A.len, A.inner, kArg)) {
        A.segs = uint32_t(f.chunks);
        A.seglen = f.seglen;
        if (f.chunks > 1) {
          const size_t bytes = sizeof(Part) * nout * f.chunks;
          A.part = one_pass || w.chunks == 1 ? partials(bytes, where) : workspace(bytes);
          if (!A.part) return false;
        }
        const FlatArgs F{f.T, f.R, MagicDiv::make(uint32_t(A.inner))};
        const dim3 grid{unsigned(A.rows), unsigned(f.chunks), 1u};
        red_cols_flat_kernel<Prod, Comb><<<grid, kFlatBlock, 0, stream()>>>(A1, prod, F);
        if (f.chunks > 1) launch_cols_finalize<Prod, Comb>(A1, prod, nout, f.chunks);
        return true;
      }
    }
    if (!multi && col_width(A.rows, A.len, A.inner, kArg) == 1) vec = false;
    const uint32_t W = vec ? 4 : 1;
    const ColChunks w = col_chunks(A.rows, A.len, A.inner, W, kColMinRows<Prod>, PLAST_COL_BLOCKS);
    const uint32_t xblocks = uint32_t(w.slices);
    const uint64_t chunks = w.chunks;
    A.segs = uint32_t(chunks);
    A.seglen = w.seglen;
    // the slices of a row share its lanes evenly, in whole 128-byte lines
    A.lanes = ceil_div(ceil_div(A.inner, W), xblocks);
    A.lanes = vec && A.lanes < 56 ? (A.lanes + 7) / 8 * 8 : 64;
    const uint64_t base_blocks = w.slices * A.rows;
    if (base_blocks <= max_blocks(kBlock)) {
      if (chunks > 1) {
        const size_t bytes = sizeof(Part) * nout * chunks;
        A.part = multi || one_pass ? partials(bytes, where) : workspace(bytes);
        if (!A.part) return false;
      }
      const dim3 grid{unsigned(base_blocks), unsigned(chunks), 1u};
      if constexpr (kMultiCols) {
        if (multi) {
          if (vec)
            red_cols_kernel<Prod, Comb, true, false, true, true><<<grid, kBlock, 0, stream()>>>(A, prod, xblocks);
          else
            red_cols_kernel<Prod, Comb, false, false, true, false><<<grid, kBlock, 0, stream()>>>(A, prod, xblocks);
          if (chunks > 1) launch_cols_finalize<Prod, Comb>(A, prod, nout, chunks);
          return true;
        }
      }
      const bool ragged = A.inner % 4 != 0 || A.lanes < 64;
      if (vec && allv && ragged)
        red_cols_kernel<Prod, Comb, true, true, false, true><<<grid, kBlock, 0, stream()>>>(A1, prod, xblocks);
      else if (vec && allv)
        red_cols_kernel<Prod, Comb, true, true, false, false><<<grid, kBlock, 0, stream()>>>(A1, prod, xblocks);
      else if (vec)
        red_cols_kernel<Prod, Comb, true, false, false, true><<<grid, kBlock, 0, stream()>>>(A1, prod, xblocks);
      else
        red_cols_kernel<Prod, Comb, false, false, false, false><<<grid, kBlock, 0, stream()>>>(A1, prod, xblocks);
      if (chunks > 1) launch_cols_finalize<Prod, Comb>(A1, prod, nout, chunks);
      return true;
    }
  }

  // ---- generic
  if constexpr (kStores<Prod>) return false;
  GenArgs<NIN> G;
  memset(&G, 0, sizeof G);
  for (int k = 0; k < NIN; ++k) G.in[k] = static_cast<const float *>(in[k]);
  G.out = out;
  G.len = 1;
  for (int d = 0; d < r; ++d) {
    const bool red = s.st[NIN][d] == 0 && s.shape[d] > 1;
    if (red) {
      G.rext[G.nr] = s.shape[d];
      for (int k = 0; k < NIN; ++k) G.rst[k][G.nr] = s.st[k][d];
      G.len *= s.shape[d];
      ++G.nr;
    } else {
      G.kext[G.nk] = s.shape[d];
      for (int k = 0; k <= NIN; ++k) G.kst[k][G.nk] = s.st[k][d];
      ++G.nk;
    }
  }
  G.nout = nout;
  G.post = int(post);
  G.divisor = divisor;
  uint64_t blocks = (nout + kBlock - 1) / kBlock;
  if (blocks > 65536) blocks = 65536;
  if (blocks == 0) blocks = 1;
  red_generic_kernel<Prod, Comb><<<unsigned(blocks), kBlock, 0, stream()>>>(G, prod);
  (void)where;
  return true;
}

// Accumulating sum into a broadcast target: target[t] += sum over its broadcast axes of prod.
template <class Prod>
bool reduce_accumulate(const Prod &prod, const void *const *in, float *target, Space s,
                       const char *where) {
  return launch_reduction<Prod, SumComb>(prod, in, target, s, Post::Accum, 1.0f, where);
}

}  // namespace plast
