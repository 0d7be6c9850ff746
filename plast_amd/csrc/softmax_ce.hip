// softmax_ce.hip — fused softmax cross-entropy over the rows of [N, C] logits with int32 labels,
// and softmax / log-softmax over the last axis.
//
// Forward, per row (the reference chain MAX -> SUB -> EXP -> SUM -> LOG -> SUB -> MUL(onehot) ->
// SUM -> NEG of src/api/loss.c:97-169, one HBM read):
//   m = the reference's max fold from -FLT_MAX (bit-exact, NaN and signed-zero rules included)
//   s = sum_j expf(x_j - m)         (parallel sum; the reference sums serially)
//   l = logf(s)
//   t = 0 + ((x_label - m) - l), or NaN when any other term 0 * ((x_j - m) - l) is NaN
//   loss = 0 - t inside the reference's SIMD blocks of its NEG node, -t in its tail
// stats[row] = (m, l) for the backward.
// Backward: dx[row, j] (+)= dloss[row] * (exp((x - m) - l) - onehot).
// The fast paths evaluate exp with exp_le0 (about 1 ulp); the exact-refold paths use expf.
#include <atomic>
#include <cfloat>
#include <type_traits>

#include "common.hpp"

namespace plast {
namespace {

constexpr int kCeBlock = 256;
constexpr int kCeWaves = kCeBlock / 64;

// exp(t) for the shifted logits of a softmax (t <= 0), from the hardware base-2 exponential
// (v_exp_f32, accurate to 1 ulp). t*log2(e) is carried as p + d: p = t*L rounded, d = that
// product's rounding error (one FMA) plus t times the error of L itself, so
// exp(t) = 2^p * 2^d with 2^d = 1 + d*ln2 (|d| < 2^-17 for |t| < 87). About 1 ulp from the
// correctly rounded result; 6 VALU ops where the library expf takes about 15. Below t = -87 the
// result would be subnormal (< 2^-125.5) and 0 is returned; -inf gives 0 and NaN stays NaN.
// Used only where the result feeds a sum or a gradient compared to 1e-5 relative.
__device__ __forceinline__ float exp_le0(float t) {
  constexpr float kL = 1.44269502162933349609375f;   // log2(e) rounded to fp32
  constexpr float kLlo = 1.925963033500011079e-8f;   // log2(e) - kL
  constexpr float kLn2 = 0.693147180559945309f;
  const float p = t * kL;
  const float d = __builtin_fmaf(t, kLlo, __builtin_fmaf(t, kL, -p));
  const float r = __builtin_amdgcn_exp2f(p);
  const float e = __builtin_fmaf(r, d * kLn2, r);
  return t < -87.0f ? 0.0f : e;
}

// exp_le0 without the range clamp, for finite t <= 0 only (-inf would give NaN): below t = -87 it
// returns the subnormal or zero that 2^p gives. Two instructions fewer.
__device__ __forceinline__ float exp_le0_finite(float t) {
  constexpr float kL = 1.44269502162933349609375f;
  constexpr float kLlo = 1.925963033500011079e-8f;
  constexpr float kLn2 = 0.693147180559945309f;
  const float p = t * kL;
  const float d = __builtin_fmaf(t, kLlo, __builtin_fmaf(t, kL, -p));
  const float r = __builtin_amdgcn_exp2f(p);
  return __builtin_fmaf(r, d * kLn2, r);
}

// Block-wide reductions over W waves (lds holds W + 1 floats), combined in wave order.
template <int W = kCeWaves>
__device__ __forceinline__ float block_sum(float v, float *lds) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = 0.0f;
#pragma unroll
  for (int w = 0; w < W; ++w) r += lds[w];
  return r;
}

template <int W = kCeWaves>
__device__ __forceinline__ float block_fmax(float v, float *lds) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = lds[0];
#pragma unroll
  for (int w = 1; w < W; ++w) r = fmaxf(r, lds[w]);
  return r;
}

template <int W = kCeWaves>
__device__ __forceinline__ bool block_any(bool b, float *lds) {
  return block_sum<W>(b ? 1.0f : 0.0f, lds) > 0.0f;
}

// The reference's serial max fold, for rows whose fast-path extreme is ambiguous (NaN or zero).
__device__ float serial_max_fold(const float *row, uint32_t C) {
  float acc = -FLT_MAX;
  for (uint32_t j = 0; j < C; ++j) acc = acc > row[j] ? acc : row[j];
  return acc;
}

// The same fold by a wave: a NaN restarts it (the result is the fold of what follows the last one),
// and the last of several zeros that tie decides a zero result's sign.
__device__ float wave_max_fold(const float *row, uint32_t C, int lane) {
  int last_nan = -1;
  for (uint32_t j = lane; j < C; j += 64)
    if (row[j] != row[j]) last_nan = int(j);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    const int o = __shfl_xor(last_nan, m);
    last_nan = o > last_nan ? o : last_nan;
  }
  const uint32_t s = uint32_t(last_nan + 1);
  if (s >= C) return last_nan < 0 ? -FLT_MAX : row[last_nan];
  float r = -__builtin_huge_valf();
  for (uint32_t j = s + lane; j < C; j += 64) r = fmaxf(r, row[j]);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) r = fmaxf(r, __shfl_xor(r, m));
  if (r == 0.0f) {
    int zero = -1;
    for (uint32_t j = s + lane; j < C; j += 64)
      if (row[j] == 0.0f) zero = int(j);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      const int o = __shfl_xor(zero, m);
      zero = o > zero ? o : zero;
    }
    r = row[zero];
  }
  return last_nan >= 0 || r > -FLT_MAX ? r : -FLT_MAX;
}

// Row max with exact reference bits: fast block fmax + NaN flag; wave 0 refolds when
// the fast value could differ (a NaN in the row, or a zero maximum whose sign depends on order).
template <int W = kCeWaves>
__device__ __forceinline__ float row_max_exact(float m, bool nan, const float *row, uint32_t C,
                                               float *lds) {
  m = block_fmax<W>(m, lds);
  nan = block_any<W>(nan, lds);
  if (nan || m == 0.0f) {
    __syncthreads();
    if (threadIdx.x < 64) {
      const float f = wave_max_fold(row, C, int(threadIdx.x));
      if (threadIdx.x == 0) lds[W] = f;
    }
    __syncthreads();
    return lds[W];
  }
  return m > -FLT_MAX ? m : -FLT_MAX;
}

// Rows of any length and alignment in float4 units: unit q covers elements 4q .. 4q + 3, the last
// one partial. A partial unit of a row of four and more is read from four elements before the row's
// end (its first `lo` elements are the unit before's), a shorter row's element by element; elements
// [lo, hi) are the unit's own.
struct RowUnit {
  uint32_t pos, lo, hi;
};
__device__ __forceinline__ RowUnit row_unit(uint32_t q, uint32_t C) {
  const uint32_t at = 4 * q;
  if (C < 4) return RowUnit{0, 0, q == 0 ? C : 0};
  const uint32_t pos = at + 4 <= C ? at : C - 4;
  return RowUnit{pos, at < C ? at - pos : 4u, 4u};
}
// The unit's four elements (those past a row shorter than four repeat its last one).
__device__ __forceinline__ f4 load_row_part(const float *row, const RowUnit &r, uint32_t C) {
  if (C >= 4) return __builtin_nontemporal_load(reinterpret_cast<const f4u *>(row + r.pos));
  f4 v;
#pragma unroll
  for (uint32_t c = 0; c < 4; ++c) v[c] = row[c < C ? c : C - 1];
  return v;
}
// Stores the unit's own elements.
__device__ __forceinline__ void store_row_part(f4 v, float *row, const RowUnit &r) {
  if (r.lo == 0 && r.hi == 4) {
    store_unit<true>(v, row + r.pos);
    return;
  }
#pragma unroll
  for (uint32_t c = 0; c < 4; ++c)
    if (c >= r.lo && c < r.hi) row[r.pos + c] = v[c];
}

// Sum and maximum over the T lanes that share a row (T a power of two up to 64).
template <int T>
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
  for (int m = T / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m);
  return v;
}
template <int T>
__device__ __forceinline__ float group_max(float v) {
#pragma unroll
  for (int m = T / 2; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m));
  return v;
}
template <int T>
__device__ __forceinline__ float group_min(float v) {
#pragma unroll
  for (int m = T / 2; m >= 1; m >>= 1) v = fminf(v, __shfl_xor(v, m));
  return v;
}

// Lanes per row and float4 units per lane for rows held in a wave's registers: about four units a
// lane, so that a wave always has 64 lanes of loads in flight however short the rows are (a
// 256-lane workgroup per row of 10 used 10 of its lanes). f(lanes, units) with constants.
constexpr uint32_t kWaveRow = 2048;  // the longest: 64 lanes of 8 units
// Softmax takes a workgroup per row beyond these (its backward holds three operands). Forward and
// backward over three rotating inputs, wave / workgroup per row: forward [60000, 600] 145 / 181 us,
// [16384, 1000] 66.5 / 69.8, and with both in 8 units [30000, 1500] 185 / 163; backward [60000, 600]
// 145 / 157, [60000, 700] 169 / 171, [16384, 1000] 70.2 / 66.5.
constexpr uint32_t kSoftmaxWaveRow = 1024, kSoftmaxBwdWaveRow = 768;
// and with fewer rows than these, which leave the chip idle: a lane of a wave's row has 16 elements to
// exponentiate one after the other, of a workgroup's four. Wave / workgroup per row: forward [64, 300]
// 4.8 / 4.0 us, [1500, 300] 5.3 / 5.0, [3000, 300] 5.8 / 6.6, [2048, 1000] 6.4 / 6.3, [3000, 1000]
// 7.4 / 8.3; log-softmax [1024, 300] 5.0 / 4.5, [2048, 300] 5.1 / 5.5.
template <bool LOG>
constexpr uint64_t kSoftmaxFewRows = LOG ? 1536 : 2048;
// The backward's, in whole 128-byte lines, wave / workgroup: [64, 128] 3.1 / 2.6, [1024, 128] 3.2 / 3.1,
// [2048, 128] 3.2 / 3.9, [1500, 256] 4.3 / 4.7; log-softmax's [64, 512] 4.4 / 3.5, [2048, 512] 5.3 / 5.8. Where
// rows share lines, workgroups of other XCDs update them at once, and a wave's neighbours are its own:
// [64, 4] 2.9 / 4.0, [64, 300] 3.3 / 3.3, [1024, 300] 3.5 / 4.1; log-softmax's [64, 300] 3.6 / 3.3, [1024, 300]
// 3.9 / 4.2. Rows that are no whole float4 (the workgroup's three passes): [2400, 10] 3.2 / 3.7, [4096, 3]
// 3.8 / 4.3, [2048, 301] 4.3 / 4.1, [2400, 514] 5.4 / 5.7; log-softmax's [2048, 514] 5.4 / 4.6, [3000, 129]
// 4.9 / 4.4, [3000, 301] 5.4 / 5.2, [4096, 301] 5.7 / 5.9, [3000, 514] 6.3 / 6.8.
template <bool LOG>
bool softmax_bwd_waves(uint64_t N, uint64_t C) {
  if (C > kSoftmaxBwdWaveRow) return false;
  if (C % 4 != 0) return N >= (LOG ? 3072 : 2176);
  if (C % 32 != 0) return !LOG || C <= 16 || N >= 768;
  return N >= (LOG ? 1700 : 1280);
}
// Rows that are no whole float4 and no longer than this take the forward's three passes rather than a
// workgroup's registers, of whose lanes they leave most idle: [1024, 301] 4.1 / 4.5 us, [1024, 514]
// 4.7 / 4.6.
constexpr uint32_t kSoftmaxPasses = 2 * kCeBlock;
// The backward's, whose 512 lanes have twice as many idle: rows that are all resident at once (2048
// workgroups), and more of short ones while the tensors stay in the caches. Three passes / registers:
// [512, 1001] 4.1 / 4.1, [1024, 301] 3.5 / 4.5, [2048, 1001] 6.7 / 7.6, [2400, 1001] 9.1 / 8.6;
// [1024, 1301] 5.2 / 5.3, [2048, 1301] 7.9 / 8.6, [2048, 1602] 10.3 / 10.1, [512, 1301] 4.6 / 4.3; [4096, 770]
// 10.3 / 11.5, [8192, 901] 21.2 / 21.2, [8192, 1021] 26.5 / 22.4, [30000, 770] 71.6 / 64.8.
bool softmax_bwd_passes(uint64_t N, uint64_t C) {
  if (N <= 2048) return C <= (N > 1024 ? 1344u : 1024u);
  return C <= 900 && N * C < uint64_t(1) << 23;
}
template <uint32_t MAX_ROW, class F>
void with_row_lanes(uint32_t C, F &&f) {
  using std::integral_constant;
  if (C <= 32) f(integral_constant<int, 2>{}, integral_constant<int, 4>{});
  else if (C <= 128) f(integral_constant<int, 8>{}, integral_constant<int, 4>{});
  else if (C <= 512) f(integral_constant<int, 32>{}, integral_constant<int, 4>{});
  else if constexpr (MAX_ROW > 512) {
    if (C <= 1024) f(integral_constant<int, 64>{}, integral_constant<int, 4>{});
    else if constexpr (MAX_ROW > 1024) f(integral_constant<int, 64>{}, integral_constant<int, 8>{});
  }
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m));
  return v;
}
__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = fminf(v, __shfl_xor(v, m));
  return v;
}

constexpr int kCeUnroll = PLAST_CE_UNROLL;  // float4 loads in flight per lane

// A row whose fast values could differ from the reference chain's bits, by one wave from memory: the
// chain element by element. Every lane returns the row max, the log of the exp-sum, and whether a
// term of the one-hot product other than the label's is not finite.
__device__ void ce_wave_exact(const float *xr, uint32_t C, int32_t y, int lane, float &mx, float &l,
                              bool &bad) {
  mx = wave_max_fold(xr, C, lane);
  float t = 0.0f;
  for (uint32_t j = lane; j < C; j += 64) t += expf(xr[j] - mx);
  l = logf(wave_sum(t));
  bool b = false;
  for (uint32_t j = lane; j < C; j += 64) {
    const float ls = (xr[j] - mx) - l;
    if (int32_t(j) != y) b = b || !(fabsf(ls) <= FLT_MAX);
  }
  bad = __any(b);
}

// A row's loss and statistics, by one lane.
__device__ __forceinline__ void ce_row_out(const float *xr, uint32_t C, int32_t y, float mx, float l,
                                           bool bad, uint64_t row, uint64_t simd_end,
                                           float *__restrict__ loss, float *__restrict__ stats) {
  float t;
  if (bad) t = __builtin_nanf("");
  else if (y >= 0 && uint32_t(y) < C) t = 0.0f + ((xr[y] - mx) - l);
  else t = 0.0f;
  loss[row] = row < simd_end ? 0.0f - t : -t;
  stats[2 * row] = mx;
  stats[2 * row + 1] = l;
}

// Whether a row's fast maximum M, exp-sum S or smallest logit mn could stand for values the
// reference chain would give other bits: a non-finite or zero maximum, a NaN or overflowed sum, or a
// shifted and normalised logit that overflows (0 * -inf = NaN in the one-hot product).
__device__ __forceinline__ bool ce_needs_exact(float M, float S, float mn, float l) {
  return !(fabsf(M) <= FLT_MAX) || M == 0.0f || !(S <= FLT_MAX) || !(fabsf((mn - M) - l) <= FLT_MAX);
}

// Forward over rows of at most 4 * L * U floats held in registers, L lanes each. Twenty-odd
// instructions a logit at most; what bounds it is the one read. [60000, 10]: 89.9 us with a workgroup
// per row.
constexpr uint32_t kCeWaveRow = 512;  // longer rows stream through ce_fwd_wave_kernel
template <int L, int U>
__global__ __launch_bounds__(kCeBlock) void ce_fwd_rows_kernel(const float *__restrict__ x,
                                                               const int32_t *__restrict__ lab,
                                                               float *__restrict__ stats,
                                                               float *__restrict__ loss, uint64_t N,
                                                               uint32_t C, uint64_t simd_end) {
  const int lane = threadIdx.x & 63, l = lane % L;
  const uint64_t row0 = (uint64_t(blockIdx.x) * kCeWaves + (threadIdx.x >> 6)) * (64 / L);
  if (row0 >= N) return;  // whole wave
  const uint64_t row = row0 + lane / L;
  const bool valid = row < N;
  const float *xr = x + (valid ? row : N - 1) * C;
  const int32_t y = lab[valid ? row : N - 1];
  f4 v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) v[u] = load_row_part(xr, row_unit(uint32_t(l) + u * L, C), C);
  float M = -__builtin_huge_valf(), mn = __builtin_huge_valf();
#pragma unroll
  for (int u = 0; u < U; ++u)  // elements read twice change neither
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      M = fmaxf(M, v[u][c]);
      mn = fminf(mn, v[u][c]);
    }
  M = group_max<L>(M);
  mn = group_min<L>(mn);
  float S = 0.0f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const RowUnit r = row_unit(uint32_t(l) + u * L, C);
#pragma unroll
    for (uint32_t c = 0; c < 4; ++c) {
      const float e = exp_le0(v[u][c] - M);
      S += c >= r.lo && c < r.hi ? e : 0.0f;
    }
  }
  S = group_sum<L>(S);
  float mx = M, lg = logf(S);
  bool bad = false;
  for (uint64_t todo = __ballot(valid && l == 0 && ce_needs_exact(M, S, mn, lg)); todo; todo &= todo - 1) {
    const int first = __ffsll((unsigned long long)todo) - 1;  // the row's first lane
    float m1, l1;
    bool b1;
    ce_wave_exact(x + (row0 + first / L) * C, C, __shfl(y, first), lane, m1, l1, b1);
    if (lane == first) mx = m1, lg = l1, bad = b1;
  }
  if (valid && l == 0) ce_row_out(xr, C, y, mx, lg, bad, row, simd_end, loss, stats);
}

// One wave64 per row, a single read of the row. Each lane keeps an online (max, exp-sum) pair,
// rescaling its sum when its max grows; the wave merges the pairs. Rows for which ce_needs_exact
// holds are recomputed by the same wave from memory.
constexpr int kCeFwdWaves = PLAST_CE_FWD_WAVES;  // rows (waves) per workgroup

__global__ __launch_bounds__(64 * kCeFwdWaves) void ce_fwd_wave_kernel(const float *__restrict__ x,
                                                          const int32_t *__restrict__ lab,
                                                          float *__restrict__ stats,
                                                          float *__restrict__ loss, uint64_t N,
                                                          uint32_t C, uint64_t simd_end) {
  const int lane = threadIdx.x & 63;
  const uint64_t row = uint64_t(blockIdx.x) * kCeFwdWaves + (threadIdx.x >> 6);
  if (row >= N) return;  // whole wave
  const float *xr = x + row * C;
  const int32_t y = lab[row];
  const float ninf = -__builtin_huge_valf();
  float m = ninf, s = 0.0f, mn = __builtin_huge_valf();
  const uint32_t C4 = C / 4;
  const auto grow = [&](float g) {  // raise the lane's maximum to g
    s = m == ninf ? s * 0.0f : s * exp_le0(m - g);
    m = g;
  };
  for (uint32_t q0 = lane; q0 < C4; q0 += 64 * kCeUnroll) {
    f4 v[kCeUnroll];
#pragma unroll
    for (int u = 0; u < kCeUnroll; ++u) {
      const uint32_t q = q0 + uint32_t(u) * 64;
      if (q < C4) v[u] = __builtin_nontemporal_load(reinterpret_cast<const f4u *>(xr + 4 * q));
    }
#pragma unroll
    for (int u = 0; u < kCeUnroll; ++u) {
      if (q0 + uint32_t(u) * 64 >= C4) continue;
      const float g = fmaxf(fmaxf(v[u][0], v[u][1]), fmaxf(v[u][2], v[u][3]));
      if (g > m) grow(g);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float e = v[u][c];
        mn = fminf(mn, e);
        s += exp_le0(e - m);
      }
    }
  }
  if (C4 * 4 + lane < C) {  // the up to three logits after the last float4
    const float e = xr[C4 * 4 + lane];
    if (e > m) grow(e);
    mn = fminf(mn, e);
    s += exp_le0(e - m);
  }
  const float M = wave_max(m);
  const float sc = m == ninf ? s * 0.0f : s * exp_le0(m - M);
  const float S = wave_sum(sc);
  mn = wave_min(mn);
  float mx = M, l = logf(S);
  bool bad = false;
  // a NaN logit reaches the sum (fmaxf skips NaN, exp(NaN - m) does not); an infinite one makes M
  // or the minimum non-finite
  if (ce_needs_exact(M, S, mn, l)) ce_wave_exact(xr, C, y, lane, mx, l, bad);
  if (lane == 0) ce_row_out(xr, C, y, mx, l, bad, row, simd_end, loss, stats);
}

// Backward, float4 path over the flattened [N, C] gradient: one float4 per lane, its row found by
// magic division; the per-row constants are cached vector loads shared by the wave.
constexpr int kCeFlatBlock = PLAST_CE_BWD_BLOCK;

template <bool OVERWRITE>
__global__ __launch_bounds__(kCeFlatBlock) void ce_bwd_flat_kernel(const float *__restrict__ x,
                                                               const int32_t *__restrict__ lab,
                                                               const float *__restrict__ stats,
                                                               const float *__restrict__ dloss,
                                                               float *dx, MagicDiv dc4,
                                                               uint32_t units) {
  const uint32_t q = (PLAST_CE_BWD_XCD ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x) * kCeFlatBlock + threadIdx.x;
  if (q >= units) return;
  const uint32_t row = dc4.div(q);
  const uint32_t j4 = q - row * dc4.d;
  const f4 xv = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(x) + q);
  f4 dv;
  if constexpr (!OVERWRITE) dv = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(dx) + q);
  const float m = stats[2 * uint64_t(row)], l = stats[2 * uint64_t(row) + 1], g = dloss[row];
  const int32_t y = lab[row];
  f4 r;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const float sm = exp_le0((xv[c] - m) - l);
    const float oh = int32_t(j4 * 4 + c) == y ? 1.0f : 0.0f;
    const float gv = g * (sm - oh);
    if constexpr (OVERWRITE) r[c] = gv;
    else r[c] = dv[c] + gv;
  }
  store_stream<PLAST_CE_NT_STORE>(r, reinterpret_cast<f4 *>(dx) + q);
}

// The same over rows that are no whole float4: a unit's elements fall in the row of its first one and
// in those after it. [60000, 10]: 18.7 us with a workgroup per row.
template <bool OVERWRITE>
__global__ __launch_bounds__(kCeFlatBlock) void ce_bwd_ragged_kernel(const float *__restrict__ x,
                                                                 const int32_t *__restrict__ lab,
                                                                 const float *__restrict__ stats,
                                                                 const float *__restrict__ dloss,
                                                                 float *dx, MagicDiv dc, uint32_t n) {
  const uint32_t q = (PLAST_CE_BWD_XCD ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x) * kCeFlatBlock + threadIdx.x;
  const uint64_t at = uint64_t(q) * 4;
  if (at >= n) return;
  const bool whole = at + 4 <= n;
  f4 xv = f4(0.0f), dv = f4(0.0f);
  if (whole) {
    xv = __builtin_nontemporal_load(reinterpret_cast<const f4u *>(x + at));
    if constexpr (!OVERWRITE) dv = __builtin_nontemporal_load(reinterpret_cast<const f4u *>(dx + at));
  } else {
#pragma unroll
    for (uint32_t c = 0; c < 3; ++c) {
      if (at + c >= n) continue;
      xv[c] = x[at + c];
      if constexpr (!OVERWRITE) dv[c] = dx[at + c];
    }
  }
  uint32_t row = dc.div(uint32_t(at));
  uint32_t col = uint32_t(at) - row * dc.d;
  float m = stats[2 * uint64_t(row)], l = stats[2 * uint64_t(row) + 1], g = dloss[row];
  int32_t y = lab[row];
  f4 r;
#pragma unroll
  for (uint32_t c = 0; c < 4; ++c) {
    const float sm = exp_le0((xv[c] - m) - l);
    const float oh = int32_t(col) == y ? 1.0f : 0.0f;
    const float gv = g * (sm - oh);
    r[c] = OVERWRITE ? gv : dv[c] + gv;
    if (++col == dc.d && at + c + 1 < n) {  // the next element starts a row
      col = 0;
      ++row;
      m = stats[2 * uint64_t(row)], l = stats[2 * uint64_t(row) + 1], g = dloss[row];
      y = lab[row];
    }
  }
  if (whole) {
    store_unit<PLAST_CE_NT_STORE>(r, dx + at);
  } else {
#pragma unroll
    for (uint32_t c = 0; c < 3; ++c)
      if (at + c < n) dx[at + c] = r[c];
  }
}

// ---- a whole cross-entropy training step in one pass: the forward's row statistics and loss,
// the backward's dx = dloss * (softmax - onehot), and the bias gradient sum_rows dx, reading each
// logit once and writing each gradient once. Persistent workgroups of kStepBlock lanes walk rows
// in pairs taken from a device counter (in deterministic mode, rows b, b + G, b + 2G, ...); a row
// is held in registers (V float4 per lane; lanes past the row are
// masked), and the next row's loads are issued into a second register set before the current row is
// reduced, so memory keeps streaming through the row's two block reductions. Per row, with the
// forward kernel's semantics (ce_fwd_wave_kernel): M = the block max, S = sum exp(x - M) in the
// block's fixed order, l = logf(S); rows whose fast values could differ from the reference chain's
// bits (a non-finite S or M, a zero M, an overflowing shifted-normalised logit) are recomputed
// exactly from memory. Each lane adds the dx of its columns into the workgroup's column sums in LDS
// (a slot per lane and unit; a lane only ever touches its own slots, so no synchronisation is
// needed) across the workgroup's rows; at the end the workgroup writes them to part[b][C], and
// ce_step_tail adds the G rows of part in workgroup order. No atomics: the bias gradient is fixed
// by which rows each workgroup took (the static schedule of deterministic mode fixes that too).
// Registers hold the two row sets only (the column sums there would spill at 1024 lanes per
// workgroup, whose wave count caps a lane at 128 VGPRs).
// A persistent row kernel's workgroup number b, which picks its rows and its partial-sum row:
// the dispatch index, or (PLAST_ROW_XCD) that index renumbered so that each XCD holds a
// contiguous range of b.
__device__ __forceinline__ uint32_t row_block() {
  if constexpr (PLAST_ROW_XCD) return xcd_block(blockIdx.x, gridDim.x);
  else return blockIdx.x;
}

// The rows a persistent row kernel's workgroup walks under the static schedule: r, r + S, ...
// below rend, that is rows b, b + G, ..., so the grid sweeps the tensor front to back.
__device__ __forceinline__ void row_range(uint32_t N, uint32_t G, uint32_t &r, uint32_t &S,
                                          uint32_t &rend) {
  r = row_block();
  rend = N;
  S = G;
}

// Dynamic row order for the persistent row kernels. Workgroups take pairs of rows (2P, 2P + 1) in
// increasing P from a device counter, so the rows in flight across the chip stay a compact band at
// the front of the tensor and a workgroup that runs faster (on MI355X the odd XCDs stream about 8%
// slower than the even ones under these loads) takes more rows; a static schedule of rows b, b + G,
// ... leaves the fast XCDs idle at the end and spreads the band. One counter pair per kernel
// family: [next pair, workgroups done]. The workgroup that finishes last returns both to zero for
// the next launch (every earlier ticket has returned by then), so no reset is launched and a
// captured graph replays it unchanged. Launches of one family overlapping on one device would
// share the counter: the library issues them on its one stream.
enum : int { kTicketStep = 0, kTicketSoftmax = 2 };
static __device__ unsigned int g_row_tickets[4];

// One ticket (a pair index), taken by lane 0 of wave 0; every other lane gets 0. The register is
// set to 0 before the branch and the atomic returns into it, so nothing reads the atomic's result
// where the branch rejoins: the wait for it falls where lane 0 first uses it. An increment
// (global_atomic_inc, bounded by 2^32 - 1, so it never wraps here) rather than an add: the
// compiler turns a uniform add into a wave-wide form whose result it reads, with a wait for every
// outstanding load, right after the branch.
__device__ __forceinline__ uint32_t take_ticket(int family) {
  uint32_t v = 0;
  if (threadIdx.x == 0) v = atomicInc(&g_row_tickets[family], 0xffffffffu);
  return v;
}

// The end of a workgroup's ticket walk: `last` is its final ticket (its value makes lane 0 wait
// for that atomic to return); the last workgroup out zeroes the family's counters.
__device__ __forceinline__ void tickets_done(int family, uint32_t last) {
  if (threadIdx.x != 0) return;
  asm volatile("" ::"v"(last));
  __threadfence();
  if (atomicAdd(&g_row_tickets[family + 1], 1u) == gridDim.x - 1) {
    __hip_atomic_store(&g_row_tickets[family], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&g_row_tickets[family + 1], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// A row unit of the persistent row kernels: nontemporal (NT) or ordinary load.
template <bool NT>
__device__ __forceinline__ f4 load_row_unit(const f4 *p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}

// Keeps the row loads just issued where they are. Without it the compiler may move a prefetch of
// the next row down to where its values are first used (past the loop's back edge, behind the
// wait for the current row), which shortens the registers' live ranges but leaves nothing in
// flight while the current row is reduced. A compiler-only barrier: no instruction is emitted.
__device__ __forceinline__ void pin_loads() {
  asm volatile("" ::: "memory");
}

constexpr int kStepBlock = PLAST_CE_STEP_BLOCK;
// The widest row the LDS column sums allow: a float4 slot per lane and unit within 159 KiB of a
// CU's 160 (1024 lanes: 8 units, rows up to 32768 floats; 512 lanes: 16 units, 65536 floats).
constexpr int step_max_units() {
  int v = 16;
  while (v > 1 && size_t(kStepBlock) * size_t(v) * 16 > size_t(159) * 1024) v /= 2;
  return v;
}
constexpr int kStepMaxV = step_max_units();
constexpr uint64_t kStepMaxC = uint64_t(kStepBlock) * 4 * kStepMaxV;
static_assert(kScratchFloats / kStepMaxC >= 256, "the device array holds a CU-sized grid of the widest rows");

// Exact row statistics for the rare rows the fast path cannot take: the reference's serial max
// fold, then the exp-sum with expf and the "some other term is non-finite" flag of the one-hot
// product (the whole block takes this branch).
template <int W>
__device__ void ce_row_exact(const float *row, uint32_t C, int32_t y, float *lds, float &mx,
                             float &l, bool &bad) {
  constexpr int BS = W * 64;
  __syncthreads();
  if (threadIdx.x == 0) lds[W] = serial_max_fold(row, C);
  __syncthreads();
  mx = lds[W];
  float t = 0.0f;
  for (uint32_t j = threadIdx.x; j < C; j += BS) t += expf(row[j] - mx);
  l = logf(block_sum<W>(t, lds));
  bool b = false;
  for (uint32_t j = threadIdx.x; j < C; j += BS) {
    const float ls = (row[j] - mx) - l;
    if (int32_t(j) != y) b = b || !(fabsf(ls) <= FLT_MAX);
  }
  bad = block_any<W>(b, lds);
}

// RAGGED: rows of any length and alignment. A row's last unit is then partial: it is read from four
// elements before the row's end and owns its last C % 4 (a lane past the row reads it too).
template <int V, bool DYN, bool RAGGED>
__global__ __launch_bounds__(kStepBlock) void ce_step_kernel(
    const float *__restrict__ x, const int32_t *__restrict__ lab, const float *__restrict__ dloss,
    float *__restrict__ stats, float *__restrict__ loss, float *__restrict__ dx,
    float *__restrict__ part, uint32_t N, uint32_t C, uint32_t simd_end) {
  constexpr int BS = kStepBlock, W = BS / 64;
  // one area per reduction of a row: a reduction's single barrier orders its writes after every
  // read of the same area in the previous row (which precede the other reduction's barrier)
  __shared__ float red1[2 * W], red2[W], ex[W + 2];
  __shared__ uint32_t tk;  // the next pair, from lane 0 of wave 0 (dynamic order)
  extern __shared__ f4 colsum[];  // BS * V float4: the workgroup's column sums, then padding
  const uint32_t C4 = C / 4, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  // row indices are 32-bit (the host checks N < 2^32): a 64-bit bound compare would be made in
  // vector registers, which the loop head may find still tied to an in-flight memory operation
  const uint32_t G = gridDim.x;
  const uint32_t rem = RAGGED ? C % 4 : 0;
  // the first element of unit q that the unit owns (4: none)
  const auto own = [&](uint32_t q) -> uint32_t { return q < C4 ? 0 : q == C4 ? 4 - rem : 4; };
  const float ninf = -__builtin_huge_valf(), pinf = __builtin_huge_valf();
#pragma unroll
  for (int u = 0; u < V; ++u) colsum[t + uint32_t(u) * BS] = f4(0.0f);

  // The lane index is made opaque in each row step, so the per-unit offsets and masks derived
  // from it are recomputed there (a few adds) instead of being hoisted out of the row loop, where
  // they would be spilled to scratch at this register budget.
  auto lane_index = [&]() {
    uint32_t i = t;
    asm volatile("" : "+v"(i));
    return i;
  };
  // Every load is issued unconditionally (a lane past the row reads the row's last float4, and the
  // prefetch past the last row re-reads that row): a load under a branch may not have been issued,
  // so the wait before the current row's first use could not count the prefetch as outstanding and
  // would wait for it too. Lanes past the row are masked where their values are used.
  // Addresses are a row base (uniform) plus a 32-bit byte offset per lane, which the loads and
  // stores take in one register (a 64-bit address per unit would take two).
  // The row's label and upstream gradient are loaded with it, a row ahead of their use (a load
  // issued when the row's processing starts would stall it for a memory round trip).
  auto load_row = [&](uint32_t r, f4 (&v)[V], int32_t &yl, float &gl) {
    const uint32_t rc = r < N ? r : N - 1;
    yl = lab[rc];
    gl = dloss[rc];
    const char *xr = reinterpret_cast<const char *>(x + uint64_t(rc) * C);
    const uint32_t ti = lane_index();
#pragma unroll
    for (int u = 0; u < V; ++u) {
      const uint32_t q = ti + uint32_t(u) * BS;
      if constexpr (RAGGED) {
        const uint32_t off = q < C4 ? q * 16u : (C - 4) * 4u;
        v[u] = __builtin_nontemporal_load(reinterpret_cast<const f4u *>(xr + off));
      } else {
        const uint32_t off = (q < C4 ? q : C4 - 1) * 16u;
        v[u] = load_row_unit<PLAST_CE_STEP_NT_LOAD>(reinterpret_cast<const f4 *>(xr + off));
      }
    }
    pin_loads();
  };

  // One row held in v: v is overwritten with e = exp(x - M) by the sum pass, so the gradient
  // pass is one multiply per element, dx = e * (dloss / S) (the softmax exp((x - m) - l) as
  // e / S, within 2 ulp of it), with the one-hot term applied to the label's element alone. A
  // row's VALU work is then about 14 instructions per element, under the memory time (the
  // recomputed-exponential form took 36 and was issue-bound).
  // With `next`, lane 0 of wave 0 publishes `give` (a ticket) before the row's first barrier and
  // every lane reads it into *next after it.
  auto process = [&](uint32_t r, f4 (&v)[V], const int32_t y, const float g, uint32_t give,
                     uint32_t *next) {
    // Consume every unit of the row here, on every path: a unit used only under a branch that some
    // waves skip (the row's ragged last unit) would leave its load pending past the loop's back
    // edge, and reusing its registers there would wait for every load, the prefetch included.
#pragma unroll
    for (int u = 0; u < V; ++u) asm volatile("" ::"v"(v[u][0]), "v"(v[u][1]), "v"(v[u][2]), "v"(v[u][3]));
    if (next && t == 0) tk = give;
    const uint32_t ti = lane_index();
    const uint32_t full = C4 / BS;  // units every lane holds inside the row
    // first reduction: the row's max and min (lanes past the row hold a copy of its last float4, which
    // changes neither)
    float m = ninf, mn = pinf;
#pragma unroll
    for (int u = 0; u < V; ++u)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        m = fmaxf(m, v[u][c]);
        mn = fminf(mn, v[u][c]);
      }
    m = wave_max(m);
    mn = wave_min(mn);
    if (lane == 0) {
      red1[wave] = m;
      red1[W + wave] = mn;
    }
    // the label's logit, taken by the lane that holds it before the sum pass overwrites v
    const bool live = y >= 0 && uint32_t(y) < C;
    const uint32_t yq = live ? uint32_t(y) >> 2 : 0;
    // the label's element of its unit
    const int yc = RAGGED && yq == C4 ? int(uint32_t(y) - (C - 4)) : int(y & 3);
    const bool owner = ti == yq % BS;
    float xy = 0.0f;
    if (owner) {
#pragma unroll
      for (int u = 0; u < V; ++u)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (uint32_t(u) == yq / BS && c == yc) xy = v[u][c];
    }
    __syncthreads();
    if (next) *next = tk;
    float M = red1[0], MN = red1[W];
#pragma unroll
    for (int w = 1; w < W; ++w) {
      M = fmaxf(M, red1[w]);
      MN = fminf(MN, red1[W + w]);
    }
    // second reduction: e = exp(x - M) into v, and its sum. A NaN logit reaches the sum; an infinite one,
    // or an x - M that overflows, sends the row to the exact path below, so every value used from
    // here on came from a finite argument and the unclamped exponential is exact enough.
    float sl = 0.0f;
#pragma unroll
    for (int u = 0; u < V; ++u) {
      const bool in = uint32_t(u) < full || ti + uint32_t(u) * BS < C4;
      const uint32_t lo = RAGGED ? own(ti + uint32_t(u) * BS) : 0;
#pragma unroll
      for (uint32_t c = 0; c < 4; ++c) {
        const float e = exp_le0_finite(v[u][c] - M);
        v[u][c] = e;
        sl += (RAGGED ? c >= lo : in) ? e : 0.0f;
      }
    }
    sl = wave_sum(sl);
    if (lane == 0) red2[wave] = sl;
    __syncthreads();
    float S = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w) S += red2[w];
    float mx = M, l = 0.0f;
    bool exact = !(fabsf(M) <= FLT_MAX) || M == 0.0f || !(S <= FLT_MAX);
    if (!exact) {
      l = logf(S);
      // the most negative shifted-normalised logit must stay finite (else 0 * -inf = NaN)
      exact = !(fabsf((MN - mx) - l) <= FLT_MAX);
    }
    bool bad = false;
    if (exact) ce_row_exact<W>(x + uint64_t(r) * C, C, y, ex, mx, l, bad);
    // the lane holding the label's logit writes the loss and the statistics
    if (owner) {
      float tt = 0.0f;
      if (bad) tt = __builtin_nanf("");
      else if (live) tt = 0.0f + ((xy - mx) - l);
      loss[r] = r < simd_end ? 0.0f - tt : -tt;
      stats[2 * uint64_t(r)] = mx;
      stats[2 * uint64_t(r) + 1] = l;
    }
    // the gradient, written once and added into the lane's column sums
    f4 *d4 = reinterpret_cast<f4 *>(dx + uint64_t(r) * C);
    char *dr = reinterpret_cast<char *>(d4);
    if (!exact) {
      const float gs = g * (1.0f / S);
      const float inv = 1.0f / S;
      // each unit's gradient stored as soon as it is formed (the stores go out first), then the
      // column sums, whose LDS reads and writes then run back to back without a branch between
      // them (+1.4% over adding each unit before its store, in one process)
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const uint32_t q = ti + uint32_t(u) * BS;
        f4 o = v[u] * gs;
        if (owner && uint32_t(u) == yq / BS && live) {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (c == yc) o[c] = g * (v[u][c] * inv - 1.0f);
        }
        if (uint32_t(u) < full || q < C4) {
          if constexpr (RAGGED) store_unit<PLAST_CE_NT_STORE>(o, reinterpret_cast<float *>(dr + q * 16u));
          else store_stream<PLAST_CE_NT_STORE>(o, reinterpret_cast<f4 *>(dr + q * 16u));
        } else if (RAGGED && q == C4) {
#pragma unroll
          for (uint32_t c = 0; c < 4; ++c) {
            if (c >= 4 - rem) reinterpret_cast<float *>(dr)[C - 4 + c] = o[c];
            else o[c] = 0.0f;  // the unit before's column
          }
        }
        v[u] = o;
      }
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const uint32_t q = ti + uint32_t(u) * BS;
        colsum[q] = colsum[q] + v[u];  // lanes past the row add into padding slots
      }
    } else {
      // the exact statistics: the gradient from memory, as the backward op computes it
      const f4 *x4 = reinterpret_cast<const f4 *>(x + uint64_t(r) * C);
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const uint32_t q = ti + uint32_t(u) * BS;
        if (RAGGED ? q * 4 >= C : q >= C4) continue;
        const uint32_t pos = RAGGED && q == C4 ? C - 4 : q * 4;
        const f4 xv = RAGGED ? f4(*reinterpret_cast<const f4u *>(x + uint64_t(r) * C + pos)) : x4[q];
        const uint32_t lo = RAGGED ? own(q) : 0;
        f4 o;
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
          const float sm = exp_le0((xv[c] - mx) - l);
          const float oh = int32_t(pos + c) == y ? 1.0f : 0.0f;
          o[c] = c >= lo ? g * (sm - oh) : 0.0f;
        }
        colsum[q] = colsum[q] + o;
        if constexpr (!RAGGED) {
          store_stream<PLAST_CE_NT_STORE>(o, d4 + q);
        } else {
#pragma unroll
          for (uint32_t c = 0; c < 4; ++c)
            if (c >= lo) dx[uint64_t(r) * C + pos + c] = o[c];
        }
      }
    }
  };

  // Two register sets used in turn (a copy out of a set whose loads are in flight would wait for
  // them), each reloaded right after its row is processed, so one row is always in flight and the
  // youngest memory operations at the loop's back edge are loads: the loop head may reuse a
  // register a store of the previous row still reads, and that wait then leaves the prefetch alone
  // (with the stores last, it would wait for every load too). Rows go in pairs, an odd last row
  // after the loop: an exit between the pair's two rows would join the loop's back edge, and the
  // waits at the loop head would then have to assume the first set's loads were the latest issued
  // (waiting for the second set's prefetch too).
  f4 xa[V], xb[V];
  int32_t ya, yb;
  float ga, gb;
  if constexpr (DYN) {
    // pairs of rows (2P, 2P + 1) from the ticket counter; the ticket for the pair after next is
    // taken right before the first set's reload, so the wait for that reload covers it
    if (t == 0) tk = take_ticket(kTicketStep);
    __syncthreads();
    uint32_t P = tk, Pn = 0;
    uint32_t ahead = take_ticket(kTicketStep);
    load_row(2 * P, xa, ya, ga);
    load_row(2 * P + 1, xb, yb, gb);
    while (2 * P + 1 < N) {
      process(2 * P, xa, ya, ga, ahead, &Pn);
      ahead = take_ticket(kTicketStep);
      load_row(2 * Pn, xa, ya, ga);
      process(2 * P + 1, xb, yb, gb, 0, nullptr);
      load_row(2 * Pn + 1, xb, yb, gb);
      P = Pn;
    }
    if (2 * P < N) process(2 * P, xa, ya, ga, 0, nullptr);
    tickets_done(kTicketStep, ahead);
  } else {
    uint32_t r, S, rend;
    row_range(N, G, r, S, rend);
    load_row(r, xa, ya, ga);
    load_row(r + S, xb, yb, gb);
    for (; r + S < rend; r += 2 * S) {
      process(r, xa, ya, ga, 0, nullptr);
      load_row(r + 2 * S, xa, ya, ga);
      process(r + S, xb, yb, gb, 0, nullptr);
      load_row(r + 3 * S, xb, yb, gb);
    }
    if (r < rend) process(r, xa, ya, ga, 0, nullptr);
  }
  // the workgroup's column sums: partial row b of part, in dispatch order under the dynamic
  // order (the rows each workgroup took vary from run to run) and by the static schedule's
  // numbering otherwise
  if (!part) return;
  float *pb = part + uint64_t(DYN ? blockIdx.x : row_block()) * C;
#pragma unroll
  for (int u = 0; u < V; ++u) {
    const uint32_t q = t + uint32_t(u) * BS;
    if (q < C4) {
      if constexpr (RAGGED) store_unit<false>(colsum[q], pb + 4 * q);
      else reinterpret_cast<f4 *>(pb)[q] = colsum[q];
    } else if (RAGGED && q == C4) {
#pragma unroll
      for (uint32_t c = 0; c < 4; ++c)
        if (c >= 4 - rem) pb[C - 4 + c] = colsum[q][c];
    }
  }
}

// The step's tail, one launch after the row kernel: with `mean`, workgroup 0 writes the mean of
// the rows' losses; the next `nfin` workgroups (with `dbias`) sum the row kernel's column sums.
//
// dbias[c] = the sum over workgroups b = 0 .. G-1 of part[b][c], deterministically: a workgroup
// takes 32 columns; its lane group q (of 8) sums the q-th eighth of the b range in order (32 lanes
// read 32 adjacent columns, 128 B, per row), then lane c adds the 8 group sums in q order.
//
// The mean is the reference chain's last node: MEAN over the rows' losses (loss.c:161-163; the
// full reduction of reduce_ops.c:24-31 with POST_MEAN, acc / n). Its order is that of 1024 virtual
// lanes: virtual lane L sums rows L, L + 1024, ... in order, each virtual wave of 64 lanes combines
// its sums in a butterfly, and the 16 wave sums are added in wave order; a sum that overflowed
// (finite terms, not a NaN) is summed again serially in row order, as the reference's order
// decides it. Then divided by N (N = 0: 0 / 0, NaN, as the reference's mean of nothing). Lane p of
// the 256 holds virtual lanes p + 256k (k < 4), which fall in virtual wave p / 64 + 4k at the same
// position, so its four butterflies are those of the virtual waves; each lane keeps 32 loads in
// flight (8 rows of 1024 at a time), as many as four rounds over config 5's 32768 rows.
constexpr int kFinCols = 32, kFinGroups = kCeBlock / kFinCols;
// partial rows (column sums) and rows of 1024 losses (mean) loaded at a time; 16 or 32 and 16
// measured no faster (the launch's duration is not its loads' latency)
constexpr uint32_t kFinBatch = 8, kMeanRounds = 8;
constexpr uint32_t kMeanVirt = 1024, kMeanHold = kMeanVirt / kCeBlock;
static_assert(kMeanVirt % kCeBlock == 0, "the mean's virtual lanes split evenly over the workgroup");
__global__ __launch_bounds__(kCeBlock) void ce_step_tail(const float *__restrict__ part,
                                                         float *__restrict__ dbias, uint32_t C,
                                                         uint32_t G, const float *__restrict__ loss,
                                                         float *__restrict__ mean, uint32_t N) {
  __shared__ float sh[kFinGroups][kFinCols];
  const uint32_t t = threadIdx.x;
  if (mean && blockIdx.x == 0) {
    const uint32_t lane = t & 63, wave = t >> 6;
    float s[kMeanHold] = {};
    for (uint32_t i0 = t; i0 < N; i0 += kMeanVirt * kMeanRounds) {
      float v[kMeanRounds][kMeanHold];
#pragma unroll
      for (uint32_t m = 0; m < kMeanRounds; ++m)
#pragma unroll
        for (uint32_t k = 0; k < kMeanHold; ++k) {
          const uint32_t i = i0 + m * kMeanVirt + k * kCeBlock;
          v[m][k] = loss[i < N ? i : N - 1];
        }
#pragma unroll
      for (uint32_t m = 0; m < kMeanRounds; ++m)
#pragma unroll
        for (uint32_t k = 0; k < kMeanHold; ++k)
          if (i0 + m * kMeanVirt + k * kCeBlock < N) s[k] += v[m][k];
    }
    float *ws = &sh[0][0];  // the virtual waves' sums, in virtual wave order
#pragma unroll
    for (uint32_t k = 0; k < kMeanHold; ++k) {
      const float w = wave_sum(s[k]);
      if (lane == 0) ws[wave + k * (kCeBlock / 64)] = w;
    }
    __syncthreads();
    if (t != 0) return;
    float p = 0.0f;
#pragma unroll
    for (uint32_t w = 0; w < kMeanVirt / 64; ++w) p += ws[w];
    if (!(fabsf(p) <= FLT_MAX) && p == p) {
      p = 0.0f;
      for (uint32_t i = 0; i < N; ++i) p = p + loss[i];
    }
    mean[0] = p / float(N);
    return;
  }
  const uint32_t cl = t % kFinCols, q = t / kFinCols;
  const uint32_t c = (blockIdx.x - (mean ? 1u : 0u)) * kFinCols + cl;
  const uint32_t per = (G + kFinGroups - 1) / kFinGroups;
  const uint32_t b0 = q * per, b1 = b0 + per < G ? b0 + per : G;
  float s = 0.0f;
  if (c < C) {
    for (uint32_t b = b0; b < b1; b += kFinBatch) {
      float v[kFinBatch];
#pragma unroll
      for (uint32_t k = 0; k < kFinBatch; ++k)
        v[k] = b + k < b1 ? part[uint64_t(b + k) * C + c] : 0.0f;
#pragma unroll
      for (uint32_t k = 0; k < kFinBatch; ++k)
        if (b + k < b1) s += v[k];
    }
  }
  sh[q][cl] = s;
  __syncthreads();
  if (q != 0 || c >= C) return;
  float u = sh[0][cl];
#pragma unroll
  for (int g = 1; g < kFinGroups; ++g) u += sh[g][cl];
  dbias[c] = u;
}

// The step for rows of at most 4 * L * U floats (kWaveRow): L lanes hold a row in registers, 64 / L
// rows per wave, and persistent workgroups of W waves walk the row groups with the next group's loads
// in flight. A lane always holds the same columns, so their gradient sums stay in its registers
// until the end, when the workgroup's waves add up through LDS in a fixed tree and write part[b]:
// the bias gradient is the same bits on every call in either mode. Without BIAS neither the sums nor
// their registers are there ([4096, 1000] 14.9 us with, 12.0 without). One read and one write per logit
// and no barrier per row (the workgroup-per-row kernel above takes 450 us for 60000 rows of 12 to
// 1024 logits, all of it barriers and idle lanes).
// Waves per workgroup, one workgroup per CU: 16, or 8 where two sets of eight units want more than the
// 128 registers that 16 leave a lane. [60000, 128] / [60000, 512] / [60000, 1024]: 22.4 / 53.6 / 95.8 us
// with 16, 25.2 / 63.2 / 116.5 with 8, 31.6 / 96.1 / 188 with 4.
template <int U>
constexpr int kStepRowsWaves = U == 8 ? 8 : 16;

template <int L, int U, bool BIAS>
__global__ __launch_bounds__(64 * kStepRowsWaves<U>) void ce_step_rows_kernel(
    const float *__restrict__ x, const int32_t *__restrict__ lab, const float *__restrict__ dloss,
    float *__restrict__ stats, float *__restrict__ loss, float *__restrict__ dx,
    float *__restrict__ part, uint32_t N, uint32_t C, uint32_t simd_end) {
  constexpr int W = kStepRowsWaves<U>, P = 64 / L;  // rows per wave
  __shared__ f4 sh[W / 2][L * U];
  const int lane = threadIdx.x & 63, l = lane % L;
  const uint32_t wave = threadIdx.x >> 6, groups = (N + P - 1) / P;
  f4 acc[U];
#pragma unroll
  for (int u = 0; u < U; ++u) acc[u] = f4(0.0f);
  // group `gr`'s row of this lane (the last row again past the end), its label and upstream gradient
  const auto load = [&](uint32_t gr, f4 (&v)[U], int32_t &y, float &g) {
    const uint32_t r = gr * P + lane / L < N && gr < groups ? gr * P + lane / L : N - 1;
    y = lab[r];
    g = dloss[r];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = load_row_part(x + uint64_t(r) * C, row_unit(uint32_t(l) + u * L, C), C);
    pin_loads();
  };
  const auto process = [&](uint32_t gr, f4 (&v)[U], const int32_t y, const float g) {
    const uint32_t r = gr * P + lane / L;
    const bool valid = r < N;
    float M = -__builtin_huge_valf(), mn = __builtin_huge_valf();
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        M = fmaxf(M, v[u][c]);
        mn = fminf(mn, v[u][c]);
      }
    M = group_max<L>(M);
    mn = group_min<L>(mn);
    float S = 0.0f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const RowUnit ru = row_unit(uint32_t(l) + u * L, C);
#pragma unroll
      for (uint32_t c = 0; c < 4; ++c) {
        const float e = exp_le0(v[u][c] - M);
        v[u][c] = e;
        S += c >= ru.lo && c < ru.hi ? e : 0.0f;
      }
    }
    S = group_sum<L>(S);
    float mx = M, lg = logf(S);
    bool bad = false, exact = valid && ce_needs_exact(M, S, mn, lg);
    for (uint64_t todo = __ballot(exact && l == 0); todo; todo &= todo - 1) {
      const int first = __ffsll((unsigned long long)todo) - 1;  // the row's first lane
      float m1, l1;
      bool b1;
      ce_wave_exact(x + uint64_t(gr * P + first / L) * C, C, __shfl(y, first), lane, m1, l1, b1);
      if (lane / L == first / L) mx = m1, lg = l1, bad = b1;
    }
    if (!valid) return;
    const float *xr = x + uint64_t(r) * C;
    float *dr = dx + uint64_t(r) * C;
    if (l == 0) ce_row_out(xr, C, y, mx, lg, bad, r, simd_end, loss, stats);
    const float inv = 1.0f / S, gs = g * inv;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const RowUnit ru = row_unit(uint32_t(l) + u * L, C);
      f4 o;
      if (exact) {  // from memory, as the backward op computes it
        const f4 xv = load_row_part(xr, ru, C);
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
          const float sm = exp_le0((xv[c] - mx) - lg);
          o[c] = g * (sm - (int32_t(ru.pos + c) == y ? 1.0f : 0.0f));
        }
      } else {
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c)
          o[c] = int32_t(ru.pos + c) == y ? g * (v[u][c] * inv - 1.0f) : v[u][c] * gs;
      }
      store_row_part(o, dr, ru);
#pragma unroll
      for (uint32_t c = 0; BIAS && c < 4; ++c) acc[u][c] += c >= ru.lo && c < ru.hi ? o[c] : 0.0f;
    }
  };
  // wave w of workgroup b takes groups (w, b), (w + W, b), ... numbered w * G + b: the first G groups
  // go to the workgroups' first waves
  const uint32_t G = gridDim.x, step = G * W;
  f4 va[U], vb[U];
  int32_t ya, yb;
  float ga, gb;
  uint32_t gr = wave * G + blockIdx.x;
  load(gr, va, ya, ga);
  for (; gr < groups; gr += 2 * step) {
    load(gr + step, vb, yb, gb);
    process(gr, va, ya, ga);
    load(gr + 2 * step, va, ya, ga);
    if (gr + step < groups) process(gr + step, vb, yb, gb);
  }
  if constexpr (!BIAS) return;
  // the wave's rows: lanes with the same l
#pragma unroll
  for (int m = L; m < 64; m <<= 1)
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[u][c] += __shfl_xor(acc[u][c], m);
  // the workgroup's waves: the upper half hands its sums to the lower half, which halves again
#pragma unroll
  for (uint32_t h = W / 2; h >= 1; h /= 2) {
    if (wave >= h && wave < 2 * h && lane < L) {
#pragma unroll
      for (int u = 0; u < U; ++u) sh[wave - h][l + u * L] = acc[u];
    }
    __syncthreads();
    if (wave < h && lane < L) {
#pragma unroll
      for (int u = 0; u < U; ++u) acc[u] = acc[u] + sh[wave][l + u * L];
    }
    __syncthreads();
  }
  if (wave != 0 || lane >= L) return;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const RowUnit ru = row_unit(uint32_t(l) + u * L, C);
#pragma unroll
    for (uint32_t c = 0; c < 4; ++c)
      if (c >= ru.lo && c < ru.hi) part[uint64_t(blockIdx.x) * C + ru.pos + c] = acc[u][c];
  }
}

// Whether ce_step_kernel<V> may be launched with its dynamic LDS (raising its limit once: beyond
// the default the kernel has to opt in).
template <int V>
bool ce_step_lds_ok() {
  static bool granted = false;
  if (granted) return true;
  const int bytes = kStepBlock * V * int(sizeof(f4));
  for (const void *k : {reinterpret_cast<const void *>(&ce_step_kernel<V, true, false>),
                        reinterpret_cast<const void *>(&ce_step_kernel<V, false, false>),
                        reinterpret_cast<const void *>(&ce_step_kernel<V, false, true>)})
    if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
      (void)hipGetLastError();  // not an error of the call: the caller takes the three passes
      return false;
    }
  granted = true;
  return true;
}

// The float4 units per lane for rows of C floats from V up (0: none of this build's kernels).
template <int V>
int ce_step_units(uint64_t C) {
  if constexpr (V > kStepMaxV) {
    return 0;
  } else {
    if (C <= uint64_t(kStepBlock) * 4 * V) return ce_step_lds_ok<V>() ? V : 0;
    return ce_step_units<V * 2>(C);
  }
}

// The one-pass step with V units per lane over `grid` workgroups, their column sums in
// part[grid][C].
template <int V>
void ce_step_launch_v(int want, unsigned grid, float *part, const float *logits,
                      const int32_t *labels, const float *dloss, float *stats, float *loss,
                      float *dlogits, uint32_t N, uint32_t C) {
  if constexpr (V <= kStepMaxV) {
    if (want != V) {
      ce_step_launch_v<V * 2>(want, grid, part, logits, labels, dloss, stats, loss, dlogits, N, C);
      return;
    }
    const size_t lds = size_t(kStepBlock) * V * sizeof(f4);
    const auto run = [&](auto dynamic, auto ragged) {
      ce_step_kernel<V, decltype(dynamic)::value, decltype(ragged)::value>
          <<<grid, kStepBlock, lds, stream()>>>(logits, labels, dloss, stats, loss, dlogits, part, N, C,
                                                uint32_t(simd_end(N)));
    };
    // the dynamic row order unless results must not depend on timing (plast_hip_set_deterministic);
    // rows that are no whole float4 and short ones always keep the static one, as their bias gradient
    // has been the same bits on every call
    if (C % 4 != 0 || !aligned16(logits) || !aligned16(dlogits)) run(std::false_type{}, std::true_type{});
    else if (deterministic() || C <= kWaveRow) run(std::false_type{}, std::false_type{});
    else run(std::true_type{}, std::false_type{});
  }
}

// Whether the step's rows share waves (ce_step_rows_kernel): rows up to kWaveRow, but for so few that
// each CU has one at most, which a workgroup per row does in one round ([64, 10] 7.4 us, 9.7 in
// waves, [256, 1000] 9.0 and 9.8, [16, 2048] 7.2 and 11.7; [400, 300] 10.2 and 9.9).
bool step_in_waves(uint64_t N, uint64_t C) {
  return C <= kWaveRow && (C < 4 || N > uint64_t(num_cus()));
}

// The one-pass step's arguments: -1 (after reporting) when unusable, 0 when the rows need the three
// passes, else the float4 units per lane of the register-resident row (its LDS opt-in granted).
int ce_step_form(const float *logits, const int32_t *labels, const float *dloss, const float *stats,
                 const float *loss, const float *dlogits, uint64_t N, uint64_t C,
                 const char *where) {
  if (!logits || !labels || !dloss || !stats || !loss || !dlogits) {
    report_error(where, "logits, labels, dloss, stats, loss and dlogits are required");
    return -1;
  }
  if (C == 0 || C >= (uint64_t(1) << 31)) {
    report_error(where, "rows of %llu elements are not supported", (unsigned long long)C);
    return -1;
  }
  if (N >= (uint64_t(1) << 31)) {
    report_error(where, "more than 2^31 rows are not supported (%llu)", (unsigned long long)N);
    return -1;
  }
  // the column sums live in LDS (one float4 slot per lane and unit, the row's plus padding): the
  // kernel must be allowed that much of it
  if (step_in_waves(N, C)) return 1;
  if (C <= kStepMaxC) return ce_step_units<1>(C);
  return 0;
}

// The one-pass step's workgroup count, shared by the allocating and the allocation-free entry
// points so that both sum the bias gradient in the same order: one workgroup per row up to
// PLAST_CE_STEP_WPC per CU, and no more than the allocation-free step's device array holds column
// sums for (kScratchFloats / C; on MI355X, 256 CUs of rows up to 32768 floats, never binding).
uint64_t ce_step_grid(uint64_t N, uint64_t C) {
  uint64_t grid = uint64_t(num_cus()) * PLAST_CE_STEP_WPC;
  if (step_in_waves(N, C)) {
    // four row groups per workgroup before another one is added: each adds a row to the tail's sum
    uint64_t rows = 1;
    with_row_lanes<kWaveRow>(uint32_t(C), [&](auto lanes, auto) { rows = 4 * (64 / decltype(lanes)::value); });
    const uint64_t need = (N + rows - 1) / rows;
    return need < grid ? need : grid;
  }
  if (grid > kScratchFloats / C) grid = kScratchFloats / C;
  return N < grid ? N : grid;
}

// The step's tail: dbias from the column sums part[G][C] when dbias is wanted, and the mean of
// loss[0 .. N) when mean_loss is; one launch, or none when neither is wanted.
void step_tail(const float *part, float *dbias, uint64_t C, unsigned G, const float *loss,
               float *mean_loss, uint64_t N) {
  const uint64_t nfin = dbias ? ceil_div(C, kFinCols) : 0;
  const uint64_t blocks = nfin + (mean_loss ? 1 : 0);
  if (blocks)
    ce_step_tail<<<unsigned(blocks), kCeBlock, 0, stream()>>>(part, dbias, uint32_t(C), G, loss,
                                                             mean_loss, uint32_t(N));
}

// The one-pass step over `grid` workgroups with their column sums in part[grid][C], then the tail:
// their sum into dbias and the loss's mean, as wanted.
void ce_step_launch(int V, unsigned grid, float *part, const float *logits, const int32_t *labels,
                    const float *dloss, float *stats, float *loss, float *dlogits, float *dbias,
                    float *mean_loss, uint64_t N, uint64_t C) {
  const uint32_t c32 = uint32_t(C);
  if (!dbias) part = nullptr;  // the kernels then leave their sums where they are
  if (step_in_waves(N, C))
    with_row_lanes<kWaveRow>(c32, [&](auto lanes, auto units) {
      constexpr int L = decltype(lanes)::value, U = decltype(units)::value;
      const auto rows = [&](auto bias) {
        ce_step_rows_kernel<L, U, decltype(bias)::value><<<grid, 64 * kStepRowsWaves<U>, 0, stream()>>>(
            logits, labels, dloss, stats, loss, dlogits, part, uint32_t(N), c32, uint32_t(simd_end(N)));
      };
      if (part) rows(std::true_type{});
      else rows(std::false_type{});
    });
  else
    ce_step_launch_v<1>(V, grid, part, logits, labels, dloss, stats, loss, dlogits, uint32_t(N), c32);
  step_tail(part, dbias, C, grid, loss, mean_loss, N);
}

bool check_ce(const Tensor *x, const Tensor *lab, const Tensor *st, const char *where) {
  if (x->dtype != FLOAT32 || x->ndim != 2 || !contiguous(x)) {
    report_error(where, "logits must be a contiguous fp32 [N, C] tensor");
    return false;
  }
  if (lab->dtype != INT32 || numel(lab) != x->shape[0] || !contiguous(lab)) {
    report_error(where, "labels must be a contiguous int32 tensor of N elements");
    return false;
  }
  if (st->dtype != FLOAT32 || numel(st) != 2 * x->shape[0] || !contiguous(st)) {
    report_error(where, "stats must be a contiguous fp32 tensor of 2N elements");
    return false;
  }
  if (x->shape[1] >= (uint64_t(1) << 31)) {
    report_error(where, "rows longer than 2^31 elements are not supported");
    return false;
  }
  return true;
}

// ---- softmax and log-softmax over the last axis. The reference composes them in Python
// (plast/nn/functional.py:75-97): MAX(dim, keepdim) -> SUB -> EXP -> SUM(dim, keepdim) -> DIV for
// softmax, -> LOG -> SUB for log-softmax. One workgroup per row: the reference's max (bit-exact),
// s = sum_j expf(x_j - m) in the block's fixed order (the reference sums serially), then
// y = expf(x - m) / s or (x - m) - logf(s): every other step is the reference's own operation.
template <bool LOG>
__global__ __launch_bounds__(kCeBlock) void softmax_fwd_kernel(const float *__restrict__ x,
                                                               float *__restrict__ y, uint32_t C) {
  __shared__ float lds[kCeWaves + 1];
  const uint64_t row = blockIdx.x;
  const float *xr = x + row * C;
  float *yr = y + row * C;
  float m = -__builtin_huge_valf();
  bool nan = false;
  for (uint32_t j = threadIdx.x; j < C; j += kCeBlock) {
    const float v = xr[j];
    m = fmaxf(m, v);
    nan = nan || v != v;
  }
  const float mx = row_max_exact(m, nan, xr, C, lds);
  float s = 0.0f;
  for (uint32_t j = threadIdx.x; j < C; j += kCeBlock) s += expf(xr[j] - mx);
  s = block_sum(s, lds);
  if constexpr (LOG) {
    const float l = logf(s);
    for (uint32_t j = threadIdx.x; j < C; j += kCeBlock) yr[j] = (xr[j] - mx) - l;
  } else {
    for (uint32_t j = threadIdx.x; j < C; j += kCeBlock) yr[j] = expf(xr[j] - mx) / s;
  }
}

// Softmax / log-softmax forward over rows of at most 4 * L * U floats in a wave's registers, L lanes
// each: the operations of softmax_fwd_kernel, with the row's sum in the lanes' fixed tree. No
// barrier, and a wave's loads fill its lanes whatever the row length.
template <bool LOG, int L, int U>
__global__ __launch_bounds__(kCeBlock) void softmax_fwd_rows_kernel(const float *__restrict__ x,
                                                                    float *__restrict__ y, uint64_t N,
                                                                    uint32_t C) {
  const int lane = threadIdx.x & 63, l = lane % L;
  const uint64_t row0 = (uint64_t(blockIdx.x) * kCeWaves + (threadIdx.x >> 6)) * (64 / L);
  if (row0 >= N) return;  // whole wave
  const uint64_t row = row0 + lane / L;
  const bool valid = row < N;
  const float *xr = x + (valid ? row : N - 1) * C;
  f4 v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) v[u] = load_row_part(xr, row_unit(uint32_t(l) + u * L, C), C);
  float M = -__builtin_huge_valf(), nan = 0.0f;
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      M = fmaxf(M, v[u][c]);
      nan = v[u][c] != v[u][c] ? 1.0f : nan;
    }
  M = group_max<L>(M);
  nan = group_max<L>(nan);
  float mx = M > -FLT_MAX ? M : -FLT_MAX;
  for (uint64_t todo = __ballot(valid && l == 0 && (nan != 0.0f || M == 0.0f)); todo; todo &= todo - 1) {
    const int first = __ffsll((unsigned long long)todo) - 1;  // the row's first lane
    const float m1 = wave_max_fold(x + (row0 + first / L) * C, C, lane);
    if (lane / L == first / L) mx = m1;
  }
  float s = 0.0f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const RowUnit r = row_unit(uint32_t(l) + u * L, C);
#pragma unroll
    for (uint32_t c = 0; c < 4; ++c) {
      const float t = v[u][c] - mx;
      const float e = expf(t);
      v[u][c] = LOG ? t : e;
      s += c >= r.lo && c < r.hi ? e : 0.0f;
    }
  }
  s = group_sum<L>(s);
  const float lg = LOG ? logf(s) : 0.0f;
  if (!valid) return;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const RowUnit r = row_unit(uint32_t(l) + u * L, C);
    f4 o;
#pragma unroll
    for (int c = 0; c < 4; ++c) o[c] = LOG ? v[u][c] - lg : v[u][c] / s;
    store_row_part(o, y + row * C, r);
  }
}

constexpr int kSoftmaxBlock = PLAST_SOFTMAX_BLOCK;

// The same with the row held in registers, for rows of up to BS * 4 * V floats: one read and one
// write per element. Each lane keeps V units of the row; lanes past the row hold -inf, which adds
// exp(-inf) = 0 to no sum (they are masked) and never wins the max. Same operations and order as
// softmax_fwd_kernel's three passes but the exp-sum's grouping (per lane, then the block's fixed
// tree). RAGGED: rows of any length and alignment (RowUnit; [30000, 1500] forward and backward 180 us
// with it, 164 without).
template <bool LOG, int V, bool RAGGED, int BS = kSoftmaxBlock>
__global__ __launch_bounds__(BS) void softmax_fwd_reg_kernel(const float *__restrict__ x,
                                                             float *__restrict__ y, uint32_t C) {
  constexpr int W = BS / 64;
  __shared__ float lds[W + 1];
  const uint64_t row = blockIdx.x;
  const float *xr = x + row * C;
  const uint32_t C4 = (C + 3) / 4;
  const float ninf = -__builtin_huge_valf();
  f4 v[V];
  float m = ninf;
  bool nan = false;
#pragma unroll
  for (int u = 0; u < V; ++u) {
    const uint32_t q = threadIdx.x + uint32_t(u) * BS;
    if constexpr (RAGGED) v[u] = q < C4 ? load_row_part(xr, row_unit(q, C), C) : f4(ninf);
    else v[u] = q < C4 ? __builtin_nontemporal_load(reinterpret_cast<const f4 *>(xr) + q) : f4(ninf);
  }
#pragma unroll
  for (int u = 0; u < V; ++u) {
    m = fmaxf(m, fmaxf(fmaxf(v[u][0], v[u][1]), fmaxf(v[u][2], v[u][3])));
    nan = nan || v[u][0] != v[u][0] || v[u][1] != v[u][1] || v[u][2] != v[u][2] ||
          v[u][3] != v[u][3];
  }
  const float mx = row_max_exact<W>(m, nan, xr, C, lds);
  float s = 0.0f;
#pragma unroll
  for (int u = 0; u < V; ++u) {
    const uint32_t q = threadIdx.x + uint32_t(u) * BS;
    const uint32_t lo = RAGGED && q < C4 ? row_unit(q, C).lo : 0;
#pragma unroll
    for (uint32_t c = 0; c < 4; ++c) {
      const float t = v[u][c] - mx;
      const float e = expf(t);
      v[u][c] = LOG ? t : e;
      s += q < C4 && c >= lo ? e : 0.0f;
    }
  }
  s = block_sum<W>(s, lds);
  const float l = LOG ? logf(s) : 0.0f;
#pragma unroll
  for (int u = 0; u < V; ++u) {
    const uint32_t q = threadIdx.x + uint32_t(u) * BS;
    if (q >= C4) continue;
    f4 r;
#pragma unroll
    for (int c = 0; c < 4; ++c) r[c] = LOG ? v[u][c] - l : v[u][c] / s;
    if constexpr (RAGGED) store_row_part(r, y + row * C, row_unit(q, C));
    else reinterpret_cast<f4 *>(y + row * C)[q] = r;
  }
}

// Softmax / log-softmax forward over rows of whole float4 (up to kStepBlock * 4 * V floats) by
// persistent kStepBlock-lane workgroups, one per CU, walking rows G apart with the next row's loads
// in flight while the current one is reduced: the row loop of ce_step_kernel (two register sets,
// unconditional clamped loads, every loaded value consumed on every path). Per row: the reference's
// max (row_max_exact's rules: the fast maximum unless the row holds a NaN or its maximum is zero,
// then the serial fold), then e = exp(x - max) and its sum in the block's fixed order, then
// y = e * (1 / S) or (x - max) - log S. Without a NaN every x - max is <= 0 or -inf, where exp_le0
// holds (about 1 ulp); a row with a NaN, whose fold may stop below some elements, takes expf and a
// division.
template <bool LOG, int V, bool DYN>
__global__ __launch_bounds__(kStepBlock) void softmax_fwd_step_kernel(const float *__restrict__ x,
                                                                      float *__restrict__ y,
                                                                      uint32_t N, uint32_t C) {
  constexpr int BS = kStepBlock, W = BS / 64;
  // one area per reduction of a row (see ce_step_kernel)
  __shared__ float red1[2 * W], red2[W], ex[2];
  __shared__ uint32_t tk;  // the next pair, from lane 0 of wave 0 (dynamic order)
  const uint32_t C4 = C / 4, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint32_t G = gridDim.x;
  const float ninf = -__builtin_huge_valf();
  auto lane_index = [&]() {
    uint32_t i = t;
    asm volatile("" : "+v"(i));
    return i;
  };
  auto load_row = [&](uint32_t r, f4 (&v)[V]) {
    const char *xr = reinterpret_cast<const char *>(x + uint64_t(r < N ? r : N - 1) * C);
    const uint32_t ti = lane_index();
#pragma unroll
    for (int u = 0; u < V; ++u) {
      const uint32_t q = ti + uint32_t(u) * BS;
      const uint32_t off = (q < C4 ? q : C4 - 1) * 16u;
      v[u] = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(xr + off));
    }
    pin_loads();
  };
  // process(r, v, give, next): with `next`, lane 0 of wave 0 publishes `give` (a ticket) before the
  // row's first barrier and every lane reads it into *next after it
  auto process = [&](uint32_t r, f4 (&v)[V], uint32_t give, uint32_t *next) {
#pragma unroll
    for (int u = 0; u < V; ++u) asm volatile("" ::"v"(v[u][0]), "v"(v[u][1]), "v"(v[u][2]), "v"(v[u][3]));
    if (next && t == 0) tk = give;
    const uint32_t ti = lane_index();
    const uint32_t full = C4 / BS;
    // first reduction: the fast maximum and whether the row holds a NaN (lanes past the row hold a copy of
    // its last float4, which changes neither)
    float m = ninf;
    bool nan = false;
#pragma unroll
    for (int u = 0; u < V; ++u)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        m = fmaxf(m, v[u][c]);
        nan = nan || v[u][c] != v[u][c];
      }
    m = wave_max(m);
    const float nanw = wave_max(nan ? 1.0f : 0.0f);
    if (lane == 0) {
      red1[wave] = m;
      red1[W + wave] = nanw;
    }
    __syncthreads();
    if (next) *next = tk;
    float M = red1[0], anynan = red1[W];
#pragma unroll
    for (int w = 1; w < W; ++w) {
      M = fmaxf(M, red1[w]);
      anynan = fmaxf(anynan, red1[W + w]);
    }
    const bool special = anynan != 0.0f;
    float mx;
    if (special || M == 0.0f) {
      if (t == 0) ex[0] = serial_max_fold(x + uint64_t(r) * C, C);
      __syncthreads();
      mx = ex[0];
    } else {
      mx = M > -FLT_MAX ? M : -FLT_MAX;
    }
    // second reduction: e = exp(x - mx), kept in v (log-softmax keeps x - mx), and the row's sum. A row with
    // a NaN is summed from memory with expf instead (rare; it keeps the registers of the fast
    // path free), each lane over the same elements in the same order as the fast path.
    const f4 *x4 = reinterpret_cast<const f4 *>(x + uint64_t(r) * C);
    float sl = 0.0f;
    if (!special) {
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const bool in = uint32_t(u) < full || ti + uint32_t(u) * BS < C4;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float d = v[u][c] - mx;
          const float e = exp_le0(d);
          v[u][c] = LOG ? d : e;
          sl += in ? e : 0.0f;
        }
      }
    } else {
      for (uint32_t q = ti; q < C4; q += BS) {
        const f4 xv = x4[q];
#pragma unroll
        for (int c = 0; c < 4; ++c) sl += expf(xv[c] - mx);
      }
    }
    sl = wave_sum(sl);
    if (lane == 0) red2[wave] = sl;
    __syncthreads();
    float S = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w) S += red2[w];
    f4 *y4 = reinterpret_cast<f4 *>(y + uint64_t(r) * C);
    char *dr = reinterpret_cast<char *>(y4);
    const float l = LOG ? logf(S) : 0.0f;
    if (!special) {
      const float inv = 1.0f / S;
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const uint32_t q = ti + uint32_t(u) * BS;
        f4 o;
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] = LOG ? v[u][c] - l : v[u][c] * inv;
        if (uint32_t(u) < full || q < C4)
          store_stream<true>(o, reinterpret_cast<f4 *>(dr + q * 16u));
      }
    } else {
      for (uint32_t q = ti; q < C4; q += BS) {
        const f4 xv = x4[q];
        f4 o;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float d = xv[c] - mx;
          o[c] = LOG ? d - l : expf(d) / S;
        }
        y4[q] = o;
      }
    }
  };
  f4 xa[V], xb[V];
  if constexpr (DYN) {
    // pairs of rows (2P, 2P + 1) from the ticket counter; the ticket for the pair after next is
    // taken right before the first set's reload, so the wait for that reload covers it
    if (t == 0) tk = take_ticket(kTicketSoftmax);
    __syncthreads();
    uint32_t P = tk, Pn = 0;
    uint32_t ahead = take_ticket(kTicketSoftmax);
    load_row(2 * P, xa);
    load_row(2 * P + 1, xb);
    while (2 * P + 1 < N) {
      process(2 * P, xa, ahead, &Pn);
      ahead = take_ticket(kTicketSoftmax);
      load_row(2 * Pn, xa);
      process(2 * P + 1, xb, 0, nullptr);
      load_row(2 * Pn + 1, xb);
      P = Pn;
    }
    if (2 * P < N) process(2 * P, xa, 0, nullptr);
    tickets_done(kTicketSoftmax, ahead);
  } else {
    uint32_t r, S, rend;
    row_range(N, G, r, S, rend);
    load_row(r, xa);
    load_row(r + S, xb);
    // rows in pairs, an odd last row after the loop (see ce_step_kernel)
    for (; r + S < rend; r += 2 * S) {
      process(r, xa, 0, nullptr);
      load_row(r + 2 * S, xa);
      process(r + S, xb, 0, nullptr);
      load_row(r + 3 * S, xb);
    }
    if (r < rend) process(r, xa, 0, nullptr);
  }
}

// Backward from the forward output y: dx += y * (dy - sum_j dy_j y_j) (softmax) or
// dx += dy - expf(y) * sum_j dy_j (log-softmax), the gradient of the reference chain (its MAX
// branch contributes zero in exact arithmetic); the row sum in the block's fixed order.
template <bool LOG>
__global__ __launch_bounds__(kCeBlock) void softmax_bwd_kernel(const float *__restrict__ y,
                                                               const float *__restrict__ dy,
                                                               float *dx, uint32_t C) {
  __shared__ float lds[kCeWaves + 1];
  const uint64_t row = blockIdx.x;
  const float *yr = y + row * C, *gr = dy + row * C;
  float *dr = dx + row * C;
  float t = 0.0f;
  for (uint32_t j = threadIdx.x; j < C; j += kCeBlock) t += LOG ? gr[j] : gr[j] * yr[j];
  t = block_sum(t, lds);
  for (uint32_t j = threadIdx.x; j < C; j += kCeBlock) {
    const float g = LOG ? gr[j] - expf(yr[j]) * t : yr[j] * (gr[j] - t);
    dr[j] = dr[j] + g;
  }
}

// The same over rows of at most 4 * L * U floats in a wave's registers, L lanes each.
template <bool LOG, int L, int U>
__global__ __launch_bounds__(kCeBlock) void softmax_bwd_rows_kernel(const float *__restrict__ y,
                                                                    const float *__restrict__ dy,
                                                                    float *dx, uint64_t N, uint32_t C) {
  const int lane = threadIdx.x & 63, l = lane % L;
  const uint64_t row0 = (uint64_t(blockIdx.x) * kCeWaves + (threadIdx.x >> 6)) * (64 / L);
  if (row0 >= N) return;  // whole wave
  const bool valid = row0 + lane / L < N;
  const uint64_t row = valid ? row0 + lane / L : N - 1;
  f4 yv[U], gv[U], dv[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const RowUnit r = row_unit(uint32_t(l) + u * L, C);
    yv[u] = load_row_part(y + row * C, r, C);
    gv[u] = load_row_part(dy + row * C, r, C);
    dv[u] = load_row_part(dx + row * C, r, C);
  }
  float t = 0.0f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const RowUnit r = row_unit(uint32_t(l) + u * L, C);
#pragma unroll
    for (uint32_t c = 0; c < 4; ++c)
      t += c >= r.lo && c < r.hi ? (LOG ? gv[u][c] : gv[u][c] * yv[u][c]) : 0.0f;
  }
  t = group_sum<L>(t);
  if (!valid) return;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const RowUnit r = row_unit(uint32_t(l) + u * L, C);
    f4 d = dv[u];
#pragma unroll
    for (int c = 0; c < 4; ++c)
      d[c] = d[c] + (LOG ? gv[u][c] - expf(yv[u][c]) * t : yv[u][c] * (gv[u][c] - t));
    store_row_part(d, dx + row * C, r);
  }
}

// The backward with y and dy of a row held in registers (rows of whole float4 up to BS * 4 * V
// floats): y, dy and dx are each read once and dx written once. The sum's grouping is per lane,
// then the block's fixed tree.
// RAGGED: rows of any length and alignment, their last unit partial (RowUnit).
template <bool LOG, int V, int BS, bool RAGGED>
__global__ __launch_bounds__(BS) void softmax_bwd_reg_kernel(const float *__restrict__ y,
                                                             const float *__restrict__ dy,
                                                             float *dx, uint32_t C) {
  constexpr int W = BS / 64;
  __shared__ float lds[W + 1];
  const uint64_t row = blockIdx.x;
  const uint32_t C4 = RAGGED ? (C + 3) / 4 : C / 4;
  const f4 *y4 = reinterpret_cast<const f4 *>(y + row * C);
  const f4 *g4 = reinterpret_cast<const f4 *>(dy + row * C);
  f4 *d4 = reinterpret_cast<f4 *>(dx + row * C);
  // Loads are unconditional (a lane past the row reads the row's last float4, masked where it is
  // used): the compiler waits for every outstanding load before the first use of a lane-masked
  // one.
  // the first kPre units of dx (all of them by default) are loaded with y and dy, so that their
  // latency overlaps the row's reduction
  constexpr int kPre = PLAST_SOFTMAX_BWD_PRE < V ? PLAST_SOFTMAX_BWD_PRE : V;
  f4 yv[V], gv[V], dv[kPre > 0 ? kPre : 1];
#pragma unroll
  for (int u = 0; u < V; ++u) {
    const uint32_t q = threadIdx.x + uint32_t(u) * BS;
    const uint32_t qc = q < C4 ? q : C4 - 1;
    if constexpr (RAGGED) {
      const RowUnit r = row_unit(qc, C);
      yv[u] = load_row_part(y + row * C, r, C);
      gv[u] = load_row_part(dy + row * C, r, C);
      if (u < kPre) dv[u] = load_row_part(dx + row * C, r, C);
      continue;
    }
    yv[u] = __builtin_nontemporal_load(y4 + qc);
    gv[u] = __builtin_nontemporal_load(g4 + qc);
    if (u < kPre) dv[u] = PLAST_SOFTMAX_BWD_NT ? __builtin_nontemporal_load(d4 + qc) : d4[qc];
  }
  float t = 0.0f;
#pragma unroll
  for (int u = 0; u < V; ++u) {
    const uint32_t q = threadIdx.x + uint32_t(u) * BS;
    const uint32_t lo = RAGGED && q < C4 ? row_unit(q, C).lo : 0;
#pragma unroll
    for (uint32_t c = 0; c < 4; ++c) t += q < C4 && c >= lo ? (LOG ? gv[u][c] : gv[u][c] * yv[u][c]) : 0.0f;
  }
  t = block_sum<W>(t, lds);
#pragma unroll
  for (int u = 0; u < V; ++u) {
    const uint32_t q = threadIdx.x + uint32_t(u) * BS;
    if (q >= C4) continue;
    f4 d;
    if (u < kPre) d = dv[u < kPre ? u : 0];
    else if constexpr (RAGGED) d = load_row_part(dx + row * C, row_unit(q, C), C);
    else d = PLAST_SOFTMAX_BWD_NT ? __builtin_nontemporal_load(d4 + q) : d4[q];
#pragma unroll
    for (int c = 0; c < 4; ++c)
      d[c] = d[c] + (LOG ? gv[u][c] - expf(yv[u][c]) * t : yv[u][c] * (gv[u][c] - t));
    if constexpr (RAGGED) store_row_part(d, dx + row * C, row_unit(q, C));
    else store_stream<PLAST_SOFTMAX_BWD_NT>(d, d4 + q);
  }
}

bool check_softmax(const Tensor *x, const Tensor *y, KernelParams p, const char *where) {
  if (x->dtype != FLOAT32 || x->ndim < 1 || !contiguous(x)) {
    report_error(where, "input must be a contiguous fp32 tensor");
    return false;
  }
  if (y->dtype != FLOAT32 || !contiguous(y) || y->ndim != x->ndim || numel(y) != numel(x)) {
    report_error(where, "output must be a contiguous fp32 tensor shaped like the input");
    return false;
  }
  if (p.dim != x->ndim - 1) {
    report_error(where, "only the last axis (dim %llu) is supported, got dim %llu",
                 (unsigned long long)(x->ndim - 1), (unsigned long long)p.dim);
    return false;
  }
  if (x->shape[x->ndim - 1] >= (uint64_t(1) << 31)) {
    report_error(where, "rows longer than 2^31 elements are not supported");
    return false;
  }
  return true;
}

template <bool LOG>
void softmax_forward(const Tensor **inputs, Tensor *output, KernelParams params,
                     const char *where) {
  if (!ensure_init()) return;
  const Tensor *x = inputs[0];
  if (!check_softmax(x, output, params, where)) return;
  const uint32_t C = uint32_t(x->shape[x->ndim - 1]);
  const uint64_t N = C ? numel(x) / C : 0;
  const uint64_t R = max_blocks(kCeBlock);
  const float *px0 = static_cast<const float *>(x->data);
  float *py0 = static_cast<float *>(output->data);
  if (C <= kSoftmaxWaveRow && N >= kSoftmaxFewRows<LOG>) {
    for (uint64_t r0 = 0; r0 < N; r0 += R) {
      const uint64_t n = N - r0 < R ? N - r0 : R;
      with_row_lanes<kSoftmaxWaveRow>(C, [&](auto lanes, auto units) {
        constexpr int L = decltype(lanes)::value, U = decltype(units)::value;
        softmax_fwd_rows_kernel<LOG, L, U>
            <<<unsigned(ceil_div(n, kCeWaves * (64 / L))), kCeBlock, 0, stream()>>>(
                px0 + r0 * C, py0 + r0 * C, n, C);
      });
    }
    finish(where);
    return;
  }
  // float4 units per lane for a register-resident row (0: the three-pass kernel)
  int V = 0;
  const bool ragged = C % 4 != 0 || !aligned16(px0) || !aligned16(py0);
  if (!ragged || C > kSoftmaxPasses)
    for (int v = 1; v <= 32 && !V; v *= 2)
      if (uint64_t(C) <= uint64_t(kSoftmaxBlock) * 4 * v) V = v;
  // long rows of whole float4: the persistent form (rows at a time below 2^31)
  constexpr int SV = 8;
  if (!ragged && C >= PLAST_SOFTMAX_PERSISTENT && C <= uint32_t(kStepBlock) * 4 * SV &&
      N < (uint64_t(1) << 31)) {
    const unsigned G = unsigned(N < uint64_t(num_cus()) ? N : uint64_t(num_cus()));
    softmax_fwd_step_kernel<LOG, SV, PLAST_ROW_DYNAMIC><<<G, kStepBlock, 0, stream()>>>(px0, py0, uint32_t(N), C);
    finish(where);
    return;
  }
  for (uint64_t r0 = 0; r0 < N; r0 += R) {
    const unsigned n = unsigned(N - r0 < R ? N - r0 : R);
    const float *px = static_cast<const float *>(x->data) + r0 * C;
    float *py = static_cast<float *>(output->data) + r0 * C;
    const auto reg = [&](auto units) {
      constexpr int U = decltype(units)::value;
      if (ragged) softmax_fwd_reg_kernel<LOG, U, true><<<n, kSoftmaxBlock, 0, stream()>>>(px, py, C);
      else softmax_fwd_reg_kernel<LOG, U, false><<<n, kSoftmaxBlock, 0, stream()>>>(px, py, C);
    };
    switch (V) {
      case 1: reg(std::integral_constant<int, 1>{}); break;
      case 2: reg(std::integral_constant<int, 2>{}); break;
      case 4: reg(std::integral_constant<int, 4>{}); break;
      case 8: reg(std::integral_constant<int, 8>{}); break;
      case 16: reg(std::integral_constant<int, 16>{}); break;
      case 32: reg(std::integral_constant<int, 32>{}); break;
      default: softmax_fwd_kernel<LOG><<<n, kCeBlock, 0, stream()>>>(px, py, C); break;
    }
  }
  finish(where);
}

template <bool LOG>
void softmax_backward(Tensor **inputs, const Tensor *output, KernelParams params,
                      const char *where) {
  if (!ensure_init()) return;
  Tensor *x = inputs[0];
  if (!x->requires_grad || !x->grad) return;
  if (!check_softmax(x, output, params, where)) return;
  if (!output->grad || !contiguous(output->grad) || !contiguous(x->grad)) {
    report_error(where, "needs the output gradient and a contiguous input gradient");
    return;
  }
  const uint32_t C = uint32_t(x->shape[x->ndim - 1]);
  const uint64_t N = C ? numel(x) / C : 0;
  const uint64_t R = max_blocks(kCeBlock);
  constexpr int BS = PLAST_SOFTMAX_BWD_BLOCK;  // y and dy in registers: 512 lanes keep V at 16
                                              // for 32768-float rows
  int V = 0;
  const bool ragged = C % 4 != 0 || !aligned16(output->data) || !aligned16(output->grad->data) ||
                      !aligned16(x->grad->data);
  if (!ragged || !softmax_bwd_passes(N, C))
    for (int v = 1; v <= 16 && !V && v * BS <= 8192; v *= 2)
      if (uint64_t(C) <= uint64_t(BS) * 4 * v) V = v;
  for (uint64_t r0 = 0; r0 < N; r0 += R) {
    const unsigned n = unsigned(N - r0 < R ? N - r0 : R);
    const float *py = static_cast<const float *>(output->data) + r0 * C;
    const float *pg = static_cast<const float *>(output->grad->data) + r0 * C;
    float *pd = static_cast<float *>(x->grad->data) + r0 * C;
    if (softmax_bwd_waves<LOG>(N, C)) {
      with_row_lanes<kSoftmaxWaveRow>(C, [&](auto lanes, auto units) {
        constexpr int L = decltype(lanes)::value, U = decltype(units)::value;
        softmax_bwd_rows_kernel<LOG, L, U>
            <<<unsigned(ceil_div(n, kCeWaves * (64 / L))), kCeBlock, 0, stream()>>>(py, pg, pd, n, C);
      });
      continue;
    }
    const auto reg = [&](auto units) {
      constexpr int U = decltype(units)::value;
      if (ragged) softmax_bwd_reg_kernel<LOG, U, BS, true><<<n, BS, 0, stream()>>>(py, pg, pd, C);
      else softmax_bwd_reg_kernel<LOG, U, BS, false><<<n, BS, 0, stream()>>>(py, pg, pd, C);
    };
    switch (V) {
      case 1: reg(std::integral_constant<int, 1>{}); break;
      case 2: reg(std::integral_constant<int, 2>{}); break;
      case 4: reg(std::integral_constant<int, 4>{}); break;
      case 8: reg(std::integral_constant<int, 8>{}); break;
      case 16: reg(std::integral_constant<int, 16>{}); break;
      default: softmax_bwd_kernel<LOG><<<n, kCeBlock, 0, stream()>>>(py, pg, pd, C); break;
    }
  }
  finish(where);
}

}  // namespace
}  // namespace plast

using namespace plast;

extern "C" {

void softmax_cross_entropy_hip_forward(const Tensor **inputs, Tensor *output, KernelParams params) {
  (void)params;
  const char *where = "softmax_cross_entropy_hip_forward";
  if (!ensure_init()) return;
  const Tensor *x = inputs[0], *lab = inputs[1], *st = inputs[2];
  if (!check_ce(x, lab, st, where)) return;
  const uint64_t N = x->shape[0];
  const uint32_t C = uint32_t(x->shape[1]);
  if (output->dtype != FLOAT32 || numel(output) != N || !contiguous(output)) {
    report_error(where, "output must be a contiguous fp32 tensor of N elements");
    return;
  }
  if (N == 0) return;
  // The NEG node of the reference chain runs over the [N] (or [N,1]) loss tensor.
  const uint64_t se = simd_end(N);
  // rows per launch: at most one workgroup for each
  const uint64_t R = max_blocks(kCeBlock);
  for (uint64_t r0 = 0; r0 < N; r0 += R) {
    const uint64_t n = N - r0 < R ? N - r0 : R;
    const float *px = static_cast<const float *>(x->data) + r0 * C;
    const int32_t *pl = static_cast<const int32_t *>(lab->data) + r0;
    float *ps = static_cast<float *>(st->data) + 2 * r0;
    float *po = static_cast<float *>(output->data) + r0;
    const uint64_t ser = se > r0 ? se - r0 : 0;  // the rule's boundary, relative to this range
    if (C > 0 && C <= kCeWaveRow)
      with_row_lanes<kCeWaveRow>(C, [&](auto lanes, auto units) {
        constexpr int L = decltype(lanes)::value, U = decltype(units)::value;
        ce_fwd_rows_kernel<L, U><<<unsigned(ceil_div(n, kCeWaves * (64 / L))), kCeBlock, 0, stream()>>>(
            px, pl, ps, po, n, C, ser);
      });
    else
      ce_fwd_wave_kernel<<<unsigned(ceil_div(n, kCeFwdWaves)), 64 * kCeFwdWaves, 0, stream()>>>(
          px, pl, ps, po, n, C, ser);
  }
  finish(where);
}

// params.keepdim == 1 writes the gradient instead of accumulating it, for callers that own a
// gradient buffer with no other contribution (saves one HBM read of [N, C]).
void softmax_cross_entropy_hip_backward(Tensor **inputs, const Tensor *output, KernelParams params) {
  const char *where = "softmax_cross_entropy_hip_backward";
  if (!ensure_init()) return;
  Tensor *x = inputs[0];
  const Tensor *lab = inputs[1], *st = inputs[2];
  if (!x->requires_grad || !x->grad) return;
  if (!check_ce(x, lab, st, where)) return;
  if (!output->grad || !contiguous(x->grad)) {
    report_error(where, "needs the loss gradient and a contiguous logits gradient");
    return;
  }
  const uint64_t N = x->shape[0];
  const uint32_t C = uint32_t(x->shape[1]);
  if (N == 0 || C == 0) return;

  const bool vec = C % 4 == 0 && aligned16(x->data) && aligned16(x->grad->data);
  const bool over = params.keepdim == 1;
  // rows per launch, so that every grid below stays within the dispatch limit and element numbers
  // within 32 bits
  uint64_t R = (vec ? max_blocks(kCeFlatBlock) * kCeFlatBlock : (uint64_t(1) << 32) - 4) /
               (vec ? C / 4 : C);
  if (R == 0) R = 1;
  for (uint64_t r0 = 0; r0 < N; r0 += R) {
    const uint64_t n = N - r0 < R ? N - r0 : R;
    const float *px = static_cast<const float *>(x->data) + r0 * C;
    float *pd = static_cast<float *>(x->grad->data) + r0 * C;
    const int32_t *pl = static_cast<const int32_t *>(lab->data) + r0;
    const float *ps = static_cast<const float *>(st->data) + 2 * r0;
    const float *pg = static_cast<const float *>(output->grad->data) + r0;
    const uint64_t units = (n * C + 3) / 4;
    const MagicDiv dc = MagicDiv::make(vec ? C / 4 : C);
    const unsigned g = unsigned(ceil_div(units, kCeFlatBlock));
    if (vec && over)
      ce_bwd_flat_kernel<true><<<g, kCeFlatBlock, 0, stream()>>>(px, pl, ps, pg, pd, dc, uint32_t(units));
    else if (vec)
      ce_bwd_flat_kernel<false><<<g, kCeFlatBlock, 0, stream()>>>(px, pl, ps, pg, pd, dc, uint32_t(units));
    else if (over)
      ce_bwd_ragged_kernel<true><<<g, kCeFlatBlock, 0, stream()>>>(px, pl, ps, pg, pd, dc, uint32_t(n * C));
    else
      ce_bwd_ragged_kernel<false><<<g, kCeFlatBlock, 0, stream()>>>(px, pl, ps, pg, pd, dc, uint32_t(n * C));
  }
  finish(where);
}

void softmax_cross_entropy_step_hip(const float *logits, const int32_t *labels, const float *dloss,
                                    float *stats, float *loss, float *dlogits, float *dbias,
                                    float *mean_loss, u64 N, u64 C) {
  const char *where = "softmax_cross_entropy_step_hip";
  if (!ensure_init()) return;
  if (N == 0) {
    step_tail(nullptr, nullptr, 0, 0, loss, mean_loss, 0);
    if (mean_loss) finish(where);
    return;
  }
  const int V = ce_step_form(logits, labels, dloss, stats, loss, dlogits, N, C, where);
  if (V < 0) return;
  const bool whole = C % 4 == 0 && aligned16(logits) && aligned16(dlogits);
  if (V == 0) {
    // any other row: the forward, the overwriting backward and the column sum as three passes
    Tensor tx, tl, ts, to, tg, tdx;
    memset(&tx, 0, sizeof tx);
    tx.ndim = 2;
    tx.shape[0] = N, tx.shape[1] = C, tx.strides[0] = C, tx.strides[1] = 1;
    tx.data = const_cast<float *>(logits), tx.dtype = FLOAT32, tx.device = GPU;
    tx.requires_grad = true;
    tdx = tx;
    tdx.data = dlogits, tdx.requires_grad = false;
    tx.grad = &tdx;
    tl = tx;
    tl.ndim = 1, tl.shape[0] = N, tl.strides[0] = 1, tl.data = const_cast<int32_t *>(labels);
    tl.dtype = INT32, tl.requires_grad = false, tl.grad = nullptr;
    ts = tl;
    ts.shape[0] = 2 * N, ts.data = stats, ts.dtype = FLOAT32;
    to = tl;
    to.data = loss, to.dtype = FLOAT32;
    tg = to;
    tg.data = const_cast<float *>(dloss);
    to.grad = &tg;
    const Tensor *fin[3] = {&tx, &tl, &ts};
    softmax_cross_entropy_hip_forward(fin, &to, KernelParams{0, 0, 0.0f});
    Tensor *bin[3] = {&tx, &tl, &ts};
    softmax_cross_entropy_hip_backward(bin, &to, KernelParams{0, 1, 0.0f});
    if (dbias) bias_grad_reduce_hip(dlogits, dbias, N * C, C);
    if (mean_loss) {
      step_tail(nullptr, nullptr, 0, 0, loss, mean_loss, N);
      finish(where);
    }
    return;
  }
  const uint64_t grid = ce_step_grid(N, C);
  // the workgroups' column sums
  // (a capture of rows that are no whole float4 needs no workspace sized before it)
  float *part = static_cast<float *>(whole ? workspace(sizeof(float) * grid * C)
                                           : partials(sizeof(float) * grid * C, where));
  if (!part) return;
  ce_step_launch(V, unsigned(grid), part, logits, labels, dloss, stats, loss, dlogits, dbias,
                 mean_loss, N, C);
  finish(where);
}

void softmax_cross_entropy_step_noalloc_hip(const float *logits, const int32_t *labels,
                                            const float *dloss, float *stats, float *loss,
                                            float *dlogits, float *dbias, float *mean_loss, u64 N,
                                            u64 C) {
  const char *where = "softmax_cross_entropy_step_noalloc_hip";
  if (!ensure_init()) return;
  if (N == 0) {
    step_tail(nullptr, nullptr, 0, 0, loss, mean_loss, 0);
    if (mean_loss) finish(where);
    return;
  }
  const int V = ce_step_form(logits, labels, dloss, stats, loss, dlogits, N, C, where);
  if (V < 0) return;
  if (V == 0 || C % 4 != 0 || !aligned16(logits) || !aligned16(dlogits)) {
    report_error(where, "rows of %llu floats are not one-pass rows of this call, which takes whole "
                 "float4, 16-byte aligned logits and dlogits and at most %llu floats",
                 (unsigned long long)C, (unsigned long long)kStepMaxC);
    return;
  }
  float *part = fixed_scratch(where);
  if (!part) return;
  const uint64_t grid = ce_step_grid(N, C);
  ce_step_launch(V, unsigned(grid), part, logits, labels, dloss, stats, loss, dlogits, dbias,
                 mean_loss, N, C);
  finish(where);
}

void softmax_hip_forward(const Tensor **inputs, Tensor *output, KernelParams params) {
  softmax_forward<false>(inputs, output, params, "softmax_hip_forward");
}
void softmax_hip_backward(Tensor **inputs, const Tensor *output, KernelParams params) {
  softmax_backward<false>(inputs, output, params, "softmax_hip_backward");
}
void log_softmax_hip_forward(const Tensor **inputs, Tensor *output, KernelParams params) {
  softmax_forward<true>(inputs, output, params, "log_softmax_hip_forward");
}
void log_softmax_hip_backward(Tensor **inputs, const Tensor *output, KernelParams params) {
  softmax_backward<true>(inputs, output, params, "log_softmax_hip_backward");
}

}  // extern "C"
