// elementwise.hip — binary and unary ops (forward and backward), and the view ops' metadata forwards
// and GPU backwards. The fused elementwise-chain op is in fused.hip.
#include "ew_impl.hpp"
#include "red_impl.hpp"

namespace plast {
namespace {

// ------------------------------------------------------------------------- binary

template <Bin OP>
void binary_forward(const Tensor **in, Tensor *out, const char *where) {
  if (!ensure_init()) return;
  const Tensor *a = in[0], *b = in[1];
  if (!check_f32(a, where) || !check_f32(b, where) || !check_f32(out, where)) return;
  uint64_t bshape[kMaxRank];
  int brank;
  if (!broadcast_shape(a, b, bshape, &brank)) {
    report_error(where, "shapes are not broadcastable");
    return;
  }
  if (brank > int(out->ndim) || numel(out) != [&] {
        uint64_t n = 1;
        for (int d = 0; d < brank; ++d) n *= bshape[d];
        return n;
      }()) {
    report_error(where, "output shape does not match the broadcast shape");
    return;
  }
  Space s;
  init_space(s, out->shape, int(out->ndim));
  set_operand(s, 0, a);
  set_operand(s, 1, b);
  set_own(s, 2, out);
  const void *ins[2] = {a->data, b->data};
  launch_elementwise(BinBody<OP>{}, ins, out->data, s, where);
  finish(where);
}

// One past the largest element offset that shape and strides address (0 for an empty shape).
uint64_t extent(const uint64_t *shape, const uint64_t *strides, uint64_t ndim) {
  uint64_t hi = 0;
  for (uint64_t d = 0; d < ndim; ++d) {
    if (shape[d] == 0) return 0;
    hi += (shape[d] - 1) * strides[d];
  }
  return hi + 1;
}

// Gradient term of one operand, for the reduction path: g and the operands the term reads.
template <Bin OP, bool B>
struct BinTerm {
  static constexpr int NIN = 1 + int(kGradUsesA<OP, B>) + int(kGradUsesB<OP, B>);
  __device__ __forceinline__ float eval(const float *v) const {
    return bin_grad_term<OP, B>(v, false);
  }
};

// Accumulate one operand's gradient. The reference's broadcast backward addresses the gradient
// buffer with the operand's *data* strides (kernel_macros.h:314-317 passes a->strides as
// da_strides; its contiguous path indexes da flat, the same offsets for a contiguous operand). A
// view's grad keeps the layout it was allocated with (tensor.c:66-78) while the view's forward
// rewrote its data strides (shape_ops.c:59-80), so on a transposed view the two layouts differ, and
// this follows the reference. Elementwise when those offsets are distinct, otherwise a
// deterministic reduction over the axes that repeat an offset (broadcast or expanded axes; the
// reference uses `omp atomic` here: kernel_macros.h:283-299). Offsets past the gradient's own
// extent (the reference would write out of bounds) are refused.
template <Bin OP, bool B>
void grad_into(const Tensor *x, const Tensor *out, const Tensor *a, const Tensor *b,
               uint64_t simd, const char *where) {
  using Elem = BinGradBody<OP, B>;
  const Tensor *g = out->grad;
  const int rank = int(g->ndim);
  int64_t tst[kMaxRank];
  bcast_strides(x, g->shape, rank, tst);
  const uint64_t need = extent(x->shape, x->strides, x->ndim);
  const uint64_t have = extent(x->grad->shape, x->grad->strides, x->grad->ndim);
  if (need > have) {
    report_error(where, "the operand's strides address %llu gradient elements, its gradient holds "
                 "%llu", (unsigned long long)need, (unsigned long long)have);
    return;
  }
  bool repeats = false;
  for (int d = 0; d < rank; ++d) repeats = repeats || (tst[d] == 0 && g->shape[d] > 1);
  Space s;
  init_space(s, g->shape, rank);
  // the terms' operands: g and what the term reads of a and b, behind the gradient itself when the
  // target is elementwise
  const void *ins[Elem::NIN];
  int n = 0;
  if (!repeats) ins[n++] = x->grad->data;
  set_own(s, n, g);
  ins[n++] = g->data;
  if (kGradUsesA<OP, B>) {
    set_operand(s, n, a);
    ins[n++] = a->data;
  }
  if (kGradUsesB<OP, B>) {
    set_operand(s, n, b);
    ins[n++] = b->data;
  }
  for (int d = 0; d < rank; ++d) s.st[n][d] = tst[d];
  if (!repeats) {
    for (int d = 0; d < rank; ++d) s.st[0][d] = tst[d];
    Elem elem;
    elem.simd_end = simd;
    launch_elementwise(elem, ins, x->grad->data, s, where);
  } else {
    reduce_accumulate(BinTerm<OP, B>{}, ins, static_cast<float *>(x->grad->data), s, where);
  }
}

// Both gradients of a binary op over contiguous operands of one shape in one pass: g and the operands
// are read once (28 bytes an element for mul where two launches moved 32, 20 for add and 24), and a
// small op is one launch. Each element's operations are those of the two launches. One float4 unit
// a lane in XCD order, as the vector kernel streams. leaky_relu(a * b + c) and its gradients node by
// node, eight launches to six: [4096, 4096] 300 -> 275 us, [93, 24] 37 -> 29.
template <Bin OP>
__global__ __launch_bounds__(PLAST_EW_BLOCK) void bin_grad_pair_kernel(const float *g, const float *a,
                                                                       const float *b, float *da,
                                                                       float *db, uint64_t n,
                                                                       uint64_t simd_end) {
  constexpr bool kA = kGradUsesA<OP, false> || kGradUsesA<OP, true>;
  constexpr bool kB = kGradUsesB<OP, false> || kGradUsesB<OP, true>;
  const uint64_t e = (uint64_t(xcd_block(blockIdx.x, gridDim.x)) * PLAST_EW_BLOCK + threadIdx.x) * 4;
  if (e >= n) return;
  const uint32_t m = n - e < 4 ? uint32_t(n - e) : 4u;
  const f4 gv = load_part<false>(g + e, m);
  f4 av = f4(0.0f), bv = f4(0.0f);
  if constexpr (kA) av = load_part<false>(a + e, m);
  if constexpr (kB) bv = load_part<false>(b + e, m);
  f4 dav = load_part<false>(da + e, m), dbv = load_part<false>(db + e, m);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const bool simd = e + c < simd_end;
    dav[c] = dav[c] + grad_a<OP>(gv[c], av[c], bv[c]);
    dbv[c] = dbv[c] + grad_b<OP>(gv[c], av[c], bv[c], simd);
  }
  store_part<false>(dav, da + e, m);
  store_part<false>(dbv, db + e, m);
}

// Launches it where it applies: every operand, gradient and the output's gradient contiguous fp32 of
// one shape, and neither gradient's buffer shared with anything else the op touches (x * x has one
// gradient for both operands); false (launching nothing) otherwise.
template <Bin OP>
bool grad_pair(const Tensor *a, const Tensor *b, const Tensor *g, uint64_t simd) {
  const Tensor *t[5] = {a->grad, b->grad, g, a, b};
  for (const Tensor *x : t)
    if (!same_shape(x, g) || !contiguous(x)) return false;
  const uint64_t n = numel(g), blocks = ((n + 3) / 4 + PLAST_EW_BLOCK - 1) / PLAST_EW_BLOCK;
  if (n == 0 || blocks > max_blocks(PLAST_EW_BLOCK)) return false;
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 5; ++j) {
      const float *p = static_cast<const float *>(t[i]->data), *q = static_cast<const float *>(t[j]->data);
      if (i != j && p < q + n && q < p + n) return false;
    }
  bin_grad_pair_kernel<OP><<<unsigned(blocks), PLAST_EW_BLOCK, 0, stream()>>>(
      static_cast<const float *>(g->data), static_cast<const float *>(a->data),
      static_cast<const float *>(b->data), static_cast<float *>(a->grad->data),
      static_cast<float *>(b->grad->data), n, simd);
  return true;
}

template <Bin OP>
void binary_backward(Tensor **in, const Tensor *out, const char *where) {
  if (!ensure_init()) return;
  const Tensor *a = in[0], *b = in[1];
  if (!check_f32(a, where) || !check_f32(b, where)) return;
  if (!out->grad) {
    report_error(where, "output has no gradient");
    return;
  }
  const bool da = a->requires_grad && a->grad, db = b->requires_grad && b->grad;
  const uint64_t n = numel(out);
  // The reference's contiguous same-shape path (kernel_macros.h:306-311) rounds the B-gradient of
  // sub/div from 0 - g inside its SIMD blocks.
  const bool ref_contig = contiguous(a) && contiguous(b) && contiguous(out) && same_shape(a, b);
  const uint64_t simd = ref_contig ? simd_end(n) : 0;
  if (da && db && grad_pair<OP>(a, b, out->grad, simd)) {
    finish(where);
    return;
  }
  if (da) grad_into<OP, false>(a, out, a, b, 0, where);
  if (db) grad_into<OP, true>(b, out, a, b, simd, where);
  finish(where);
}

// ------------------------------------------------------------------------- unary

template <Un OP>
void unary_forward(const Tensor **in, Tensor *out, KernelParams p, const char *where) {
  if (!ensure_init()) return;
  const Tensor *a = in[0];
  if (!check_f32(a, where) || !check_f32(out, where)) return;
  if (numel(out) != numel(a)) {
    report_error(where, "output has %llu elements, input %llu", (unsigned long long)numel(out),
                 (unsigned long long)numel(a));
    return;
  }
  const uint64_t n = numel(a);
  UnBody<OP> body;
  body.alpha = p.fval;
  body.simd_end = (contiguous(a) && contiguous(out)) ? simd_end(n) : 0;
  Space s;
  init_space(s, a->shape, int(a->ndim));
  set_own(s, 0, a);
  // the reference indexes the output with its own strides over the input's shape
  for (int d = 0; d < s.rank; ++d) s.st[1][d] = a->shape[d] == 1 ? 0 : int64_t(out->strides[d]);
  const void *ins[1] = {a->data};
  launch_elementwise(body, ins, out->data, s, where);
  finish(where);
}

template <Un OP>
void unary_backward(Tensor **in, const Tensor *out, KernelParams p, const char *where) {
  if (!ensure_init()) return;
  const Tensor *a = in[0];
  if (!a->requires_grad || !a->grad) return;
  if (!check_f32(a, where)) return;
  if (!out->grad) {
    report_error(where, "output has no gradient");
    return;
  }
  UnGradBody<OP> body;
  body.alpha = p.fval;
  body.contig = contiguous(a) && contiguous(out);
  Space s;
  init_space(s, a->shape, int(a->ndim));
  set_own(s, 0, a->grad);
  for (int d = 0; d < s.rank; ++d)
    s.st[1][d] = a->shape[d] == 1 ? 0 : int64_t(out->grad->strides[d]);
  set_own(s, 2, a);
  set_own(s, 3, a->grad);
  const void *ins[3] = {a->grad->data, out->grad->data, a->data};
  launch_elementwise(body, ins, a->grad->data, s, where);
  finish(where);
}

// ------------------------------------------------------------------------- view ops

// Backward of a view that kept numel: da[i] += dout[i] over contiguous buffers
// (shape_ops.c:14-26).
void reshape_accumulate(float *da, const float *dout, uint64_t n, const char *where) {
  Space s;
  s.rank = 1;
  s.shape[0] = n;
  s.st[0][0] = s.st[1][0] = s.st[2][0] = 1;
  const void *ins[2] = {da, dout};
  launch_elementwise(AccumBody{}, ins, da, s, where);
}

void alias_meta(const Tensor *a, Tensor *out) {
  out->data = a->data;
  out->dtype = a->dtype;
  out->device = a->device;
  out->requires_grad = a->requires_grad;
}

// Row-major strides of the caller-provided output shape (cpu_utils.c:19-26).
void row_major(Tensor *out) {
  uint64_t s = 1;
  for (uint64_t d = out->ndim; d-- > 0;) {
    out->strides[d] = s;
    s *= out->shape[d];
  }
}

void view_like_forward(const Tensor **in, Tensor *out) {
  alias_meta(in[0], out);
  row_major(out);
}

void view_like_backward(Tensor **in, const Tensor *out, const char *where) {
  if (!ensure_init()) return;
  Tensor *a = in[0];
  if (!a->requires_grad || !out->grad || !a->grad) return;
  reshape_accumulate(static_cast<float *>(a->grad->data),
                     static_cast<const float *>(out->grad->data), numel(a), where);
  finish(where);
}

// expand / broadcast forward (shape_ops.c:54-57 with cpu_utils.c:59-119): stride 0 on new and on
// expanded size-1 axes. The output shares the input's grad, so their backward is a no-op
// (kernel_macros.h:141-153).
void expand_like_forward(const Tensor **in, Tensor *out) {
  const Tensor *a = in[0];
  alias_meta(a, out);
  out->grad = a->grad;
  const uint64_t lead = out->ndim - a->ndim;
  for (uint64_t d = 0; d < out->ndim; ++d) {
    if (d < lead) {
      out->strides[d] = 0;
    } else {
      const uint64_t s = d - lead;
      out->strides[d] = (a->shape[s] == 1 && out->shape[d] > 1) ? 0 : a->strides[s];
    }
  }
}

}  // namespace
}  // namespace plast

using namespace plast;

extern "C" {

#define BINARY_ENTRY(name, OPV)                                                                    \
  void name##_hip_forward(const Tensor **inputs, Tensor *output, KernelParams params) {            \
    (void)params;                                                                                  \
    binary_forward<OPV>(inputs, output, #name "_hip_forward");                                     \
  }                                                                                                \
  void name##_hip_backward(Tensor **inputs, const Tensor *output, KernelParams params) {           \
    (void)params;                                                                                  \
    binary_backward<OPV>(inputs, output, #name "_hip_backward");                                   \
  }
BINARY_ENTRY(add, Bin::Add)
BINARY_ENTRY(sub, Bin::Sub)
BINARY_ENTRY(mul, Bin::Mul)
BINARY_ENTRY(div, Bin::Div)
#undef BINARY_ENTRY

#define UNARY_ENTRY(name, OPV)                                                                     \
  void name##_hip_forward(const Tensor **inputs, Tensor *output, KernelParams params) {            \
    unary_forward<OPV>(inputs, output, params, #name "_hip_forward");                              \
  }                                                                                                \
  void name##_hip_backward(Tensor **inputs, const Tensor *output, KernelParams params) {           \
    unary_backward<OPV>(inputs, output, params, #name "_hip_backward");                            \
  }
UNARY_ENTRY(exp, Un::Exp)
UNARY_ENTRY(log, Un::Log)
UNARY_ENTRY(neg, Un::Neg)
UNARY_ENTRY(abs, Un::Abs)
UNARY_ENTRY(sin, Un::Sin)
UNARY_ENTRY(cos, Un::Cos)
UNARY_ENTRY(tan, Un::Tan)
UNARY_ENTRY(leaky_relu, Un::Leaky)
#undef UNARY_ENTRY

#define VIEW_ENTRY(name)                                                                           \
  void name##_hip_forward(const Tensor **inputs, Tensor *output, KernelParams params) {            \
    (void)params;                                                                                  \
    view_like_forward(inputs, output);                                                             \
  }                                                                                                \
  void name##_hip_backward(Tensor **inputs, const Tensor *output, KernelParams params) {           \
    (void)params;                                                                                  \
    view_like_backward(inputs, output, #name "_hip_backward");                                     \
  }
VIEW_ENTRY(view)
VIEW_ENTRY(flatten)
VIEW_ENTRY(squeeze)
VIEW_ENTRY(unsqueeze)
#undef VIEW_ENTRY

void expand_hip_forward(const Tensor **inputs, Tensor *output, KernelParams params) {
  (void)params;
  expand_like_forward(inputs, output);
}
void expand_hip_backward(Tensor **inputs, const Tensor *output, KernelParams params) {
  (void)inputs;
  (void)output;
  (void)params;
}
void broadcast_hip_forward(const Tensor **inputs, Tensor *output, KernelParams params) {
  (void)params;
  expand_like_forward(inputs, output);
}
void broadcast_hip_backward(Tensor **inputs, const Tensor *output, KernelParams params) {
  (void)inputs;
  (void)output;
  (void)params;
}

// shape_ops.c:59-80
void transpose_hip_forward(const Tensor **inputs, Tensor *output, KernelParams params) {
  const Tensor *a = inputs[0];
  const uint64_t x = params.dim, y = params.keepdim;
  if (x >= a->ndim || y >= a->ndim) {
    report_error("transpose_hip_forward", "axes (%llu, %llu) out of range for rank %llu",
                 (unsigned long long)x, (unsigned long long)y, (unsigned long long)a->ndim);
    return;
  }
  alias_meta(a, output);
  output->ndim = a->ndim;
  for (uint64_t d = 0; d < a->ndim; ++d) {
    output->shape[d] = a->shape[d];
    output->strides[d] = a->strides[d];
  }
  std::swap(output->shape[x], output->shape[y]);
  std::swap(output->strides[x], output->strides[y]);
}

// shape_ops.c:82-120: da[c] += dout[c with axes swapped].
void transpose_hip_backward(Tensor **inputs, const Tensor *output, KernelParams params) {
  Tensor *a = inputs[0];
  if (!a->requires_grad || !output->grad || !a->grad) return;
  transpose_backward_hip(static_cast<float *>(a->grad->data),
                         static_cast<const float *>(output->grad->data), a->shape,
                         a->grad->strides, output->grad->strides, a->ndim, params.dim,
                         params.keepdim, numel(a));
}

void reshape_backward_hip(float *da, const float *dout, u64 num_elements) {
  if (!ensure_init()) return;
  reshape_accumulate(da, dout, num_elements, "reshape_backward_hip");
  finish("reshape_backward_hip");
}

void transpose_backward_hip(float *da, const float *dout, const u64 *a_shape, const u64 *da_strides,
                            const u64 *dout_strides, u64 ndim, u64 axis1, u64 axis2,
                            u64 num_elements) {
  if (!ensure_init()) return;
  if (ndim > uint64_t(kMaxRank) || axis1 >= ndim || axis2 >= ndim) {
    report_error("transpose_backward_hip", "bad rank/axes");
    return;
  }
  (void)num_elements;
  Space s;
  s.rank = int(ndim);
  for (uint64_t d = 0; d < ndim; ++d) s.shape[d] = a_shape[d];
  for (uint64_t d = 0; d < ndim; ++d) {
    s.st[0][d] = a_shape[d] == 1 ? 0 : int64_t(da_strides[d]);
    // coordinate d of `a` is coordinate swap(d) of the transposed gradient
    const uint64_t td = d == axis1 ? axis2 : (d == axis2 ? axis1 : d);
    s.st[1][d] = a_shape[d] == 1 ? 0 : int64_t(dout_strides[td]);
    s.st[2][d] = s.st[0][d];
  }
  const void *ins[2] = {da, dout};
  launch_elementwise(AccumBody{}, ins, da, s, "transpose_backward_hip");
  finish("transpose_backward_hip");
}

}  // extern "C"
