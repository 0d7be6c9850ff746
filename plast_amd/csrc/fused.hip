// fused.hip — the fused elementwise-chain op (forward), and the interpreter of its arithmetic and exp
// op sets; fused_wide.hip holds the wider sets, epilogue.hip the one chain that carries a gradient
// (beside the bias-gradient kernels it shares).
#include "tape_launch.hpp"

namespace plast {

template void launch_tape<kTapeArith>(const PlastFusedTape &, uint64_t, uint32_t, int,
                                      const void *const *, void *, const Space &, const char *);
template void launch_tape<kTapeExp>(const PlastFusedTape &, uint64_t, uint32_t, int,
                                      const void *const *, void *, const Space &, const char *);

namespace {

// Does tensor t cover every element of `shape` exactly once (no broadcast axis)?
bool covers(const Tensor *t, const uint64_t *shape, int rank) {
  if (int(t->ndim) > rank) return false;
  int lead = rank - int(t->ndim);
  for (int d = 0; d < rank; ++d) {
    uint64_t e = d < lead ? 1 : t->shape[d - lead];
    if (e != shape[d]) return false;
  }
  return true;
}

}  // namespace
}  // namespace plast

using namespace plast;

extern "C" {

void fused_elementwise_hip_forward(const Tensor **inputs, Tensor *output, KernelParams params) {
  const char *where = "fused_elementwise_hip_forward";
  if (!ensure_init()) return;
  const PlastFusedTape *tape = reinterpret_cast<const PlastFusedTape *>(uintptr_t(params.dim));
  if (!tape || tape->num_inputs == 0 || tape->num_inputs > PLAST_TAPE_MAX_INPUTS ||
      tape->num_ins == 0 || tape->num_ins > PLAST_TAPE_MAX_INS || tape->ins[0].op != TAPE_LOAD) {
    report_error(where, "malformed tape");
    return;
  }
  for (uint32_t i = 0; i < tape->num_ins; ++i) {
    const PlastTapeIns &t = tape->ins[i];
    if (t.op >= TAPE_NUM_OPS || ((t.src == TAPE_SRC_INPUT || t.op == TAPE_LOAD) &&
                                 t.idx >= tape->num_inputs)) {
      report_error(where, "tape instruction %u is invalid", i);
      return;
    }
  }
  if (!check_f32(output, where)) return;
  for (uint32_t k = 0; k < tape->num_inputs; ++k)
    if (!check_f32(inputs[k], where)) return;
  const uint64_t n = numel(output);
  Space s;
  init_space(s, output->shape, int(output->ndim));
  const void *ins[PLAST_TAPE_MAX_INPUTS];
  for (uint32_t k = 0; k < tape->num_inputs; ++k) {
    if (!covers(inputs[k], output->shape, int(output->ndim))) {
      // broadcast inputs are fine; shapes that do not broadcast are not
      uint64_t bs[kMaxRank];
      int br;
      if (!broadcast_shape(inputs[k], output, bs, &br) || br != int(output->ndim)) {
        report_error(where, "input %u does not broadcast to the output", k);
        return;
      }
    }
    set_operand(s, int(k), inputs[k]);
    ins[k] = inputs[k]->data;
  }
  const int nin = int(tape->num_inputs);
  set_own(s, nin, output);
  // The reference's neg takes its 8-wide SIMD path (0 - x below simd_end) only when its input and
  // its output are both contiguous (DEFINE_UNARY_CPU_FORWARD, kernel_macros.h:19-31), and -x
  // otherwise. Every intermediate of the unfused chain is a fresh contiguous tensor, so only a NEG
  // reading the loaded input directly or writing the chain's output can meet a strided tensor.
  uint32_t neg_simd = 0;
  for (uint32_t i = 1; i < tape->num_ins; ++i) {
    if (tape->ins[i].op != TAPE_NEG) continue;
    const bool in_ok = i > 1 || contiguous(inputs[tape->ins[0].idx]);
    const bool out_ok = i + 1 < tape->num_ins || contiguous(output);
    if (in_ok && out_ok) neg_simd |= 1u << i;
  }
  const uint64_t se = simd_end(n);
  switch (tape_ops_class(*tape)) {
  case kTapeArith: launch_tape<kTapeArith>(*tape, se, neg_simd, nin, ins, output->data, s, where); break;
  case kTapeExp: launch_tape<kTapeExp>(*tape, se, neg_simd, nin, ins, output->data, s, where); break;
  case kTapeExp | kTapeLog:
    launch_tape<kTapeExp | kTapeLog>(*tape, se, neg_simd, nin, ins, output->data, s, where);
    break;
  default:
    launch_tape<kTapeExp | kTapeLog | kTapeTrig>(*tape, se, neg_simd, nin, ins, output->data, s, where);
    break;
  }
  finish(where);
}

}  // extern "C"
