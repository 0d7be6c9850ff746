// tape_launch.hpp — a fused chain on the interpreter instantiated for one op set; each set is
// instantiated in one translation unit (fused.hip, fused_wide.hip), which build in parallel.
#pragma once

#include "ew_impl.hpp"

namespace plast {

// Launches tape t on the interpreter of op set OPS and nin inputs.
template <uint32_t OPS>
void launch_tape(const PlastFusedTape &t, uint64_t se, uint32_t neg_simd, int nin,
                 const void *const *ins, void *out, const Space &s, const char *where) {
  switch (nin) {
  case 1: launch_elementwise(TapeBody<1, OPS>{t, se, neg_simd}, ins, out, s, where); break;
  case 2: launch_elementwise(TapeBody<2, OPS>{t, se, neg_simd}, ins, out, s, where); break;
  case 3: launch_elementwise(TapeBody<3, OPS>{t, se, neg_simd}, ins, out, s, where); break;
  default: launch_elementwise(TapeBody<4, OPS>{t, se, neg_simd}, ins, out, s, where); break;
  }
}

extern template void launch_tape<kTapeArith>(const PlastFusedTape &, uint64_t, uint32_t, int,
                                             const void *const *, void *, const Space &, const char *);
extern template void launch_tape<kTapeExp>(const PlastFusedTape &, uint64_t, uint32_t, int,
                                           const void *const *, void *, const Space &, const char *);
extern template void launch_tape<kTapeExp | kTapeLog>(const PlastFusedTape &, uint64_t, uint32_t, int,
                                                      const void *const *, void *, const Space &,
                                                      const char *);
extern template void launch_tape<kTapeExp | kTapeLog | kTapeTrig>(const PlastFusedTape &, uint64_t,
                                                                  uint32_t, int, const void *const *,
                                                                  void *, const Space &, const char *);

}  // namespace plast
