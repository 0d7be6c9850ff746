// fused_wide.hip — the tape interpreter of the op sets with log, and with every op.
#include "tape_launch.hpp"

namespace plast {

template void launch_tape<kTapeExp | kTapeLog>(const PlastFusedTape &, uint64_t, uint32_t, int,
                                               const void *const *, void *, const Space &,
                                               const char *);
template void launch_tape<kTapeExp | kTapeLog | kTapeTrig>(const PlastFusedTape &, uint64_t, uint32_t, int,
                                               const void *const *, void *, const Space &,
                                               const char *);

}  // namespace plast
