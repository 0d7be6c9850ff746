// launch_rules.hpp — dispatch rules that are arithmetic on sizes alone: host code without HIP, so
// that the CPU tests evaluate them over whole ranges of sizes.
#pragma once

#include <cstdint>

namespace plast {

// The dispatch packet's grid size is 32-bit: a launch holds fewer than 2^32 work-items per
// dimension, i.e. at most max_blocks(threads) workgroups of `threads` lanes along x.
constexpr uint64_t max_blocks(uint64_t threads) { return (uint64_t(1) << 32) / threads - 1; }

// Threads that share a row of the one-read max/min backward, about four float4 units each; 0 where the
// two passes run: a few rows too long for one workgroup each, and more rows than one launch holds.
inline uint32_t ext_row_threads(uint64_t rows, uint64_t len) {
  constexpr uint64_t kRowsBlock = 256, kLongBlock = 512;  // lanes per workgroup
  if (len > 32768 && rows < 256) return 0;
  const uint32_t t = len <= 128 ? 8 : len <= 2048 ? 64 : uint32_t(kLongBlock);
  const uint64_t per_block = t > 64 ? 1 : kRowsBlock / t;  // rows of a workgroup
  const uint64_t blocks = (rows + per_block - 1) / per_block;
  return blocks <= max_blocks(t > 64 ? kLongBlock : kRowsBlock) ? t : 0;
}

}  // namespace plast
