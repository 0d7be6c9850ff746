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

// ------------------------------------------------------------------------- elementwise launches

// Whether a space of n elements with a transposed operand goes to the 64x64 tiles rather than to one
// element a lane. `staged`: operands read through LDS. One, whole tiles: always. Several: a workgroup
// stages them one after the other, 5.6 us however small the space (d += g * b, both transposed:
// [128, 128] 5.6 us in tiles, 3.6 so, [512, 512] 5.8 and 4.9, [512, 1024] 5.9 and 6.9). Partial tiles:
// config 3's chain [8, 301, 150] 5.82 and 4.12, [8, 301, 301] 5.95 and 6.58, [64, 513, 301] 22 and
// 56; of whole float4 units with nothing read past LDS (`quads`), over extents that fill a tile: exp
// of [600, 600] 4.5 and 4.6, of [700, 700] 4.6 and 5.0, but of [100000, 4] 5.6 and 3.1.
inline bool tile_pays(uint64_t n, bool tape, uint32_t staged, bool full, bool quads, uint64_t least_extent) {
  if (staged > 1 && !tape) return n >= uint64_t(1) << 19;
  return full || n >= (quads && !tape && least_extent >= 64 ? uint64_t(3) << 17 : uint64_t(1) << 19);
}

// Whether a contiguous output whose rows are no whole float4 goes to the flat kernel rather than to one
// element a lane, `outer` axes decoded outside the innermost one. Fixed bodies, a row added:
// [30000, 77] 3.5 us flat and 3.4, [400000 / 77, 77] 3.7 and 3.8, [1.2M / 77, 77] 4.4 and 5.1; three
// outer axes: 0.3M elements 4.6 and 3.7, 1.2M 6.0 and 5.8, 4.9M 13.9 and 15.4. Fused chains beyond the
// smallest (which never come here) gain from it at once, with three outer axes from 1.3M elements:
// 0.4M 6.9 and 4.9, 1.1M 8.5 and 7.9, 1.5M 8.8 and 9.5.
inline bool flat_elementwise_pays(uint64_t n, bool tape, int outer) {
  if (tape) return outer < 3 || n >= uint64_t(5) << 18;
  return n >= (outer < 3 ? uint64_t(3) << 17 : uint64_t(3) << 20);
}

// ------------------------------------------------------------------------- leading-axis reductions
// A reduction of [rows, len, inner] over len, the `inner` columns kept.

inline uint64_t div_up(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// Row chunks of the column kernel with lanes of `width` columns: slices of 64 lanes, and the reduced
// axis in chunks of at least `min_rows` rows until the grid has about `blocks` workgroups.
struct ColChunks {
  uint64_t slices;  // of one row's columns
  uint64_t chunks, seglen;
};
inline ColChunks col_chunks(uint64_t rows, uint64_t len, uint64_t inner, uint64_t width,
                            uint64_t min_rows, uint64_t blocks) {
  ColChunks c;
  c.slices = div_up(inner, 64 * width);
  const uint64_t base = c.slices * rows;
  c.chunks = 1;
  if (base < blocks && len >= 2 * min_rows) {
    c.chunks = div_up(blocks, base);
    if (c.chunks > len / min_rows) c.chunks = len / min_rows;
    if (c.chunks > 65535) c.chunks = 65535;
  }
  c.seglen = div_up(len, c.chunks);
  c.chunks = div_up(len, c.seglen);
  return c;
}

// Narrow columns read as one flat array: T of kFlatBlock lanes take consecutive float4 units, 4 T
// floats being R whole rows (a step). Chunks of whole steps: one up to eight of them, else eight
// steps each up to about `blocks` workgroups, down to two where that leaves the chip idle (sum and
// max of [60000, 10]: 16.0 us with chunks of eight, 13.4 of two; the bias gradient of [16384, 250]:
// 28.3 and 30.6).
constexpr uint32_t kFlatBlock = 512, kFlatInner = 256;  // inner is below kFlatInner
struct FlatCols {
  uint32_t T, R;
  uint64_t chunks, seglen;
};
inline FlatCols flat_cols(uint64_t rows, uint64_t len, uint64_t inner, uint64_t blocks) {
  const uint32_t in = uint32_t(inner);
  const uint32_t units = in % 4 == 0 ? in / 4 : in % 2 == 0 ? in / 2 : in;  // of the shortest whole rows
  FlatCols f;
  f.T = kFlatBlock / units * units;
  f.R = uint32_t(uint64_t(4) * f.T / in);
  const uint64_t steps = div_up(len, f.R);
  const uint64_t most = div_up(blocks, rows), least = div_up(256, rows);
  uint64_t c = steps / 8;
  if (c > most) c = most;
  if (c < least) c = steps / 2 < least ? steps / 2 : least;
  if (c > 65535) c = 65535;
  if (steps <= 8 || c < 1) c = 1;
  f.seglen = div_up(steps, c) * f.R;
  f.chunks = div_up(len, f.seglen);
  return f;
}

// Whether the flat array beats the column kernel at one column a lane (`w`: its chunks). A flat
// workgroup is 512 lanes and pays its merge through LDS however little it reads (an argmax, whose
// partials are 16 bytes of value and index, twice that), so over many outer rows of a short axis
// the column kernel's small workgroups win: sum of [20000, 8, 10] over the 8 16 us against 64,
// argmax 20 and 200, sum of [1024, 100, 10] 5.4 and 6.7. The flat array wins where it needs one
// launch and the chunks two (sum of [256, 512, 10] 4.4 us, 8.3 in chunks), where each column
// workgroup would walk more than some 64 rows (max of [256, 2048, 8] 7.9 and 27.7, of [16, 6000, 10]
// 8.4 and 9.5), where the partials of many chunks are left to merge (sum of [60000, 10] 7.1 and
// 8.9), over a few rows of nearly the chunks' 128 (max of [100, 10] 4.8 and 5.3), where its workgroups
// have thousands of elements each of a large input (max of [1000, 100, 100] 9.2 and 13.3), and, at widths of which a wave's slice leaves a part idle, on large inputs (sum of [16384, 250]
// 8.4 and 9.6; of [8192, 250] 7.5 and 7.2).
inline bool flat_pays(const ColChunks &w, const FlatCols &f, uint64_t rows, uint64_t len, uint64_t inner,
                      bool argmax) {
  const uint64_t steps = div_up(len, f.R);
  if (w.chunks == 1)
    return len >= 256 || (len >= 96 && len * inner >= 8192 && rows * len * inner >= uint64_t(11) << 19) ||
           (!argmax && ((len >= 128 && rows <= 1024) ||
                        (len >= 96 && rows <= 256 && inner >= 8 && inner < 128)));
  if (f.chunks == 1 && steps <= (!argmax ? 8 : inner < 64 ? 4 : 7)) return true;
  if (inner < 128) return w.seglen >= 80 || w.chunks > 320;
  return w.seglen >= 128 || (inner > 192 && !argmax && rows * len * inner >= uint64_t(7) << 19);
}

// Columns a lane of the column kernel owns where rows allow float4 units: 4 only where the launch is
// bound by its loads or by its workgroup count. Below some 5.8 million elements it is bound by
// the rows each wave walks one after the other, and one column a lane makes four times the
// waves (max of [2048, 1001] 7.9 us, 11 with four, of [8192, 1001] 14.4 and 13.1; sum of [4096, 513]
// 7.3 and 10.1). Rows of at most 64 columns would leave most of a wave idle with four. Sums of many
// short columns are bound by the workgroups (sum of [4096, 8, 250] 14.1 us, 7.9 with four; argmax,
// which does more per column, is not: [20000, 16, 77] 44 and 66).
inline uint32_t col_width(uint64_t rows, uint64_t len, uint64_t inner, bool argmax) {
  if (inner <= 64 || (argmax && inner < kFlatInner)) return 1;
  if (!argmax && rows * div_up(inner, 64) >= 4096) return 4;
  return rows * len * inner >= uint64_t(11) << 19 ? 4 : 1;
}

// Whether a sum of whole float4 columns (partial at a row's end) goes to the one-launch slices, each
// lane walking its share of the rows: from a few rows on, below 128 only where the slices are few
// (they read 16 or 32 bytes a row: sum of [256, 100, 77] 6.9 us, 5.2 in columns), up to what one
// workgroup walks in the time of the second launch it saves. Producers of one operand: sum of
// [6000, 64] 6.0 us, in chunks 7.3, of [12000, 64] 8.6 and 7.4. Of two and three: the gradient of a
// multiplied [4000, 64] 7.2 and 8.0, of [6000, 64] 9.0 and 7.8, of [4096, 301] 13.7 and 8.2. Storing
// ones, whose stores off a 16-byte boundary cost more: the one-pass epilogue at [2048, 64] 6.5 and
// 7.9, at [1500, 301] 7.1 and 8.2, at [2048, 30] 8.2 and 7.6; config 1's step at [2048, 256] 8.3
// and 9.4, at [2048, 64] 10.3 and 8.6, at [2048, 8] 6.3 and 7.5.
inline bool col_slices(uint64_t rows, uint64_t len, uint64_t inner, int nin, bool stores) {
  const uint64_t n = rows * len * inner;
  if (len < (stores ? 24 : 48) || (len < 128 && rows * div_up(inner, 64) >= 128)) return false;
  if (!stores) return len <= (nin == 1 ? 6144 : n <= (uint64_t(1) << 19) ? 4096 : 2048);
  if (n <= (uint64_t(1) << 15)) return len <= 2048;
  return len <= (inner % 4 == 0 && (nin == 2 || inner >= 256) ? 2048 : 1536);
}

}  // namespace plast
