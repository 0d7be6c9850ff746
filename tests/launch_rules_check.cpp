// Evaluates the launches' size rules (plast_amd/csrc/launch_rules.hpp): prints "ok" or the first rule
// broken, and exits non-zero on failure.
#include <cstdint>
#include <cstdio>
#include <initializer_list>

#include "launch_rules.hpp"

static int g_fail = 0;

#define CHECK(cond, ...)                                          \
  do {                                                            \
    if (!(cond)) {                                                \
      std::printf("line %d: %s: ", __LINE__, #cond);              \
      std::printf(__VA_ARGS__);                                   \
      std::printf("\n");                                          \
      g_fail = 1;                                                 \
    }                                                             \
  } while (0)

using u64 = uint64_t;
static const u64 k32 = u64(1) << 32;

// Max/min backward in one read: every launch it takes has fewer than 2^32 work-items, and what it
// leaves to the two passes is the few long rows and the launches past that bound.
static void ext_rows() {
  const u64 lens[] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 127, 128, 129, 2047, 2048, 2049, 32768, 32769, 1 << 20};
  for (u64 len : lens) {
    for (int e = 0; e <= 32; ++e)
      for (int d = -2; d <= 2; ++d) {
        const u64 rows = (u64(1) << e) + u64(int64_t(d));
        if (rows == 0 || rows > k32 || rows * len >= k32) continue;
        const u64 t = plast::ext_row_threads(rows, len);
        const u64 want = len <= 128 ? 8 : len <= 2048 ? 64 : 512;
        const u64 per = want == 512 ? 1 : 256 / want, lanes = want == 512 ? 512 : 256;
        const bool fits = (rows + per - 1) / per * lanes < k32;
        const bool few = len > 32768 && rows < 256;
        CHECK(t == 0 || t == want, "rows %llu len %llu", (unsigned long long)rows, (unsigned long long)len);
        CHECK(t == 0 || (fits && !few), "rows %llu len %llu", (unsigned long long)rows, (unsigned long long)len);
        if (!few && rows < (u64(1) << 28))
          CHECK(t != 0, "rows %llu len %llu", (unsigned long long)rows, (unsigned long long)len);
      }
  }
  CHECK(plast::ext_row_threads((u64(1) << 29) - 64, 7) == 8, "below the bound");
  CHECK(plast::ext_row_threads(u64(1) << 29, 4) == 0, "2^29 rows of 8 threads");
}

// Leading-axis reductions: every plan covers its rows, the flat array's merge fits its lanes, and it is
// never taken where each workgroup would read little of a short axis.
static void columns() {
  const u64 blocks = 1024;
  for (u64 inner = 1; inner < plast::kFlatInner; ++inner) {
    const plast::FlatCols one = plast::flat_cols(1, 100, inner, blocks);
    CHECK(one.T >= 1 && one.T <= plast::kFlatBlock && u64(4) * one.T == u64(one.R) * inner, "inner %llu", (unsigned long long)inner);
    // a merge round writes ceil(rows / 8) rows of `inner` sums, one a lane, from the first round's R rows
    CHECK((one.R + 7) / 8 * inner <= plast::kFlatBlock, "inner %llu", (unsigned long long)inner);
  }
  const u64 outers[] = {1, 2, 3, 16, 64, 255, 256, 257, 1000, 1024, 1025, 4096, 20000, 100000, 1 << 24};
  const u64 lens[] = {2, 3, 8, 32, 64, 95, 96, 100, 127, 128, 129, 200, 256, 512, 1000, 4096, 60000, 1 << 20, (1 << 26) + 1};
  const u64 inners[] = {1, 2, 3, 8, 10, 63, 64, 65, 77, 127, 128, 129, 192, 193, 250, 255, 256, 257, 1001, 65536};
  for (u64 rows : outers)
    for (u64 len : lens)
      for (u64 inner : inners) {
        if (rows * len * inner >= k32) continue;
        for (u64 width : {u64(1), u64(4)}) {
          const plast::ColChunks c = plast::col_chunks(rows, len, inner, width, 64, blocks);
          CHECK(c.chunks >= 1 && c.chunks <= 65535 && c.chunks * c.seglen >= len && (c.chunks - 1) * c.seglen < len &&
                    c.slices * 64 * width >= inner, "rows %llu len %llu inner %llu", (unsigned long long)rows,
                (unsigned long long)len, (unsigned long long)inner);
          CHECK(c.chunks == 1 || (c.slices * rows < blocks && c.seglen >= 64), "chunks of at least 64 rows");
        }
        const u64 w1 = (inner + 63) / 64 * rows;
        for (int arg = 0; arg < 2; ++arg) {
          const u64 w = plast::col_width(rows, len, inner, arg);
          CHECK(w == 1 || (w == 4 && inner > 64), "width");
          CHECK(w == 1 || rows * len * inner >= u64(5500000) || (!arg && w1 >= 4096), "rows %llu len %llu inner %llu",
                (unsigned long long)rows, (unsigned long long)len, (unsigned long long)inner);
        }
        CHECK(!plast::col_slices(rows, len, inner, 1, false) || (len <= 6144 && (len >= 128 || w1 < 128)), "slices");
        if (inner >= plast::kFlatInner) continue;
        const plast::FlatCols f = plast::flat_cols(rows, len, inner, blocks);
        CHECK(f.chunks >= 1 && f.chunks <= 65535 && f.chunks * f.seglen >= len && (f.chunks - 1) * f.seglen < len &&
                  f.seglen % f.R == 0, "rows %llu len %llu inner %llu", (unsigned long long)rows,
              (unsigned long long)len, (unsigned long long)inner);
        for (int arg = 0; arg < 2; ++arg) {
          const bool pays = plast::flat_pays(plast::col_chunks(rows, len, inner, 1, 64, blocks), f, rows, len, inner, arg);
          CHECK(!pays || len >= 96, "short axes keep the small workgroups");
          CHECK(!pays || rows <= 1024 || len >= 256 || len * inner >= 8192, "rows %llu len %llu inner %llu", (unsigned long long)rows,
                (unsigned long long)len, (unsigned long long)inner);
        }
      }
}

// Elementwise launches: a small space never pays for a workgroup's staging, a large one always leaves
// the one-element-a-lane kernel, and each rule keeps its side once a space has grown past it.
static void elementwise() {
  for (int tape = 0; tape < 2; ++tape) {
    for (int outer = 0; outer < 6; ++outer) {
      bool was = false;
      for (u64 n = 1; n < k32; n = n * 5 / 4 + 1) {
        const bool pays = plast::flat_elementwise_pays(n, tape, outer);
        CHECK(pays || !was, "n %llu", (unsigned long long)n);
        CHECK(tape || !pays || n > 300000, "n %llu", (unsigned long long)n);
        CHECK(pays || n < 4000000, "n %llu", (unsigned long long)n);
        was = pays;
      }
    }
    for (uint32_t staged = 1; staged < 4; ++staged)
      for (int form = 0; form < 4; ++form)
        for (u64 n = 1; n < k32; n = n * 5 / 4 + 1) {
          const bool pays = plast::tile_pays(n, tape, staged, form & 1, form & 2, n < 64 ? n : 64);
          CHECK(pays || n < 600000, "n %llu", (unsigned long long)n);
          CHECK(!pays || n > 390000 || ((form & 1) && (staged == 1 || tape)), "n %llu", (unsigned long long)n);
        }
  }
}

int main() {
  ext_rows();
  elementwise();
  columns();
  if (!g_fail) std::printf("ok\n");
  return g_fail;
}
