// Evaluates the launches' size rules (plast_amd/csrc/launch_rules.hpp): prints "ok" or the first rule
// broken, and exits non-zero on failure.
#include <cstdint>
#include <cstdio>

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

int main() {
  ext_rows();
  if (!g_fail) std::printf("ok\n");
  return g_fail;
}
