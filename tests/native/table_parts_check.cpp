// Host-side check of split_tables (caps_amd/csrc/engine.h): for plans of every
// kind of step and windows from the smallest on, each step's table lies in its
// part, whole and unchanged, behind the part's copy of the split constants, and
// the parts cover all steps in order.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <set>

#include "../../caps_amd/csrc/engine.h"

using namespace caps;

static int fails = 0;
#define CHECK(c, ...)                    \
  do {                                   \
    if (!(c)) {                          \
      printf("FAIL %s: ", #c);           \
      printf(__VA_ARGS__);               \
      printf("\n");                      \
      if (++fails > 20) return;          \
    }                                    \
  } while (0)

static size_t up64(size_t x) { return (x + 63) / 64 * 64; }
static std::set<int> kinds;

static void check(int n, int r, int bs, const char *pat, int mode, int moduli, bool fuse,
                  int cutoff) {
  const caps_desc d{n, r, 1, 1, 1, 1, bs};
  const auto build = [&](Plan &p) {
    return build_plan(p, (double *)0x1000, (double *)0x2000, (double *)0x3000, d, pat, mode, moduli,
                      cutoff, (void *)0x100000, fuse);
  };
  Plan whole;
  CHECK(build(whole) == CAPS_OK, "n=%d %s", n, pat);
  // the sizes: a step's table ends where the next one (or the constants) starts,
  // but for alignment
  std::set<size_t> starts{whole.host_tables.size()};
  if (whole.oz_moduli) starts.insert(whole.oz_const);
  for (const Step &st : whole.steps) starts.insert(st.table);
  size_t largest = 0;
  for (const Step &st : whole.steps) {
    const size_t bytes = step_table_bytes(st), next = *starts.upper_bound(st.table);
    CHECK(bytes > 0 && st.table + bytes <= next && up64(st.table + bytes) >= next,
          "n=%d %s kind %d: %zu bytes at %zu, next %zu", n, pat, st.kind, bytes, st.table, next);
    largest = std::max(largest, bytes);
    kinds.insert(st.kind);
  }
  const size_t consts = whole.oz_moduli ? sizeof(OzakiConsts) : 0;
  const size_t least = up64(consts) + largest;
  Plan none;
  build(none);
  CHECK(!split_tables(none, least - 1), "n=%d %s: window %zu", n, pat, least - 1);
  for (size_t window : {least, least + 64, least + 4096, whole.host_tables.size() + 65536}) {
    Plan p;
    build(p);
    CHECK(split_tables(p, window), "n=%d %s: window %zu", n, pat, window);
    CHECK(p.steps.size() == whole.steps.size() && !p.parts.empty() && p.parts[0].first_step == 0,
          "n=%d %s", n, pat);
    if (window > whole.host_tables.size()) CHECK(p.parts.size() == 1, "n=%d %s", n, pat);
    for (size_t i = 0; i < p.parts.size(); i++) {
      const TablePart &t = p.parts[i];
      const size_t last = i + 1 < p.parts.size() ? p.parts[i + 1].first_step : p.steps.size();
      CHECK(last > t.first_step && t.bytes <= window && t.offset + t.bytes <= p.host_tables.size(),
            "n=%d %s part %zu", n, pat, i);
      const unsigned char *part = p.host_tables.data() + t.offset;
      CHECK(p.oz_const + consts <= t.bytes &&
                !memcmp(part + p.oz_const, whole.host_tables.data() + whole.oz_const, consts),
            "n=%d %s part %zu: constants", n, pat, i);
      for (size_t s = t.first_step; s < last; s++) {
        const Step &a = p.steps[s], &b = whole.steps[s];
        const size_t bytes = step_table_bytes(b);
        CHECK(a.kind == b.kind && a.table % 64 == 0 && a.table >= consts &&
                  a.table + bytes <= t.bytes &&
                  !memcmp(part + a.table, whole.host_tables.data() + b.table, bytes),
              "n=%d %s step %zu", n, pat, s);
      }
    }
  }
}

int main() {
  const int modes[] = {CAPS_MODE_FP64, CAPS_MODE_OZAKI_INT8, CAPS_MODE_CRT_INT8,
                       CAPS_MODE_CRT_BF16};
  for (int mode : modes)
    for (int fuse = 0; fuse < 2; fuse++) {
      const int k = mode == CAPS_MODE_FP64 ? 0 : 14;
      for (const char *pat : {"ddd", "bdd", "dbd", "bbb", "dbb", "bbd", "hdb"}) {
        check(392, 3, 7, pat, mode, k, fuse, 0);
        check(136, 3, 1, pat, mode, k, fuse, 0);
      }
      check(512, 2, 1, "bb", mode, k, fuse, 0);
      check(8192, 2, 1, "bb", mode, k, fuse, 0);
      check(64, 0, 1, "", mode, k, fuse, 0);
      if (mode != CAPS_MODE_OZAKI_INT8) check(1024, 3, 1, "bdd", mode, k, fuse, 1);
    }
  for (int kind : {STEP_EW, STEP_GEMM_F64, STEP_REORDER, STEP_OZ_SCALE, STEP_OZ_SPLIT,
                   STEP_OZ_GEMM, STEP_OZ_RECON, STEP_REW, STEP_CRT_SCALE, STEP_CRT_SPLIT,
                   STEP_CRT_RECON, STEP_BB_PRE, STEP_BB_POST, STEP_BB_SPLIT_A, STEP_BB_SPLIT_B,
                   STEP_FUSED_PRE, STEP_FUSED_POST})
    if (!kinds.count(kind)) {
      printf("FAIL no step of kind %d\n", kind);
      fails++;
    }
  if (!fails) printf("OK\n");
  return fails != 0;
}
