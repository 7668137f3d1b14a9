// Host-side check of merge_key (caps_amd/csrc/engine.cpp): products written in
// interleaved segments (RGemm::cseg), which the 256-tile kernels alone write, never
// join a segmented launch, whatever block tile the estimate gives for it.
// residue_block_tile here takes the place of the library's: 256 for the products'
// own launch, 192 for the launch that merging asks about.
#include <cstdio>

#include "../../caps_amd/csrc/engine.cpp"

namespace caps {
int residue_block_tile(int, int, int, long long problems) {
  return problems < (1 << 20) ? 256 : 192;
}
}  // namespace caps

int main() {
  using namespace caps;
  int products[2] = {0, 0}, merged[2] = {0, 0};  // plain, in segments
  for (const char *pat : {"bb", "bd"}) {
    Plan plan;
    const caps_desc d{4096, 2, 1, 1, 1, 1, 1};
    if (build_plan(plan, (double *)0x1000, (double *)0x2000, (double *)0x3000, d, pat,
                   CAPS_MODE_CRT_INT8, 14, 0, (void *)0x100000) != CAPS_OK) {
      printf("FAIL build %s\n", pat);
      return 1;
    }
    for (const Step &st : plan.steps)
      if (st.kind == STEP_OZ_GEMM) {
        const RGemm *g = reinterpret_cast<const RGemm *>(&plan.host_tables[st.table]);
        for (int p = 0; p < st.count; p++)
          if (g[p].cseg != g[0].cseg) {
            printf("FAIL one step, two segment strides\n");
            return 1;
          }
        products[g->cseg != 128]++;
        merged[g->cseg != 128] += merge_key(plan, st).kind >= 0;
      }
  }
  if (products[0] == 0 || products[1] != 1 || merged[0] != products[0] || merged[1] != 0) {
    printf("FAIL %d plain products, %d may merge; %d in segments, %d may merge\n", products[0],
           merged[0], products[1], merged[1]);
    return 1;
  }
  printf("OK\n");
  return 0;
}
