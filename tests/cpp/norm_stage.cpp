// Host-only: for each "batch rows cols kept" of the arguments, whether norm_stage_pays joins the norm
// and the exact staging of that many padded rows x cols matrices, with or without kept scales.
#include <stdio.h>
#include <stdlib.h>

#include "../../dmuon_amd/csrc/dmuon_amd_internal.h"

int main(int argc, char** argv) {
  for (int i = 1; i + 3 < argc; i += 4) {
    static float scale;
    float* const kept[1] = {&scale};
    dmuon::PreArgs p{};
    p.L = atoi(argv[i]);
    p.Rp = atoi(argv[i + 1]);
    p.Cp = atoi(argv[i + 2]);
    dmuon::NormArgs a{};
    a.L = p.L;
    a.nparts = dmuon::pre_blocks_per_mat(p.Rp, p.Cp);
    a.est_ptrs = atoi(argv[i + 3]) ? kept : nullptr;
    printf("%d", dmuon::norm_stage_pays(&a, 1, &p, 1) ? 1 : 0);
  }
  printf("\n");
  return 0;
}
