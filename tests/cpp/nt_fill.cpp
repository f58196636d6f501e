// Host-only: for each "m batch tile" of the arguments, whether nt_fill_pays puts the Q update of
// that many m x m matrices into three triangle launches of theirs on a GPU of 256 CUs.
#include <stdio.h>
#include <stdlib.h>

#include "../../dmuon_amd/csrc/dmuon_amd_internal.h"

int main(int argc, char** argv) {
  for (int i = 1; i + 2 < argc; i += 3) {
    const int m = atoi(argv[i]), tile = atoi(argv[i + 2]);
    dmuon::NtArgs a{};
    a.M = a.N = a.K = (m + tile - 1) / tile * tile;
    a.k_loop = (m + 63) / 64 * 64;
    a.live_rows = a.live_cols = a.k_loop < a.M ? a.k_loop : 0;
    a.L = atoi(argv[i + 1]);
    a.mt = a.nt = a.M / tile;
    a.tiles_per_mat = a.mt * a.nt;
    dmuon::NtArgs t = a;
    t.tri = 1;
    t.tiles_per_mat = a.mt * (a.mt + 1) / 2;
    printf("%d", dmuon::nt_fill_pays(&t, &a, 1, tile, 256) ? 1 : 0);
  }
  printf("\n");
  return 0;
}
