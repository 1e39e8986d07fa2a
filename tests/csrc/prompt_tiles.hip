// Host check of lbk::prompt_tile (lowbit_amd/csrc/lb_internal.h), the workgroup -> tile map
// of the prompt GEMMs: for every grid of 1..40 x 1..70 tiles each tile is taken by one
// workgroup, the surplus ones are told so, and nothing is divided by zero on the way.
// Prints "tiles <count> bad <count>".
#include <cstdio>
#include <vector>

#include "lb_internal.h"

int main() {
  long tiles = 0, bad = 0;
  for (int mt = 1; mt <= 40; mt++)
    for (int nt = 1; nt <= 70; nt++) {
      std::vector<int> hits((size_t)mt * nt);
      const unsigned grid = lbk::prompt_grid(mt, nt);
      for (unsigned b = 0; b < grid; b++) {
        int tm = -1, tn = -1;
        if (!lbk::prompt_tile(b, mt, nt, tm, tn)) continue;
        if (tm < 0 || tm >= mt || tn < 0 || tn >= nt) bad++;
        else hits[(size_t)tm * nt + tn]++;
      }
      for (const int h : hits) tiles++, bad += h != 1;
    }
  std::printf("tiles %ld bad %ld\n", tiles, bad);
  return bad != 0;
}
