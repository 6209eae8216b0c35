// fstage_place (fx_place.h): every workgroup's share of every group of blocks
// is taken once, those of one group lie on one XCD and so do the neighbouring
// groups of an eighth of a row, and a launch of few groups uses every XCD alike.
// tile_turns: every row of V with an input is stored, and no turn has none.
#include <algorithm>
#include <cstdio>
#include <vector>
#include "../../difx-svn2git-try3_amd/csrc/fx_place.h"

static int check(unsigned groups, unsigned rows, unsigned PW) {
  const fxg::FsGrid dims = fxg::fstage_grid(groups, rows, PW);
  const unsigned all = groups * rows, eighth = (groups + 7) / 8;
  if (dims.x % (8 * PW)) return 1;
  std::vector<int> taken(all * PW, 0), xcd(all, -1), on(8, 0);
  for (unsigned y = 0; y < dims.y; y++)
    for (unsigned x = 0; x < dims.x; x++) {
      const fxg::FsPlace p = fxg::fstage_place(x, y, dims.x, groups, PW);
      if (p.row >= rows || p.grp >= groups) continue;
      if (p.pw >= PW) return 2;
      const unsigned g = p.row * groups + p.grp;
      const int at = (int)((x + y * dims.x) % 8);
      taken[g * PW + p.pw]++;
      if (xcd[g] >= 0 && xcd[g] != at) return 3;
      xcd[g] = at;
      on[at]++;
    }
  for (int t : taken)
    if (t != 1) return 4;
  for (unsigned g = 0; g < all; g++)
    if (g % groups % eighth && xcd[g] != xcd[g - 1]) return 5;
  // below 64 groups, eight rows give every XCD the same and fewer none more than
  // eight would; from there on no XCD has more than an eighth of each row
  const unsigned most = groups < 64 ? (rows + 7) / 8 * groups * PW : rows * eighth * PW;
  if (*std::max_element(on.begin(), on.end()) > (int)most) return 6;
  return groups < 8 && dims.x * dims.y >= (all + 8 * groups) * PW ? 7 : 0;
}

int main() {
  int bad = 0;
  for (unsigned PW = 1; PW <= 8; PW *= 2)
    for (unsigned rows : {1u, 2u, 7u, 24u, 144u})
      for (unsigned groups = 1; groups <= 80; groups++)
        if (const int e = check(groups, rows, PW)) {
          if (!bad) printf("%u groups, %u rows, %u a group: %d\n", groups, rows, PW, e);
          bad++;
        }
  for (int nin = 1; nin <= 130; nin++)
    for (int row0 = 0; row0 < 128; row0 += 32)
      for (int g = 0; g < 4; g++) bad += (row0 + 8 * g < nin) != (g < fxg::tile_turns(nin - row0));
  printf("%s: %d\n", bad ? "FAIL" : "PASS", bad);
  return bad ? 1 : 0;
}
