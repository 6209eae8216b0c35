// turn_units (fx_bits.h) against the definition, field by field, for every
// unit size and channel count the corner turn takes.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "../../difx-svn2git-try3_amd/csrc/fx_bits.h"

template <int U, int N> static int check() {
  const int nch = 1 << N, per = 32 / U;
  const uint32_t mask = (1u << U) - 1u;
  std::vector<uint32_t> in(nch), out;
  for (auto& w : in) w = ((uint32_t)rand() << 17) ^ ((uint32_t)rand() << 5) ^ (uint32_t)rand();
  out = in;
  fxg::turn_units<U, N>(out.data());
  for (int i = 0; i < nch; i++) {
    const int c = fxg::turned_channel<U, N>(i);
    for (int t = 0; t < per; t++) {
      const int bit = (t * nch + c) * U;
      if (((out[i] >> (t * U)) & mask) != ((in[bit / 32] >> (bit % 32)) & mask)) {
        printf("U %d channels %d: word %d time %d\n", U, nch, i, t);
        return 1;
      }
    }
  }
  return 0;
}
template <int U> static int check_all() {
  return check<U, 0>() + check<U, 1>() + check<U, 2>() + check<U, 3>() + check<U, 4>() + check<U, 5>() + check<U, 6>();
}

int main() {
  const int bad = check_all<2>() + check_all<4>() + check_all<8>() + check_all<16>();
  if (!bad) printf("ok\n");
  return bad ? 1 : 0;
}
