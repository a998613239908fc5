// The rows of a fast step's tiles as the kernels find them (FastTilesInverse),
// against the division: for steps of one to six levels every tiles-per-row and
// every row that a level's sides allow, the first and the last tile of each row.
// Both quotients only grow with the tile, so the tiles between are right too.
#include <stdio.h>

#include "groups.hpp"

using namespace nvpro_pyramid;

template <int COUNT>
static uint64_t check()
{
  const uint32_t most = 65535u >> COUNT;
  uint64_t wrong = 0;
  for(uint32_t x = 1; x <= most; ++x)
  {
    const FastTilesInverse<COUNT> tiles(x, x * most, FastTilesInverse<COUNT>::inverseOf(x));
    uint64_t bad = 0;
    for(uint32_t row = 0; row < most; ++row)
      bad += (tiles.row(row * x) != row) + (tiles.row(row * x + x - 1u) != row);
    if(bad && wrong == 0)
      fprintf(stderr, "%d levels, %u tiles a row: %llu wrong\n", COUNT, x, (unsigned long long)bad);
    wrong += bad;
  }
  return wrong;
}

int main()
{
  const uint64_t wrong = check<1>() + check<2>() + check<3>() + check<4>() + check<5>() + check<6>();
  printf("%llu wrong\n", (unsigned long long)wrong);
  return wrong ? 1 : 0;
}
