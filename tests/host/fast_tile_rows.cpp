// The rows of a fast step's tiles as the kernels find them (FastTilesInverse),
// against the division: every tiles-per-row a level can have, the first and the
// last tile of every row.  Both quotients only grow with the tile, so the tiles
// between are right too.  The one-level step has the most tiles of either
// direction; the ranges of the steps of more levels are part of its.
#include <stdio.h>

#include "groups.hpp"

using namespace nvpro_pyramid;

int main()
{
  const uint32_t most = 65535u >> 1;
  uint64_t checked = 0, wrong = 0;
  for(uint32_t x = 1; x <= most; ++x)
  {
    const FastTilesInverse tiles(x, x * most, FastTilesInverse::inverseOf(x));
    uint64_t bad = 0;
    for(uint32_t row = 0; row < most; ++row)
      bad += (tiles.row(row * x) != row) + (tiles.row(row * x + x - 1u) != row);
    if(bad && wrong == 0)
      fprintf(stderr, "%u tiles a row: %llu wrong\n", x, (unsigned long long)bad);
    wrong += bad;
    checked += 2u * most;
  }
  printf("%llu rows checked, %llu wrong\n", (unsigned long long)checked, (unsigned long long)wrong);
  return wrong ? 1 : 0;
}
