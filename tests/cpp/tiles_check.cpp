// Lines per work-group that public_amd/csrc/tiles.hpp chooses.
// Prints one line per grid, direction and precision: n1 n2 n3 d fp64 lines.
#include <cstdio>

#include "../../public_amd/csrc/tiles.hpp"

int main() {
  const int sizes[] = {16, 24, 32, 48, 64, 72, 128, 256, 512, 1024, 4096};
  for (int n1 : sizes)
    for (int n2 : sizes)
      for (int n3 : sizes) {
        const int np[3] = {n1, n2, n3};
        for (int d = 0; d < 3; ++d)
          for (int fp64 = 0; fp64 < 2; ++fp64)
            std::printf("%d %d %d %d %d %d\n", n1, n2, n3, d, fp64, cruna::auto_tile_lines(np, d, fp64, 512));
      }
  return 0;
}
