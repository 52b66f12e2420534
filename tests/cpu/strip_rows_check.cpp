// strip_rows_check.cpp -- the source rows of the strip kernel's tiles
// (mapRowNear where tileRowsNear holds, custen_amd/csrc/kernels.h) on periodic
// grids at least as tall as the window.  A tile holds rows [y0 - T, y0 + TH + B):
// every one of them has to be mapped to the right row of the grid.
//
// Prints "<rows looked up> <outside the grid> <wrong> <grids left to mapRow>".
#define __HIP_PLATFORM_AMD__ 1
#include <cstdio>

#include "../../custen_amd/csrc/kernels.h"

int main()
{
    long looked = 0, outside = 0, wrong = 0, left = 0;
    for (int TH : {16, 32, 64})
        for (int V : {1, 3, 5, 9, 13})
            for (int T = 0; T < V; T++)
                for (int ny = V; ny < 3 * TH; ny++) {
                    const int B = V - 1 - T;
                    const custen::RowMap m{1, ny, 0, ny - 1};
                    if (!custen::tileRowsNear(m, ny, V, T, TH)) {
                        left++;
                        continue;
                    }
                    for (int y0 = 0; y0 < ny; y0 += TH)
                        for (int gy = y0 - T; gy < y0 + TH + B; gy++) {
                            const int sy = custen::mapRowNear(m, gy);
                            looked++;
                            outside += sy < 0 || sy >= ny;
                            wrong += sy != ((gy % ny) + ny) % ny;
                        }
                }
    std::printf("%ld %ld %ld %ld\n", looked, outside, wrong, left);
    return 0;
}
