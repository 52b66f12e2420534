// batch_rules_check.cpp -- which grids of a batch take several steps to a pass
// (chooseSteps, custen_amd/csrc/batch_rules.h).
//
// usage: batch_rules_check <bytes per element> <H> <single> <count>x<nx>x<ny> ...
// prints "<rows per band> <stepped grids of each group> ..."
#define __HIP_PLATFORM_AMD__ 1
#include <cstdio>
#include <cstdlib>

#include "../../custen_amd/csrc/batch_rules.h"

int main(int argc, char** argv)
{
    std::vector<custen::GridSize> grids;
    std::vector<size_t> ends;
    for (int i = 4; i < argc; i++) {
        int n, nx, ny;
        if (std::sscanf(argv[i], "%dx%dx%d", &n, &nx, &ny) != 3) return 2;
        grids.insert(grids.end(), n, {nx, ny});
        ends.push_back(grids.size());
    }
    const custen::StepsChoice c = custen::chooseSteps(grids, std::atoi(argv[1]), std::atoi(argv[2]),
                                                      std::atoi(argv[3]) != 0);
    std::printf("%d", c.rows);
    size_t k = 0;
    for (size_t e : ends) {
        int n = 0;
        for (; k < e; k++) n += c.stepped[k];
        std::printf(" %d", n);
    }
    std::printf("\n");
    return 0;
}
