// batch_rules.h -- which grids of a batch take several steps in one pass over
// memory (stencil_steps.h), and in bands of how many rows.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdint>
#include <vector>

namespace custen {
namespace dev {

constexpr int kFusedSteps = 3;

// Columns that a strip of a pass of K steps stores, of 128: whole 64-byte pieces
// (with 124 and 120 FP32 columns the pass was 10-15 % slower for the lines
// shared by two strips).
__host__ __device__ constexpr int stepsColumns(int size, int H, int K)
{
    return (128 - (K - 1) * (H - 1)) / (64 / size) * (64 / size);
}

// Strips and bands of a grid's pass: bands of `rows` rows, at most `most`.
struct StepsGrid {
    int strips, bands, rows;
};
__host__ __device__ inline StepsGrid stepsGrid(int size, int H, int nx, int ny, int most)
{
    StepsGrid g;
    const int ow = stepsColumns(size, H, kFusedSteps);
    g.strips = (nx + ow - 1) / ow;
    g.bands = (ny + most - 1) / most;
    g.rows = (ny + g.bands - 1) / g.bands;
    return g;
}

}  // namespace dev

// The grids that passes are for: one wrap correction must do for every column
// and row a wave starts at, and a row's bytes for the 31 bits of a buffer's
// range.
inline bool stepsApply(int nx, int ny) { return nx >= 128 && nx < (1 << 28) && ny >= 16; }

// A 5x5 grid of 128 columns takes two strips of a pass for the one of single
// steps; us per step, passes against single steps, 60 M points:
//   128 columns, FP64, 16 rows: 215, 164   128: 167, 164   FP32, 16: 124, 88   1000: 101, 85
//   256 columns, FP64, 16 rows: 167, 169   256: 128, 169   FP32, 16: 93, 92    1000: 92, 92
//   130 columns, FP64, 64 rows: 169, 269                   FP32, 64: 99, 152
// and 3x3, which has the FMAs to spare, 128 columns: FP64, 16 rows 118, 160,
// FP32 82, 84.  Such grids are left out where they are most of the batch, but a
// few beside wider ones cost less in the pass than as three small launches of
// their own (128 grids of 128 to 2048 points a side, ten steps: 2710 us with them,
// 2775 without).
inline bool stepsDouble(int size, int H, int nx)
{
    return H == 5 && dev::stepsGrid(size, H, nx, 16, 16).strips >= 2 * ((nx + 127) / 128);
}

// Several steps in one pass pay once the two sides no longer stay in the L2s
// (8 x 4 MiB): single steps then wait for memory, and a pass takes a third of
// its traffic.  In L2 a single step costs 4-6 us and a pass is bound by its
// chain of rows.  31 steps, single against passes, in us, by MiB a side:
//   FP64 5x5   16: 196, 288   32:  470, 412   64:  957, 699   128: 1720, 1164
//   FP32 5x5   16: 220, 280   32:  560, 429   64: 1056, 707
//   FP64 3x3   16: 174, 160   32:  495, 238   64:  918, 434   128: 1668, 760
//   FP32 3x3   16: 188, 165   32:  516, 279   64:  979, 552
constexpr int64_t kStepBytes5 = 24 << 20, kStepBytes3 = 16 << 20;
// Most rows of a pass's band.  Short bands repeat more rows (V - 1 for each
// step) and long ones come in few rounds of waves.  In FP64 a batch takes the
// length of 128, 64, 32, 16 for which rounds times rows is least, where a wave
// holds 11 KB of LDS (14 on a CU) and the last round counts 0.4.  In FP32, with
// twice as many waves on a CU, it takes the longest that gives 12 waves to a
// CU.  Waves of lower grids count by their length, and each XCD runs an eighth of
// the items, in order: where tall grids' long waves would all be on the first
// XCDs, it is the share of those that counts in FP64, and FP32 takes shorter bands
// (four 1024 x 1024 grids beside 1000 of 300 x 20: 44 us a step with bands of 128
// rows, 20 with 32).  5x5, us per step, by rows:
//   FP64, forty 2048 x 2048 grids     64: 268   128: 262   256: 268
//   FP64, sixteen 2048 x 2048 grids   64: 115   128: 125
//   FP64, sixteen 1024 x 1024 grids   16: 41.3   32: 37.5
//   FP32, sixteen 2048 x 2048 grids   64: 69.5   128: 64.1
//   FP32, 32 1024 x 1024 grids        32: 43.8   64: 37.5
constexpr int kStepRows = 128;
constexpr int kStepSlots = 14 * 256, kStepWaves32 = 12 * 256;
constexpr double kStepUneven = 1.25;  // most work of an XCD against the mean

struct GridSize {
    int nx, ny;
};
struct StepsChoice {
    std::vector<char> stepped;  // of each grid
    int rows = 16;              // most rows per band
};

// What a batch of H x H stencils on elements of `size` bytes takes in passes.
// `single`: the caller configured single steps.
inline StepsChoice chooseSteps(const std::vector<GridSize>& grids, int size, int H, bool single)
{
    StepsChoice c;
    c.stepped.assign(grids.size(), 0);
    int64_t bytes = 0, doubled = 0;
    for (size_t i = 0; i < grids.size(); i++) {
        const GridSize& g = grids[i];
        if (single || !stepsApply(g.nx, g.ny)) continue;
        c.stepped[i] = 1;
        bytes += (int64_t)g.nx * g.ny * size;
        if (stepsDouble(size, H, g.nx)) doubled += (int64_t)g.nx * g.ny * size;
    }
    if (doubled > bytes - doubled) {
        bytes -= doubled;
        for (size_t i = 0; i < grids.size(); i++)
            if (stepsDouble(size, H, grids[i].nx)) c.stepped[i] = 0;
    }
    if (bytes <= (H == 5 ? kStepBytes5 : kStepBytes3)) {
        c.stepped.assign(grids.size(), 0);
        return c;
    }
    double least = 0;
    for (int rows = kStepRows; rows >= 16; rows /= 2) {
        int64_t items = 0;
        for (size_t i = 0; i < grids.size(); i++) {
            if (!c.stepped[i]) continue;
            const dev::StepsGrid s = dev::stepsGrid(size, H, grids[i].nx, grids[i].ny, rows);
            items += (int64_t)s.strips * s.bands;
        }
        // row-steps of the longest wave and of an XCD's (6: what a wave costs beside)
        const int64_t share = std::max<int64_t>(1, (items + 7) / 8);
        double longest = 0, work = 0, most = 0, here = 0;
        int64_t room = share;
        for (size_t i = 0; i < grids.size(); i++) {
            if (!c.stepped[i]) continue;
            const dev::StepsGrid s = dev::stepsGrid(size, H, grids[i].nx, grids[i].ny, rows);
            const double wave = std::min(rows, grids[i].ny) + dev::kFusedSteps * (H - 1) + 6;
            longest = std::max(longest, wave);
            for (int64_t n = (int64_t)s.strips * s.bands; n > 0;) {
                const int64_t k = std::min(n, room);
                work += wave * k;
                here += wave * k;
                most = std::max(most, here);
                n -= k;
                room -= k;
                if (room == 0) {
                    here = 0;
                    room = share;
                }
            }
        }
        const double time = std::max(1.0, 8 * most / longest / kStepSlots + 0.4) * longest;
        if (rows == kStepRows || size == 4 || time < least) {
            least = time;
            c.rows = rows;
        }
        if (size == 4 && work / longest >= kStepWaves32 && 8 * most <= kStepUneven * work) break;
    }
    return c;
}

}  // namespace custen
