// stencil_steps.h -- several steps of a periodic xy stencil in one pass over the
// grid (batched grids, batch.hip).
//
// A single step reads and writes the field once, 16 bytes a point in FP64,
// and runs at the memory's copy rate with two thirds of the FMA units idle.
// Here one wave takes K = 3 steps of its strip before it stores, so a step's
// share of the memory time falls to a third; the FP64 5x5 pass then takes
// longer for its FMAs than for memory, so more steps would gain nothing.
//
// The wave walks down a band one row at a time.  A row of step k's input adds
// to the V output rows it belongs to, whose sums are in registers, and
// completes one of them; that row goes through one row of LDS (neighbouring
// columns are other lanes') to step k+1, or to memory after step K.  A row is
// thus read from LDS once per step, and LDS holds only the input rows in
// flight (D of them) and one row per step: 11 KB for FP64 5x5, so that 14 waves
// fit on a CU.  (With chunks of four output rows from a window of eight rows in
// LDS, 29 KB and five waves, a pass over forty 2048 x 2048 grids took 960 us;
// 787 here when it is repeated for long, 661 when it is not: random data draw
// more power than the clock holds under, and a pass over zeros takes 593.  Three
// single steps take 1330.)
//
// Step k of a strip is computed for 128 - (k-1)(H-1) columns, each step's
// range inside the last one's by the stencil's extents, so a strip stores at
// most 128 - (K-1)(H-1) columns (120 of 128 for 5x5), and a band of n rows
// computes n + (K-k)(V-1) rows of step k.  Neighbouring strips and bands compute the
// overlap from the same values in the same order, so every point has the bits
// of K single steps.
#pragma once

#include <type_traits>

#include "batch_rules.h"
#include "lds_ring.h"  // row buffers
#include "stencil_band.h"

#pragma clang fp contract(off)

namespace custen {
namespace dev {

template <typename T, int H, int V, int K>
struct StepsShape {
    static constexpr int D = 8;                          // input rows in flight or in use
    static constexpr int OW = stepsColumns(sizeof(T), H, K);  // columns stored per strip
    static constexpr int HLP = ((H - 1) + 1) & ~1;       // halo columns staged per side
    static constexpr int LD = kTW + 2 * HLP;             // input ring row
    static constexpr int MID = kTW + 2 * HLP;            // row between steps (reads of its unused
                                                         // last columns run on)
    static constexpr int ELEMS = D * LD + (K - 1) * MID;
};

// Rows that lanes wrote to LDS may be read by other lanes of the wave from here
// on.  The LDS takes a wave's operations in order, so this costs no
// instruction, but the compiler sees one lane, whose reads of its neighbours'
// columns do not alias what it wrote, and might move them up.
__device__ __forceinline__ void rowsWritten()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// K steps of wave item g of a grid (periodic, nx x ny, row stride nx).  `lds`
// is the wave's StepsShape::ELEMS elements.
template <typename T, int H, int V, int K>
__device__ __forceinline__ void stepsWalk(const Glob<T>* __restrict__ in, Glob<T>* __restrict__ out,
                                          int nx, int ny, int L, int Tt, const T (&w)[H * V],
                                          Lds<T>* __restrict__ lds, int most, int g)
{
    using SH = StepsShape<T, H, V, K>;
    using V2 = typename Vec2<T>::type;
    constexpr int D = SH::D, HLP = SH::HLP, LD = SH::LD;
    constexpr int TAIL = 2 * HLP * (int)sizeof(T) / 4;  // dwords of a ring row past 128 columns
    constexpr int FLAT = sizeof(T) == 8 ? 4 : 2;  // 4-byte loads of a row body
    static_assert((H + 1) % 2 == 0, "pair reads");
    const int lane = threadIdx.x;
    const StepsGrid sg = stepsGrid(sizeof(T), H, nx, ny, most);
    const int band = __builtin_amdgcn_readfirstlane(g / sg.strips);
    const int strip = g - band * sg.strips;
    const int n = __builtin_amdgcn_readfirstlane(sg.rows);
    const int yS = min(band * n, ny - n);
    const int x0 = min(strip * SH::OW, nx - SH::OW);
    const int x1 = x0 - (K - 1) * L;  // first column of step 1

    auto wrapCol = [&](int c) { return c < 0 ? c + nx : (c >= nx ? c - nx : c); };
    // FP64 rows: 16 bytes per lane, unless a pair of columns straddles the wrap
    // (odd position or width); then, and for FP32, 4 bytes per lane.
    const bool wide = sizeof(T) == 8 && ((x1 >= HLP && x1 - HLP + kTW <= nx) || ((x1 | nx) & 1) == 0);
    const int xs = x1 - HLP;  // first column staged
    const uint32_t bodyOff = (uint32_t)wrapCol(xs + 2 * lane) * sizeof(T);
    uint32_t flatOff[FLAT];
#pragma unroll
    for (int i = 0; i < FLAT; i++) {
        const int dword = i * kLanes + lane;
        flatOff[i] = sizeof(T) == 8
                         ? (uint32_t)wrapCol(xs + (dword >> 1)) * 8u + (uint32_t)(dword & 1) * 4u
                         : (uint32_t)wrapCol(xs + dword) * 4u;
    }
    const int tl = min(lane, TAIL - 1);
    const uint32_t tailOff =
        sizeof(T) == 8 ? (uint32_t)wrapCol(xs + kTW + (tl >> 1)) * 8u + (uint32_t)(tl & 1) * 4u
                       : (uint32_t)wrapCol(xs + kTW + tl) * 4u;

    // input row t (of the rows from the first that step 1 reads) is in ring
    // slot t mod D; rows are loaded in order.  A row is a buffer with its base
    // in scalar registers, so a load has no vector address arithmetic.
    int sy = yS - K * Tt;
    if (sy < 0) sy += ny;
    int loaded = 0;
    const int need = n + K * (V - 1);
    auto loadRow = [&]() {
        const __amdgpu_buffer_rsrc_t rs = rowBuffer((const void*)(in + (int64_t)sy * nx));
        // past the last row needed, that row again (the count of loads in flight
        // stays what it is)
        sy = __builtin_amdgcn_readfirstlane(loaded + 1 >= need ? sy : (sy + 1 == ny ? 0 : sy + 1));
        Lds<char>* l = (Lds<char>*)(lds + (loaded & (D - 1)) * LD);
        loaded = __builtin_amdgcn_readfirstlane(loaded + 1);
        if (wide) {
            rowDma<16>(rs, l, bodyOff, 0);
        } else {
#pragma unroll
            for (int i = 0; i < FLAT; i++)
                rowDma<4>(rs, l + i * kLanes * 4, flatOff[i], 0);
        }
        if (lane < TAIL) rowDma<4>(rs, l + kTW * sizeof(T), tailOff, 0);
    };
    // Row t + 1 has landed once no more than the loads of the D-1 rows after it
    // are outstanding, and the stores of the iterations since it was loaded
    // where each of them stored.
    constexpr int FIRST = V - 1 + (K - 1) * V;  // the iteration of the first store
    auto waitRow = [&](int t) {
        const bool stored = t >= FIRST + D - 1 && t <= FIRST + n;
        if (wide && stored) waitVmcnt<(D - 1) * 3>();
        else if (wide) waitVmcnt<(D - 1) * 2>();
        else waitVmcnt<(D - 1) * (FLAT + 1)>();
    };
    auto readPairs = [&](T(&v)[H + 1], const Lds<T>* row) {
#pragma unroll
        for (int q = 0; q < (H + 1) / 2; q++) {
            const V2 p = ((const Lds<V2>*)row)[q];
            v[2 * q] = p.x;
            v[2 * q + 1] = p.y;
        }
    };
    auto readInput = [&](T(&v)[H + 1], int t) {
        const Lds<T>* row = lds + (t & (D - 1)) * LD + (HLP - L) + 2 * lane;
        if (((HLP - L) & 1) == 0) {
            readPairs(v, row);
        } else {
#pragma unroll
            for (int k = 0; k < H + 1; k++) v[k] = row[k];
        }
    };
    Lds<T>* mid[K];
#pragma unroll
    for (int k = 1; k < K; k++) mid[k] = lds + D * LD + (k - 1) * SH::MID + 2 * lane;

    // Row t of step k's input (k = 0 .. K-1 here): adds weight row j to output
    // row t - j, whose sums are acc[k][(t - j) mod V].  Step k+1 takes at
    // iteration t the row that step k completed at iteration t-1, its input
    // row t - V: all steps have the same row modulo V, which is p here.
    T acc[K][V][2];
#pragma unroll
    for (int k = 0; k < K; k++)
#pragma unroll
        for (int s = 0; s < V; s++) acc[k][s][0] = acc[k][s][1] = T(0);
    auto addRow = [&](T(&a)[V][2], const T(&v)[H + 1], auto pc) {
        constexpr int p = decltype(pc)::value;
#pragma unroll
        for (int j = V - 1; j >= 0; j--) {
            constexpr int VV = V;
            const int s = (p - j + VV) % VV;
            if (j == 0) a[s][0] = a[s][1] = T(0);
#pragma unroll
            for (int i = 0; i < H; i++) {
                a[s][0] = fmaT(w[j * H + i], v[i], a[s][0]);
                a[s][1] = fmaT(w[j * H + i], v[i + 1], a[s][1]);
            }
        }
        // The sums are taken here, not where the compiler would rather have
        // them: it sinks the chains of a whole group to the rows that complete
        // them, keeping five rows' values in registers instead (246 of them).
#pragma unroll
        for (int s = 0; s < V; s++) __asm__ __volatile__("" : "+v"(a[s][0]), "+v"(a[s][1]));
    };
    T v0[H + 1];
    // One iteration.  A step adds nothing before its first row is there (3 % of
    // ten FP64 5x5 steps over 178 M points in grids of 256 to 2048 points a
    // side); after its last row it goes on, and what it adds reaches no sum that
    // is stored.  (A second body of code for the band's ends took twice the
    // registers.)
    auto iterate = [&](auto pc, int t) {
        constexpr int p = decltype(pc)::value;
        constexpr int done = (p + 1) % V;  // the sums that this row completes
        T v[K][H + 1];
#pragma unroll
        for (int k = 1; k < K; k++) readPairs(v[k], mid[k]);
        __builtin_amdgcn_sched_barrier(0);
        addRow(acc[0], v0, pc);
        __builtin_amdgcn_sched_barrier(0);
        loadRow();
        waitRow(t);
        readInput(v0, t + 1);
#pragma unroll
        for (int k = 1; k < K; k++) {
            *(Lds<V2>*)mid[k] = V2{acc[k - 1][done][0], acc[k - 1][done][1]};
            __builtin_amdgcn_sched_barrier(0);
            if (t >= k * V) addRow(acc[k], v[k], pc);
            __builtin_amdgcn_sched_barrier(0);
        }
        rowsWritten();
        const int o = t - (V - 1) - (K - 1) * V;
        if (o >= 0 && o < n) {
            const V2 r = {acc[K - 1][done][0], acc[K - 1][done][1]};
            if (lane < SH::OW / 2)
                __builtin_nontemporal_store(
                    ElemVec2<T>(r), reinterpret_cast<Glob<ElemVec2<T>>*>(
                                        out + (int64_t)(yS + o) * nx + x0 + 2 * lane));
        }
    };
    static_assert(V == 3 || V == 5, "the unrolled groups");
#pragma unroll 1
    for (int r = 0; r < D; r++) loadRow();
    waitRow(-1);
    readInput(v0, 0);
    // iterations, in groups of V that the last one need not fill (3-6 % of 100
    // FP64 5x5 steps, by the length of the bands)
    const int total = n + K * V - 1;
    for (int t = 0; t < total;) {
        iterate(std::integral_constant<int, 0>{}, t);
        if (t + 1 == total) break;
        iterate(std::integral_constant<int, 1>{}, t + 1);
        if (t + 2 == total) break;
        iterate(std::integral_constant<int, 2>{}, t + 2);
        if constexpr (V == 5) {
            if (t + 3 == total) break;
            iterate(std::integral_constant<int, 3>{}, t + 3);
            if (t + 4 == total) break;
            iterate(std::integral_constant<int, 4>{}, t + 4);
        }
        t = __builtin_amdgcn_readfirstlane(t + V);  // (kept in a scalar register)
    }
}

}  // namespace dev
}  // namespace custen
