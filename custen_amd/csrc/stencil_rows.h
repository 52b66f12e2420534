// stencil_rows.h -- row-streaming band kernel for the wide FP64 xy stencils.
//
// The chunked band walker (stencil_band.h) reads each input row from LDS once
// for every output row that it belongs to and has no registers left for 49 or
// 81 FP64 weights, which it loads from the scalar cache before the FMAs of each
// row.  Here a wave walks its band one input row at a time: the row is read
// from LDS once and added to the V output rows it belongs to, whose sums stay in
// registers, and it completes one of them.  Every weight is then used once a
// row, so they stay in registers too, part of them scalar.  The FMAs bound it,
// and on random data the clock that their power leaves: 9x9 at 4096 x 4096 takes
// 66 us (43 TFLOP/s with the rows repeated at the bands' ends), 84 in chunks.
//
// A band of n rows adds V - 1 rows more, whose sums are not all stored, so it
// needs long bands: launches with too few rows for them keep the chunks.
// Sums are formed in the order of the other stencil kernels.
#pragma once

#include <type_traits>

#include "stencil_band.h"

#pragma clang fp contract(off)

namespace custen {
namespace dev {

// Stencils that stream rows, and the least rows of a band that they do it for.
template <typename T, int H, int V>
constexpr bool kStreamRows = sizeof(T) == 8 && H == V && (H == 7 || H == 9);
constexpr int kStreamBand = 28;

template <int H, int V>
struct RowsShape {
    static constexpr int D = 8;                        // input rows in flight or in use
    static constexpr int HLP = ((H - 1) + 1) & ~1;     // halo columns staged per side
    static constexpr int LD = kTW + 2 * HLP;
    static constexpr int NS = 34;                      // weights in scalar registers
    static constexpr int LDS_BYTES = D * LD * 8;
};

// Bands of about 4 * chunks rows, of equal length; the last ends at the last
// row.  (The host counts waves with the same function.)
constexpr int kRowsRPW = 4;
__host__ __device__ inline int rowsBands(const BandGrid& g, int chunks)
{
    const int most = kRowsRPW * chunks;
    return (g.yb - g.ya + most - 1) / most;
}

template <int H, int V>
__global__ __launch_bounds__(kLanes) void stencilRows(StencilLaunch a)
{
    using SH = RowsShape<H, V>;
    using V2 = typename Vec2<double>::type;
    constexpr int D = SH::D, HLP = SH::HLP, LD = SH::LD, HL = HLP * 2;
    __shared__ __attribute__((aligned(16))) double lds[D * LD];
    Lds<double>* ring = (Lds<double>*)lds;
    double w[H * V];
#pragma unroll
    for (int k = 0; k < H * V; k++) w[k] = a.weights[k];
#pragma unroll
    for (int k = SH::NS; k < H * V; k++) {
        // an empty asm with a vector-register result keeps the value there
        double o;
        __asm__ __volatile__("" : "=v"(o) : "0"(w[k]));
        w[k] = o;
    }

    const int lane = threadIdx.x;
    const BandGrid bg = bandGrid(a, kRowsRPW);
    const int g = xcdRemap(blockIdx.x, gridDim.x);
    const int strip = g % bg.strips, band = g / bg.strips;
    const int bands = rowsBands(bg, a.chunks);
    const int n = __builtin_amdgcn_readfirstlane((bg.yb - bg.ya + bands - 1) / bands);
    const int yS = min(bg.ya + band * n, bg.yb - n);
    const int x0 = bg.x0(strip);
    const int nx = a.nx, L = a.L;
    const Glob<double>* __restrict__ in = globalPtr<double>(a.in);
    Glob<double>* __restrict__ out = globalPtr<double>(a.out);

    // halo columns staged by this lane (lanes < HL, one dword each)
    int colL = x0 - HLP + (lane >> 1), colR = x0 + kTW + (lane >> 1);
    if (a.xWrap) {
        if (colL < 0) colL += nx;
        if (colR >= nx) colR -= nx;
    } else {
        colL = colL < 0 ? 0 : colL;
        colR = colR >= nx ? nx - 1 : colR;
    }

    // Input row t (row 0 is yS - T) goes to ring slot t mod D.
    const RowMap rows = a.rows;
    const int need = n + V - 1;
    int loaded = 0;
    int gy = yS - a.T, sy = mapRowNear(rows, gy);
    auto loadRow = [&]() {
        const Glob<double>* row = in + (int64_t)sy * a.ldIn;
        Lds<double>* l = ring + (loaded & (D - 1)) * LD;
        loaded = __builtin_amdgcn_readfirstlane(loaded + 1);
        // past the last row needed, that row again (the count of loads in
        // flight stays what it is)
        if (loaded < need) {
            gy++;
            if (rows.wrap) sy = sy + 1 == rows.rowWrap ? 0 : sy + 1;
            else sy = min(max(gy, rows.rowMin), rows.rowMax);
        }
        sy = __builtin_amdgcn_readfirstlane(sy);
        ldsDma16<kDmaDefault>(row + x0 + 2 * lane, l + HLP);
        if (lane < HL) {
            ldsDma4<kDmaDefault>((const Glob<unsigned>*)(row + colL) + (lane & 1), l);
            ldsDma4<kDmaDefault>((const Glob<unsigned>*)(row + colR) + (lane & 1), l + HLP + kTW);
        }
    };

    double acc[V][2];
#pragma unroll
    for (int s = 0; s < V; s++) acc[s][0] = acc[s][1] = 0.0;
    // Row t adds weight row j to output row t - j, whose sums are
    // acc[(t - j) mod V], and completes output row t - (V - 1).
    auto iterate = [&](auto pc, int t) {
        constexpr int p = decltype(pc)::value;
        constexpr int done = (p + 1) % V;
        // row t has landed once no more than the loads of the D - 1 rows after
        // it are outstanding, and the stores since it was loaded where each
        // iteration stored
        if (t >= V - 1 + D && t <= n + V - 1) waitVmcnt<(D - 1) * 4>();
        else waitVmcnt<(D - 1) * 3>();
        const Lds<double>* row = ring + (t & (D - 1)) * LD + (HLP - L) + 2 * lane;
        double v[H + 1];
        if (((HLP - L) & 1) == 0) {
#pragma unroll
            for (int q = 0; q < (H + 1) / 2; q++) {
                const V2 e = ((const Lds<V2>*)row)[q];
                v[2 * q] = e.x;
                v[2 * q + 1] = e.y;
            }
        } else {
#pragma unroll
            for (int k = 0; k < H + 1; k++) v[k] = row[k];
        }
#pragma unroll
        for (int j = V - 1; j >= 0; j--) {
            const int s = (p - j + V) % V;
            if (j == 0) acc[s][0] = acc[s][1] = 0.0;
#pragma unroll
            for (int i = 0; i < H; i++) {
                acc[s][0] = fmaT(w[j * H + i], v[i], acc[s][0]);
                acc[s][1] = fmaT(w[j * H + i], v[i + 1], acc[s][1]);
            }
        }
        // the sums are taken here: the compiler would rather keep the rows
        // and form the chains where they end
#pragma unroll
        for (int s = 0; s < V; s++) __asm__ __volatile__("" : "+v"(acc[s][0]), "+v"(acc[s][1]));
        loadRow();  // into the slot of the row just read
        const int o = t - (V - 1);
        if (o >= 0 && o < n) {
            const V2 r = {acc[done][0], acc[done][1]};
            __builtin_nontemporal_store(
                ElemVec2<double>(r),
                reinterpret_cast<Glob<ElemVec2<double>>*>(out + (int64_t)(yS + o) * a.ldOut + x0 +
                                                          2 * lane));
        }
    };
#pragma unroll 1
    for (int r = 0; r < D; r++) loadRow();
    static_assert(V == 7 || V == 9, "the unrolled groups");
    for (int t = 0; t < need;) {
        iterate(std::integral_constant<int, 0>{}, t);
        iterate(std::integral_constant<int, 1>{}, t + 1);
        iterate(std::integral_constant<int, 2>{}, t + 2);
        iterate(std::integral_constant<int, 3>{}, t + 3);
        iterate(std::integral_constant<int, 4>{}, t + 4);
        iterate(std::integral_constant<int, 5>{}, t + 5);
        iterate(std::integral_constant<int, 6>{}, t + 6);
        if constexpr (V == 9) {
            iterate(std::integral_constant<int, 7>{}, t + 7);
            iterate(std::integral_constant<int, 8>{}, t + 8);
        }
        t = __builtin_amdgcn_readfirstlane(t + V);
    }
}

}  // namespace dev
}  // namespace custen
