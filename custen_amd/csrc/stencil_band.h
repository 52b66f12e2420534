// stencil_band.h -- the band-walker stencil kernel: one wave streams a band
// of rows down its own 128-column strip, with no workgroup barrier.
//
// Rows go from HBM straight into LDS (global_load_lds: each lane's 16 or 4
// bytes land at LDS base + 16 * lane or 4 * lane, so one instruction stages a
// 128-column FP64 row body and two stage an FP32 one; one 4-byte load per
// side by the lanes that cover HLP columns stages the halo).  The wave keeps
// a ring of S row slots,
//     S = (D + 1) * RPW + V - 1,
// and while it computes chunk c (RPW output rows from RPW + V - 1 input rows)
// the rows of chunks c+1 .. c+D are in flight into the other slots, so no
// registers are spent on staging and the V-1 rows shared by consecutive
// chunks are never copied.  Completion is tracked with the vector-memory
// counter, which retires loads and stores in issue order: before chunk c the
// wave waits until no more than (loads issued after chunk c's) + (stores
// issued after chunk c's) operations are outstanding.
//
// Every point of a walked strip is written, so there are no store masks: the
// walked strips tile the written columns of the launch, the last one ending
// at the last written column (it overlaps its neighbour, and so may the first,
// when the window is not made of whole strips), and the chunks tile the written
// rows, the last band ending at the last of them.  Points in an overlap are computed by both
// waves from the same values in the same order.  A strip may start at any
// column and rows at any alignment of an element: the loads and stores need
// element alignment only.  At 4099 x 3001 (5x5, FP64, written window inside a
// two-cell border, odd rows) the apply takes 32.0 us (197 MB, 6.1
// TB/s), against 49.4 when such rows took the strip kernel's per-element path.
//
// Arithmetic is the fma chain of the other stencil kernels (row j outer,
// column i inner, from 0.0), so every configuration gives identical bits.
// The point-wise transform of the cube-minus point function (u^3 - u,
// unfused) is applied to each value as it is read from the ring; the strip
// kernel applies the same function while staging, so the values agree.
#pragma once

#include "stencil_tile.h"

#pragma clang fp contract(off)

namespace custen {
namespace dev {

// LDS (address space 3) views: the ring is addressed through them from the
// kernel down, so the compiler never has to turn a generic pointer into an
// LDS address.
typedef __attribute__((address_space(3))) void LdsVoid;
template <typename T> using Lds = __attribute__((address_space(3))) T;

// s_waitcnt with vmcnt = N and the other counters unconstrained (gfx9
// encoding: vmcnt[3:0] and [15:14], expcnt [6:4], lgkmcnt [11:8]).
template <int N>
__device__ __forceinline__ void waitVmcnt()
{
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
    __asm__ __volatile__("" ::: "memory");
}

// Wait for a chunk given la = chunks of loads and sa = chunks of stores
// issued after it (la < D, sa <= D): the immediate is la*NL + sa*NS.
template <int NL, int NS, int D, int A = 0, int B = 0>
__device__ __forceinline__ void waitChunk(int la, int sa)
{
    if constexpr (A >= D) {
        waitVmcnt<0>();
    } else if constexpr (B > D) {
        waitChunk<NL, NS, D, A + 1, 0>(la, sa);
    } else {
        if (la == A && sa == B) waitVmcnt<A * NL + B * NS>();
        else waitChunk<NL, NS, D, A, B + 1>(la, sa);
    }
}

// Direct-to-LDS loads use the default cache policy.  Non-temporal row loads
// were measured: 6-10 % faster when the same input is applied again and
// again (the unchanged input then stays partly in the last-level cache), but
// within 2 % either way in a time-stepping loop that alternates input and
// output, and 10-40 % slower for tall stencils and FP32 fields.  Since the
// autotuner times repeated applies of one input, that policy would also
// mislead it, so it is not used.
constexpr int kDmaDefault = 0;

template <int POLICY>
__device__ __forceinline__ void ldsDma16(const Glob<double>* g, Lds<double>* l)
{
    __builtin_amdgcn_global_load_lds((const Glob<void>*)g, (LdsVoid*)l, 16, 0, POLICY);
}
template <int POLICY, typename T>
__device__ __forceinline__ void ldsDma4(const Glob<unsigned>* g, Lds<T>* l)
{
    __builtin_amdgcn_global_load_lds((const Glob<void>*)g, (LdsVoid*)l, 4, 0, POLICY);
}

// A pair of elements at element alignment.
template <typename T> struct ElemPair;
template <> struct ElemPair<double> { typedef double type __attribute__((ext_vector_type(2), aligned(8))); };
template <> struct ElemPair<float> { typedef float type __attribute__((ext_vector_type(2), aligned(4))); };
template <typename T> using ElemVec2 = typename ElemPair<T>::type;

// FP64 stencils of more than 36 points have more weights than the scalar
// registers hold next to the walker's own state; held for the whole walk they
// are spilled and read back lane by lane.  The walk of those stencils instead
// loads each weight row from the scalar cache just before its FMAs (the
// weights are not written during a launch, so the constant address space
// applies).
template <typename T, int H, int V>
constexpr bool kStreamWeights = sizeof(T) == 8 && H * V > 36;

// FP32 stencils of more than 36 points: the weights (converted from the
// FP64 array on the vector unit) stay in vector registers, 49 or 81 of them,
// instead of being moved to scalar registers that then spill.
template <typename T, int H, int V>
constexpr bool kWeightsInVgprs = sizeof(T) == 4 && H * V > 36;

template <int H>
__device__ __forceinline__ void loadWeightRow(const double* weights, int j, double (&wr)[H],
                                              double after)
{
    // The empty asm makes the address opaque at each use and orders it after
    // `after` (the accumulator the row updates), so the loads stay next to
    // the FMAs that consume them instead of being hoisted out of the walk.
    uint64_t p = (uint64_t)weights;
    __asm__ __volatile__("" : "+s"(p) : "v"(after));
    typedef __attribute__((address_space(4))) const double CDouble;
    const CDouble* q = (const CDouble*)p;
#pragma unroll
    for (int i = 0; i < H; i++) wr[i] = q[j * H + i];
}

// Ring geometry of a band-walker instantiation (2 columns per lane).  A row
// body is one 16-byte load per lane for FP64 and two 4-byte loads (columns
// lane and 64 + lane) for FP32; each halo side is one 4-byte load by the
// lanes that cover HLP columns.
template <typename T, int H, int V, int RPW>
struct BandShape {
    static constexpr int D = 8 / RPW;                  // chunks in flight ahead
    static constexpr int HLP = ((H - 1) + 1) & ~1;     // halo columns staged per side
    static constexpr int LD = kTW + 2 * HLP;           // slot length (elements)
    static constexpr int S = (D + 1) * RPW + V - 1;    // slots in the ring
    static constexpr int BODY = sizeof(T) == 8 ? 1 : 2;      // body loads per row
    static constexpr int HALO_LANES = HLP * (int)sizeof(T) / 4;  // dwords per side
    static constexpr int NL = RPW * (BODY + (H > 1 ? 2 : 0));  // load instructions per chunk
    static constexpr int LDS_BYTES = S * LD * (int)sizeof(T);
};

// What a launch of the band walker covers: written columns [xa, xb) in strips
// of 128 and written rows [ya, yb) in chunks of rpw rows, `chunks` to a band.
struct BandGrid {
    int xa, xb, x00, ya, yb, strips, total, chunks, bands;
    // first column of a strip
    __host__ __device__ int x0(int strip) const
    {
        const int x = x00 + strip * kTW;
        return x < xa ? xa : (x < xb - kTW ? x : xb - kTW);
    }
};
__host__ __device__ inline BandGrid bandGrid(const StencilLaunch& a, int rpw)
{
    BandGrid g;
    g.xa = a.wx0;
    g.xb = a.wx1;
    g.ya = a.wy0 > a.yGlobal0 ? a.wy0 - a.yGlobal0 : 0;
    g.yb = a.wy1 - a.yGlobal0 < a.ny ? a.wy1 - a.yGlobal0 : a.ny;
    const int rows = g.yb - g.ya;
    // Where every row starts at a 128-byte line, strips start at multiples of
    // 128 columns, so that only the first and the last share lines with their
    // neighbours (8192 x 8192 FP64, written window from column 2 on: 5x5 194.6
    // us with strips from column 2, 177.5 so).
    const int line = a.dtype == Dtype::F64 ? 16 : 32;
    g.x00 = a.ldIn % line == 0 && a.ldOut % line == 0 ? g.xa / kTW * kTW : g.xa;
    g.strips = (g.xb - g.x00 + kTW - 1) / kTW;
    g.total = (rows + rpw - 1) / rpw;
    // fewer rows than a band: the ragged last chunk gets a band of its own,
    // which ends at the last row without starting before the first
    g.chunks = a.chunks < rows / rpw ? a.chunks : rows / rpw;
    g.bands = g.chunks > 0 ? (g.total + g.chunks - 1) / g.chunks : 0;
    return g;
}
// The walker's conditions: a full strip of written columns, a full chunk of
// written rows, and at most one wrap correction for every row it touches.
__host__ __device__ inline bool bandApplies(const StencilLaunch& a, int rpw)
{
    const BandGrid g = bandGrid(a, rpw);
    return g.xb - g.xa >= kTW && g.yb - g.ya >= rpw &&
           (!a.rows.wrap || (a.rows.rowWrap >= a.V + rpw && a.ny <= a.rows.rowWrap));
}

// Band walk of wave g of a launch (one wave per workgroup): strip
// g % strips, band g / strips.  `ring` is the wave's BandShape::S x LD LDS ring
// and `w` the H*V weights; X the point-wise transform of the values read.
// With kStreamWeights the weights come from a.weights and `w` is not read.
template <typename T, int H, int V, int RPW, Xform X = Xform::Identity>
__device__ __forceinline__ void bandWalk(const StencilLaunch& a, const T (&w)[H * V],
                                         Lds<T>* __restrict__ ring, int g)
{
    using BS = BandShape<T, H, V, RPW>;
    constexpr int D = BS::D, HLP = BS::HLP, LD = BS::LD, S = BS::S, NL = BS::NL;
    constexpr int HL = BS::HALO_LANES;

    const int lane = threadIdx.x;
    const BandGrid bg = bandGrid(a, RPW);
    const int strip = g % bg.strips, band = g / bg.strips;
    const int nChunks = min(bg.chunks, bg.total - band * bg.chunks);
    const int yS = min(bg.ya + band * bg.chunks * RPW, bg.yb - nChunks * RPW);

    const Glob<T>* __restrict__ in = globalPtr<T>(a.in);
    Glob<T>* __restrict__ out = globalPtr<T>(a.out);
    const int nx = a.nx;
    const int x0 = bg.x0(strip);
    const int L = a.L;
    const int R = H - 1 - L;
    // x-np (V == 1): the last strip's waves also write 0 to the R columns right
    // of it
    const bool zeros = V == 1 && a.zeroRight && strip == bg.strips - 1;

    // halo columns staged for this lane (lanes < HL, one dword each)
    const int hcol = sizeof(T) == 8 ? lane >> 1 : lane;
    const int hword = sizeof(T) == 8 ? lane & 1 : 0;
    int colL = x0 - HLP + hcol;
    int colR = x0 + kTW + hcol;
    if (a.xWrap) {
        if (colL < 0) colL += nx;
        if (colR >= nx) colR -= nx;
    } else {
        colL = colL < 0 ? 0 : colL;
        colR = colR >= nx ? nx - 1 : colR;
    }

    // Rows are loaded in order; syNext is the source row of the next one.
    const RowMap rows = a.rows;
    int gyNext = yS - a.T;
    int syNext = mapRowNear(rows, gyNext);
    auto loadRow = [&](int slot) {
        const Glob<T>* row = in + (int64_t)syNext * a.ldIn;
        gyNext++;
        if (rows.wrap) syNext = syNext + 1 == rows.rowWrap ? 0 : syNext + 1;
        else syNext = min(max(gyNext, rows.rowMin), rows.rowMax);
        Lds<T>* l = ring + slot * LD;
        if constexpr (sizeof(T) == 8) {
            ldsDma16<kDmaDefault>((const Glob<double>*)(row + x0 + 2 * lane),
                                  (Lds<double>*)(l + HLP));
        } else {
            ldsDma4<kDmaDefault>((const Glob<unsigned>*)(row + x0 + lane), l + HLP);
            ldsDma4<kDmaDefault>((const Glob<unsigned>*)(row + x0 + kLanes + lane),
                                 l + HLP + kLanes);
        }
        if constexpr (H > 1) {
            if (lane < HL) {
                ldsDma4<kDmaDefault>((const Glob<unsigned>*)(row + colL) + hword, l);
                ldsDma4<kDmaDefault>((const Glob<unsigned>*)(row + colR) + hword, l + HLP + kTW);
            }
        }
    };
    auto loadChunk = [&](int slot0) {
#pragma unroll
        for (int r = 0; r < RPW; r++) {
            int sl = slot0 + r;
            if (sl >= S) sl -= S;
            loadRow(sl);
        }
    };

    // Chunk c computes region rows [yS + c*RPW, +RPW) from relative input rows
    // [c*RPW, c*RPW + RPW + V - 1) (relative row 0 is yS - T), held in slots
    // (relative row) mod S.  Its loads are the rows [c*RPW + V-1, (c+1)*RPW + V-1);
    // chunk 0 also loads rows [0, V-1) first.
#pragma unroll
    for (int r = 0; r < V - 1; r++) loadRow(r);
    int slotLoad = V - 1;
    for (int c = 0; c < D; c++) {
        if (c < nChunks) loadChunk(slotLoad);
        slotLoad += RPW;
        if (slotLoad >= S) slotLoad -= S;
    }

    int slotBase = 0;
    for (int c = 0; c < nChunks; c++) {
        if (zeros) {
            waitVmcnt<0>();  // its extra stores are not in the count
        } else {
            const int la = min(c + D - 1, nChunks - 1) - c;
            const int sa = min(c, D);
            waitChunk<NL, RPW, D>(la, sa);
        }
        // chunk c + D reuses the slots of chunk c - 1's first RPW rows
        if (c + D < nChunks) loadChunk(slotLoad);
        slotLoad += RPW;
        if (slotLoad >= S) slotLoad -= S;

        T acc[RPW][2];
#pragma unroll
        for (int r = 0; r < RPW; r++) acc[r][0] = acc[r][1] = T(0);
#pragma unroll
        for (int ir = 0; ir < RPW + V - 1; ir++) {
            int sl = slotBase + ir;
            if (sl >= S) sl -= S;
            const Lds<T>* row = ring + sl * LD + (HLP - L) + 2 * lane;
            T v[H + 1];
            // Pair reads only for stencils of at most 25 points: the wider
            // ones were measured slower with a second read path in the loop.
            if (H * V <= 25 && ((HLP - L) & 1) == 0 && (H + 1) % 2 == 0) {
                // window pair-aligned: one 2-element read per pair (FP64:
                // ds_read_b128, 16 lanes x 16 B cover all banks once)
                using V2 = typename Vec2<T>::type;
                const Lds<V2>* rp = (const Lds<V2>*)row;
#pragma unroll
                for (int k = 0; k < (H + 1) / 2; k++) {
                    const V2 p = rp[k];
                    v[2 * k] = xformValue<T, X>(p.x);
                    v[2 * k + 1] = xformValue<T, X>(p.y);
                }
            } else {
#pragma unroll
                for (int k = 0; k < H + 1; k++) v[k] = xformValue<T, X>(row[k]);
            }
#pragma unroll
            for (int r = 0; r < RPW; r++) {
                const int j = ir - r;
                if (j >= 0 && j < V) {
                    T wr[H];
                    if constexpr (kStreamWeights<T, H, V>) {
                        loadWeightRow<H>(a.weights, j, wr, acc[r][1]);
                    } else {
#pragma unroll
                        for (int i = 0; i < H; i++) wr[i] = w[j * H + i];
                    }
#pragma unroll
                    for (int i = 0; i < H; i++) {
                        acc[r][0] = fmaT(wr[i], v[i], acc[r][0]);
                        acc[r][1] = fmaT(wr[i], v[i + 1], acc[r][1]);
                    }
                }
            }
        }

#pragma unroll
        for (int r = 0; r < RPW; r++) {
            const typename Vec2<T>::type v = {acc[r][0], acc[r][1]};
            Glob<T>* orow = out + (int64_t)(yS + c * RPW + r) * a.ldOut;
            __builtin_nontemporal_store(ElemVec2<T>(v),
                                        reinterpret_cast<Glob<ElemVec2<T>>*>(orow + x0 + 2 * lane));
            if (zeros && lane < R) orow[nx - R + lane] = T(0);
        }
        slotBase += RPW;
        if (slotBase >= S) slotBase -= S;
    }
}

// Single-region launch: one wave per workgroup, waves in XCD-aware order.
template <typename T, int H, int V, int RPW, Xform X = Xform::Identity>
__global__ __launch_bounds__(kLanes) void stencilBand(StencilLaunch a)
{
    using BS = BandShape<T, H, V, RPW>;
    __shared__ __attribute__((aligned(16))) T ring[BS::S * BS::LD];
    T w[H * V];
    if constexpr (!kStreamWeights<T, H, V>) {
#pragma unroll
        for (int k = 0; k < H * V; k++) w[k] = static_cast<T>(a.weights[k]);
    }
    if constexpr (kWeightsInVgprs<T, H, V>) {
        // an empty asm with a vector-register result: the compiler treats
        // the value as per-lane and keeps it there
#pragma unroll
        for (int k = 0; k < H * V; k++) {
            T o;
            __asm__ __volatile__("" : "=v"(o) : "0"(w[k]));
            w[k] = o;
        }
    }
    bandWalk<T, H, V, RPW, X>(a, w, (Lds<T>*)ring, xcdRemap(blockIdx.x, gridDim.x));
}

}  // namespace dev
}  // namespace custen
