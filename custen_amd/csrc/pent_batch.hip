// pent_batch.hip -- batched pentadiagonal factorisation and solve on
// interleaved systems (cuPentCahnADI/src/cuPentBatch.cu:35-198): element i of
// system k lives at [i * batch + k], every system has its own diagonals.
//
// One lane per system, so each row access of a wave is contiguous in every
// array.  The recurrences are sequential in the row.  Two forms:
//   factorKernel, solveKernel  many systems: a wave of 64 loads, computes and
//       stores its own rows, prefetching kPF rows in registers
//       (double-buffered); several waves per SIMD hide the rest of the latency
//       and the kernel runs at the memory's rate;
//   factorRingKernel, solveRingKernel  fewer systems than that takes: other
//       waves of the workgroup fetch the rows ahead into LDS.
// Arithmetic is the reference's, one IEEE operation at a time (contraction
// off), identical to the CPU restatement.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "../../include/custen_pent.h"
#include "lds_ring.h"
#include "plan_internal.h"
#include "short_division.h"

#pragma clang fp contract(off)

namespace custen {
namespace pentdev {

constexpr int kPF = 8;
constexpr int kBlock = 64;

// ---------------------------------------------------------------------------
// Ring kernels: SYS systems per workgroup, one per lane of wave 0, which runs
// the recurrences.  Waves 1 and 2 bring chunks of CR rows of every array the
// sweep reads from memory straight into an LDS ring, wave 3 (of a solve) adds
// the reciprocals of the pivots, and wave 0 reads a chunk ahead of the one it
// computes and stores its rows itself.
//
// With one wave doing all of it a row costs a share of the memory latency that
// few waves cannot hide (8 rows in flight, drained by the register copies of
// the double buffer): 340 ns per row of a factorisation and 260 ns of a solve
// at 4096 systems.  Here a row takes 120 and 130 ns, most of them the
// instructions wave 0 issues for it (a lone wave issues one per 4 to 5
// cycles, and a stored row costs it about 14).
// ---------------------------------------------------------------------------
constexpr int CR = 8;  // rows per chunk

using dev::kMaxDivisor;
using dev::kMinDivisor;
using dev::kMinQuotient;
using dev::Lds;
using dev::quotient;
using dev::recipOf;
typedef int i32x4 __attribute__((ext_vector_type(4)));

struct __attribute__((aligned(16))) Progress {
    int landed[2];  // chunks in LDS, by loading wave
    int recips;     // chunks whose reciprocals are in LDS
    int read;       // chunks read out of their slot
};

// The counters as wave 0 last saw them: they are read a chunk before they are
// needed, so that a wait which is already over costs no LDS round trip.
struct Seen {
    i32x4 f;
    __device__ __forceinline__ void look(const Progress& P)
    {
        __asm__ __volatile__("" ::: "memory");
        f = *reinterpret_cast<const i32x4*>(&P);
        __asm__ __volatile__("" ::: "memory");
    }
    __device__ __forceinline__ void waitLanded(const Progress& P, int v)
    {
        while (__builtin_amdgcn_readfirstlane(min(f.x, f.y)) < v) again(P);
        __asm__ __volatile__("" ::: "memory");
    }
    __device__ __forceinline__ void waitRecips(const Progress& P, int v)
    {
        while (__builtin_amdgcn_readfirstlane(f.z) < v) again(P);
        __asm__ __volatile__("" ::: "memory");
    }
    __device__ __forceinline__ void again(const Progress& P)
    {
        __builtin_amdgcn_s_sleep(1);
        look(P);
    }
};

// The chunks of a sweep over rows [lo, hi) of m-row arrays: upwards (dir > 0)
// chunk c starts at row lo + c CR; downwards it ends at row hi - 1 - c CR.
struct Sweep {
    int lo, hi, dir, m;
    __device__ __forceinline__ int chunks() const { return (hi - lo + CR - 1) / CR; }
    // first (lowest) row held by chunk c's slot
    __device__ __forceinline__ int base(int c) const
    {
        return dir > 0 ? lo + c * CR : max(hi - (c + 1) * CR, 0);
    }
};

// LDS of a workgroup: 56 rows of a solve's arrays at 64 systems (one workgroup
// per CU), 96 at 16 (two per CU).
template <int SYS>
constexpr int kRingBytes = SYS == 64 ? 140 * 1024 : 60 * 1024;

// The slots of a sweep that reads NA arrays and keeps NX more rows' worth of
// derived values per row (reciprocals).
template <int SYS, int NA, int NX>
struct Ring {
    static constexpr int ROW = SYS * 8;                   // bytes of a row of one array
    static constexpr int ARRAY = CR * ROW;                // of an array's rows in a slot
    static constexpr int SLOT = (NA + NX) * ARRAY;
    static constexpr int NB = kRingBytes<SYS> / SLOT;     // slots
};

// Waves 1 and 2 (LW = 0, 1): every other load of a chunk.  A load instruction
// takes BYTES per lane, 64 BYTES of consecutive rows of one array: 16 for
// even batches of 16-byte aligned arrays, else 4.
template <int SYS, int NA, int NX, int BYTES, int LW>
__device__ __forceinline__ void loadSweep(const double* const (&arr)[NA], const Sweep& sw,
                                          int64_t batch, int64_t k0, Lds<char>* ring, Progress& P,
                                          int lane)
{
    using RG = Ring<SYS, NA, NX>;
    constexpr int TI = RG::ARRAY / (64 * BYTES);        // loads per array and chunk
    constexpr int NL = (NA * TI - LW + 1) / 2;          // of them this wave's
    constexpr int Q = 63 / NL < RG::NB - 2 ? 63 / NL : RG::NB - 2;  // chunks in flight behind
    static_assert(Q >= 1 && RG::NB >= 3, "at least one chunk in flight");
    const int nCh = sw.chunks();
    const int last = (int)min((int64_t)(SYS - 1), batch - 1 - k0);
    const uint32_t stride = (uint32_t)batch * 8u;
    // row and byte offset in the row of this lane's part of load t; systems
    // past the last one repeat it
    uint32_t row[TI], col[TI], voff[TI];
#pragma unroll
    for (int t = 0; t < TI; t++) {
        const int e = (t * 64 + lane) * BYTES;
        row[t] = (uint32_t)(e / RG::ROW);
        const int sys = e % RG::ROW / 8;
        col[t] = BYTES == 16 ? (uint32_t)min(sys, last - 1) * 8u
                             : (uint32_t)min(sys, last) * 8u + (uint32_t)(e & 4);
        voff[t] = row[t] * stride + col[t];
    }
    int slot = 0;
    for (int c = 0; c < nCh; c++) {
        if (c >= RG::NB) dev::waitFor(P.read, c - RG::NB + 1);
        const int row0 = sw.base(c);
        const int end = sw.m - 1 - row0;  // last row of the arrays, from row0
        const bool whole = end >= CR - 1;  // else: rows past the end repeat it
#pragma unroll
        for (int q = LW; q < NA * TI; q += 2) {
            const int a = q / TI, t = q % TI;
            const __amdgpu_buffer_rsrc_t rs =
                dev::rowBuffer(arr[a] + (int64_t)row0 * batch + k0);
            const uint32_t v = whole ? voff[t] : min(row[t], (uint32_t)end) * stride + col[t];
            dev::rowDma<BYTES>(rs, ring + slot * RG::SLOT + q * 64 * BYTES, v, 0);
        }
        if (c >= Q) {
            dev::waitVmcnt<Q * NL>();
            dev::post(P.landed[LW], c - Q + 1);
        }
        if (++slot == RG::NB) slot = 0;
    }
    dev::waitVmcnt<0>();
    dev::post(P.landed[LW], nCh);
    dev::sweepBarrier();
}

template <int NA>
using Rows = double[NA][CR];

// Wave 0: the CR rows of a slot's first N arrays.
template <class RG, int N>
__device__ __forceinline__ void readChunk(double (&r)[N][CR], const Lds<char>* ring, int slot,
                                          int lane)
{
    const Lds<double>* p = (const Lds<double>*)(ring + slot * RG::SLOT) + lane;
#pragma unroll
    for (int a = 0; a < N; a++)
#pragma unroll
        for (int k = 0; k < CR; k++) r[a][k] = p[a * (RG::ARRAY / 8) + k * (RG::ROW / 8)];
}

// pentFactorBatch (cuPentBatch.cu:35-113).  LATE: a chunk's rows are stored when
// its quotients are known to be in the short division's range, and then once;
// otherwise as they are computed, and again after a chunk that left it.
template <int SYS, int BYTES, bool LATE>
__global__ __launch_bounds__(192) void factorRingKernel(double* __restrict__ ds,
                                                        double* __restrict__ dl,
                                                        double* __restrict__ d,
                                                        double* __restrict__ du,
                                                        double* __restrict__ dw, int m,
                                                        int64_t batch)
{
    __shared__ __attribute__((aligned(16))) char ringMem[kRingBytes<SYS>];
    __shared__ Progress P;
    using RG = Ring<SYS, 5, 0>;
    Lds<char>* ring = (Lds<char>*)ringMem;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t k0 = (int64_t)blockIdx.x * SYS;
    const Sweep sw{2, m, 1, m};
    if (threadIdx.x == 0) P = Progress{};
    __syncthreads();
    if (wave > 0) {
        const double* const arr[5] = {ds, dl, d, du, dw};
        if (wave == 1) loadSweep<SYS, 5, 0, BYTES, 0>(arr, sw, batch, k0, ring, P, lane);
        else loadSweep<SYS, 5, 0, BYTES, 1>(arr, sw, batch, k0, ring, P, lane);
        return;
    }
    if (lane >= SYS) return;
    // Lanes past the last system repeat it: they store the same bits.
    const int sys = (int)min((int64_t)lane, batch - 1 - k0);
    const int64_t k = k0 + sys;
    const int64_t s = batch;
    const uint32_t col8 = (uint32_t)sys * 8u, stride = (uint32_t)batch * 8u;
    // row 0
    const double d0 = d[k];
    const double du0 = du[k] / d0;
    const double dw0 = dw[k] / d0;
    // row 1
    const double dl1 = dl[k + s];
    const double d1 = d[k + s] - dl1 * du0;
    const double du1 = (du[k + s] - dl1 * dw0) / d1;
    const double dw1 = dw[k + s] / d1;
    du[k] = du0;
    dw[k] = dw0;
    d[k + s] = d1;
    du[k + s] = du1;
    dw[k + s] = dw1;
    double duPP = du0, dwPP = dw0, duP = du1, dwP = dw1;
    Seen seen;
    const int nCh = sw.chunks();
    const int nFull = max(m - 4, 0) / CR;  // chunks of interior rows (below m - 2) only

    auto compute = [&](const Rows<5>& x, int c) {
        const int64_t at = (int64_t)(2 + c * CR) * s + k0;
        const __amdgpu_buffer_rsrc_t rl = dev::rowBuffer(dl + at), rd = dev::rowBuffer(d + at),
                                     ru = dev::rowBuffer(du + at), rw = dev::rowBuffer(dw + at);
        const double duPPs = duPP, dwPPs = dwPP, duPs = duP, dwPs = dwP;
        double vl[CR], vd[CR], vu[CR], vw[CR];
        auto storeRow = [&](int j) {
            const uint32_t o = (uint32_t)j * stride;
            dev::rowStore(rl, vl[j], col8, o);
            dev::rowStore(rd, vd[j], col8, o);
            dev::rowStore(ru, vu[j], col8, o);
            dev::rowStore(rw, vw[j], col8, o);
        };
        double qmin = 0x1p900, dmin = 0x1p900, dmax = 0.0;
#pragma unroll
        for (int j = 0; j < CR; j++) {
            const double lv = x[1][j] - x[0][j] * duPP;
            const double dv = (x[2][j] - x[0][j] * dwPP) - lv * duP;
            const double y = recipOf(dv);
            const double uv = quotient(x[3][j] - lv * dwP, dv, y);
            const double wv = quotient(x[4][j], dv, y);
            qmin = __builtin_fmin(qmin, __builtin_fmin(__builtin_fabs(uv), __builtin_fabs(wv)));
            dmin = __builtin_fmin(dmin, __builtin_fabs(dv));
            dmax = __builtin_fmax(dmax, __builtin_fabs(dv));
            vl[j] = lv;
            vd[j] = dv;
            vu[j] = uv;
            vw[j] = wv;
            if constexpr (!LATE) storeRow(j);
            duPP = duP;
            dwPP = dwP;
            duP = uv;
            dwP = wv;
        }
        // out of the short division's range (zero and tiny quotients, extreme
        // pivots), or not finite: an infinity or NaN stays in the recurrence
        if (!(qmin >= kMinQuotient && dmin >= kMinDivisor && dmax <= kMaxDivisor &&
              __builtin_fabs(duP) < __builtin_inf() && __builtin_fabs(dwP) < __builtin_inf())) {
            duPP = duPPs;
            dwPP = dwPPs;
            duP = duPs;
            dwP = dwPs;
#pragma unroll
            for (int j = 0; j < CR; j++) {
                vl[j] = x[1][j] - x[0][j] * duPP;
                vd[j] = (x[2][j] - x[0][j] * dwPP) - vl[j] * duP;
                vu[j] = (x[3][j] - vl[j] * dwP) / vd[j];
                vw[j] = x[4][j] / vd[j];
                if constexpr (!LATE) storeRow(j);
                duPP = duP;
                dwPP = dwP;
                duP = vu[j];
                dwP = vw[j];
            }
        }
        if constexpr (LATE) {
#pragma unroll
            for (int j = 0; j < CR; j++) storeRow(j);
        }
    };
    Rows<5> A, B;
    int slot = 0;
    // one chunk: the next one's rows are read first, then this one's computed
    auto chunk = [&](const Rows<5>& cur, Rows<5>& next, int c) {
        if (++slot == RG::NB) slot = 0;
        if (c + 1 < nCh) {
            seen.waitLanded(P, c + 2);
            readChunk<RG>(next, ring, slot, sys);
            dev::post(P.read, c + 2);
            seen.look(P);
        }
        __builtin_amdgcn_sched_barrier(0);
        compute(cur, c);
    };
    seen.look(P);
    seen.waitLanded(P, 1);
    readChunk<RG>(A, ring, 0, sys);
    dev::post(P.read, 1);
    int c = 0;
    for (; c + 2 <= nFull; c += 2) {
        chunk(A, B, c);
        chunk(B, A, c + 1);
    }
    if (c < nFull) chunk(A, B, c++);
    // the last 2 .. CR + 1 rows, one at a time: rows up to m-2 update du,
    // interior rows also dw
    seen.waitLanded(P, nCh);
    for (int i = 2 + nFull * CR; i < m; i++) {
        const int ci = (i - 2) / CR;
        const Lds<double>* x = (const Lds<double>*)(ring + ci % RG::NB * RG::SLOT) +
                               (i - 2) % CR * SYS + sys;
        const double lv = x[CR * SYS] - x[0] * duPP;
        const double dv = (x[2 * CR * SYS] - x[0] * dwPP) - lv * duP;
        const int64_t o = (int64_t)i * s + k;
        dl[o] = lv;
        d[o] = dv;
        double uv = 0.0, wv = x[4 * CR * SYS];
        if (i < m - 1) {
            uv = (x[3 * CR * SYS] - lv * dwP) / dv;
            du[o] = uv;
        }
        if (i < m - 2) {
            wv = wv / dv;
            dw[o] = wv;
        }
        duPP = duP;
        dwPP = dwP;
        duP = uv;
        dwP = wv;
    }
    dev::sweepBarrier();
}

// pentSolveBatch (cuPentBatch.cu:119-198)
template <int SYS, int BYTES>
__global__ __launch_bounds__(256) void solveRingKernel(const double* __restrict__ ds,
                                                       const double* __restrict__ dl,
                                                       const double* __restrict__ d,
                                                       const double* __restrict__ du,
                                                       const double* __restrict__ dw,
                                                       double* __restrict__ b, int m,
                                                       int64_t batch)
{
    __shared__ __attribute__((aligned(16))) char ringMem[kRingBytes<SYS>];
    __shared__ Progress P[2];
    using RF = Ring<SYS, 4, 1>;  // ds, dl, d, b and 1/d
    using RB = Ring<SYS, 3, 0>;  // du, dw, b
    Lds<char>* ring = (Lds<char>*)ringMem;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t k0 = (int64_t)blockIdx.x * SYS;
    const Sweep fw{2, m, 1, m}, bw{0, m - 2, -1, m};
    if (threadIdx.x == 0) P[0] = P[1] = Progress{};
    __syncthreads();
    if (wave == 1 || wave == 2) {
        const double* const af[4] = {ds, dl, d, b};
        const double* const ab[3] = {du, dw, b};
        if (wave == 1) {
            loadSweep<SYS, 4, 1, BYTES, 0>(af, fw, batch, k0, ring, P[0], lane);
            loadSweep<SYS, 3, 0, BYTES, 0>(ab, bw, batch, k0, ring, P[1], lane);
        } else {
            loadSweep<SYS, 4, 1, BYTES, 1>(af, fw, batch, k0, ring, P[0], lane);
            loadSweep<SYS, 3, 0, BYTES, 1>(ab, bw, batch, k0, ring, P[1], lane);
        }
        return;
    }
    Seen seen;
    const int nF = fw.chunks(), nB = bw.chunks();
    if (wave == 3) {
        // reciprocals of the pivots (0: out of the short division's range)
        int slot = 0;
        for (int c = 0; c < nF; c++) {
            seen.look(P[0]);
            seen.waitLanded(P[0], c + 1);
            Lds<double>* x = (Lds<double>*)(ring + slot * RF::SLOT) + min(lane, SYS - 1);
            double v[CR];
#pragma unroll
            for (int j = 0; j < CR; j++) v[j] = x[(2 * CR + j) * SYS];
#pragma unroll
            for (int j = 0; j < CR; j++) {
                const double a = __builtin_fabs(v[j]);
                x[(4 * CR + j) * SYS] =
                    a >= kMinDivisor && a <= kMaxDivisor ? recipOf(v[j]) : 0.0;
            }
            dev::post(P[0].recips, c + 1);
            if (++slot == RF::NB) slot = 0;
        }
        dev::sweepBarrier();
        dev::sweepBarrier();
        return;
    }
    if (lane >= SYS) return;
    // Lanes past the last system repeat it: they store the same bits.
    const int sys = (int)min((int64_t)lane, batch - 1 - k0);
    const int64_t k = k0 + sys;
    const int64_t s = batch;
    const uint32_t col8 = (uint32_t)sys * 8u, stride = (uint32_t)batch * 8u;

    // forward substitution
    double b2 = b[k] / d[k];
    double b1 = (b[k + s] - dl[k + s] * b2) / d[k + s];
    b[k] = b2;
    b[k + s] = b1;
    {
        const int nFull = (m - 2) / CR;
        auto compute = [&](const Rows<5>& x, int c) {
            const __amdgpu_buffer_rsrc_t rb =
                dev::rowBuffer(b + (int64_t)(2 + c * CR) * s + k0);
            const double b2s = b2, b1s = b1;
            double qmin = 0x1p900;
#pragma unroll
            for (int j = 0; j < CR; j++) {
                const double num = (x[3][j] - x[0][j] * b2) - x[1][j] * b1;
                const double v = quotient(num, x[2][j], x[4][j]);
                qmin = __builtin_fmin(qmin, __builtin_fabs(v));
                dev::rowStore(rb, v, col8, (uint32_t)j * stride);
                b2 = b1;
                b1 = v;
            }
            // a zero or tiny quotient, a pivot without a reciprocal (its
            // quotient is 0), or not finite: these rows again, with IEEE
            // division
            if (!(qmin >= kMinQuotient && __builtin_fabs(b1) < __builtin_inf())) {
                b2 = b2s;
                b1 = b1s;
#pragma unroll
                for (int j = 0; j < CR; j++) {
                    const double v = ((x[3][j] - x[0][j] * b2) - x[1][j] * b1) / x[2][j];
                    dev::rowStore(rb, v, col8, (uint32_t)j * stride);
                    b2 = b1;
                    b1 = v;
                }
            }
        };
        Rows<5> A, B;
        int slot = 0;
        auto chunk = [&](const Rows<5>& cur, Rows<5>& next, int c) {
            if (++slot == RF::NB) slot = 0;
            if (c + 1 < nF) {
                seen.waitRecips(P[0], c + 2);
                readChunk<RF>(next, ring, slot, sys);
                dev::post(P[0].read, c + 2);
                seen.look(P[0]);
            }
            __builtin_amdgcn_sched_barrier(0);
            compute(cur, c);
        };
        seen.look(P[0]);
        seen.waitRecips(P[0], 1);
        readChunk<RF>(A, ring, 0, sys);
        dev::post(P[0].read, 1);
        int c = 0;
        for (; c + 2 <= nFull; c += 2) {
            chunk(A, B, c);
            chunk(B, A, c + 1);
        }
        if (c < nFull) chunk(A, B, c++);
        seen.waitRecips(P[0], nF);
        const Lds<double>* x = (const Lds<double>*)(ring + c % RF::NB * RF::SLOT) + sys;
        for (int j = 0; 2 + c * CR + j < m; j++, x += SYS) {
            const double v = ((x[3 * CR * SYS] - x[0] * b2) - x[CR * SYS] * b1) /
                             x[2 * CR * SYS];
            b[(int64_t)(2 + c * CR + j) * s + k] = v;
            b2 = b1;
            b1 = v;
        }
    }
    dev::sweepBarrier();

    // backward substitution: x[m-1] = b1, x[m-2] = b2 - du[m-2] x[m-1]
    double a1 = b1;
    double a0 = b2 - du[(int64_t)(m - 2) * s + k] * a1;
    b[(int64_t)(m - 2) * s + k] = a0;
    {
        const int nFull = (m - 2) / CR;
        auto compute = [&](const Rows<3>& x, int c) {
            const __amdgpu_buffer_rsrc_t rb = dev::rowBuffer(b + (int64_t)bw.base(c) * s + k0);
#pragma unroll
            for (int j = CR - 1; j >= 0; j--) {
                const double v = (x[2][j] - x[0][j] * a0) - x[1][j] * a1;
                dev::rowStore(rb, v, col8, (uint32_t)j * stride);
                a1 = a0;
                a0 = v;
            }
        };
        Rows<3> A, B;
        int slot = 0;
        auto chunk = [&](const Rows<3>& cur, Rows<3>& next, int c) {
            if (++slot == RB::NB) slot = 0;
            if (c + 1 < nB) {
                seen.waitLanded(P[1], c + 2);
                readChunk<RB>(next, ring, slot, sys);
                dev::post(P[1].read, c + 2);
                seen.look(P[1]);
            }
            __builtin_amdgcn_sched_barrier(0);
            compute(cur, c);
        };
        seen.look(P[1]);
        seen.waitLanded(P[1], 1);
        readChunk<RB>(A, ring, 0, sys);
        dev::post(P[1].read, 1);
        int c = 0;
        for (; c + 2 <= nFull; c += 2) {
            chunk(A, B, c);
            chunk(B, A, c + 1);
        }
        if (c < nFull) chunk(A, B, c++);
        seen.waitLanded(P[1], nB);
        const int rest = (m - 2) % CR;  // rows rest-1 .. 0, from row 0 of their slot
        const Lds<double>* x = (const Lds<double>*)(ring + c % RB::NB * RB::SLOT) + sys;
        for (int j = rest - 1; j >= 0; j--) {
            const double v = (x[(2 * CR + j) * SYS] - x[j * SYS] * a0) -
                             x[(CR + j) * SYS] * a1;
            b[(int64_t)j * s + k] = v;
            a1 = a0;
            a0 = v;
        }
    }
    dev::sweepBarrier();
}

// pentFactorBatch (cuPentBatch.cu:35-113)
__global__ __launch_bounds__(kBlock) void factorKernel(double* __restrict__ ds,
                                                       double* __restrict__ dl,
                                                       double* __restrict__ d,
                                                       double* __restrict__ du,
                                                       double* __restrict__ dw, int m,
                                                       int64_t batch)
{
    const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (k >= batch) return;
    ds += k;
    dl += k;
    d += k;
    du += k;
    dw += k;
    const int64_t s = batch;
    // row 0
    const double d0 = d[0];
    const double du0 = du[0] / d0;
    const double dw0 = dw[0] / d0;
    du[0] = du0;
    dw[0] = dw0;
    // row 1
    const double dl1 = dl[s];
    const double d1 = d[s] - dl1 * du0;
    const double du1 = (du[s] - dl1 * dw0) / d1;
    const double dw1 = dw[s] / d1;
    d[s] = d1;
    du[s] = du1;
    dw[s] = dw1;
    double duPP = du0, dwPP = dw0, duP = du1, dwP = dw1;

    double cs[kPF], cl[kPF], cd[kPF], cu[kPF], cw[kPF];
    double ns[kPF], nl[kPF], nd[kPF], nu[kPF], nw[kPF];
#pragma unroll
    for (int j = 0; j < kPF; j++) {
        const int i = 2 + j;
        if (i < m) {
            const int64_t o = (int64_t)i * s;
            cs[j] = ds[o];
            cl[j] = dl[o];
            cd[j] = d[o];
            cu[j] = du[o];
            cw[j] = dw[o];
        }
    }
    for (int i0 = 2; i0 < m; i0 += kPF) {
#pragma unroll
        for (int j = 0; j < kPF; j++) {
            const int i = i0 + kPF + j;
            if (i < m) {
                const int64_t o = (int64_t)i * s;
                ns[j] = ds[o];
                nl[j] = dl[o];
                nd[j] = d[o];
                nu[j] = du[o];
                nw[j] = dw[o];
            }
        }
#pragma unroll
        for (int j = 0; j < kPF; j++) {
            const int i = i0 + j;
            if (i < m) {
                const int64_t o = (int64_t)i * s;
                const double lv = cl[j] - cs[j] * duPP;
                const double dv = (cd[j] - cs[j] * dwPP) - lv * duP;
                dl[o] = lv;
                d[o] = dv;
                double uv = 0.0, wv = cw[j];
                if (i < m - 1) {  // rows up to m-2 update du
                    uv = (cu[j] - lv * dwP) / dv;
                    du[o] = uv;
                }
                if (i < m - 2) {  // interior rows also update dw
                    wv = cw[j] / dv;
                    dw[o] = wv;
                }
                duPP = duP;
                dwPP = dwP;
                duP = uv;
                dwP = wv;
            }
        }
#pragma unroll
        for (int j = 0; j < kPF; j++) {
            cs[j] = ns[j];
            cl[j] = nl[j];
            cd[j] = nd[j];
            cu[j] = nu[j];
            cw[j] = nw[j];
        }
    }
}

// pentSolveBatch (cuPentBatch.cu:119-198)
__global__ __launch_bounds__(kBlock) void solveKernel(const double* __restrict__ ds,
                                                      const double* __restrict__ dl,
                                                      const double* __restrict__ d,
                                                      const double* __restrict__ du,
                                                      const double* __restrict__ dw,
                                                      double* __restrict__ b, int m, int64_t batch)
{
    const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (k >= batch) return;
    ds += k;
    dl += k;
    d += k;
    du += k;
    dw += k;
    b += k;
    const int64_t s = batch;

    // forward substitution
    double b2 = b[0] / d[0];
    b[0] = b2;
    double b1 = (b[s] - dl[s] * b2) / d[s];
    b[s] = b1;
    double cs[kPF], cl[kPF], cd[kPF], cb[kPF];
    double ns[kPF], nl[kPF], nd[kPF], nb[kPF];
#pragma unroll
    for (int j = 0; j < kPF; j++) {
        const int i = 2 + j;
        if (i < m) {
            const int64_t o = (int64_t)i * s;
            cs[j] = ds[o];
            cl[j] = dl[o];
            cd[j] = d[o];
            cb[j] = b[o];
        }
    }
    for (int i0 = 2; i0 < m; i0 += kPF) {
#pragma unroll
        for (int j = 0; j < kPF; j++) {
            const int i = i0 + kPF + j;
            if (i < m) {
                const int64_t o = (int64_t)i * s;
                ns[j] = ds[o];
                nl[j] = dl[o];
                nd[j] = d[o];
                nb[j] = b[o];
            }
        }
#pragma unroll
        for (int j = 0; j < kPF; j++) {
            const int i = i0 + j;
            if (i < m) {
                const double v = ((cb[j] - cs[j] * b2) - cl[j] * b1) / cd[j];
                b[(int64_t)i * s] = v;
                b2 = b1;
                b1 = v;
            }
        }
#pragma unroll
        for (int j = 0; j < kPF; j++) {
            cs[j] = ns[j];
            cl[j] = nl[j];
            cd[j] = nd[j];
            cb[j] = nb[j];
        }
    }

    // backward substitution: x[m-1] = b1, x[m-2] = b2 - du[m-2] x[m-1]
    double a1 = b1;
    double a0 = b2 - du[(int64_t)(m - 2) * s] * a1;
    b[(int64_t)(m - 2) * s] = a0;
    double cuu[kPF], cww[kPF], nuu[kPF], nww[kPF];
#pragma unroll
    for (int j = 0; j < kPF; j++) {
        const int i = m - 3 - j;
        if (i >= 0) {
            const int64_t o = (int64_t)i * s;
            cuu[j] = du[o];
            cww[j] = dw[o];
            cb[j] = b[o];
        }
    }
    for (int i0 = m - 3; i0 >= 0; i0 -= kPF) {
#pragma unroll
        for (int j = 0; j < kPF; j++) {
            const int i = i0 - kPF - j;
            if (i >= 0) {
                const int64_t o = (int64_t)i * s;
                nuu[j] = du[o];
                nww[j] = dw[o];
                nb[j] = b[o];
            }
        }
#pragma unroll
        for (int j = 0; j < kPF; j++) {
            const int i = i0 - j;
            if (i >= 0) {
                const double v = (cb[j] - cuu[j] * a0) - cww[j] * a1;
                b[(int64_t)i * s] = v;
                a1 = a0;
                a0 = v;
            }
        }
#pragma unroll
        for (int j = 0; j < kPF; j++) {
            cuu[j] = nuu[j];
            cww[j] = nww[j];
            cb[j] = nb[j];
        }
    }
}

}  // namespace pentdev

namespace {

int check(const char* fn, const void* const* ptrs, int nptr, int m, int batchCount)
{
    if (m < 4) {
        setError(CUSTEN_ERROR_INVALID_VALUE, std::string(fn) + ": m must be >= 4");
        return CUSTEN_ERROR_INVALID_VALUE;
    }
    if (batchCount < 1) {
        setError(CUSTEN_ERROR_INVALID_VALUE, std::string(fn) + ": batchCount must be >= 1");
        return CUSTEN_ERROR_INVALID_VALUE;
    }
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        setHipError(e, fn);
        return lastError();
    }
    for (int i = 0; i < nptr; i++) {
        if (ptrs[i] == nullptr) {
            setError(CUSTEN_ERROR_INVALID_VALUE, std::string(fn) + ": null array");
            return CUSTEN_ERROR_INVALID_VALUE;
        }
        if (classify(ptrs[i], dev) != MemKind::Device) {
            setError(CUSTEN_ERROR_INVALID_VALUE,
                     std::string(fn) + ": arrays must be device memory of the current device");
            return CUSTEN_ERROR_INVALID_VALUE;
        }
    }
    return CUSTEN_SUCCESS;
}

// Where the ring kernels are the faster ones (us at 1022 rows, one-wave kernel
// -> ring kernel): a factorisation of 4096 systems 342 -> 120, 16384 398 ->
// 213, 32768 520 -> 443, 40960 638 -> 618; a solve of 4096 262 -> 131, 16384 358
// -> 244, 20480 431 -> 432, 32768 476 -> 504.  Above the limits the one-wave
// kernel has several waves on every SIMD and runs at the memory's rate, while the
// ring kernel has one workgroup on a CU, and short systems lose in its third
// round (factorisation of 40960: 32 rows 22.3 -> 27.9, 64 rows 39.5 -> 44.7).
constexpr int kFactorRingMax = 32768;
// Rows stored late cost nothing (4096 systems 122 -> 120 us, 24576 389 -> 388) and
// spare a chunk with a zero quotient its second stores (a zero above the diagonal
// in every third row, us: 24576 systems 538 -> 412, where the one-wave kernel
// takes 501), but where rows are not 16-byte aligned and workgroups few, the
// burst of stores is waited for (898 rows, 245 systems 102.8 -> 108.0, 4095
// 107.3 -> 109.5, 8191 164.9 -> 162.7).
constexpr int kFactorEarlyMax = 4096;
constexpr int kSolveRingMax = 16384;
// A solve of few systems takes 16 per workgroup, so that four times as many CUs
// fetch (their outstanding loads are what a CU's share of a sweep waits for):
// 4096 systems 142 -> 131 us, 1023 168 -> 132; 8192 as fast either way, 12288
// 112 -> 172.  A factorisation issues more per row and gains nothing.
constexpr int kSolve16Max = 8192;

unsigned blocksOf(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

// 16-byte loads: rows 16-byte aligned in every array.
bool wideRows(const void* const* ptrs, int nptr, int batchCount)
{
    bool ok = batchCount % 2 == 0;
    for (int i = 0; i < nptr; i++) ok = ok && reinterpret_cast<uintptr_t>(ptrs[i]) % 16 == 0;
    return ok;
}

}  // namespace
}  // namespace custen

using namespace custen;

extern "C" int custenPentFactorBatch(double* ds, double* dl, double* d, double* du, double* dw,
                                     int m, int batchCount, hipStream_t stream)
{
    const void* ptrs[] = {ds, dl, d, du, dw};
    int rc = check("custenPentFactorBatch", ptrs, 5, m, batchCount);
    if (rc != CUSTEN_SUCCESS) return rc;
    const int64_t n = batchCount;
    if (batchCount > kFactorRingMax)
        hipLaunchKernelGGL(pentdev::factorKernel, dim3(blocksOf(n, pentdev::kBlock)),
                           dim3(pentdev::kBlock), 0, stream, ds, dl, d, du, dw, m, n);
    else if (wideRows(ptrs, 5, batchCount))
        hipLaunchKernelGGL((pentdev::factorRingKernel<64, 16, true>), dim3(blocksOf(n, 64)),
                           dim3(192), 0, stream, ds, dl, d, du, dw, m, n);
    else if (batchCount > kFactorEarlyMax)
        hipLaunchKernelGGL((pentdev::factorRingKernel<64, 4, true>), dim3(blocksOf(n, 64)),
                           dim3(192), 0, stream, ds, dl, d, du, dw, m, n);
    else
        hipLaunchKernelGGL((pentdev::factorRingKernel<64, 4, false>), dim3(blocksOf(n, 64)),
                           dim3(192), 0, stream, ds, dl, d, du, dw, m, n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        setHipError(e, "custenPentFactorBatch");
        return lastError();
    }
    return CUSTEN_SUCCESS;
}

extern "C" int custenPentSolveBatch(const double* ds, const double* dl, const double* d,
                                    const double* du, const double* dw, double* b, int m,
                                    int batchCount, hipStream_t stream)
{
    const void* ptrs[] = {ds, dl, d, du, dw, b};
    int rc = check("custenPentSolveBatch", ptrs, 6, m, batchCount);
    if (rc != CUSTEN_SUCCESS) return rc;
    const int64_t n = batchCount;
    const bool wide = wideRows(ptrs, 6, batchCount);
    if (batchCount > kSolveRingMax)
        hipLaunchKernelGGL(pentdev::solveKernel, dim3(blocksOf(n, pentdev::kBlock)),
                           dim3(pentdev::kBlock), 0, stream, ds, dl, d, du, dw, b, m, n);
    else if (batchCount > kSolve16Max && wide)
        hipLaunchKernelGGL((pentdev::solveRingKernel<64, 16>), dim3(blocksOf(n, 64)), dim3(256), 0,
                           stream, ds, dl, d, du, dw, b, m, n);
    else if (batchCount > kSolve16Max)
        hipLaunchKernelGGL((pentdev::solveRingKernel<64, 4>), dim3(blocksOf(n, 64)), dim3(256), 0,
                           stream, ds, dl, d, du, dw, b, m, n);
    else if (wide)
        hipLaunchKernelGGL((pentdev::solveRingKernel<16, 16>), dim3(blocksOf(n, 16)), dim3(256), 0,
                           stream, ds, dl, d, du, dw, b, m, n);
    else
        hipLaunchKernelGGL((pentdev::solveRingKernel<16, 4>), dim3(blocksOf(n, 16)), dim3(256), 0,
                           stream, ds, dl, d, du, dw, b, m, n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        setHipError(e, "custenPentSolveBatch");
        return lastError();
    }
    return CUSTEN_SUCCESS;
}
