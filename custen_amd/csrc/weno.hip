// weno.hip -- fifth-order WENO upwind advection, periodic in x and y:
// out = u * Fx + v * Fy (cuSten/src/kernels/2d_xyADVWENO_p_kernel.cu:51-401).
//
// One workgroup of 256 threads covers a 64-column x 4*RPW-row tile.  It stages
// the scaled differences of the advected field in LDS, in x and in y, with the
// halo that either sign of the velocity needs, so each is taken once; a lane
// then evaluates its column for RPW rows.  The upwind choice is a lane's address
// and stride in LDS (the negative side reads the same differences from the other
// end), so both signs run the same code with no selection of operands.
//
// The kernel is bound by its vector instructions, so the flux is written for
// their number: products by powers of two go into the addition that follows
// them, and divisions run without the scaling and special cases of IEEE
// division, which the range of the denominators makes needless.  A tile that
// staged a difference outside that range (kWenoWide) evaluates its points
// operation by operation instead: 4096 x 4096 with 1 % of the points at 1e9,
// 185 us, where evaluating a row again after the short forms had left their range
// took 335 and IEEE divisions throughout 242.
// Those two forms and the reference's source order with IEEE divisions have the
// same bits (each shortened step is argued below), so results are bit-identical
// to the CPU restatement.  Contraction is off; the optional single-precision
// squares round to float, square in float and widen, as powf does on the
// reference's double arguments.  4096 x 4096, single-precision squares: 144 us,
// the vector unit busy 92 % of the time with 252 instructions a point (memory
// alone would take 88 at the copy rate); with differences and selections per lane
// and IEEE divisions it took 192.
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "lds_ring.h"  // row buffers
#include "short_division.h"
#include "stencil_tile.h"

#pragma clang fp contract(off)

namespace custen {
namespace dev {

constexpr int kWenoTW = 64;            // columns per tile (one per lane)
constexpr int kWenoLX = kWenoTW + 6;   // LDS row of x differences (69 in use)

template <bool SS>
__device__ __forceinline__ double wenoSq(double d)
{
    if constexpr (SS) {
        const float f = static_cast<float>(d);
        const float f2 = f * f;
        return static_cast<double>(f2);
    } else {
        return d * d;
    }
}

// wenoSten (2d_xyADVWENO_p_kernel.cu:51-86), same operation order.
template <bool SS>
__device__ __forceinline__ double wenoFlux(double v1, double v2, double v3, double v4, double v5)
{
    const double phi1 = ((1.0 / 3.0) * v1 - (7.0 / 6.0) * v2) + (11.0 / 6.0) * v3;
    const double phi2 = (-(1.0 / 6.0) * v2 + (5.0 / 6.0) * v3) + (1.0 / 3.0) * v4;
    const double phi3 = ((1.0 / 3.0) * v3 + (5.0 / 6.0) * v4) - (1.0 / 6.0) * v5;
    const double s1 = (13.0 / 12.0) * wenoSq<SS>((v1 - 2.0 * v2) + v3) +
                      0.25 * wenoSq<SS>((v1 - 4.0 * v2) + 3.0 * v3);
    const double s2 = (13.0 / 12.0) * wenoSq<SS>((v2 - 2.0 * v3) + v4) + 0.25 * wenoSq<SS>(v2 - v4);
    const double s3 = (13.0 / 12.0) * wenoSq<SS>((v3 - 2.0 * v4) + v5) +
                      0.25 * wenoSq<SS>((3.0 * v3 - 4.0 * v4) + v5);
    const double a1 = 0.1 / wenoSq<SS>(s1 + 1e-06);
    const double a2 = 0.6 / wenoSq<SS>(s2 + 1e-06);
    const double a3 = 0.3 / wenoSq<SS>(s3 + 1e-06);
    const double denom = 1.0 / ((a1 + a2) + a3);
    const double w1 = a1 * denom, w2 = a2 * denom, w3 = a3 * denom;
    return (phi1 * w1 + phi2 * w2) + phi3 * w3;
}

// n / d with the bits of IEEE division, for a positive normal float d that is
// 2^125 at most, widened: the reciprocal has 44 good bits after one Newton step
// from the float estimate, the remainder of the quotient is exact (24 by 53
// bits), and the quotient's last correction leaves an error of 2^-88, where no
// quotient by a 24-bit divisor lies within 2^-78 of a rounding boundary.
__device__ __forceinline__ double quotientF(double n, float d)
{
    const double w = static_cast<double>(d);
    double y = static_cast<double>(__builtin_amdgcn_rcpf(d));
    y = __builtin_fma(y, __builtin_fma(-w, y, 1.0), y);
    const double q = n * y;
    return __builtin_fma(__builtin_fma(-w, q, n), y, q);
}
// Differences below 2^28 (2^92 where the squares are double) stay in the range of
// wenoFluxFast: a sum of squares is below 33.4 of their squares, so its own square
// is below 2^123 (2^380).
template <bool SS>
constexpr uint32_t kWenoWide = SS ? 0x41b00000u : 0x45b00000u;  // their high words
__device__ __forceinline__ uint32_t magnitude(double d)
{
    return (uint32_t)(__builtin_bit_cast(uint64_t, d) >> 32) & 0x7fffffffu;
}

// wenoFlux with the same bits for differences below kWenoWide.
// - x - 2 y and x - 4 y as one fma: the product is exact.
// - s + 0.25 b as one fma: the product is exact unless it is subnormal, and 1e-6
//   is added to the sum.
// - the squares that divide are 1e-12 at least; the sum of the quotients is then
//   within the range of the reciprocal's steps.
template <bool SS>
__device__ __forceinline__ double wenoFluxFast(double v1, double v2, double v3, double v4,
                                               double v5)
{
    const double phi1 = ((1.0 / 3.0) * v1 - (7.0 / 6.0) * v2) + (11.0 / 6.0) * v3;
    const double phi2 = (-(1.0 / 6.0) * v2 + (5.0 / 6.0) * v3) + (1.0 / 3.0) * v4;
    const double phi3 = ((1.0 / 3.0) * v3 + (5.0 / 6.0) * v4) - (1.0 / 6.0) * v5;
    const double v33 = 3.0 * v3;
    const double s1 = __builtin_fma(0.25, wenoSq<SS>(__builtin_fma(-4.0, v2, v1) + v33),
                                    (13.0 / 12.0) * wenoSq<SS>(__builtin_fma(-2.0, v2, v1) + v3));
    const double s2 = __builtin_fma(0.25, wenoSq<SS>(v2 - v4),
                                    (13.0 / 12.0) * wenoSq<SS>(__builtin_fma(-2.0, v3, v2) + v4));
    const double s3 = __builtin_fma(0.25, wenoSq<SS>(__builtin_fma(-4.0, v4, v33) + v5),
                                    (13.0 / 12.0) * wenoSq<SS>(__builtin_fma(-2.0, v4, v3) + v5));
    double a1, a2, a3;
    if constexpr (SS) {
        const float f1 = static_cast<float>(s1 + 1e-06), f2 = static_cast<float>(s2 + 1e-06),
                    f3 = static_cast<float>(s3 + 1e-06);
        a1 = quotientF(0.1, f1 * f1);
        a2 = quotientF(0.6, f2 * f2);
        a3 = quotientF(0.3, f3 * f3);
    } else {
        const double f1 = s1 + 1e-06, f2 = s2 + 1e-06, f3 = s3 + 1e-06;
        const double g1 = f1 * f1, g2 = f2 * f2, g3 = f3 * f3;
        a1 = quotient(0.1, g1, recipOf(g1));
        a2 = quotient(0.6, g2, recipOf(g2));
        a3 = quotient(0.3, g3, recipOf(g3));
    }
    const double sum = (a1 + a2) + a3;
    const double y = recipOf(sum);
    const double denom = __builtin_fma(__builtin_fma(-sum, y, 1.0), y, y);
    const double w1 = a1 * denom, w2 = a2 * denom, w3 = a3 * denom;
    return (phi1 * w1 + phi2 * w2) + phi3 * w3;
}

template <int RPW, bool SS>
__global__ __launch_bounds__(kThreads) void wenoKernel(WenoLaunch a, int tilesX,
                                                         uint32_t tilesInv)
{
    constexpr int TH = kWaves * RPW;
    // x differences: row r, column j is (q(x0 - 2 + j) - q(x0 - 3 + j)) / dx;
    // y differences: row r is (q(y0 - 2 + r) - q(y0 - 3 + r)) / dy
    __shared__ double diffX[TH * kWenoLX];
    __shared__ double diffY[(TH + 5) * kWenoTW];
    __shared__ int wideWave[kWaves];  // the wave staged a difference that is kWenoWide or more

    const int g = xcdRemap(blockIdx.x, gridDim.x);
    // g / tilesX from the rounded-down reciprocal, at most one too small
    int tileY = (int)(((uint64_t)(uint32_t)g * tilesInv) >> 32);
    if (g - tileY * tilesX >= tilesX) tileY++;
    const int x0 = (g - tileY * tilesX) * kWenoTW;
    const int y0 = tileY * TH;
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);

    // Every load of a wave's share is issued before the first is waited for, and
    // so are its velocities.  Rows of a tile inside the grid are buffers with
    // their bases in scalar registers: no address arithmetic on the vector unit.
    constexpr int PER = (TH + 5 + kWaves - 1) / kWaves;
    const int rBegin = wave * PER, yBegin = y0 + wave * RPW;
    double q[PER + 1], qa[RPW], qb[RPW], ta, tb, uv[RPW], vv[RPW];
    auto row = [&](int y) { return a.in + (int64_t)mapRow(a.rows, y) * a.ldIn; };
    // the last five x differences of the wave's rows: a lane for each
    const int tr = min(lane / 5, RPW - 1), tc = lane - 5 * (lane / 5);
    if (x0 >= 3 && x0 + kWenoTW + 3 <= a.nx) {
        const uint32_t off = lane * 8u;
#pragma unroll
        for (int k = 0; k <= PER; k++)
            q[k] = rowLoad(rowBuffer(row(y0 - 3 + rBegin + k) + x0), off);
#pragma unroll
        for (int k = 0; k < RPW; k++) {
            const __amdgpu_buffer_rsrc_t rs = rowBuffer(row(yBegin + k) + x0 - 3);
            qa[k] = rowLoad(rs, off + 8);
            qb[k] = rowLoad(rs, off);
        }
    } else {
        const int64_t xc = wrapIndex(x0 + lane, a.nx);
        const int64_t xa = wrapIndex(x0 - 2 + lane, a.nx), xb = wrapIndex(x0 - 3 + lane, a.nx);
#pragma unroll
        for (int k = 0; k <= PER; k++) q[k] = row(y0 - 3 + rBegin + k)[xc];
#pragma unroll
        for (int k = 0; k < RPW; k++) {
            qa[k] = row(yBegin + k)[xa];
            qb[k] = row(yBegin + k)[xb];
        }
    }
    {
        const double* last = row(yBegin + tr);
        ta = last[wrapIndex(x0 + kWenoTW - 2 + tc, a.nx)];
        tb = last[wrapIndex(x0 + kWenoTW - 3 + tc, a.nx)];
    }
    const uint32_t here = (uint32_t)min(lane, a.nx - 1 - x0) * 8u;
#pragma unroll
    for (int k = 0; k < RPW; k++) {
        const int64_t at = (int64_t)min(yBegin + k, a.ny - 1) * a.ldSide + x0;
        uv[k] = rowLoad(rowBuffer(a.u + at), here);
        vv[k] = rowLoad(rowBuffer(a.v + at), here);
    }
    uint32_t most = 0;
    auto stage = [&](double* at, double d) {
        *at = d;
        most = max(most, magnitude(d));
    };
#pragma unroll
    for (int k = 0; k < PER; k++)
        if (rBegin + k < TH + 5)
            stage(diffY + (rBegin + k) * kWenoTW + lane, (q[k + 1] - q[k]) * a.coeDy);
#pragma unroll
    for (int k = 0; k < RPW; k++)
        stage(diffX + (wave * RPW + k) * kWenoLX + lane, (qa[k] - qb[k]) * a.coeDx);
    if (lane < 5 * RPW)
        stage(diffX + (wave * RPW + tr) * kWenoLX + kWenoTW + tc, (ta - tb) * a.coeDx);
    wideWave[wave] = __ballot(most >= kWenoWide<SS>) != 0;
    __syncthreads();
    int wide = 0;
#pragma unroll
    for (int k = 0; k < kWaves; k++) wide |= wideWave[k];
    wide = __builtin_amdgcn_readfirstlane(wide);

    const int x = x0 + lane;
    if (x >= a.nx) return;
    auto rows = [&](auto flux) {
#pragma unroll
        for (int r = 0; r < RPW; r++) {
            const int ly = wave * RPW + r;
            const int y = y0 + ly;
            if (y >= a.ny) break;
            // the middle one of the five differences, and the way to the others
            const bool px = uv[r] > 0.0, py = vv[r] > 0.0;
            const double* mx = diffX + ly * kWenoLX + lane + (px ? 2 : 3);
            const double* my = diffY + (ly + (py ? 2 : 3)) * kWenoTW + lane;
            const int sx = px ? 1 : -1, sy = py ? kWenoTW : -kWenoTW;
            const double fx = flux(mx[-2 * sx], mx[-sx], mx[0], mx[sx], mx[2 * sx]);
            const double fy = flux(my[-2 * sy], my[-sy], my[0], my[sy], my[2 * sy]);
            __builtin_nontemporal_store(uv[r] * fx + vv[r] * fy,
                                        a.out + (int64_t)y * a.ldOut + x);
        }
    };
    if (__builtin_expect(wide, 0)) {
        rows([](double v1, double v2, double v3, double v4, double v5) {
            return wenoFlux<SS>(v1, v2, v3, v4, v5);
        });
    } else {
        rows([](double v1, double v2, double v3, double v4, double v5) {
            return wenoFluxFast<SS>(v1, v2, v3, v4, v5);
        });
    }
}

template <int RPW>
hipError_t launchWenoRpw(const WenoLaunch& w, hipStream_t st)
{
    constexpr int TH = kWaves * RPW;
    const int64_t tilesX = (w.nx + kWenoTW - 1) / kWenoTW;
    const int64_t tiles = tilesX * ((w.ny + TH - 1) / TH);
    if (tiles > 0x7fffffff) return hipErrorInvalidValue;
    // (2^32 - 1) / tilesX: also fits where tilesX is 1
    const uint32_t inv = 0xffffffffu / (uint32_t)tilesX;
    auto* kernel = w.singleSquares ? wenoKernel<RPW, true> : wenoKernel<RPW, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(kThreads), 0, st, w, (int)tilesX, inv);
    return hipGetLastError();
}

}  // namespace dev

// 4 rows per wave unless 8 is asked for: the same time at 4096 x 4096 (147 and
// 146 us) and less where there are few tiles (300 x 500: 6.5 and 10.0 us).
int wenoLdsBytes(int rowsPerWave)
{
    const int rpw = rowsPerWave == 8 ? 8 : 4;
    const int rows = dev::kWaves * rpw;
    return (rows * dev::kWenoLX + (rows + 5) * dev::kWenoTW) * (int)sizeof(double) +
           dev::kWaves * (int)sizeof(int);
}

hipError_t launchWeno(const WenoLaunch& w, hipStream_t st)
{
    if (w.nx < 1 || w.ny < 1) return hipSuccess;
    if (w.rowsPerWave == 8) return dev::launchWenoRpw<8>(w, st);
    return dev::launchWenoRpw<4>(w, st);
}

}  // namespace custen
