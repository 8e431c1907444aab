// A.1 MC points (src/isspa_force_cuda.cu:73-107), Philox instead of curand,
// as a per-point device function shared by the points kernel and the MD
// engine's step prologue.
#pragma once

#include "device_common.hpp"
#include "kernels.hpp"

namespace isspa {


// x + R * (v 2^-24) with two roundings, never fused into one FMA, so the
// oracle forms the same bits (v 2^-24 itself is exact)
__device__ __forceinline__ float point_coord(float x, float R, int v)
{
#pragma clang fp contract(off)
    const float u = (float)v * 5.9604644775390625e-08f;
    const float du = R * u;
    return x + du;
}

// Draw d of point m (window-local index): true if its 24-bit signed lattice
// vector lies in the unit ball.
__device__ __forceinline__ bool mc_draw(uint64_t seed, uint32_t m, uint32_t d, uint32_t step,
                                        uint32_t sys, int &c0, int &c1, int &c2)
{
    const uint4 o = philox_draw(seed, m, kStreamPoints, d, step, sys);
    c0 = 2 * (int)(o.x >> 8) - (1 << 24);
    c1 = 2 * (int)(o.y >> 8) - (1 << 24);
    c2 = 2 * (int)(o.z >> 8) - (1 << 24);
    const uint64_t r2 = (uint64_t)((int64_t)c0 * c0 + (int64_t)c1 * c1 + (int64_t)c2 * c2);
    return r2 <= kMcAcceptMax;
}

// the point of owner x at lattice vector (v0, v1, v2); .w is the owner's rmax^2
__device__ __forceinline__ float4 mc_place(float4 x, float R, float R2, int v0, int v1, int v2)
{
    return make_float4(point_coord(x.x, R, v0), point_coord(x.y, R, v1), point_coord(x.z, R, v2),
                       R2);
}

// Point gp (global index; window w owns points [a0_w nMC, (a0_w + n_w) nMC),
// point m of the window belongs to atom m / nMC) is drawn with counter
// {m, draw, step, sys_w}: the first draw whose 24-bit signed lattice vector
// lies in the unit ball.  .w of each point carries the owner's rmax^2.
//
// A block of 256 work-items draws kMcBlockPts points, kMcLanes lanes each: the
// lanes try consecutive draws side by side and the first accepted one counts.
// A wave repeats until its last point is placed, and a draw, ten Philox
// rounds, is a chain of some 150 dependent operations: with one lane a point
// that was seven draws in a row, now it is two, the same work in four times
// the waves.  The owner's position and radii are requested before the first
// draw, and the owner is found by a 32-bit division (a model has fewer than 2^29
// points).
// Launch of 1,100 atoms, nMC = 20: 5.6 -> 3.1 us; 19,998 atoms 12.7 -> 11.9 us.
constexpr int kMcLanes = 4, kMcBlockPts = 256 / kMcLanes;

__device__ __forceinline__ void mc_points_block(const PointsArgs &a, long long block)
{
    static_assert(kMcLanes == 4 && kMcMaxAttempts % kMcLanes == 0, "quads, whole rounds");
    const long long total = (long long)a.ntot * a.nmc;
    const int sub = threadIdx.x % kMcLanes;
    const long long at = block * kMcBlockPts + threadIdx.x / kMcLanes;
    const long long gp = min(at, total - 1);
    const int k = (int)((uint32_t)gp / (uint32_t)a.nmc);
    const float4 x = a.xyzq[k];
    const int t = a.itype[k];
    const WinDesc W = a.nwin == 1 ? a.wins[0] : a.wins[a.atom_win[k]];
    const float R = a.rmax[t], R2 = a.rmax2[t];
    const uint32_t step = a.step_d ? *a.step_d : a.step;
    const uint32_t m = (uint32_t)(gp - (long long)W.a0 * a.nmc);
    const int quad = (int)threadIdx.x % kWave & ~(kMcLanes - 1);
    bool open = at < total;
    for (int d = 0; d < kMcMaxAttempts && wave_any(open); d += kMcLanes) {
        int c0, c1, c2;
        const bool ok = mc_draw(a.seed, m, (uint32_t)(d + sub), step, W.sys, c0, c1, c2);
        const int hits = (int)(__builtin_amdgcn_ballot_w64(ok) >> quad) & (kMcLanes * 4 - 1);
        if (open && hits != 0) {
            if (sub == __builtin_ctz(hits)) a.pts[gp] = mc_place(x, R, R2, c0, c1, c2);
            open = false;
        }
    }
    // every draw refused: the point at its atom
    if (open && sub == 0) a.pts[gp] = mc_place(x, R, R2, 0, 0, 0);
}

}  // namespace isspa
