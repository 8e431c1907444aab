// Per-window minimum-image flag, computed by one 256-thread block.
#pragma once

#include "kernels.hpp"

namespace isspa {

// flag = 1 when some pair separation of window W may exceed half a box
// (minimum image needed); 0 when (extent + rmax + margin) < L/2 on every axis,
// in which case the single-image minimum image is the identity for every
// atom-atom and point-atom pair and the kernels take their shift-free loops.
// Every thread of the block must call it.
__device__ inline void pbc_flag_block(const WinDesc &W, const float4 *__restrict__ xyzq,
                                      float rmax_all, int *flag)
{
    constexpr int kU = 8;  // atoms in flight a work-item
    float l[3] = {3.0e38f, 3.0e38f, 3.0e38f}, u[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
    for (int i0 = threadIdx.x; i0 < W.n; i0 += kU * 256) {
        float4 x[kU];
#pragma unroll
        for (int k = 0; k < kU; ++k) x[k] = xyzq[W.a0 + min(i0 + k * 256, W.n - 1)];
#pragma unroll
        for (int k = 0; k < kU; ++k) {
            l[0] = fminf(l[0], x[k].x); u[0] = fmaxf(u[0], x[k].x);
            l[1] = fminf(l[1], x[k].y); u[1] = fmaxf(u[1], x[k].y);
            l[2] = fminf(l[2], x[k].z); u[2] = fmaxf(u[2], x[k].z);
        }
    }
    // the waves by shuffles, their extents through LDS
    __shared__ float lo[3][4], hi[3][4];
    for (int w = kWave / 2; w > 0; w >>= 1)
        for (int k = 0; k < 3; ++k) {
            l[k] = fminf(l[k], __shfl_xor(l[k], w));
            u[k] = fmaxf(u[k], __shfl_xor(u[k], w));
        }
    if (threadIdx.x % kWave == 0)
        for (int k = 0; k < 3; ++k) {
            lo[k][threadIdx.x / kWave] = l[k];
            hi[k][threadIdx.x / kWave] = u[k];
        }
    __syncthreads();
    if (threadIdx.x == 0) {
        int need = 0;
        for (int k = 0; k < 3; ++k) {
            const float ext = fmaxf(fmaxf(hi[k][0], hi[k][1]), fmaxf(hi[k][2], hi[k][3])) -
                              fminf(fminf(lo[k][0], lo[k][1]), fminf(lo[k][2], lo[k][3]));
            if (!(ext + rmax_all + 1.0e-2f < W.h)) need = 1;  // NaN -> need
        }
        *flag = need;
    }
}

// The same decision taken by a block for its own use, atom by atom: none of
// the window's atoms is far from the first one, x0, if every one lies within
// (L/2 - rmax - margin) / 2 of it on every axis.  It may say far where the
// flag says 0; the image loop then shifts nothing.
__device__ __forceinline__ bool atoms_far(const WinDesc &W, float4 x, float4 x0, float rmax_all)
{
    const float lim = 0.5f * (W.h - rmax_all - 1.0e-2f);
    // NaN -> far
    return !(fabsf(x.x - x0.x) < lim && fabsf(x.y - x0.y) < lim && fabsf(x.z - x0.z) < lim);
}

// for the whole window, by a block's first NT work-items (two barriers)
template <int NT>
__device__ __forceinline__ bool needs_image(const WinDesc &W, const float4 *__restrict__ xyzq,
                                            float rmax_all)
{
    const float4 x0 = xyzq[W.a0];
    bool far = false;
    for (int i = threadIdx.x; i < W.n; i += NT)
        far = far || atoms_far(W, xyzq[W.a0 + i], x0, rmax_all);
    __shared__ int need;
    if (threadIdx.x == 0) need = 0;
    __syncthreads();
    if (far) need = 1;
    __syncthreads();
    return need != 0;
}

}  // namespace isspa
