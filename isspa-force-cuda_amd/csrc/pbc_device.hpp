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
    __shared__ float lo[3][256], hi[3][256];
    float l[3] = {3.0e38f, 3.0e38f, 3.0e38f}, u[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
    for (int i = W.a0 + (int)threadIdx.x; i < W.a0 + W.n; i += 256) {
        const float4 x = xyzq[i];
        l[0] = fminf(l[0], x.x); u[0] = fmaxf(u[0], x.x);
        l[1] = fminf(l[1], x.y); u[1] = fmaxf(u[1], x.y);
        l[2] = fminf(l[2], x.z); u[2] = fmaxf(u[2], x.z);
    }
    for (int k = 0; k < 3; ++k) {
        lo[k][threadIdx.x] = l[k];
        hi[k][threadIdx.x] = u[k];
    }
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int k = 0; k < 3; ++k) {
                lo[k][threadIdx.x] = fminf(lo[k][threadIdx.x], lo[k][threadIdx.x + w]);
                hi[k][threadIdx.x] = fmaxf(hi[k][threadIdx.x], hi[k][threadIdx.x + w]);
            }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        int need = 0;
        for (int k = 0; k < 3; ++k) {
            const float ext = hi[k][0] - lo[k][0];
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
