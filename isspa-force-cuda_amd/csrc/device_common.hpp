// Device helpers shared by every gfx950 kernel of the IS-SPA engine.
//
// Arithmetic contract with the CPU oracle: decision values (squared pair
// distances for the in-sphere / LJ-versus-CDD tests, minimum-image shifts,
// MC point coordinates) are formed with the exact FP32 operation sequence
// written here -- explicit fmaf where a fused op is used, __fmul_rn /
// __fadd_rn where contraction must not happen -- so the oracle can form the
// same values bit for bit and both take the same branch.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace isspa {

constexpr int kWave = 64;

// ---------------------------------------------------------------------------
// Langevin moments <P1>, <P2>, <P3> (= c1, 1.5 c2 - 0.5, 2.5 c3 - 1.5 c1 of
// src/isspa_force_cuda.cu:270-287) in FP64.  Below x = 5, <P_l> = i_l / i_0
// with the all-positive power series
//   i_l(x) / x^l = sum_k a_lk h^k,  h = x^2 / 2,  a_l0 = 1 / (2l+1)!!,
//   a_l(k+1) = a_lk / ((k+1)(2l+2k+3)),
// by Horner's rule, one fused multiply-add a term with compile-time
// coefficients; 19 terms, as the next one is below 1e-19 of the sum at x = 5.
// Above 5 the upward recurrence from coth, which then cancels by at most ~3x.
// (Term by term, with three operations a term and 30 terms, the epilogue
// launch took 5.9 us at 1,100 atoms, now 5.1, and the small-window launch of 44
// atoms 17.5, now 16.7 us.)
// ---------------------------------------------------------------------------
constexpr int kLgTerms = 19;
struct LangevinCoef {
    double a[4][kLgTerms];
};
constexpr LangevinCoef make_langevin_coef()
{
    LangevinCoef c{};
    double f = 1.0;
    for (int l = 0; l < 4; ++l) {
        if (l > 0) f /= (double)(2 * l + 1);
        double t = f;
        for (int k = 0; k < kLgTerms; ++k) {
            c.a[l][k] = t;
            t /= (double)(k + 1) * (double)(2 * l + 2 * k + 3);
        }
    }
    return c;
}
__constant__ constexpr LangevinCoef kLangevin = make_langevin_coef();

// coth x for x >= 5
__device__ __forceinline__ double coth_large(double x)
{
    const double u = exp(-2.0 * x);
    return (1.0 + u) / (1.0 - u);
}

// ---------------------------------------------------------------------------
// Philox4x32-10 (Salmon et al., SC'11).  Counter layout:
//   ctr = { index, (stream << 24) | draw, step, system }, key = { seed lo, hi }
// ---------------------------------------------------------------------------
constexpr uint32_t kStreamPoints = 0u;
constexpr uint32_t kStreamAndersen = 1u;

__device__ __forceinline__ uint4 philox4x32_10(uint4 c, uint2 k)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint32_t hi0 = __umulhi(0xD2511F53u, c.x);
        const uint32_t lo0 = 0xD2511F53u * c.x;
        const uint32_t hi1 = __umulhi(0xCD9E8D57u, c.z);
        const uint32_t lo1 = 0xCD9E8D57u * c.z;
        c = make_uint4(hi1 ^ c.y ^ k.x, lo1, hi0 ^ c.w ^ k.y, lo0);
        k.x += 0x9E3779B9u;
        k.y += 0xBB67AE85u;
    }
    return c;
}

__device__ __forceinline__ uint4 philox_draw(uint64_t seed, uint32_t index, uint32_t stream,
                                             uint32_t draw, uint32_t step, uint32_t sys)
{
    return philox4x32_10(make_uint4(index, (stream << 24) | draw, step, sys),
                         make_uint2((uint32_t)seed, (uint32_t)(seed >> 32)));
}

// MC rejection sampling on the 2^-24 lattice: accept iff |2v - 2^24|^2 summed
// over the three axes is <= floor(0.99 * 2^48)  (u in the ball |u|^2 < 0.99).
constexpr uint64_t kMcAcceptMax = 278660226943549ULL;
constexpr int kMcMaxAttempts = 64;

// ---------------------------------------------------------------------------
// single-image minimum image (src/cuda_vector_routines.h:28-47):
//   r > h -> r - L ; r < -h -> r + L, with one rounding.
// As k = [|r| > h] and r - k copysign(L, r): k is clamp(|r| S - h S) to [0, 1]
// of one fused multiply-add, S a power of two that takes h to 2^100.  The
// fma's sign is exact and |r| > h exceeds h by at least 2^-24 h, so k is
// exactly 0 or 1 (a NaN gives 0) for every h from 2^-102 up.  Bounded by VALU
// issue: 3 operations an axis, none with an SGPR or a mask operand, measured
// 7.2 cycles against 20.6 of compare, compare, select, select, fma; at 4,510
// periodic atoms the field pass took 311 and now 241 us, the force pass 506 and
// 433 us.
// ---------------------------------------------------------------------------
struct MinImage {
    float L, S, nhS;  // box length, scale, -h scale
};

__device__ __forceinline__ MinImage min_image_of(float L, float h)
{
    const int e = __builtin_amdgcn_frexp_expf(h);  // h = m 2^e, m in [1/2, 1)
    const float S = __builtin_amdgcn_ldexpf(1.0f, min(126, 100 - e));
    return MinImage{L, S, -h * S};
}

__device__ __forceinline__ float min_image1(float r, const MinImage &b)
{
    const float k =
        __builtin_amdgcn_fmed3f(__builtin_fmaf(__builtin_fabsf(r), b.S, b.nhS), 0.0f, 1.0f);
    return __builtin_fmaf(-k, __builtin_copysignf(b.L, r), r);
}

// squared distance in the operation order the oracle reproduces
__device__ __forceinline__ float dist2_f32(float rx, float ry, float rz)
{
    return __builtin_fmaf(rz, rz, __builtin_fmaf(ry, ry, rx * rx));
}

__device__ __forceinline__ float rsqrt_f32(float x) { return __builtin_amdgcn_rsqf(x); }

// wave-uniform "any lane" test
__device__ __forceinline__ bool wave_any(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0ull; }

// A read-only input seen through the constant address space.  Its loads at a
// wave-uniform index are scalar loads whatever else the kernel writes: the
// compiler otherwise turns them into per-lane vector loads when it cannot
// prove that no store of the kernel reaches them (as in a kernel that also
// runs the all-pairs blocks, which write their partials).  Only for memory
// that no work-item writes during the launch.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T *read_only(const T *p)
{
    return (const __attribute__((address_space(4))) T *)p;
}

// float4s read through the constant address space: scalar loads, whatever the
// compiler knows about the kernel's stores and asm statements
struct ScalarRecords {
    const __attribute__((address_space(4))) float *p;
    __device__ __forceinline__ ScalarRecords operator+(int k) const { return {p + 4 * k}; }
    __device__ __forceinline__ float4 operator[](int k) const
    {
        const auto *q = p + 4 * k;
        return make_float4(q[0], q[1], q[2], q[3]);
    }
};

}  // namespace isspa
