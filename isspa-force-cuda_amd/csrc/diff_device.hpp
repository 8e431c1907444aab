// Analytic per-type functions of the differentiable IS-SPA model (FP32,
// device side).  The FP64 restatement and its derivation live in the oracle;
// the definitions are:
//
//   sigma_ts = (sigma + sigma_s)/2, eps_ts = sqrt(eps eps_s)
//   r_lo = max(x0 - sqrt(g0/alpha), core sigma_ts), r_hi = x0 + sqrt((g0 - 1)/alpha)
//   S(d) = smoothstep((d - r_lo)/delta + 1)
//   g(d) = S(d) max(0, g0 - alpha (d - x0)^2) for d < r_hi, 1 beyond
//   E(d) = c exp(-(d - x0)^2/2) S(d)
//   F(d) = 24 eps_ts/d (2 (sigma_ts/d)^12 - (sigma_ts/d)^6) S(d)
//
// Derivatives are with respect to theta = (sigma, eps, x0, g0, alpha).
#pragma once

#include <hip/hip_runtime.h>

namespace isspa {

// per-type constants, 64 bytes (one scalar load)
struct DiffType {
    float sts, ets;      // sigma_ts, eps_ts
    float x0, g0, al, c; // parabola and E-field amplitude
    float rlo, rhi;      // switch end and parabola end
    float idel;          // 1 / delta
    float eps;           // eps (dF/deps = F / (2 eps))
    float drlo[5];       // d r_lo / d theta
    float pad;
};

// S(d)
__device__ __forceinline__ float diff_switch(const DiffType &T, float d)
{
    const float z = (d - T.rlo) * T.idel + 1.0f;
    return z <= 0.0f ? 0.0f : (z >= 1.0f ? 1.0f : z * z * (3.0f - 2.0f * z));
}

__device__ __forceinline__ float diff_g(const DiffType &T, float d)
{
    if (d >= T.rhi) return 1.0f;
    const float u = d - T.x0;
    const float P = T.g0 - T.al * u * u;
    if (P <= 0.0f) return 0.0f;
    return diff_switch(T, d) * P;
}

__device__ __forceinline__ float diff_E(const DiffType &T, float d)
{
    const float u = d - T.x0;
    return T.c * expf(-0.5f * u * u) * diff_switch(T, d);
}

// the four constants diff_F needs, held in registers by the force pass
struct DiffFParams {
    float sts, ets, rlo, idel;
};

__device__ __forceinline__ DiffFParams diff_f_params(const DiffType &T)
{
    return DiffFParams{T.sts, T.ets, T.rlo, T.idel};
}

__device__ __forceinline__ float diff_F(const DiffFParams &T, float d, float rinv)
{
    const float z = (d - T.rlo) * T.idel + 1.0f;
    const float S = z <= 0.0f ? 0.0f : (z >= 1.0f ? 1.0f : z * z * (3.0f - 2.0f * z));
    const float sr = T.sts * rinv;
    const float sr2 = sr * sr;
    const float sr6 = sr2 * sr2 * sr2;
    return 24.0f * T.ets * rinv * (2.0f * sr6 * sr6 - sr6) * S;
}

// x / b for r = 1 / b rounded: a product, then two of Markstein's corrections
// by the exact remainder (P. Markstein, IBM J. Res. Dev. 34, 1990), which leave
// the correctly rounded quotient; 5 operations against 11 of the division
__device__ __forceinline__ float div_by(float x, float b, float r)
{
    float q = x * r;
    q = __builtin_fmaf(__builtin_fmaf(-b, q, x), r, q);
    return __builtin_fmaf(__builtin_fmaf(-b, q, x), r, q);
}

// What the adjoint needs of a lane's type, kept in registers: the constants,
// the reciprocals of the two it divides by, and d r_lo / d theta but for eps,
// on which r_lo never depends.
struct DiffVjpType {
    float sts, ets, x0, g0, al, c, rlo, rhi, idel;
    float eps2;            // 2 eps
    float rsts, reps2;     // 1 / sts, 1 / (2 eps)
    float d0, d2, d3, d4;  // d r_lo / d {sigma, x0, g0, al}
    __device__ __forceinline__ explicit DiffVjpType(const DiffType &T)
        : sts(T.sts), ets(T.ets), x0(T.x0), g0(T.g0), al(T.al), c(T.c), rlo(T.rlo), rhi(T.rhi),
          idel(T.idel), eps2(2.0f * T.eps), rsts(1.0f / T.sts), reps2(1.0f / (2.0f * T.eps)),
          d0(T.drlo[0]), d2(T.drlo[2]), d3(T.drlo[3]), d4(T.drlo[4])
    {
    }
};

// g and the derivatives of g, E and F by {sigma, x0, g0, al}, and of F by eps
struct DiffDerivs {
    float g;
    float dg[4], dE[4], dF[4], dFeps;
};

__device__ __forceinline__ DiffDerivs diff_derivs(const DiffVjpType &T, float d, float rinv)
{
    DiffDerivs o;
    const float z = (d - T.rlo) * T.idel + 1.0f;
    float S = 0.0f, dSdz = 0.0f;
    if (z >= 1.0f) {
        S = 1.0f;
    } else if (!(z <= 0.0f)) {  // NaN stays
        S = z * z * (3.0f - 2.0f * z);
        dSdz = 6.0f * z * (1.0f - z);
    }
    const float dS = -dSdz * T.idel;
    const float dS0 = dS * T.d0, dS2 = dS * T.d2, dS3 = dS * T.d3, dS4 = dS * T.d4;
    const float u = d - T.x0;
    o.g = 1.0f;
    o.dg[0] = o.dg[1] = o.dg[2] = o.dg[3] = 0.0f;
    if (!(d >= T.rhi)) {
        const float P = T.g0 - T.al * u * u;
        o.g = 0.0f;
        if (!(P <= 0.0f)) {
            o.g = S * P;
            o.dg[0] = dS0 * P;
            o.dg[1] = dS2 * P + S * (2.0f * T.al * u);
            o.dg[2] = dS3 * P + S;
            o.dg[3] = dS4 * P - S * (u * u);
        }
    }
    const float Er = T.c * expf(-0.5f * u * u);
    o.dE[0] = Er * dS0;
    o.dE[1] = Er * dS2 + Er * u * S;
    o.dE[2] = Er * dS3;
    o.dE[3] = Er * dS4;
    const float sr = T.sts * rinv;
    const float sr2 = sr * sr;
    const float sr6 = sr2 * sr2 * sr2;
    const float FLJ = 24.0f * T.ets * rinv * (2.0f * sr6 * sr6 - sr6);
    const float dFds =
        div_by(24.0f * T.ets * rinv * (24.0f * sr6 * sr6 - 6.0f * sr6), T.sts, T.rsts);
    o.dF[0] = FLJ * dS0 + 0.5f * dFds * S;
    o.dF[1] = FLJ * dS2;
    o.dF[2] = FLJ * dS3;
    o.dF[3] = FLJ * dS4;
    o.dFeps = div_by(FLJ, T.eps2, T.reps2) * S;
    return o;
}

}  // namespace isspa
