// Differentiable IS-SPA + nonbond model: parameter preparation, forward
// reduction and the hand-written adjoint (vector-Jacobian product) for gfx950.
//
// Forward (reusing the plain kernels with analytic per-type functions):
//   points -> field -> epilogue -> force partials -> k_diff_reduce
//   F_i = -q_i vtot_i S_e,i - vtot_i S_lj,i  (+ nonbond)
// Adjoint for a cotangent lambda = dL/dF, in reverse order:
//   k_vjp_points   lanes = MC points, receivers streamed: bars of the point
//                  record (E-hat, A1..A3, E0c, w) from every receiver
//   k_vjp_epilogue per point, FP64: back through |E|, E-hat, the Langevin
//                  moments and w = g/cnt to dL/dE, dL/dE0, g dL/dg
//   k_vjp_atoms    lanes = atoms, points streamed: dL/dq_j through the field,
//                  and the per-atom bars of the type parameters through g, E
//                  (field side) and F (receiver side)
//   k_vjp_nonbond  lanes = receivers, partners streamed
//   k_vjp_finish   per atom: sum the chunk partials in order, add the direct
//                  charge term lambda_i . (-vtot_i S_e,i)
//   k_type_reduce  per type, FP64, fixed order
// Every accumulation is an FP32 tile sum flushed into FP64, summed over
// partials in a fixed order: results are deterministic.
#include <algorithm>

#include "device_common.hpp"
#include "diff_device.hpp"
#include "kernels.hpp"
#include "reduce_device.hpp"

namespace isspa {

constexpr int kB = 256;
constexpr int kTile = 64;

static inline int nblk(long long n) { return (int)((n + kB - 1) / kB); }

// ---------------------------------------------------------------------------
// parameters -> per-type constants and LJ pair tables
// ---------------------------------------------------------------------------
__device__ __forceinline__ void diff_prep_types(const DiffPrepArgs &a)
{
    const int T = a.T;
    for (int t = threadIdx.x; t < T; t += kB) {
        const double sig = a.theta[5 * t], eps = a.theta[5 * t + 1], x0 = a.theta[5 * t + 2];
        const double g0 = a.theta[5 * t + 3], al = a.theta[5 * t + 4];
        const double sts = 0.5 * (sig + a.sig_s), ets = sqrt(eps * a.eps_s);
        const double w = sqrt(g0 / al);
        DiffType d;
        d.sts = (float)sts;
        d.ets = (float)ets;
        d.x0 = (float)x0;
        d.g0 = (float)g0;
        d.al = (float)al;
        d.c = (float)a.camp[t];
        d.rhi = (float)(x0 + sqrt((g0 - 1.0) / al));
        d.idel = (float)(1.0 / a.delta);
        d.eps = (float)eps;
        for (int p = 0; p < 5; ++p) d.drlo[p] = 0.0f;
        if (x0 - w >= a.core * sts) {
            d.rlo = (float)(x0 - w);
            d.drlo[2] = 1.0f;
            d.drlo[3] = (float)(-1.0 / (2.0 * w * al));
            d.drlo[4] = (float)(w / (2.0 * al));
        } else {
            d.rlo = (float)(a.core * sts);
            d.drlo[0] = (float)(0.5 * a.core);
        }
        d.pad = 0.0f;
        a.types[t] = d;
    }
    for (int k = threadIdx.x; k < T * T; k += kB) {
        const int i = k / T, j = k % T;
        const double s = 0.5 * (a.theta[5 * i] + a.theta[5 * j]);
        const double e = sqrt(a.theta[5 * i + 1] * a.theta[5 * j + 1]);
        const double s2 = s * s, s6 = s2 * s2 * s2;
        const double A = 4.0 * e * s6 * s6, B = 4.0 * e * s6;
        a.nb_lj[k] = make_float2((float)(12.0 * A), (float)(6.0 * B));
        // {A, B, dA/dsigma_ij, dB/dsigma_ij}
        a.nb_ld[k] = make_float4((float)A, (float)B, (float)(12.0 * A / s), (float)(6.0 * B / s));
    }
}

// positions with the charges as FP32 .w; receiver records for the adjoint
__device__ __forceinline__ void diff_prep_atoms(const DiffAtomArgs &a, int block)
{
    const int i = block * kB + (int)threadIdx.x;
    if (i >= a.n) return;
    const float4 x = a.xyz[i];
    const double q = a.q[i];
    a.xq[i] = make_float4(x.x, x.y, x.z, (float)q);
    if (!a.lam) return;
    const int t = a.itype[i];
    const double vt = a.vtot[t];
    const double l0 = a.lam[3 * i], l1 = a.lam[3 * i + 1], l2 = a.lam[3 * i + 2];
    const double cq = -q * vt;
    float4 *r = a.arec + 4 * (size_t)i;
    r[0] = make_float4(x.x, x.y, x.z, a.rmax2[t]);
    r[1] = make_float4((float)(cq * l0), (float)(cq * l1), (float)(cq * l2), __int_as_float(t));
    r[2] = make_float4((float)(-vt * l0), (float)(-vt * l1), (float)(-vt * l2), (float)q);
    r[3] = make_float4((float)l0, (float)l1, (float)l2, 0.0f);
}

// the types by the first block, the atoms by the others
__global__ __launch_bounds__(kB) void k_diff_prep(DiffPrepArgs t, DiffAtomArgs a)
{
    if (blockIdx.x == 0)
        diff_prep_types(t);
    else
        diff_prep_atoms(a, (int)blockIdx.x - 1);
}

// F_i = -q_i vtot_i S_e - vtot_i S_lj, plus the all-pairs sum where its partials
// are given (overwrites f); S_e kept for the adjoint.
// Latency bound: a block of 16 atoms x 16 entry slices (reduce_device.hpp) with
// eight entries in flight a slice.  One lane per atom over all chunks
// took 53.9 us at 550 atoms (3 blocks, 181 dependent rounds) and 121 us for
// 32 x 1,100 atoms; now 7.4 and 16 us (86 MB, 5.4 TB/s).
__global__ __launch_bounds__(kB) void k_diff_reduce(DiffReduceArgs a)
{
    __shared__ double red[kSumSlices][9][kSumAtoms];
    const int al = threadIdx.x % kSumAtoms, sl = threadIdx.x / kSumAtoms;
    const int i = blockIdx.x * kSumAtoms + al;
    const bool valid = i < a.n;
    double s[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};  // S_e, S_lj; all pairs
    if (valid) {
        const WinDesc W = window_of(a.wins, a.nwin, a.atom_win, i);
        sum_batches<6, 8>(ForceEntry<6>(W, a.part, i), sl, W.fents, s);
        if (a.nb_part) {
            const WinDesc Wn = window_of(a.nb_wins, a.nwin, a.atom_win, i);
            sum_batches<3, 4>(nonbond_entry<3>(Wn, a.nb_part, a.nb_B, i), sl, Wn.nte, s + 6);
        }
    }
    combine_slices<9>(red, al, sl, s);
    if (sl != 0 || !valid) return;
    const double vt = a.vtot[a.itype[i]];
    const double qv = -a.q[i] * vt;
    for (int c = 0; c < 3; ++c) {
        a.se[3 * i + c] = s[c];
        a.f[3 * i + c] = qv * s[c] - vt * s[3 + c] + s[6 + c];
    }
}

// ---------------------------------------------------------------------------
// adjoint, point side: lanes own MC points, receivers stream (wave-uniform)
// ---------------------------------------------------------------------------
struct PointBar {
    float hx, hy, hz;   // E-hat bar
    float a1, a2, a3;   // A1..A3 bar
    float cx, cy, cz;   // E0c bar
    float w;            // w bar
};

template <bool PBC>
__device__ __forceinline__ void vjp_points_tile(const VjpArgs &a, int j0, int j1,
                                                const MinImage &mi, float px, float py, float pz,
                                                float Ex, float Ey, float Ez, float A1, float A2,
                                                float A3, const Progress &pg, PointBar &b)
{
    // wave-uniform records, the next one requested while this one is used
    ScalarRecords nr{read_only(reinterpret_cast<const float *>(a.arec + 4 * j0))};
    float4 n0 = nr[0], n1 = nr[1], n2 = nr[2];
    for (int j = j0; j < j1;) {
        const int stop = j0 + pg.rank(j - j0, j1 - j0);
        for (; j < stop; ++j) {
            const float4 r0 = n0, r1 = n1, r2 = n2;
            if (j + 1 < j1) nr = nr + 4;
            n0 = nr[0];
            n1 = nr[1];
            n2 = nr[2];
            float rx = px - r0.x, ry = py - r0.y, rz = pz - r0.z;
            if (PBC) {
                rx = min_image1(rx, mi);
                ry = min_image1(ry, mi);
                rz = min_image1(rz, mi);
            }
            const float d2 = dist2_f32(rx, ry, rz);
            const float rinv = rsqrt_f32(d2);
            const float u = __builtin_fmaf(Ez, rz, __builtin_fmaf(Ey, ry, Ex * rx)) * rinv;
            const float u2 = u * u;
            const float P2 = __builtin_fmaf(7.5f, u2, -1.5f);
            const float P3 = __builtin_fmaf(17.5f, u2, -7.5f) * u;
            const float dP2 = 15.0f * u;
            const float dP3 = __builtin_fmaf(52.5f, u2, -7.5f);
            const float rinv2 = rinv * rinv;
            const float rinv3 = rinv2 * rinv;
            const float rinv4 = rinv2 * rinv2;
            const float rinv5 = rinv4 * rinv;
            const float rinv6 = rinv4 * rinv2;
            const float la = __builtin_fmaf(r1.z, rz, __builtin_fmaf(r1.y, ry, r1.x * rx));  // Lambda.r
            const float lb = __builtin_fmaf(r1.z, Ez, __builtin_fmaf(r1.y, Ey, r1.x * Ex));  // Lambda.E-hat
            const float u3 = 3.0f * u;
            b.a1 += la * u3 * rinv4 - lb * rinv3;
            b.a2 += la * rinv5 * P2 - lb * u3 * rinv4;
            b.a3 += la * rinv6 * P3 - lb * rinv5 * P2;
            const float dal = 3.0f * A1 * rinv4 + A2 * dP2 * rinv5 + A3 * dP3 * rinv6;
            const float dk = 3.0f * A2 * rinv4 + dP2 * A3 * rinv5;
            const float k = u3 * A2 * rinv4 + P2 * A3 * rinv5;
            const float cu = (la * dal - lb * dk) * rinv;
            const float ce = -(rinv3 * A1 + k);
            b.hx += cu * rx + ce * r1.x;
            b.hy += cu * ry + ce * r1.y;
            b.hz += cu * rz + ce * r1.z;
            if (d2 > r0.w) {
                const float c5 = rinv5 * la, c3 = rinv3 * (1.0f / 3.0f);
                b.cx += c5 * rx - c3 * r1.x;
                b.cy += c5 * ry - c3 * r1.y;
                b.cz += c5 * rz - c3 * r1.z;
            } else {
                const float lp = __builtin_fmaf(r2.z, rz, __builtin_fmaf(r2.y, ry, r2.x * rx));
                // the atom's type is wave-uniform: its constants come by scalar loads
                const auto *T = read_only(reinterpret_cast<const float *>(
                    a.dtypes + __builtin_amdgcn_readfirstlane(__float_as_int(r1.w))));
                const DiffFParams fp{T[offsetof(DiffType, sts) / 4], T[offsetof(DiffType, ets) / 4],
                                     T[offsetof(DiffType, rlo) / 4], T[offsetof(DiffType, idel) / 4]};
                b.w += diff_F(fp, d2 * rinv, rinv) * lp * rinv;
            }
        }
    }
}

// A block takes W.fg splits of the same 256 / fg points and adds their FP64
// sums in split order through LDS, as the field pass: the epilogue, which is
// bound by the partials it reads, takes 39 us instead of 117 at 32 x 1,100
// atoms (nMC = 20) and 7.4 instead of 11.2 at 550.  The loop issues some 70
// VALU operations a pair; the next atom's record is requested one atom ahead,
// which hides the scalar load where few waves share a SIMD (550 atoms: 28.0 ->
// 24.6 us) and costs nothing where many do (1,130 us at 32 x 1,100).
__global__ __launch_bounds__(kB) void k_vjp_points(VjpArgs a)
{
    __shared__ double red[10][3 * kWave];  // fg = 4: 3 splits of 64 points
    const int4 bt = a.gblk[blockIdx.x];
    const WinDesc W = a.wins[bt.x];
    const int P = W.n * a.nmc;
    const int fg = W.fg, np = kB / fg;
    // wave-uniform, so the atom range stays on scalar loads
    const int sub = __builtin_amdgcn_readfirstlane((int)threadIdx.x / np);
    const int lt = (int)threadIdx.x - sub * np;
    const int m = bt.y * np + lt;
    const int j0 = W.a0 + (bt.z * fg + sub) * W.aps;
    const int j1 = min(W.a0 + W.n, j0 + W.aps);
    const bool valid = m < P;
    const long long gp = (long long)W.a0 * a.nmc + (valid ? m : 0);
    const float4 q0 = a.rec4[4 * gp + 0];  // p, Ehat.x
    const float4 q1 = a.rec4[4 * gp + 1];  // Ehat.yz
    const float4 q3 = a.rec4[4 * gp + 3];  // A2, 3 A2, A3, w
    const float A1 = a.aux4[gp].w;
    const bool pbc = a.pbc_flag[bt.x] != 0;
    const MinImage mi = min_image_of(W.L, W.h);
    double acc[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    Progress pg(a.ranked_from, j1 - j0);
    for (int jt = j0; jt < j1; jt += kTile) {
        const int je = min(j1, jt + kTile);
        pg.done = jt - j0;
        PointBar b{0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        if (pbc)
            vjp_points_tile<true>(a, jt, je, mi, q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, A1, q3.x,
                                  q3.z, pg, b);
        else
            vjp_points_tile<false>(a, jt, je, mi, q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, A1, q3.x,
                                   q3.z, pg, b);
        acc[0] += b.hx; acc[1] += b.hy; acc[2] += b.hz;
        acc[3] += b.a1; acc[4] += b.a2; acc[5] += b.a3;
        acc[6] += b.cx; acc[7] += b.cy; acc[8] += b.cz;
        acc[9] += b.w;
    }
    if (sub > 0)
        for (int k = 0; k < 10; ++k) red[k][(sub - 1) * np + lt] = acc[k];
    __syncthreads();
    if (sub > 0 || !valid) return;
    const long long o = W.fpo + (long long)bt.z * P + m;
    for (int k = 0; k < 10; ++k) {
        for (int w = 0; w + 1 < fg; ++w) acc[k] += red[k][w * np + lt];
        a.ppart[k * a.F + o] = acc[k];
    }
}

// Langevin moments and their derivatives, as the forward epilogue
__device__ __forceinline__ void moments_derivs(double x, double m[3], double dm[3])
{
    if (x < 5.0) {
        const double h = 0.5 * x * x;
        double s[4], ds[4];  // the series and their derivatives by h
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            s[l] = kLangevin.a[l][kLgTerms - 1];
            ds[l] = 0.0;
        }
#pragma unroll
        for (int k = kLgTerms - 2; k >= 0; --k)
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                ds[l] = __builtin_fma(ds[l], h, s[l]);
                s[l] = __builtin_fma(s[l], h, kLangevin.a[l][k]);
            }
        const double s0 = s[0];
        double xl = 1.0;
#pragma unroll
        for (int l = 1; l <= 3; ++l) {
            const double xl1 = xl;  // x^(l-1)
            xl *= x;                // x^l
            m[l - 1] = xl * s[l] / s0;
            dm[l - 1] = (double)l * xl1 * s[l] / s0 + xl * x * (ds[l] * s0 - s[l] * ds[0]) / (s0 * s0);
        }
        return;
    }
    const double coth = coth_large(x);
    const double sh = sinh(x);
    m[0] = coth - 1.0 / x;
    m[1] = 1.0 - 3.0 * m[0] / x;
    m[2] = m[0] - 5.0 * m[1] / x;
    dm[0] = 1.0 / (x * x) - 1.0 / (sh * sh);
    dm[1] = -3.0 * dm[0] / x + 3.0 * m[0] / (x * x);
    dm[2] = dm[0] - 5.0 * dm[1] / x + 5.0 * m[1] / (x * x);
}

__device__ __forceinline__ void vjp_epilogue_block(const VjpArgs &a)
{
    const long long gp = (long long)blockIdx.x * kB + threadIdx.x;
    if (gp >= a.Ptot) return;
    const WinDesc W = a.wins[a.atom_win[gp / a.nmc]];
    const int P = W.n * a.nmc;
    const long long m = gp - (long long)W.a0 * a.nmc;
    double b[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int s = 0; s < W.splits / W.fg; ++s) {
        const long long o = W.fpo + (long long)s * P + m;
        for (int k = 0; k < 10; ++k) b[k] += a.ppart[k * a.F + o];
    }
    const double E[3] = {a.E_out[3 * gp], a.E_out[3 * gp + 1], a.E_out[3 * gp + 2]};
    const double g = a.g_out[gp];
    const double cnt = (double)a.cnt_out[gp];
    const double x = sqrt(E[0] * E[0] + E[1] * E[1] + E[2] * E[2]);
    double eh[3];
    for (int c = 0; c < 3; ++c) eh[c] = x > 0.0 ? E[c] / x : 0.0;
    double mm[3], dm[3];
    moments_derivs(x, mm, dm);
    const double w = g / cnt, cp = (double)a.p0 / cnt;
    const double p0 = a.p0, q0 = a.q0, o0 = a.o0;
    const double wbar = b[9] + p0 * mm[0] * b[3] + q0 * mm[1] * b[4] + o0 * mm[2] * b[5];
    const double gbar = wbar / cnt;
    const double xbar = w * (p0 * dm[0] * b[3] + q0 * dm[1] * b[4] + o0 * dm[2] * b[5]);
    const double hdot = b[0] * eh[0] + b[1] * eh[1] + b[2] * eh[2];
    double Eb[3], E0b[3];
    for (int c = 0; c < 3; ++c) {
        Eb[c] = xbar * eh[c] + (x > 0.0 ? (b[c] - hdot * eh[c]) / x : 0.0);
        E0b[c] = cp * b[6 + c];
    }
    const float4 p = a.pts[gp];
    float4 *r = a.prec + 4 * gp;
    r[0] = p;
    r[1] = make_float4((float)Eb[0], (float)Eb[1], (float)Eb[2], (float)(g * gbar));
    r[2] = make_float4((float)E0b[0], (float)E0b[1], (float)E0b[2], (float)w);
    r[3] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// ---------------------------------------------------------------------------
// adjoint, atom side: lanes own atoms, point records stream (wave-uniform)
// ---------------------------------------------------------------------------
template <bool PBC>
__device__ __forceinline__ void vjp_atoms_tile(const VjpArgs &a, const float4 *__restrict__ pr,
                                               const DiffVjpType &Tj, int m0, int m1,
                                               const MinImage &mi, float4 xj, float R2j, float lpx,
                                               float lpy, float lpz, const Progress &pg, float &qb,
                                               double tb[5])
{
    const float e0 = a.e0;
    // wave-uniform records, the next one requested while this one is used
    ScalarRecords nr{read_only(reinterpret_cast<const float *>(pr + 4 * m0))};
    float4 n0 = nr[0], n1 = nr[1], n2 = nr[2];
    for (int m = m0; m < m1;) {
        const int stop = m0 + pg.rank(m - m0, m1 - m0);
#pragma unroll 2
        for (; m < stop; ++m) {
            const float4 p = n0, eb = n1, e0b = n2;
            if (m + 1 < m1) nr = nr + 4;
            n0 = nr[0];
            n1 = nr[1];
            n2 = nr[2];
            float rx = p.x - xj.x, ry = p.y - xj.y, rz = p.z - xj.z;
            if (PBC) {
                rx = min_image1(rx, mi);
                ry = min_image1(ry, mi);
                rz = min_image1(rz, mi);
            }
            const float d2 = dist2_f32(rx, ry, rz);
            const float rinv = rsqrt_f32(d2);
            const float er = __builtin_fmaf(eb.z, rz, __builtin_fmaf(eb.y, ry, eb.x * rx));
            const float e0r = __builtin_fmaf(e0b.z, rz, __builtin_fmaf(e0b.y, ry, e0b.x * rx));
            const bool in_own = d2 <= p.w;
            const bool in_rec = d2 <= R2j;
            const float s = -e0 * rinv * rinv * rinv;
            qb = __builtin_fmaf(s, in_own ? er : er + e0r, qb);
            if (in_own || in_rec) {
                const float d = d2 * rinv;
                const DiffDerivs D = diff_derivs(Tj, d, rinv);
                if (in_own) {
                    const float ce = er * rinv;
                    const float cg = (eb.w != 0.0f && D.g != 0.0f) ? eb.w / D.g : 0.0f;
                    tb[0] += (double)(ce * D.dE[0] + cg * D.dg[0]);
                    for (int k = 1; k < 4; ++k) tb[k + 1] += (double)(ce * D.dE[k] + cg * D.dg[k]);
                }
                if (in_rec) {
                    const float lp = __builtin_fmaf(lpz, rz, __builtin_fmaf(lpy, ry, lpx * rx));
                    const float cf = e0b.w * lp * rinv;
                    tb[0] += (double)(cf * D.dF[0]);
                    tb[1] += (double)(cf * D.dFeps);
                    for (int k = 1; k < 4; ++k) tb[k + 1] += (double)(cf * D.dF[k]);
                }
            }
        }
    }
}

// A block's four waves take the same 64 atoms and one chunk each, and add
// their FP64 sums in chunk order through LDS (as the force pass): a quarter of
// the partials to write and to sum, and no idle wave in a window's last block.
// 32 x 1,100 atoms: k_vjp_finish behind it 81 -> 24 us.
// Bounded by the in-sphere branch, some 200 operations for the few lanes of a
// wave that are in a sphere.  The lane's type record stays in registers (read
// from LDS through a flat pointer in the branch, each read waited for both
// memories) and the next point is requested one point ahead: 52.8 -> 36 us at
// 550 atoms, 985 -> 880 us at 32 x 1,100.  Without the terms that are zero for
// every type, and with the divisions by the type's constants as products
// (div_by), 32 and 840 us.  Six waves a SIMD: held to seven or
// eight the branch spills (934 us and worse), left alone it takes five (1,006).
__global__ __launch_bounds__(kB, 6) void k_vjp_atoms(VjpArgs a)
{
    __shared__ double red[3][6][kWave];
    const int4 bt = a.vblk[blockIdx.x];
    const WinDesc W = a.wins[bt.x];
    const int lane = threadIdx.x % kWave;
    // read from the first lane so the compiler knows it is wave-uniform
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int il = bt.y * kWave + lane;
    const long long pbase = (long long)W.a0 * a.nmc;
    const float4 *__restrict__ pr = a.prec + 4 * pbase;  // this window's point bars
    const int P = W.n * a.nmc;
    const int m0 = min(P, (4 * bt.z + wv) * W.ppc);  // window-local point range
    const int m1 = min(P, m0 + W.ppc);
    const bool valid = il < W.n;
    const int j = W.a0 + (valid ? il : 0);
    const float4 xj = a.xq[j];
    const int tj = a.itype[j];
    const float R2j = valid ? a.rmax2[tj] : -1.0f;
    const float4 lp = a.arec[4 * (size_t)j + 2];  // Lambda' = -vtot lambda
    const bool pbc = a.pbc_flag[bt.x] != 0;
    const DiffVjpType Tj(a.dtypes[tj]);
    const MinImage mi = min_image_of(W.L, W.h);
    double qsum = 0.0, tb[5] = {0, 0, 0, 0, 0};  // q, theta
    Progress pg(a.ranked_from, m1 - m0);
    for (int mt = m0; mt < m1; mt += kTile) {
        const int me = min(m1, mt + kTile);
        pg.done = mt - m0;
        float qb = 0.0f;
        if (pbc)
            vjp_atoms_tile<true>(a, pr, Tj, mt, me, mi, xj, R2j, lp.x, lp.y, lp.z, pg, qb, tb);
        else
            vjp_atoms_tile<false>(a, pr, Tj, mt, me, mi, xj, R2j, lp.x, lp.y, lp.z, pg, qb, tb);
        qsum += (double)qb;
    }
    double acc[6] = {qsum, tb[0], tb[1], tb[2], tb[3], tb[4]};
    if (wv > 0)
        for (int k = 0; k < 6; ++k) red[wv - 1][k][lane] = acc[k];
    __syncthreads();
    if (wv > 0 || !valid) return;
    const long long o = W.vpo + (long long)bt.z * W.n + il;
    for (int k = 0; k < 6; ++k) {
        for (int w = 0; w < 3; ++w) acc[k] += red[w][k][lane];
        a.apart[k * a.C + o] = acc[k];
    }
}

// ---------------------------------------------------------------------------
// adjoint of the all-pairs term: lanes own receivers i, partners stream
// ---------------------------------------------------------------------------
__device__ __forceinline__ void vjp_nonbond_block(const VjpNbArgs &a, int block, float4 *lds_ld)
{
    for (int t = threadIdx.x; t < a.T * a.T; t += kB) lds_ld[t] = a.ld[t];
    __syncthreads();
    const int4 bt = a.blocks[block];
    const WinDesc W = a.wins[bt.x];
    const int lane = (int)threadIdx.x % kWave;
    // read from the first lane, so the compiler knows it is wave-uniform
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int il = bt.y * kWave + lane;
    const int j0 = W.a0 + min(W.n, (kNbGroup * bt.z + wv) * W.apc);
    const int j1 = min(W.a0 + W.n, j0 + W.apc);
    const bool valid = il < W.n;
    const int i = W.a0 + (valid ? il : W.n - 1);
    const float4 xi = a.xq[i];
    const float4 auxi = a.aux[i];
    const int ti = __float_as_int(auxi.w);
    const float4 li4 = a.arec[4 * (size_t)i + 3];
    uint32_t ex[4];
    for (int k = 0; k < 4; ++k) ex[k] = a.excl[4 * i + k];
    const bool pbc = !a.pbc_flag || a.pbc_flag[bt.x] != 0;
    const MinImage mi = min_image_of(W.L, W.h);
    const int wave_lo = W.a0 + bt.y * kWave;
    const float4 *ldrow = lds_ld + ti * a.T;
    double qacc = 0.0, sacc = 0.0, eacc = 0.0;
    for (int jt = j0; jt < j1; jt += kTile) {
        const int je = min(j1, jt + kTile);
        const bool near = (jt < wave_lo + kWave + 64) && (je > wave_lo - 64);
        float qb = 0.0f, sb = 0.0f, eb = 0.0f;
        for (int j = jt; j < je; ++j) {
            const float4 xj = a.xq[j];  // wave-uniform
            const float4 auxj = a.aux[j];
            const float4 lj4 = a.arec[4 * (size_t)j + 3];
            float rx = xi.x - xj.x, ry = xi.y - xj.y, rz = xi.z - xj.z;
            if (pbc) {
                rx = min_image1(rx, mi);
                ry = min_image1(ry, mi);
                rz = min_image1(rz, mi);
            }
            const float d2 = dist2_f32(rx, ry, rz);
            const float inv = rsqrt_f32(d2);
            const float inv2 = inv * inv;
            const float d = d2 * inv;
            const float lri = __builtin_fmaf(li4.z, rz, __builtin_fmaf(li4.y, ry, li4.x * rx));
            const float lrj = __builtin_fmaf(lj4.z, rz, __builtin_fmaf(lj4.y, ry, lj4.x * rx));
            const float c = lri - lrj;
            bool excl = false;
            if (near) {
                const int w = j - i + 64;
                if (w >= 0 && w < 128) excl = (ex[w >> 5] >> (w & 31)) & 1u;
            }
            if (a.excl_ptr) {
                const int e0 = a.excl_ptr[i], e1 = a.excl_ptr[i + 1];
                for (int e = e0; e < e1; ++e) excl |= (a.excl_idx[e] == j);
            }
            const bool self = (j == i);
            // pair term phi(d, R): far -2 fep/(3 d^3), near cA + cB d
            const float phj = d2 > auxj.x ? a.cfar * inv2 * inv : __builtin_fmaf(auxj.z, d, auxj.y);
            const float phi = d2 > auxi.x ? a.cfar * inv2 * inv : __builtin_fmaf(auxi.z, d, auxi.y);
            float dq = xj.w * (lri * phj - lrj * phi);
            float ds = 0.0f, de = 0.0f;
            if (!excl) {
                const float4 pt = ldrow[__float_as_int(auxj.w)];
                const float r6 = inv2 * inv2 * inv2;
                ds = 0.5f * c * (12.0f * pt.z * r6 * r6 - 6.0f * pt.w * r6) * inv2;
                de = c * (12.0f * pt.x * r6 * r6 - 6.0f * pt.y * r6) * inv2;
                dq = __builtin_fmaf(c * xj.w, inv2 * inv, dq);
            }
            qb += self ? 0.0f : dq;
            sb += (self || excl) ? 0.0f : ds;
            eb += (self || excl) ? 0.0f : de;
        }
        qacc += (double)qb;
        sacc += (double)sb;
        eacc += (double)eb;
    }
    // the chunks' sums in order, as the forward blocks; every wave is done
    // with the table
    double *red = reinterpret_cast<double *>(lds_ld) + lane;
    __syncthreads();
    if (wv > 0) {
        double *d = red + (wv - 1) * 3 * kWave;
        d[0] = qacc;
        d[kWave] = sacc;
        d[2 * kWave] = eacc;
    }
    __syncthreads();
    if (wv > 0 || !valid) return;
    for (int w = 0; w < kNbGroup - 1; ++w) {
        const double *d = red + w * 3 * kWave;
        qacc += d[0];
        sacc += d[kWave];
        eacc += d[2 * kWave];
    }
    const long long o = W.npo + (long long)bt.z * W.n + il;
    a.part[o] = qacc;
    a.part[a.B + o] = sacc;
    a.part[2 * a.B + o] = eacc;
}

__global__ __launch_bounds__(kB) void k_vjp_epilogue(VjpArgs a)
{
    vjp_epilogue_block(a);
}

__global__ __launch_bounds__(kB) void k_vjp_nonbond(VjpNbArgs a)
{
    extern __shared__ __align__(16) float4 lds_ld[];
    vjp_nonbond_block(a, blockIdx.x, lds_ld);
}

// The epilogue with the all-pairs blocks behind its own where a block a CU
// holds both: each is a chain that leaves the chip idle (550 atoms: 7.4 us
// with 43 blocks and 8.7 with 81).
__global__ __launch_bounds__(kB) void k_vjp_epilogue_nonbond(VjpArgs a, VjpNbArgs n, int nepi)
{
    extern __shared__ __align__(16) float4 lds_ld[];
    if ((int)blockIdx.x < nepi)
        vjp_epilogue_block(a);
    else
        vjp_nonbond_block(n, (int)blockIdx.x - nepi, lds_ld);
}

// Per atom: the chunk partials + the direct charge term.  Latency bound like
// k_diff_reduce and split the same way, four entries in flight a slice: one lane per atom took 74.7 us at 550 atoms and
// 133 us for 32 x 1,100 atoms; now 9.2 and 24 us.
__global__ __launch_bounds__(kB) void k_vjp_finish(VjpFinishArgs a)
{
    __shared__ double red[kSumSlices][9][kSumAtoms];
    const int al = threadIdx.x % kSumAtoms, sl = threadIdx.x / kSumAtoms;
    const int i = blockIdx.x * kSumAtoms + al;
    const bool valid = i < a.n;
    double s[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};  // q, theta(5); nonbond q, sigma, eps
    if (valid) {
        const WinDesc W = window_of(a.wins, a.nwin, a.atom_win, i);
        const WinDesc Wn = window_of(a.nb_wins, a.nwin, a.atom_win, i);
        const int il = i - W.a0;
        sum_batches<6, 4>(PlanarEntry<6>{a.apart, a.C, W.vpo + il, W.n}, sl, W.vents, s);
        sum_batches<3, 4>(PlanarEntry<3>{a.nbpart, a.B, Wn.npo + il, Wn.n}, sl, Wn.nbc, s + 6);
    }
    combine_slices<9>(red, al, sl, s);
    if (sl != 0 || !valid) return;
    const int ti = a.itype[i];
    const double vt = a.vtot[ti];
    const double direct = -vt * (a.lam[3 * i] * a.se[3 * i] + a.lam[3 * i + 1] * a.se[3 * i + 1] +
                                 a.lam[3 * i + 2] * a.se[3 * i + 2]);
    a.gq[i] = s[0] + s[6] + direct;
    a.gatom[5 * i + 0] = s[1] + s[7];
    a.gatom[5 * i + 1] = s[2] + s[8] / (2.0 * a.theta[5 * ti + 1]);
    for (int k = 2; k < 5; ++k) a.gatom[5 * i + k] = s[1 + k];
}

// Per-type sums of the per-atom bars, FP64, fixed order: one block per type
// and atom range [kTypeRange b, kTypeRange (b + 1)), then, with more than one
// range, one block per type over the ranges.  Latency bound: a block that
// walks all 35,200 atoms of 32 x 1,100 alone takes 137 dependent rounds
// (81.6 us); in ranges it takes 7.7 + 4.6 us.
constexpr int kTypeRange = 2048;

__device__ __forceinline__ void type_tree(double (&red)[5][kB], const double (&s)[5])
{
    for (int k = 0; k < 5; ++k) red[k][threadIdx.x] = s[k];
    __syncthreads();
    for (int w = kB / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int k = 0; k < 5; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + w];
        __syncthreads();
    }
}

// out[(type * gridDim.y + range) * 5 + k]
__global__ __launch_bounds__(kB) void k_type_reduce(const double *__restrict__ gatom,
                                                    const int *__restrict__ itype, int n,
                                                    double *out)
{
    __shared__ double red[5][kB];
    const int t = blockIdx.x;
    double s[5] = {0, 0, 0, 0, 0};
    const int i0 = blockIdx.y * kTypeRange + threadIdx.x;
#pragma unroll
    for (int u = 0; u < kTypeRange / kB; ++u) {
        const int i = i0 + u * kB;
        if (i < n && itype[i] == t)
            for (int k = 0; k < 5; ++k) s[k] += gatom[5 * (size_t)i + k];
    }
    type_tree(red, s);
    if (threadIdx.x < 5)
        out[5 * ((size_t)t * gridDim.y + blockIdx.y) + threadIdx.x] = red[threadIdx.x][0];
}

__global__ __launch_bounds__(kB) void k_type_sum(const double *__restrict__ part, int ranges,
                                                 double *gtheta)
{
    __shared__ double red[5][kB];
    const int t = blockIdx.x;
    double s[5] = {0, 0, 0, 0, 0};
    for (int r = threadIdx.x; r < ranges; r += kB)
        for (int k = 0; k < 5; ++k) s[k] += part[5 * ((size_t)t * ranges + r) + k];
    type_tree(red, s);
    if (threadIdx.x < 5) gtheta[5 * t + threadIdx.x] = red[threadIdx.x][0];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_diff_prep(const DiffPrepArgs &t, const DiffAtomArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(k_diff_prep, dim3(1 + nblk(a.n)), dim3(kB), 0, s, t, a);
    return hipGetLastError();
}

hipError_t launch_diff_reduce(const DiffReduceArgs &a, hipStream_t s)
{
    if (a.n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_diff_reduce, dim3((a.n + kSumAtoms - 1) / kSumAtoms), dim3(kB), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_vjp_points(const VjpArgs &a, int nblocks, hipStream_t s)
{
    if (nblocks == 0) return hipSuccess;
    VjpArgs b = a;
    b.ranked_from = ranked_from(nblocks);
    hipLaunchKernelGGL(k_vjp_points, dim3(nblocks), dim3(kB), 0, s, b);
    return hipGetLastError();
}

// the point epilogue and the all-pairs adjoint, in one launch up to a block a CU
hipError_t launch_vjp_epilogue_nonbond(const VjpArgs &a, const VjpNbArgs &n, int nb_blocks,
                                       hipStream_t s)
{
    const int nepi = nblk(a.Ptot);
    const size_t lds = std::max(sizeof(float4) * n.T * n.T, nonbond_share_bytes(3));
    if (nepi + nb_blocks <= 256) {
        if (nepi + nb_blocks > 0)
            hipLaunchKernelGGL(k_vjp_epilogue_nonbond, dim3(nepi + nb_blocks), dim3(kB), lds, s, a,
                               n, nepi);
        return hipGetLastError();
    }
    if (nepi > 0) hipLaunchKernelGGL(k_vjp_epilogue, dim3(nepi), dim3(kB), 0, s, a);
    if (nb_blocks > 0) hipLaunchKernelGGL(k_vjp_nonbond, dim3(nb_blocks), dim3(kB), lds, s, n);
    return hipGetLastError();
}

hipError_t launch_vjp_atoms(const VjpArgs &a, int nblocks, hipStream_t s)
{
    if (nblocks == 0) return hipSuccess;
    VjpArgs b = a;
    b.ranked_from = ranked_from(nblocks);
    hipLaunchKernelGGL(k_vjp_atoms, dim3(nblocks), dim3(kB), 0, s, b);
    return hipGetLastError();
}

hipError_t launch_vjp_finish(const VjpFinishArgs &a, hipStream_t s)
{
    if (a.n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_vjp_finish, dim3((a.n + kSumAtoms - 1) / kSumAtoms), dim3(kB), 0, s, a);
    return hipGetLastError();
}

int type_reduce_ranges(int n) { return std::max(1, (n + kTypeRange - 1) / kTypeRange); }

hipError_t launch_type_reduce(const double *gatom, const int *itype, int n, int T, double *part,
                              double *gtheta, hipStream_t s)
{
    if (T == 0) return hipSuccess;
    const int ranges = type_reduce_ranges(n);
    hipLaunchKernelGGL(k_type_reduce, dim3(T, ranges), dim3(kB), 0, s, gatom, itype, n,
                       ranges > 1 ? part : gtheta);
    if (ranges > 1)
        hipLaunchKernelGGL(k_type_sum, dim3(T), dim3(kB), 0, s, part, ranges, gtheta);
    return hipGetLastError();
}

}  // namespace isspa
