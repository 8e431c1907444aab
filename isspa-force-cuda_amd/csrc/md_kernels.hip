// Nonbond, bonded, integrator, restraint and utility kernels for gfx950.
//
// Semantics follow the reference kernels cited at each function; the
// decomposition is this engine's own: one lane per receiving atom with a
// wave-uniform partner stream for the all-pairs term, per-term contribution
// slots plus a per-atom gather for the bonded terms (no float atomics), and
// single-workgroup FP64 tree reductions for the umbrella centres of mass.
// The all-pairs, integrator and restraint kernels are window-aware (kernels.hpp).
#include <algorithm>

#include "device_common.hpp"
#include "kernels.hpp"
#include "pbc_device.hpp"
#include "reduce_device.hpp"
#include "points_device.hpp"
#include "nonbond_device.hpp"
#include "bonded_device.hpp"

namespace isspa {

constexpr int kBlk = 256;
static inline int nblocks(long long n) { return (int)((n + kBlk - 1) / kBlk); }

template <bool SPLIT>
__global__ __launch_bounds__(kBlk) void k_nonbond(NonbondArgs a)
{
    extern __shared__ float2 lds_lj[];
    nonbond_block<SPLIT, !SPLIT, false>(a, blockIdx.x, lds_lj);
}

hipError_t launch_nonbond(const NonbondArgs &a, int nb, bool split, hipStream_t s)
{
    if (nb == 0) return hipSuccess;
    const size_t lds = nonbond_lds_bytes(a.T, a.sym != 0, split);
    if (split)
        hipLaunchKernelGGL(k_nonbond<true>, dim3(nb), dim3(kBlk), lds, s, a);
    else
        hipLaunchKernelGGL(k_nonbond<false>, dim3(nb), dim3(kBlk), lds, s, a);
    return hipGetLastError();
}

// sum [comps][B] partials over the window's groups of partner chunks in the fixed
// slice order of reduce_device.hpp; comps == 3: f += sum; comps == 9: three FP64
// outputs.  FEW: an atom a work-item (few_entries).
template <int COMPS, bool FEW>
__global__ __launch_bounds__(kBlk) void k_chunk_reduce3(const WinDesc *__restrict__ wins,
                                                        int nwin,
                                                        const int *__restrict__ atom_win,
                                                        const double *__restrict__ part,
                                                        long long B, int ntot, float4 *f,
                                                        double *o0, double *o1, double *o2)
{
    constexpr int kAtoms = FEW ? kBlk : kSumAtoms;
    const int al = threadIdx.x % kAtoms, sl = threadIdx.x / kAtoms;
    const int i = blockIdx.x * kAtoms + al;
    const bool valid = i < ntot;
    double s[COMPS];
    for (int k = 0; k < COMPS; ++k) s[k] = 0.0;
    if (valid) {
        const WinDesc W = window_of(wins, nwin, atom_win, i);
        sum_batches<COMPS, FEW ? kFewBatch : 4, FEW ? 1 : kSumSlices>(nonbond_entry<COMPS>(W, part, B, i), sl,
                                                    COMPS == 3 ? W.nte : W.nbc, s);
    }
    if constexpr (!FEW) {
        __shared__ double red[kSumSlices][COMPS][kSumAtoms];
        combine_slices<COMPS>(red, al, sl, s);
    }
    if (sl != 0 || !valid) return;
    if constexpr (COMPS == 3) {
        float4 v = f[i];
        v.x += (float)s[0];
        v.y += (float)s[1];
        v.z += (float)s[2];
        f[i] = v;
    } else {
        for (int k = 0; k < 3; ++k) {
            o0[3 * i + k] = s[k];
            o1[3 * i + k] = s[3 + k];
            o2[3 * i + k] = s[6 + k];
        }
    }
}

hipError_t launch_chunk_reduce3(const WinDesc *wins, int nwin, const int *atom_win,
                                const double *part, long long B, int max_entries, int ntot,
                                int comps, float4 *f, double *o0, double *o1, double *o2,
                                hipStream_t s)
{
    if (ntot == 0) return hipSuccess;
    const bool few = few_entries(max_entries, ntot);
    const int atoms = few ? kBlk : kSumAtoms;
    const dim3 g((ntot + atoms - 1) / atoms), t(kBlk);
#define REDUCE(C, F) \
    hipLaunchKernelGGL((k_chunk_reduce3<C, F>), g, t, 0, s, wins, nwin, atom_win, part, B, ntot, f, o0, o1, o2)
    switch ((few ? 2 : 0) + (comps == 3 ? 0 : 1)) {
    case 0: REDUCE(3, false); break;
    case 1: REDUCE(9, false); break;
    case 2: REDUCE(3, true); break;
    default: REDUCE(9, true); break;
    }
#undef REDUCE
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// bonded terms.  Each term writes its per-atom forces into fixed contribution
// slots; k_bonded_gather sums each atom's slots in FP64 in a fixed order.
// Slot layout: bonds [0, 2nb), angles [2nb, 2nb+3na), dihedrals 6 per term
// (atoms i, j, k, l, then the 1-4 pair's i and l).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlk) void k_bonded_terms(BondedArgs a)
{
    bonded_one(a, blockIdx.x * kBlk + threadIdx.x);
}

hipError_t launch_bonded_terms(const BondedArgs &a, hipStream_t s)
{
    const long n = (long)a.nb + a.na + a.nd;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_bonded_terms, dim3(nblocks(n)), dim3(kBlk), 0, s, a);
    return hipGetLastError();
}

// One energy of n terms, stride apart: a work-item's terms in order, four loads
// in flight
template <int COMPS>
__device__ __forceinline__ void energy_terms(const double *__restrict__ e, int n, double *acc)
{
    constexpr int kU = 4;
    for (int q0 = threadIdx.x; q0 < n; q0 += kU * kBlk) {
        double v[kU][COMPS];
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int k = 0; k < COMPS; ++k)
                v[u][k] = e[COMPS * (size_t)min(q0 + u * kBlk, n - 1) + k];
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int k = 0; k < COMPS; ++k) acc[k] += q0 + u * kBlk < n ? v[u][k] : 0.0;
    }
}

// energies: bond, angle, torsion, 1-4 Coulomb, 1-4 LJ (one workgroup, fixed tree)
__device__ __forceinline__ void bonded_energy_block(const double *__restrict__ e, int nb, int na,
                                                    int nd, double *out, double (*red)[kBlk])
{
    double acc[5] = {0, 0, 0, 0, 0};
    energy_terms<1>(e, nb, acc);
    energy_terms<1>(e + nb, na, acc + 1);
    energy_terms<3>(e + (size_t)nb + na, nd, acc + 2);
    for (int k = 0; k < 5; ++k) red[k][threadIdx.x] = acc[k];
    __syncthreads();
    for (int w = kBlk / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int k = 0; k < 5; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int k = 0; k < 5; ++k) out[k] = red[k][0];
}

// A block owns kSumAtoms atoms and kSumSlices slot slices: slice t sums slots
// t, t + S, ... of its atom in order, then the slices are added in order (a
// fixed order independent of scheduling, with S times the waves of one lane
// per atom).  With g.energy the first block sums the energies instead: like the
// gather they need the terms only, and a launch of their own took 4.7 us
// behind the gather's 3.2 (550 atoms; the loop of separate calls 69.5 -> 65.9 us).
__global__ __launch_bounds__(kBlk) void k_bonded_gather(BondedSumArgs g)
{
    __shared__ double lds[5 * kBlk];
    static_assert(5 * kBlk >= kSumSlices * 3 * kSumAtoms, "both sums fit");
    int b = blockIdx.x;
    if (g.energy) {
        if (b == 0) {
            bonded_energy_block(g.eterm, g.nb, g.na, g.nd, g.energy,
                                reinterpret_cast<double (*)[kBlk]>(lds));
            return;
        }
        --b;
    }
    auto &red = *reinterpret_cast<double (*)[kSumSlices][3][kSumAtoms]>(lds);
    const int al = threadIdx.x % kSumAtoms, sl = threadIdx.x / kSumAtoms;
    const int i = b * kSumAtoms + al;
    const bool valid = i < g.n;
    double s[3] = {0.0, 0.0, 0.0};
    if (valid) bonded_sum(g.contrib, g.idx, g.ptr[i] + sl, g.ptr[i + 1], s);
    combine_slices<3>(red, al, sl, s);
    if (sl != 0 || !valid) return;
    float4 v = g.f[i];
    v.x += (float)s[0];
    v.y += (float)s[1];
    v.z += (float)s[2];
    g.f[i] = v;
}

hipError_t launch_bonded_gather(const BondedSumArgs &g, hipStream_t s)
{
    const int grid = (g.n + kSumAtoms - 1) / kSumAtoms + (g.energy ? 1 : 0);
    if (grid == 0) return hipSuccess;
    hipLaunchKernelGGL(k_bonded_gather, dim3(grid), dim3(kBlk), 0, s, g);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// A.15 leap-frog + Andersen (src/leapfrog_cuda.cu:33-67).  On a collision the
// velocity is redrawn from Maxwell-Boltzmann, then half-kicked (quirk Q21).
// Atom i of window w draws with counter {i - a0_w, draw, step, sys_w}.
// ---------------------------------------------------------------------------
// atom i of window W: position x and velocity v before, collision draw o
__device__ __forceinline__ uint4 collision_draw(const WinDesc &W, int i, uint64_t seed,
                                                uint32_t step)
{
    return philox_draw(seed, (uint32_t)(i - W.a0), kStreamAndersen, 0u, step, W.sys);
}
__device__ __forceinline__ void leapfrog_atom(const WinDesc &W, int i, float4 x, float4 v, uint4 o,
                                              float4 *xyzq, float4 *vel, const float4 fi, float kT,
                                              float dt, uint32_t thr, uint64_t seed, uint32_t step)
{
    const uint32_t il = (uint32_t)(i - W.a0);
    const float m = v.w;
    if (o.x < thr) {
        const uint4 z = philox_draw(seed, il, kStreamAndersen, 1u, step, W.sys);
        const float s24 = 5.9604644775390625e-08f;
        const float u1a = (float)((z.x >> 8) + 1u) * s24, u2a = (float)(z.y >> 8) * s24;
        const float u1b = (float)((z.z >> 8) + 1u) * s24, u2b = (float)(z.w >> 8) * s24;
        const float ra = sqrtf(-2.0f * logf(u1a)), rb = sqrtf(-2.0f * logf(u1b));
        const float twopi = 6.283185307179586f;
        const float sc = sqrtf(kT / m);
        const float hk = dt / (m * 2.0f);
        v.x = ra * cosf(twopi * u2a) * sc + fi.x * hk;
        v.y = ra * sinf(twopi * u2a) * sc + fi.y * hk;
        v.z = rb * cosf(twopi * u2b) * sc + fi.z * hk;
    } else {
        const float kk = dt / m;
        v.x += fi.x * kk;
        v.y += fi.y * kk;
        v.z += fi.z * kk;
    }
    x.x += v.x * dt;
    x.y += v.y * dt;
    x.z += v.z * dt;
    // wrap (src/cuda_vector_routines.h:49-68)
    const float L = W.L;
    x.x = x.x > L ? x.x - L : (x.x < 0.0f ? x.x + L : x.x);
    x.y = x.y > L ? x.y - L : (x.y < 0.0f ? x.y + L : x.y);
    x.z = x.z > L ? x.z - L : (x.z < 0.0f ? x.z + L : x.z);
    vel[i] = v;
    xyzq[i] = x;
}

__global__ __launch_bounds__(kBlk) void k_leapfrog(const WinDesc *__restrict__ wins,
                                                   const int *__restrict__ atom_win, WinDesc one,
                                                   int ntot,
                                                   float4 *xyzq, float4 *vel,
                                                   const float4 *__restrict__ f, float kT,
                                                   float dt, uint32_t thr, uint64_t seed,
                                                   uint32_t step_arg,
                                                   const uint32_t *step_d)
{
    const int i = blockIdx.x * kBlk + threadIdx.x;
    const uint32_t step = step_d ? *step_d : step_arg;
    if (i >= ntot) return;
    const WinDesc W = atom_win ? wins[atom_win[i]] : one;
    leapfrog_atom(W, i, xyzq[i], vel[i], collision_draw(W, i, seed, step), xyzq, vel, f[i], kT, dt,
                  thr, seed, step);
}

hipError_t launch_leapfrog(const WinDesc *wins, const int *atom_win, const WinDesc &one,
                           int ntot, float4 *xyzq, float4 *vel, const float4 *f, float kT,
                           float dt, uint32_t thr, uint64_t seed, uint32_t step,
                           const uint32_t *step_d, hipStream_t s)
{
    if (ntot == 0) return hipSuccess;
    hipLaunchKernelGGL(k_leapfrog, dim3(nblocks(ntot)), dim3(kBlk), 0, s, wins, atom_win, one, ntot,
                       xyzq, vel, f, kT, dt, thr, seed, step, step_d);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The MD engine's per-step force: f = ((bonded + IS-SPA) + all-pairs) per atom,
// plus the restraint force of restrained atoms.  Each term is summed by the
// same helper and in the same order as its own reduction kernel and added in
// the order the separate calls add them into a zeroed f, so the result equals
// zero + gather + IS-SPA reduction + chunk reduction + restraint bit for bit,
// in one launch.  With lf.xyzq the same thread then integrates its atom
// (leap-frog + Andersen, as k_leapfrog) and the first block advances the step,
// so a whole step ends with this launch.
//
// Bounded by the latency of dependent loads, so the loads of all terms are
// issued level by level before any of them is used: the windows, slot ranges
// and the atom's own data; then the first batch of each term's entries; then
// the bonded contributions.  Whole steps, against one term after the other in
// 32 atoms x 8 slices and a step counter that the last finished block moved
// on: 44 atoms 28.9 -> 26.3 us, 1,100 atoms 92.2 -> 89.4 us, 64 windows 70.2
// -> 66.2 us, 19,998 atoms 8.00 -> 7.99 ms.  Held to 128 VGPRs it spills, and
// a launch with scratch starts later: 30.2 us at 44 atoms.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlk) void k_assemble_forces(AssembleArgs a)
{
    constexpr int nc = 12;  // bonded xyz, IS-SPA 6, all-pairs xyz
    constexpr int kBI = 6, kBN = 5;
    __shared__ double red[kSumSlices][nc][kSumAtoms];
    const int al = threadIdx.x % kSumAtoms, sl = threadIdx.x / kSumAtoms;
    const int ia = blockIdx.x * kSumAtoms + al;
    const bool valid = ia < a.n;
    const int i = valid ? ia : a.n - 1;  // idle work-items mirror the last atom
    // level 1
    const uint32_t step = a.lf.step_d ? a.lf.step_d[kStepNow] : 0u;
    WinDesc Wi{}, Wn{}, Wl{};
    if (a.isspa.part) Wi = window_of(a.isspa.wins, a.isspa.nwin, a.isspa.atom_win, i);
    if (a.nb_part) Wn = window_of(a.nb_wins, a.nb_nwin, a.nb_atom_win, i);
    int e0 = 0, e1 = 0;
    if (a.contrib) {
        e0 = a.gptr[i] + sl;
        e1 = a.gptr[i + 1];
    }
    float4 x = make_float4(0.0f, 0.0f, 0.0f, 0.0f), v = x, u = x;
    float vtot = 0.0f;
    uint4 draw = make_uint4(0u, 0u, 0u, 0u);
    if (sl == 0) {
        if (a.lf.xyzq) {
            Wl = window_of(a.lf.wins, a.lf.nwin, a.lf.atom_win, i);
            v = a.lf.vel[i];
        }
        if (a.fus) u = a.fus[i];
        if (a.isspa.part) {
            x = a.isspa.xyzq[i];
            vtot = a.isspa.vtot[a.isspa.itype[i]];
        } else if (a.lf.xyzq) {
            x = a.lf.xyzq[i];
        }
    }
    // level 2
    const ForceEntry<6> ei(Wi, a.isspa.part, i);
    const PlanarEntry<3> en = nonbond_entry<3>(Wn, a.nb_part, a.nb_B, i);
    double vi[kBI][6], vn[kBN][3];
    BondBatch bb;
    const bool hi = sl < Wi.fents, hn = sl < Wn.nte, hb = e0 < e1;
    if (hi) load_batch<6, kBI>(ei, sl, Wi.fents, vi);
    if (hn) load_batch<3, kBN>(en, sl, Wn.nte, vn);
    if (hb) bonded_load_idx(a.gidx, e0, e1, bb);
    if (sl == 0 && a.lf.xyzq) draw = collision_draw(Wl, i, a.lf.seed, step);
    // level 3
    if (hb) bonded_load(a.contrib, bb);
    double s[nc];
    for (int k = 0; k < nc; ++k) s[k] = 0.0;
    if (hi) {
        add_batch<6, kBI>(sl, Wi.fents, vi, s + 3);
        sum_batches<6, kBI>(ei, sl + kBI * kSumSlices, Wi.fents, s + 3);
    }
    if (hn) {
        add_batch<3, kBN>(sl, Wn.nte, vn, s + 9);
        sum_batches<3, kBN>(en, sl + kBN * kSumSlices, Wn.nte, s + 9);
    }
    if (hb) {
        bonded_add(e0, e1, bb, s);
        bonded_sum(a.contrib, a.gidx, e0 + kBondBatch * kSumSlices, e1, s);
    }
    combine_slices<nc>(red, al, sl, s);
    if (sl == 0 && valid) {
        float4 f = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (a.contrib) {
            f.x += (float)s[0];
            f.y += (float)s[1];
            f.z += (float)s[2];
        }
        if (a.isspa.part) {
            const float3 fi = isspa_atom_force(x.w, vtot, s + 3);
            f.x += fi.x;
            f.y += fi.y;
            f.z += fi.z;
        }
        if (a.nb_part) {
            f.x += (float)s[9];
            f.y += (float)s[10];
            f.z += (float)s[11];
        }
        if (a.fus && u.w != 0.0f) {
            f.x += u.x;
            f.y += u.y;
            f.z += u.z;
        }
        a.f[i] = f;
        if (a.lf.xyzq)
            leapfrog_atom(Wl, i, x, v, draw, a.lf.xyzq, a.lf.vel, f, a.lf.kT, a.lf.dt, a.lf.thr,
                          a.lf.seed, step);
    }
    if (a.lf.step_d && blockIdx.x == 0 && threadIdx.x == 0) a.lf.step_d[kStepNext] = step + 1u;
}

hipError_t launch_assemble_forces(const AssembleArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(k_assemble_forces, dim3((a.n + kSumAtoms - 1) / kSumAtoms), dim3(kBlk), 0,
                       s, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// A.16 umbrella restraint (src/us_force_cuda.cu:14-47).  One workgroup per
// restraint: the two centres of mass by an FP64 tree reduction (the
// reference synchronises only within a block, quirk Q12), then each bias
// atom's force.  Atoms in a restraint are unique, so the updates do not race.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlk) void k_us(const int *__restrict__ boff,
                                             const int2 *__restrict__ atoms,
                                             const float *__restrict__ mass,
                                             const float2 *__restrict__ kx,
                                             const float *__restrict__ Ls,
                                             const float4 *__restrict__ xyzq, float4 *f,
                                             double *com)
{
    __shared__ double red[6][kTermBlock];
    us_block(blockIdx.x, boff, atoms, mass, kx, Ls, xyzq, f, com, false, red);
}

hipError_t launch_us(int nres, const int *boff, const int2 *atoms, const float *mass,
                     const float2 *kx, const float *L, const float4 *xyzq, float4 *f, double *com,
                     hipStream_t s)
{
    if (nres == 0) return hipSuccess;
    hipLaunchKernelGGL(k_us, dim3(nres), dim3(kBlk), 0, s, boff, atoms, mass, kx, L, xyzq, f, com);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// MD engine step prologue: what of a step depends only on the coordinates and
// does not ride on the epilogue, as block ranges of one grid -- minimum-image
// flags (one block per window), bonded terms (256 terms a block), restraints
// (one block each, bias forces stored for the force assembly) and the MC points.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlk) void k_step_prologue(PrologueArgs a)
{
    int b = blockIdx.x;
    if (b == 0 && threadIdx.x == 0) a.step_d[kStepNow] = a.step_d[kStepNext];
    if (b < a.nflag) {
        const WinDesc W = a.pts.wins[b];
        pbc_flag_block(W, a.pts.xyzq, a.rmax_all, a.flag + b);
        return;
    }
    b -= a.nflag;
    if (b < a.bonded_blocks) {
        bonded_one(a.bonded, b * kBlk + (int)threadIdx.x);
        return;
    }
    b -= a.bonded_blocks;
    if (b < a.us.nres) {
        __shared__ double red[6][kTermBlock];
        us_block(b, a.us.boff, a.us.us_atoms, a.us.us_mass, a.us.kx, a.us.Ls, a.pts.xyzq, a.us.fus,
                 a.us.com, true, red);
        return;
    }
    b -= a.us.nres;
    if ((long long)a.pts.ntot * a.pts.nmc > 0) mc_points_block(a.pts, b);
}

hipError_t launch_step_prologue(PrologueArgs a, hipStream_t s)
{
    const long nterms = (long)a.bonded.nb + a.bonded.na + a.bonded.nd;
    a.bonded_blocks = a.bonded.contrib ? nblocks(nterms) : 0;
    const long long P = (long long)a.pts.ntot * a.pts.nmc;
    const long long grid = (long long)a.nflag + a.bonded_blocks + a.us.nres + (P + kMcBlockPts - 1) / kMcBlockPts;
    // at least one block: the first one hands the step on
    hipLaunchKernelGGL(k_step_prologue, dim3((unsigned)std::max(grid, 1LL)), dim3(kBlk), 0, s, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// utilities
// ---------------------------------------------------------------------------
// flag[w] for every window w: one block per window
__global__ __launch_bounds__(256) void k_pbc_flag(const WinDesc *__restrict__ wins,
                                                  const float4 *__restrict__ xyzq,
                                                  float rmax_all, int *flag)
{
    const WinDesc W = wins[blockIdx.x];
    pbc_flag_block(W, xyzq, rmax_all, flag + blockIdx.x);
}

hipError_t launch_pbc_flag(const WinDesc *wins, int W, const float4 *xyzq, float rmax_all,
                           int *flag, hipStream_t s)
{
    if (W == 0) return hipSuccess;
    hipLaunchKernelGGL(k_pbc_flag, dim3(W), dim3(256), 0, s, wins, xyzq, rmax_all, flag);
    return hipGetLastError();
}

__global__ void k_zero16(uint4 *p, size_t n16)
{
    for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < n16;
         k += (size_t)gridDim.x * blockDim.x)
        p[k] = make_uint4(0u, 0u, 0u, 0u);
}
__global__ void k_zero1(unsigned char *p, size_t n)
{
    for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < n;
         k += (size_t)gridDim.x * blockDim.x)
        p[k] = 0;
}

hipError_t launch_zero(void *p, size_t bytes, hipStream_t s)
{
    if (bytes == 0) return hipSuccess;
    if (((uintptr_t)p & 15u) == 0 && (bytes & 15u) == 0) {
        const size_t n16 = bytes / 16;
        const int g = (int)std::min<size_t>(4096, (n16 + kBlk - 1) / kBlk);
        hipLaunchKernelGGL(k_zero16, dim3(g), dim3(kBlk), 0, s, (uint4 *)p, n16);
    } else {
        const int g = (int)std::min<size_t>(4096, (bytes + kBlk - 1) / kBlk);
        hipLaunchKernelGGL(k_zero1, dim3(g), dim3(kBlk), 0, s, (unsigned char *)p, bytes);
    }
    return hipGetLastError();
}

__global__ __launch_bounds__(kBlk) void k_add4(float4 *dst, const float4 *__restrict__ src, int n)
{
    const int i = blockIdx.x * kBlk + threadIdx.x;
    if (i >= n) return;
    float4 d = dst[i];
    const float4 s = src[i];
    d.x += s.x;
    d.y += s.y;
    d.z += s.z;
    dst[i] = d;
}

hipError_t launch_add4(float4 *dst, const float4 *src, int n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_add4, dim3(nblocks(n)), dim3(kBlk), 0, s, dst, src, n);
    return hipGetLastError();
}

__global__ void k_set_word(uint32_t *dst, uint32_t v) { *dst = v; }

hipError_t launch_set_word(uint32_t *dst, uint32_t v, hipStream_t s)
{
    hipLaunchKernelGGL(k_set_word, dim3(1), dim3(1), 0, s, dst, v);
    return hipGetLastError();
}

}  // namespace isspa
