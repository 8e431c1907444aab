// Fixed-order per-atom sums shared by the reduction kernels: the IS-SPA chunk
// reduction, the bonded gather, the all-pairs chunk reduction and the MD
// engine's force assembly, which does all three in one launch.  Each kernel
// that sums a term calls the same helper, so a term's per-atom sum has the
// same operations in the same order whichever kernel computes it.
#pragma once

#include "kernels.hpp"

namespace isspa {

// A 256-thread reduction block owns kSumAtoms atoms and kSumSlices slices of
// each atom's list: slice t takes entries t, t + S, t + 2S, ... in order, and
// slice 0 then adds slices 1..S-1 in order.  The sums are bounded by the
// latency of a few dependent loads, so the slices are many and short: with 16
// slices the 60 or so entries of a large system are one batch of loads a
// slice.  (32 atoms x 8 slices: the reduction of 44 atoms over 677 entries
// took 16.1 us, the solvent force of which it is a part 45.8, now 40.4 us;
// the all-pairs force of 2,222 atoms 25.7, now 22.3 us.)
constexpr int kSumAtoms = 16;
constexpr int kSumSlices = 16;

// Every slice's sums into slice 0, added in slice order (slice 0's value,
// then slices 1, 2, ...).  Component k is added up by the work-items of slice
// k mod kSumSlices, so each chain of LDS reads is kSumSlices long rather than
// (kSumSlices - 1) x NC in slice 0 alone; each sum has the same additions in
// the same order, so the same bits.  Every work-item of the block calls it
// (two barriers).
template <int NC>
__device__ __forceinline__ void combine_slices(double (&red)[kSumSlices][NC][kSumAtoms], int al,
                                               int sl, double (&s)[NC])
{
#pragma unroll
    for (int k = 0; k < NC; ++k) red[sl][k][al] = s[k];
    __syncthreads();
    for (int k = sl; k < NC; k += kSumSlices) {
        double v[kSumSlices];
#pragma unroll
        for (int t = 0; t < kSumSlices; ++t) v[t] = red[t][k][al];
        double acc = v[0];
#pragma unroll
        for (int t = 1; t < kSumSlices; ++t) acc += v[t];
        red[0][k][al] = acc;
    }
    __syncthreads();
    if (sl == 0)
#pragma unroll
        for (int k = 0; k < NC; ++k) s[k] = red[0][k][al];
}

// the window of atom i; one window needs no lookup
__device__ __forceinline__ WinDesc window_of(const WinDesc *__restrict__ wins, int nwin,
                                             const int *__restrict__ atom_win, int i)
{
    return nwin == 1 ? wins[0] : wins[atom_win[i]];
}

// One batch of a slice's entries: entries c, c + S, ... (B of them, those
// below n), the loads of all of them issued before the first is used.  The
// missing ones read entry n - 1 again and count as zero, so the last batch
// waits once, as every other.  load(entry, v) reads an entry's COMPS values.
// S = 1: one slice, every entry in turn.
template <int COMPS, int B, int S = kSumSlices, typename Load>
__device__ __forceinline__ void load_batch(Load load, int c, int n, double (&v)[B][COMPS])
{
#pragma unroll
    for (int u = 0; u < B; ++u) load(min(c + u * S, n - 1), v[u]);
}
template <int COMPS, int B, int S = kSumSlices>
__device__ __forceinline__ void add_batch(int c, int n, const double (&v)[B][COMPS], double *s)
{
#pragma unroll
    for (int u = 0; u < B; ++u) {
        const bool in = c + u * S < n;
#pragma unroll
        for (int k = 0; k < COMPS; ++k) s[k] += in ? v[u][k] : 0.0;
    }
}
template <int COMPS, int B, int S = kSumSlices, typename Load>
__device__ __forceinline__ void sum_batches(Load load, int c, int n, double *s)
{
    for (; c < n; c += B * S) {
        double v[B][COMPS];
        load_batch<COMPS, B, S>(load, c, n, v);
        add_batch<COMPS, B, S>(c, n, v, s);
    }
}

// Sums of few entries for many atoms: one work-item an atom, kFewBatch entries in
// flight.  With at most kSumSlices entries a slice holds one entry or none, so the
// entries in turn give the slices' sum bit for bit; and most of sixteen work-items an
// atom would have nothing to read, behind two barriers.  From 8,192 atoms on the atoms
// alone hide the latency: the force reduction of 3,520 atoms and 16 entries takes 4.2 us
// so and 3.5 in slices, of 8,800 atoms 4.2 and 4.8 (one entry 3.0 and 3.5), of 160,600
// atoms and 4 entries 7.1 and 25.7, of 440,000 atoms 17.7 (4.8 TB/s) and 66.6; components
// of 160,600 atoms 227 and 266 us a call.
constexpr int kFewAtoms = 8192, kFewBatch = 4;
inline bool few_entries(int entries, int atoms)
{
    return entries <= kSumSlices && atoms >= kFewAtoms;
}

// Reads the COMPS components (6, or 9 in split mode) of the force partial of
// (entry, atom i of window W), stored as double2 pairs.
template <int COMPS>
struct ForceEntry {
    const double2 *part;
    long long base, n;
    __device__ __forceinline__ ForceEntry(const WinDesc &W, const double *p, int i)
        : part(reinterpret_cast<const double2 *>(p)), base(W.ppo + (i - W.a0)), n(W.n)
    {
    }
    __device__ __forceinline__ void operator()(int c, double (&v)[COMPS]) const
    {
        const double2 *e = part + (base + c * n) * (force_part_stride(COMPS == 9) / 2);
#pragma unroll
        for (int h = 0; h < (COMPS + 1) / 2; ++h) {
            const double2 d = e[h];
            v[2 * h] = d.x;
            if (2 * h + 1 < COMPS) v[2 * h + 1] = d.y;
        }
    }
};

// Reads COMPS component-major partials [COMPS][stride] of entry c, n apart.
template <int COMPS>
struct PlanarEntry {
    const double *part;
    long long stride, base, n;
    __device__ __forceinline__ void operator()(int c, double (&v)[COMPS]) const
    {
#pragma unroll
        for (int k = 0; k < COMPS; ++k) v[k] = part[k * stride + base + c * n];
    }
};

// all-pairs partials of atom i (COMPS = 3: the total force, entries of the
// total-force layout; 9: the split components, one per group of partner chunks)
template <int COMPS>
__device__ __forceinline__ PlanarEntry<COMPS> nonbond_entry(const WinDesc &W, const double *part,
                                                            long long B, int i)
{
    return PlanarEntry<COMPS>{part, B, (COMPS == 3 ? W.spo : W.npo) + (i - W.a0), W.n};
}

// F_i = -q_i vtot_i S_e - vtot_i S_lj from the summed IS-SPA partials
__device__ __forceinline__ float3 isspa_atom_force(float q, float vtot, const double *s)
{
    const double vt = (double)vtot;
    const double qv = -(double)q * vt;
    return make_float3((float)(qv * s[0] - vt * s[3]), (float)(qv * s[1] - vt * s[4]),
                       (float)(qv * s[2] - vt * s[5]));
}

// bonded contribution slots [e0, e1) of an atom, slots e0 + sl, + kSumSlices,
// ...: the indices of a batch, then its contributions
constexpr int kBondBatch = 4;
struct BondBatch {
    int idx[kBondBatch];
    float4 c[kBondBatch];
};
__device__ __forceinline__ void bonded_load_idx(const int *__restrict__ idx, int e, int e1,
                                                BondBatch &b)
{
#pragma unroll
    for (int u = 0; u < kBondBatch; ++u) b.idx[u] = idx[max(0, min(e + u * kSumSlices, e1 - 1))];
}
__device__ __forceinline__ void bonded_load(const float4 *__restrict__ contrib, BondBatch &b)
{
#pragma unroll
    for (int u = 0; u < kBondBatch; ++u) b.c[u] = contrib[b.idx[u]];
}
__device__ __forceinline__ void bonded_add(int e, int e1, const BondBatch &b, double *s)
{
#pragma unroll
    for (int u = 0; u < kBondBatch; ++u) {
        const bool in = e + u * kSumSlices < e1;
        s[0] += in ? (double)b.c[u].x : 0.0;
        s[1] += in ? (double)b.c[u].y : 0.0;
        s[2] += in ? (double)b.c[u].z : 0.0;
    }
}
__device__ __forceinline__ void bonded_sum(const float4 *__restrict__ contrib,
                                           const int *__restrict__ idx, int e, int e1, double *s)
{
    for (; e < e1; e += kBondBatch * kSumSlices) {
        BondBatch b;
        bonded_load_idx(idx, e, e1, b);
        bonded_load(contrib, b);
        bonded_add(e, e1, b, s);
    }
}

}  // namespace isspa
