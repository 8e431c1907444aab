// Launch interface between the C-ABI host code (capi_*.hip) and the gfx950
// kernels.  Every launcher enqueues on `stream` and returns the launch status.
//
// All kernels are window-aware: a launch covers W independent systems
// ("windows", e.g. umbrella-sampling windows of uneven size) whose atoms are
// concatenated.  Window w owns atoms [a0, a0 + n) and MC points
// [a0 nMC, (a0 + n) nMC).  A single system is the case W = 1.  Grids are 1-D
// over a per-block work table (int4 {window, block, split/chunk, -}), so
// uneven windows share one launch without idle blocks.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "diff_device.hpp"
#include "xcd_runs.hpp"

namespace isspa {

struct WinDesc {
    int a0, n;          // atoms of the window
    int splits, aps;    // field pass: atom splits, atoms per split
    int chunks, ppc;    // force pass: point chunks, points per chunk
    int nbc, apc;       // nonbond: groups of kNbGroup partner chunks, atoms per chunk
    long long fpo;      // field partial offset:  sum over earlier windows of splits / fg * P
    long long ppo;      // force partial offset:  sum of fents * n
    long long npo;      // nonbond partial offset: sum of nbc * n (nbc entries per atom)
    uint32_t sys;       // Philox counter word 3
    float L, h;         // box length and half length
    int nte;            // nonbond total force: entries per atom (nbc, or the
                        // number of 256-atom blocks when pairs are taken once)
    int fg;             // field pass: splits per block (1, 2 or 4; divides splits);
                        // the block's waves take fg splits of 256 / fg points
                        // and leave one partial per group of fg splits
    int fents;          // force pass: partial entries per atom, ceil(chunks / force_group(n))
    long long spo;      // nonbond total-force partial offset: sum of nte * n
    long long vpo;      // adjoint atom-pass partial offset: sum of vents * n
    int vents, vpad;    // adjoint atom pass: entries per atom, ceil(chunks / 4)
};

// splits per field block for a window of `splits` splits
inline int field_group(int splits) { return splits % 4 == 0 ? 4 : (splits % 2 == 0 ? 2 : 1); }

// Per-type tables on the device, each type padded with one trailing zero row
// so that a lerp at the last row reads 0 (the reference reads the next type's
// first row there, 0 in every shipped table; quirk Q4).  All windows share the
// grid; their types are concatenated.  The E table is read at the g table's
// row, so the two are stored as pairs {g, E}: both ends of both lerps are one
// 16-byte read (E rows beyond the g table are never read).
struct TableView {
    const float2 *ge;
    const float *f;  // directly behind ge
    int n_g, n_f;    // logical rows
    int ld_g, ld_f;  // padded rows per type
    int ntypes;
    float g_r0, g_dr, g_inv;
    float e_r0, e_dr, e_inv;
    float f_r0, f_dr, f_inv;
};

// Per-point record written by the field epilogue and streamed by the force pass.
// 16 floats = one 64-byte scalar load per point.
//   [0..2]  p      MC point position
//   [3..5]  Ehat   unit mean-field direction
//   [6..8]  V      A1*Ehat + cp*E0/3  (E-hat-like terms of dipole + CDD)
//   [9..11] D      3 A1 Ehat + cp*E0  (r-coefficient vector of dipole + CDD)
//   [12] A2 = q0 <P2> w   [13] 3 A2   [14] A3 = o0 <P3> w   [15] w = g/cnt
// with A1 = p0 <P1> w.  A second array of P float4 {cp*E0, A1} (read only by
// the in-sphere branch, the component split and the adjoint) follows the
// records in the same allocation.
constexpr int kRecFloats = 16;
constexpr int kAuxFloats = 4;

// all-pairs blocks of 256 work-items; kinds of the block table's .w
constexpr int kNbBlock = 256;
constexpr int kNbKindChunk = 0;  // 64 receivers x kNbGroup partner chunks, every pair in both orders
constexpr int kNbKindNear = 1;   // receiver block x itself or a neighbouring block, ordered
constexpr int kNbKindSym = 2;    // super-tile: receiver block x partner block, each pair once
constexpr int kSymMinAtoms = 4096;            // windows that take each pair once
constexpr int kSymLdsDoubles = 3 * kNbBlock;  // a super-tile's partner sums in LDS

struct NonbondArgs {
    const WinDesc *wins;
    const int4 *blocks;    // {w, receiver block, group of partner chunks or block, kind}
    const float4 *xyzq;
    const float4 *aux;     // per atom j: {4 R_j^2, cA_j, cB_j, LJ type (int bits)}
    const float2 *lj;      // [T*T] {12A, 6B}
    int T;
    const uint32_t *excl;  // [N][4] bit window j - i + 64 in [0,128)
    const int *excl_ptr;   // CSR fallback (null when the windows are complete)
    const int *excl_idx;
    float cfar;
    const int *pbc_flag;
    double *part;          // [comps][B], in the layout of the launch's mode
    long long B;
    int sym;               // the block table holds super-tiles
};

// chunks of a block: one a wave, all for the same 64 receivers
constexpr int kNbGroup = 4;
constexpr size_t nonbond_share_bytes(int comps) { return sizeof(double) * 3 * 64 * comps; }

// dynamic LDS of an all-pairs block: the T x T LJ table, then (super-tiles)
// the partner sums on an 8-byte boundary; the chunks' sums take the table's place
inline size_t nonbond_lds_bytes(int T, bool sym, bool split = false)
{
    const size_t tab = sym ? sizeof(float) * 2 * (((size_t)T * T + 1) & ~(size_t)1) +
                                 sizeof(double) * kSymLdsDoubles
                           : sizeof(float) * 2 * (size_t)T * T;
    const size_t sums = nonbond_share_bytes(split ? 9 : 3);
    return tab > sums ? tab : sums;
}

struct FieldArgs {
    const WinDesc *wins;
    const int4 *blocks;   // {w, point block, split, -}
    const float4 *pts;
    const float4 *xyzq;
    const int *itype;
    TableView tab;
    const DiffType *dtypes;  // non-null: analytic functions instead of tables
    int nmc;
    float e0;
    const int *pbc_flag;  // per window
    double *part_g;       // [F] product of the in-sphere g factors
    int *part_cnt;        // [F]
    double *part_s0;      // [3][F]  sum_out q r / d^3
    double *part_ein;     // [3][F]  sum_in (-e0 q / d^3 + Etab / d) r
    long long F;          // total field partial length
    // all-pairs partials computed by nb_blocks extra blocks of the same launch
    // (tables only, nb_blocks = 0: none); nfield is set by the launcher
    NonbondArgs nb;
    int nb_blocks, nfield;
    int ranked_from;  // blocks from here on rank their waves by progress (set at launch)
    int max_fg;  // the largest W.fg of the launch (its LDS holds the split exchange if > 1)
};

struct EpilogueArgs {
    const WinDesc *wins;
    int nwin;
    const int *atom_win;
    const float4 *pts;
    long long Ptot;
    int nmc;
    const double *part_g;
    const int *part_cnt;
    const double *part_s0, *part_ein;
    long long F;
    float e0, p0, q0, o0;
    float *rec;         // [P][16]
    float4 *aux;        // [P] {cp E0, A1}
    double *g_out;      // [P]      inspection outputs, each may be null
    int *cnt_out;       // [P]
    double *E_out;      // [P][3]
    double *E0_out;     // [P][3]
};

struct ForceArgs {
    const WinDesc *wins;
    const int4 *blocks;   // {w, receiver block (64 atoms), chunk group, -}
    const float4 *rec4;   // [P][4] float4 view of the records
    const float4 *aux4;   // [P] {cp E0, A1}
    const float4 *xyzq;
    const int *itype;
    const float *rmax2;   // per type
    TableView tab;
    const DiffType *dtypes;  // non-null: analytic F instead of the table
    int nmc;
    const int *pbc_flag;
    double *part;         // [C][stride]: (S_e, S_lj), or (pol, lj, cdd, pad) split
    long long C;
    int red_off;          // float offset of the share-sum area in the dynamic LDS (set at launch)
    int ranked_from;      // blocks from here on rank their waves by progress (set at launch)
};

// The first block of a launch of nb whose waves rank themselves by progress
// (Progress, below); the blocks before it have the top priority.
//   nb <= 512:   none; with one or two waves a SIMD there is little to even
//                out (field of 550 atoms, 430 blocks: 9.8 us, ranked 10.1).
//   nb <= 1536:  all; they run at once (6 to 7 blocks fit a CU).
//   above:       the last 1,280, 5 a CU: those before must leave in turn, so
//                that the rest find room early.  Force pass of 4,510 atoms
//                (2,272 blocks): 195 us unranked, 175 with the last 1,280, 183
//                with 1,536, 198 with 1,664 and 199 with 2,048; 187 with 768.
// The split force pass, the analytic field and force passes and both sides of the
// adjoint follow the same lines, though they hold four to seven blocks a CU.  Measured
// none / this rule / all ranked / the last 1,280, in us:
//   split force   414 blocks   21.9 /  22.2 /  22.3 /  22.1;  990  48.5 / 44.5 / 44.4 / 44.5;
//               2,135         146.6 / 136.0 / 140.7 / 135.6; 3,328 424 / 405 / 413 / 408
//   analytic field 516         19.7 /  20.2 /  20.2 /  20.2; 1,116 30.2 / 28.8 / 28.7 / 28.9;
//               2,064          33.9 /  34.7 /  34.9 /  34.7; 8,256 99.2 / 99.2 / 101.9 / 97.9
//   analytic force 384         10.3 /  10.5 /  11.4 /  11.1;  975  33.7 / 31.2 / 31.2 / 31.0;
//               2,484          52.2 /  50.3 /  54.7 /  50.2; 7,920 195.5 / 194.5 / 196.0 / 192.3
//   adjoint, points 416        15.2 /  15.3 /  15.5 /  15.3; 1,032 38.2 / 34.0 / 33.7 / 33.8;
//               2,064          59.9 /  55.2 /  58.8 /  55.1; 8,256 245 / 243 / 245 / 240
//   adjoint, atoms  384        17.0 /  17.1 /  17.3 /  17.3;  828  41.7 / 37.7 / 37.3 / 37.6;
//               2,484          78.3 /  70.7 /  71.7 /  70.9; 29,376 838 / 830 / 850 / 831
// Over 62 launches of 315 to 29,376 blocks the rule is within 2.6% of the best of the
// four, and up to 12% faster than unranked.
constexpr int kUnranked = 0x7fffffff;
constexpr int kRankMin = 512, kRankAll = 1536, kRankLast = 1280;
inline int ranked_from(int nb)
{
    return nb <= kRankMin ? kUnranked : (nb <= kRankAll ? 0 : nb - kRankLast);
}

// A wave's issue priority by its progress.  The arbiter serves the oldest of a
// SIMD's waves first, so of four that start together the first is done at half
// the time of the last, which ends up alone, at a third of the SIMD's rate.
// Here a wave with three quarters of its work to go outranks one with two:
// they stay within a quarter of each other and end together.
// Against the arbiter alone: force pass of 1,100 atoms (nMC = 20) 37.5 ->
// 32.7 us, of 2,200 (nMC = 10) 69 -> 59, of 6,600 359 -> 335, of 19,998 (nMC =
// 20) 5,420 -> 5,320 us; field pass of 1,100 atoms 22.9 -> 22.3, of 2,200 36.4
// -> 32.3, of 6,600 166 -> 153, of 19,998 2,268 -> 2,265 us.  (Looking at the
// rank every 16 records instead of at the quarters: field of 19,998 atoms
// 2,335 us.)
struct Progress {
    int done = 0;     // work before the tile
    int quarter = 0;  // of the wave's work, rounded up; 0: not ranked
    __device__ __forceinline__ Progress(int from, int work)
    {
        if (from == kUnranked) return;
        if ((int)blockIdx.x < from)
            __builtin_amdgcn_s_setprio(3);
        else
            quarter = (work + 3) / 4;
    }
    // ranks the wave at place m of the tile; returns where the rank changes
    // next, at most m1
    __device__ __forceinline__ int rank(int m, int m1) const
    {
        if (quarter == 0) return m1;
        const int x = done + m;
        int next = quarter;
        if (x < quarter) {
            __builtin_amdgcn_s_setprio(3);
        } else if (x < 2 * quarter) {
            __builtin_amdgcn_s_setprio(2);
            next = 2 * quarter;
        } else if (x < 3 * quarter) {
            __builtin_amdgcn_s_setprio(1);
            next = 3 * quarter;
        } else {
            __builtin_amdgcn_s_setprio(0);
            return m1;
        }
        return min(m1, next - done);
    }
};

// A force block's four waves serve the same 64 receivers, each with its own
// share of the MC points, and the block adds the shares' sums in order before
// it writes one partial: a quarter of the partials of a block that gives each
// wave its own receivers, at the same number of waves, and no idle wave in
// the last receiver block.  A share is a whole chunk, or, in windows of at
// most 128 (64) atoms, a half (quarter) of one; the block takes force_group
// consecutive chunks.  Against 256 receivers a block: the force assembly, which
// reads the partials, 78 -> 38 us at 19,998 atoms and 13.9 -> 10.4 us at
// 1,100, the force pass there 43.0 -> 40.9 us, the differentiable model's
// reduction of 32 x 1,100 atoms 81 -> 16 us.
__host__ __device__ constexpr int force_shares(int n) { return n <= 64 ? 4 : (n <= 128 ? 2 : 1); }
__host__ __device__ constexpr int force_group(int n) { return 4 / force_shares(n); }
// doubles of the share-sum area: shares 1..3 of 64 receivers
__host__ __device__ constexpr int force_share_doubles(bool split)
{
    return 3 * 64 * (split ? 9 : 6);
}

// The force pass's partials are stored entry by entry, entry
// (chunk group, atom) holding its components together: 6 doubles (S_e, S_lj), or
// 10 in split mode (pol, lj, cdd and a pad, so every entry stays 16-byte
// aligned), read and written as double2.
__host__ __device__ constexpr int force_part_stride(bool split) { return split ? 10 : 6; }

struct ReduceArgs {
    const WinDesc *wins;
    int nwin;
    const int *atom_win;
    const double *part;
    long long C;
    int max_fents;        // the most entries of a window
    int ntot;
    const float4 *xyzq;
    const int *itype;
    const float *vtot;    // per type
    float4 *f;            // += total (may be null)
    float4 *f_alone;      // = total, the IS-SPA force kept apart (may be null)
    double *f_lj, *f_pol, *f_cdd;  // component outputs (split mode)
};

// MC points: one per (atom, draw) of every window
struct PointsArgs {
    const WinDesc *wins;
    const int *atom_win;
    const float4 *xyzq;
    const int *itype;
    const float *rmax, *rmax2;
    int ntot, nmc;
    uint64_t seed;
    uint32_t step;            // used when step_d is null
    const uint32_t *step_d;
    float4 *pts;
    int nwin;
};

// bonded terms (window-agnostic: they carry global atom indices)
struct BondedArgs {
    const float4 *xyzq;
    float L, h;
    int nb, na, nd;
    const int4 *bond_atoms;
    const float2 *bond_params;
    const int4 *angle_atoms;
    const float2 *angle_params;
    const int4 *dih_atoms;
    const int *dih_types;
    const float4 *dih_params;
    const float2 *sc14;
    const int *ityp;
    const float2 *lj;      // [T*T] {A, B}
    int T;
    float4 *contrib;       // [2 nb + 3 na + 6 nd]
    double *energy;        // per-term energies (3 per dihedral: torsion, 1-4 Coulomb, 1-4 LJ)
    int terms;
};
// umbrella restraints: nres blocks, bias entries [boff[r], boff[r+1])
struct RestraintArgs {
    int nres;
    const int *boff;
    const int2 *us_atoms;
    const float *us_mass;
    const float2 *kx;
    const float *Ls;
    float4 *fus;  // bias forces stored (w = 1)
    double *com;
};

// Bonded terms, restraints and all-pairs blocks (no super-tiles) riding on the
// epilogue, after its own blocks (each part skipped when empty).
struct RiderArgs {
    const float4 *xyzq;
    BondedArgs bonded;
    int bonded_blocks;      // set by the launcher
    RestraintArgs us;
    NonbondArgs nb;
    int nb_blocks;
};

// The IS-SPA pass of a model of small windows in one launch (k_window), with
// the all-pairs, bonded and restraint blocks of an engine step riding on it
// (each part skipped when empty).
struct WindowArgs {
    const WinDesc *wins;
    const int4 *blocks;   // {w, -, chunk group, -}
    int nblocks;
    const float4 *xyzq;
    const int *itype;
    const float *rmax, *rmax2;
    float rmax_all;
    TableView tab;
    int nmc;
    float e0, p0, q0, o0;
    uint64_t seed;
    uint32_t step;
    const uint32_t *step_d;
    float4 *pts;
    double *part;         // force partials, as k_force leaves them
    uint32_t *step_now;   // an engine step's kStepNow word, or null
    NonbondArgs nb;
    int nb_blocks;
    BondedArgs bonded;
    int bonded_blocks;    // set by the launcher
    RestraintArgs us;
    int off_atoms, off_pts, off_x, cap_pts;  // LDS layout in floats (set by the launcher)
};

hipError_t launch_mc_points(const WinDesc *wins, const int *atom_win, const float4 *xyzq,
                            const int *itype, const float *rmax, const float *rmax2, int ntot,
                            int nmc, uint64_t seed, uint32_t step, const uint32_t *step_d,
                            float4 *pts, hipStream_t s, int nwin = 0, float rmax_all = 0.0f,
                            int *flag = nullptr);
hipError_t launch_field(const FieldArgs &a, int nblocks, hipStream_t s);
hipError_t launch_epilogue(const EpilogueArgs &a, hipStream_t s);
// the epilogue with riders, where it is short of blocks
bool epilogue_takes_riders(long long P, const RiderArgs &r);
hipError_t launch_step_epilogue(const EpilogueArgs &a, RiderArgs r, hipStream_t s);
// k_window: whether a model's windows, chunk groups and tables fit it, whether it is
// the faster route (windows w of the present tiling), and the launch (max_atoms,
// max_points: of the largest window and chunk group; max_items: the most (point,
// field split) pairs of a group)
bool window_fits(const TableView &t, int max_atoms, int max_points, int nblocks);
bool window_pays(const WinDesc *w, int nwin, int nmc, int nblocks, int max_items);
hipError_t launch_window(const WindowArgs &a, int max_points, int max_items, hipStream_t s);
hipError_t launch_force(const ForceArgs &a, int nblocks, bool split, hipStream_t s);
hipError_t launch_force_reduce(const ReduceArgs &a, bool split, hipStream_t s);

// One step's force of the MD engine in one launch: f = bonded gather + IS-SPA
// reduction + all-pairs chunk reduction (each optional: null contrib, null
// isspa.part, null nb_part), overwriting f (w = 0).
struct AssembleArgs {
    int n;
    float4 *f;
    const float4 *contrib;  // bonded contribution slots
    const int *gptr, *gidx;
    ReduceArgs isspa;       // IS-SPA chunk partials (isspa.f unused)
    const WinDesc *nb_wins; // all-pairs chunk partials
    int nb_nwin;
    const int *nb_atom_win;
    const double *nb_part;
    long long nb_B;
    const float4 *fus;      // restraint bias forces (w = 1 marks a restrained atom), added last
    struct {                // leap-frog + Andersen of the assembled atoms (xyzq null: none)
        const WinDesc *wins;    // integrator windows, both required with xyzq
        int nwin;
        const int *atom_win;
        float4 *xyzq, *vel;
        float kT, dt;
        uint32_t thr;
        uint64_t seed;
        uint32_t *step_d;   // kStepNext: written step + 1; kStepNow: this step
    } lf;
};
hipError_t launch_assemble_forces(const AssembleArgs &a, hipStream_t s);

// The engine's step counter is two words.  The first launch of a step reads
// kStepNext and copies it to kStepNow; the assembly, its last launch, reads
// kStepNow and writes kStepNow + 1 to kStepNext.  No launch both reads a word
// and writes it, so no block waits for or counts the others.
constexpr int kStepNext = 0, kStepNow = 1;

// ---- nonbond ----
hipError_t launch_nonbond(const NonbondArgs &a, int nblocks, bool split, hipStream_t s);
// max_entries: the most entries of a window
hipError_t launch_chunk_reduce3(const WinDesc *wins, int nwin, const int *atom_win, const double *part,
                                long long B, int max_entries, int ntot, int comps, float4 *f,
                                double *o0, double *o1, double *o2, hipStream_t s);

// ---- bonded ----
hipError_t launch_bonded_terms(const BondedArgs &a, hipStream_t s);
// the terms' forces summed per atom into f and, with energy, their energies
struct BondedSumArgs {
    const float4 *contrib;
    const int *ptr, *idx;   // an atom's contribution slots
    int n;
    float4 *f;
    const double *eterm;
    int nb, na, nd;
    double *energy;         // out [5], or null
};
hipError_t launch_bonded_gather(const BondedSumArgs &g, hipStream_t s);
// The MD engine's step prologue: what of a step depends only on the coordinates
// and does not ride on the epilogue, in one grid.  Each part is skipped when empty (nflag 0,
// bonded.contrib null, us.nres 0, pts.ntot 0).
struct PrologueArgs {
    int nflag;              // minimum-image flags of the IS-SPA windows
    float rmax_all;
    int *flag;
    BondedArgs bonded;      // bonded terms into their contribution slots
    int bonded_blocks;      // set by the launcher
    RestraintArgs us;       // bias forces stored into fus
    PointsArgs pts;         // MC points (pts.wins also serves the flags)
    uint32_t *step_d;       // the step counter's two words
};
hipError_t launch_step_prologue(PrologueArgs a, hipStream_t s);


// ---- differentiable model: parameter preparation, forward reduction, adjoint ----
struct DiffPrepArgs {
    int T;
    const double *theta;   // [T][5] sigma, eps, x0, g0, alpha
    const double *camp;    // [T]
    double sig_s, eps_s, core, delta;
    DiffType *types;       // out [T]
    float2 *nb_lj;         // out [T*T] {12A, 6B} for the nonbond kernel
    float4 *nb_ld;         // out [T*T] {A, B, dA/dsigma_ij, dB/dsigma_ij}
};
struct DiffAtomArgs {
    int n;
    const float4 *xyz;     // positions (.w ignored)
    const double *q;       // charges
    const double *lam;     // [N][3] cotangent, or null (forward)
    const int *itype;
    const float *vtot, *rmax2;
    float4 *xq;            // out: positions with FP32 charges
    float4 *arec;          // out [N][4]: {x, R2}, {-q vtot lam, type}, {-vtot lam, q}, {lam, 0}
};
struct DiffReduceArgs {
    int n;
    const WinDesc *wins;
    int nwin;
    const int *atom_win;
    const double *part;    // force partials [6][C] (S_e, S_lj)
    long long C;
    const int *itype;
    const float *vtot;
    const double *q;
    double *se;            // out [N][3]
    double *f;             // out [N][3] (overwritten)
    const WinDesc *nb_wins;  // all-pairs partials added to f, or null
    const double *nb_part;
    long long nb_B;
};
struct VjpArgs {
    const WinDesc *wins;
    const int *atom_win;
    const int4 *gblk, *vblk;   // point-lane and atom-lane block tables
    int nmc;
    long long Ptot;
    const float4 *pts, *rec4, *aux4, *arec, *xq;
    const int *itype;
    const float *rmax2;
    const DiffType *dtypes;
    int ranked_from;           // as ForceArgs (set at launch)
    const int *pbc_flag;
    const double *g_out, *E_out;
    const int *cnt_out;
    float e0, p0, q0, o0;
    double *ppart;             // [10][F] point-record bars
    long long F;
    float4 *prec;              // [P][4] {p, R2}, {dL/dE, g dL/dg}, {dL/dE0, w}, -
    double *apart;             // [6][C] atom bars: q, theta(5)
    long long C;               // sum of vents * n
};
struct VjpNbArgs {
    const WinDesc *wins;
    const int4 *blocks;
    const float4 *xq, *aux, *arec;
    const uint32_t *excl;
    const int *excl_ptr, *excl_idx;
    float cfar;
    const int *pbc_flag;
    const float4 *ld;          // [T*T] {A, B, dA, dB}
    int T;
    double *part;              // [3][B] q, sigma, eps bars
    long long B;
};
struct VjpFinishArgs {
    int n;
    const WinDesc *wins, *nb_wins;
    int nwin;
    const int *atom_win;
    const double *apart;
    long long C;
    const double *nbpart;
    long long B;
    const int *itype;
    const float *vtot;
    const double *lam, *se, *theta;
    double *gq;                // out [N]
    double *gatom;             // out [N][5]
};
hipError_t launch_diff_prep(const DiffPrepArgs &t, const DiffAtomArgs &a, hipStream_t s);
hipError_t launch_diff_reduce(const DiffReduceArgs &a, hipStream_t s);
hipError_t launch_vjp_points(const VjpArgs &a, int nblocks, hipStream_t s);
hipError_t launch_vjp_epilogue_nonbond(const VjpArgs &a, const VjpNbArgs &n, int nb_blocks,
                                       hipStream_t s);
hipError_t launch_vjp_atoms(const VjpArgs &a, int nblocks, hipStream_t s);
hipError_t launch_vjp_finish(const VjpFinishArgs &a, hipStream_t s);
// part: scratch of 5 T type_reduce_ranges(n) doubles
int type_reduce_ranges(int n);
hipError_t launch_type_reduce(const double *gatom, const int *itype, int n, int T, double *part,
                              double *gtheta, hipStream_t s);

// ---- integrator / restraint / utilities ----
// atom_win == null: every atom belongs to the single window `one`
hipError_t launch_leapfrog(const WinDesc *wins, const int *atom_win, const WinDesc &one,
                           int ntot, float4 *xyzq, float4 *vel, const float4 *f, float kT,
                           float dt, uint32_t thr, uint64_t seed, uint32_t step,
                           const uint32_t *step_d, hipStream_t s);
// one workgroup per restraint; bias entries [boff[r], boff[r+1]) {atom, group}
hipError_t launch_us(int nres, const int *boff, const int2 *atoms, const float *mass,
                     const float2 *kx /* {k, x0} */, const float *L, const float4 *xyzq,
                     float4 *f, double *com, hipStream_t s);
hipError_t launch_pbc_flag(const WinDesc *wins, int W, const float4 *xyzq, float rmax_all,
                           int *flag, hipStream_t s);
hipError_t launch_zero(void *p, size_t bytes, hipStream_t s);
hipError_t launch_add4(float4 *dst, const float4 *src, int n, hipStream_t s);
hipError_t launch_set_word(uint32_t *dst, uint32_t v, hipStream_t s);

}  // namespace isspa
