// IS-SPA solvent kernels for gfx950 (CDNA4): MC points, field pass, per-point
// epilogue, force pass, chunk reduction.
//
// Semantics follow src/isspa_force_cuda.cu:73-327 of the reference; the
// decomposition does not.  The reference launches one thread per (point,
// atom) pair and folds results with wave32 shuffles and float atomics.  Here:
//
//  * field pass: one lane owns one MC point; the atom stream is wave-uniform
//    (scalar loads), so each pair costs ~14 VALU ops + one v_rsq.  In-sphere
//    pairs (<2% of wave iterations) take a skipped-when-empty branch.
//  * epilogue: per point, in FP64: |E|, E-hat, Langevin moments by series or
//    recurrence (no tanh cancellation, quirk Q22), and the hoisted constants
//    of the force pass packed in a 64-byte record.
//  * force pass: one lane owns one receiving atom; the point-record stream is
//    wave-uniform.  Per-atom factors (-q_i vtot_i, -vtot_i) are applied once
//    in the reduction.  The CDD term is taken for every pair in the main path
//    and undone in the rare in-sphere branch, so the main path has no select.
//  * no float atomics: lanes keep FP32 partials over short tiles, flush them
//    into FP64, and write per-chunk partials that a reduction kernel sums in a
//    fixed order (quirk Q10).
//  * every launch covers any number of independent windows (kernels.hpp).
//  * the field and force kernels are templated on AN: table lookups (the
//    plain path) or the analytic per-type functions of the differentiable
//    model (diff_device.hpp); only the rare in-sphere branches differ.
#include <algorithm>

#include "device_common.hpp"
#include "diff_device.hpp"
#include "kernels.hpp"
#include "pbc_device.hpp"
#include "points_device.hpp"
#include "nonbond_device.hpp"
#include "bonded_device.hpp"
#include "reduce_device.hpp"

namespace isspa {

constexpr int kBlock = 256;
constexpr int kFieldTile = 128;
constexpr int kForceTile = 128;
// per-type tables up to this many floats (16 KB) are staged in LDS for the
// in-sphere branches; 8 resident blocks per CU then hold 128 of its 160 KB
constexpr int kTabLdsFloats = 4096;

__host__ __device__ inline int field_tab_floats(const TableView &t)
{
    return 2 * t.ntypes * t.ld_g;
}
__host__ __device__ inline int force_tab_floats(const TableView &t) { return t.ntypes * t.ld_f; }
// per-type records of the analytic model (one DiffType per type)
__host__ __device__ inline int diff_tab_floats(const TableView &t)
{
    return t.ntypes * (int)(sizeof(DiffType) / sizeof(float));
}

// copy n floats into LDS with the whole block (n is block-uniform); eight
// loads per thread are issued before their stores, so a small system's
// kernel waits for the table once rather than once per 256 floats
__device__ __forceinline__ void stage_lds(float *dst, const float *__restrict__ src, int n)
{
    constexpr int kU = 8;
    for (int t0 = threadIdx.x; t0 < n; t0 += kU * kBlock) {
        float v[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int t = t0 + u * kBlock;
            v[u] = t < n ? src[t] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int t = t0 + u * kBlock;
            if (t < n) dst[t] = v[u];
        }
    }
}

// ---------------------------------------------------------------------------
// A.1 MC points (mc_points_block).  The first nflag blocks (one
// per window, none when nflag = 0) compute instead the per-window
// minimum-image flags that the field and force passes read, which saves a
// launch.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_mc_points(PointsArgs a, int nflag, float rmax_all,
                                                     int *flag)
{
    if ((int)blockIdx.x < nflag) {
        const WinDesc W = a.wins[blockIdx.x];
        pbc_flag_block(W, a.xyzq, rmax_all, flag + blockIdx.x);
        return;
    }
    mc_points_block(a, blockIdx.x - nflag);
}

// ---------------------------------------------------------------------------
// A.2 field pass (src/isspa_force_cuda.cu:110-206)
// ---------------------------------------------------------------------------
// in-sphere state of one point: g product and count over the split, and the
// E_in sum of the current tile (flushed into FP64 per tile)
struct FieldRare {
    float g;
    int cnt;
    float ex, ey, ez;
};

// GE: {g, E} rows, [type][ld_g].  No branch (each costs a lone wave some 30
// cycles): a lane outside the table reads the nearest row and drops it.  With
// one paired read and no nested branches here and in table_force the step of
// 44 atoms went from 30.2 to 29.3 us, of 1,100 atoms from 94.7 to 93.4 us.
__device__ __forceinline__ void field_in_sphere(const TableView &tb, const float2 *GE, int tj,
                                                float d2, float inv, float s, float rx, float ry,
                                                float rz, float e0, FieldRare &st)
{
    // every rounding spelt out: the bin from a fused d2 inv - r0, the phases
    // from the rounded distance
#pragma clang fp contract(off)
    const float d = d2 * inv;
    // truncation, as the reference's int()
    const int b = (int)(__builtin_fmaf(d2, inv, -tb.g_r0) * tb.g_inv);
    const int row = max(0, min(b, tb.n_g - 2));
    const float2 t0 = GE[tj * tb.ld_g + row], t1 = GE[tj * tb.ld_g + row + 1];
    const float og = d - __builtin_fmaf(tb.g_dr, (float)row, tb.g_r0);
    const float oe = d - __builtin_fmaf(tb.e_dr, (float)row, tb.e_r0);
    float fac = __builtin_fmaf(t1.x, og * tb.g_inv, t0.x * __builtin_fmaf(-tb.g_inv, og, 1.0f));
    float et = __builtin_fmaf(t1.y, oe * tb.e_inv, t0.y * __builtin_fmaf(-tb.e_inv, oe, 1.0f));
    fac = b < 0 ? 0.0f : (b < tb.n_g - 1 ? fac : 1.0f);
    et = b == row ? et : 0.0f;
    st.g *= fac;
    st.cnt += 1;
    const float c = __builtin_fmaf(-e0, s, et * inv);
    st.ex = __builtin_fmaf(c, rx, st.ex);
    st.ey = __builtin_fmaf(c, ry, st.ey);
    st.ez = __builtin_fmaf(c, rz, st.ez);
}

// the same with the analytic g and E of the differentiable model
__device__ __forceinline__ void field_in_sphere_an(const DiffType &T, float d2, float inv, float s,
                                                   float rx, float ry, float rz, float e0,
                                                   FieldRare &st)
{
    const float d = d2 * inv;
    st.g *= diff_g(T, d);
    st.cnt += 1;
    const float c = __builtin_fmaf(-e0, s, diff_E(T, d) * inv);
    st.ex = __builtin_fmaf(c, rx, st.ex);
    st.ey = __builtin_fmaf(c, ry, st.ey);
    st.ez = __builtin_fmaf(c, rz, st.ez);
}

// One (point, atom) pair; type(): the atom's type, asked for only in a sphere
template <bool PBC, bool AN, typename Type>
__device__ __forceinline__ void field_pair(const TableView &tab, float e0, const float2 *GE,
                                           const DiffType *dtypes, float4 q, Type type,
                                           const MinImage &mi, float px, float py, float pz,
                                           float R2, float &ax, float &ay, float &az,
                                           FieldRare &st)
{
    float rx = px - q.x, ry = py - q.y, rz = pz - q.z;
    if (PBC) {
        rx = min_image1(rx, mi);
        ry = min_image1(ry, mi);
        rz = min_image1(rz, mi);
    }
    const float d2 = dist2_f32(rx, ry, rz);
    const float inv = rsqrt_f32(d2);
    const float s = q.w * (inv * inv * inv);
    const bool in = d2 <= R2;
    const float so = in ? 0.0f : s;
    ax = __builtin_fmaf(so, rx, ax);
    ay = __builtin_fmaf(so, ry, ay);
    az = __builtin_fmaf(so, rz, az);
    if (in) {
        if (AN)
            field_in_sphere_an(dtypes[type()], d2, inv, s, rx, ry, rz, e0, st);
        else
            field_in_sphere(tab, GE, type(), d2, inv, s, rx, ry, rz, e0, st);
    }
}

template <bool PBC, bool AN>
__device__ __forceinline__ void field_tile(const FieldArgs &a, const float2 *GE,
                                           const DiffType *dtypes, int j0, int j1,
                                           const MinImage &mi, float px, float py, float pz,
                                           float R2, const Progress &pr, float &ax, float &ay,
                                           float &az, FieldRare &st)
{
    // the tile's atoms by a pointer that advances 16 bytes an atom (an index
    // recomputed from j costs the scalar unit a sign extension and a shift
    // before every load)
    const auto *xq = read_only(reinterpret_cast<const float *>(a.xyzq + j0));
    const auto *ity = read_only(a.itype);
    for (int j = j0; j < j1;) {
        const int stop = j0 + pr.rank(j - j0, j1 - j0);
#pragma unroll 2
        for (; j < stop; ++j, xq += 4)  // wave-uniform
            field_pair<PBC, AN>(a.tab, a.e0, GE, dtypes, make_float4(xq[0], xq[1], xq[2], xq[3]),
                                [=]() { return ity[j]; }, mi, px, py, pz, R2, ax, ay, az, st);
    }
}

// a point's sums over atoms [j0, j1) of its split
struct FieldSums {
    double sx = 0.0, sy = 0.0, sz = 0.0, ex = 0.0, ey = 0.0, ez = 0.0;
    FieldRare st{1.0f, 0, 0.0f, 0.0f, 0.0f};
};

template <bool AN>
__device__ __forceinline__ void field_span(const FieldArgs &a, const float2 *GE,
                                           const DiffType *dtypes, int j0, int j1,
                                           const WinDesc &W, bool pbc, float4 p, FieldSums &fs)
{
    FieldRare &st = fs.st;
    const MinImage mi = min_image_of(W.L, W.h);
    Progress pr(a.ranked_from, j1 - j0);
    for (int jt = j0; jt < j1; jt += kFieldTile) {
        const int je = min(j1, jt + kFieldTile);
        pr.done = jt - j0;
        float ax = 0.0f, ay = 0.0f, az = 0.0f;
        st.ex = st.ey = st.ez = 0.0f;
        if (pbc)
            field_tile<true, AN>(a, GE, dtypes, jt, je, mi, p.x, p.y, p.z, p.w, pr, ax, ay, az,
                                 st);
        else
            field_tile<false, AN>(a, GE, dtypes, jt, je, mi, p.x, p.y, p.z, p.w, pr, ax, ay, az,
                                  st);
        fs.sx += (double)ax;
        fs.sy += (double)ay;
        fs.sz += (double)az;
        fs.ex += (double)st.ex;
        fs.ey += (double)st.ey;
        fs.ez += (double)st.ez;
    }
}

// A block takes fg splits (W.fg: 1, 2 or 4) of the same 256 / fg points, one
// split for each 256 / fg work-items, and adds its splits' sums in split order
// through LDS: it leaves one partial per group of fg splits, so the epilogue
// reads fg times fewer.
struct FieldXchg {
    double s[6];
    float g;
    int cnt;
};
constexpr int kFieldXchgBytes = 3 * 64 * (int)sizeof(FieldXchg);  // fg = 4: 3 splits of 64 points

// NB: the launch also carries the all-pairs blocks after the field blocks (a
// separate instantiation, so the plain field loop keeps its own registers)
template <bool AN, bool NB>
__global__ __launch_bounds__(kBlock) void k_field(FieldArgs a)
{
    extern __shared__ __align__(16) float lds_tab[];
    if (NB && (int)blockIdx.x >= a.nfield) {
        // an all-pairs block riding on this launch (its LJ table in the LDS)
        nonbond_block<false, false, false>(a.nb, blockIdx.x - a.nfield, reinterpret_cast<float2 *>(lds_tab));
        return;
    }
    const int4 bt = a.blocks[blockIdx.x];
    const WinDesc W = a.wins[bt.x];
    const int P = W.n * a.nmc;
    const int fg = W.fg, np = kBlock / fg;
    // the block's split for this work-item (a whole number of waves each),
    // read from the first lane so the compiler knows it is wave-uniform and
    // the atom range stays on scalar loads
    const int sub = __builtin_amdgcn_readfirstlane((int)threadIdx.x / np);
    const int lt = (int)threadIdx.x - sub * np;
    const int m = bt.y * np + lt;  // point within the window
    const int split = bt.z * fg + sub;
    const int j0 = W.a0 + split * W.aps;
    const int j1 = min(W.a0 + W.n, j0 + W.aps);
    const bool valid = m < P;
    const long long gp = (long long)W.a0 * a.nmc + m;
    const float4 p = valid ? a.pts[gp] : make_float4(0.0f, 0.0f, 0.0f, -1.0f);
    const bool pbc = a.pbc_flag[bt.x] != 0;
    // Warm-up: the 128-byte lines of the split's atoms (8 atoms a line, up to
    // two lines a work-item) are requested at block start, so that the loop's
    // scalar atom loads find them in L2 instead of waiting for each line in
    // turn (the positions were last written by another XCD).  The values are
    // only kept alive by the empty asm after the loop.
    float w0 = 0.0f, w1 = 0.0f;
    if (j1 > j0) {
        const int l0 = (j0 >> 3) + lt, last = (j1 - 1) >> 3;
        if (l0 <= last) w0 = a.xyzq[8 * l0].x;
        if (l0 + np <= last) w1 = a.xyzq[8 * (l0 + np)].x;
    }
    // g and E tables (or the analytic records) for the in-sphere branch: LDS
    // when they fit.  Separate call sites give each table pointer one address
    // space, so the LDS ones compile to LDS reads.
    FieldSums fs;
    if (!AN && field_tab_floats(a.tab) <= kTabLdsFloats) {
        stage_lds(lds_tab, reinterpret_cast<const float *>(a.tab.ge), field_tab_floats(a.tab));
        __syncthreads();
        field_span<AN>(a, reinterpret_cast<const float2 *>(lds_tab), a.dtypes, j0, j1, W, pbc, p,
                       fs);
    } else if (AN && diff_tab_floats(a.tab) <= kTabLdsFloats) {
        stage_lds(lds_tab, reinterpret_cast<const float *>(a.dtypes), diff_tab_floats(a.tab));
        __syncthreads();
        field_span<AN>(a, a.tab.ge, reinterpret_cast<const DiffType *>(lds_tab), j0, j1, W, pbc, p,
                       fs);
    } else {
        field_span<AN>(a, a.tab.ge, a.dtypes, j0, j1, W, pbc, p, fs);
    }
    asm volatile("" ::"v"(w0), "v"(w1));
    FieldRare &st = fs.st;
    double sx = fs.sx, sy = fs.sy, sz = fs.sz, ex = fs.ex, ey = fs.ey, ez = fs.ez;
    // the g factors of a split multiply in FP32; splits multiply in FP64 (a
    // product over several splits can leave the FP32 range)
    double g = (double)st.g;
    if (fg > 1) {
        // the group's splits in split order, through LDS (the tables are done)
        FieldXchg *xc = reinterpret_cast<FieldXchg *>(lds_tab);
        __syncthreads();
        if (sub > 0) {
            FieldXchg &e = xc[(sub - 1) * np + lt];
            e.s[0] = sx; e.s[1] = sy; e.s[2] = sz;
            e.s[3] = ex; e.s[4] = ey; e.s[5] = ez;
            e.g = st.g;
            e.cnt = st.cnt;
        }
        __syncthreads();
        if (sub > 0) return;
        for (int k = 1; k < fg; ++k) {
            const FieldXchg &e = xc[(k - 1) * np + lt];
            sx += e.s[0]; sy += e.s[1]; sz += e.s[2];
            ex += e.s[3]; ey += e.s[4]; ez += e.s[5];
            g *= (double)e.g;
            st.cnt += e.cnt;
        }
    }
    if (!valid) return;
    const long long o = W.fpo + (long long)bt.z * P + m;
    a.part_g[o] = g;
    a.part_cnt[o] = st.cnt;
    a.part_s0[o] = sx;
    a.part_s0[a.F + o] = sy;
    a.part_s0[2 * a.F + o] = sz;
    a.part_ein[o] = ex;
    a.part_ein[a.F + o] = ey;
    a.part_ein[2 * a.F + o] = ez;
}

// ---------------------------------------------------------------------------
// per-point epilogue in FP64
// ---------------------------------------------------------------------------
__device__ __forceinline__ void langevin_moments(double x, double inv_x, double &m1, double &m2,
                                                 double &m3)
{
    if (x < 5.0) {
        // the four series advance together: independent FP64 chains
        const double h = 0.5 * x * x;
        double s[4];
#pragma unroll
        for (int l = 0; l < 4; ++l) s[l] = kLangevin.a[l][kLgTerms - 1];
#pragma unroll
        for (int k = kLgTerms - 2; k >= 0; --k)
#pragma unroll
            for (int l = 0; l < 4; ++l) s[l] = __builtin_fma(s[l], h, kLangevin.a[l][k]);
        const double r = 1.0 / s[0];
        m1 = x * s[1] * r;
        m2 = x * x * s[2] * r;
        m3 = x * x * x * s[3] * r;
        return;
    }
    m1 = coth_large(x) - inv_x;
    m2 = 1.0 - 3.0 * m1 * inv_x;
    m3 = m1 - 5.0 * m2 * inv_x;
}

// One point's epilogue: its field partials (one per group of W.fg splits)
// summed in group order (B groups' loads in flight at a time), then the FP64
// Langevin moments, the 16-float force record {p, Ehat, V, D, A2, 3 A2, A3,
// w} and the aux entry {cp E0, A1}.  The epilogue kernel writes them to
// memory; the small-window kernel keeps them in LDS.  Both run this same
// code, so the records are the same bit for bit.
struct PointRecord {
    float4 r[4];
    float4 aux;
    double g;
    int cnt;
    double E[3], E0[3];
};

// the record of point p from its summed field
__device__ __forceinline__ void point_record(float fe0, float fp0, float fq0, float fo0, float4 p,
                                             double g, int cnt, const double *s0, const double *ei,
                                             PointRecord &out)
{
    double E0[3], E[3];
    for (int c = 0; c < 3; ++c) {
        E0[c] = -(double)fe0 * s0[c];
        E[c] = E0[c] + ei[c];
    }
    const double x = sqrt(E[0] * E[0] + E[1] * E[1] + E[2] * E[2]);
    const double inv_x = x > 0.0 ? 1.0 / x : 0.0;
    double eh[3];
    for (int c = 0; c < 3; ++c) eh[c] = E[c] * inv_x;
    double m1, m2, m3;
    langevin_moments(x, inv_x, m1, m2, m3);
    // cnt >= 1 always: the owner atom lies inside its own sphere
    const double inv_cnt = 1.0 / (double)(cnt > 0 ? cnt : 1);
    const double w = g * inv_cnt;
    const double cp = (double)fp0 * inv_cnt;
    const double A1 = (double)fp0 * m1 * w;
    const double A2 = (double)fq0 * m2 * w;
    const double A3 = (double)fo0 * m3 * w;
    double c3[3];  // cp E0 / 3
    for (int c = 0; c < 3; ++c) c3[c] = cp * E0[c] * (1.0 / 3.0);
    out.r[0] = make_float4(p.x, p.y, p.z, (float)eh[0]);
    out.r[1] = make_float4((float)eh[1], (float)eh[2], (float)(A1 * eh[0] + c3[0]),
                           (float)(A1 * eh[1] + c3[1]));
    out.r[2] = make_float4((float)(A1 * eh[2] + c3[2]),
                           (float)(3.0 * A1 * eh[0] + cp * E0[0]),
                           (float)(3.0 * A1 * eh[1] + cp * E0[1]),
                           (float)(3.0 * A1 * eh[2] + cp * E0[2]));
    out.r[3] = make_float4((float)A2, (float)(3.0 * A2), (float)A3, (float)w);
    out.aux = make_float4((float)(cp * E0[0]), (float)(cp * E0[1]), (float)(cp * E0[2]), (float)A1);
    out.g = g;
    out.cnt = cnt;
    for (int c = 0; c < 3; ++c) {
        out.E[c] = E[c];
        out.E0[c] = E0[c];
    }
}

template <int B>
__device__ __forceinline__ void epilogue_point(const EpilogueArgs &a, const WinDesc &W,
                                               long long gp, PointRecord &out)
{
    const int P = W.n * a.nmc;
    const long long m = gp - (long long)W.a0 * a.nmc;
    const float4 p = a.pts[gp];  // requested with the partials, used at the end
    double g = 1.0, s0[3] = {0, 0, 0}, ei[3] = {0, 0, 0};
    int cnt = 0;
    const int ngr = W.splits / W.fg;  // one partial per group of splits
    for (int sp = 0; sp < ngr; sp += B) {
        double pg[B];
        int pc[B];
        double ps[B][3], pe[B][3];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            pg[u] = 1.0;
            pc[u] = 0;
            for (int c = 0; c < 3; ++c) ps[u][c] = pe[u][c] = 0.0;
            if (sp + u < ngr) {
                const long long o = W.fpo + (long long)(sp + u) * P + m;
                pg[u] = a.part_g[o];
                pc[u] = a.part_cnt[o];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    ps[u][c] = a.part_s0[c * a.F + o];
                    pe[u][c] = a.part_ein[c * a.F + o];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
            if (sp + u >= ngr) break;
            g *= pg[u];
            cnt += pc[u];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                s0[c] += ps[u][c];
                ei[c] += pe[u][c];
            }
        }
    }
    point_record(a.e0, a.p0, a.q0, a.o0, p, g, cnt, s0, ei, out);
}

// B groups' loads in flight at a time: 8 for launches with fewer blocks than
// CUs, where each batch costs a full memory latency, and 2 for larger ones,
// where the 8-wide batch's registers would cost occupancy in an HBM-bound
// pass
constexpr int kEpiWideGrid = 256;

template <int B>
__device__ __forceinline__ void epilogue_block(const EpilogueArgs &a)
{
    const long long gp = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (gp >= a.Ptot) return;
    // one window: no per-point window lookup
    const WinDesc W = a.nwin == 1 ? a.wins[0] : a.wins[a.atom_win[gp / a.nmc]];
    PointRecord pr;
    epilogue_point<B>(a, W, gp, pr);
    float4 *r4 = reinterpret_cast<float4 *>(a.rec + gp * kRecFloats);
    for (int k = 0; k < 4; ++k) r4[k] = pr.r[k];
    a.aux[gp] = pr.aux;
    if (a.g_out) a.g_out[gp] = pr.g;
    if (a.cnt_out) a.cnt_out[gp] = pr.cnt;
    if (a.E_out)
        for (int c = 0; c < 3; ++c) a.E_out[3 * gp + c] = pr.E[c];
    if (a.E0_out)
        for (int c = 0; c < 3; ++c) a.E0_out[3 * gp + c] = pr.E0[c];
}

template <int B>
__global__ __launch_bounds__(kBlock) void k_field_epilogue(EpilogueArgs a)
{
    epilogue_block<B>(a);
}

// The wide epilogue with other blocks behind its own.  An engine step's bonded
// and restraint blocks depend on the coordinates alone, and a bonded block, a
// chain of FP64 operations about as long as a point's epilogue, was the longest
// block of the launch before the field pass (5.3 us at 1,100 atoms, the points
// 3.1).  The differentiable model's all-pairs blocks were a launch of 6.4 us at
// 550 atoms.
__global__ __launch_bounds__(kBlock) void k_step_epilogue(EpilogueArgs a, RiderArgs r, int nepi)
{
    __shared__ double red[6][kTermBlock];
    extern __shared__ __align__(16) float2 lds_lj[];
    int b = (int)blockIdx.x - nepi;
    if (b < 0) {
        epilogue_block<8>(a);
        return;
    }
    if (b < r.bonded_blocks) {
        bonded_one(r.bonded, b * kBlock + (int)threadIdx.x);
        return;
    }
    b -= r.bonded_blocks;
    if (b < r.us.nres) {
        us_block(b, r.us.boff, r.us.us_atoms, r.us.us_mass, r.us.kx, r.us.Ls, r.xyzq, r.us.fus,
                 r.us.com, true, red);
        return;
    }
    nonbond_block<false, false, false>(r.nb, b - r.us.nres, lds_lj);
}

// ---------------------------------------------------------------------------
// A.3 force pass (src/isspa_force_cuda.cu:208-327)
//
// For receiver i and point m (r = p_m - x_i, d = |r|, u = Ehat.r/d,
// P2 = 7.5u^2-1.5, P3 = (17.5u^2-7.5)u), the reference's three multipole
// terms plus the CDD term, with -q_i vtot_i factored out, are
//     S += alpha r - d^-3 V - k Ehat
//     alpha = d^-4 (3 A1 u + d^-1 (A2 P2 + d^-1 A3 P3)) + d^-5 (E0c.r)
//     k     = d^-4 (3 u A2 + d^-1 P2 A3)
// with V = A1 Ehat + cp E0/3 and E0c = cp E0.  With e = Ehat.r (u = e/d),
// t = e/d^2 and P3' = 17.5u^2-7.5, both coefficients collapse onto d^-5:
//     alpha = d^-5 (D.r + A2 P2 + A3 P3' t),   D = 3 A1 Ehat + E0c
//     k     = d^-5 (3 A2 e + A3 P2)
// which is 37 VALU operations per pair (one of them v_rsq).  Inside the
// receiver's sphere the CDD part (d^-5 (E0c.r) r - d^-3 E0c/3) is removed
// again and the LJ table term is added instead (with -vtot_i factored out).
// ---------------------------------------------------------------------------
struct ForceAcc {
    double ex, ey, ez;  // electrostatic (pol + CDD) sum, or pol in split mode
    double lx, ly, lz;  // LJ sum
    double cx, cy, cz;  // CDD sum (split mode only)
};

// d^-5 (E0c.r) r - d^-3 E0c/3 for one pair, E0c = c.xyz
__device__ __forceinline__ float3 cdd_term(float4 c, float rx, float ry, float rz, float rinv3,
                                           float rinv5)
{
    const float ec = __builtin_fmaf(c.z, rz, __builtin_fmaf(c.y, ry, c.x * rx));
    const float ac = ec * rinv5;
    const float bc = rinv3 * (1.0f / 3.0f);
    return make_float3(__builtin_fmaf(ac, rx, -bc * c.x), __builtin_fmaf(ac, ry, -bc * c.y),
                       __builtin_fmaf(ac, rz, -bc * c.z));
}

// F of the receiver type's table at d = d2 rinv.  No branch: a lane outside the
// table reads the nearest row and drops it; roundings as in field_in_sphere.
__device__ __forceinline__ float table_force(const TableView &tb, const float *F, float d2,
                                             float rinv)
{
#pragma clang fp contract(off)
    const int b =
        (int)__builtin_fmaf(tb.f_inv, __builtin_fmaf(d2, rinv, -tb.f_r0), 0.5f);
    const int row = max(0, min(b, tb.n_f - 1));
    const float o = d2 * rinv - __builtin_fmaf(tb.f_dr, (float)row, tb.f_r0);
    const float f =
        __builtin_fmaf(F[row + 1], o * tb.f_inv, F[row] * __builtin_fmaf(-tb.f_inv, o, 1.0f));
    return b == row ? f : 0.0f;
}

// FP32 sums of one tile: the electrostatic (or, split, polarisation) sum s and
// the in-sphere LJ sum l; flushed into the FP64 ForceAcc per tile
struct TileSums {
    float sx, sy, sz;
    float lx, ly, lz;
};

// Rec: const float4 * (records in LDS) or ScalarRecords (in memory)
template <bool PBC, bool SPLIT, bool AN, bool RANK, typename Rec>
__device__ __forceinline__ void force_tile(const ForceArgs &a, Rec rec, Rec aux, int m0, int m1,
                                           const MinImage &mi, float xi, float yi, float zi,
                                           float R2, const float *Ftab,
                                           const DiffFParams &fp, const Progress &pr, TileSums &ts,
                                           ForceAcc &acc)
{
    float &sx = ts.sx, &sy = ts.sy, &sz = ts.sz;
    // the next point's record (wave-uniform) is fetched while this one is
    // evaluated, which hides the scalar load latency when few waves share a
    // SIMD; 32-bit point indices within the window keep the loop test on the
    // SALU
    // the next record's pointers advance one record an iteration and stop at
    // the last one (an index recomputed from m costs the scalar unit a clamp,
    // a sign extension and shifts before every load)
    Rec nr = rec + 4 * m0, nx = aux + m0;
    float4 n0 = nr[0], n1 = nr[1], n2 = nr[2], n3 = nr[3], na = nx[0];
    for (int m = m0; m < m1;) {
        const int stop = RANK ? pr.rank(m, m1) : m1;
#pragma unroll 2
        for (; m < stop; ++m) {
            const float4 q0 = n0, q1 = n1, q2 = n2, q3 = n3, c4 = na;
            if (m + 1 < m1) {
                nr = nr + 4;
                nx = nx + 1;
            }
            n0 = nr[0];
            n1 = nr[1];
            n2 = nr[2];
            n3 = nr[3];
            na = nx[0];
            const float Ex = q0.w, Ey = q1.x, Ez = q1.y;
            const float Vx = q1.z, Vy = q1.w, Vz = q2.x;
            const float Dx = q2.y, Dy = q2.z, Dz = q2.w;
            const float A2 = q3.x, A2x3 = q3.y, A3 = q3.z, w = q3.w;
            float rx = q0.x - xi, ry = q0.y - yi, rz = q0.z - zi;
            if (PBC) {
                rx = min_image1(rx, mi);
                ry = min_image1(ry, mi);
                rz = min_image1(rz, mi);
            }
            const float d2 = dist2_f32(rx, ry, rz);
            const float rinv = rsqrt_f32(d2);
            const float e = __builtin_fmaf(Ez, rz, __builtin_fmaf(Ey, ry, Ex * rx));
            const float rinv2 = rinv * rinv;
            const float t = e * rinv2;
            const float u2 = e * t;
            const float P2 = __builtin_fmaf(7.5f, u2, -1.5f);
            const float P3p = __builtin_fmaf(17.5f, u2, -7.5f);
            const float rinv3 = rinv2 * rinv;
            const float rinv5 = rinv3 * rinv2;
            const float k = __builtin_fmaf(A2x3, e, A3 * P2) * rinv5;
            const bool in = d2 <= R2;
            if (!SPLIT) {
                const float dr = __builtin_fmaf(Dz, rz, __builtin_fmaf(Dy, ry, Dx * rx));
                const float alpha = __builtin_fmaf(A2, P2, __builtin_fmaf(A3, P3p * t, dr)) * rinv5;
                sx = __builtin_fmaf(alpha, rx, sx);
                sy = __builtin_fmaf(alpha, ry, sy);
                sz = __builtin_fmaf(alpha, rz, sz);
                sx = __builtin_fmaf(-rinv3, Vx, sx);
                sy = __builtin_fmaf(-rinv3, Vy, sy);
                sz = __builtin_fmaf(-rinv3, Vz, sz);
                sx = __builtin_fmaf(-k, Ex, sx);
                sy = __builtin_fmaf(-k, Ey, sy);
                sz = __builtin_fmaf(-k, Ez, sz);
            } else {
                // polarisation alone: alpha_p r - (d^-3 A1 + k) Ehat, alpha_p
                // being alpha without the E0c.r part
                const float A1 = c4.w;
                const float ap =
                    __builtin_fmaf(A2, P2, __builtin_fmaf(A3, P3p * t, (3.0f * A1) * e)) * rinv5;
                const float bp = __builtin_fmaf(rinv3, A1, k);
                sx = __builtin_fmaf(ap, rx, __builtin_fmaf(-bp, Ex, sx));
                sy = __builtin_fmaf(ap, ry, __builtin_fmaf(-bp, Ey, sy));
                sz = __builtin_fmaf(ap, rz, __builtin_fmaf(-bp, Ez, sz));
                if (!in) {
                    const float3 c = cdd_term(c4, rx, ry, rz, rinv3, rinv5);
                    acc.cx += (double)c.x;
                    acc.cy += (double)c.y;
                    acc.cz += (double)c.z;
                }
            }
            if (in) {
                float fs;
                if (AN) {
                    fs = diff_F(fp, d2 * rinv, rinv) * w;
                } else {
                    fs = table_force(a.tab, Ftab, d2, rinv) * w;
                }
                const float fl = fs * rinv;
                ts.lx = __builtin_fmaf(fl, rx, ts.lx);
                ts.ly = __builtin_fmaf(fl, ry, ts.ly);
                ts.lz = __builtin_fmaf(fl, rz, ts.lz);
                if (!SPLIT) {
                    // remove the CDD part taken in the main path
                    const float3 c = cdd_term(c4, rx, ry, rz, rinv3, rinv5);
                    sx -= c.x;
                    sy -= c.y;
                    sz -= c.z;
                }
            }
        }
    }
}

// The 128-byte lines of the records and aux entries of points [m, m + kForceTile)
// requested by the wave, one record line a lane and an aux line in 16 lanes,
// those below m1.
struct TileLines {
    float r = 0.0f, x = 0.0f;
};
__device__ __forceinline__ void request_tile(const float4 *__restrict__ rec,
                                             const float4 *__restrict__ aux, int m, int m1,
                                             TileLines &t)
{
    static_assert(kForceTile == 2 * kWave, "a record line a lane");
    const int lane = (int)threadIdx.x % kWave;
    const int mr = m + 2 * lane, mx = m + 8 * lane;
    if (mr < m1) t.r = rec[4 * mr].x;
    if (lane < kForceTile / 8 && mx < m1) t.x = aux[mx].x;
}

// Points [m0, m1) of one chunk for one receiver, in tiles of kForceTile.
// AHEAD: the records are in memory, and a wave requests each tile's lines
// while it evaluates the one before.  Right after the epilogue has written
// them they sit in another XCD's L2 or in memory, and the loop's
// one-record-ahead scalar loads would wait for each line in turn.  The values
// are only kept alive (an empty asm takes them a tile later), never used.
// (Lines dealt over a group's blocks once at block start leave the groups
// uncovered whose blocks do not all run at once: the solvent force of 10,758
// atoms with 7 points an atom took 1,019 us, now 925; the step of 1,100 atoms 90.0,
// now 87.9 us.)
template <bool SPLIT, bool AN, bool AHEAD>
__device__ __forceinline__ void force_chunk(const ForceArgs &a, const float4 *__restrict__ rec,
                                            const float4 *__restrict__ aux, int m0, int m1,
                                            const WinDesc &W, bool pbc, float4 xi, float R2,
                                            const float *Ftab, const DiffFParams &fp,
                                            ForceAcc &acc)
{
    const MinImage mi = min_image_of(W.L, W.h);
    Progress pr(AHEAD ? a.ranked_from : kUnranked, m1 - m0);
    for (int mt = m0; mt < m1; mt += kForceTile) {
        const int me = min(m1, mt + kForceTile);
        pr.done = mt - m0;
        TileLines next;
        if (AHEAD) request_tile(rec, aux, me, m1, next);
        TileSums ts{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        // tile-local point indices from the tile's first record
        auto tile = [&](auto r, auto x) {
            if (pbc)
                force_tile<true, SPLIT, AN, AHEAD>(a, r, x, 0, me - mt, mi, xi.x, xi.y, xi.z, R2,
                                                   Ftab, fp, pr, ts, acc);
            else
                force_tile<false, SPLIT, AN, AHEAD>(a, r, x, 0, me - mt, mi, xi.x, xi.y, xi.z, R2,
                                                    Ftab, fp, pr, ts, acc);
        };
        if constexpr (AHEAD)
            tile(ScalarRecords{read_only(reinterpret_cast<const float *>(rec + 4 * mt))},
                 ScalarRecords{read_only(reinterpret_cast<const float *>(aux + mt))});
        else
            tile(rec + 4 * mt, aux + mt);
        acc.ex += (double)ts.sx;
        acc.ey += (double)ts.sy;
        acc.ez += (double)ts.sz;
        acc.lx += (double)ts.lx;
        acc.ly += (double)ts.ly;
        acc.lz += (double)ts.lz;
        if (AHEAD) asm volatile("" ::"v"(next.r), "v"(next.x));
    }
}

// Waves 1..3 leave their shares' sums in LDS; wave 0 adds them in share
// order.  Every wave of the block reaches the barrier.  Returns false on the
// waves whose sums were handed over.
template <bool SPLIT>
__device__ __forceinline__ bool share_sum(double *red, int wv, int lane, ForceAcc &acc)
{
    constexpr int nc = SPLIT ? 9 : 6;
    if (wv > 0) {
        double *d = red + ((wv - 1) * kWave + lane) * nc;
        d[0] = acc.ex; d[1] = acc.ey; d[2] = acc.ez;
        d[3] = acc.lx; d[4] = acc.ly; d[5] = acc.lz;
        if (SPLIT) { d[6] = acc.cx; d[7] = acc.cy; d[8] = acc.cz; }
    }
    __syncthreads();
    if (wv > 0) return false;
    for (int k = 0; k < 3; ++k) {
        const double *d = red + (k * kWave + lane) * nc;
        acc.ex += d[0]; acc.ey += d[1]; acc.ez += d[2];
        acc.lx += d[3]; acc.ly += d[4]; acc.lz += d[5];
        if (SPLIT) { acc.cx += d[6]; acc.cy += d[7]; acc.cz += d[8]; }
    }
    return true;
}

// the window-local points [ms, me) of wave wv's share of chunk group gr
__device__ __forceinline__ void share_range(const WinDesc &W, int P, int gr, int wv, int &ms,
                                            int &me)
{
    const int shares = force_shares(W.n), group = force_group(W.n);
    const int ch = gr * group + wv / shares, part = wv % shares;
    const int c0 = min(P, ch * W.ppc), c1 = min(P, c0 + W.ppc);
    const int sub = (c1 - c0 + shares - 1) / shares;
    ms = min(c1, c0 + part * sub);
    me = min(c1, ms + sub);
}

template <bool SPLIT>
__device__ __forceinline__ void write_force_entry(const ForceArgs &a, const WinDesc &W, int gr,
                                                  int il, const ForceAcc &acc)
{
    const long long o = W.ppo + (long long)gr * W.n + il;
    double2 *e = reinterpret_cast<double2 *>(a.part + o * force_part_stride(SPLIT));
    e[0] = make_double2(acc.ex, acc.ey);
    e[1] = make_double2(acc.ez, acc.lx);
    e[2] = make_double2(acc.ly, acc.lz);
    if (SPLIT) {
        e[3] = make_double2(acc.cx, acc.cy);
        e[4] = make_double2(acc.cz, 0.0);
    }
}

template <bool SPLIT, bool AN>
__global__ __launch_bounds__(kBlock) void k_force(ForceArgs a)
{
    const int4 bt = a.blocks[xcd_run_entry(blockIdx.x, gridDim.x)];
    const WinDesc W = a.wins[bt.x];
    const int lane = (int)threadIdx.x % kWave;
    // the wave index read from the first lane, so the compiler knows it is
    // wave-uniform and the share's point range stays on scalar loads
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int il = bt.y * kWave + lane;  // receiver within the window
    const int P = W.n * a.nmc;
    const long long pbase = (long long)W.a0 * a.nmc;
    const float4 *__restrict__ rec = a.rec4 + 4 * pbase;  // this window's records
    const float4 *__restrict__ aux = a.aux4 + pbase;
    int ms, me;
    share_range(W, P, bt.z, wv, ms, me);
    TileLines first;
    request_tile(rec, aux, ms, me, first);
    const bool valid = il < W.n;
    const int i = W.a0 + (valid ? il : 0);
    const float4 xi = a.xyzq[i];
    const int ti = a.itype[i];
    const float R2 = valid ? a.rmax2[ti] : -1.0f;
    // the receiver type's F table for the in-sphere branch: LDS when it fits;
    // the analytic model keeps its four F constants in registers
    extern __shared__ __align__(16) float lds_tab[];
    DiffFParams fp{0.0f, 0.0f, 0.0f, 0.0f};
    if (AN) fp = diff_f_params(a.dtypes[ti]);
    const bool pbc = a.pbc_flag[bt.x] != 0;
    ForceAcc acc{0, 0, 0, 0, 0, 0, 0, 0, 0};
    // two call sites, so the table pointer of each has one address space and
    // the LDS one compiles to LDS reads
    if (!AN && force_tab_floats(a.tab) <= kTabLdsFloats) {
        stage_lds(lds_tab, a.tab.f, force_tab_floats(a.tab));
        __syncthreads();
        force_chunk<SPLIT, AN, true>(a, rec, aux, ms, me, W, pbc, xi, R2,
                                     lds_tab + ti * a.tab.ld_f, fp, acc);
    } else {
        force_chunk<SPLIT, AN, true>(a, rec, aux, ms, me, W, pbc, xi, R2,
                                     AN ? nullptr : a.tab.f + ti * a.tab.ld_f, fp, acc);
    }
    asm volatile("" ::"v"(first.r), "v"(first.x));
    if (!share_sum<SPLIT>(reinterpret_cast<double *>(lds_tab + a.red_off), wv, lane, acc)) return;
    if (valid) write_force_entry<SPLIT>(a, W, bt.z, il, acc);
}

// ---------------------------------------------------------------------------
// Models of small windows (at most kWinMaxAtoms atoms each): the whole IS-SPA
// pass of a chunk group -- its points, their field over all atoms, the
// epilogue and the force on every receiver -- in one block, with everything
// in LDS: no other block needs a group's points or fields.  Bounded by
// latency: each phase is one short chain per wave, so a block has eight waves
// (one wave alone issues a VALU operation every 8 cycles, two on a SIMD one
// every 2.7), the draws of a point's rejection loop are tried by several
// lanes at once, and all field splits of 64 points run side by side.
// Splits, FP32 tiles, shares and the order of every sum are those of the
// separate launches, so the forces are the same bit for bit.
// Whole step of 44 atoms, nMC = 100, ten steps a graph: 34.5 us in separate
// launches (prologue 6.1, field 6.5, epilogue + force 10.0 us), 22.2 us so.
// The step's all-pairs, bonded and restraint blocks, which depend on the
// coordinates alone, ride on the launch (work-items from 256 up leave).
// ---------------------------------------------------------------------------
// Windows alone of more than 144 atoms gain nothing from having each group of points
// in one block: the blocks are few and the separate passes spread the same chains over
// the chip.  Engine step of 132 atoms, nMC = 20, 25.5 us here and 29.3 in the separate
// launches, of 154 atoms 32.6 and 30.9, of 242 atoms 36.5 and 33.6; their solvent force
// 23.0 and 26.7, 28.2 and 24.2, 32.1 and 27.4.  Batches with windows on both sides
// follow window_pays.
constexpr int kWinMaxAtoms = 256, kWinSmallAtoms = 144;
constexpr int kWinMaxPts = 256;
// One round of two blocks a CU.  More blocks are throughput, not latency: a
// step takes 29.0 us here against 37.5 in the separate launches with 474
// blocks (44 atoms, nMC = 700), 51.1 against 55.3 with 454 (242 atoms, nMC =
// 150), but 58.8 against 56.3 with 632 (64 umbrella windows) and 89.8 against
// 86.4 with 908 (242 atoms, nMC = 300).
constexpr int kWinMaxBlocks = 512;

struct WindowLds {
    const float4 *atoms;
    const int *types;
    const float *rmax, *rmax2;  // per atom
    const float2 *GE;
};

template <bool PBC>
__device__ __forceinline__ void window_field_span(const WindowArgs &a, const WindowLds &l, int j0,
                                                  int j1, const MinImage &mi, float4 p,
                                                  FieldSums &fs)
{
    FieldRare &st = fs.st;
    for (int jt = j0; jt < j1; jt += kFieldTile) {
        const int je = min(j1, jt + kFieldTile);
        float ax = 0.0f, ay = 0.0f, az = 0.0f;
        st.ex = st.ey = st.ez = 0.0f;
        // the next atom and its type are read while this pair is evaluated
        float4 nx = l.atoms[jt];
        int nt = l.types[jt];
        for (int j = jt; j < je; ++j) {
            const float4 x = nx;
            const int t = nt;
            const int jn = min(j + 1, je - 1);
            nx = l.atoms[jn];
            nt = l.types[jn];
            field_pair<PBC, false>(a.tab, a.e0, l.GE, nullptr, x, [=]() { return t; }, mi, p.x,
                                   p.y, p.z, p.w, ax, ay, az, st);
        }
        fs.sx += (double)ax;
        fs.sy += (double)ay;
        fs.sz += (double)az;
        fs.ex += (double)st.ex;
        fs.ey += (double)st.ey;
        fs.ez += (double)st.ez;
    }
}

// the points [m0, m0 + np) of window W into LDS and memory; D lanes a point
// (lt, of atom il) try D consecutive draws at a time, the first accepted one
// counts
__device__ __forceinline__ void window_points(const WindowArgs &a, const WinDesc &W, int m0, int np,
                                              int lt, int il, int sub, int D, uint32_t step,
                                              const WindowLds &l, float4 *lrec, int *best)
{
    const bool mine = lt < np && sub < D;
    for (int base = 0;; base += D) {
        int c0 = 0, c1 = 0, c2 = 0;
        const int d = base + sub;
        const bool open = mine && d < kMcMaxAttempts && best[lt] > d;
        const bool ok = open && mc_draw(a.seed, (uint32_t)(m0 + lt), (uint32_t)d, step, W.sys, c0, c1, c2);
        if (ok) atomicMin(best + lt, d);
        __syncthreads();
        const int b = mine ? best[lt] : 0;
        const bool last = base + D >= kMcMaxAttempts;
        // the winner, or, after the last draw, the point at its atom
        const bool none = mine && last && sub == 0 && b == kMcMaxAttempts;
        if ((ok && b == d) || none) {
            const float4 p = none ? mc_place(l.atoms[il], l.rmax[il], l.rmax2[il], 0, 0, 0)
                                  : mc_place(l.atoms[il], l.rmax[il], l.rmax2[il], c0, c1, c2);
            lrec[4 * lt] = p;
            a.pts[(long long)W.a0 * a.nmc + m0 + lt] = p;
        }
        // every work-item of the block sees the same answer
        if (!__syncthreads_or(mine && b == kMcMaxAttempts) || last) break;
    }
}

// NT: work-items of a block, a multiple of 512
template <int NT>
__global__ __launch_bounds__(NT, 4) void k_window(WindowArgs a)
{
    extern __shared__ __align__(16) float lds_tab[];
    int b = blockIdx.x;
    if (a.step_now && b == 0 && threadIdx.x == 0) *a.step_now = a.step_d ? *a.step_d : a.step;
    if (b >= a.nblocks) {
        // a riding block
        b -= a.nblocks;
        if (threadIdx.x >= (unsigned)kBlock) return;
        if (b < a.nb_blocks) {
            nonbond_block<false, false, true>(a.nb, b, reinterpret_cast<float2 *>(lds_tab));
            return;
        }
        b -= a.nb_blocks;
        if (b < a.bonded_blocks) {
            bonded_one(a.bonded, b * kBlock + (int)threadIdx.x);
            return;
        }
        b -= a.bonded_blocks;
        us_block(b, a.us.boff, a.us.us_atoms, a.us.us_mass, a.us.kx, a.us.Ls, a.xyzq, a.us.fus,
                 a.us.com, true, reinterpret_cast<double (*)[kTermBlock]>(lds_tab));
        return;
    }
    const int tid = threadIdx.x, lane = tid % kWave;
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    // LDS: g/E and F tables; atoms; point records (until they are written the
    // points, in each record's first entry, and the draws' counters); then the
    // splits' field sums, later the shares' force sums
    float4 *atoms = reinterpret_cast<float4 *>(lds_tab + a.off_atoms);
    int *types = reinterpret_cast<int *>(atoms + kWinMaxAtoms);
    float *rmax = reinterpret_cast<float *>(types + kWinMaxAtoms), *rmax2 = rmax + kWinMaxAtoms;
    float4 *lrec = reinterpret_cast<float4 *>(lds_tab + a.off_pts);
    float4 *laux = lrec + 4 * a.cap_pts;
    int *best = reinterpret_cast<int *>(laux);
    float *area = lds_tab + a.off_x;
    FieldXchg *xc = reinterpret_cast<FieldXchg *>(area);
    __shared__ int far_flag;
    // The loads of the tables (which depend on nothing) are in flight while
    // the block's window is looked up and its atoms are requested.
    const int ntab = field_tab_floats(a.tab) + force_tab_floats(a.tab);
    const float *tab = reinterpret_cast<const float *>(a.tab.ge);  // F follows
    constexpr int kU = 6;
    float tv[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) tv[u] = tab[min(tid + u * NT, ntab - 1)];
    const int4 bt = a.blocks[b];
    const WinDesc W = a.wins[bt.x];
    const uint32_t step = a.step_d ? *a.step_d : a.step;
    const int n = W.n, P = n * a.nmc;
    const float4 x = a.xyzq[W.a0 + min(tid, n - 1)], x0 = a.xyzq[W.a0];
    const int t = a.itype[W.a0 + min(tid, n - 1)];
    const float rm = a.rmax[t], rm2 = a.rmax2[t];
    const int span = force_group(n) * W.ppc;
    const int m0 = min(P, bt.z * span), np = min(P, m0 + span) - m0;
    // lt: the work-item's point, of atom il; sub: its draw or field split, wave-uniform
    const int npr = (np + kWave - 1) & ~(kWave - 1);
    const int D = NT / npr;
    const int sub = __builtin_amdgcn_readfirstlane(tid / npr);
    const int lt = tid - sub * npr;
    const int il = lt < np && sub < D ? (m0 + lt) / a.nmc : 0;
    if (tid == 0) far_flag = 0;
    if (tid < npr) best[tid] = kMcMaxAttempts;
#pragma unroll
    for (int u = 0; u < kU; ++u)
        if (tid + u * NT < ntab) lds_tab[tid + u * NT] = tv[u];
    for (int k = tid + kU * NT; k < ntab; k += NT) lds_tab[k] = tab[k];
    if (tid < n) {
        atoms[tid] = x;
        types[tid] = t;
        rmax[tid] = rm;
        rmax2[tid] = rm2;
    }
    __syncthreads();
    if (atoms_far(W, x, x0, a.rmax_all)) far_flag = 1;
    const WindowLds l{atoms, types, rmax, rmax2, reinterpret_cast<const float2 *>(lds_tab)};
    // (its barriers also publish the flag)
    window_points(a, W, m0, np, lt, il, sub, D, step, l, lrec, best);
    const bool pbc = far_flag != 0;
    const MinImage mi = min_image_of(W.L, W.h);
    // field: D splits side by side, added in order, groups of W.fg at a time
    const float4 p = lt < np ? lrec[4 * lt] : make_float4(0.0f, 0.0f, 0.0f, -1.0f);
    double g = 1.0, s0[3] = {0, 0, 0}, ei[3] = {0, 0, 0};
    double gg = 1.0, gs[3] = {0, 0, 0}, ge[3] = {0, 0, 0};
    int cnt = 0;
    for (int sp = 0; sp < W.splits; sp += D) {
        const int split = sp + sub;
        if (sub < D && split < W.splits) {
            const int j0 = split * W.aps, j1 = min(n, j0 + W.aps);
            FieldSums fs;
            if (pbc)
                window_field_span<true>(a, l, j0, j1, mi, p, fs);
            else
                window_field_span<false>(a, l, j0, j1, mi, p, fs);
            FieldXchg &e = xc[tid];
            e.s[0] = fs.sx; e.s[1] = fs.sy; e.s[2] = fs.sz;
            e.s[3] = fs.ex; e.s[4] = fs.ey; e.s[5] = fs.ez;
            e.g = fs.st.g;
            e.cnt = fs.st.cnt;
        }
        __syncthreads();
        if (tid < np)
            for (int k = 0; k < D && sp + k < W.splits; ++k) {
                const FieldXchg &e = xc[k * npr + tid];
                cnt += e.cnt;
                if ((sp + k) % W.fg == 0) {
                    gg = (double)e.g;
                    for (int c = 0; c < 3; ++c) { gs[c] = e.s[c]; ge[c] = e.s[3 + c]; }
                } else {
                    gg *= (double)e.g;
                    for (int c = 0; c < 3; ++c) { gs[c] += e.s[c]; ge[c] += e.s[3 + c]; }
                }
                if ((sp + k) % W.fg == W.fg - 1) {
                    g *= gg;
                    for (int c = 0; c < 3; ++c) { s0[c] += gs[c]; ei[c] += ge[c]; }
                }
            }
        if (sp + D < W.splits) __syncthreads();
    }
    if (tid < np) {
        PointRecord pr;
        point_record(a.e0, a.p0, a.q0, a.o0, lrec[4 * tid], g, cnt, s0, ei, pr);
        for (int k = 0; k < 4; ++k) lrec[4 * tid + k] = pr.r[k];
        laux[tid] = pr.aux;
    }
    __syncthreads();
    // force: up to 128 receivers, a wave for each 64 and share; above, a wave
    // for each 64 and pair of shares.  The wave of the first share keeps its
    // sums and adds the others' from LDS, in share order.
    ForceArgs fa{};
    fa.tab = a.tab;
    fa.part = a.part;
    const int nrw = (n + kWave - 1) / kWave;
    const int per = nrw <= 2 ? 1 : 2;  // shares of a wave
    const int rg = wv * per / 4, q0 = wv * per % 4;
    const int ir = rg * kWave + lane;  // the lane's receiver
    double *sh = reinterpret_cast<double *>(area);  // [share - per][receiver][6]
    const DiffFParams fp{0.0f, 0.0f, 0.0f, 0.0f};
    ForceAcc own{0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (rg < nrw) {
        const int ic = min(ir, n - 1);
        const float4 xi = atoms[ic];
        const float R2 = ir < n ? rmax2[ic] : -1.0f;
        const float *F = lds_tab + field_tab_floats(a.tab) + types[ic] * a.tab.ld_f;
        for (int q = q0; q < q0 + per; ++q) {
            int ms, me;
            share_range(W, P, bt.z, q, ms, me);
            ForceAcc acc{0, 0, 0, 0, 0, 0, 0, 0, 0};
            force_chunk<false, false, false>(fa, lrec, laux, ms - m0, me - m0, W, pbc, xi, R2, F, fp,
                                             acc);
            if (q0 == 0) {
                own.ex += acc.ex; own.ey += acc.ey; own.ez += acc.ez;
                own.lx += acc.lx; own.ly += acc.ly; own.lz += acc.lz;
            } else {
                double *d = sh + 6 * ((size_t)(q - per) * nrw * kWave + ir);
                d[0] = acc.ex; d[1] = acc.ey; d[2] = acc.ez;
                d[3] = acc.lx; d[4] = acc.ly; d[5] = acc.lz;
            }
        }
    }
    __syncthreads();
    if (q0 != 0 || ir >= n) return;
    for (int q = per; q < 4; ++q) {
        const double *d = sh + 6 * ((size_t)(q - per) * nrw * kWave + ir);
        own.ex += d[0]; own.ey += d[1]; own.ez += d[2];
        own.lx += d[3]; own.ly += d[4]; own.lz += d[5];
    }
    write_force_entry<false>(fa, W, bt.z, ir, own);
}

// the force of atom i, or its components, from its summed partials
template <bool SPLIT>
__device__ __forceinline__ void write_force(const ReduceArgs &a, int i, const double *s)
{
    if (!SPLIT) {
        const float3 fi = isspa_atom_force(a.xyzq[i].w, a.vtot[a.itype[i]], s);
        float4 f = a.f[i];
        f.x += fi.x;
        f.y += fi.y;
        f.z += fi.z;
        a.f[i] = f;
        if (a.f_alone) a.f_alone[i] = make_float4(fi.x, fi.y, fi.z, 0.0f);
    } else {
        const float4 x = a.xyzq[i];
        const double vt = (double)a.vtot[a.itype[i]];
        const double qv = -(double)x.w * vt;
        for (int c = 0; c < 3; ++c) {
            a.f_pol[3 * i + c] = qv * s[c];
            a.f_lj[3 * i + c] = -vt * s[3 + c];
            a.f_cdd[3 * i + c] = qv * s[6 + c];
        }
    }
}

// F_i = -q_i vtot_i S_e - vtot_i S_lj over the chunk partials, summed in the
// fixed slice order of reduce_device.hpp (kSumAtoms atoms x kSumSlices chunk
// slices a block).  FEW: an atom a work-item (few_entries).
template <bool SPLIT, bool FEW>
__global__ __launch_bounds__(kBlock) void k_force_reduce(ReduceArgs a)
{
    constexpr int comps = SPLIT ? 9 : 6;
    double s[comps];
    for (int k = 0; k < comps; ++k) s[k] = 0.0;
    if constexpr (FEW) {
        const int i = blockIdx.x * kBlock + threadIdx.x;
        if (i >= a.ntot) return;
        const WinDesc W = window_of(a.wins, a.nwin, a.atom_win, i);
        sum_batches<comps, kFewBatch, 1>(ForceEntry<comps>(W, a.part, i), 0, W.fents, s);
        write_force<SPLIT>(a, i, s);
    } else {
        __shared__ double red[kSumSlices][comps][kSumAtoms];
        const int al = threadIdx.x % kSumAtoms, sl = threadIdx.x / kSumAtoms;
        const int i = blockIdx.x * kSumAtoms + al;
        const bool valid = i < a.ntot;
        if (valid) {
            const WinDesc W = window_of(a.wins, a.nwin, a.atom_win, i);
            sum_batches<comps, 8>(ForceEntry<comps>(W, a.part, i), sl, W.fents, s);
        }
        combine_slices<comps>(red, al, sl, s);
        if (sl == 0 && valid) write_force<SPLIT>(a, i, s);
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline int blocks_for(long long n) { return (int)((n + kBlock - 1) / kBlock); }

hipError_t launch_mc_points(const WinDesc *wins, const int *atom_win, const float4 *xyzq,
                            const int *itype, const float *rmax, const float *rmax2, int ntot,
                            int nmc, uint64_t seed, uint32_t step, const uint32_t *step_d,
                            float4 *pts, hipStream_t s, int nwin, float rmax_all, int *flag)
{
    const long long P = (long long)ntot * nmc;
    const int nflag = flag ? nwin : 0;
    if (P == 0 && nflag == 0) return hipSuccess;
    const PointsArgs a{wins, atom_win, xyzq, itype, rmax, rmax2, ntot, nmc, seed, step, step_d, pts, nwin};
    hipLaunchKernelGGL(k_mc_points, dim3((unsigned)((P + kMcBlockPts - 1) / kMcBlockPts) + nflag), dim3(kBlock), 0, s, a, nflag,
                       rmax_all, flag);
    return hipGetLastError();
}

hipError_t launch_field(const FieldArgs &a0, int nblocks, hipStream_t s)
{
    FieldArgs a = a0;
    a.nfield = nblocks;
    a.ranked_from = ranked_from(nblocks);
    if (a.dtypes) {
        if (nblocks == 0) return hipSuccess;
        const int nt = diff_tab_floats(a.tab);
        const size_t lds = std::max<size_t>(nt <= kTabLdsFloats ? (size_t)nt * sizeof(float) : 0,
                                            a.max_fg > 1 ? kFieldXchgBytes : 0);
        hipLaunchKernelGGL((k_field<true, false>), dim3(nblocks), dim3(kBlock), lds, s, a);
    } else {
        if (nblocks + a.nb_blocks == 0) return hipSuccess;
        const int nt = field_tab_floats(a.tab);
        size_t lds = std::max<size_t>(nt <= kTabLdsFloats ? (size_t)nt * sizeof(float) : 0,
                                      a.max_fg > 1 ? kFieldXchgBytes : 0);
        if (a.nb_blocks) {
            lds = std::max(lds, nonbond_lds_bytes(a.nb.T, false));
            hipLaunchKernelGGL((k_field<false, true>), dim3(nblocks + a.nb_blocks), dim3(kBlock),
                               lds, s, a);
        } else {
            hipLaunchKernelGGL((k_field<false, false>), dim3(nblocks), dim3(kBlock), lds, s, a);
        }
    }
    return hipGetLastError();
}

static int rider_blocks(const RiderArgs &r)
{
    return r.bonded.contrib ? (int)blocks_for((long)r.bonded.nb + r.bonded.na + r.bonded.nd) : 0;
}

// a block a CU: with a second round the step of 64 umbrella windows (184
// blocks and 104 riders) takes 57.0 us, with the riders before the field 56.0
bool epilogue_takes_riders(long long P, const RiderArgs &r)
{
    return P > 0 && blocks_for(P) + rider_blocks(r) + r.us.nres + r.nb_blocks <= kEpiWideGrid;
}

hipError_t launch_step_epilogue(const EpilogueArgs &a, RiderArgs r, hipStream_t s)
{
    const int eb = (int)blocks_for(a.Ptot);
    r.bonded_blocks = rider_blocks(r);
    const int grid = eb + r.bonded_blocks + r.us.nres + r.nb_blocks;
    const size_t lds = r.nb_blocks ? nonbond_lds_bytes(r.nb.T, false) : 0;
    hipLaunchKernelGGL(k_step_epilogue, dim3(grid), dim3(kBlock), lds, s, a, r, eb);
    return hipGetLastError();
}

hipError_t launch_epilogue(const EpilogueArgs &a, hipStream_t s)
{
    if (a.Ptot == 0) return hipSuccess;
    const int eb = (int)blocks_for(a.Ptot);
    if (eb < kEpiWideGrid)
        hipLaunchKernelGGL(k_field_epilogue<8>, dim3(eb), dim3(kBlock), 0, s, a);
    else
        hipLaunchKernelGGL(k_field_epilogue<2>, dim3(eb), dim3(kBlock), 0, s, a);
    return hipGetLastError();
}

// LDS of k_window in floats: tables, atoms, point records, then the splits' or
// the shares' sums
static int window_lds(const TableView &t, int nt, int max_points, WindowArgs &a)
{
    const int tab = (field_tab_floats(t) + force_tab_floats(t) + 3) & ~3;
    a.off_atoms = tab;
    a.off_pts = a.off_atoms + 7 * kWinMaxAtoms;
    a.cap_pts = (max_points + kWave - 1) / kWave * kWave;
    a.off_x = a.off_pts + (kRecFloats + kAuxFloats) * a.cap_pts;
    const int nxc = nt * (int)(sizeof(FieldXchg) / sizeof(float));
    const int nsh = 2 * 6 * std::max(3 * 2 * kWave, 2 * 4 * kWave);
    return a.off_x + std::max(nxc, nsh);
}

bool window_fits(const TableView &t, int max_atoms, int max_points, int nblocks)
{
    return max_atoms <= kWinMaxAtoms && max_points <= kWinMaxPts && nblocks <= kWinMaxBlocks &&
           field_tab_floats(t) <= kTabLdsFloats && force_tab_floats(t) <= kTabLdsFloats;
}

// Work-items of a k_window block: sixteen waves where a pass of eight holds less
// than a group's field splits and a CU has a block to itself (242 atoms, nMC = 20,
// 72 blocks: a step takes 36.7 against 41.2 us; but nMC = 100, 303 blocks, 63.5
// against 49.4 us).
static int window_threads(int max_items, int nblocks)
{
    return max_items > 512 && nblocks <= 256 ? 1024 : 512;
}

// Whether k_window is the faster route for windows that fit it.
//
// With windows on both sides of kWinSmallAtoms it depends on where the longest chains
// are.  k_window lasts as long as its longest block, which makes its field passes one
// after the other (each a split's atoms a lane) and then its waves' shares of the
// force: a least-squares fit gives the solvent force 14 us + 0.3 us an atom of those
// passes + 0.2 us a point of those shares.  The separate passes pay their launches,
// wait for the longest share of any window, read a point's partial fields one after the
// other and take longer with more pairs: 20 us + 0.14 us a point of that share + 0.3 us
// an entry of the longest row of partial fields + 2.7 us a million pairs; in an engine
// step, whose other terms ride on k_window, both take 5 to 8 us more.  The rule is that
// comparison in units of 0.3 us, its constants moved to where the measured times divide
// best.
//
// Measured on 382 batches drawn from windows of 2 to 242 atoms, nMC 3 to 100, both
// routes each: where the rule takes k_window (212), the step is 10% and the solvent
// force alone 2.6% faster than in separate passes; where it does not (170), k_window
// would take the same time for the step and 10.8% more for the force.  Without the term
// of the entries, which a window of 22 splits has 11 of and one of 20 five, batches of a
// single 220-atom window were sent the slower way: 39 pairs and 40 chains of 22 atoms
// beside it (nMC = 20), a step of 35.9 us instead of 32.1.  Four windows of 220 atoms,
// nMC = 10: with two pairs of atoms the step takes 35.1 us separate and 36.6 here, the
// force 28.4 and 32.8; with two chains of 22 atoms, whose shares are the longest, 41.1
// and 37.7, and 33.8 and 32.6.
bool window_pays(const WinDesc *w, int nwin, int nmc, int nblocks, int max_items)
{
    int lo = w[0].n, hi = w[0].n;
    for (int k = 1; k < nwin; ++k) {
        lo = std::min(lo, w[k].n);
        hi = std::max(hi, w[k].n);
    }
    if (hi <= kWinSmallAtoms) return true;
    if (lo > kWinSmallAtoms) return false;
    const int nt = window_threads(max_items, nblocks);
    double chain = 0.0, longest = 0.0, entries = 0.0, pairs = 0.0;
    for (int k = 0; k < nwin; ++k) {
        const WinDesc &d = w[k];
        const long long P = (long long)d.n * nmc;
        const long long np = std::min(P, (long long)force_group(d.n) * d.ppc);
        if (np > kWinMaxPts) return false;
        const int side = nt / (int)((np + kWave - 1) / kWave * kWave);  // splits of a pass
        const int passes = (d.splits + side - 1) / side;
        const int shares = force_shares(d.n), share = (d.ppc + shares - 1) / shares;
        const int per = d.n <= 2 * kWave ? 1 : 2;  // shares of a wave
        chain = std::max(chain, passes * d.aps + 0.6 * per * share);
        longest = std::max(longest, (double)share);
        entries = std::max(entries, (double)(d.splits / d.fg));
        pairs += (double)d.n * (double)P;
    }
    return chain <= 20.0 + 0.6 * longest + 0.8 * entries + 8.0e-6 * pairs;
}

hipError_t launch_window(const WindowArgs &a0, int max_points, int max_items, hipStream_t s)
{
    WindowArgs a = a0;
    const int nt = window_threads(max_items, a.nblocks);
    size_t lds = sizeof(float) * window_lds(a.tab, nt, max_points, a);
    if (a.nb_blocks) lds = std::max(lds, nonbond_lds_bytes(a.nb.T, false));
    const long terms = (long)a.bonded.nb + a.bonded.na + a.bonded.nd;
    a.bonded_blocks = a.bonded.contrib ? blocks_for(terms) : 0;
    const int grid = a.nblocks + a.nb_blocks + a.bonded_blocks + a.us.nres;
    if (grid == 0) return hipSuccess;
    if (nt == 512)
        hipLaunchKernelGGL(k_window<512>, dim3(grid), dim3(nt), lds, s, a);
    else
        hipLaunchKernelGGL(k_window<1024>, dim3(grid), dim3(nt), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_force(const ForceArgs &a, int nblocks, bool split, hipStream_t s)
{
    if (nblocks == 0) return hipSuccess;
    // dynamic LDS: the F table when it fits (table model), then the
    // share-sum area
    ForceArgs b = a;
    const int nt = force_tab_floats(a.tab);
    b.red_off = (!a.dtypes && nt <= kTabLdsFloats) ? (nt + 3) & ~3 : 0;
    b.ranked_from = ranked_from(nblocks);
    const size_t lds = (size_t)(b.red_off + 2 * force_share_doubles(split)) * sizeof(float);
    const dim3 g(nblocks), t(kBlock);
    switch ((a.dtypes ? 2 : 0) + (split ? 1 : 0)) {
    case 0: hipLaunchKernelGGL((k_force<false, false>), g, t, lds, s, b); break;
    case 1: hipLaunchKernelGGL((k_force<true, false>), g, t, lds, s, b); break;
    case 2: hipLaunchKernelGGL((k_force<false, true>), g, t, lds, s, b); break;
    default: hipLaunchKernelGGL((k_force<true, true>), g, t, lds, s, b); break;
    }
    return hipGetLastError();
}

hipError_t launch_force_reduce(const ReduceArgs &a, bool split, hipStream_t s)
{
    if (a.ntot == 0) return hipSuccess;
    const bool few = few_entries(a.max_fents, a.ntot);
    const int atoms = few ? kBlock : kSumAtoms;
    const dim3 g((a.ntot + atoms - 1) / atoms), t(kBlock);
    switch ((few ? 2 : 0) + (split ? 1 : 0)) {
    case 0: hipLaunchKernelGGL((k_force_reduce<false, false>), g, t, 0, s, a); break;
    case 1: hipLaunchKernelGGL((k_force_reduce<true, false>), g, t, 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_force_reduce<false, true>), g, t, 0, s, a); break;
    default: hipLaunchKernelGGL((k_force_reduce<true, true>), g, t, 0, s, a); break;
    }
    return hipGetLastError();
}


}  // namespace isspa
