// cmf_device.hpp -- device-side data layout and per-cell physics of the MI355X
// CaMa-Flood substep. Shared by the kernels (cmf_kernels.hip) and the host glue.
//
// Layout in HBM (one structure of arrays per handle):
//  * cells: the domains of the handle concatenated, each domain in depth-first
//    river order (or NSEQ order); static arrays are indexed by cell c.
//  * members: a handle runs NMEM = 2^lgm members (runoff realisations) of every
//    domain. Per-member state is member-minor: state slot s = (c << lgm) | m, so
//    the members of a cell are adjacent, static map values are read once per
//    cell for all its members, and the neighbour gathers (j << lgm) | m of a
//    wavefront stay as coalesced as the cells themselves. Instance k = dom*NMEM+m
//    has its own adaptive step (InstStep). A single model is NMEM=1, one domain.
//  * static map: the seven float32 source maps (every reference map is read from
//    a float32 file, so float32 holds them exactly) and the NLFP float32 profile
//    planes; the derived tables (RIVSTOMAX, RIVELV, FLDSTOMAX, FLDGRD) are
//    recomputed in FP64 in registers with the reference's own statements, so the
//    FP64 path reads 4 B instead of 8-16 B per map value and stays bit-identical.
//  * topology: I1NEXT (0-based) and the upstream CSR (ascending sources).
//  * state: storages FP64; flux/stage arrays of type R (double for the FP64
//    path, float for the mixed path); inflow accumulators FP64.
//
// Arithmetic of the FP64 path keeps the reference's statement order (the Fortran
// left-to-right product order, x**(-1.) = 1/x, x**0.5 = sqrt(x), default-kind
// literals widened from float). Files are compiled with -ffp-contract=off.
#pragma once
#include <hip/hip_runtime.h>
#include <utility>
#include <stdint.h>

namespace cmf {

// default-kind (float) literals of the reference, widened
constexpr double K_1EM5F  = (double)1.e-5f;
constexpr double K_1EM10F = (double)1.e-10f;
constexpr double K_0P01F  = (double)0.01f;
constexpr double K_2O3F   = (double)(2.f / 3.f);
constexpr double K_0P1F   = (double)0.1f;
constexpr double K_0P2F   = (double)0.2f;
constexpr double K_1E18F  = (double)1.e18f;
constexpr double K_P7O3   = -7.0 / 3.0;     // -7._JPRB/3._JPRB
constexpr double K_P4O3   = -4.0 / 3.0;     // -4._JPRB/3._JPRB
constexpr double K_P7O3F  = (double)(-7.f / 3.f);   // default-real -7./3.
constexpr double K_P4O3F  = (double)(-4.f / 3.f);   // default-real -4./3.
constexpr double K_LEVSENT = 1.e18;         // 1.E18_JPRB sentinel of non-levee cells

constexpr int NGLB = 11;
constexpr int NPART = 2 * NGLB;                // budget sums of a tile: high parts, then low parts
enum { G_STOPRE, G_STONXT, G_STONEW, G_RIVINF, G_RIVOUT,
       G_STOPRE2, G_STONEW2, G_RIVSTO, G_FLDSTO, G_FLDARE, G_LEVSTO };

constexpr int NLFP_MAX = 16;
constexpr int NMEM_MAX = 64;                   // members per domain (power of two)
constexpr int NDOM_ARG = 32;                   // domain offsets carried in the kernel arguments

template <class T> __device__ __forceinline__ T vmax(T a, T b) { return a > b ? a : b; }
template <class T> __device__ __forceinline__ T vmin(T a, T b) { return a < b ? a : b; }
__device__ __forceinline__ double vpow(double x, double y) { return pow(x, y); }
__device__ __forceinline__ float vpow(float x, float y) { return powf(x, y); }
__device__ __forceinline__ double vsqrt(double x) { return sqrt(x); }
__device__ __forceinline__ float vsqrt(float x) { return sqrtf(x); }
__device__ __forceinline__ double vabs(double x) { return fabs(x); }
__device__ __forceinline__ float vabs(float x) { return fabsf(x); }

struct DevMap {
    int32_t n, nseqriv, nlfp, npth, npthlev, ndam;
    int32_t lfplain, nlevcell;
    int32_t lgm, nmem;                         // members per domain = nmem = 1 << lgm
    int32_t ns, nsp;                           // state slots: n << lgm, npth << lgm
    double dfrcinc;
    const int32_t* cell_dom;                   // domain of each cell (NULL: one domain)
    int32_t ndom_arg;                          // > 0: domains found from dom_off_arg instead
    int32_t dom_off_arg[NDOM_ARG + 1];         // first cell of each domain (device order)
    const int32_t* pth_dom;                    // domain of each path (NULL: one domain)
    const int32_t* next;                       // 0-based downstream, <0 for mouths
    const int32_t* up_ptr;                     // upstream CSR (n+1)
    const int32_t* up_idx;
    const float *elevtn, *rivhgt, *nxtdst, *rivwth, *rivman, *rivlen, *grarea;
    const float* fldhgt;                       // [nlfp][n]
    const double* dwnelv;                      // boundary elevation (mouths)
    const int32_t* i2mask;
    // bifurcation paths, 0-based endpoints (-1 outside domain)
    const int32_t *pth_upst, *pth_down;
    const double *pth_dst, *pth_elv, *pth_wth, *pth_man;   // elv/wth [npthlev][npth]
    const int32_t *pout_ptr, *pout_idx, *pinf_ptr, *pinf_idx;
    // levee: compact table of levee cells, lev_idx[i] = row or -1
    const int32_t* lev_idx;
    const double* lev_tab;                     // [7][nlevcell]
    // dams
    const int32_t* i1dam;                      // per cell (0,1,10,11)
    const int32_t* dam_of_cell;                // per cell: dam row; -2 other cells with I1DAM > 0; -1
    const int32_t* damstat;
    const double *dam_convol, *dam_emevol, *dam_adjvol, *dam_qa, *dam_qn, *dam_qf;
    // Hanazaki-2022 rule (LDAMH22): NorVol and R_VolUpa of every dam
    int32_t ldamh22;
    const double *dam_norvol, *dam_r_volupa;
};

// Per-instance step of the current outer step (written by the host after the
// CFL bound is known): DT, PGRV*DT, NADD = sum of DT over the NT substeps.
// input matrix of the runoff interpolation (INPX, INPY, INPA of YOS_CMF_MAP), device
// cell order, entry-planar: entry k of cell c at k * n + c
struct RoffMap {
    int inpn, nxin, nyin, n;
    const int* inpx;
    const int* inpy;
    const double* inpa;
    double drofunit, rmis;
};

// output-period accumulators (D2*_oAVG / D2*_oMAX of YOS_CMF_DIAG), FP64 in both
// precisions, one value per state slot; pthflw [npthlev][nsp]
struct OutState {
    double *rivout, *fldout, *outflw, *rivvel, *pthout, *runoff, *daminf;
    double *outflw_max, *rivdph_max, *storge_max;
    double* pthflw;
};

struct InstStep {
    double dt, gdt, nadd;
    int32_t nt;                                // substeps of this instance
    int32_t swapfix;                           // odd number of idle substeps: RIVDPH pair swapped
};

template <class R>
struct DevState {
    double *rivsto, *fldsto, *levsto, *damsto, *daminf;
    R *rivout, *fldout;                        // limited outflow == *_PRE after a substep
    const R* rivout_vel;                       // D2RIVOUT read by OUTFLW for RIVVEL
    R *qr_u, *qf_u;                            // outflow before the inflow limiter
    R *rivdph_pre, *fldsto_pre;
    R* rivdph_next;                            // buffer receiving the new RIVDPH (k_update)
    R *rivdph, *flddph, *fldfrc, *fldare, *sfcelv, *storge, *outflw, *rivvel, *levdph;
    double *rivinf, *fldinf, *pthout;
    R* rate;
    R* runoff;
    R* upsinf;                                 // LUPSINF: D2UPSINF [m3/s] (NULL when off)
    R *pthflw, *pthflw_u, *pthflwsum, *pthflwsum_u;   // [npthlev][nsp], [nsp]
    R *rivout_avg, *fldout_avg, *outflw_avg, *rivvel_avg, *pthout_avg, *runoff_avg;
    R *outflw_max, *rivdph_max, *storge_max, *daminf_avg;
    R *pthflw_avg, *pthflwsum_avg;
    double* partials;                          // [nt][ntiles][NPART] (single instance only)
    double* glb_hist;                          // [nt_cap][NGLB]
    unsigned long long* cfl;                   // [ninst]: bits of the CFL bound (positive doubles)
    double* cfl_part;                          // single instance: CFL bound of each stage block
    const InstStep* inst;                      // [ninst]
    unsigned* bar;                             // [2]: grid barrier of the fused substep kernel
    int32_t* err;                              // [1]: device error flag (barrier time-out)
};

struct StepArgs {
    double pgrv, pmanfld, pdstmth, pcadp, pminslp;
    int32_t lfldout, lpthout, ldamout, llevee;
    int32_t it;                                // substep index within the outer step
    int32_t prow;                              // row of S.partials this substep's budget sums go to
    int32_t budget;                            // write the per-tile water-budget sums
    int32_t xcd;                               // XCD-contiguous tile order
    int32_t lupsinf;                           // add S.upsinf to the river in STONXT
    int32_t lkine;                             // kinematic-wave outflow (LKINE)
    int32_t lslpmix;                           // slope-mixed outflow (LSLPMIX, without LKINE)
    int32_t daminf_sparse;                     // DAMINF is zero in every cell with I1DAM == 0
};

// ---------------------------------------------------------------------------
// Compensated sums of the eleven budget terms (TwoSum, Knuth): every partial sum
// is carried as hi + lo with lo the exact rounding error of each addition, so the
// result is the correctly rounded sum up to O(2^-106) relative terms, whatever the
// number of cells. Needs IEEE additions without contraction (the files are compiled
// with -ffp-contract=off).
__device__ __forceinline__ void two_sum(double a, double b, double& s, double& e) {
    s = a + b;
    const double bb = s - a;
    e = (a - (s - bb)) + (b - bb);
}

// lanes 0-31 of a and 32-63 of b in a; the other halves in b (permlane32_swap);
// with 16: odd rows of 16 lanes of a against the even rows of b
template <int W>
__device__ __forceinline__ void lane_swap(double& a, double& b) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    unsigned al = (unsigned)__double2loint(a), ah = (unsigned)__double2hiint(a);
    unsigned bl = (unsigned)__double2loint(b), bh = (unsigned)__double2hiint(b);
    u2 l, h;
    if (W == 32) {
        l = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
        h = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
    } else {
        l = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
        h = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
    }
    a = __hiloint2double((int)h[0], (int)l[0]);
    b = __hiloint2double((int)h[1], (int)l[1]);
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
    const int l = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true);
    const int h = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true);
    return __hiloint2double(h, l);
}
constexpr int DPP_ROR8 = 0x128;                // rotation by 8 inside a row of 16 lanes
constexpr int DPP_HALF_MIRROR = 0x141;         // lane i of 8 takes lane 7 - i
constexpr int DPP_QUAD_1032 = 0xb1, DPP_QUAD_2301 = 0x4e;
__device__ __forceinline__ void comp_add(double& h, double& l, double oh, double ol) {
    double s, e;
    two_sum(h, oh, s, e);
    h = s;
    l = (l + ol) + e;
}
// one halving step of N values a lane: lanes with `up` keep the values from (N+1)/2
// on, the others those before, and each adds what its partner lane held of them
template <int CTRL, int N>
__device__ __forceinline__ void comp_halve(double (&h)[N], double (&l)[N], double (&ho)[(N + 1) / 2],
                                           double (&lo)[(N + 1) / 2], bool up) {
    constexpr int H = (N + 1) / 2;
#pragma unroll
    for (int i = 0; i < H; ++i) {
        if (N == 1) {
            ho[i] = h[i]; lo[i] = l[i];
            comp_add(ho[i], lo[i], dpp_move<CTRL>(h[i]), dpp_move<CTRL>(l[i]));
        } else {
            const double bh = i + H < N ? h[i + H < N ? i + H : 0] : 0.0, bl = i + H < N ? l[i + H < N ? i + H : 0] : 0.0;
            ho[i] = up ? bh : h[i];
            lo[i] = up ? bl : l[i];
            const double oh = up ? h[i] : bh, ol = up ? l[i] : bl;
            comp_add(ho[i], lo[i], dpp_move<CTRL>(oh), dpp_move<CTRL>(ol));
        }
    }
}

// Sums of N terms over a wavefront into hi[(base + k) * stride + col], lo[...].
// At every step half of the lanes take half of the terms (a half-swap of terms i
// and i + N/2 leaves one in the lower lanes and the other in the upper ones, each
// ready to be added to its other half), so eleven terms need 14 compensated
// additions instead of the 66 of eleven butterflies, and no LDS permutes: a substep is
// bound by its instructions where the state fits the caches (FP64, 239,520 cells 39.9
// -> 33.8 us; 1,500,120 cells 209 -> 200 us).
// vl: low parts of the terms, NULL where they are exact.
template <int N>
__device__ __forceinline__ void wave_sum_comp(const double* v, double* hi, double* lo, int stride, int col,
                                              int base = 0, const double* vl = nullptr) {
    constexpr int N1 = (N + 1) / 2, N2 = (N1 + 1) / 2, N3 = (N2 + 1) / 2, N4 = (N3 + 1) / 2;
    static_assert(N > 2 && N4 == 1, "laid out for 3 to 16 terms");
    const int lane = threadIdx.x & 63;
    double h1[N1], l1[N1], h2[N2], l2[N2], h3[N3], l3[N3], h4[1], l4[1];
#pragma unroll
    for (int i = 0; i < N1; ++i) {
        double a = v[i], b = i + N1 < N ? v[i + N1 < N ? i + N1 : 0] : 0.0;
        lane_swap<32>(a, b);
        two_sum(a, b, h1[i], l1[i]);
        if (vl) {
            double al = vl[i], bl = i + N1 < N ? vl[i + N1 < N ? i + N1 : 0] : 0.0;
            lane_swap<32>(al, bl);
            l1[i] = l1[i] + (al + bl);
        }
    }
#pragma unroll
    for (int i = 0; i < N2; ++i) {
        double bh = i + N2 < N1 ? h1[i + N2 < N1 ? i + N2 : 0] : 0.0, bl = i + N2 < N1 ? l1[i + N2 < N1 ? i + N2 : 0] : 0.0;
        h2[i] = h1[i]; l2[i] = l1[i];
        lane_swap<16>(h2[i], bh);
        lane_swap<16>(l2[i], bl);
        comp_add(h2[i], l2[i], bh, bl);
    }
    comp_halve<DPP_ROR8>(h2, l2, h3, l3, (lane & 8) != 0);
    comp_halve<DPP_HALF_MIRROR>(h3, l3, h4, l4, (lane & 4) != 0);
    comp_add(h4[0], l4[0], dpp_move<DPP_QUAD_1032>(h4[0]), dpp_move<DPP_QUAD_1032>(l4[0]));
    comp_add(h4[0], l4[0], dpp_move<DPP_QUAD_2301>(h4[0]), dpp_move<DPP_QUAD_2301>(l4[0]));
    // which term a lane ended up with
    if ((lane & 3) == 0) {
        int k = N3 > 1 && (lane & 4) ? N4 : 0;
        bool ok = k < N3 && (N3 > 1 || !(lane & 4));
        if (N2 > 1) { k += lane & 8 ? N3 : 0; ok = ok && k < N2; } else ok = ok && !(lane & 8);
        if (N1 > 1) { k += lane & 16 ? N2 : 0; ok = ok && k < N1; } else ok = ok && !(lane & 16);
        k += lane & 32 ? N1 : 0;
        ok = ok && k < N;
        if (ok) { hi[(base + k) * stride + col] = h4[0]; lo[(base + k) * stride + col] = l4[0]; }
    }
}
// term k over nw wavefront sums, in wavefront order. Tiles hand on both parts, so
// that the sum over all of them does not depend on how the cells are cut into tiles.
__device__ __forceinline__ void comp_total(const double* hi, const double* lo, int nw, int k, double& h, double& l) {
    h = 0.0; l = 0.0;
    for (int w = 0; w < nw; ++w) comp_add(h, l, hi[k * nw + w], lo[k * nw + w]);
}

// Cell / path slot -> static index, member and instance. MB = false is the
// single-instance handle (one domain, one member): slot = cell, instance 0,
// known at compile time.
struct Slot {
    int c, m, inst;
};
template <bool MB>
__device__ __forceinline__ Slot cell_slot(const DevMap& M, int s) {
    Slot x;
    if (!MB) { x.c = s; x.m = 0; x.inst = 0; return x; }
    x.c = s >> M.lgm;
    x.m = s & (M.nmem - 1);
    int d = 0;
    if (M.ndom_arg > 0) {
        // compare against the offsets in the kernel arguments: no dependent load
        for (int k = 1; k < M.ndom_arg; ++k) d += x.c >= M.dom_off_arg[k];
    } else if (M.cell_dom) {
        d = M.cell_dom[x.c];
    }
    x.inst = d * M.nmem + x.m;
    return x;
}
template <bool MB>
__device__ __forceinline__ Slot path_slot(const DevMap& M, int q) {
    Slot x;
    if (!MB) { x.c = q; x.m = 0; x.inst = 0; return x; }
    x.c = q >> M.lgm;
    x.m = q & (M.nmem - 1);
    x.inst = (M.pth_dom ? M.pth_dom[x.c] * M.nmem : 0) + x.m;
    return x;
}
template <bool MB>
__device__ __forceinline__ int sidx(const DevMap& M, int c, int m) { return MB ? ((c << M.lgm) | m) : c; }

// ---------------------------------------------------------------------------
// Floodplain profile table recomputed on the fly: SET_FLDSTG
// (src/cmf_ctrl_maps_mod.F90:984-995) and, identically, CMF_LEVEE_INIT :169-181.
struct Geom {                 // float32 map values of one cell, widened
    double rivlen, rivwth, grarea, rivhgt;
};
__device__ __forceinline__ Geom load_geom(const DevMap& M, int i) {
    Geom g;
    g.rivlen = (double)M.rivlen[i]; g.rivwth = (double)M.rivwth[i];
    g.grarea = (double)M.grarea[i]; g.rivhgt = (double)M.rivhgt[i];
    return g;
}

// FLDHGT of layer l (1-based) of one cell, from the map planes; the row is formed where
// the layers are asked for, in flooded cells only (formed for all cells it made the
// update 1-3% slower)
struct MapHgt {
    struct Row {
        const float* h;      // &fldhgt[i], stride n
        int n;
        __device__ __forceinline__ float operator()(int l) const { return h[(size_t)(l - 1) * n]; }
    };
    const DevMap& M;
    int i;
    __device__ __forceinline__ MapHgt(const DevMap& map, int cell) : M(map), i(cell) {}
    __device__ __forceinline__ Row row() const { return {M.fldhgt + i, M.n}; }
};
template <class H>
struct FldTab {
    decltype(std::declval<const H&>().row()) h;
    double rivlen, rivwth, dwthinc, stopre, hpre;
    __device__ __forceinline__ FldTab(const DevMap& M, const H& hgt, const Geom& g, double rivstomax) : h(hgt.row()) {
        rivlen = g.rivlen;
        rivwth = g.rivwth;
        dwthinc = (g.grarea * (1.0 / rivlen)) * M.dfrcinc;
        stopre = rivstomax; hpre = 0.0;
    }
    // next layer l (1-based, consecutive calls): FLDSTOMAX(l), FLDGRD(l), FLDHGT(l)
    __device__ __forceinline__ void layer(int l, double& smax, double& grd, double& hgt) {
        const double hl = (double)h(l);
        const double dstonow = (rivlen * (rivwth + dwthinc * ((double)l - 0.5))) * (hl - hpre);
        smax = stopre + dstonow;
        grd = (hl - hpre) * (1.0 / dwthinc);
        hgt = hl;
        stopre = smax; hpre = hl;
    }
};

__device__ __forceinline__ double rivstomax_of(const DevMap& M, int i) {
    // maps:716-721
    return M.lfplain ? ((double)M.rivlen[i] * (double)M.rivwth[i]) * (double)M.rivhgt[i] : K_1E18F;
}
__device__ __forceinline__ double rivstomax_of(const DevMap& M, const Geom& g) {
    return M.lfplain ? (g.rivlen * g.rivwth) * g.rivhgt : K_1E18F;
}
__device__ __forceinline__ double rivelv_of(const DevMap& M, int i) {
    return (double)M.elevtn[i] - (double)M.rivhgt[i];            // maps:722
}

// The two ends of a bifurcation path: riverbed elevations, depths, and for a levee end
// (lev_*) its LEVDPH and ground elevation
template <class R>
struct PathEnds {
    double ri_d, rj_d;
    R di, dj, dpi, dpj;
    bool lev_i = false, lev_j = false;
    R ldi = R(0), ldj = R(0);
    float ei = 0.f, ej = 0.f;
};
// Water surface slope along a path. Surface terms are in difference form with R =
// float: each surface height relative to a level elevation is a depth plus the exact
// FP64 elevation difference rounded once.
template <class R>
__device__ __forceinline__ R path_slope(const PathEnds<R>& e, R dst) {
    constexpr bool kDiff = sizeof(R) == sizeof(float);
    const R si = R(e.ri_d) + e.di, sj = R(e.rj_d) + e.dj;
    const R dslp = (kDiff ? (e.di - e.dj) + R(e.ri_d - e.rj_d) : si - sj) / dst;
    return vmax(R(-0.005), vmin(R(0.005), dslp));
}
// Flow of level l of a path before its limits, pthout:20-83 / levee:497-590.
// load(w, man, pre): width, roughness and the flow before, asked for where the level is wet
template <class R, class Load>
__device__ __forceinline__ R path_level(const PathEnds<R>& e, R dslp, int llevee, int l, double elv_d, R gdt, Load load) {
    constexpr bool kDiff = sizeof(R) == sizeof(float);
    const R zero = R(0), one = R(1);
    // max(si, sj) - elv, max(pi, pj) - elv and max(li, lj) - elv
    R hs, hp, hl;
    if (kDiff) {
        const R ai = R(e.ri_d - elv_d), aj = R(e.rj_d - elv_d);
        hs = vmax(e.di + ai, e.dj + aj);
        hp = vmax(e.dpi + ai, e.dpj + aj);
        const R lvi = e.lev_i ? vmin(e.ldi + R((double)e.ei - elv_d), e.di + ai) : e.di + ai;
        const R lvj = e.lev_j ? vmin(e.ldj + R((double)e.ej - elv_d), e.dj + aj) : e.dj + aj;
        hl = vmax(lvi, lvj);
    } else {
        const R elv = R(elv_d), ri = R(e.ri_d), rj = R(e.rj_d);
        const R si = ri + e.di, sj = rj + e.dj;
        const R li = e.lev_i ? vmin(R(e.ei) + e.ldi, si) : si, lj = e.lev_j ? vmin(R(e.ej) + e.ldj, sj) : sj;   // D2SFCELV_LEV
        hs = vmax(si, sj) - elv;
        hp = vmax(ri + e.dpi, rj + e.dpj) - elv;
        hl = vmax(li, lj) - elv;
    }
    R dflw, dflw_im;
    if (!llevee || l == 0) {
        dflw = vmax(hs, zero);
        const R dflw_pr = vmax(hp, zero);
        dflw_im = vsqrt(dflw * dflw_pr);
        if (llevee) { if (dflw_im <= zero) dflw_im = dflw; }
        else dflw_im = vmax(dflw_im, vsqrt(dflw * R(0.01)));
    } else {
        dflw = vmax(hl, zero);
        dflw_im = dflw;
    }
    if (!(dflw_im > R(1.e-5))) return zero;
    R w, man, pre;
    load(w, man, pre);
    const R dout_pr = (llevee && l > 0) ? pre * (one / w) : pre / w;
    return (w * (dout_pr + (gdt * dflw_im) * dslp)) /
           (one + ((gdt * (man * man)) * vabs(dout_pr)) * vpow(dflw_im, R(K_P7O3)));
}

struct Stage {
    double rivsto, fldsto, levsto;
    double rivdph, flddph, fldfrc, fldare, levdph;
};

// CMF_CALC_FLDSTG_DEF per cell, src/cmf_calc_fldstg_mod.F90:49-95. CLAMP = false:
// the same inversion as CMF_LEVEE_FLDSTG states it for a cell without a levee
// (src/cmf_ctrl_levee_mod.F90:312-349), which does not bound the river storage by
// the total.
template <bool CLAMP = true, class H>
__device__ __forceinline__ void stage_def(const DevMap& M, const H& hgt_of, const Geom& geo, double rivsto,
                                          double fldsto, Stage& o) {
    const double pstoall = rivsto + fldsto;
    const double dstoall = pstoall;
    const double rivstomax = rivstomax_of(M, geo);
    const double rivlen = geo.rivlen, rivwth = geo.rivwth;
    o.levsto = 0.0; o.levdph = 0.0;
    if (pstoall > rivstomax) {
        const int nl = M.nlfp;
        FldTab<H> T(M, hgt_of, geo, rivstomax);
        const double dwth_inc = (geo.grarea / rivlen) * M.dfrcinc;
        int I = 1;
        double dsto_fil = rivstomax, dwth_fil = rivwth, ddph_fil = 0.0;
        double smax, grd, hgt;
        T.layer(1, smax, grd, hgt);
        while (pstoall > smax) {                      // :59-65
            dsto_fil = smax;
            dwth_fil = dwth_fil + dwth_inc;
            ddph_fil = ddph_fil + grd * dwth_inc;
            I = I + 1;
            if (I > nl) break;
            T.layer(I, smax, grd, hgt);
        }
        double dwth_add;
        if (I > nl) {                                 // :66-70
            const double dsto_add = dstoall - dsto_fil;
            dwth_add = 0.0;
            o.flddph = ddph_fil + (dsto_add / dwth_fil) / rivlen;
        } else {                                      // :71-74
            const double dsto_add = dstoall - dsto_fil;
            dwth_add = -dwth_fil + sqrt(dwth_fil * dwth_fil + ((2.0 * dsto_add) / rivlen) / grd);
            o.flddph = ddph_fil + grd * dwth_add;
        }
        double rs = rivstomax + (rivlen * rivwth) * o.flddph;     // :76-77
        if (CLAMP) rs = vmin(rs, pstoall);
        o.rivsto = rs;
        o.rivdph = (rs / rivlen) / rivwth;
        const double fs = pstoall - rs;
        o.fldsto = vmax(fs, 0.0);
        double fr = ((-rivwth + dwth_fil) + dwth_add) / (dwth_inc * (double)nl);
        fr = vmax(fr, 0.0);
        fr = vmin(fr, 1.0);
        o.fldfrc = fr;
        o.fldare = geo.grarea * fr;
    } else {                                          // :87-95
        o.rivsto = pstoall;
        const double d = (dstoall / rivlen) / rivwth;
        o.rivdph = vmax(d, 0.0);
        o.fldsto = 0.0; o.flddph = 0.0; o.fldfrc = 0.0; o.fldare = 0.0;
    }
}

// levee parameters of one cell (sentinels of CMF_LEVEE_INIT for cells without one)
struct Lev {
    double levhgt, levfrc, bashgt, levdst, levbassto, levtopsto, levfilsto;
};
__device__ __forceinline__ Lev load_lev_row(const DevMap& M, int li) {
    Lev L{0.0, 1.0, K_LEVSENT, K_LEVSENT, K_LEVSENT, K_LEVSENT, K_LEVSENT};
    const int nlc = M.nlevcell;
    if (li >= 0) {
        L.levhgt = M.lev_tab[li]; L.levfrc = M.lev_tab[nlc + li]; L.bashgt = M.lev_tab[2 * nlc + li];
        L.levdst = M.lev_tab[3 * nlc + li]; L.levbassto = M.lev_tab[4 * nlc + li];
        L.levtopsto = M.lev_tab[5 * nlc + li]; L.levfilsto = M.lev_tab[6 * nlc + li];
    }
    return L;
}
__device__ __forceinline__ Lev load_lev(const DevMap& M, int i) { return load_lev_row(M, M.lev_idx[i]); }

// CMF_LEVEE_FLDSTG per cell, src/cmf_ctrl_levee_mod.F90:302-473. Every case
// computes the same eight local values and the result is written once, so the
// compiler keeps the whole inversion in registers.
template <class H>
__device__ __forceinline__ void stage_levee(const DevMap& M, const H& hgt_of, const Geom& geo, const Lev& L,
                                            double rivsto, double fldsto, double levsto, Stage& o) {
    const int nl = M.nlfp;
    const double levhgt = L.levhgt, levfrc = L.levfrc, bashgt = L.bashgt, levdst = L.levdst;
    const double levbassto = L.levbassto, levtopsto = L.levtopsto, levfilsto = L.levfilsto;
    const double pstoall = (rivsto + fldsto) + levsto;
    const double dstoall = pstoall;
    const double rivstomax = rivstomax_of(M, geo);
    const double rl = geo.rivlen, rw = geo.rivwth, ga = geo.grarea;
    const double dwth_inc = (ga / rl) * M.dfrcinc;
    double r_riv = 0.0, r_fld = 0.0, r_lev = 0.0, r_rdph = 0.0, r_fdph = 0.0, r_frc = 0.0, r_are = 0.0,
           r_ldph = 0.0;
    // case selection (:308-311): 0 in bank; 1 below the levee base; 2 river side
    // below the crown; 3 protected side filling; 4 above the protected-side fill
    int kase;
    if (!(dstoall > rivstomax)) kase = 0;
    else if (dstoall < levbassto) kase = 1;
    else if (dstoall < levtopsto) kase = 2;
    else if (dstoall < levfilsto) kase = 3;
    else kase = 4;
    if (kase == 1 || kase == 4) {
        // case 1 (:312-349) and case 4 (:424-461) share the layer search
        FldTab<H> T(M, hgt_of, geo, rivstomax);
        int I = 1;
        double dsto_fil = rivstomax, dwth_fil = rw, ddph_fil = 0.0, dwth_add;
        double smax, grd, hgt;
        T.layer(1, smax, grd, hgt);
        while (dstoall > smax) {
            dsto_fil = smax;
            dwth_fil = dwth_fil + dwth_inc;
            ddph_fil = ddph_fil + grd * dwth_inc;
            I = I + 1;
            if (I > nl) break;
            T.layer(I, smax, grd, hgt);
        }
        if (I <= nl) {
            const double dsto_add = dstoall - dsto_fil;
            dwth_add = -dwth_fil + sqrt(dwth_fil * dwth_fil + ((2.0 * dsto_add) / rl) / grd);
            r_fdph = ddph_fil + grd * dwth_add;
        } else {
            const double dsto_add = dstoall - dsto_fil;
            dwth_add = 0.0;
            r_fdph = ddph_fil + (dsto_add / dwth_fil) / rl;
        }
        if (kase == 1) {
            r_riv = rivstomax + (rl * rw) * r_fdph;
            r_rdph = (r_riv / rl) / rw;
            const double fs = pstoall - r_riv;
            r_fld = vmax(fs, 0.0);
            double fr = ((-rw + dwth_fil) + dwth_add) / (dwth_inc * (double)nl);
            fr = vmax(fr, 0.0);
            fr = vmin(fr, 1.0);
            r_frc = fr;
            r_are = ga * fr;
        } else {
            r_frc = ((-rw + dwth_fil) + dwth_add) / (dwth_inc * (double)nl);
            r_are = ga * r_frc;
            r_riv = rivstomax + (rl * rw) * r_fdph;
            r_rdph = (r_riv / rl) / rw;
            const double dsto_add = ((r_fdph - levhgt) * (levdst + rw)) * rl;
            const double fs = (levtopsto + dsto_add) - r_riv;
            r_fld = vmax(fs, 0.0);
            const double ls = (pstoall - r_riv) - r_fld;
            r_lev = vmax(ls, 0.0);
            r_ldph = r_fdph;
        }
    } else if (kase == 2) {                           // (:353-368)
        const double dsto_add = dstoall - levbassto;
        const double dwth_add = levdst + rw;
        r_fdph = bashgt + (dsto_add / dwth_add) / rl;
        r_riv = rivstomax + (rl * rw) * r_fdph;
        r_rdph = (r_riv / rl) / rw;
        const double fs = pstoall - r_riv;
        r_fld = vmax(fs, 0.0);
        r_frc = levfrc;
        r_are = ga * r_frc;
    } else if (kase == 3) {                           // (:372-420): river side full
        r_fdph = levhgt;
        r_riv = rivstomax + (rl * rw) * r_fdph;
        r_rdph = (r_riv / rl) / rw;
        const double fs = levtopsto - r_riv;
        r_fld = vmax(fs, 0.0);
        const double ls = (pstoall - r_riv) - r_fld;
        r_lev = vmax(ls, 0.0);
        const int ilev = (int)(levfrc * (double)nl) + 1;
        double dsto_fil = levtopsto, dwth_fil = 0.0, ddph_fil = 0.0;
        FldTab<H> T(M, hgt_of, geo, rivstomax);
        double smax = 0.0, grd = 0.0, hgt = 0.0;
        for (int l = 1; l < ilev && l <= nl; ++l) T.layer(l, smax, grd, hgt);
        int I = ilev;
        while (I <= nl) {
            T.layer(I, smax, grd, hgt);
            const double dsto_add = ((levdst + rw) * (levhgt - hgt)) * rl;
            if (dstoall < smax + dsto_add) break;
            dsto_fil = smax + dsto_add;
            dwth_fil = dwth_inc * (double)I - levdst;
            ddph_fil = hgt - bashgt;
            I = I + 1;
        }
        if (I <= nl) {
            const double dsto_add = dstoall - dsto_fil;
            const double dwth_add = -dwth_fil + sqrt(dwth_fil * dwth_fil + ((2.0 * dsto_add) / rl) / grd);
            const double ddph_add = dwth_add * grd;
            r_ldph = (bashgt + ddph_fil) + ddph_add;
            double fr = (dwth_fil + levdst) / (dwth_inc * (double)nl);
            fr = vmax(fr, 0.0);
            fr = vmin(fr, 1.0);
            r_frc = fr;
            r_are = ga * fr;
        } else {
            const double dsto_add = dstoall - dsto_fil;
            const double ddph_add = (dsto_add / dwth_fil) / rl;
            r_ldph = (bashgt + ddph_fil) + ddph_add;
            r_frc = 1.0;
            r_are = ga * r_frc;
        }
    } else {                                          // case 0 (:463-473)
        r_riv = pstoall;
        const double d = (dstoall / rl) / rw;
        r_rdph = vmax(d, 0.0);
    }
    o.rivsto = r_riv; o.fldsto = r_fld; o.levsto = r_lev;
    o.rivdph = r_rdph; o.flddph = r_fdph; o.fldfrc = r_frc; o.fldare = r_are; o.levdph = r_ldph;
}

// ---------------------------------------------------------------------------
// CMF_CALC_OUTFLW per cell, src/cmf_calc_outflw_mod.F90:45-182, from values in
// registers: the water surface (surface_of), RIVVEL (river_vel), river (or mouth)
// and floodplain flow and the reverse-flow storage limiter (local_inertial).
template <class R>
struct FlowIn {
    R rivdph, rivdph_pre, qr_pre, qr_old;      // D2RIVOUT_PRE, D2RIVOUT (for RIVVEL)
    R fldsto, flddph, fldsto_pre, fldout_pre;  // floodplain terms (LFLDOUT)
    R storge;
    float elevtn, rivhgt, rivwth, rivman, nxtdst, rivlen;
    bool river;                                // has a downstream cell
    R dj, dj_pre;                              // its RIVDPH, RIVDPH_PRE
    double zdn;                                // its RIVELV; mouths: DWNELV
};

//   hs  = SFCELV - DWNELV          (slope numerator)
//   hr  = max(SFCELV, DWNELV) - RIVELV,  hrp the same with the _PRE values
//   (mouths: hr = RIVDPH, hrp = RIVDPH_PRE)
//   fa  = surface above ELEVTN for the floodplain (outflw:88, :147), fap the _PRE one
template <class R>
struct Surface {
    R hs, hr, hrp, fa, fap;
    R dflw_im;                                 // semi-implicit flow depth
    R dare;                                    // flow area
    bool wet;                                  // deep enough to flow
};
template <class R>
__device__ __forceinline__ Surface<R> surface_of(const FlowIn<R>& c) {
    const R rivdph = c.rivdph, rivdph_pre = c.rivdph_pre;
    // Water-surface terms of outflw:45-58. With R = double they are evaluated as
    // the reference writes them (SFCELV = RIVELV + RIVDPH, slopes and depths from
    // SFCELV). With R = float the same quantities are formed from depths and the
    // exact FP64 elevation difference, rounded once: a ~250 m surface elevation
    // keeps only ~1.5e-5 m in FP32, which the slope (a difference of a few cm)
    // would otherwise inherit.
    R hs, hr, hrp, fa, fap;
    if (sizeof(R) == sizeof(double)) {
        const R rivelv = R((double)c.elevtn - (double)c.rivhgt);    // maps:722
        const R elevtn = R(c.elevtn);
        const R sfcelv = rivelv + rivdph;                           // outflw:45-47
        const R sfcelv_pre = rivelv + rivdph_pre;
        if (c.river) {                                               // outflw:52-57
            const R rivelv_j = R(c.zdn);
            const R dwn = rivelv_j + c.dj;
            const R dwn_pre = rivelv_j + c.dj_pre;
            const R dsfc = vmax(sfcelv, dwn), dsfc_pr = vmax(sfcelv_pre, dwn_pre);
            hs = sfcelv - dwn;
            hr = dsfc - rivelv;
            hrp = dsfc_pr - rivelv;
            fa = dsfc - elevtn;
            fap = dsfc_pr - elevtn;
        } else {
            hs = sfcelv - R(c.zdn);
            hr = rivdph;
            hrp = rivdph_pre;
            fa = sfcelv - elevtn;
            fap = sfcelv_pre - elevtn;
        }
    } else {
        const double e_i = (double)c.elevtn - (double)c.rivhgt;
        const R dz = R(c.zdn - e_i);                                 // RIVELV(j) or DWNELV above RIVELV(i)
        if (c.river) {
            hs = (rivdph - c.dj) - dz;
            hr = vmax(rivdph, dz + c.dj);
            hrp = vmax(rivdph_pre, dz + c.dj_pre);
        } else {
            hs = rivdph - dz;
            hr = rivdph;
            hrp = rivdph_pre;
        }
        const R hgt = R(c.rivhgt);                                   // ELEVTN = RIVELV + RIVHGT
        fa = hr - hgt;
        fap = hrp - hgt;
    }
    Surface<R> f;
    f.hs = hs; f.hr = hr; f.hrp = hrp; f.fa = fa; f.fap = fap;
    R dare = R(c.rivwth) * hr;                                       // outflw:60-66, :119-125
    f.dare = vmax(dare, R(1.e-10));
    R dflw_im = vsqrt(hr * hrp);
    f.dflw_im = vmax(dflw_im, R(1.e-6));
    f.wet = (f.dflw_im > R(K_1EM5F)) && (f.dare > R(K_1EM5F));
    return f;
}
// RIVVEL of outflw:75, :134 (from the flow before this substep)
template <class R>
__device__ __forceinline__ R river_vel(const FlowIn<R>& c, const Surface<R>& f) {
    const R dvel = c.qr_old * (R(1) / f.dare);
    return f.wet ? dvel : R(0);
}

template <class R>
__device__ __forceinline__ void local_inertial(const FlowIn<R>& c, const Surface<R>& sf, int lfldout, double pmanfld,
                                               double pdstmth, double dt, double gdt_d, R& q_r, R& q_f) {
    const R zero = R(0), one = R(1);
    const R gdt = R(gdt_d);
    const R rivwth = R(c.rivwth), rivman = R(c.rivman);
    const R rdst = one / (c.river ? R(c.nxtdst) : R(pdstmth));
    const R hs = sf.hs;
    q_f = zero;
    // ---- river channel: outflw:60-80 (river), :119-139 (mouth)
    {
        const R dslp = hs * rdst;
        const R dout_pr = c.qr_pre * (one / rivwth);
        const R dout = (rivwth * (dout_pr + (gdt * sf.dflw_im) * dslp)) *
                       (one / (one + ((gdt * (rivman * rivman)) * vabs(dout_pr)) * vpow(sf.dflw_im, R(K_P7O3))));
        q_r = sf.wet ? dout : zero;
    }
    // ---- floodplain: outflw:84-116 (river), :143-171 (mouth). Surface heights
    // above ELEVTN = RIVELV + RIVHGT: max(SFCELV, DWNELV) - ELEVTN = hr - RIVHGT.
    if (lfldout) {
        const R gdtn2 = gdt * (R(pmanfld) * R(pmanfld));
        const R flddph_pre = vmax(c.rivdph_pre - R(c.rivhgt), zero);
        const R rrl = one / R(c.rivlen);
        R dslp = hs * rdst;
        dslp = vmax(R(-0.005), vmin(R(0.005), dslp));
        const R dflw = c.river ? vmax(sf.fa, zero) : sf.fa, dflw_pr = sf.fap;
        const R dare = vmax(c.fldsto * rrl - c.flddph * rivwth, zero);
        const R dare_pr = vmax(c.fldsto_pre * rrl - flddph_pre * rivwth, R(1.e-6));
        const R t = dflw * dflw_pr;
        R dflw_im = vsqrt(vmax(t, zero));
        dflw_im = vmax(dflw_im, R(1.e-6));
        R dare_im = vsqrt(dare * dare_pr);
        dare_im = vmax(dare_im, R(1.e-6));
        const R dout_pr = c.fldout_pre;
        const R thr = c.river ? R(1.e-5) : R(K_1EM5F);
        const R dout = (dout_pr + (gdt * dare_im) * dslp) *
                       (one / (one + ((gdtn2 * vabs(dout_pr)) * vpow(dflw_im, R(K_P4O3))) * (one / dare_im)));
        const bool mask = (dflw_im > thr) && (dare > thr);
        const R f = mask ? dout : zero;
        q_f = (f * q_r > zero) ? f : zero;
    }
    // ---- reverse-flow storage limiter, river cells: outflw:175-182
    if (c.river) {
        R dout = ((-q_r) - q_f) * R(dt);
        dout = vmax(dout, R(K_1EM10F));
        R rate = (R(0.05) * c.storge) / dout;
        rate = vmin(rate, one);
        q_r = q_r * rate;
        q_f = q_f * rate;
    }
}

// Hanazaki-2022 reservoir operation (LDAMH22), src/cmf_ctrl_damout_mod.F90:354-378,
// before the storage limiter. Zones: normal (<= NorVol), water supply (<= ConVol),
// flood control (< EmeVol), emergency. r_volupa is the dam's own flood-control
// volume over its upstream area (damout:204 stores every dam's ratio at index NDAM;
// here each dam reads its own). Default-real constants 1. and 0.2 widened.
__device__ __forceinline__ double dam_rule_h22(double vol, double inflow, double norvol, double convol,
                                               double emevol, double qn, double qf, double r_volupa) {
    if (vol <= norvol) return qn * (vol / convol);
    const double quad = (vol - norvol) / (emevol - norvol);        // ((V-NorVol)/(EmeVol-NorVol))**2
    const double pre = qn * 0.5 + (quad * quad) * (qf - qn);
    if (vol <= convol) {
        if (qf <= inflow) return qn * 0.5 + ((vol - norvol) / (convol - norvol)) * (qf - qn);
        return pre;
    }
    if (vol < emevol) {
        if (qf <= inflow) {
            const double cut = vmax(1.0 - r_volupa / K_0P2F, 0.0);
            return qf + ((cut * (vol - convol)) / (emevol - convol)) * (inflow - qf);
        }
        return pre;
    }
    return vmax(inflow, qf);
}

__device__ __attribute__((noinline)) static double rare_pow(double x, double y) { return pow(x, y); }

// Manning factors of the kinematic wave in a cell i above a dam (damout:471-480):
// (1/n) S^(1/2) of the river and, with the slope bounded by 0.005, of the
// floodplain; j its downstream cell.
__device__ __forceinline__ void dam_kine_factors(const DevMap& M, double pminslp, double pmanfld, int i, int j,
                                                 double& vk, double& vf) {
    double dslope = ((double)M.elevtn[i] - (double)M.elevtn[j]) * (1.0 / (double)M.nxtdst[i]);
    dslope = vmax(dslope, pminslp);
    vk = (1.0 / (double)M.rivman[i]) * sqrt(dslope);
    const double dslope_f = vmin(0.005, dslope);
    vf = (1.0 / pmanfld) * sqrt(dslope_f);
}

// Outflow of a cell with I1DAM > 0 (damout:344-419, :466-493) from its DAMINF:
// nothing by default; the kinematic wave (factors vk, vf) where `kine` is set; the
// operation rule of dam row d (Yamazaki & Funato or Hanazaki-2022) where `active`.
template <class R>
__device__ __forceinline__ void dam_outflow(const DevMap& M, bool kine, double vk, double vf, float rivwth,
                                            float rivlen, bool active, int d, double inf, double dt, R rivdph,
                                            R flddph, double rivsto, double fldsto, double damsto, R& q_r, R& q_f,
                                            R& vel) {
    q_r = R(0); q_f = R(0);
    if (kine) {                                                  // :471-493
        const double rd = (double)rivdph;
        const double dvel = vk * rare_pow(rd, K_2O3F);
        const double darea = (double)rivwth * rd;
        vel = R(dvel);
        double q = darea * dvel;
        q_r = R(vmin(q, rivsto / dt));
        const double fd = (double)flddph;
        // most floodplains above a dam are dry, and the wavefront of these cells is what
        // a block waits for: 1,500,120 cells with 2,500 dams and levees, mixed, 680
        // substeps 67.1 -> 62.1 ms without the second power
        const double dvel_f = vf * (fd == 0.0 ? 0.0 : rare_pow(fd, K_2O3F));
        double dare_f = fldsto * (1.0 / (double)rivlen);
        dare_f = vmax(dare_f - fd * (double)rivwth, 0.0);
        const double qf = dare_f * dvel_f;
        q_f = R(vmin(qf, fldsto / dt));
    }
    if (active) {                                                // :344-419
        const double vol = damsto;
        const double cv = M.dam_convol[d], av = M.dam_adjvol[d], ev = M.dam_emevol[d];
        const double qn = M.dam_qn[d], qf = M.dam_qf[d], qa = M.dam_qa[d];
        double out = 0.0;
        if (M.ldamh22) {
            out = dam_rule_h22(vol, inf, M.dam_norvol[d], cv, ev, qn, qf, M.dam_r_volupa[d]);
        } else if (vol <= cv) {
            out = qn * sqrt(vol / cv);
        } else if (vol > cv && vol <= av) {
            const double xx = (vol - cv) / (av - cv);
            out = qn + (xx * (xx * xx)) * (qa - qn);
        } else if (vol > av && vol <= ev) {
            const double tmp = qa + rare_pow((vol - av) / (ev - av), K_0P1F) * (qf - qa);
            if (inf >= qf) {
                out = qn + ((vol - cv) / (ev - cv)) * (inf - qn);
                out = vmax(out, tmp);
            } else {
                out = tmp;
            }
        } else if (vol > ev) {
            out = (inf >= qf) ? inf : qf;
        }
        out = vmin(vmin(out, vol / dt), (rivsto + fldsto) / dt);
        out = vmax(out, 0.0);
        q_r = R(out);
        q_f = R(0);
    }
}

// CMF_CALC_STONXT per cell, src/cmf_calc_stonxt_mod.F90:54-98: the storages rs, fs
// before the stage inversion, and the budget terms it forms. rinf, finf, pout are
// the FP64 inflows and path outflow, qrl, qfl the limited outflows.
template <class R>
__device__ __forceinline__ void storage_next(double& rs, double& fs, double rinf, double finf, double pout, R qrl,
                                             R qfl, double dt, R runoff, R fldfrc, int lupsinf, R upsinf,
                                             double (&g)[NGLB]) {
    g[G_STOPRE] = rs + fs;
    g[G_RIVINF] = rinf * dt + finf * dt;
    g[G_RIVOUT] = ((double)qrl * dt + (double)qfl * dt) + pout * dt;
    rs = (rs + rinf * dt) - (double)qrl * dt;
    if (rs < 0.0) { fs = fs + rs; rs = 0.0; }
    fs = ((fs + finf * dt) - (double)qfl * dt) - pout * dt;
    if (fs < 0.0) { rs = vmax(rs + fs, 0.0); fs = 0.0; }
    g[G_STONXT] = rs + fs;
    R drivrof = (runoff * (R(1) - fldfrc)) * R(dt);
    const R dfldrof = (runoff * fldfrc) * R(dt);
    if (lupsinf) drivrof = drivrof + upsinf * R(dt);               // stonxt:81
    rs = rs + (double)drivrof;
    fs = fs + (double)dfldrof;
}

}  // namespace cmf
