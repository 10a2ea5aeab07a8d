// kh_step.hpp -- device code shared by the stage update (kh_update.hip) and the
// task-level kernels (kh_step.hip): ghost images, zone indices, the geometric
// source, flux divergence, the tiles of the curved-space kernels.
#pragma once
#include <cfloat>

#include "kh_internal.hpp"

namespace kh {

static constexpr int BS = 256;
static inline dim3 grid_for(long n, int bs = BS) { return dim3((unsigned)((n + bs - 1) / bs)); }
static inline long ninterior_host(const BlockDims& b) {
    return (long)b.nx1 * (b.ndim > 1 ? b.nx2 : 1) * (b.ndim > 2 ? b.nx3 : 1);
}

// ------------------------------------------------------------ ghost images
// Images of interior zone (k,j,i) in ghost regions: per axis, the zone's
// offset in the image block's layout (0 = no image) and the index offset of
// that block (0: this block, a periodic axis of a one-block mesh; otherwise
// the neighbour across the face the zone lies within ng of).  With nx >= 2 ng
// on every image axis a zone has at most one image per axis, so up to 7 image
// copies (edges and corners land in the diagonal neighbour, whose block offset
// is the sum of the axes' offsets).
struct ImageSet {
    long oi, oj, ok;
    int bi, bj, bk;
};
__device__ __forceinline__ void image_set(const BlockDims& b, int k, int j, int i, ImageSet& s) {
    s.oi = s.oj = s.ok = 0;
    s.bi = s.bj = s.bk = 0;
    if (b.img[0][0] && i - b.is < b.ng) { s.oi = b.nx1; s.bi = b.nbd[0][0]; }
    else if (b.img[0][1] && b.ie - i < b.ng) { s.oi = -b.nx1; s.bi = b.nbd[0][1]; }
    if (b.ndim > 1) {
        if (b.img[1][0] && j - b.js < b.ng) { s.oj = (long)b.nx2 * b.s2; s.bj = b.nbd[1][0]; }
        else if (b.img[1][1] && b.je - j < b.ng) { s.oj = -(long)b.nx2 * b.s2; s.bj = b.nbd[1][1]; }
    }
    if (b.ndim > 2) {
        if (b.img[2][0] && k - b.ks < b.ng) { s.ok = (long)b.nx3 * b.s3; s.bk = b.nbd[2][0]; }
        else if (b.img[2][1] && b.ke - k < b.ng) { s.ok = -(long)b.nx3 * b.s3; s.bk = b.nbd[2][1]; }
    }
}
// base[c] = val and the same at every image; bstride: elements between the
// same array of consecutive blocks (NV nc for a state, nc for a flag array).
template <typename T>
__device__ __forceinline__ void store_with_images(const BlockDims&, const ImageSet& s, T* base, long c, T val,
                                                  long bstride) {
    base[c] = val;
    if ((s.oi | s.oj | s.ok) == 0) return;
    const long di = s.oi + s.bi * bstride, dj = s.oj + s.bj * bstride, dk = s.ok + s.bk * bstride;
    if (s.oi) base[c + di] = val;
    if (s.oj) base[c + dj] = val;
    if (s.ok) base[c + dk] = val;
    if (s.oi && s.oj) base[c + di + dj] = val;
    if (s.oi && s.ok) base[c + di + dk] = val;
    if (s.oj && s.ok) base[c + dj + dk] = val;
    if (s.oi && s.oj && s.ok) base[c + di + dj + dk] = val;
}

__device__ __forceinline__ void interior_index(const BlockDims& b, unsigned t, int& k, int& j, int& i) {
    const unsigned nij = (unsigned)b.nx1 * (unsigned)(b.ndim > 1 ? b.nx2 : 1);
    const unsigned kk = t / nij;
    const unsigned rem = t - kk * nij;
    const unsigned jj = rem / (unsigned)b.nx1;
    i = b.is + (int)(rem - jj * (unsigned)b.nx1);
    j = b.js + (int)jj;
    k = b.ks + (int)kk;
}
__device__ __forceinline__ long ninterior(const BlockDims& b) {
    return (long)b.nx1 * (b.ndim > 1 ? b.nx2 : 1) * (b.ndim > 2 ? b.nx3 : 1);
}

// Metric of cell centre (j, i): flat, or read from the geometry cache.
template <int GEO, class Fn>
__device__ __forceinline__ void with_center_geom(const GeomDev& gd, int j, int i, Fn&& fn) {
    if constexpr (GEO) {
        CachedGeom<double> g(gd.g[GLOC_CENTER], gd.np, (long)j * gd.gn1 + i);
        fn(g);
    } else {
        MinkowskiGeom<double> g;
        fn(g);
    }
}
// Geometric floors of cell centre (j, i) (floors_functions.hpp:97-108)
template <int GEO>
__device__ __forceinline__ void geom_floors(const StepConsts& c, const GeomDev& gd, int j, int i, double& rf, double& uf) {
    if constexpr (GEO) {
        const long q = (long)j * gd.gn1 + i;
        rf = gd.flr[q];
        uf = gd.flr[gd.np + q];
    } else {
        rf = c.floors.rho_min_const;
        uf = c.floors.u_min_const;
    }
}
// KDomain::GetPhysicalRange (domain.hpp:161-187): the entire block, less the
// ghosts across physical-boundary faces (the ghosts of periodic faces and of
// faces shared with another block are in range).
__device__ __forceinline__ bool in_physical(const BlockDims& b, int k, int j, int i) {
    if (i < 0 || i >= b.n1 || j < 0 || j >= b.n2 || k < 0 || k >= b.n3) return false;
    if ((i < b.is && !b.img[0][0]) || (i > b.ie && !b.img[0][1])) return false;
    if (b.ndim > 1 && ((j < b.js && !b.img[1][0]) || (j > b.je && !b.img[1][1]))) return false;
    if (b.ndim > 2 && ((k < b.ks && !b.img[2][0]) || (k > b.ke && !b.img[2][1]))) return false;
    return true;
}

// Flux::AddGeoSource (flux/flux.cpp:395-444): the T^mu_nu Gamma contraction of
// zone (j, i) added to the energy and momentum rates,
// S_lam = sum_{mu, nu} T^mu_nu sqrt(-g) Gamma^nu_{lam mu}.  conn holds
// sqrt(-g) Gamma^a_{b c} at index 16 a + 4 b + c, exactly symmetric in (b, c)
// (the geometry build stores the mean of the two finite-difference orders), so
// each of the 40 distinct components is loaded once and serves both (lam, mu)
// and (mu, lam): 40 loads instead of 64 (the reference sums all 64; the sum
// here differs from it by rounding only).  No test for zero components: a
// branch per component would make every load wait for the one before it.
// conn(n) returns component n = 16 a + 4 b + c of this zone's table.
template <class G, class C>
__device__ __forceinline__ void add_geo_source_c(const G& g, const C& conn, const double Psub[NV], double gam,
                                                 double dudt[NV]) {
    FourVec<double> D;
    calc_4vecs<double>(g, Psub, D);
    const double bsq = bsq_of<G>(D.bcon, D.bcov);
    const double pgas = (gam - 1.) * Psub[UU];
    const double eta = pgas + Psub[RHO] + Psub[UU] + bsq;
    const double ptot = pgas + 0.5 * bsq;
    double nd[4] = {0., 0., 0., 0.};
    double T[4][4];   // T^mu_nu
#pragma unroll
    for (int mu = 0; mu < 4; ++mu)
#pragma unroll
        for (int nu = 0; nu < 4; ++nu) T[mu][nu] = eta * D.ucon[mu] * D.ucov[nu] + (mu == nu ? ptot : 0.) - D.bcon[mu] * D.bcov[nu];
#pragma unroll
    for (int nu = 0; nu < 4; ++nu) {
        double cs[10];
#pragma unroll
        for (int lam = 0, n = 0; lam < 4; ++lam)
#pragma unroll
            for (int mu = lam; mu < 4; ++mu, ++n) cs[n] = conn(nu * 16 + lam * 4 + mu);
#pragma unroll
        for (int lam = 0, n = 0; lam < 4; ++lam)
#pragma unroll
            for (int mu = lam; mu < 4; ++mu, ++n) {
                nd[lam] += T[mu][nu] * cs[n];
                if (mu != lam) nd[mu] += T[lam][nu] * cs[n];
            }
    }
    dudt[UU] += nd[0];
    dudt[U1] += nd[1];
    dudt[U2] += nd[2];
    dudt[U3] += nd[3];
}
template <class G>
__device__ __forceinline__ void add_geo_source(const G& g, const GeomDev& gd, long q, const double Psub[NV], double gam,
                                               double dudt[NV]) {
    add_geo_source_c(g, [&](int n) { return gd.conn[(long)n * gd.np + q]; }, Psub, gam, dudt);
}


// Flux divergence of all 8 variables of zone c (FluxDivHelper form:
// -(sum_d A_d (F_d(hi) - F_d(lo))) / V), with the flux-CT B fluxes
// evaluated from the EMFs when `ct` is set.
template <typename R>
__device__ __forceinline__ void zone_divergence(const BlockDims& b, const FluxVars<const R>& F, const R* __restrict__ emf,
                                                long c, bool ct, double dudt[NV], bool skip_b = false) {
    const double A1 = b.dx2 * b.dx3, A2 = b.dx1 * b.dx3, A3 = b.dx1 * b.dx2, V = b.dx1 * b.dx2 * b.dx3;
    const double iV = 1. / V;   // one division per zone instead of eight
    const Vars<const R>& F1 = F[0];
    const Vars<const R>& F2 = F[1];
    const Vars<const R>& F3 = F[2];
    const long s2 = b.s2, s3 = b.s3;
    const int nd = b.ndim;
    double f1lo[NV], f1hi[NV], f2lo[NV], f2hi[NV], f3lo[NV], f3hi[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        f1lo[v] = f1hi[v] = f2lo[v] = f2hi[v] = f3lo[v] = f3hi[v] = 0.;
        if (skip_b && v >= B1) continue;   // face-centred B: the cell B comes from the faces
        f1lo[v] = (double)F1[v][c];
        f1hi[v] = (double)F1[v][c + 1];
        if (nd >= 2 && !(ct && v >= B1)) { f2lo[v] = (double)F2[v][c]; f2hi[v] = (double)F2[v][c + s2]; }
        if (nd == 3 && !(ct && v >= B1)) { f3lo[v] = (double)F3[v][c]; f3hi[v] = (double)F3[v][c + s3]; }
    }
    if (ct) {
        const R* e1 = emf;
        const R* e2 = emf + b.nc;
        const R* e3 = emf + 2 * b.nc;
        f1lo[B1] = 0.; f1hi[B1] = 0.;
        f1lo[B2] = (double)(R(0.5) * (e3[c] + e3[c + s2]));
        f1hi[B2] = (double)(R(0.5) * (e3[c + 1] + e3[c + 1 + s2]));
        f2lo[B1] = (double)(R(-0.5) * (e3[c] + e3[c + 1]));
        f2hi[B1] = (double)(R(-0.5) * (e3[c + s2] + e3[c + s2 + 1]));
        f2lo[B2] = 0.; f2hi[B2] = 0.;
        if (nd == 3) {
            f1lo[B3] = (double)(R(-0.5) * (e2[c] + e2[c + s3]));
            f1hi[B3] = (double)(R(-0.5) * (e2[c + 1] + e2[c + 1 + s3]));
            f2lo[B3] = (double)(R(0.5) * (e1[c] + e1[c + s3]));
            f2hi[B3] = (double)(R(0.5) * (e1[c + s2] + e1[c + s2 + s3]));
            f3lo[B1] = (double)(R(0.5) * (e2[c] + e2[c + 1]));
            f3hi[B1] = (double)(R(0.5) * (e2[c + s3] + e2[c + s3 + 1]));
            f3lo[B2] = (double)(R(-0.5) * (e1[c] + e1[c + s2]));
            f3hi[B2] = (double)(R(-0.5) * (e1[c + s3] + e1[c + s3 + s2]));
            f3lo[B3] = 0.; f3hi[B3] = 0.;
        } else {
            // 2D: B3 keeps its Riemann fluxes
            f2lo[B3] = (double)F2[B3][c];
            f2hi[B3] = (double)F2[B3][c + s2];
        }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        double du = (A1 * f1hi[v] - A1 * f1lo[v]);
        if (nd >= 2) du += (A2 * f2hi[v] - A2 * f2lo[v]);
        if (nd == 3) du += (A3 * f3hi[v] - A3 * f3lo[v]);
        dudt[v] = -du * iV;
    }
}

__device__ __forceinline__ double zone_ndt(const BlockDims& b, double c1, double c2, double c3) {
    // GRMHD::EstimateTimestep, grmhd.cpp:320-322, with c_d = max(cmax_d, cmin_d)
    return 1.0 / (1 / (b.dx1 / c1) + 1 / (b.dx2 / c2) + 1 / (b.dx3 / c3));
}

// Block-wide min / max (wavefront shuffles, then LDS across the block's waves).
__device__ __forceinline__ double block_min(double v) {
    __shared__ double red[1024 / 64];
    v = wave_min(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    double m = red[0];
    for (int q = 1; q < (int)(blockDim.x >> 6); ++q) m = fmin(m, red[q]);
    return m;
}
__device__ __forceinline__ double block_max(double v) {
    __shared__ double red[1024 / 64];
    v = wave_max(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    double m = red[0];
    for (int q = 1; q < (int)(blockDim.x >> 6); ++q) m = fmax(m, red[q]);
    return m;
}

// Corner EMFs of flux-CT (b_flux_ct.cpp:331-342) evaluated from the Riemann
// B fluxes at corner c.
template <typename R>
__device__ __forceinline__ R emf3_at(const R* F1B2, const R* F2B1, long c, long s2) {
    return R(0.25) * (F1B2[c] + F1B2[c - s2] - F2B1[c] - F2B1[c - 1]);
}
template <typename R>
__device__ __forceinline__ R emf1_at(const R* F2B3, const R* F3B2, long c, long s2, long s3) {
    return R(0.25) * (F2B3[c] + F2B3[c - s3] - F3B2[c] - F3B2[c - s2]);
}
template <typename R>
__device__ __forceinline__ R emf2_at(const R* F3B1, const R* F1B3, long c, long s3) {
    return R(0.25) * (F3B1[c] + F3B1[c - 1] - F1B3[c] - F1B3[c - s3]);
}

// Divergence of zone c with the flux-CT B fluxes (b_flux_ct.cpp:347-369) built
// from EMFs computed here from the Riemann fluxes, so neither the EMFs nor the
// rewritten B fluxes make a trip through HBM.
// ND (2 or 3) fixes the dimensionality at compile time; ND = 0 reads b.ndim.
template <typename R, int ND = 0>
__device__ __forceinline__ void zone_divergence_ct(const BlockDims& b, const R* __restrict__ F, long c, double dudt[NV]) {
    const double A1 = b.dx2 * b.dx3, A2 = b.dx1 * b.dx3, A3 = b.dx1 * b.dx2, V = b.dx1 * b.dx2 * b.dx3;
    const double iV = 1. / V;   // one division per zone instead of eight
    const R* F1 = F;
    const R* F2 = F + 8 * b.nc;
    const R* F3 = F + 16 * b.nc;
    const long s2 = b.s2, s3 = b.s3, nc = b.nc;
    const int nd = ND ? ND : b.ndim;
    double f1lo[NV], f1hi[NV], f2lo[NV], f2hi[NV], f3lo[NV], f3hi[NV];
#pragma unroll
    for (int v = 0; v < B1; ++v) {
        f1lo[v] = (double)F1[v * nc + c];
        f1hi[v] = (double)F1[v * nc + c + 1];
        f2lo[v] = (double)F2[v * nc + c];
        f2hi[v] = (double)F2[v * nc + c + s2];
        if (nd == 3) { f3lo[v] = (double)F3[v * nc + c]; f3hi[v] = (double)F3[v * nc + c + s3]; }
        else { f3lo[v] = 0.; f3hi[v] = 0.; }
    }
    const R* F1B2 = F1 + B2 * nc;
    const R* F2B1 = F2 + B1 * nc;
    const R e3_00 = emf3_at(F1B2, F2B1, c, s2), e3_10 = emf3_at(F1B2, F2B1, c + 1, s2);
    const R e3_01 = emf3_at(F1B2, F2B1, c + s2, s2), e3_11 = emf3_at(F1B2, F2B1, c + s2 + 1, s2);
    f1lo[B1] = 0.; f1hi[B1] = 0.;
    f1lo[B2] = (double)(R(0.5) * (e3_00 + e3_01));
    f1hi[B2] = (double)(R(0.5) * (e3_10 + e3_11));
    f2lo[B1] = (double)(R(-0.5) * (e3_00 + e3_10));
    f2hi[B1] = (double)(R(-0.5) * (e3_01 + e3_11));
    f2lo[B2] = 0.; f2hi[B2] = 0.;
    f3lo[B1] = f3hi[B1] = f3lo[B2] = f3hi[B2] = f3lo[B3] = f3hi[B3] = 0.;
    if (nd == 3) {
        const R* F2B3 = F2 + B3 * nc;
        const R* F3B2 = F3 + B2 * nc;
        const R* F3B1 = F3 + B1 * nc;
        const R* F1B3 = F1 + B3 * nc;
        const R e1_000 = emf1_at(F2B3, F3B2, c, s2, s3), e1_010 = emf1_at(F2B3, F3B2, c + s2, s2, s3);
        const R e1_001 = emf1_at(F2B3, F3B2, c + s3, s2, s3), e1_011 = emf1_at(F2B3, F3B2, c + s2 + s3, s2, s3);
        const R e2_000 = emf2_at(F3B1, F1B3, c, s3), e2_100 = emf2_at(F3B1, F1B3, c + 1, s3);
        const R e2_001 = emf2_at(F3B1, F1B3, c + s3, s3), e2_101 = emf2_at(F3B1, F1B3, c + s3 + 1, s3);
        f1lo[B3] = (double)(R(-0.5) * (e2_000 + e2_001));
        f1hi[B3] = (double)(R(-0.5) * (e2_100 + e2_101));
        f2lo[B3] = (double)(R(0.5) * (e1_000 + e1_001));
        f2hi[B3] = (double)(R(0.5) * (e1_010 + e1_011));
        f3lo[B1] = (double)(R(0.5) * (e2_000 + e2_100));
        f3hi[B1] = (double)(R(0.5) * (e2_001 + e2_101));
        f3lo[B2] = (double)(R(-0.5) * (e1_000 + e1_010));
        f3hi[B2] = (double)(R(-0.5) * (e1_001 + e1_011));
    } else {
        // 2D: B3 keeps its Riemann fluxes
        f1lo[B3] = (double)F1[B3 * nc + c];
        f1hi[B3] = (double)F1[B3 * nc + c + 1];
        f2lo[B3] = (double)F2[B3 * nc + c];
        f2hi[B3] = (double)F2[B3 * nc + c + s2];
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        double du = (A1 * f1hi[v] - A1 * f1lo[v]);
        du += (A2 * f2hi[v] - A2 * f2lo[v]);
        if (nd == 3) du += (A3 * f3hi[v] - A3 * f3lo[v]);
        dudt[v] = -du * iV;
    }
}

// The U->P solver of inverter/type (inverter.cpp:53-70): INV 0 onedw, 1 Kastaun.
template <int INV, class G>
__device__ __forceinline__ int invert_zone(const G& g, const double U[NV], double P[NV], const StepConsts& cst) {
    if constexpr (INV == 1) return u_to_p_kastaun(g, U, P, cst.gam, cst.floors, cst.iter_max, cst.err_tol);
    else return u_to_p_onedw(g, U, P, cst.gam, cst.iter_max, cst.err_tol);
}

// The curved-space kernels walk the interior in (j, k, i) order, i fastest, with
// the workgroups renumbered so each XCD (workgroup w runs on XCD w % 8) owns one
// contiguous range of j: the axisymmetric geometry tables ([comp][j][i]) a
// workgroup reads then stay within one eighth of the table per XCD L2.
constexpr unsigned N_XCD = 8;
__device__ __forceinline__ unsigned xcd_logical_block(unsigned b, unsigned nb) {
    const unsigned x = b % N_XCD, r = b / N_XCD, q = nb / N_XCD, m = nb % N_XCD;
    return x * q + (x < m ? x : m) + r;
}
__device__ __forceinline__ void interior_index_jki(const BlockDims& b, unsigned t, int& k, int& j, int& i) {
    const unsigned n3 = (unsigned)(b.ndim > 2 ? b.nx3 : 1);
    const unsigned row = t / (unsigned)b.nx1;
    const unsigned jj = row / n3;
    i = b.is + (int)(t - row * (unsigned)b.nx1);
    k = b.ks + (int)(row - jj * n3);
    j = b.js + (int)jj;
}

// In 3-D they run on tiles of TI = 64 x1 cells by 4 x3 rows at one x2 row, one x3
// row per wavefront: the four wavefronts of a work-group share the geometry of
// their 64 (j, i) columns (the 22 metric components and the 2 geometric floors),
// which the work-group stages once in LDS as [component][64] instead of each zone
// loading its own.  A block whose x1 width is an odd multiple of 32 (the 96-wide
// blocks of a 2x2x4 mesh of the 192x128x128 torus) runs TI = 32 by 8 rows instead,
// two rows per wavefront, so that no tile is half empty.  Tiles are numbered i
// fastest, then k, then j, and renumbered per XCD as above.
constexpr int STG_GEOM = GEO_NCOMP + 2;
template <int TI> __host__ __device__ __forceinline__ int tiles_i(const BlockDims& b) { return (b.nx1 + TI - 1) / TI; }
template <int TI> __host__ __device__ __forceinline__ int tiles_k(const BlockDims& b) {
    return (b.nx3 + BS / TI - 1) / (BS / TI);
}
// The tile width for block b: 32 where it leaves fewer idle lanes.
static inline int tile_width(const BlockDims& b) {
    return (tiles_i<32>(b) * 32 - b.nx1 < tiles_i<64>(b) * 64 - b.nx1) ? 32 : 64;
}
static inline long update_tiles_host(const BlockDims& b) {
    return tile_width(b) == 32 ? (long)tiles_i<32>(b) * tiles_k<32>(b) * b.nx2
                                   : (long)tiles_i<64>(b) * tiles_k<64>(b) * b.nx2;
}
// Zone (k, j, i) of this thread; i0 is the tile's first x1 cell.
template <int TI>
__device__ __forceinline__ bool tile_zone(const BlockDims& b, int& k, int& j, int& i, int& i0) {
    const unsigned lb = xcd_logical_block(blockIdx.x, gridDim.x);
    const unsigned nti = (unsigned)tiles_i<TI>(b), ntk = (unsigned)tiles_k<TI>(b);
    const unsigned ti = lb % nti, rest = lb / nti;
    const unsigned tk = rest % ntk, jj = rest / ntk;
    const int row = (TI == 64) ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x / TI)) : (int)(threadIdx.x / TI);
    i0 = b.is + (int)ti * TI;
    i = i0 + (int)(threadIdx.x % TI);
    k = b.ks + (int)tk * (BS / TI) + row;
    j = b.js + (int)jj;
    return i <= b.ie && k <= b.ke;
}
// Stage the tile's metric and floors (x1 clamped to the table for a ragged
// last tile) into sg; every thread of the work-group calls it.
template <int TI>
__device__ __forceinline__ void stage_tile_geometry(const GeomDev& gd, int j, int i0, double* sg) {
    const int lane = (int)(threadIdx.x % TI);
    const int w = (TI == 64) ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x / TI)) : (int)(threadIdx.x / TI);
    const long q = (long)j * gd.gn1 + min(i0 + lane, gd.gn1 - 1);
#pragma unroll
    for (int c0 = 0; c0 < STG_GEOM; c0 += BS / TI) {
        const int comp = c0 + w;
        if (comp < STG_GEOM)
            sg[comp * TI + lane] = comp < GEO_NCOMP ? gd.g[GLOC_CENTER][(long)comp * gd.np + q]
                                                    : gd.flr[(long)(comp - GEO_NCOMP) * gd.np + q];
    }
    __syncthreads();
}

}  // namespace kh
