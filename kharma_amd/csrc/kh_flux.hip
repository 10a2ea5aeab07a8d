// kh_flux.hip -- fused face-flux kernels: reconstruction + reconstruction floors
// + prim_to_flux + signal speeds + LLF/HLLE in one pass per direction.
//
// Replaces the four kernels of Flux::GetFlux<Recon,dir> (flux/get_flux.hpp:60-373:
// calc_flux_recon, calc_flux_left, calc_flux_right, flux_llf), which stage
// Pl/Pr/Ul/Ur/Fl/Fr through HBM scratch.  Here each work-item reconstructs ONE
// cell (both of its face values, sharing the smoothness indicators), publishes
// the right-face value through LDS, and then computes the flux through its
// cell's left face from its own left-face value and its neighbour's right-face
// value.  Only the 8 fluxes and 2 signal speeds per face reach HBM.
//
// X1: 256-thread blocks walk the cells of consecutive x1 rows (flattened,
// consecutive blocks overlap by one cell); loads and stores are contiguous.
// X2/X3: 64 x TY blocks; x is a flattened transverse index with x1 fastest (so
// a wavefront reads 64 consecutive values), y walks TY cells along the face
// normal, consecutive tiles overlapping by one cell.
// Small blocks run the tiles of all directions in one launch (flux_all_kernel);
// FP64 fluxes of large 3-D meshes are taken by lanes that walk along the normal
// (flux_march_kernel, flux_x1_march_kernel).
#include "kh_internal.hpp"
#include "kh_lane_geom.hpp"

namespace kh {

// The FP32 kernels, which are VALU-bound, address their arrays through 32-bit
// offsets (at32: 5-6 % fewer VALU instructions, 6-7 % faster X2/X3); the FP64
// tile kernels keep 64-bit indices, which measured faster for them (X1 8 %).
template <typename R> struct A32Of { static constexpr bool value = sizeof(R) == 4; };
template <bool A32, class T> __device__ __forceinline__ T& at_idx(T* p, long e) {
    if constexpr (A32) return at32(p, (unsigned)e);
    else return p[e];
}

template <int RECON, typename R>
__device__ __forceinline__ void cell_states(R x1, R x2, R x3, R x4, R x5, R& lout, R& rout) {
    if constexpr (RECON == RECON_WENO5) {
        weno5_cell(x1, x2, x3, x4, x5, lout, rout);
    } else if constexpr (RECON == RECON_LINEAR_MC) {
        const R dq = mc_lim(x3 - x2, x4 - x3) * (x4 - x3);
        rout = x3 + R(0.5) * dq;
        lout = x3 - R(0.5) * dq;
    } else if constexpr (RECON == RECON_PPM) {
        ppm(x1, x2, x3, x4, x5, lout, rout);
    } else {
        lout = x3;
        rout = x3;
    }
}

// Flux through one face from its two states (get_flux.hpp:237-367).
// SPEEDS: SPEEDS_BOTH writes cmax and cmin (Flux.cmax/cmin), SPEEDS_CTOP writes
// max(cmax, cmin) (all the timestep uses) into cmax_out, SPEEDS_NONE writes none.
template <int DIR, int SPEEDS, typename R, class G>
__device__ __forceinline__ void face_flux_g(const StepConsts& c, const BlockDims& b, const G& g, R rflr, R uflr,
                                            R Pl[NV], R Pr[NV], long ci,
                                            const Vars<R>& F, R* __restrict__ cmax_out, R* __restrict__ cmin_out) {
    constexpr bool A32 = A32Of<R>::value;
    const R gam = R(c.gam);
    // get_flux.hpp:170-182: geometric floors of the face's cell centre on both states
    if (c.recon_floors) {
        apply_geo_floors<R>(Pl, rflr, uflr);
        apply_geo_floors<R>(Pr, rflr, uflr);
    }
    R Ul[NV], Fl[NV], Ur[NV], Fr[NV];
    R cmaxL, cminL, cmaxR, cminR;
    {
        FourVec<R> D;
        calc_4vecs<R>(g, Pl, D);
        prim_to_u_and_flux<R, G, DIR>(g, Pl, D, gam, Ul, Fl);
        vchar<R, G, DIR>(g, Pl, D, gam, cmaxL, cminL);
    }
    {
        FourVec<R> D;
        calc_4vecs<R>(g, Pr, D);
        prim_to_u_and_flux<R, G, DIR>(g, Pr, D, gam, Ur, Fr);
        vchar<R, G, DIR>(g, Pr, D, gam, cmaxR, cminR);
    }
    // get_flux.hpp:275-276 and 331-332: cmin is stored as a positive speed
    const R cmx = smax(smax(R(0), cmaxL), cmaxR);
    const R cmn = -smin(smin(R(0), cminL), cminR);
    if constexpr (SPEEDS == SPEEDS_BOTH) {
        at_idx<A32>(cmax_out, ci) = cmx;
        at_idx<A32>(cmin_out, ci) = cmn;
    } else if constexpr (SPEEDS == SPEEDS_CTOP) {
        at_idx<A32>(cmax_out, ci) = smax(cmx, cmn);
    }
    if (c.use_hlle) {
        const R inv = rcp(cmx + cmn);
#pragma unroll
        for (int v = 0; v < NV; ++v)
            at_idx<A32>(F[v], ci) = (cmx * Fl[v] + cmn * Fr[v] - cmx * cmn * (Ur[v] - Ul[v])) * inv;
    } else {
        const R ctop = smax(cmx, cmn);
#pragma unroll
        for (int v = 0; v < NV; ++v)
            at_idx<A32>(F[v], ci) = R(0.5) * (Fl[v] + Fr[v] - ctop * (Ur[v] - Ul[v]));
    }
}

template <typename R> __device__ __forceinline__ const R* geo_table(const GeomDev& gd, int loc);
template <> __device__ __forceinline__ const double* geo_table<double>(const GeomDev& gd, int loc) { return gd.g[loc]; }
template <> __device__ __forceinline__ const float* geo_table<float>(const GeomDev& gd, int loc) { return gd.g32[loc]; }
template <typename R> __device__ __forceinline__ R geo_floor(const GeomDev& gd, int which, long q);
template <> __device__ __forceinline__ double geo_floor<double>(const GeomDev& gd, int which, long q) { return gd.flr[which * gd.np + q]; }
template <> __device__ __forceinline__ float geo_floor<float>(const GeomDev& gd, int which, long q) { return gd.flr32[which * gd.np + q]; }

// Face at entire-block indices (j, i): flat metric (GEO == 0) or the cached
// metric of the face locus (X1 face, X2 face, or the centre for X3 faces of the
// axisymmetric metric) with the floors of cell (j, i).
template <int DIR, int SPEEDS, typename R, int GEO>
__device__ __forceinline__ void face_flux(const StepConsts& c, const BlockDims& b, const GeomDev& gd, int j, int i,
                                          R Pl[NV], R Pr[NV], long ci,
                                          const Vars<R>& F, R* __restrict__ cmax_out, R* __restrict__ cmin_out) {
    if constexpr (GEO) {
        const long q = (long)j * gd.gn1 + i;
        const int loc = (DIR == 1) ? GLOC_FACE1 : (DIR == 2) ? GLOC_FACE2 : GLOC_CENTER;
        CachedGeom<R, A32Of<R>::value> g(geo_table<R>(gd, loc), gd.np, q);
        face_flux_g<DIR, SPEEDS, R>(c, b, g, geo_floor<R>(gd, 0, q), geo_floor<R>(gd, 1, q), Pl, Pr, ci, F, cmax_out, cmin_out);
    } else {
        MinkowskiGeom<R> g;
        face_flux_g<DIR, SPEEDS, R>(c, b, g, R(c.floors.rho_min_const), R(c.floors.u_min_const), Pl, Pr, ci, F, cmax_out, cmin_out);
    }
}

// X1 faces i in [is, ie+1] of rows j in [j0, j0+nj), k in [k0, k0+nk).
// Cells i in [is-1, ie+1] (L per row); block b handles flattened cells
// [255 b, 255 b + 256) and emits the faces of all but its first cell.
// Waves per SIMD the FP32 flux kernels are built for (the second launch bound): 6,
// which holds them to 48-69 VGPRs (7-8 waves fit); unbounded they took 90-115 and X2/X3
// were 11-14 % slower on the 192x128x128 torus.  The FP64 tiles are not bounded: 101-126
// VGPRs, four waves.
template <typename R> struct FluxOcc { static constexpr int w = sizeof(R) == 4 ? 6 : 1; };
template <int RECON, int SPEEDS, typename R, typename PT, int GEO>
__device__ __forceinline__ void x1_tile(const BlockDims& b, const StepConsts& c, const GeomDev& gd, const Vars<const PT>& P,
                                        const Vars<R>& F, R* __restrict__ cmax_out, R* __restrict__ cmin_out, int j0,
                                        int nj, int k0, int nk, unsigned bx, int tid, R (*sr)[256]) {
    const int L = b.nx1 + 2;
    // cell counts stay below 2^31 (the C ABI bounds a block's size), so the
    // flattened index is divided in 32 bits
    const unsigned g = bx * 255u + (unsigned)tid;
    const bool valid = g < (unsigned)L * (unsigned)nj * (unsigned)nk;
    int ii = 0, jf = 0;
    long ci = 0;
    R lo[NV];
    if (valid) {
        const int row = (int)(g / (unsigned)L);
        ii = (int)(g - (unsigned)row * (unsigned)L);
        const int jj = (int)((unsigned)row % (unsigned)nj), kk = (int)((unsigned)row / (unsigned)nj);
        jf = j0 + jj;
        ci = (long)(k0 + kk) * b.s3 + (long)(j0 + jj) * b.s2 + (b.is - 1 + ii);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            R ro;
            if constexpr (A32Of<R>::value) {
                const PT* __restrict__ q = P[v];
                const unsigned cu = (unsigned)ci;
                cell_states<RECON, R>(R(at32(q, cu - 2)), R(at32(q, cu - 1)), R(at32(q, cu)), R(at32(q, cu + 1)),
                                      R(at32(q, cu + 2)), lo[v], ro);
            } else {
                const PT* __restrict__ q = P[v] + ci;
                cell_states<RECON, R>(R(q[-2]), R(q[-1]), R(q[0]), R(q[1]), R(q[2]), lo[v], ro);
            }
            sr[v][tid] = ro;
        }
    }
    __syncthreads();
    if (!valid || tid == 0 || ii == 0) return;
    R Pl[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) Pl[v] = sr[v][tid - 1];
    face_flux<1, SPEEDS, R, GEO>(c, b, gd, jf, b.is - 1 + ii, Pl, lo, ci, F, cmax_out, cmin_out);
}
template <int RECON, int SPEEDS, typename R, typename PT, int GEO, bool PK>
__global__ void __launch_bounds__(256, FluxOcc<R>::w)
flux_x1_kernel(BlockDims b, StepConsts c, GeomDev gd, Vars<const PT> P, Vars<R> F,
               R* __restrict__ cmax_out, R* __restrict__ cmin_out, int j0, int nj, int k0, int nk,
               const BlockEntry* __restrict__ pk) {
    __shared__ R sr[NV][256];
    if constexpr (PK) {
        const long blk = pack_select(pk, b, gd);
        P = pack_at(P, blk * NV * b.nc);
        F = pack_at(F, blk * 3 * NV * b.nc);
        cmax_out = pack_at(cmax_out, blk * 3 * b.nc);
        cmin_out = pack_at(cmin_out, blk * 3 * b.nc);
    }
    x1_tile<RECON, SPEEDS, R, PT, GEO>(b, c, gd, P, F, cmax_out, cmin_out, j0, nj, k0, nk, blockIdx.x, threadIdx.x, sr);
}

// X2 / X3 faces.  Transverse columns: flattened (outer, i) with i in [is-1, ie+1]
// fastest; outer = k (X2) or j (X3) from o0.  Along the normal: faces s in
// [s0, s1]; tile y covers cells s0-1+(TY-1)y .. s0-2+TY+(TY-1)y.  64 x 8 blocks, two
// per CU in FP64 (101-118 VGPRs), three or four in FP32 (48-67): 64 x 10 and 64 x 16
// FP32 blocks measured 24 % and 2 % slower, 64 x 4, 64 x 12 and 64 x 16 FP64 blocks 5, 3
// and 4 % (192x128x128 torus).
constexpr int XT_TY = 8;
template <int DIR, int RECON, int SPEEDS, typename R, typename PT, int GEO, int TY>
__device__ __forceinline__ void xt_tile(const BlockDims& b, const StepConsts& c, const GeomDev& gd, const Vars<const PT>& P,
                                        const Vars<R>& F, R* __restrict__ cmax_out, R* __restrict__ cmin_out, int o0,
                                        int no, int s0, int s1, int bx, int by, int tx, int ty, R (*sr)[TY][64]) {
    const int ni = b.nx1 + 2;
    const int col = bx * 64 + tx;
    const int s = s0 - 1 + by * (TY - 1) + ty;
    const bool valid = col < ni * no && s <= s1;
    const long st = (DIR == 2) ? b.s2 : b.s3;
    long ci = 0;
    int jf = 0, if_ = 0;
    R lo[NV];
    if (valid) {
        const int outer = o0 + col / ni;
        const int i = b.is - 1 + col % ni;
        const int j = (DIR == 2) ? s : outer;
        const int k = (DIR == 2) ? outer : s;
        jf = j; if_ = i;
        ci = (long)k * b.s3 + (long)j * b.s2 + i;
        constexpr bool A = A32Of<R>::value;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            R ro;
            if constexpr (A) {
                const PT* __restrict__ q = P[v];
                cell_states<RECON, R>(R(at32(q, unsigned(ci - 2 * st))), R(at32(q, unsigned(ci - st))),
                                      R(at32(q, unsigned(ci))), R(at32(q, unsigned(ci + st))),
                                      R(at32(q, unsigned(ci + 2 * st))), lo[v], ro);
            } else {
                const PT* __restrict__ q = P[v] + ci;
                cell_states<RECON, R>(R(q[-2 * st]), R(q[-st]), R(q[0]), R(q[st]), R(q[2 * st]), lo[v], ro);
            }
            sr[v][ty][tx] = ro;
        }
    }
    __syncthreads();
    if (!valid || ty == 0) return;
    R Pl[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) Pl[v] = sr[v][ty - 1][tx];
    face_flux<DIR, SPEEDS, R, GEO>(c, b, gd, jf, if_, Pl, lo, ci, F, cmax_out, cmin_out);
}
template <int DIR, int RECON, int SPEEDS, typename R, typename PT, int GEO, bool PK>
__global__ void __launch_bounds__(64 * XT_TY, FluxOcc<R>::w)
flux_xt_kernel(BlockDims b, StepConsts c, GeomDev gd, Vars<const PT> P, Vars<R> F,
               R* __restrict__ cmax_out, R* __restrict__ cmin_out, int o0, int no, int s0, int s1,
               const BlockEntry* __restrict__ pk) {
    __shared__ R sr[NV][XT_TY][64];
    if constexpr (PK) {
        const long blk = pack_select(pk, b, gd);
        P = pack_at(P, blk * NV * b.nc);
        F = pack_at(F, blk * 3 * NV * b.nc);
        cmax_out = pack_at(cmax_out, blk * 3 * b.nc);
        cmin_out = pack_at(cmin_out, blk * 3 * b.nc);
    }
    xt_tile<DIR, RECON, SPEEDS, R, PT, GEO, XT_TY>(b, c, gd, P, F, cmax_out, cmin_out, o0, no, s0, s1, (int)blockIdx.x,
                                                   (int)blockIdx.y, (int)threadIdx.x, (int)threadIdx.y, sr);
}

// The faces of all directions in one launch, the X1 tiles first, then X2 and X3
// tiles of 64 x 4.  A direction's launch of a small block fills a fraction of the
// chip (64^2: 17 and 20 work-groups on 256 CUs) and ends in a tail that nothing
// follows; in one launch the directions fill each other's tails, and the smaller
// X2 / X3 tiles shorten the longest chain.  FP64 64^2: 18.9 + 6.3 -> 11.2 us, 256^2 8.9 +
// 9 -> 13.5 us, 256x128 torus 10 + 8.1 -> 11.6 us; FP32 128^2 6.8 + 6.1 -> 7.5 us.
constexpr int ALL_TY = 4;
// One direction's tiles: its first tile, tiles along the columns, and the face ranges.
struct FluxTiles { int first, nx, o0, no, s0, s1; };
template <int RECON, int SPEEDS, typename R, typename PT, int GEO>
__global__ void __launch_bounds__(256, FluxOcc<R>::w)
flux_all_kernel(BlockDims b, StepConsts c, GeomDev gd, Vars<const PT> P, Vars<R> F, R* __restrict__ ctop, FluxTiles x1,
                  FluxTiles x2, FluxTiles x3) {
    __shared__ R sr[NV][256];
    R (*st)[ALL_TY][64] = reinterpret_cast<R (*)[ALL_TY][64]>(sr);
    const int t = (int)blockIdx.x, tx = (int)threadIdx.x % 64, ty = (int)threadIdx.x / 64;
    if (t >= x3.first) {
        const int q = t - x3.first;
        xt_tile<3, RECON, SPEEDS, R, PT, GEO, ALL_TY>(b, c, gd, P, pack_at(F, 2 * NV * b.nc), pack_at(ctop, 2 * b.nc), nullptr,
                                                     x3.o0, x3.no, x3.s0, x3.s1, q % x3.nx, q / x3.nx, tx, ty, st);
    } else if (t >= x2.first) {
        const int q = t - x2.first;
        xt_tile<2, RECON, SPEEDS, R, PT, GEO, ALL_TY>(b, c, gd, P, pack_at(F, NV * b.nc), pack_at(ctop, b.nc), nullptr,
                                                     x2.o0, x2.no, x2.s0, x2.s1, q % x2.nx, q / x2.nx, tx, ty, st);
    } else {
        x1_tile<RECON, SPEEDS, R, PT, GEO>(b, c, gd, P, F, ctop, nullptr, x1.o0, x1.no, x1.s0, x1.s1 - x1.s0 + 1, (unsigned)t,
                                           (int)threadIdx.x, sr);
    }
}

// ---------------------------------------------------- FP64, large 3-D meshes
// The FP64 tiles wait for half of a wavefront's life (four per SIMD): 40 stencil
// loads, a barrier, the metric's loads, all in one short pass per face.  The
// marching kernels walk instead.
//
// X2 / X3 faces.  Each lane walks its own column of cells
// along the face normal, over a chunk of faces, with the five cells of the stencil
// in registers, so a row costs 8 loads of P instead of 40 and each cell is
// reconstructed once.
//
// Nothing in a row waits for memory: the cell that enters the next row's stencil
// and (X2) the next row's metric are requested at the row's start and used a row
// later, and no other load follows them (loads complete in order, so any later one
// would wait for both).  The metric of the row sits in the lane's own LDS slots,
// as do the two face states, which frees the registers the window needs (172-240
// VGPRs on the torus, two waves per SIMD).  Lanes share nothing: there is no barrier.
//
// Bound by FP64 issue and its dependent chains at two wavefronts: VALU issue 0.56-0.63
// of the chip's capacity on the 192x128x128 torus, waiting 0.31-0.37 of a wavefront's
// life.  Against the tiles there X2 234 -> 157-163 us, X3 226 -> 139 us.  Asking for the next
// row before the metric (249 us X2: the metric's waits included the prefetch) and the
// metric straight from memory behind it (250 us X2, 182 us X3) were slower.
//
// The marching kernels' reconstruction: WENO5 in its lean form (X2 172 -> 165 us, X3 154 ->
// 144, X1 171 -> 160 on the 192x128x128 torus), which rounds differently from the tiles'.
template <int RECON>
__device__ __forceinline__ void march_states(double x1, double x2, double x3, double x4, double x5, double& lout, double& rout) {
    if constexpr (RECON == RECON_WENO5) weno5_cell_lean(x1, x2, x3, x4, x5, lout, rout);
    else cell_states<RECON, double>(x1, x2, x3, x4, x5, lout, rout);
}
template <int DIR, int RECON, int SPEEDS, int GEO, bool PK>
__global__ void __launch_bounds__(256, 2)
flux_march_kernel(BlockDims b, StepConsts c, GeomDev gd, Vars<const double> P, Vars<double> F,
                  double* __restrict__ cmax_out, double* __restrict__ cmin_out, int o0, int no, int s0, int s1, int chunk,
                  const BlockEntry* __restrict__ pk) {
    if constexpr (PK) {
        const long blk = pack_select(pk, b, gd);
        P = pack_at(P, blk * NV * b.nc);
        F = pack_at(F, blk * 3 * NV * b.nc);
        cmax_out = pack_at(cmax_out, blk * 3 * b.nc);
        cmin_out = pack_at(cmin_out, blk * 3 * b.nc);
    }
    __shared__ double sl[NV][256], sr[NV][256], sm[GEO ? MG_N : 1][256];
    const int tid = threadIdx.x;
    const int ni = b.nx1 + 2;
    const unsigned col = blockIdx.x * 256u + threadIdx.x;
    if (col >= (unsigned)ni * (unsigned)no) return;
    const int outer = o0 + (int)(col / (unsigned)ni);
    const int i = b.is - 1 + (int)(col % (unsigned)ni);
    const int first = s0 + (int)blockIdx.y * chunk;
    const int last = min(first + chunk - 1, s1);
    const unsigned st = (unsigned)((DIR == 2) ? b.s2 : b.s3);
    unsigned ci = (unsigned)((DIR == 2) ? outer * b.s3 : outer * b.s2) + (unsigned)i + (unsigned)(first - 1) * st;
    // the metric of the row's faces: X2 rows have their own, X3 rows share one
    unsigned q = (unsigned)((DIR == 2) ? first : outer) * (unsigned)gd.gn1 + (unsigned)i;
    constexpr int loc = (DIR == 2) ? GLOC_FACE2 : GLOC_CENTER;
    double mg[GEO ? MG_N : 1];
    auto load_metric = [&](unsigned at) {
        if constexpr (GEO) {
#pragma unroll
            for (int m = 0; m < MG_RF; ++m) mg[m] = at32(gd.g[loc] + (long)LaneGeom<DIR>::src(m) * gd.np, at);
            mg[MG_RF] = at32(gd.flr, at);
            mg[MG_UF] = at32(gd.flr + gd.np, at);
        }
    };
    auto store_metric = [&]() {
        if constexpr (GEO) {
#pragma unroll
            for (int m = 0; m < MG_N; ++m) sm[m][tid] = mg[m];
        }
    };
    double w[NV][5];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
#pragma unroll
        for (int m = 0; m < 5; ++m) w[v][m] = at32(P[v], ci + (unsigned)(m - 2) * st);
    }
    unsigned ahead = ci + 3 * st;
    double pre[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) pre[v] = at32(P[v], ahead);
    load_metric(q);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        double lo, hi;
        march_states<RECON>(w[v][0], w[v][1], w[v][2], w[v][3], w[v][4], lo, hi);
        sl[v][tid] = hi;
    }
    store_metric();
    for (int s = first; s <= last; ++s) {
        ci += st;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            w[v][0] = w[v][1]; w[v][1] = w[v][2]; w[v][2] = w[v][3]; w[v][3] = w[v][4];
            w[v][4] = pre[v];
        }
        // (the last row requests its own again rather than past the stencil)
        if (s < last) {
            ahead += st;
            if (DIR == 2) q += (unsigned)gd.gn1;
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) pre[v] = at32(P[v], ahead);
        if constexpr (DIR == 2) load_metric(q);
        __builtin_amdgcn_sched_barrier(0);
        double Pl[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            double lo, hi;
            march_states<RECON>(w[v][0], w[v][1], w[v][2], w[v][3], w[v][4], lo, hi);
            sr[v][tid] = lo;
            Pl[v] = sl[v][tid];
            sl[v][tid] = hi;
        }
        double Pr[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) Pr[v] = sr[v][tid];
        if constexpr (GEO) {
            LaneGeom<DIR> g{sm, tid};
            face_flux_g<DIR, SPEEDS, double>(c, b, g, sm[MG_RF][tid], sm[MG_UF][tid], Pl, Pr, (long)ci, F, cmax_out, cmin_out);
        } else {
            MinkowskiGeom<double> g;
            face_flux_g<DIR, SPEEDS, double>(c, b, g, c.floors.rho_min_const, c.floors.u_min_const, Pl, Pr, (long)ci, F,
                                             cmax_out, cmin_out);
        }
        if constexpr (DIR == 2) store_metric();
    }
}

// X1 faces of large 3-D blocks in FP64: each lane walks along x3 with one cell of
// a row, the rows flattened over (x2, x1) with three cells beyond either end, so
// a wavefront's 64 cells and two more on each side hold every stencil.  A row's 68
// cells pass through LDS (one load a cell instead of five, requested a row ahead);
// the metric, which x3 does not change, is read once.  A wavefront takes 63 faces
// and shares nothing with the others: the LDS exchange needs no barrier, only that
// its accesses stay in order.  192x128x128 torus 192 -> 150 us (VALU issue 0.59).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <int RECON, int SPEEDS, bool PK>
__global__ void __launch_bounds__(256, 2)
flux_x1_march_kernel(BlockDims b, StepConsts c, GeomDev gd, Vars<const double> P, Vars<double> F,
                     double* __restrict__ cmax_out, double* __restrict__ cmin_out, int j0, int nj, int k0, int k1, int chunk,
                     const BlockEntry* __restrict__ pk) {
    if constexpr (PK) {
        const long blk = pack_select(pk, b, gd);
        P = pack_at(P, blk * NV * b.nc);
        F = pack_at(F, blk * 3 * NV * b.nc);
        cmax_out = pack_at(cmax_out, blk * 3 * b.nc);
        cmin_out = pack_at(cmin_out, blk * 3 * b.nc);
    }
    __shared__ double row[NV][4][68], sh[NV][256], sm[MG_N][256];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int L = b.nx1 + 6, total = L * nj;
    const int g0 = ((int)blockIdx.x * 4 + wv) * 63;   // the wavefront's first cell
    if (g0 >= total) return;                           // (whole wavefronts)
    auto offset = [&](int g) {                         // of flattened cell g, clamped into the rows
        g = min(max(g, 0), total - 1);
        const int jj = (int)((unsigned)g / (unsigned)L);
        return (unsigned)((j0 + jj) * b.s2) + (unsigned)(b.is - 3 + (g - jj * L));
    };
    const int g = g0 + lane;
    const int jj = (int)((unsigned)min(g, total - 1) / (unsigned)L), ii = g - jj * L;
    const bool face = lane > 0 && g < total && ii >= 3 && ii <= b.nx1 + 3;
    const int first = k0 + (int)blockIdx.y * chunk;
    const int last = min(first + chunk - 1, k1);
    const unsigned s3 = (unsigned)b.s3;
    unsigned ci = offset(g) + (unsigned)first * s3;
    // lanes 0-3 also fetch the two cells before and after the wavefront's
    const int hm = lane < 2 ? lane : 64 + lane;
    const bool halo = lane < 4;
    unsigned hi_ci = offset(g0 - 2 + hm) + (unsigned)first * s3;
    {
        const unsigned q = (unsigned)(j0 + jj) * (unsigned)gd.gn1 + (unsigned)(b.is - 3 + min(ii, L - 1));
#pragma unroll
        for (int m = 0; m < MG_RF; ++m) sm[m][tid] = at32(gd.g[GLOC_FACE1] + (long)LaneGeom<1>::src(m) * gd.np, q);
        sm[MG_RF][tid] = at32(gd.flr, q);
        sm[MG_UF][tid] = at32(gd.flr + gd.np, q);
    }
    double pre[NV], prh[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) pre[v] = at32(P[v], ci);
#pragma unroll
    for (int v = 0; v < NV; ++v) prh[v] = halo ? at32(P[v], hi_ci) : 0.;
    for (int k = first; k <= last; ++k) {
        double own[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            own[v] = pre[v];
            row[v][wv][lane + 2] = pre[v];
            if (halo) row[v][wv][hm] = prh[v];
        }
        wave_lds_fence();
        const unsigned at = ci;
        if (k < last) { ci += s3; hi_ci += s3; }   // (the last row requests its own again)
#pragma unroll
        for (int v = 0; v < NV; ++v) pre[v] = at32(P[v], ci);
#pragma unroll
        for (int v = 0; v < NV; ++v) prh[v] = halo ? at32(P[v], hi_ci) : 0.;
        __builtin_amdgcn_sched_barrier(0);
        double lo[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            double hi;
            const double* r = &row[v][wv][lane];
            march_states<RECON>(r[0], r[1], own[v], r[3], r[4], lo[v], hi);
            sh[v][tid] = hi;
        }
        wave_lds_fence();
        double Pl[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) Pl[v] = sh[v][lane > 0 ? tid - 1 : tid];
        wave_lds_fence();   // the next row overwrites row and sh
        if (face) {
            LaneGeom<1> gm{sm, tid};
            face_flux_g<1, SPEEDS, double>(c, b, gm, sm[MG_RF][tid], sm[MG_UF][tid], Pl, lo, (long)at, F, cmax_out, cmin_out);
        }
    }
}

// Zones per resident lane (two wavefronts per SIMD, 131072 lanes) from which the
// marching kernels are used.  A walk pays its start (five rows of loads, one extra
// reconstruction) once per chunk, and two wavefronts hide less latency than the
// tiles' four, so short walks lose.
//
// The zones counted are the whole mesh's, not the launch's: the two families round
// differently (see march_states), and one block, blocks in one launch and blocks
// launched one by one give the same bits only if they take the same one.
//
// FP64 steps, the tiles in one launch (flux_all_kernel) against marching, us: flat 80^3
// 322 / 350, 96^3 541 / 544, 112^3 835 / 797, 128^3 1259 / 1132 (7 zones a lane: 97^3);
// torus 84x72x60 313 / 345, 102x84x66 475 / 494, 126x90x61 537 / 547, 128x96x96 869 / 839,
// 160x112x96 1270 / 1171.  The task entry points, which launch a direction at a time, gain
// earlier (126x90x61, X2/X3 a face launch 57 / 51 us), so curved space starts at 5.  X1,
// curved space only: 126x90x61 49 / 52 us, 192x96x64 81 / 79, 150x110x100 111 / 105,
// 192x128x128 210 / 180; X1 flat 128^3 112 / 118 (four wavefronts of 103 registers: the
// tiles stay).  (2-D blocks have one row of each along x3 and too few faces: tiles.)
constexpr long MARCH_LANES = 2L * 4 * 256 * 64;
FluxRoute flux_route(const BlockDims& b, long mesh_zones, bool lane_form) {
    FluxRoute rt;
    rt.xt = b.ndim == 3 && (b.geo ? lane_form && mesh_zones >= 5 * MARCH_LANES : mesh_zones >= 7 * MARCH_LANES);
    rt.x1 = rt.xt && b.geo && mesh_zones >= 8 * MARCH_LANES;
    return rt;
}
// Faces per chunk: the fewest rounds of work for the busiest CU, a round being one
// block's chunk plus its start, 0.6 of a row's work (flat 160^3, X2: chunks of 1, 2, 4, 22
// faces 299, 233, 193, 171 us); a CU holds two blocks, and one alone on it takes 0.6 of
// the time of a pair (flat 64x64x32, X2: 198 blocks of 3 faces 15.1 us, 297 of 2 18.2, 585
// of 1 19.0).
static int march_chunk(long blocks_x, int nfaces) {
    int best = nfaces;
    double cost = 1e300;
    for (int ch = 1; ch <= nfaces; ++ch) {
        const long blocks = blocks_x * ((nfaces + ch - 1) / ch);
        const double per_cu = (double)((blocks + 255) / 256);
        const double t = (per_cu > 1.2 ? per_cu : 1.2) * (ch + 0.6);
        if (t < cost) { cost = t; best = ch; }
    }
    return best;
}

template <int RECON, int SPEEDS, typename R, typename PT, int GEO, bool PK>
static hipError_t launch_recon(const BlockDims& b, const StepConsts& c, const GeomDev& gd, FluxRoute rt, int dir, const Vars<const PT>& P, const Vars<R>& F,
                               R* cmax, R* cmin, hipStream_t s, const Pack* pk) {
    const BlockEntry* pd = pack_dev(pk);
    // Face ranges consumed by flux-CT and the divergence: the face-normal index
    // covers [start, end+1]; transverse indices extend one zone each side.
    const int jlo = (b.ndim > 1) ? b.js - 1 : b.js, jhi = (b.ndim > 1) ? b.je + 1 : b.je;
    const int klo = (b.ndim > 2) ? b.ks - 1 : b.ks, khi = (b.ndim > 2) ? b.ke + 1 : b.ke;
    const int nblk = pk ? pk->nblk : 1;
    if constexpr (sizeof(R) == 8) {
        if (dir == 1) {
            const int nj = jhi - jlo + 1, nk = khi - klo + 1;
            const long cells = (long)(b.nx1 + 6) * nj;
            if (rt.x1) {
                const unsigned bx = (unsigned)((cells + 4 * 63 - 1) / (4 * 63));
                const int chunk = march_chunk((long)bx * nblk, nk);
                const dim3 grid = pack_grid(dim3(bx, (unsigned)((nk + chunk - 1) / chunk)), pk);
                hipLaunchKernelGGL((flux_x1_march_kernel<RECON, SPEEDS, PK>), grid, dim3(256), 0, s, b, c, gd, P, F, cmax, cmin, jlo, nj, klo, khi, chunk, pd);
                return hipGetLastError();
            }
        } else {
            const int o0 = dir == 2 ? klo : jlo, no = dir == 2 ? khi - klo + 1 : jhi - jlo + 1;
            const int s0 = dir == 2 ? b.js : b.ks, s1 = dir == 2 ? b.je + 1 : b.ke + 1;
            const long cols = (long)(b.nx1 + 2) * no;
            const int nfaces = s1 - s0 + 1;
            if (rt.xt) {
                const unsigned bx = (unsigned)((cols + 255) / 256);
                const int chunk = march_chunk((long)bx * nblk, nfaces);
                const dim3 grid = pack_grid(dim3(bx, (unsigned)((nfaces + chunk - 1) / chunk)), pk);
                if (dir == 2)
                    hipLaunchKernelGGL((flux_march_kernel<2, RECON, SPEEDS, GEO, PK>), grid, dim3(256), 0, s, b, c, gd, P, F, cmax, cmin, o0, no, s0, s1, chunk, pd);
                else
                    hipLaunchKernelGGL((flux_march_kernel<3, RECON, SPEEDS, GEO, PK>), grid, dim3(256), 0, s, b, c, gd, P, F, cmax, cmin, o0, no, s0, s1, chunk, pd);
                return hipGetLastError();
            }
        }
    }
    if (dir == 1) {
        const int nj = jhi - jlo + 1, nk = khi - klo + 1;
        const long cells = (long)(b.nx1 + 2) * nj * nk;
        const dim3 grid = pack_grid(dim3((unsigned)((cells - 1 + 254) / 255)), pk);
        hipLaunchKernelGGL((flux_x1_kernel<RECON, SPEEDS, R, PT, GEO, PK>), grid, dim3(256), 0, s, b, c, gd, P, F, cmax, cmin, jlo, nj, klo, nk, pd);
    } else if (dir == 2) {
        const int no = khi - klo + 1;
        const int ncol = (b.nx1 + 2) * no;
        const int nfaces = b.nx2 + 1;
        constexpr int TY = XT_TY;
        const dim3 grid = pack_grid(dim3((unsigned)((ncol + 63) / 64), (unsigned)((nfaces + TY - 2) / (TY - 1))), pk);
        hipLaunchKernelGGL((flux_xt_kernel<2, RECON, SPEEDS, R, PT, GEO, PK>), grid, dim3(64, TY), 0, s, b, c, gd, P, F, cmax, cmin, klo, no, b.js, b.je + 1, pd);
    } else {
        const int no = jhi - jlo + 1;
        const int ncol = (b.nx1 + 2) * no;
        const int nfaces = b.nx3 + 1;
        constexpr int TY = XT_TY;
        const dim3 grid = pack_grid(dim3((unsigned)((ncol + 63) / 64), (unsigned)((nfaces + TY - 2) / (TY - 1))), pk);
        hipLaunchKernelGGL((flux_xt_kernel<3, RECON, SPEEDS, R, PT, GEO, PK>), grid, dim3(64, TY), 0, s, b, c, gd, P, F, cmax, cmin, jlo, no, b.ks, b.ke + 1, pd);
    }
    return hipGetLastError();
}

template <int SPEEDS, typename R, typename PT, int GEO, bool PK>
static hipError_t launch_speeds(const BlockDims& b, const StepConsts& c, const GeomDev& gd, FluxRoute rt, int dir, int recon, const Vars<const PT>& P, const Vars<R>& F,
                                R* cmax, R* cmin, hipStream_t s, const Pack* pk) {
    switch (recon) {
    case RECON_DONOR: return launch_recon<RECON_DONOR, SPEEDS, R, PT, GEO, PK>(b, c, gd, rt, dir, P, F, cmax, cmin, s, pk);
    case RECON_LINEAR_MC: return launch_recon<RECON_LINEAR_MC, SPEEDS, R, PT, GEO, PK>(b, c, gd, rt, dir, P, F, cmax, cmin, s, pk);
    case RECON_PPM: return launch_recon<RECON_PPM, SPEEDS, R, PT, GEO, PK>(b, c, gd, rt, dir, P, F, cmax, cmin, s, pk);
    default: return launch_recon<RECON_WENO5, SPEEDS, R, PT, GEO, PK>(b, c, gd, rt, dir, P, F, cmax, cmin, s, pk);
    }
}

template <typename R, typename PT, int GEO, bool PK>
static hipError_t launch_geo(const BlockDims& b, const StepConsts& c, const GeomDev& gd, FluxRoute rt, int dir, int recon, int speeds,
                             const Vars<const PT>& P, const Vars<R>& F, R* cmax, R* cmin, hipStream_t s, const Pack* pk) {
    if (speeds == SPEEDS_CTOP) return launch_speeds<SPEEDS_CTOP, R, PT, GEO, PK>(b, c, gd, rt, dir, recon, P, F, cmax, cmin, s, pk);
    if (speeds == SPEEDS_NONE) return launch_speeds<SPEEDS_NONE, R, PT, GEO, PK>(b, c, gd, rt, dir, recon, P, F, cmax, cmin, s, pk);
    if constexpr (!PK) return launch_speeds<SPEEDS_BOTH, R, PT, GEO, PK>(b, c, gd, rt, dir, recon, P, F, cmax, cmin, s, pk);
    return hipErrorInvalidValue;   // a pack launch is a stage's: no cmin array
}

template <typename R, typename PT, bool PK = false>
static hipError_t launch_prec(const BlockDims& b, const StepConsts& c, const GeomDev& gd, FluxRoute rt, int dir, int recon, int speeds,
                              const Vars<const PT>& P, const Vars<R>& F, R* cmax, R* cmin, hipStream_t s,
                              const Pack* pk = nullptr) {
    if (b.geo) return launch_geo<R, PT, 1, PK>(b, c, gd, rt, dir, recon, speeds, P, F, cmax, cmin, s, pk);
    return launch_geo<R, PT, 0, PK>(b, c, gd, rt, dir, recon, speeds, P, F, cmax, cmin, s, pk);
}

hipError_t launch_flux(const BlockDims& b, const StepConsts& c, const GeomDev& gd, FluxRoute rt, int dir, int recon, int prec,
                       const Vars<const double>& P, const Vars<void>& F, void* cmax, void* cmin, hipStream_t s) {
    if (dir == 2 && b.ndim < 2) return hipSuccess;
    if (dir == 3 && b.ndim < 3) return hipSuccess;
    if (prec == PREC_SPLIT)
        return launch_prec<float, double>(b, c, gd, rt, dir, recon, SPEEDS_BOTH, P, vars_cast<float>(F), (float*)cmax,
                                          (float*)cmin, s);
    return launch_prec<double, double>(b, c, gd, rt, dir, recon, SPEEDS_BOTH, P, vars_cast<double>(F), (double*)cmax,
                                       (double*)cmin, s);
}

hipError_t launch_flux_stage(const BlockDims& b, const StepConsts& c, const GeomDev& gd, FluxRoute rt, int dir, int recon, int prec,
                             int speeds, const double* P, const float* P32, void* F, void* ctop, hipStream_t s,
                             const Pack* pk) {
    if (dir == 2 && b.ndim < 2) return hipSuccess;
    if (dir == 3 && b.ndim < 3) return hipSuccess;
    if (pk) {
        if (prec == PREC_SPLIT)
            return launch_prec<float, float, true>(b, c, gd, rt, dir, recon, speeds, vars_of(P32, b.nc),
                                                   vars_of((float*)F, b.nc), (float*)ctop, nullptr, s, pk);
        return launch_prec<double, double, true>(b, c, gd, rt, dir, recon, speeds, vars_of(P, b.nc),
                                                 vars_of((double*)F, b.nc), (double*)ctop, nullptr, s, pk);
    }
    if (prec == PREC_SPLIT)
        return launch_prec<float, float>(b, c, gd, rt, dir, recon, speeds, vars_of(P32, b.nc), vars_of((float*)F, b.nc),
                                         (float*)ctop, nullptr, s);
    return launch_prec<double, double>(b, c, gd, rt, dir, recon, speeds, vars_of(P, b.nc), vars_of((double*)F, b.nc),
                                       (double*)ctop, nullptr, s);
}

// Tiles up to which the directions run in one launch.  Steps of a block, one launch a
// direction against one: FP64 64^2 82 / 53 us, 256^2 75 / 66, 512^2 135 / 128, 1024^2
// 433 / 431, 64^3 flat 212 / 195, 1024x512 torus 431 / 416; FP32 fluxes 64^3 flat 173 / 156,
// 128^3 (31500 tiles) 1004 / 992, 192x128x128 torus (46400 tiles) 1820 / 1837: there the
// 64 x 8 tiles' fewer overlapping cells win.  FP64 3-D blocks from the size of the
// marching kernels on take those.
constexpr long ALL_TILES = 32768;
// Tiles of the one-launch form, all directions; 0 where a direction is missing.
static int all_tiles(const BlockDims& b, FluxTiles (&x)[3]) {
    const int jlo = (b.ndim > 1) ? b.js - 1 : b.js, jhi = (b.ndim > 1) ? b.je + 1 : b.je;
    const int klo = (b.ndim > 2) ? b.ks - 1 : b.ks, khi = (b.ndim > 2) ? b.ke + 1 : b.ke;
    const long ni = b.nx1 + 2;
    const long n1 = (ni * (jhi - jlo + 1) * (khi - klo + 1) - 1 + 254) / 255;
    x[0] = {0, 0, jlo, jhi - jlo + 1, klo, khi};
    x[1] = {0, (int)((ni * (khi - klo + 1) + 63) / 64), klo, khi - klo + 1, b.js, b.je + 1};
    x[2] = {0, (int)((ni * (jhi - jlo + 1) + 63) / 64), jlo, jhi - jlo + 1, b.ks, b.ke + 1};
    const long n2 = b.ndim > 1 ? (long)x[1].nx * ((b.nx2 + 1 + ALL_TY - 2) / (ALL_TY - 1)) : 0;
    const long n3 = b.ndim > 2 ? (long)x[2].nx * ((b.nx3 + 1 + ALL_TY - 2) / (ALL_TY - 1)) : 0;
    const long n = n1 + n2 + n3;
    if (n > ALL_TILES) return 0;
    x[1].first = (int)n1;
    x[2].first = (int)(n1 + n2);
    return (int)n;
}
template <int SPEEDS, typename R, int GEO>
static hipError_t launch_all(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int recon, const Vars<const R>& P,
                               const Vars<R>& F, R* ctop, const FluxTiles (&x)[3], int n, hipStream_t s) {
#define KH_ALL(RECON) \
    hipLaunchKernelGGL((flux_all_kernel<RECON, SPEEDS, R, R, GEO>), dim3((unsigned)n), dim3(256), 0, s, b, c, gd, P, F, ctop, x[0], x[1], x[2])
    switch (recon) {
    case RECON_DONOR: KH_ALL(RECON_DONOR); break;
    case RECON_LINEAR_MC: KH_ALL(RECON_LINEAR_MC); break;
    case RECON_PPM: KH_ALL(RECON_PPM); break;
    default: KH_ALL(RECON_WENO5);
    }
#undef KH_ALL
    return hipGetLastError();
}
template <typename R>
static hipError_t launch_all_prec(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int recon, int speeds,
                                    const R* P, R* F, R* ctop, const FluxTiles (&x)[3], int n, hipStream_t s) {
    const Vars<const R> Pv = vars_of(P, b.nc);
    const Vars<R> Fv = vars_of(F, b.nc);
    if (b.geo)
        return speeds == SPEEDS_CTOP ? launch_all<SPEEDS_CTOP, R, 1>(b, c, gd, recon, Pv, Fv, ctop, x, n, s)
                                     : launch_all<SPEEDS_NONE, R, 1>(b, c, gd, recon, Pv, Fv, ctop, x, n, s);
    return speeds == SPEEDS_CTOP ? launch_all<SPEEDS_CTOP, R, 0>(b, c, gd, recon, Pv, Fv, ctop, x, n, s)
                                 : launch_all<SPEEDS_NONE, R, 0>(b, c, gd, recon, Pv, Fv, ctop, x, n, s);
}
hipError_t launch_flux_stage_all(const BlockDims& b, const StepConsts& c, const GeomDev& gd, FluxRoute rt, int recon, int prec,
                                 int speeds, const double* P, const float* P32, void* F, void* ctop, hipStream_t s) {
    FluxTiles x[3];
    const bool march = prec == PREC_FP64 && rt.xt;
    const int n = (speeds == SPEEDS_BOTH || march) ? 0 : all_tiles(b, x);
    if (n)
        return prec == PREC_SPLIT
                   ? launch_all_prec<float>(b, c, gd, recon, speeds, P32, (float*)F, (float*)ctop, x, n, s)
                   : launch_all_prec<double>(b, c, gd, recon, speeds, P, (double*)F, (double*)ctop, x, n, s);
    const long e = prec == PREC_SPLIT ? sizeof(float) : sizeof(double);
    for (int dir = 1; dir <= b.ndim; ++dir) {
        const hipError_t r = launch_flux_stage(b, c, gd, rt, dir, recon, prec, speeds, P, P32, (char*)F + e * (dir - 1) * NV * b.nc,
                                               (char*)ctop + e * (dir - 1) * b.nc, s, nullptr);
        if (r != hipSuccess) return r;
    }
    return hipSuccess;
}

// ---------------------------------------------- first-order flux correction
// Flux::FOFC (flux/fofc.cpp:113-226) with its defaults (LLF, speeds from both
// states, cell-centred B): each face of the consumed ranges next to a marked
// zone gets the LLF flux of the two zones' own primitives, and its speeds.
// `mark` holds the interior marks; a ghost zone reads the mark of its periodic
// image or, across a physical face, of the nearest interior zone -- what the
// outflow and reflecting fills of the synced flag give for the one ghost layer
// a consumed face touches.
__device__ __forceinline__ int fofc_source(int v, int s, int e, int n, int periodic) {
    if (v >= s && v <= e) return v;
    if (periodic) return v < s ? v + n : v - n;
    return v < s ? s : e;
}
template <int DIR, int SPEEDS, int GEO>
__global__ void __launch_bounds__(256)
fofc_flux_kernel(BlockDims b, StepConsts c, GeomDev gd, Vars<const double> P, const int* __restrict__ mark,
                 Vars<double> F, double* __restrict__ cmax_out, double* __restrict__ cmin_out, bool ghost_marks) {
    const int m1 = (DIR == 1) ? b.nx1 + 1 : b.nx1 + 2;
    const int m2 = (b.ndim < 2) ? 1 : (DIR == 2) ? b.nx2 + 1 : b.nx2 + 2;
    const int m3 = (b.ndim < 3) ? 1 : (DIR == 3) ? b.nx3 + 1 : b.nx3 + 2;
    const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;   // face counts stay below 2^31
    if (t >= (unsigned)m1 * (unsigned)m2 * (unsigned)m3) return;
    const int i = ((DIR == 1) ? b.is : b.is - 1) + (int)(t % (unsigned)m1);
    const unsigned r = t / (unsigned)m1;
    const int j = ((b.ndim < 2 || DIR == 2) ? b.js : b.js - 1) + (int)(r % (unsigned)m2);
    const int k = ((b.ndim < 3 || DIR == 3) ? b.ks : b.ks - 1) + (int)(r / (unsigned)m2);
    // a ghost of a shared face keeps its own (synced) mark when ghost_marks is set
    auto src = [&](int v, int s, int e, int n, int d) {
        if (ghost_marks && ((v < s && b.img[d][0]) || (v > e && b.img[d][1]))) return v;
        return fofc_source(v, s, e, n, b.periodic[d]);
    };
    auto marked = [&](int kk, int jj, int ii) {
        ii = src(ii, b.is, b.ie, b.nx1, 0);
        if (b.ndim > 1) jj = src(jj, b.js, b.je, b.nx2, 1);
        if (b.ndim > 2) kk = src(kk, b.ks, b.ke, b.nx3, 2);
        return mark[(long)kk * b.s3 + (long)jj * b.s2 + ii] != 0;
    };
    if (!marked(k, j, i) && !marked(DIR == 3 ? k - 1 : k, DIR == 2 ? j - 1 : j, DIR == 1 ? i - 1 : i)) return;
    const long ci = (long)k * b.s3 + (long)j * b.s2 + i;
    const long st = (DIR == 1) ? 1 : (DIR == 2) ? b.s2 : b.s3;
    double Pl[NV], Pr[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        Pl[v] = P[v][ci - st];
        Pr[v] = P[v][ci];
    }
    face_flux<DIR, SPEEDS, double, GEO>(c, b, gd, j, i, Pl, Pr, ci, F, cmax_out, cmin_out);
}

template <int DIR, int SPEEDS>
static hipError_t launch_fofc_dir(const BlockDims& b, const StepConsts& c, const GeomDev& gd, const Vars<const double>& P,
                                  const int* mark, const Vars<double>& F, double* cmax, double* cmin, hipStream_t s,
                                  bool gm) {
    const long m1 = (DIR == 1) ? b.nx1 + 1 : b.nx1 + 2;
    const long m2 = (b.ndim < 2) ? 1 : (DIR == 2) ? b.nx2 + 1 : b.nx2 + 2;
    const long m3 = (b.ndim < 3) ? 1 : (DIR == 3) ? b.nx3 + 1 : b.nx3 + 2;
    const dim3 grid((unsigned)((m1 * m2 * m3 + 255) / 256));
    if (b.geo) fofc_flux_kernel<DIR, SPEEDS, 1><<<grid, 256, 0, s>>>(b, c, gd, P, mark, F, cmax, cmin, gm);
    else fofc_flux_kernel<DIR, SPEEDS, 0><<<grid, 256, 0, s>>>(b, c, gd, P, mark, F, cmax, cmin, gm);
    return hipGetLastError();
}

template <int SPEEDS>
static hipError_t launch_fofc_speeds(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int dir,
                                     const Vars<const double>& P, const int* mark, const Vars<double>& F, double* cmax,
                                     double* cmin, hipStream_t s, bool gm) {
    if (dir == 1) return launch_fofc_dir<1, SPEEDS>(b, c, gd, P, mark, F, cmax, cmin, s, gm);
    if (dir == 2) return launch_fofc_dir<2, SPEEDS>(b, c, gd, P, mark, F, cmax, cmin, s, gm);
    return launch_fofc_dir<3, SPEEDS>(b, c, gd, P, mark, F, cmax, cmin, s, gm);
}

hipError_t launch_fofc_flux(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int speeds,
                            const Vars<const double>& P, const int* mark, const FluxVars<double>& F, double* cmax,
                            double* cmin, hipStream_t s, bool ghost_marks) {
    StepConsts cl = c;   // first-order states: no reconstruction floors; LLF whatever flux/type says
    cl.recon_floors = 0;
    cl.use_hlle = 0;
    for (int dir = 1; dir <= b.ndim; ++dir) {
        double* cx = cmax ? cmax + (long)(dir - 1) * b.nc : nullptr;
        double* cn = cmin ? cmin + (long)(dir - 1) * b.nc : nullptr;
        hipError_t e;
        if (speeds == SPEEDS_CTOP) e = launch_fofc_speeds<SPEEDS_CTOP>(b, cl, gd, dir, P, mark, F[dir - 1], cx, cn, s, ghost_marks);
        else if (speeds == SPEEDS_BOTH) e = launch_fofc_speeds<SPEEDS_BOTH>(b, cl, gd, dir, P, mark, F[dir - 1], cx, cn, s, ghost_marks);
        else e = launch_fofc_speeds<SPEEDS_NONE>(b, cl, gd, dir, P, mark, F[dir - 1], cx, cn, s, ghost_marks);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace kh
