// kh_update_geo.hpp -- the stage update in curved space.  The kernels for FP64 and
// for FP32 fluxes are compiled in files of their own (kh_update_f64.hip,
// kh_update_f32.hip), which build side by side.
#pragma once
#include "kh_step.hpp"

namespace kh {

// U->P from the guess P, B from U, floors in frame FRAME, P->U of one zone (k, j, i)
// at c; STG: metric and floors from the tile's LDS copy sg.
template <int FRAME, int INV, bool STG, int TI>
__device__ __forceinline__ void recover_zone(const BlockDims& b, const StepConsts& cst, const GeomDev& gd, int stage,
                                             double* Uout, double* __restrict__ Pout,
                                             float* __restrict__ Pout32, int* __restrict__ pflag,
                                             int* __restrict__ fflag, int* __restrict__ fail_list,
                                             DeviceState* __restrict__ ds, double* __restrict__ Ustar,
                                             const double* sg, int k, int j, int i, long c, double (&U)[NV],
                                             double (&P)[NV]) {
    const double gam = cst.gam;
    int pf = 0, ff = 0;
    double rf, uf;
    const int lane = (int)(threadIdx.x % TI);
    if (Ustar) {   // the stage's U* for the differentiation form's record
#pragma unroll
        for (int v = 0; v < NV; ++v) Ustar[v * b.nc + c] = U[v];
    }
    if constexpr (STG) {
        rf = sg[GEO_NCOMP * TI + lane];
        uf = sg[(GEO_NCOMP + 1) * TI + lane];
    } else {
        geom_floors<1>(cst, gd, j, i, rf, uf);
    }
    {
        CachedGeom<double> g(STG ? sg : gd.g[GLOC_CENTER], STG ? TI : gd.np, STG ? lane : (long)j * gd.gn1 + i);
        pf = invert_zone<INV>(g, U, P, cst);
        const int ff0 = (pf / F_GEOM_RHO) * F_GEOM_RHO;
        pf = pf % F_GEOM_RHO;
        const double gd_ = g.gdet();
        const double igd = rcp(gd_);
        P[B1] = U[B1] * igd; P[B2] = U[B2] * igd; P[B3] = U[B3] * igd;
        FourVec<double> D;
        calc_4vecs<double, true>(g, P, D);
        ff = ff0;
        if (cst.floors.on) ff = floors_zone<FRAME>(g, P, U, D, gam, cst.floors, rf, uf, ff0, pf);
        p_to_u_D(g, P, D, gam, U);
    }
    ImageSet s;
    image_set(b, k, j, i, s);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        store_with_images(b, s, Uout + v * b.nc, c, U[v], NV * b.nc);
        store_with_images(b, s, Pout + v * b.nc, c, P[v], NV * b.nc);
        if (Pout32) store_with_images(b, s, Pout32 + v * b.nc, c, (float)P[v], NV * b.nc);
    }
    store_with_images(b, s, pflag, c, pf, b.nc);
    fflag[c] = ff;
    if (pf > 0) {
        const int slot = atomicAdd(&ds->fail_count[stage - 1], 1);
        fail_list[slot] = (int)c;
    }
}

// --------------------------------------------- curved-space stage update
// The same update in curved space: flux-CT divergence, geometric source
// (flux.cpp:395-444) and RK combination give U*, then the recovery.  ND:
// dimensionality (flux-CT for 2 and 3); SAME: the stage with gam0 = 0 and U_sub ==
// U_full, which reads the state once (0*U + 1*U == U) and estimates no timestep.
//
// One launch: as two (combination to U*, recovery from it) it made a round trip of
// U* and the guess through memory (200 bytes per zone), loaded the metric twice,
// and the first of the two spent its life waiting on loads while the second, bound
// by FP64 chains, left memory idle.  Fused, the recovery of one wavefront overlaps
// the loads of another.  192x128x128 torus, stage 1 / stage 2: FP64 551 / 601 ->
// 418 / 473 us, FP32 fluxes 500 / 536 -> 383 / 446 us, these as 2x2x4 blocks 572 / 645 ->
// 494 / 541 us; 256x128, FP64: 18 / 20 -> 13.5 / 14.5 us.  The bytes that cannot be avoided
// take 270-330 us at the rate of a copy.
//
// In 3-D the zones run on tiles with the metric and floors staged in LDS, which
// both halves read (stage 1 / 2 unstaged 499 / 562 us).  Three wavefronts per SIMD
// (118-168 VGPRs; with FP32 fluxes and onedw stage 1 takes 124-126 in the drift frame
// and runs four): a bound of four spills 28-76 bytes and slows stage 2 (482 -> 525 us).  Staging
// the 40 connection components too measured 455 / 499 us, requesting the primitives
// ahead of the staging barrier 441 / 487 us.
//
// The source is summed apart, before the state and the fluxes are loaded, but for FP64
// fluxes in 2-D (and 1-D), which add it to the divergence, after requesting the fluxes,
// with the halves kept apart for the scheduler and a bound of two wavefronts.  The two
// round differently: this form keeps the bits of 2-D FP64 runs and their gradients.
// In time it holds its own in small blocks only.  Stage 1 / 2 of the 2-D torus in this
// form against the 3-D one (three wavefronts): 256x128 14.8 / 15.9 and 14.5 / 16.2 us,
// 512x256 28 / 30 and 26 / 28.5, 1024x512 107 / 116 and 98 / 109, 2048x1536 624 / 699 and
// 602 / 662.
//
// The guess passes through an empty asm: the source and the solver form the same
// products of it, and sharing them would round the solver's differently from a
// solver that loads its guess.
template <int ND> struct UpdateGeoOcc { static constexpr int w = ND == 3 ? 3 : 2; };
template <typename R, int ND, bool SAME, int FRAME, int INV, bool PK, int TI = 64>
__global__ void __launch_bounds__(BS, UpdateGeoOcc<ND>::w)
update_geo_kernel(BlockDims b, StepConsts cst, GeomDev gd, int stage, const R* __restrict__ F, const R* __restrict__ ctop,
                  const double* __restrict__ Usub, const double* Ufull, const double* __restrict__ Psub, double* Uout,
                  double* __restrict__ Pout, float* __restrict__ Pout32, int* __restrict__ pflag,
                  int* __restrict__ fflag, int* __restrict__ fail_list, DeviceState* __restrict__ ds,
                  double* __restrict__ dt_part, double* __restrict__ Ustar, const BlockEntry* __restrict__ pk) {
    constexpr bool STG = ND == 3;
    __shared__ double sg[STG ? STG_GEOM * TI : 1];
    if constexpr (PK) {
        const long blk = pack_select(pk, b, gd);
        const long sv = blk * NV * b.nc;
        F = pack_at(F, 3 * sv);
        ctop = pack_at(ctop, blk * 3 * b.nc);
        Usub = pack_at(Usub, sv); Ufull = pack_at(Ufull, sv); Psub = pack_at(Psub, sv); Uout = pack_at(Uout, sv);
        Pout = pack_at(Pout, sv); Pout32 = pack_at(Pout32, sv); Ustar = pack_at(Ustar, sv);
        pflag = pack_at(pflag, blk * b.nc); fflag = pack_at(fflag, blk * b.nc); fail_list = pack_at(fail_list, blk * b.nc);
        ds += blk;
        dt_part = pack_at(dt_part, blk * gridDim.x);
    }
    int k, j, i;
    bool active;
    if constexpr (STG) {
        int i0;
        active = tile_zone<TI>(b, k, j, i, i0);
        stage_tile_geometry<TI>(gd, j, i0, sg);
    } else {
        const unsigned t = xcd_logical_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
        active = t < (unsigned)ninterior(b);
        if (active) interior_index_jki(b, t, k, j, i);
    }
    double ndt = DBL_MAX;
    if (active) {
        const long c = (long)k * b.s3 + (long)j * b.s2 + i;
        const double g0 = cst.gam0[stage - 1], g1 = cst.gam1[stage - 1];
        constexpr bool SRC_FIRST = sizeof(R) == 4 || ND == 3;
        auto source = [&](double acc[NV]) {
            double Ps[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) Ps[v] = Psub[v * b.nc + c];
            const long q = (long)j * gd.gn1 + i;
            CachedGeom<double> g(STG ? sg : gd.g[GLOC_CENTER], STG ? TI : gd.np, STG ? (long)(threadIdx.x % TI) : q);
            add_geo_source(g, gd, q, Ps, cst.gam, acc);
        };
        double dS[NV] = {0., 0., 0., 0., 0., 0., 0., 0.};
        if constexpr (SRC_FIRST) source(dS);
        double U[NV], P[NV];   // U first holds the stage's base state, requested early
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double uf = Ufull[v * b.nc + c];
            U[v] = SAME ? uf : g0 * Usub[v * b.nc + c] + g1 * uf;
        }
        double dudt[NV];
        if constexpr (ND > 1) zone_divergence_ct<R, ND>(b, F, c, dudt);
        else zone_divergence<R>(b, flux_vars_of(F, b.nc), nullptr, c, false, dudt);
        if constexpr (SRC_FIRST) {
#pragma unroll
            for (int v = UU; v <= U3; ++v) dudt[v] += dS[v];
        } else {
            source(dudt);
        }
        const double beta_dt = cst.beta[stage - 1] * ds->dt;
#pragma unroll
        for (int v = 0; v < NV; ++v) U[v] = 1.0 * U[v] + beta_dt * dudt[v];
        if constexpr (!SAME) {   // without an estimate to make, ctop is any readable array
            const double n = zone_ndt(b, (double)ctop[c], ND > 1 ? (double)ctop[b.nc + c] : 0.,
                                      ND > 2 ? (double)ctop[2 * b.nc + c] : 0.);
            if (!(n != n)) ndt = n;
        }
        if constexpr (ND < 3) __builtin_amdgcn_sched_barrier(0);
        // the guess: the stage's starting fluid primitives (kharma_driver.cpp:379-384)
#pragma unroll
        for (int v = 0; v < 5; ++v) P[v] = Psub[v * b.nc + c];
#pragma unroll
        for (int v = 0; v < 5; ++v) asm("" : "+v"(P[v]));
        recover_zone<FRAME, INV, STG, TI>(b, cst, gd, stage, Uout, Pout, Pout32, pflag, fflag, fail_list, ds, Ustar, sg,
                                          k, j, i, c, U, P);
    }
    if (!SAME && dt_part) {
        const double m = block_min(ndt);
        if (threadIdx.x == 0) dt_part[blockIdx.x] = m;
    }
}

template <typename R, bool PK>
static void launch_update_geo_k(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int stage, bool do_dt,
                                const void* F, const void* ctop, const double* Usub, const double* Ufull,
                                const double* Psub, double* Uout, double* Pout, float* Pout32, int* pflag, int* fflag,
                                int* fail_list, DeviceState* ds, double* dt_part, hipStream_t s, double* Ustar,
                                const Pack* pk) {
    const dim3 g = pack_grid(dim3((unsigned)dt_blocks(b)), pk);
    const bool ti32 = tile_width(b) == 32;
    const BlockEntry* pd = pack_dev(pk);
    const bool same = (c.gam0[stage - 1] == 0.) && (Usub == Ufull) && !do_dt;
    if (!do_dt) { ctop = F; dt_part = nullptr; }
#define KH_UG(ND, SAME, FR, INV, TI)                                                                                  \
    hipLaunchKernelGGL((update_geo_kernel<R, ND, SAME, FR, INV, PK, TI>), g, dim3(BS), 0, s, b, c, gd, stage, (const R*)F, \
                       (const R*)ctop, Usub, Ufull, Psub, Uout, Pout, Pout32, pflag, fflag, fail_list, ds, dt_part, Ustar, pd)
#define KH_UG_ND(SAME, FR, INV)                                                                                       \
    do {                                                                                                              \
        if (b.ndim == 3 && ti32) KH_UG(3, SAME, FR, INV, 32);                                                         \
        else if (b.ndim == 3) KH_UG(3, SAME, FR, INV, 64);                                                            \
        else if (b.ndim == 2) KH_UG(2, SAME, FR, INV, 64);                                                            \
        else KH_UG(1, SAME, FR, INV, 64);                                                                             \
    } while (0)
#define KH_UG_SAME(FR, INV) do { if (same) KH_UG_ND(true, FR, INV); else KH_UG_ND(false, FR, INV); } while (0)
    if (c.inverter == 1) {
        if (c.floors.frame == 0) KH_UG_SAME(0, 1);
        else if (c.floors.frame == 1) KH_UG_SAME(1, 1);
        else KH_UG_SAME(2, 1);
    } else {
        if (c.floors.frame == 0) KH_UG_SAME(0, 0);
        else if (c.floors.frame == 1) KH_UG_SAME(1, 0);
        else KH_UG_SAME(2, 0);
    }
#undef KH_UG_SAME
#undef KH_UG_ND
#undef KH_UG
}
template <typename R>
void launch_update_geo(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int stage, bool do_dt,
                       const void* F, const void* ctop, const double* Usub, const double* Ufull,
                       const double* Psub, double* Uout, double* Pout, float* Pout32, int* pflag, int* fflag,
                       int* fail_list, DeviceState* ds, double* dt_part, hipStream_t s, double* Ustar, const Pack* pk) {
    if (pk) launch_update_geo_k<R, true>(b, c, gd, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, Pout32, pflag,
                                         fflag, fail_list, ds, dt_part, s, Ustar, pk);
    else launch_update_geo_k<R, false>(b, c, gd, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, Pout32, pflag,
                                       fflag, fail_list, ds, dt_part, s, Ustar, pk);
}

}  // namespace kh
