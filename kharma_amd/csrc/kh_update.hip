// kh_update.hip -- the fused stage update.  For one interior zone and in registers:
//   flux-CT B fluxes from the corner EMFs (B_FluxCT::FluxCT, b_flux_ct.cpp:347-369)
//   + flux divergence (KHARMADriver::FluxDivergence, kharma_driver.hpp:208-231)
//   + RK state update (KHARMADriver::AddStateUpdate, kharma_driver.cpp:339-387)
//   + onedw U->P (Inverter::BlockUtoP, inverter.cpp:131-182) and B U->P (b_flux_ct.cpp:195-217)
//   + floors (Floors::ApplyGRMHDFloors, floors_impl.hpp:45-128)
//   + P->U (Flux::MeshPtoU, flux.cpp:276-322)
//   + (last stage) the CFL estimate (GRMHD::EstimateTimestep, grmhd.cpp:313-328)
// and writes U, P and the flags once, also into the periodic ghost images of
// the zone (the boundary exchange), so no separate sync pass reads the state.
#include "kh_step.hpp"

namespace kh {

// --------------------------------------- fused stage update, flat space
// Compiled for 4 work-groups per CU (128 VGPRs).
// Stage 1 (gam0 = 0 and U_sub == U_full) reads the state once: 0*U + 1*U == U.
// ND: the dimensionality where it is known at compile time, else 0.  Known, the
// fluxes are requested in one go instead of in two parts about a branch, which suits
// 2-D blocks and FP32 fluxes: FP64 256^2 13.4 / 15.9 -> 12.2 / 14.7 us, split 128^3 213 /
// 270 -> 212 / 257 us (stage 1 / 2).  The 48 FP64 fluxes of a 3-D zone do not fit 128
// registers at once (168-196 byte spill; at three wavefronts 64^3 29 / 34 -> 32 / 40 us);
// in two parts 24-52 bytes spill.
// BM: 0 no B transport (1-D), 1 flux-CT EMFs from the face fluxes, 2 face-centred
// B (B_CT): the cell B is the average of the stage's new faces fB (B_CT::BlockUtoP,
// b_ct.cpp:173-205, which the reference runs before the inversion).
template <typename R, bool DO_DT, int ND, int BM, int INV = 0, bool PK = false>
__global__ void __launch_bounds__(BS, 4)
update_kernel(BlockDims b, StepConsts cst, GeomDev gd, int stage, const R* __restrict__ F, const R* __restrict__ ctop,
              const double* __restrict__ Usub, const double* Ufull, const double* __restrict__ Psub,
              double* Uout, double* __restrict__ Pout, float* __restrict__ Pout32,
              int* __restrict__ pflag, int* __restrict__ fflag, int* __restrict__ fail_list,
              DeviceState* __restrict__ ds, double* __restrict__ dt_part, const double* __restrict__ fB,
              const BlockEntry* __restrict__ pk) {
    if constexpr (PK) {
        const long blk = pack_select(pk, b, gd);
        const long sv = blk * NV * b.nc;
        F = pack_at(F, 3 * sv);
        ctop = pack_at(ctop, blk * 3 * b.nc);
        Usub = pack_at(Usub, sv); Ufull = pack_at(Ufull, sv); Psub = pack_at(Psub, sv);
        Uout = pack_at(Uout, sv); Pout = pack_at(Pout, sv); Pout32 = pack_at(Pout32, sv);
        pflag = pack_at(pflag, blk * b.nc); fflag = pack_at(fflag, blk * b.nc); fail_list = pack_at(fail_list, blk * b.nc);
        ds += blk;
        dt_part = pack_at(dt_part, blk * gridDim.x);
    }
    const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = t < (unsigned)ninterior(b);
    double ndt = DBL_MAX;
    if (active) {
        int k, j, i;
        interior_index(b, t, k, j, i);
        const long c = (long)k * b.s3 + (long)j * b.s2 + i;
        const double gam = cst.gam;
        const int nd = ND ? ND : b.ndim;
        double dudt[NV];
        if constexpr (BM == 1) zone_divergence_ct<R, ND>(b, F, c, dudt);
        else zone_divergence<R>(b, flux_vars_of(F, b.nc), nullptr, c, false, dudt, BM == 2);
        const double g0 = cst.gam0[stage - 1], g1 = cst.gam1[stage - 1];
        const double beta_dt = cst.beta[stage - 1] * ds->dt;
        const bool same = (g0 == 0.) && (Usub == Ufull);
        double U[NV], P[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double uf = Ufull[v * b.nc + c];
            const double u = same ? uf : g0 * Usub[v * b.nc + c] + g1 * uf;
            U[v] = 1.0 * u + beta_dt * dudt[v];
        }
        if constexpr (BM == 2) {
            const long f = (long)k * b.fs3 + (long)j * b.fs2 + i;
            U[B1] = (fB[f] + fB[f + 1]) / 2;
            U[B2] = (fB[b.nf + f] + fB[b.nf + f + b.fs2]) / 2;
            U[B3] = (b.ndim > 2) ? (fB[2 * b.nf + f] + fB[2 * b.nf + f + b.fs3]) / 2 : fB[2 * b.nf + f];
        }
        // U->P guess: the stage's starting primitives (kharma_driver.cpp:379-384)
#pragma unroll
        for (int v = 0; v < 5; ++v) P[v] = Psub[v * b.nc + c];
        int pf = 0, ff = 0;
        double rf, uf;
        geom_floors<0>(cst, gd, j, i, rf, uf);
        with_center_geom<0>(gd, j, i, [&](const auto& g) {
            pf = invert_zone<INV>(g, U, P, cst);
            const int ff0 = (pf / F_GEOM_RHO) * F_GEOM_RHO;
            pf = pf % F_GEOM_RHO;
            const double gd_ = g.gdet();
            const double igd = rcp(gd_);
            P[B1] = U[B1] * igd; P[B2] = U[B2] * igd; P[B3] = U[B3] * igd;
            FourVec<double> D;
            calc_4vecs<double>(g, P, D);
            ff = ff0;
            if (cst.floors.on) ff = floors_zone(g, P, U, D, gam, cst.floors, rf, uf, ff0, pf);
            p_to_u_D(g, P, D, gam, U);
        });
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
        if (DO_DT) {
            const double n = zone_ndt(b, (double)ctop[c], nd > 1 ? (double)ctop[b.nc + c] : 0.,
                                      nd > 2 ? (double)ctop[2 * b.nc + c] : 0.);
            if (!(n != n)) ndt = n;
        }
    }
    if (DO_DT) {
        const double m = block_min(ndt);
        if (threadIdx.x == 0) dt_part[blockIdx.x] = m;
    }
}

long update_blocks(const BlockDims& b) { return (ninterior_host(b) + BS - 1) / BS; }
long dt_blocks(const BlockDims& b) { return (b.geo && b.ndim == 3) ? update_tiles_host(b) : update_blocks(b); }

// The curved-space update (kh_update_geo.hpp), R the element type of the fluxes;
// with Ustar non-null the interior zones' U* is stored there too.
template <typename R>
void launch_update_geo(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int stage, bool do_dt,
                       const void* F, const void* ctop, const double* Usub, const double* Ufull,
                       const double* Psub, double* Uout, double* Pout, float* Pout32, int* pflag, int* fflag,
                       int* fail_list, DeviceState* ds, double* dt_part, hipStream_t s, double* Ustar, const Pack* pk);
extern template void launch_update_geo<float>(
    const BlockDims&, const StepConsts&, const GeomDev&, int, bool, const void*, const void*, const double*,
    const double*, const double*, double*, double*, float*, int*, int*, int*, DeviceState*, double*, hipStream_t,
    double*, const Pack*);
extern template void launch_update_geo<double>(
    const BlockDims&, const StepConsts&, const GeomDev&, int, bool, const void*, const void*, const double*,
    const double*, const double*, double*, double*, float*, int*, int*, int*, DeviceState*, double*, hipStream_t,
    double*, const Pack*);
template <typename R, bool PK>
static void launch_update_t_k(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int stage, bool do_dt,
                            const void* F, const void* ctop, const double* Usub, const double* Ufull, const double* Psub,
                            double* Uout, double* Pout, float* Pout32, int* pflag, int* fflag,
                            int* fail_list, DeviceState* ds, double* dt_part, hipStream_t s, const double* fB,
                            const Pack* pk) {
    const dim3 g = pack_grid(grid_for(ninterior_host(b)), pk);
    const int bm = fB ? 2 : (b.ndim > 1 ? 1 : 0);
    const BlockEntry* pd = pack_dev(pk);
    constexpr int ND3 = sizeof(R) == 4 ? 3 : 0;
#define KH_UPD(DT, ND, BM, INV)                                                                                         \
    hipLaunchKernelGGL((update_kernel<R, DT, ND, BM, INV, PK>), g, dim3(BS), 0, s, b, c, gd, stage, (const R*)F, (const R*)ctop, \
                       Usub, Ufull, Psub, Uout, Pout, Pout32, pflag, fflag, fail_list, ds, dt_part, fB, pd)
#define KH_UPD_BM(DT, INV)                                                                                            \
    {                                                                                                                 \
        if (bm == 2) KH_UPD(DT, 0, 2, INV);                                                                           \
        else if (bm == 0) KH_UPD(DT, 0, 0, INV);                                                                      \
        else if (b.ndim == 2) KH_UPD(DT, 2, 1, INV);                                                                  \
        else KH_UPD(DT, ND3, 1, INV);                                                                                 \
    }
    if (c.inverter == 1) {
        if (do_dt) KH_UPD_BM(true, 1) else KH_UPD_BM(false, 1)
    } else {
        if (do_dt) KH_UPD_BM(true, 0) else KH_UPD_BM(false, 0)
    }
#undef KH_UPD_BM
#undef KH_UPD
}
template <typename R>
static void launch_update_t(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int stage, bool do_dt,
                            const void* F, const void* ctop, const double* Usub, const double* Ufull, const double* Psub,
                            double* Uout, double* Pout, float* Pout32, int* pflag, int* fflag,
                            int* fail_list, DeviceState* ds, double* dt_part, hipStream_t s, const double* fB = nullptr,
                            const Pack* pk = nullptr) {
    if (pk) launch_update_t_k<R, true>(b, c, gd, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, Pout32,
                                            pflag, fflag, fail_list, ds, dt_part, s, fB, pk);
    else launch_update_t_k<R, false>(b, c, gd, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, Pout32,
                                          pflag, fflag, fail_list, ds, dt_part, s, fB, pk);
}
hipError_t launch_update_faces(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int prec, int stage,
                               bool do_dt, const void* F, const void* ctop, const double* Usub, const double* Ufull,
                               const double* Psub, double* Uout, double* Pout, float* Pout32, int* pflag, int* fflag,
                               int* fail_list, DeviceState* ds, double* dt_part, const double* fB, hipStream_t s) {
    if (b.geo || !fB) return hipErrorInvalidValue;
    if (prec == PREC_SPLIT)
        launch_update_t<float>(b, c, gd, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, Pout32, pflag, fflag,
                                  fail_list, ds, dt_part, s, fB);
    else
        launch_update_t<double>(b, c, gd, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, Pout32, pflag, fflag,
                                   fail_list, ds, dt_part, s, fB);
    return hipGetLastError();
}
hipError_t launch_update(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int prec, int stage, bool do_dt,
                         const void* F, const void* ctop, const double* Usub, const double* Ufull, const double* Psub,
                         double* Uout, double* Pout, float* Pout32, int* pflag, int* fflag,
                         int* fail_list, DeviceState* ds, double* dt_part, hipStream_t s, const Pack* pk) {
    if (prec == PREC_SPLIT) {
        if (b.geo) launch_update_geo<float>(b, c, gd, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, Pout32, pflag, fflag, fail_list, ds, dt_part, s, nullptr, pk);
        else launch_update_t<float>(b, c, gd, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, Pout32, pflag, fflag, fail_list, ds, dt_part, s, nullptr, pk);
    } else {
        if (b.geo) launch_update_geo<double>(b, c, gd, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, Pout32, pflag, fflag, fail_list, ds, dt_part, s, nullptr, pk);
        else launch_update_t<double>(b, c, gd, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, Pout32, pflag, fflag, fail_list, ds, dt_part, s, nullptr, pk);
    }
    return hipGetLastError();
}
hipError_t launch_update_recorded(const BlockDims& b, const StepConsts& c, const GeomDev& gd, int stage, bool do_dt,
                                  const void* F, const void* ctop, const double* Usub, const double* Ufull,
                                  const double* Psub, double* Uout, double* Pout, int* pflag, int* fflag,
                                  int* fail_list, DeviceState* ds, double* dt_part, double* Ustar, hipStream_t s) {
    if (!b.geo)
        return launch_update(b, c, gd, PREC_FP64, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, nullptr, pflag,
                             fflag, fail_list, ds, dt_part, s);
    launch_update_geo<double>(b, c, gd, stage, do_dt, F, ctop, Usub, Ufull, Psub, Uout, Pout, nullptr, pflag, fflag,
                              fail_list, ds, dt_part, s, Ustar, nullptr);
    return hipGetLastError();
}

}  // namespace kh
