// kh_lane_geom.hpp -- the metric that a lane of a marching flux kernel keeps in LDS.
#pragma once
#include "kh_internal.hpp"

namespace kh {

// Slots of one lane: the metric components that the flux through a face normal to
// DIR needs, then the floors.  g_{t x2} and g_{x2 phi} have none: they vanish in
// every embedding the cache is built for (the upload checks the tables, and a block
// whose tables hold others is routed to the tiles: flux_route).
enum {
    MG_G00, MG_G01, MG_G03, MG_G11, MG_G12, MG_G13, MG_G22, MG_G33, MG_U00, MG_U01, MG_U02, MG_U03, MG_UDD, MG_GDET,
    MG_ALPHA, MG_RF, MG_UF, MG_N
};

// One lane's metric in slots [MG_N][256].  Components are named at compile time; one
// without a slot does not compile.
template <int DIR> struct LaneGeom {
    static constexpr bool flat = false;
    const double (*s)[256];
    int t;
    static __device__ __forceinline__ constexpr int src(int m) {   // component of the cached table
        return m == MG_G00 ? 0 : m == MG_G01 ? 1 : m == MG_G03 ? 3 : m == MG_G11 ? 4 : m == MG_G12 ? 5 : m == MG_G13 ? 6
             : m == MG_G22 ? 7 : m == MG_G33 ? 9 : m == MG_U00 ? 10 : m == MG_U01 ? 11 : m == MG_U02 ? 12 : m == MG_U03 ? 13
             : m == MG_UDD ? (DIR == 1 ? 14 : DIR == 2 ? 17 : 19) : m == MG_GDET ? GEO_GDET : GEO_ALPHA;
    }
    template <int A, int B> __device__ __forceinline__ double gcov() const {
        constexpr int l = A < B ? A : B, h = A < B ? B : A;
        static_assert(l >= 0 && h <= 3 && !(l == 0 && h == 2) && !(l == 2 && h == 3), "no slot for this component of g_{ab}");
        return s[l == 0 ? (h == 0 ? MG_G00 : h == 1 ? MG_G01 : MG_G03)
               : l == 1 ? (h == 1 ? MG_G11 : h == 2 ? MG_G12 : MG_G13) : l == 2 ? MG_G22 : MG_G33][t];
    }
    template <int A, int B> __device__ __forceinline__ double gcon() const {
        constexpr int l = A < B ? A : B, h = A < B ? B : A;
        static_assert(l >= 0 && h <= 3 && (l == 0 || (l == DIR && h == DIR)), "no slot for this component of g^{ab}");
        return s[l == 0 ? MG_U00 + h : MG_UDD][t];
    }
    __device__ __forceinline__ double gcon0(int v) const { return s[MG_U00 + v][t]; }
    __device__ __forceinline__ double gdet() const { return s[MG_GDET][t]; }
    __device__ __forceinline__ double alpha() const { return s[MG_ALPHA][t]; }
    // CachedGeom::lower and lorentz without the products with g_{t x2} and g_{x2 phi}
    __device__ __forceinline__ void lower(const double v[4], double o[4]) const {
        o[0] = fma(gcov<0, 3>(), v[3], fma(gcov<0, 0>(), v[0], gcov<0, 1>() * v[1]));
        o[1] = sum_a(gcov<0, 1>(), v[0], gcov<1, 1>(), v[1], gcov<1, 2>(), v[2], gcov<1, 3>(), v[3]);
        o[2] = fma(gcov<2, 2>(), v[2], gcov<1, 2>() * v[1]);
        o[3] = fma(gcov<3, 3>(), v[3], fma(gcov<0, 3>(), v[0], gcov<1, 3>() * v[1]));
    }
    __device__ __forceinline__ double lorentz(double u1, double u2, double u3) const {
        const double qsq = gcov<1, 1>() * u1 * u1 + gcov<2, 2>() * u2 * u2 + gcov<3, 3>() * u3 * u3 +
                           2. * (gcov<1, 2>() * u1 * u2 + gcov<1, 3>() * u1 * u3);
        return sqrt(1. + qsq);
    }
};
template <int A, int B, int DIR> __device__ __forceinline__ double gcon_at(const LaneGeom<DIR>& g) {
    return g.template gcon<A, B>();
}

}  // namespace kh
