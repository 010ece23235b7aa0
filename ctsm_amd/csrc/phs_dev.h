// phs_dev.h -- device pieces of plant hydraulic stress shared by phs.hip
// (the soil-side and calcstress kernels) and canopy.hip (CanopyFluxes with
// PhotosynthesisHydraulicStress): the parameter table's rows, the Weibull
// vulnerability curve plc and its derivative, and calcstress with getqflx,
// spacF, spacA and getvegwp (PhotosynthesisMod.F90:4490-5228).
#pragma once

#include "common.h"

namespace ctsm {
namespace phs {

constexpr double RPI = 3.14159265358979323846;   // SHR_CONST_PI
constexpr double C_TO_B = 2.0;                     // g biomass / g C (PhotosynthesisMod.F90:2911)
constexpr double CROOT_LATERAL_LENGTH = 0.25;      // m (:2910)

// rows of the device parameter table, CTSM_MAX_PFT values each
enum { T_KRMAX = 0, T_RADIUS = 1, T_DENSITY = 2, T_FROOT_LEAF = 3, T_PSI50 = 4, T_CK = 8, T_KMAX = 12, T_CROP = 16, T_ROWS = 17 };

// plc, vegetation_weibull branch: 2**(-(x/psi50)**ck), cut to zero below 0.005
// (lt: log's table)
__device__ __forceinline__ double plc(double x, double psi50, double ck, const double *lt)
{
    double v = cm_pow(2.0, -cm_pow_tab(x / psi50, ck, lt));
    if (v < 0.005) v = 0.0;
    return v;
}

// ---- calcstress (PhotosynthesisMod.F90:4490-4710) for one patch ---------------
// Segments 0 sun, 1 sha, 2 xyl, 3 root.  The helpers follow the reference's
// routines statement by statement, so every lane performs the Fortran's
// operations in the Fortran's order.
constexpr double RGAS = 6.02214e26 * 1.38065e-23;   // SHR_CONST_AVOGAD * SHR_CONST_BOLTZ
constexpr double LN2 = 0.6931471805599453;         // log(2._r8), correctly rounded
constexpr double SPVAL = 1.e36;
constexpr double TOL_LAI = 0.001;

struct Leaf {
    double laisun, laisha, elai, esai, tsai, htop, fdry, thm, rho, pbot, gb;
    double kmax[4], psi50[4], ck[4];
    // The soil below the patch, staged once (stage_soil): k_soil_root(p, :) and
    // 1000 z(c, :) in the lane's LDS column, and the sums over the layers that
    // no potential enters -- of k, k smp, smp - 1000 z and k (smp - 1000 z).
    const double *k, *g;
    double sum_k, sum_ks, sum_w, sum_kw;
    const double *lt;            // log's table in LDS
    const double *smp;           // layer 1 of smp_l(c, :), stride ss
    long ss;
    int n;
};
// LDS doubles per lane of a one-wave block, and the stride between layers
constexpr int SOIL_LDS = 2 * MAX_NLEVSOI;
constexpr int SOIL_STRIDE = 64;

// Fills P's soil members; lds is the lane's column of a one-wave block's
// [SOIL_LDS][SOIL_STRIDE] array.  The loads of all layers are in flight at once.
// Read from HBM layer by layer instead, as the sums of every Newton pass need
// them, they were what a pass waited for.
__device__ __forceinline__ void stage_soil(Leaf &P, const double *__restrict__ k, long sk,
                                           const double *__restrict__ smp, const double *__restrict__ z, long ss, int n,
                                           double *lds, const double *lt)
{
    P.k = lds;
    P.g = lds + MAX_NLEVSOI * SOIL_STRIDE;
    P.lt = lt;
    P.smp = smp;
    P.ss = ss;
    P.n = n;
    double kj[MAX_NLEVSOI], gj[MAX_NLEVSOI], wj[MAX_NLEVSOI];
#pragma unroll
    for (int j = 0; j < MAX_NLEVSOI; ++j) {
        const int i = j < n ? j : n - 1;
        kj[j] = k[i * sk];
        gj[j] = 1000.0 * z[i * ss];
        wj[j] = smp[i * ss];
    }
    double a = 0.0, b = 0.0, c = 0.0, d = 0.0;
#pragma unroll
    for (int j = 0; j < MAX_NLEVSOI; ++j) {
        lds[j * SOIL_STRIDE] = kj[j];
        lds[(MAX_NLEVSOI + j) * SOIL_STRIDE] = gj[j];
        if (j >= n) continue;
        a = a + kj[j];
        b = b + kj[j] * wj[j];
        c = c + (wj[j] - gj[j]);
        d = d + kj[j] * (wj[j] - gj[j]);
    }
    P.sum_k = a;
    P.sum_ks = b;
    P.sum_w = c;
    P.sum_kw = d;
}

// The four segments' vulnerability curves at x: u = (x/psi50)**ck, w = 2**-u,
// v = plc (w cut to zero below 0.005); d1plc's value from the same powers.  One
// Newton pass needs each curve and its slope; evaluated through plc and d1plc in
// spacF and spacA apart, it took 28 powers instead of 8.
struct Curves {
    double u[4], w[4], v[4];
};
__device__ __forceinline__ void curves(const Leaf &P, const double *x, Curves &C)
{
#pragma unroll
    for (int k = 0; k < 4; ++k) C.u[k] = cm_pow_tab(x[k] / P.psi50[k], P.ck[k], P.lt);
#pragma unroll
    for (int k = 0; k < 4; ++k) C.w[k] = cm_pow(2.0, -C.u[k]);
#pragma unroll
    for (int k = 0; k < 4; ++k) C.v[k] = C.w[k] < 0.005 ? 0.0 : C.w[k];
}
// d1plc
__device__ __forceinline__ double slope(const Leaf &P, const Curves &C, const double *x, int k)
{
    return -P.ck[k] * LN2 * C.w[k] * C.u[k] / x[k];
}

// getqflx (:5080-5164)
__device__ void getqflx(const Leaf &P, double qsatl, double qaf, bool havegs, double &gs_sun, double &gs_sha,
                        double &q_sun, double &q_sha)
{
    const double cf = P.pbot / (RGAS * 1.e-3 * P.thm) * 1.e6;
    const double wtl = (P.elai + P.esai) * P.gb;
    const double efpot = P.rho * wtl * (qsatl - qaf);
    if (havegs) {
        if (efpot > 0.0 && P.elai > 0.0) {
            if (gs_sun > 0.0) {
                const double rpp = P.fdry / P.gb * (P.laisun / (1.0 / P.gb + 1.0 / gs_sun)) / P.elai;
                q_sun = efpot * rpp / cf;
            } else {
                q_sun = 0.0;
            }
            if (gs_sha > 0.0) {
                const double rpp = P.fdry / P.gb * (P.laisha / (1.0 / P.gb + 1.0 / gs_sha)) / P.elai;
                q_sha = efpot * rpp / cf;
            } else {
                q_sha = 0.0;
            }
        } else {
            q_sun = 0.0;
            q_sha = 0.0;
        }
    } else {
        gs_sun = (q_sun > 0.0) ? P.gb * q_sun * cf * P.elai / (efpot * P.fdry * P.laisun - q_sun * cf * P.elai) : 0.0;
        gs_sha = (q_sha > 0.0) ? P.gb * q_sha * cf * P.elai / (efpot * P.fdry * P.laisha - q_sha * cf * P.elai) : 0.0;
    }
}

// the root's layer sum of spacF: k (x + 1000 z)
__device__ __forceinline__ double root_sum(const Leaf &P, double x)
{
    double s = 0.0;
    if (P.n == MAX_NLEVSOI) {
#pragma unroll
        for (int j = 0; j < MAX_NLEVSOI; ++j) s = s + P.k[j * SOIL_STRIDE] * (x + P.g[j * SOIL_STRIDE]);
    } else {
        for (int j = 0; j < P.n; ++j) s = s + P.k[j * SOIL_STRIDE] * (x + P.g[j * SOIL_STRIDE]);
    }
    return s;
}

// spacF (:4898-4976)
__device__ __forceinline__ void spacF(const Leaf &P, const Curves &C, const double *x, double *f, double q_sun,
                                      double q_sha)
{
    const double grav1 = P.htop * 1000.0;
    const double fsto1 = C.v[0], fsto2 = C.v[1], fx = C.v[2], fr = C.v[3];
    f[0] = q_sun * fsto1 - P.laisun * P.kmax[0] * fx * (x[2] - x[0]);
    f[1] = q_sha * fsto2 - P.laisha * P.kmax[1] * fx * (x[2] - x[1]);
    f[2] = P.laisun * P.kmax[0] * fx * (x[2] - x[0]) + P.laisha * P.kmax[1] * fx * (x[2] - x[1])
           - P.tsai * P.kmax[2] / P.htop * fr * (x[3] - x[2] - grav1);
    f[3] = P.tsai * P.kmax[2] / P.htop * fr * (x[3] - x[2] - grav1) + root_sum(P, x[3]) - P.sum_ks;
    if (P.laisha < TOL_LAI) {
        const double t = f[0];
        f[0] = f[1];
        f[1] = t;
    }
}

// spacA (:4715-4893); invA row-major; returns true when not invertible
__device__ __forceinline__ bool spacA(const Leaf &P, const Curves &C, const double *x, double *iA, double q_sun,
                                      double q_sha)
{
    double A[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) { A[i] = 0.0; iA[i] = 0.0; }
#define AA(i, j) A[((i) - 1) * 4 + (j) - 1]
#define IA(i, j) iA[((i) - 1) * 4 + (j) - 1]
    const double grav1 = P.htop * 1000.0;
    const double fx = C.v[2], fr = C.v[3];
    const double dfsto1 = slope(P, C, x, 0), dfsto2 = slope(P, C, x, 1);
    const double dfx = slope(P, C, x, 2), dfr = slope(P, C, x, 3);
    const double ks = P.kmax[0], kh = P.kmax[1], kx = P.kmax[2];
    AA(1, 1) = -(P.laisun * ks * fx) - q_sun * dfsto1;
    AA(1, 3) = P.laisun * ks * dfx * (x[2] - x[0]) + P.laisun * ks * fx;
    AA(2, 2) = -(P.laisha * kh * fx) - q_sha * dfsto2;
    AA(2, 3) = P.laisha * kh * dfx * (x[2] - x[1]) + P.laisha * kh * fx;
    AA(3, 1) = P.laisun * ks * fx;
    AA(3, 2) = P.laisha * kh * fx;
    AA(3, 3) = -(P.laisun * ks * dfx * (x[2] - x[0])) - P.laisun * ks * fx - P.laisha * kh * dfx * (x[2] - x[1])
               - P.laisha * kh * fx - P.tsai * kx / P.htop * fr;
    AA(3, 4) = P.tsai * kx / P.htop * dfr * (x[3] - x[2] - grav1) + P.tsai * kx / P.htop * fr;
    AA(4, 3) = P.tsai * kx / P.htop * fr;
    AA(4, 4) = -(P.tsai * kx / P.htop * fr) - P.tsai * kx / P.htop * dfr * (x[3] - x[2] - grav1) - P.sum_k;
    if (P.laisun > TOL_LAI && P.laisha > TOL_LAI) {
        const double determ = AA(4, 4) * AA(2, 2) * AA(3, 3) * AA(1, 1) - AA(4, 4) * AA(2, 2) * AA(3, 1) * AA(1, 3)
                              - AA(4, 4) * AA(3, 2) * AA(2, 3) * AA(1, 1) - AA(4, 3) * AA(1, 1) * AA(2, 2) * AA(3, 4);
        if (fabs(determ) <= 1.e-50) return true;
        const double ld = 1.0 / determ;
        IA(1, 1) = ld * AA(4, 4) * AA(2, 2) * AA(3, 3) - ld * AA(4, 4) * AA(3, 2) * AA(2, 3)
                   - ld * AA(4, 3) * AA(2, 2) * AA(3, 4);
        IA(2, 1) = ld * AA(2, 3) * AA(4, 4) * AA(3, 1);
        IA(3, 1) = -ld * AA(4, 4) * AA(2, 2) * AA(3, 1);
        IA(4, 1) = ld * AA(4, 3) * AA(2, 2) * AA(3, 1);
        IA(1, 2) = ld * AA(1, 3) * AA(4, 4) * AA(3, 2);
        IA(2, 2) = ld * AA(4, 4) * AA(3, 3) * AA(1, 1) - ld * AA(4, 4) * AA(3, 1) * AA(1, 3)
                   - ld * AA(4, 3) * AA(1, 1) * AA(3, 4);
        IA(3, 2) = -ld * AA(1, 1) * AA(4, 4) * AA(3, 2);
        IA(4, 2) = ld * AA(4, 3) * AA(1, 1) * AA(3, 2);
        IA(1, 3) = -ld * AA(1, 3) * AA(2, 2) * AA(4, 4);
        IA(2, 3) = -ld * AA(2, 3) * AA(1, 1) * AA(4, 4);
        IA(3, 3) = ld * AA(2, 2) * AA(1, 1) * AA(4, 4);
        IA(4, 3) = -ld * AA(4, 3) * AA(1, 1) * AA(2, 2);
        IA(1, 4) = ld * AA(1, 3) * AA(3, 4) * AA(2, 2);
        IA(2, 4) = ld * AA(2, 3) * AA(3, 4) * AA(1, 1);
        IA(3, 4) = -ld * AA(3, 4) * AA(1, 1) * AA(2, 2);
        IA(4, 4) = ld * AA(2, 2) * AA(3, 3) * AA(1, 1) - ld * AA(2, 2) * AA(3, 1) * AA(1, 3)
                   - ld * AA(3, 2) * AA(2, 3) * AA(1, 1);
    } else {
        if (P.laisha <= TOL_LAI) {
            AA(2, 2) = AA(1, 1);
            AA(3, 2) = AA(3, 1);
            AA(2, 3) = AA(1, 3);
        }
        const double determ = AA(2, 2) * AA(3, 3) * AA(4, 4) - AA(3, 4) * AA(2, 2) * AA(4, 3)
                              - AA(2, 3) * AA(3, 2) * AA(4, 4);
        if (fabs(determ) <= 1.e-50) return true;
        IA(2, 2) = AA(3, 3) * AA(4, 4) - AA(3, 4) * AA(4, 3);
        IA(2, 3) = -AA(2, 3) * AA(4, 4);
        IA(2, 4) = AA(3, 4) * AA(2, 3);
        IA(3, 2) = -AA(3, 2) * AA(4, 4);
        IA(3, 3) = AA(2, 2) * AA(4, 4);
        IA(3, 4) = -AA(3, 4) * AA(2, 2);
        IA(4, 2) = AA(3, 2) * AA(4, 3);
        IA(4, 3) = -AA(2, 2) * AA(4, 3);
        IA(4, 4) = AA(2, 2) * AA(3, 3) - AA(2, 3) * AA(3, 2);
        const double r = 1.0 / determ;
#pragma unroll
        for (int i = 0; i < 16; ++i) iA[i] = r * iA[i];
    }
#undef AA
#undef IA
    return false;
}

// getvegwp (:4979-5077); returns soilflux
__device__ double getvegwp(const Leaf &P, double *x, double gs_sun, double gs_sha, double qsatl, double qaf)
{
    const double grav1 = 1000.0 * P.htop;
    double q_sun, q_sha;
    getqflx(P, qsatl, qaf, true, gs_sun, gs_sha, q_sun, q_sha);
    if (fabs(P.sum_k) == 0.0) x[3] = P.sum_w / P.n;
    else x[3] = (P.sum_kw - q_sun - q_sha) / P.sum_k;
    const double fr = plc(x[3], P.psi50[3], P.ck[3], P.lt);
    if (P.tsai > 0.0 && fr > 0.0)
        x[2] = x[3] - grav1 - (q_sun + q_sha) / (fr * P.kmax[3] / P.htop * P.tsai);
    else
        x[2] = x[3] - grav1;
    const double fx = plc(x[2], P.psi50[2], P.ck[2], P.lt);
    x[1] = (P.laisha > 0.0 && fx > 0.0) ? x[2] - (q_sha / (fx * P.kmax[2] * P.laisha)) : x[2];
    x[0] = (P.laisun > 0.0 && fx > 0.0) ? x[2] - (q_sun / (fx * P.kmax[2] * P.laisun)) : x[2];
    double w[MAX_NLEVSOI];
#pragma unroll
    for (int j = 0; j < MAX_NLEVSOI; ++j) w[j] = P.smp[(j < P.n ? j : P.n - 1) * P.ss];
    double soilflux = 0.0;
#pragma unroll
    for (int j = 0; j < MAX_NLEVSOI; ++j)
        if (j < P.n) soilflux = soilflux + P.k[j * SOIL_STRIDE] * (w[j] - x[3] - P.g[j * SOIL_STRIDE]);
    return soilflux;
}


// calcstress for one patch: x (4) inout, bsun / bsha out; returns true where
// the call took the night branch (a positive x(sun) on entry), tran then
// holding its transpiration.  Used by the calcstress kernel and by
// PhotosynthesisHydraulicStress inside the CanopyFluxes iteration.
__device__ __forceinline__ bool calcstress(const Leaf &P, double *x, double gs_sun_in, double gs_sha_in, double qsatl,
                                           double qaf, double &bsun, double &bsha, double &tran)
{
    const bool night = x[0] > 0.0;
    if (night) x[0] = x[1];
    double gs0sun = gs_sun_in, gs0sha = gs_sha_in;
    double q_sun, q_sha;
    getqflx(P, qsatl, qaf, true, gs0sun, gs0sha, q_sun, q_sha);
    bool flag;
    if ((P.laisun > TOL_LAI || P.laisha > TOL_LAI) && (q_sun > 0.0 || q_sha > 0.0)) {
        int iter = 0;
        for (;;) {   // at most 51 passes: the iter > itmax exit
            iter = iter + 1;
            double f[4], iA[16], dx[4];
            Curves C;
            curves(P, x, C);
            spacF(P, C, x, f, q_sun, q_sha);
            double ff = 0.0;
#pragma unroll
            for (int k = 0; k < 4; ++k) ff = ff + f[k] * f[k];
            if (sqrt(ff) < 1.e-6 * (q_sun + q_sha)) { flag = false; break; }
            if (iter > 50) { flag = false; break; }
            flag = spacA(P, C, x, iA, q_sun, q_sha);
            if (flag) break;
            if (P.laisun > TOL_LAI && P.laisha > TOL_LAI) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    double s = 0.0;
#pragma unroll
                    for (int k = 0; k < 4; ++k) s = s + iA[r * 4 + k] * f[k];
                    dx[r] = s;
                }
            } else {
                dx[0] = 0.0;
#pragma unroll
                for (int r = 1; r < 4; ++r) {
                    double s = 0.0;
#pragma unroll
                    for (int k = 1; k < 4; ++k) s = s + iA[r * 4 + k] * f[k];
                    dx[r] = s;
                }
            }
            double m = fabs(dx[0]);
#pragma unroll
            for (int k = 1; k < 4; ++k) if (fabs(dx[k]) > m) m = fabs(dx[k]);
            if (m > 50000.0) {
#pragma unroll
                for (int k = 0; k < 4; ++k) dx[k] = 50000.0 * dx[k] / m;
            }
            if (P.laisun > TOL_LAI && P.laisha > TOL_LAI) {
#pragma unroll
                for (int k = 0; k < 4; ++k) x[k] = x[k] + dx[k];
            } else if (P.laisha > TOL_LAI) {
#pragma unroll
                for (int k = 0; k < 4; ++k) x[k] = x[k] + dx[k];
                x[0] = x[2];
            } else {
                x[2] = x[2] + dx[2];
                x[3] = x[3] + dx[3];
                x[0] = x[0] + dx[1];
                x[1] = x[2];
            }
            double dd = 0.0;
#pragma unroll
            for (int k = 0; k < 4; ++k) dd = dd + dx[k] * dx[k];
            if (sqrt(dd) < 1.e-9) break;
            if (x[2] > x[3]) x[2] = x[3];
            if (x[0] > x[2]) x[0] = x[2];
            if (x[1] > x[2]) x[1] = x[2];
        }
    } else {
        flag = true;
    }
    if (flag) {
        (void)getvegwp(P, x, gs0sun, gs0sha, qsatl, qaf);
        bsun = plc(x[0], P.psi50[0], P.ck[0], P.lt);
        bsha = plc(x[1], P.psi50[1], P.ck[1], P.lt);
    } else {
        double qs = q_sun * plc(x[0], P.psi50[0], P.ck[0], P.lt);
        double qh = q_sha * plc(x[1], P.psi50[1], P.ck[1], P.lt);
        getqflx(P, qsatl, qaf, false, gs0sun, gs0sha, qs, qh);
        bsun = (q_sun > 0.0) ? gs0sun / gs_sun_in : plc(x[0], P.psi50[0], P.ck[0], P.lt);
        bsha = (q_sha > 0.0) ? gs0sha / gs_sha_in : plc(x[1], P.psi50[1], P.ck[1], P.lt);
    }
    if (bsun < 0.01) bsun = 0.0;
    if (bsha < 0.01) bsha = 0.0;
    if (night) {
        gs0sun = bsun * gs_sun_in;
        gs0sha = bsha * gs_sha_in;
        double soilflux = getvegwp(P, x, gs0sun, gs0sha, qsatl, qaf);
        if (soilflux < 0.0) soilflux = 0.0;
        tran = soilflux;
    }
    return night;
}

}  // namespace phs
}  // namespace ctsm
