// canopy.hip -- CanopyFluxes (CanopyFluxesMod.F90:191-1765) for gfx950, a lane
// per patch: the set-up (root stress, roughness, Monin-Obukhov initialisation),
// rounds of the Newton / stability iteration with sun and shade photosynthesis and
// its state in registers, the post-iteration fluxes.
//
// Callees restated here: FrictionVelocity / StabilityFunc1/2 / MoninObukIni
// (FrictionVelocityMod.F90:754-1209), QSat (QSatMod.F90:61-127),
// Photosynthesis / hybrid / brent / ci_func (PhotosynthesisMod.F90:1243-2701),
// quadratic (quadraticMod.F90:17-74), calc_effective_soilporosity /
// calc_volumetric_h2oliq / calc_root_moist_stress_clm45default
// (SoilMoistStressMod.F90:70-215, 312-514), PhotosynthesisTotal
// (PhotosynthesisMod.F90:2065-2151), truncate_small_values (NumericsMod.F90:
// 60-100); plus the transpiration p2c and sink (clm_driver.F90:1714-1716,
// SoilWaterPlantSinkMod.F90:332-424) in k_root_sink.
//
// Patches are independent, so the reference's shrinking filter of
// unconverged patches becomes a per-lane loop exit; the operation sequence of
// each patch is the reference's.  Leaf-temperature factors of Photosynthesis
// (ft, fth, 2**x) depend on t_veg only, so they are evaluated once per
// iteration and shared by the sun and shade phases (the same values the
// reference computes twice).
#include <algorithm>
#include <climits>
#include <type_traits>

#include "common.h"
#include "phs_dev.h"
#include "trace.h"

namespace ctsm {
namespace canopy {

constexpr double VKC = 0.4;
constexpr double CPAIR = 1.00464e3;
constexpr double HVAP = 2.501e6;
constexpr double CWATER = 4.188e3;
constexpr double RGAS = 6.02214e26 * 1.38065e-23;
constexpr double PI = 3.14159265358979323846;
constexpr double SPVAL = 1.e36;
constexpr double TLSAI_CRIT = 2.0;
constexpr double ALPHA_AERO = 1.0;
constexpr double NU = 1.5e-5;
constexpr double CD1 = 7.5;
constexpr double CDRYBIO = 1400.0;
constexpr double C_TO_B = 2.0;
constexpr double MAX_CS = 1.e-06;
constexpr int ENDRUN = CTSM_E_ENDRUN;
// the Meier2022 fixed point u = a exp(u) converges or overflows to NaN
// within a few hundred steps for finite input; the cap only bounds a wave
constexpr int MAX_FIXED_POINT = 100000;

// PFT table field indices (rows of the device table, CTSM_MAX_PFT each)
enum {
    F_DLEAF, F_C3PSN, F_SLATOP, F_LEAFCN, F_FLNR, F_FNITR, F_MBBOPT, F_MEDSLOPE, F_MEDINT, F_SMPSO, F_SMPSC,
    F_THETA_CJ, F_Z0V_CR, F_Z0V_CS, F_Z0V_C, F_Z0V_CW, F_Z0V_LAIMAX, F_IS_TREE, F_IS_SHRUB, F_DBH, F_FBW,
    F_NSTEM, F_RSTEM, F_WOOD, N_PFT_FIELDS
};

struct CView {
    int begc, ldc, begp, ldp, begg, ldg, nlevsno, nlevsoi, nlevgrnd;
    __device__ __forceinline__ long c1(int c) const { return (long)(c - begc); }
    __device__ __forceinline__ long g1(int g) const { return (long)(g - begg); }
    __device__ __forceinline__ long p1(int p) const { return (long)(p - begp); }
    __device__ __forceinline__ long sno(int c, int j) const { return (long)(c - begc) + (long)(j + nlevsno - 1) * ldc; }
    __device__ __forceinline__ long soi(int c, int j) const { return (long)(c - begc) + (long)(j - 1) * ldc; }
    __device__ __forceinline__ long soip(int p, int j) const { return (long)(p - begp) + (long)(j - 1) * ldp; }
};

struct CSwitch {
    int z0param, stomatal, soil_resis, biomass, undercanopy, light_inhibit, itmax;
};

__device__ __forceinline__ double p4(double x) { const double x2 = x * x; return x2 * x2; }
__device__ __forceinline__ double p3(double x) { return (x * x) * x; }

// QSatMod.F90:61-127
__device__ __forceinline__ void qsat(double T, double p, double &qs, double &es, double &qsdT)
{
    const double td = fmin90(100.0, fmax90(-75.0, T - TFRZ));
    double e, d;
    if (td >= 0.0) {
        e = 6.11213476 + td * (0.444007856 + td * (0.143064234e-01 + td * (0.264461437e-03 + td * (0.305903558e-05
            + td * (0.196237241e-07 + td * (0.892344772e-10 + td * (-0.373208410e-12 + td * 0.209339997e-15)))))));
        d = 0.444017302 + td * (0.286064092e-01 + td * (0.794683137e-03 + td * (0.121211669e-04 + td * (0.103354611e-06
            + td * (0.404125005e-09 + td * (-0.788037859e-12 + td * (-0.114596802e-13 + td * 0.381294516e-16)))))));
    } else {
        e = 6.11123516 + td * (0.503109514 + td * (0.188369801e-01 + td * (0.420547422e-03 + td * (0.614396778e-05
            + td * (0.602780717e-07 + td * (0.387940929e-09 + td * (0.149436277e-11 + td * 0.262655803e-14)))))));
        d = 0.503277922 + td * (0.377289173e-01 + td * (0.126801703e-02 + td * (0.249468427e-04 + td * (0.313703411e-06
            + td * (0.257180651e-08 + td * (0.133268878e-10 + td * (0.394116744e-13 + td * 0.498070196e-16)))))));
    }
    es = e * 100.0;
    const double vp = 1.0 / (p - 0.378 * es);
    const double vp1 = 0.622 * vp;
    qs = es * vp1;
    const double esdT = d * 100.0;
    const double vp2 = vp1 * vp;
    qsdT = esdT * vp2 * p;
}

__device__ __forceinline__ double qsat_only(double T, double p, double &es)
{
    const double td = fmin90(100.0, fmax90(-75.0, T - TFRZ));
    double e;
    if (td >= 0.0)
        e = 6.11213476 + td * (0.444007856 + td * (0.143064234e-01 + td * (0.264461437e-03 + td * (0.305903558e-05
            + td * (0.196237241e-07 + td * (0.892344772e-10 + td * (-0.373208410e-12 + td * 0.209339997e-15)))))));
    else
        e = 6.11123516 + td * (0.503109514 + td * (0.188369801e-01 + td * (0.420547422e-03 + td * (0.614396778e-05
            + td * (0.602780717e-07 + td * (0.387940929e-09 + td * (0.149436277e-11 + td * 0.262655803e-14)))))));
    es = e * 100.0;
    const double vp = 1.0 / (p - 0.378 * es);
    return es * (0.622 * vp);
}

// quadraticMod.F90:17-74; false where the reference calls endrun
template <class DIV>     // the type of a as a denominator: double, or Recip
__device__ __forceinline__ bool quadratic(double a, const DIV &ra, double b, double c, double &r1, double &r2)
{
    if (a == 0.0) { r1 = r2 = 0.0; return false; }
    double root = b * b - 4.0 * a * c;
    bool ok = true;
    if (root < 0.0) {
        if (-root < 3.0 * 2.220446049250313e-16) root = 0.0;
        else { ok = false; root = 0.0; }
    }
    double q;
    if (b >= 0.0) q = -0.5 * (b + sqrt(root));
    else q = -0.5 * (b - sqrt(root));
    r1 = q / ra;
    r2 = (q != 0.0) ? c / q : 1.e36;
    return ok;
}
__device__ __forceinline__ bool quadratic(double a, double b, double c, double &r1, double &r2)
{
    return quadratic(a, a, b, c, r1, r2);
}

__device__ __forceinline__ double stab1(double zeta, const double *lt)
{
    const double chik2 = sqrt(1.0 - 16.0 * zeta);
    const double chik = sqrt(chik2);
    return 2.0 * cm_log_tab((1.0 + chik) * 0.5, lt) + cm_log_tab((1.0 + chik2) * 0.5, lt) - 2.0 * cm_atan(chik) + PI * 0.5;
}
__device__ __forceinline__ double stab2(double zeta, const double *lt)
{
    const double chik2 = sqrt(1.0 - 16.0 * zeta);
    return 2.0 * cm_log_tab((1.0 + chik2) * 0.5, lt);
}

// the temperature / humidity profile block repeated in FrictionVelocityMod.F90:916-1060;
// log_z = log(zldis / z0), which does not change over the canopy iteration.
// The lanes of a wave sit in different stability regimes; each elementary
// function a regime needs is evaluated once for all the lanes that need it
// (the very unstable and the very stable regime share the logarithm of
// their height ratio, the two unstable ones stab2(z0 / obu)) rather than once
// per regime branch.  Every lane computes its own regime's expression with
// the same operations in the same order.
// lt: log's table in LDS.
__device__ __forceinline__ double temp_profile(double zldis, double z0, const Recip &obu, double log_z, const double *lt)
{
    const double zetat = 0.465;
    const double zeta = zldis / obu;
    const bool ra = zeta < -zetat, rb = !ra && zeta < 0.0, rc = !ra && !rb && zeta <= 1.0, rd = !(ra || rb || rc);
    double lg = 0.0, sa = 0.0, sb = 0.0, pw = 0.0, lz = 0.0;
    if (ra || rd) lg = cm_log_tab(ra ? -zetat * obu.b / z0 : obu.b / z0, lt);
    if (ra || rb) sb = stab2(z0 / obu, lt);
    if (ra) {
        sa = stab2(-zetat, cm_log_table());
        pw = cm_pow(zetat, -0.333) - cm_pow_tab(-zeta, -0.333, lt);
    }
    if (rb) sa = stab2(zeta, lt);
    if (rd) lz = cm_log_tab(zeta, lt);
    double den;
    if (ra) den = lg - sa + sb + 0.8 * pw;
    else if (rb) den = log_z - sa + sb;
    else if (rc) den = log_z + 5.0 * zeta - 5.0 * z0 / obu;
    else den = lg + 5.0 - 5.0 * z0 / obu + (5.0 * lz + zeta - 1.0);
    return VKC / den;
}

__device__ __forceinline__ double fm_profile(double z, const double *lt)
{
    // dust-model fm of FrictionVelocityMod.F90:1072-1095 for z < 0
    const double tmp1 = cm_pow_tab(1.0 - 16.0 * z, 0.25, lt);
    const double tmp2 = cm_log_tab((1.0 + tmp1 * tmp1) / 2.0, lt);
    const double tmp3 = cm_log_tab((1.0 + tmp1) / 2.0, lt);
    return 2.0 * tmp3 + tmp2 - 2.0 * cm_atan(tmp1) + 1.5707963;
}

struct FV {
    double ustar, temp1, temp2, temp12m, temp22m, fm, u10, u10_clm, va, fv, vds;
};

// FrictionVelocityMod.F90:754-1117 (patch form), the part the canopy
// iteration consumes: ustar, the heat / moisture profile factors temp1 and
// temp2, and the running mean of the dust-model fm.  The heights above the
// displacement height (zldis, zht, zhq), the roughness length (one value for
// momentum, heat and moisture over vegetation) and the logarithms of height over
// it (lm: momentum, lh: heat) are the step's constants; the moisture height's is
// taken where it differs from the heat's.  The regimes' divides by obu share its
// reciprocal.
struct FVLogs {
    double lm, lh;
};
__device__ __forceinline__ void friction_velocity(double zldis, double zht, double zhq, double z0, const FVLogs &L,
                                                  double obu_, int iter, double um, FV &o, const double *lt)
{
    const double zetam = 1.574;
    const double z0m = z0, z0h = z0, z0q = z0;
    const Recip obu = recip(obu_);
    const double zeta = zldis / obu;
    // each elementary function once for the lanes whose regime needs it (as
    // in temp_profile)
    const bool ra = zeta < -zetam, rb = !ra && zeta < 0.0, rc = !ra && !rb && zeta <= 1.0, rd = !(ra || rb || rc);
    double lg = 0.0, sa = 0.0, sb = 0.0, pw = 0.0, lz = 0.0;
    if (ra || rd) lg = cm_log_tab(ra ? -zetam * obu_ / z0m : obu_ / z0m, lt);
    if (ra || rb) sb = stab1(z0m / obu, lt);
    if (ra) {
        sa = stab1(-zetam, cm_log_table());
        pw = cm_pow_tab(-zeta, 0.333, lt) - cm_pow(zetam, 0.333);
    }
    if (rb) sa = stab1(zeta, lt);
    if (rd) lz = cm_log_tab(zeta, lt);
    double den;
    if (ra) den = lg - sa + sb + 1.14 * pw;
    else if (rb) den = L.lm - sa + sb;
    else if (rc) den = L.lm + 5.0 * zeta - 5.0 * z0m / obu;
    else den = lg + 5.0 - 5.0 * z0m / obu + (5.0 * lz + zeta - 1.0);
    o.ustar = VKC * um / den;
    o.temp1 = temp_profile(zht, z0h, obu, L.lh, lt);
    if (zhq == zht) o.temp2 = o.temp1;
    else o.temp2 = temp_profile(zhq, z0q, obu, cm_log_tab(zhq / z0q, lt), lt);
    const double zm1 = fmin90(zeta, 1.0);
    const double fmnew = (zm1 < 0.0) ? fm_profile(zm1, lt) : -5.0 * zm1;
    o.fm = (iter == 1) ? fmnew : 0.5 * (o.fm + fmnew);
}

// The diagnostics FrictionVelocity computes beside them (deposition
// velocity, 10-m winds, 2-m profile factors).  Nothing in the iteration reads
// them, so they are evaluated once, from the inputs (obu, um) and the ustar
// and fm of the last iteration: the same values the reference keeps from its
// last call.
__device__ __forceinline__ void friction_velocity_diag(double hu, double displa, double z0m, double z0h, double z0q, double obu_,
                                       double ur, double um, FV &o, const double *lt)
{
    const double zetam = 1.574;
    const Recip obu = recip(obu_);
    const double zldis = hu - displa;
    const double zeta = zldis / obu;
    if (zeta < 0.0) o.vds = 2.e-3 * o.ustar * (1.0 + cm_pow_tab(300.0 / (-obu_), 0.666, lt));
    else o.vds = 2.e-3 * o.ustar;
    if (zldis - z0m <= 10.0) {
        o.u10_clm = um;
    } else {
        const double z10 = 10.0 + z0m;
        // one evaluation of each elementary function for the lanes whose
        // regime needs it (as in friction_velocity)
        const bool ra = zeta < -zetam, rb = !ra && zeta < 0.0, rc = !ra && !rb && zeta <= 1.0;
        const bool rd = !(ra || rb || rc);
        const double lg = cm_log_tab(ra ? -zetam * obu_ / z10 : (rd ? obu_ / z10 : zldis / z10), lt);
        double sa = 0.0, sb = 0.0, pw = 0.0, lz = 0.0;
        if (ra || rb) sb = stab1(z10 / obu, lt);
        if (ra) {
            sa = stab1(-zetam, cm_log_table());
            pw = cm_pow_tab(-zeta, 0.333, lt) - cm_pow(zetam, 0.333);
        }
        if (rb) sa = stab1(zeta, lt);
        if (rd) lz = cm_log_tab(zeta, lt);
        double t;
        if (ra) t = lg - sa + sb + 1.14 * pw;
        else if (rb) t = lg - sa + sb;
        else if (rc) t = lg + 5.0 * zeta - 5.0 * z10 / obu;
        else t = lg + 5.0 - 5.0 * z10 / obu + (5.0 * lz + zeta - 1.0);
        o.u10_clm = um - (o.ustar / VKC * t);
    }
    o.va = um;
    o.temp12m = temp_profile(2.0 + z0h, z0h, obu, cm_log_tab((2.0 + z0h) / z0h, lt), lt);
    if (z0q == z0h) o.temp22m = o.temp12m;
    else o.temp22m = temp_profile(2.0 + z0q, z0q, obu, cm_log_tab((2.0 + z0q) / z0q, lt), lt);
    double zeta10 = fmin90(10.0 / obu, 1.0);
    if (zeta == 0.0) zeta10 = 0.0;
    const double fm10 = (zeta10 < 0.0) ? fm_profile(zeta10, lt) : -5.0 * zeta10;
    const double tmp4 = cm_log_tab(fmax90(1.0, hu / 10.0), lt);
    o.u10 = ur - o.ustar / VKC * (tmp4 - o.fm + fm10);
    o.fv = o.ustar;
}

// the exponents of ft and fth (PhotosynthesisMod.F90:2488-2561): haq is
// ha / (rgas (tfrz + 25)), t25 = 1 - (tfrz + 25) / tl, rt the reciprocal of rgas tl
__device__ __forceinline__ double fth_arg(double tl, const Recip &rt, double hd, double se)
{
    return (-hd + se * tl) / rt;
}
__device__ __forceinline__ double fth25(double hd, double se)
{
    return 1.0 + cm_exp((-hd + se * (TFRZ + 25.0)) / (RGAS * 1.e-3 * (TFRZ + 25.0)));
}

// One ci solve: the constants of ci_func and the photosyns_inst values it writes.
struct CiSolve {
    bool c3, medlyn;
    double forc_pbot, cair, oair, gb_mol, je, lmr_z, par_z, rh_can;
    double vcmax_z, tpu_z, kp_z, cp, kc, ko, qe, bbb, mbb, theta_cj, theta_ip, mslope, mint;
    double ac, aj, ap, ag, an, gs_mol;
    Recip r_cj, r_ip, r_pbot, r_gbrh;   // of theta_cj, theta_ip, forc_pbot and Medlyn's gb_mol rh_can term
    bool bad;
};

// PhotosynthesisMod.F90:2564-2701
__device__ __forceinline__ double ci_func(double ci, CiSolve &s)
{
    double r1, r2;
    // the C3 Rubisco rate and the C4 PEP carboxylase rate are the one divide
    // of each pathway: a wave of both kinds takes it once, each lane on its
    // own pathway's operands
    const double q = (s.c3 ? s.vcmax_z * fmax90(ci - s.cp, 0.0) : s.kp_z * fmax90(ci, 0.0))
                     / (s.c3 ? ci + s.kc * (1.0 + s.oair / s.ko) : s.forc_pbot);
    if (s.c3) {
        s.ac = q;
        s.aj = s.je * fmax90(ci - s.cp, 0.0) / (4.0 * ci + 8.0 * s.cp);
        s.ap = 3.0 * s.tpu_z;
    } else {
        s.ac = s.vcmax_z;
        s.aj = s.qe * s.par_z * 4.6;
        s.ap = q;
    }
    if (!quadratic(s.theta_cj, s.r_cj, -(s.ac + s.aj), s.ac * s.aj, r1, r2)) s.bad = true;
    const double ai = fmin90(r1, r2);
    if (!quadratic(s.theta_ip, s.r_ip, -(ai + s.ap), ai * s.ap, r1, r2)) s.bad = true;
    s.ag = fmax90(0.0, fmin90(r1, r2));
    s.an = s.ag - s.lmr_z;
    if (s.an < 0.0) return 0.0;
    double cs = s.cair - 1.4 / s.gb_mol * s.an * s.forc_pbot;
    cs = fmax90(cs, MAX_CS);
    if (s.medlyn) {
        const double term = 1.6 * s.an / (cs / s.r_pbot * 1.e06);
        const double bq = -(2.0 * (s.mint * 1.e-06 + term)
                            + (s.mslope * term) * (s.mslope * term) / s.r_gbrh);
        const double cq = s.mint * s.mint * 1.e-12 + (2.0 * s.mint * 1.e-06 + term * (1.0 - s.mslope * s.mslope / s.rh_can)) * term;
        if (!quadratic(1.0, bq, cq, r1, r2)) s.bad = true;
        s.gs_mol = fmax90(r1, r2) * 1.e06;
    } else {
        const double bq = cs * (s.gb_mol - s.bbb) - s.mbb * s.an * s.forc_pbot;
        const double cq = -s.gb_mol * (cs * s.bbb + s.mbb * s.an * s.forc_pbot * s.rh_can);
        if (!quadratic(cs, bq, cq, r1, r2)) s.bad = true;
        s.gs_mol = fmax90(r1, r2);
    }
    return ci - s.cair + s.an * s.forc_pbot * (1.4 * s.gs_mol + 1.6 * s.gb_mol) / (s.gb_mol * s.gs_mol);
}

// hybrid (PhotosynthesisMod.F90:2251-2368) with its Brent fallback (brent,
// :2371-2485).  Nearly every solve takes the two starting points and one secant
// step and is done; one in sixteen, but one in most waves, goes on.  So the three
// evaluations of ci_func are straight-line code, and what follows is one loop
// with a single evaluation per pass: the stage a lane is in (a secant step, the
// Brent iteration, the re-evaluation at the best point) takes the last result and
// chooses the next point or ends, and lanes in different stages share the
// evaluation.  Each lane makes exactly the reference's sequence of evaluations and
// arithmetic (only the ci_func side effects matter to the caller).  As one loop
// over all the stages a pass spent as much on moving the lanes' state between the
// stages as on the evaluation.
__device__ __forceinline__ void hybrid(double x0, CiSolve &s)
{
    const double eps = 1.e-2, eps1 = 1.e-4;
    double f0 = ci_func(x0, s);
    if (f0 == 0.0) return;
    double minx = x0, minf = f0;
    double x1 = x0 * 0.99;
    double f1 = ci_func(x1, s);
    if (f1 == 0.0) return;
    if (f1 < minf) {
        minx = x1;
        minf = f1;
    }
    double dx = -f1 * (x1 - x0) / (f1 - f0);
    double x = x1 + dx;
    double tol = fabs(x) * eps;
    if (fabs(dx) < tol) return;
    x0 = x1;
    f0 = f1;
    x1 = x;
    double f = ci_func(x1, s);

    enum { SECANT, BRENT, LAST };
    int stage = SECANT, iter = 1, biter = 0;
    double a = 0.0, b = 0.0, c = 0.0, fa = 0.0, fb = 0.0, fc = 0.0, d = 0.0, e = 0.0;
    for (;;) {
        double xe;
        bool brent = false;
        if (stage == SECANT) {
            f1 = f;
            if (f1 < minf) {
                minx = x1;
                minf = f1;
            }
            if (fabs(f1) <= eps1) return;
            if (f1 * f0 < 0.0) {
                // brent(x0, x1, f0, f1, tol): the bracket, the signs opposite
                a = x0;
                b = x1;
                fa = f0;
                fb = f1;
                c = b;
                fc = fb;
                brent = true;
            } else if (iter > 40) {
                xe = minx;
                stage = LAST;
            } else {
                ++iter;
                dx = -f1 * (x1 - x0) / (f1 - f0);
                x = x1 + dx;
                tol = fabs(x) * eps;
                if (fabs(dx) < tol) return;
                x0 = x1;
                f0 = f1;
                x1 = x;
                xe = x1;
            }
        } else if (stage == BRENT) {
            fb = f;
            if (fb == 0.0) return;
            ++biter;
            brent = true;
        } else {
            return;     // LAST: ci_func at the best point has run
        }
        if (brent) {
            // one Brent iteration up to its evaluation of ci_func
            if (biter >= 20) return;
            if ((fb > 0.0 && fc > 0.0) || (fb < 0.0 && fc < 0.0)) {
                c = a;
                fc = fa;
                d = b - a;
                e = d;
            }
            if (fabs(fc) < fabs(fb)) {
                a = b;
                b = c;
                c = a;
                fa = fb;
                fb = fc;
                fc = fa;
            }
            const double tol1 = 2.0 * eps * fabs(b) + 0.5 * tol;
            const double xm = 0.5 * (c - b);
            if (fabs(xm) <= tol1 || fb == 0.0) return;
            if (fabs(e) >= tol1 && fabs(fa) > fabs(fb)) {
                const double ss = fb / fa;
                double p, q;
                if (a == c) {
                    p = 2.0 * xm * ss;
                    q = 1.0 - ss;
                } else {
                    q = fa / fc;
                    const double r = fb / fc;
                    p = ss * (2.0 * xm * q * (q - r) - (b - a) * (r - 1.0));
                    q = (q - 1.0) * (r - 1.0) * (ss - 1.0);
                }
                if (p > 0.0) q = -q;
                p = fabs(p);
                if (2.0 * p < fmin90(3.0 * xm * q - fabs(tol1 * q), fabs(e * q))) {
                    e = d;
                    d = p / q;
                } else {
                    d = xm;
                    e = d;
                }
            } else {
                d = xm;
                e = d;
            }
            a = b;
            fa = fb;
            if (fabs(d) > tol1) b = b + d;
            else b = b + copysign(fabs(tol1), xm);
            xe = b;
            stage = BRENT;
        }
        f = ci_func(xe, s);
    }
}

// per-phase outputs of Photosynthesis
struct Phase {
    double rs, rs_z, ci_z, lmr, lmr_z, psn, psn_z, psn_wc, psn_wj, psn_wp, gs_ph, gs_ln;
};
// photosyns_inst values shared by the phases (last writer wins, as in the reference)
struct Shared {
    double vcmax_z, tpu_z, kp_z, gb_mol, ac, aj, ap, ag, an, gs_mol, rh_leaf, vpd_can;
};
// leaf-temperature factors of one iteration (each a value the reference
// computes inside Photosynthesis; products keep the reference's order)
struct TFac {
    double kc, ko, cp;
    double ftL, fthL, dL4;          // lmr: c3 ft*fth, c4 divisor
    double ftV, fthV, dV1, dV2;     // vcmax: c3 ft*fth, c4 divisors
    double ftJ, fthJ, ftT, fthT;    // jmax, tpu
    double pow2;                    // 2**((t_veg - (tfrz+25))/10)
};
// constants of the step for one patch
struct PsnConst {
    bool c3;
    double bbb, mbb, qe, lnc, vcmax25top, jmax25top, tpu25top, kp25top, lmr25top;
    double t10c, vcmaxse, jmaxse, tpuse, vcmaxc, jmaxc, tpuc, kc25, ko25, cp25;
    double theta_cj, mslope, mint;
};

// Element `byte` bytes into an array, as a base in scalar registers and a 32-bit
// offset (a patch or column array without levels is far below 4 GiB: the state of
// 2^29 patches would not fit the card).
template <class T>
__device__ __forceinline__ T &at(T *base, uint32_t byte)
{
    return *(T *)((char *)base + byte);
}

// PhotosynthesisMod.F90:1243-2062 for one patch and one phase.
template <class PRM>
__device__ __forceinline__ void photosynthesis(const CSwitch &sw, const PRM &P, const PsnConst &K, const TFac &T,
                               int nrad, double par_z, const double *lai_z_p, const double *vcmaxcint,
                               const double *o3v, const double *o3g, uint32_t po, bool noon, double forc_pbot, double tgcm, double esat_tv, double eair, double oair,
                               double cair, double rb, double btran, Phase &ph, Shared &sh, bool &bad)
{
    const bool medlyn = sw.stomatal == CTSM_STOMATA_MEDLYN2011;
    double jmax_z = 0.0;
    if (nrad >= 1) {
        const double nscaler = at(vcmaxcint, po);
        const double lmr25 = K.lmr25top * nscaler;
        if (K.c3) {
            ph.lmr_z = lmr25 * T.ftL * T.fthL;
        } else {
            ph.lmr_z = lmr25 * T.pow2;
            ph.lmr_z = ph.lmr_z / T.dL4;
        }
        if (par_z <= 0.0) {
            sh.vcmax_z = 0.0;
            jmax_z = 0.0;
            sh.tpu_z = 0.0;
            sh.kp_z = 0.0;
        } else {
            const double vcmax25 = K.vcmax25top * nscaler;
            const double jmax25 = K.jmax25top * nscaler;
            const double tpu25 = K.tpu25top * nscaler;
            const double kp25 = K.kp25top * nscaler;
            sh.vcmax_z = vcmax25 * T.ftV * T.fthV;
            jmax_z = jmax25 * T.ftJ * T.fthJ;
            sh.tpu_z = tpu25 * T.ftT * T.fthT;
            if (!K.c3) {
                sh.vcmax_z = vcmax25 * T.pow2;
                sh.vcmax_z = sh.vcmax_z / T.dV1;
                sh.vcmax_z = sh.vcmax_z / T.dV2;
            }
            sh.kp_z = kp25 * T.pow2;
        }
        sh.vcmax_z = sh.vcmax_z * btran;
        ph.lmr_z = ph.lmr_z * btran;
        if (sw.light_inhibit && par_z > 0.0) ph.lmr_z = ph.lmr_z * 0.67;
    }
    const double rsmax0 = 2.e4;
    const double cf = forc_pbot / (RGAS * 1.e-3 * tgcm) * 1.e06;
    const double gb = 1.0 / rb;
    sh.gb_mol = gb * cf;
    double psn_wc_z = 0.0, psn_wj_z = 0.0, psn_wp_z = 0.0;
    if (nrad >= 1) {
        if (par_z <= 0.0) {
            sh.ac = 0.0;
            sh.aj = 0.0;
            sh.ap = 0.0;
            sh.ag = 0.0;
            sh.an = sh.ag - ph.lmr_z;
            ph.psn_z = 0.0;
            if (!medlyn) ph.rs_z = fmin90(rsmax0, 1.0 / K.bbb * cf);
            else ph.rs_z = fmin90(rsmax0, 1.0 / K.mint * cf);
            ph.ci_z = 0.0;
            sh.rh_leaf = 0.0;
            ph.gs_ph = cf / ph.rs_z;
        } else {
            const double ceair = fmin90(eair, esat_tv);
            double rh_can;
            if (!medlyn) {
                rh_can = ceair / esat_tv;
            } else {
                rh_can = fmax90(esat_tv - ceair, 50.0) * 0.001;
                sh.vpd_can = rh_can;
            }
            const double qabs = 0.5 * (1.0 - P.fnps) * par_z * 4.6;
            double r1, r2;
            if (!quadratic(P.theta_psii, -(qabs + jmax_z), qabs * jmax_z, r1, r2)) bad = true;
            const double je = fmin90(r1, r2);
            const double ci0 = K.c3 ? 0.7 * cair : 0.4 * cair;
            CiSolve s;
            s.c3 = K.c3;
            s.medlyn = medlyn;
            s.forc_pbot = forc_pbot;
            s.cair = cair;
            s.oair = oair;
            s.gb_mol = sh.gb_mol;
            s.je = je;
            s.lmr_z = ph.lmr_z;
            s.par_z = par_z;
            s.rh_can = rh_can;
            s.vcmax_z = sh.vcmax_z;
            s.tpu_z = sh.tpu_z;
            s.kp_z = sh.kp_z;
            s.cp = T.cp;
            s.kc = T.kc;
            s.ko = T.ko;
            s.qe = K.qe;
            s.bbb = K.bbb;
            s.mbb = K.mbb;
            s.theta_cj = K.theta_cj;
            s.theta_ip = P.theta_ip;
            s.mslope = K.mslope;
            s.mint = K.mint;
            s.ac = sh.ac;
            s.aj = sh.aj;
            s.ap = sh.ap;
            s.ag = sh.ag;
            s.an = sh.an;
            s.gs_mol = sh.gs_mol;
            s.r_cj = recip(s.theta_cj);
            s.r_ip = recip(s.theta_ip);
            s.r_pbot = recip(forc_pbot);
            s.r_gbrh = recip(s.gb_mol * 1.e-06 * rh_can);
            s.bad = false;
            hybrid(ci0, s);
            if (s.bad) bad = true;
            sh.ac = s.ac;
            sh.aj = s.aj;
            sh.ap = s.ap;
            sh.ag = s.ag;
            sh.an = s.an;
            sh.gs_mol = s.gs_mol;
            if (sh.an < 0.0) sh.gs_mol = medlyn ? K.mint : K.bbb;
            const double gs_mol = sh.gs_mol;
            ph.gs_ph = gs_mol;
            ph.gs_ln = noon ? gs_mol : SPVAL;
            const double an = sh.an;
            ph.ci_z = cair - an * forc_pbot * (1.4 * gs_mol + 1.6 * sh.gb_mol) / (sh.gb_mol * gs_mol);
            ph.ci_z = fmax90(ph.ci_z, 1.e-06);
            const double gs = gs_mol / cf;
            ph.rs_z = fmin90(1.0 / gs, rsmax0);
            ph.rs_z = ph.rs_z / at(o3g, po);
            ph.psn_z = sh.ag;
            ph.psn_z = ph.psn_z * at(o3v, po);
            if (sh.ac <= sh.aj && sh.ac <= sh.ap) psn_wc_z = ph.psn_z;
            else if (sh.aj < sh.ac && sh.aj <= sh.ap) psn_wj_z = ph.psn_z;
            else if (sh.ap < sh.ac && sh.ap < sh.aj) psn_wp_z = ph.psn_z;
            if (gs_mol < 0.0) bad = true;
            if (!medlyn) sh.rh_leaf = (sh.gb_mol * ceair + gs_mol * esat_tv) / ((sh.gb_mol + gs_mol) * esat_tv);
        }
    }
    double psncan = 0.0, psncan_wc = 0.0, psncan_wj = 0.0, psncan_wp = 0.0, lmrcan = 0.0, gscan = 0.0, laican = 0.0;
    if (nrad >= 1) {
        const double lai_z = at(lai_z_p, po);
        psncan = psncan + ph.psn_z * lai_z;
        psncan_wc = psncan_wc + psn_wc_z * lai_z;
        psncan_wj = psncan_wj + psn_wj_z * lai_z;
        psncan_wp = psncan_wp + psn_wp_z * lai_z;
        lmrcan = lmrcan + ph.lmr_z * lai_z;
        gscan = gscan + lai_z / (rb + ph.rs_z);
        laican = laican + lai_z;
    }
    if (laican > 0.0) {
        ph.psn = psncan / laican;
        ph.psn_wc = psncan_wc / laican;
        ph.psn_wj = psncan_wj / laican;
        ph.psn_wp = psncan_wp / laican;
        ph.lmr = lmrcan / laican;
        ph.rs = laican / gscan - rb;
    } else {
        ph.psn = 0.0;
        ph.psn_wc = 0.0;
        ph.psn_wj = 0.0;
        ph.psn_wp = 0.0;
        ph.lmr = 0.0;
        ph.rs = 0.0;
    }
}

#include "canopy_phs.h"

}  // namespace canopy
}  // namespace ctsm

namespace ctsm {
namespace canopy {

// constants of the time step for one patch (PhotosynthesisMod.F90:1525-1722)
// phs: PhotosynthesisHydraulicStress's constants (:3117-3300): the
// Ball-Berry minimum conductance without btran (the stress enters through
// bsun / bsha) and the top-leaf nitrogen capped at 10 g/m2
__device__ __forceinline__ void psn_static(const CSwitch &sw, const double *__restrict__ pft, int ivt, double btran,
                                           PsnConst &K, bool &bad, bool phs)
{
    const bool medlyn = sw.stomatal == CTSM_STOMATA_MEDLYN2011;
    K.c3 = ((int)rint(pft[F_C3PSN * CTSM_MAX_PFT + ivt]) == 1);
    double bbbopt = 0.0;
    if (K.c3) {
        K.qe = 0.0;
        if (!medlyn) bbbopt = 10000.0;
    } else {
        K.qe = 0.05;
        if (!medlyn) bbbopt = 40000.0;
    }
    K.bbb = phs ? bbbopt : fmax90(bbbopt * btran, 1.0);
    K.mbb = pft[F_MBBOPT * CTSM_MAX_PFT + ivt];
    const double slatop = pft[F_SLATOP * CTSM_MAX_PFT + ivt], leafcn = pft[F_LEAFCN * CTSM_MAX_PFT + ivt];
    if (slatop * leafcn <= 0.0) bad = true;
    K.lnc = 1.0 / (slatop * leafcn);
    if (phs) K.lnc = fmin90(K.lnc, 10.0);
}

// those that follow from vcmax25top, t10c and the forcing
template <class PRM>
__device__ __forceinline__ void psn_derive(const PRM &P, double forc_pbot, double oair, PsnConst &K)
{
    K.kc25 = P.kc25_coef * forc_pbot;
    K.ko25 = P.ko25_coef * forc_pbot;
    const double sco = 0.5 * 0.209 / P.cp25_yr2000;
    K.cp25 = 0.5 * oair / sco;
    K.jmax25top = ((2.59 - 0.035 * K.t10c) * K.vcmax25top) * P.jmax25top_sf;
    K.tpu25top = P.tpu25ratio * K.vcmax25top;
    K.kp25top = P.kp25ratio * K.vcmax25top;
    K.lmr25top = K.c3 ? K.vcmax25top * P.leaf_mr_vcm : K.vcmax25top * 0.025;
    K.vcmaxse = (668.39 - 1.07 * K.t10c) * P.vcmaxse_sf;
    K.jmaxse = (659.70 - 0.75 * K.t10c) * P.jmaxse_sf;
    K.tpuse = (668.39 - 1.07 * K.t10c) * P.tpuse_sf;
}

template <class PRM>
__device__ void psn_constants(const CSwitch &sw, const PRM &P, const double *__restrict__ pft, int ivt,
                              double forc_pbot, double oair, double t10, double btran, double dayl_factor,
                              PsnConst &K, bool &bad, bool phs = false)
{
    psn_static(sw, pft, ivt, btran, K, bad, phs);
    K.vcmax25top = K.lnc * pft[F_FLNR * CTSM_MAX_PFT + ivt] * P.fnr * P.act25 * dayl_factor;
    K.vcmax25top = K.vcmax25top * pft[F_FNITR * CTSM_MAX_PFT + ivt];
    K.t10c = fmin90(fmax90(t10 - TFRZ, 11.0), 35.0);
    psn_derive(P, forc_pbot, oair, K);
    K.vcmaxc = fth25(P.vcmaxhd, K.vcmaxse);
    K.jmaxc = fth25(P.jmaxhd, K.jmaxse);
    K.tpuc = fth25(P.tpuhd, K.tpuse);
    K.theta_cj = pft[F_THETA_CJ * CTSM_MAX_PFT + ivt];
    K.mslope = pft[F_MEDSLOPE * CTSM_MAX_PFT + ivt];
    K.mint = pft[F_MEDINT * CTSM_MAX_PFT + ivt];
}

// The leaf-temperature factors of one iteration.  All twelve exponentials are
// straight-line code on every lane's own arguments, so they run through each
// other: C3 and C4 lanes share a wave, each with its own pathway's argument where
// both have a factor; a factor its lane does not need is computed and ignored.
template <class PRM, class DRV>
__device__ __forceinline__ void temp_factors(const PRM &P, const DRV &D, const PsnConst &K, double tv, bool anyday,
                                             TFac &T)
{
    const double t25 = 1.0 - (TFRZ + 25.0) / tv;
    const Recip rt = recip(RGAS * 1.e-3 * tv);
    const double e_kc = cm_exp(D.kcha * t25), e_ko = cm_exp(D.koha * t25), e_cp = cm_exp(D.cpha * t25);
    T.pow2 = cm_pow(2.0, (tv - (TFRZ + 25.0)) / 10.0);
    const double eL = cm_exp(K.c3 ? D.lmrha * t25 : 1.3 * (tv - (TFRZ + 55.0)));
    const double eLh = cm_exp(fth_arg(tv, rt, P.lmrhd, P.lmrse));
    T.kc = K.kc25 * e_kc;
    T.ko = K.ko25 * e_ko;
    T.cp = K.cp25 * e_cp;
    T.ftL = eL;
    T.fthL = D.lmrc / (1.0 + eLh);
    T.dL4 = 1.0 + eL;
    if (anyday) {
        const double eV1 = cm_exp(K.c3 ? D.vcmaxha * t25 : 0.2 * ((TFRZ + 15.0) - tv));
        const double eV2 = cm_exp(K.c3 ? fth_arg(tv, rt, P.vcmaxhd, K.vcmaxse) : 0.3 * (tv - (TFRZ + 40.0)));
        const double eJ = cm_exp(D.jmaxha * t25), eJh = cm_exp(fth_arg(tv, rt, P.jmaxhd, K.jmaxse));
        const double eT = cm_exp(D.tpuha * t25), eTh = cm_exp(fth_arg(tv, rt, P.tpuhd, K.tpuse));
        T.ftV = eV1;
        T.fthV = K.vcmaxc / (1.0 + eV2);
        T.dV1 = 1.0 + eV1;
        T.dV2 = 1.0 + eV2;
        T.ftJ = eJ;
        T.fthJ = K.jmaxc / (1.0 + eJh);
        T.ftT = eT;
        T.fthT = K.tpuc / (1.0 + eTh);
    }
}

#define PF(f) pft[(f) * CTSM_MAX_PFT + ivt]

// What a patch keeps between the kernels of a call, indexed by its position in
// the filter (structure of arrays).  Between rounds: the iteration state.  Once it
// has finished: what the outputs are formed from -- FrictionVelocity's last um, obu
// and fm, its ustar in nmozsgn, temp1 in qsatl and temp2 in el, the leaf temperature
// before the last step in t_veg and the step in del, rpp in efeb, wtgq in qsatldT,
// rah2 in taf, eflx_sh_veg in qaf, qflx_evap_veg in delq, qflx_tran_veg in gs_mol.
// itlef: the iterations done, -1 for a patch whose set-up failed.  No kernel reads
// an output array of CanopyFluxes back: a caller may point those it does not want
// at one array.
struct CanopyWork {
    double *t_veg, *del, *efeb, *nmozsgn, *um, *obu, *fm, *qsatl, *el, *qsatldT, *taf, *qaf, *delq, *itlef, *gs_mol,
        *btran;
};
constexpr int N_WORK_FIELDS = 16;
static_assert(sizeof(CanopyWork) == N_WORK_FIELDS * sizeof(double *), "one pointer per saved value");

// CanopyFluxes runs as three kernels over the filter's patches, a patch per lane:
// the set-up (canopy_setup_patch: root stress, roughness, Monin-Obukhov
// initialisation), the rounds of the leaf-temperature iteration
// (canopy_iterate_patch), and the fluxes and outputs of the step
// (canopy_finish_patch).  As one kernel it held the set-up's LDS and, across the
// iteration, everything the outputs read: one wave per SIMD, and the outputs
// written once per round with the few lanes that had finished in it.  The
// iteration now keeps its state only; what the outputs need of its last pass is
// written by the passes that can be the last one (the leaf temperature had settled
// in the pass before, or itmax is reached), each later one over the earlier.
// What bounds them, by counters on 1,048,576 columns (8.9 million patches): the set-up
// moves 19.6 GB in 4.2 ms, as fast as a copy; the first round issues vector
// instructions in 63 % of the SIMDs' cycles (and moves 28.7 GB in 17.1 ms); the later
// rounds, in 35 %, wait for their slow patches; the finish moves 6.7 GB in 2.0 ms,
// three quarters of a copy's rate.  There the one kernel took 31.4 ms for its first round and 43.6 ms
// in all; the set-up takes 4.1, the rounds 26.6 (the first 17.0) and the finish
// 2.0 ms now.  (With the finish reading the outputs back, 0.3 ms less; the totals
// would then depend on the caller's arrays being distinct.)

// The column-level half of calc_effective_soilporosity, calc_volumetric_h2oliq
// and calc_root_moist_stress (SoilMoistStressMod.F90:70-126, 190-240,
// 420-514): effective porosity, volumetric liquid water and, where the level
// takes up water, the soil matric potential of CH78 before the PFT's floor
// and eff / watsat.  The reference computes them once per patch of the filter
// (CanopyFluxesMod.F90:833-891 builds a column filter with one entry per
// patch); here the 64 lanes of a wave share the work of the runs of lanes
// whose patches share a column, one (run, level) item per lane at a time, and
// each lane's patch then reads its column's terms from LDS.  Same operations on
// the same inputs as the per-patch form, so the same bits.  kNoUptake marks a
// level that takes up nothing (no liquid, or frozen below -2 C): a signalling
// NaN, which no arithmetic produces.
constexpr long long kNoUptake = 0x7ff0dead00000001LL;

struct SoilTerms {
    double smp;     // -sucsat s^-bsw, or kNoUptake
    double ratio;   // eff_porosity / watsat
};

constexpr int SOIL_RUNS = 16;     // runs whose terms are in LDS at a time

// The index of the lane's run (-1 for a lane without a valid patch), the runs'
// columns in run_col and their number; every lane of the wave calls it.
template <class CAN>
__device__ int runs_of_wave(const CView &V, const CAN &S, int p, bool active, int *run_col, int &nruns)
{
    const int lane = threadIdx.x;
    int c = -1;
    if (active) {
        // the patches canopy_setup_patch accepts (it reports the others)
        const long pp = V.p1(p);
        const int cp = S.column[pp], g = S.gridcell[pp], ivt = S.itype[pp];
        if (!(ivt < 0 || ivt >= CTSM_MAX_PFT || cp < V.begc || cp >= V.begc + V.ldc || g < V.begg ||
              g >= V.begg + V.ldg))
            c = cp;
    }
    const int prev = __shfl_up(c, 1);
    const bool lead = c >= 0 && (lane == 0 || prev != c);
    const unsigned long long leaders = __ballot(lead);
    if (lead) run_col[__popcll(leaders & ((1ull << lane) - 1ull))] = c;
    nruns = __popcll(leaders);
    wave_sync();
    return c >= 0 ? __popcll(leaders & ((2ull << lane) - 1ull)) - 1 : -1;
}

// The terms of runs r0 .. r0 + SOIL_RUNS - 1 into terms; every lane calls it.
template <class COL, class CAN>
__device__ void soil_terms_of_runs(const CView &V, const COL &col, const CAN &S, const int *run_col, int r0, int nruns,
                                   SoilTerms *terms, const double *lt)
{
    const int nl = V.nlevgrnd;
    const int items = min(nruns - r0, SOIL_RUNS) * nl;
    wave_sync();
    for (int it = threadIdx.x; it < items; it += 64) {
        const int r = it / nl, j = it - r * nl + 1;
        const int rc = run_col[r0 + r];
        const long cs = V.soi(rc, j), cn = V.sno(rc, j);
        const double watsat = col.watsat[cs], dz = col.dz[cn];
        const double vol_ice = fmin90(watsat, col.h2osoi_ice[cn] / (DENICE * dz));
        const double eff = watsat - vol_ice;
        col.eff_porosity[cs] = eff;
        const double liqvol = fmin90(eff, col.h2osoi_liq[cn] / (dz * DENH2O));
        S.h2osoi_liqvol[cs] = liqvol;
        SoilTerms t{__longlong_as_double(kNoUptake), 0.0};
        if (!(liqvol <= 0.0 || col.t_soisno[cn] <= TFRZ - 2.0)) {
            const double s_node = fmax90(liqvol / eff, 0.01);
            t.smp = -col.sucsat[cs] * cm_pow_tab(s_node, -col.bsw[cs], lt);
            t.ratio = eff / watsat;
        }
        terms[r * MAX_NLEVGRND + j - 1] = t;
    }
    wave_sync();
}

// Root moisture stress of one patch from its column's terms (SoilMoistStressMod.
// F90:420-514): rresis, rootr normalised by btran (:480-500), btran.
template <class CAN>
__device__ __forceinline__ double root_stress(const CView &V, const CAN &S, const double *__restrict__ pft, int p,
                                              int ivt, const SoilTerms *soil)
{
    const double smpsc = PF(F_SMPSC), smpso = PF(F_SMPSO);
    double btran = 0.0;
    double rr[MAX_NLEVGRND];
#pragma unroll
    for (int j = 0; j < MAX_NLEVGRND; ++j) rr[j] = j < V.nlevgrnd ? S.rootfr[V.soip(p, j + 1)] : 0.0;
#pragma unroll
    for (int j = 0; j < MAX_NLEVGRND; ++j) {
        if (j >= V.nlevgrnd) continue;
        const SoilTerms t = soil[j];
        double r = 0.0;
        if (__double_as_longlong(t.smp) != kNoUptake) {
            double smp_node = t.smp;
            smp_node = fmax90(smpsc, smp_node);
            const double rres = fmin90(t.ratio * (smp_node - smpsc) / (smpso - smpsc), 1.0);
            S.rresis[V.soip(p, j + 1)] = rres;
            r = rr[j] * rres;
            btran = btran + fmax90(r, 0.0);
        }
        rr[j] = r;
    }
#pragma unroll
    for (int j = 0; j < MAX_NLEVGRND; ++j)
        if (j < V.nlevgrnd) S.rootr[V.soip(p, j + 1)] = (btran > 0.0) ? rr[j] / btran : 0.0;
    S.btran[V.p1(p)] = btran;
    return btran;
}

// The set-up of one patch after its root stress: roughness, leaf humidity,
// initial profiles and the Monin-Obukhov initialisation.  Leaves the iteration
// state in W; a patch that fails is reported and marked (W.itlef = -1).
template <class PRM, class COL, class CAN, class WRK>
__device__ __forceinline__ void canopy_setup_patch(const CView &V, const CSwitch &sw, const PRM &P,
                                                   const double *__restrict__ pft, const COL &col, const CAN &S, int i0,
                                                   int p, ErrWord *err, const WRK &W, const double *lt)
{
    const long pp = V.p1(p);
    const int c = S.column[pp];
    const int g = S.gridcell[pp];
    const int ivt = S.itype[pp];
    const long cc = V.c1(c), gg = V.g1(g);
    bool bad = false;
    const double elai = S.elai[pp], esai = S.esai[pp], htop = S.htop[pp];

    // ---- aerodynamic parameters (CanopyFluxesMod.F90:897-943)
    double displa = S.displa[pp], z0mv = S.z0mv[pp];
    if (sw.z0param == CTSM_Z0_ZENGWANG2007) {
        const double vai = fmin90(elai + esai, TLSAI_CRIT);
        const double egvf = (1.0 - ALPHA_AERO * cm_exp(-vai)) / (1.0 - ALPHA_AERO * cm_exp(-TLSAI_CRIT));
        displa = egvf * displa;
        z0mv = cm_exp(egvf * cm_log_tab(z0mv, lt) + (1.0 - egvf) * cm_log_tab(S.z0mg[cc], lt));
    } else {
        double vai = fmax90(1.e-5, elai + esai);
        displa = htop * (1.0 - (1.0 - cm_exp(-cm_pow_tab(CD1 * vai, 0.5, lt))) / cm_pow_tab(CD1 * vai, 0.5, lt));
        vai = fmin90(vai, PF(F_Z0V_LAIMAX));
        double delt = 2.0;
        const double zc = PF(F_Z0V_C);
        const double U_ustar_ini = cm_pow_tab(PF(F_Z0V_CS) + PF(F_Z0V_CR) * vai * 0.5, -0.5, lt) * zc * vai * 0.25;
        double U_ustar = U_ustar_ini;
        int guard = 0;
        while (delt > 1.e-4) {
            const double prev = U_ustar;
            U_ustar = U_ustar_ini * cm_exp(prev);
            delt = fabs(U_ustar - prev);
            if (++guard > MAX_FIXED_POINT) { bad = true; break; }
        }
        U_ustar = 4.0 * U_ustar / vai / zc;
        const double zcw = PF(F_Z0V_CW);
        z0mv = htop * (1.0 - displa / htop) * cm_exp(-VKC * U_ustar + cm_log_tab(zcw, lt) - 1.0 + 1.0 / zcw);
    }
    const double z0hv = z0mv, z0qv = z0mv;
    const double hu = S.forc_hgt_u[gg] + z0mv + displa;
    const double ht = S.forc_hgt_t[gg] + z0hv + displa;
    const double hq = S.forc_hgt_q[gg] + z0qv + displa;
    S.displa[pp] = displa;
    S.z0mv[pp] = z0mv;
    S.z0hv[pp] = z0hv;
    S.z0qv[pp] = z0qv;
    S.forc_hgt_u_patch[pp] = hu;
    S.forc_hgt_t_patch[pp] = ht;
    S.forc_hgt_q_patch[pp] = hq;

    // ---- leaf humidity, initial profiles (:945-1002)
    const double forc_q = S.forc_q[cc], thm = S.thm[pp], qg = S.qg[cc];
    const double fu = S.forc_u[gg], fvv = S.forc_v[gg];
    const double ur = fmax90(P.wind_min, sqrt(fu * fu + fvv * fvv));
    const double zldis = hu - displa;
    const double t_veg = S.t_veg[pp];
    double qsatl, el, qsatldT;
    qsat(t_veg, S.forc_pbot[cc], qsatl, el, qsatldT);
    const double taf = (col.t_grnd[cc] + thm) / 2.0;
    const double qaf = (forc_q + qg) / 2.0;
    const double dth = thm - taf;
    const double dqh = forc_q - qaf;
    const double dthv = dth * (1.0 + 0.61 * forc_q) + 0.61 * S.forc_th[cc] * dqh;
    const int snl = col.snl[cc];
    if (zldis < 0.0 || snl < -V.nlevsno || snl > 0) {
        report_error(err, p, zldis < 0.0 ? ENDRUN : CTSM_E_ARG);
        W.itlef[i0] = -1.0;
        return;
    }
    // FrictionVelocityMod.F90:1158-1209
    const double wc = 0.5;
    double um;
    if (dthv >= 0.0) um = fmax90(ur, 0.1);
    else um = sqrt(ur * ur + wc * wc);
    const double rib = GRAV * zldis * dthv / (S.thv[cc] * um * um);
    double zeta0;
    if (rib >= 0.0) {
        zeta0 = rib * cm_log_tab(zldis / z0mv, lt) / (1.0 - 5.0 * fmin90(rib, 0.19));
        zeta0 = fmin90(P.zetamaxstable, fmax90(zeta0, 0.01));
    } else {
        zeta0 = rib * cm_log_tab(zldis / z0mv, lt);
        zeta0 = fmax90(-100.0, fmin90(zeta0, -0.01));
    }
    W.t_veg[i0] = t_veg;
    W.del[i0] = 0.0;
    W.efeb[i0] = 0.0;
    W.nmozsgn[i0] = 0.0;
    W.um[i0] = um;
    W.obu[i0] = zldis / zeta0;
    W.fm[i0] = 0.0;
    W.qsatl[i0] = qsatl;
    W.el[i0] = el;
    W.qsatldT[i0] = qsatldT;
    W.taf[i0] = taf;
    W.qaf[i0] = qaf;
    W.delq[i0] = qg - qaf;
    W.itlef[i0] = 0.0;
    W.gs_mol[i0] = S.gs_mol[pp];
    if (bad) report_error(err, p, ENDRUN);
}

// Biomass heat capacities (CanopyFluxesMod.F90:717-819), step constants.
struct Biomass {
    double frac_rad_abs_by_stem, sa_leaf, sa_stem, sa_internal, cp_leaf, cp_stem, rstem, stem_biomass, leaf_biomass;
};
template <class PRM>
__device__ __forceinline__ void biomass(const CSwitch &sw, const PRM &, const double *__restrict__ pft, int ivt,
                                        double elai, double esai, double htop, Biomass &B)
{
    const double k_vert = 0.1, k_cyl_vol = 1.0, k_cyl_area = 1.0, k_internal = 0.0;
    const double min_stem_diameter = 0.05, min_lai = 0.1;
    double frac_rad_abs_by_stem, sa_leaf, sa_stem, sa_internal, cp_leaf, cp_stem, rstem;
    double stem_biomass = 0.0, leaf_biomass = 0.0;
    if (sw.biomass) {
        frac_rad_abs_by_stem = (esai) / (elai + esai);
        if (elai > 0.0) frac_rad_abs_by_stem = k_vert * frac_rad_abs_by_stem;
        const double dbh = PF(F_DBH);
        sa_leaf = elai;
        sa_leaf = 2.0 * sa_leaf;
        sa_stem = PF(F_NSTEM) * (htop * PI * dbh);
        sa_stem = k_cyl_area * sa_stem;
        if (!((int)PF(F_IS_TREE) || (int)PF(F_IS_SHRUB)) || dbh < min_stem_diameter) {
            frac_rad_abs_by_stem = 0.0;
            sa_stem = 0.0;
            sa_leaf = sa_leaf + esai;
        } else {
            if (elai < min_lai) sa_leaf = sa_leaf + esai;
        }
        const double fbw = PF(F_FBW);
        leaf_biomass = (1.e-3 * C_TO_B / PF(F_SLATOP)) * fmax90(0.01, 0.5 * sa_leaf) / (1.0 - fbw);
        const double carea_stem = PI * ((dbh * 0.5) * (dbh * 0.5));
        stem_biomass = carea_stem * htop * k_cyl_vol * PF(F_NSTEM) * PF(F_WOOD) / (1.0 - fbw);
        sa_internal = fmin90(sa_leaf, sa_stem);
        sa_internal = k_internal * sa_internal;
        cp_leaf = leaf_biomass * (CDRYBIO * (1.0 - fbw) + (fbw) * CWATER);
        cp_stem = stem_biomass * (CDRYBIO * (1.0 - fbw) + (fbw) * CWATER);
        cp_stem = k_cyl_vol * cp_stem;
        rstem = PF(F_RSTEM) * dbh;
    } else {
        sa_leaf = (elai + esai);
        frac_rad_abs_by_stem = 0.0;
        sa_stem = 0.0;
        sa_internal = 0.0;
        cp_leaf = 0.0;
        cp_stem = 0.0;
        rstem = 0.0;
    }
    B = Biomass{frac_rad_abs_by_stem, sa_leaf, sa_stem, sa_internal, cp_leaf, cp_stem, rstem, stem_biomass,
                leaf_biomass};
}

// The weights of the heat and the moisture equation (CanopyFluxesMod.F90:1119-1250)
// from the resistances, as the iteration and the outputs need them.
struct HeatWeights {
    double wta, wtl, wtg, wtstem, wtl0, wtg0, wta0, wtstem0, wtga, wtal;
};
__device__ __forceinline__ HeatWeights heat_weights(double rah1, double rb, double rah2, double sa_leaf, double sa_stem,
                                                    double rstem)
{
    HeatWeights w;
    w.wta = 1.0 / rah1;
    w.wtl = sa_leaf / rb;
    w.wtg = 1.0 / rah2;
    w.wtstem = sa_stem / (rstem + rb);
    const double wtshi = 1.0 / (w.wta + w.wtl + w.wtstem + w.wtg);
    w.wtl0 = w.wtl * wtshi;
    w.wtg0 = w.wtg * wtshi;
    w.wta0 = w.wta * wtshi;
    w.wtstem0 = w.wtstem * wtshi;
    w.wtga = w.wta0 + w.wtg0 + w.wtstem0;
    w.wtal = w.wta0 + w.wtl0 + w.wtstem0;
    return w;
}
struct MoistureWeights {
    double wtlq, wtgq0, wtlq0, wtaq0, wtgaq, wtalq;
};
__device__ __forceinline__ MoistureWeights moisture_weights(double fvn, double lai, double raw1, double rb, double rpp,
                                                            double wtgq)
{
    MoistureWeights w;
    const double wtaq = fvn / raw1;
    w.wtlq = fvn * lai / rb * rpp;
    const double wtsqi = 1.0 / (wtaq + w.wtlq + wtgq);
    w.wtgq0 = wtgq * wtsqi;
    w.wtlq0 = w.wtlq * wtsqi;
    w.wtaq0 = wtaq * wtsqi;
    w.wtgaq = w.wtaq0 + w.wtgq0;
    w.wtalq = w.wtaq0 + w.wtlq0;
    return w;
}

// The outputs of one leaf phase, and of both, in a pass that can be the last.
// Photosynthesis writes some of them only on branches fixed for the step (nrad,
// par, the stomatal model): they are stored under the same conditions (otherwise
// the arrays keep their values, as in the reference); the PHS path writes some
// itself, to arrays of its own.
template <bool PHS, class CAN>
__device__ __forceinline__ void store_phase(const CAN &S, uint32_t po, bool sun, const Phase &ph, int nrad, bool lit)
{
    if (nrad >= 1) {
        at(sun ? S.rssun_z : S.rssha_z, po) = ph.rs_z;
        at(sun ? S.cisun_z : S.cisha_z, po) = ph.ci_z;
        at(sun ? S.lmrsun_z : S.lmrsha_z, po) = ph.lmr_z;
        at(sun ? S.psnsun_z : S.psnsha_z, po) = ph.psn_z;
        at(sun ? S.gs_mol_sun : S.gs_mol_sha, po) = ph.gs_ph;
    }
    if (!PHS && lit) at(sun ? S.gs_mol_sun_ln : S.gs_mol_sha_ln, po) = ph.gs_ln;
    at(sun ? S.rssun : S.rssha, po) = ph.rs;
    at(sun ? S.lmrsun : S.lmrsha, po) = ph.lmr;
    at(sun ? S.psnsun : S.psnsha, po) = ph.psn;
    at(sun ? S.psnsun_wc : S.psnsha_wc, po) = ph.psn_wc;
    at(sun ? S.psnsun_wj : S.psnsha_wj, po) = ph.psn_wj;
    at(sun ? S.psnsun_wp : S.psnsha_wp, po) = ph.psn_wp;
}
template <bool PHS, class CAN>
__device__ __forceinline__ void store_shared(const CAN &S, uint32_t po, const CSwitch &sw, const Shared &sh, int nrad,
                                             double parsun, double parsha)
{
    at(S.gb_mol, po) = sh.gb_mol;
    if (PHS) return;
    at(S.gs_mol, po) = sh.gs_mol;
    if (nrad < 1) return;
    const bool medlyn = sw.stomatal == CTSM_STOMATA_MEDLYN2011;
    const bool lit_sun = parsun > 0.0, lit_sha = parsha > 0.0;
    at(S.vcmax_z, po) = sh.vcmax_z;
    at(S.tpu_z, po) = sh.tpu_z;
    at(S.kp_z, po) = sh.kp_z;
    at(S.ac, po) = sh.ac;
    at(S.aj, po) = sh.aj;
    at(S.ap, po) = sh.ap;
    at(S.ag, po) = sh.ag;
    at(S.an, po) = sh.an;
    // rh_leaf: a dark phase writes 0, a lit one under Ball-Berry its value;
    // vpd_can: a lit phase under Medlyn (the last writer wins)
    if (!medlyn || !lit_sun || !lit_sha) at(S.rh_leaf, po) = sh.rh_leaf;
    if (medlyn && (lit_sun || lit_sha)) at(S.vpd_can, po) = sh.vpd_can;
}

// A phase's photosynthesis and conductance as the canopy's totals need them: the rate
// that limits it (0: none, 1: Rubisco, 2: light, 3: product) says which of psn_wc,
// psn_wj and psn_wp is psn, the others being zero.
struct PhaseSums {
    double psn = 0.0, gs = 0.0;
    int limit = 0;
    PhaseSums() = default;
    __device__ explicit PhaseSums(const Phase &ph)
        : psn(ph.psn), gs(ph.gs_ph), limit(ph.psn_wc != 0.0 ? 1 : ph.psn_wj != 0.0 ? 2 : ph.psn_wp != 0.0 ? 3 : 0)
    {
    }
    __device__ double of(int rate) const { return limit == rate ? psn : 0.0; }
};
// PhotosynthesisTotal and the noon water-use efficiency, in a pass that can be the last.
template <class CAN>
__device__ __forceinline__ void store_totals(const CAN &S, uint32_t po, bool noon, double laisun, double laisha,
                                             const PhaseSums &sun, const PhaseSums &sha)
{
    const double fpsn = sun.psn * laisun + sha.psn * laisha;
    at(S.fpsn, po) = fpsn;
    at(S.fpsn_wc, po) = sun.of(1) * laisun + sha.of(1) * laisha;
    at(S.fpsn_wj, po) = sun.of(2) * laisun + sha.of(2) * laisha;
    at(S.fpsn_wp, po) = sun.of(3) * laisun + sha.of(3) * laisha;
    double iwue = SPVAL;
    if (noon && fpsn > 0.0) {
        const double gs = 1.e-6 * (laisun * sun.gs + laisha * sha.gs);
        iwue = (gs > 0.0) ? fpsn / gs : SPVAL;
    }
    at(S.iwue_ln, po) = iwue;
}

// Step constants of the iteration that wait in LDS ([KC_N][64], the lane's column)
// instead of in registers: with log's table 20,104 bytes a wave, room for two waves
// per SIMD.  Values formed from them in a few operations are formed anew.
enum {
    KC_T10C, KC_VCMAXC, KC_JMAXC, KC_TPUC, KC_VCMAX25, KC_STOM0, KC_STOM1, KC_THETA, KC_LM, KC_LH, KC_WVEG, KC_DLEXT,
    KC_SALEAF, KC_SASTEM, KC_RSTEM, KC_CPL, KC_FR, KC_ZL, KC_ZT, KC_ZQ, KC_BIR, KC_RAD, KC_CIRLW, KC_UR, KC_SQDLEAF,
    KC_H2OCAN, KC_LAI, KC_ELAI, KC_LAISUN, KC_LAISHA, KC_FDRY, KC_FWET, KC_THM, KC_TLINI, KC_TSTEM, KC_N
};

// At most `budget` leaf-temperature iterations of one patch from the state in W.
// Returns true when the patch is still iterating (its state saved in W); false when
// it finished or its set-up had failed.
// PHS: CanopyFluxes with plant hydraulic stress, H its PhsArgs (unused
// otherwise): PhotosynthesisHydraulicStress in place of the two Photosynthesis
// calls and the branches of CanopyFluxesMod.F90:1219-1230, 1353-1356.
template <bool PHS, class PRM, class COL, class CAN, class WRK, class PHA, class DRV>
__device__ __forceinline__ bool canopy_iterate_patch(const CView &V, const CSwitch &sw, const PRM &P,
                             const double *__restrict__ pft, const COL &col, const CAN &S,
                             int i0, int p, double dtime, ErrWord *err,
                             int budget, const WRK &W, const PHA &H, const DRV &D, const double *lt, double *kc,
                             double *phs_lane)
{
    uint32_t wo = (uint32_t)i0 * 8u;
    const double it_done = at(W.itlef, wo);
    if (it_done < 0.0) return false;
    const long pp = V.p1(p);
    const int c = S.column[pp];
    const int g = S.gridcell[pp];
    const int ivt = S.itype[pp];
    const long cc = V.c1(c), gg = V.g1(g);
    const double btran0 = 0.0, zii = 1000.0, beta = 1.0, delmax = 1.0, dlemin = 0.1, dtmin = 0.01;
    const int itmin = 2;
    const double ria = 0.5;
    bool bad = false;

    // ---- the step's constants
    const int nrad = S.nrad[pp];
    const double parsun = S.parsun_z[pp], parsha = S.parsha_z[pp];
    const bool noon = S.near_local_noon[gg] != 0;
    const bool anyday = nrad >= 1 && (parsun > 0.0 || parsha > 0.0);
    const bool medlyn = sw.stomatal == CTSM_STOMATA_MEDLYN2011;
    double btran = at(W.btran, wo), sa_lw;
    bool c3;
    {
        const double elai = S.elai[pp], esai = S.esai[pp], emv = S.emv[pp], emg = col.emg[cc];
        Biomass B;
        biomass(sw, P, pft, ivt, elai, esai, S.htop[pp], B);
        kc[KC_SALEAF * 64] = B.sa_leaf;
        kc[KC_SASTEM * 64] = B.sa_stem;
        kc[KC_RSTEM * 64] = B.rstem;
        kc[KC_CPL * 64] = B.cp_leaf / dtime;
        kc[KC_FR * 64] = B.frac_rad_abs_by_stem;
        sa_lw = B.sa_internal * emv * SB;
        const double dayl = S.dayl[gg], max_dayl = S.max_dayl[gg];
        const double dayl_factor = fmin90(1.0, fmax90(0.01, (dayl * dayl) / (max_dayl * max_dayl)));
        PsnConst K;
        psn_constants(sw, P, pft, ivt, S.forc_pbot[cc], S.forc_po2[gg], S.t_a10[pp], btran, dayl_factor, K, bad, PHS);
        c3 = K.c3;
        kc[KC_T10C * 64] = K.t10c;
        kc[KC_VCMAXC * 64] = K.vcmaxc;
        kc[KC_JMAXC * 64] = K.jmaxc;
        kc[KC_TPUC * 64] = K.tpuc;
        kc[KC_VCMAX25 * 64] = K.vcmax25top;
        kc[KC_STOM0 * 64] = medlyn ? K.mslope : K.bbb;
        kc[KC_STOM1 * 64] = medlyn ? K.mint : K.mbb;
        kc[KC_THETA * 64] = K.theta_cj;
        kc[KC_SQDLEAF * 64] = sqrt(PF(F_DLEAF));
        kc[KC_H2OCAN * 64] = (S.liqcan[pp] + S.snocan[pp]) / dtime;
        kc[KC_LAI * 64] = elai + esai;
        kc[KC_ELAI * 64] = elai;
        kc[KC_LAISUN * 64] = S.laisun[pp];
        kc[KC_LAISHA * 64] = S.laisha[pp];
        kc[KC_FDRY * 64] = S.fdry[pp];
        kc[KC_FWET * 64] = S.fwet[pp];
        kc[KC_THM * 64] = S.thm[pp];
        kc[KC_TLINI * 64] = S.t_veg[pp];
        kc[KC_TSTEM * 64] = S.t_stem[pp];
        const double displa = S.displa[pp], z0mv = S.z0mv[pp];
        const double hu = S.forc_hgt_u[gg] + z0mv + displa;
        const double ht = S.forc_hgt_t[gg] + z0mv + displa;
        const double hq = S.forc_hgt_q[gg] + z0mv + displa;
        const double zl = hu - displa, zt = ht - displa, zq = hq - displa;
        kc[KC_ZL * 64] = zl;
        kc[KC_ZT * 64] = zt;
        kc[KC_ZQ * 64] = zq;
        kc[KC_LM * 64] = cm_log_tab(zl / z0mv, lt);
        kc[KC_LH * 64] = cm_log_tab(zt / z0mv, lt);
        kc[KC_WVEG * 64] = cm_exp(-(elai + esai));
        const double lai_dl_eff = P.lai_dl * (1.0 - fmin90(col.snow_depth[cc] / P.z_dl, 1.0));
        kc[KC_DLEXT * 64] = 1.0 - cm_exp(-lai_dl_eff);
        const int snl = col.snl[cc];
        const double frac_sno = col.frac_sno_eff[cc], frac_h2osfc = col.frac_h2osfc[cc];
        const double t_top = col.t_soisno[V.sno(c, snl + 1)], t_soi1 = col.t_soisno[V.sno(c, 1)];
        const double t_h2osfc = col.t_h2osfc[cc];
        const double lw_grnd = (frac_sno * p4(t_top) + (1.0 - frac_sno - frac_h2osfc) * p4(t_soi1)
                                + frac_h2osfc * p4(t_h2osfc));
        const double air = emv * (1.0 + (1.0 - emv) * (1.0 - emg)) * col.forc_lwrad[cc];
        const double cir = emv * emg * SB;
        kc[KC_BIR * 64] = -(2.0 - emv * (1.0 - emg)) * emv * SB;
        kc[KC_RAD * 64] = S.sabv[pp] + air;
        kc[KC_CIRLW * 64] = cir * lw_grnd;
        const double fu = S.forc_u[gg], fvv = S.forc_v[gg];
        kc[KC_UR * 64] = fmax90(P.wind_min, sqrt(fu * fu + fvv * fvv));
    }
    // ---- the iteration's state
    double t_veg = at(W.t_veg, wo), qsatl = at(W.qsatl, wo), el = at(W.el, wo), qsatldT = at(W.qsatldT, wo),
           taf = at(W.taf, wo), qaf = at(W.qaf, wo), delq = at(W.delq, wo), um = at(W.um, wo), obu = at(W.obu, wo);
    int nmozsgn = (int)at(W.nmozsgn, wo);
    double gs_mol_c = at(W.gs_mol, wo);
    double del = at(W.del, wo), efeb = at(W.efeb, wo), fm_c = at(W.fm, wo);
    int itlef = (int)it_done;
    const uint32_t po0 = (uint32_t)pp * 8u, co0 = (uint32_t)cc * 8u, go0 = (uint32_t)gg * 8u;
    for (int it = 0;; ++it) {
        if (it >= budget) {
            // still iterating: keep the state for the next round
            at(W.t_veg, wo) = t_veg;
            at(W.del, wo) = del;
            at(W.efeb, wo) = efeb;
            at(W.nmozsgn, wo) = (double)nmozsgn;
            at(W.um, wo) = um;
            at(W.obu, wo) = obu;
            at(W.fm, wo) = fm_c;
            at(W.qsatl, wo) = qsatl;
            at(W.el, wo) = el;
            at(W.qsatldT, wo) = qsatldT;
            at(W.taf, wo) = taf;
            at(W.qaf, wo) = qaf;
            at(W.delq, wo) = delq;
            at(W.itlef, wo) = (double)itlef;
            at(W.gs_mol, wo) = gs_mol_c;
            if (PHS) at(W.btran, wo) = btran;
            if (bad) report_error(err, p, ENDRUN);
            return true;
        }
        // whether this pass can be the patch's last: a patch converges only where
        // the pass before moved the leaf by less than dtmin too
        const bool last = itlef >= sw.itmax || (itlef >= itmin && !(del >= dtmin));
        // (offsets made opaque, here and before each part of the pass: the step's
        // constants are read where they are used, not held in registers across the
        // loop or the pass)
#define KC(name) kc[KC_##name * 64 + k_]
#define OPAQUE asm volatile("" : "+v"(k_), "+v"(po), "+v"(co), "+v"(go), "+v"(wo))
        uint32_t po = po0, co = co0, go = go0;
        int k_ = 0;
        OPAQUE;
        FV fv;
        double wtgq = 0.0;
        fv.fm = fm_c;
        {
            const FVLogs fvlog{KC(LM), KC(LH)};
            friction_velocity(KC(ZL), KC(ZT), KC(ZQ), at(S.z0mv, po), fvlog, obu, itlef + 1, um, fv, lt);
        }
        const double ustar = fv.ustar, temp1 = fv.temp1, temp2 = fv.temp2;
        const double tlbef = t_veg;
        const double del2 = del;
        const double ram1 = 1.0 / (ustar * ustar / um);
        const double rah1 = 1.0 / (temp1 * ustar);
        const double raw1 = 1.0 / (temp2 * ustar);
        const double uaf = um * sqrt(1.0 / (ram1 * um));
        const double uuc = fmin90(0.4, (0.03 * um / ustar));
        const double cf = P.cv / (sqrt(uaf) * KC(SQDLEAF));
        const double rb = 1.0 / (cf * uaf);
        const double csoilb = VKC / (P.a_coef * cm_pow_tab(at(S.z0mg, co) * uaf / NU, P.a_exp, lt));
        double csoilcn;
        {
            const double w = KC(WVEG), t_grnd = at(col.t_grnd, co);
            if (sw.undercanopy && (taf - t_grnd) > 0.0) {
                const double ri = (GRAV * at(S.htop, po) * (taf - t_grnd)) / (taf * (uaf * uaf));
                const double ricsoilc = P.csoilc / (1.00 + ria * fmin90(ri, 10.0));
                csoilcn = csoilb * w + ricsoilc * (1.0 - w);
            } else {
                csoilcn = csoilb * w + P.csoilc * (1.0 - w);
            }
        }
        const double rah2 = sw.biomass ? 1.0 / (csoilcn * uuc) : 1.0 / (csoilcn * uaf);
        const double raw2 = rah2;
        const double svpts = el;
        const double eah = at(S.forc_pbot, co) * qaf / 0.622;
        if (last) {
            at(W.obu, wo) = obu;        // the inputs of this FrictionVelocity call
            at(W.um, wo) = um;
            at(W.fm, wo) = fv.fm;
            at(W.qsatl, wo) = temp1;
            at(W.el, wo) = temp2;
            at(W.nmozsgn, wo) = ustar;
            at(W.taf, wo) = rah2;
            at(S.rh_af, po) = eah / svpts;
            at(S.vpd, po) = fmax90((svpts - eah), 50.0) * 0.001;
        }

        // Photosynthesis, sun then shade
        Shared sh = Shared{};
        sh.gs_mol = gs_mol_c;
        double rs_sun, rs_sha, qflx_tran_veg = 0.0;
        {
            OPAQUE;
            const double o2 = at(S.forc_po2, go), co2 = at(S.forc_pco2, go), forc_pbot = at(S.forc_pbot, co);
            const double thm = KC(THM);
            PsnConst K;
            K.c3 = c3;
            K.qe = c3 ? 0.0 : 0.05;
            K.t10c = KC(T10C);
            K.vcmax25top = KC(VCMAX25);
            psn_derive(P, forc_pbot, o2, K);
            K.vcmaxc = KC(VCMAXC);
            K.jmaxc = KC(JMAXC);
            K.tpuc = KC(TPUC);
            K.bbb = K.mslope = KC(STOM0);
            K.mbb = K.mint = KC(STOM1);
            K.theta_cj = KC(THETA);
            TFac T;
            temp_factors(P, D, K, t_veg, anyday, T);
            if (last) {
                at(S.kc, po) = T.kc;
                at(S.ko, po) = T.ko;
                at(S.cp, po) = T.cp;
            }
            if constexpr (PHS) {
                // sun and shade together; btran and the transpiration come from the hydraulics
                Phase sun = Phase{}, sha = Phase{};
                btran = photosynthesis_phs(V, sw, P, K, T, H, S, p, c, ivt, nrad, noon, forc_pbot, thm, svpts, eah, o2,
                                           co2, rb, qsatl, qaf, sun, sha, sh, bad, phs_lane, lt);
                qflx_tran_veg = at(S.qflx_tran_veg, po);
                rs_sun = sun.rs;
                rs_sha = sha.rs;
                if (last) {
                    at(W.btran, wo) = btran;
                    store_phase<PHS>(S, po, true, sun, nrad, false);
                    store_phase<PHS>(S, po, false, sha, nrad, false);
                    store_totals(S, po, noon, KC(LAISUN), KC(LAISHA), PhaseSums(sun), PhaseSums(sha));
                }
            } else {
                rs_sun = rs_sha = 0.0;
                PhaseSums sun{};
                // one call site for both phases: sun (k = 0), then shade
#pragma nounroll
                for (int k = 0; k < 2; ++k) {
                    const bool ks = k == 0;
                    const double par = ks ? parsun : parsha;
                    Phase ph{};
                    photosynthesis(sw, P, K, T, nrad, par, ks ? S.laisun_z : S.laisha_z,
                                   ks ? S.vcmaxcintsun : S.vcmaxcintsha, ks ? S.o3coefvsun : S.o3coefvsha,
                                   ks ? S.o3coefgsun : S.o3coefgsha, po,
                                   noon, forc_pbot, thm, svpts, eah, o2, co2, rb, btran, ph, sh, bad);
                    if (last) {
                        store_phase<PHS>(S, po, ks, ph, nrad, nrad >= 1 && par > 0.0);
                        if (!ks) store_totals(S, po, noon, KC(LAISUN), KC(LAISHA), sun, PhaseSums(ph));
                    }
                    if (ks) {
                        rs_sun = ph.rs;
                        sun = PhaseSums(ph);
                    } else {
                        rs_sha = ph.rs;
                    }
                }
            }
            if (last) store_shared<PHS>(S, po, sw, sh, nrad, parsun, parsha);
        }

        // conductances and the leaf-temperature Newton step (:1119-1331)
        OPAQUE;
        const double fvn = (double)at(S.frac_veg_nosno, po / 2);
        const double forc_rho = at(S.forc_rho, co), forc_q = at(S.forc_q, co), qg = at(S.qg, co);
        const double t_grnd = at(col.t_grnd, co), thm = KC(THM), lai = KC(LAI), t_stem = KC(TSTEM), h2ocan_dt = KC(H2OCAN);
        const HeatWeights hw = heat_weights(rah1, rb, rah2, KC(SALEAF), KC(SASTEM), KC(RSTEM));
        const double lw_stem = sa_lw * p4(t_stem);
        const double lw_leaf = sa_lw * p4(t_veg);
        const double fdry = KC(FDRY), fwet = KC(FWET);
        double rppdry;
        if (fdry > 0.0) rppdry = fdry * rb * (KC(LAISUN) / (rb + rs_sun) + KC(LAISHA) / (rb + rs_sha)) / KC(ELAI);
        else rppdry = 0.0;
        double efpot = forc_rho * (lai / rb) * (qsatl - qaf);
        double rpp;
        if (PHS) {
            if (efpot > 0.0) {
                if (btran > btran0) rpp = rppdry + fwet;
                else rpp = fwet;
                rpp = fmin90(rpp, (qflx_tran_veg + h2ocan_dt) / efpot);
            } else {
                rpp = 1.0;
            }
        } else if (efpot > 0.0) {
            if (btran > btran0) {
                qflx_tran_veg = efpot * rppdry;
                rpp = rppdry + fwet;
            } else {
                rpp = fwet;
                qflx_tran_veg = 0.0;
            }
            rpp = fmin90(rpp, (qflx_tran_veg + h2ocan_dt) / efpot);
        } else {
            rpp = 1.0;
            qflx_tran_veg = 0.0;
        }
        const double rdl = KC(DLEXT) / (0.004 * uaf);
        // the branches' divides share one evaluation (operands per lane)
        {
            const bool lee = sw.soil_resis == CTSM_SOILRESIS_LEEPIELKE1992, sl14 = sw.soil_resis == CTSM_SOILRESIS_SL14;
            if (delq < 0.0 || lee || sl14) {
                const bool wet = delq < 0.0;
                const double num = (wet || !lee) ? fvn : at(S.soilbeta, co) * fvn;
                const double den = (wet || lee) ? raw2 + rdl : raw2 + at(S.soilresis, co);
                wtgq = num / den;
            }
        }
        const MoistureWeights mw = moisture_weights(fvn, lai, raw1, rb, rpp, wtgq);
        const double dc1 = forc_rho * CPAIR * hw.wtl;
        const double dc2 = HVAP * forc_rho * mw.wtlq;
        const double efsh = dc1 * (hw.wtga * t_veg - hw.wtg0 * t_grnd - hw.wta0 * thm - hw.wtstem0 * t_stem);
        double efe = dc2 * (mw.wtgaq * qsatl - mw.wtgq0 * qg - mw.wtaq0 * forc_q);
        double erre = 0.0;
        if (efe * efeb < 0.0) {
            const double efeold = efe;
            efe = 0.1 * efeold;
            erre = efe - efeold;
        }
        const double fr = KC(FR), bir = KC(BIR), rad = KC(RAD), cirlw = KC(CIRLW), cpl = KC(CPL);
        double dt_veg = ((1.0 - fr) * (rad + bir * p4(t_veg) + cirlw)
                         - efsh - efe - lw_leaf + lw_stem - cpl * (t_veg - KC(TLINI)))
                        / ((1.0 - fr) * (-4.0 * bir * p3(t_veg)) + 4.0 * sa_lw * p3(t_veg)
                           + dc1 * hw.wtga + dc2 * mw.wtgaq * qsatldT + cpl);
        t_veg = tlbef + dt_veg;
        const double dels = dt_veg;
        del = fabs(dels);
        double errp = 0.0;
        if (del > delmax) {
            dt_veg = delmax * dels / del;
            t_veg = tlbef + dt_veg;
            errp = (1.0 - fr) * (rad + bir * p3(tlbef) * (tlbef + 4.0 * dt_veg) + cirlw)
                   - sa_lw * p3(tlbef) * (tlbef + 4.0 * dt_veg)
                   + lw_stem
                   - (efsh + dc1 * hw.wtga * dt_veg) - (efe + dc2 * mw.wtgaq * qsatldT * dt_veg)
                   - cpl * (t_veg - KC(TLINI));
        }
        efpot = forc_rho * (lai / rb) * (mw.wtgaq * (qsatl + qsatldT * dt_veg) - mw.wtgq0 * qg - mw.wtaq0 * forc_q);
        double qflx_evap_veg = rpp * efpot;
        if (!PHS) {
            if (efpot > 0.0 && btran > btran0) qflx_tran_veg = efpot * rppdry;
            else qflx_tran_veg = 0.0;
        }
        const double ecidif = fmax90(0.0, qflx_evap_veg - qflx_tran_veg - h2ocan_dt);
        qflx_evap_veg = fmin90(qflx_evap_veg, qflx_tran_veg + h2ocan_dt);
        const double eflx_sh_veg = efsh + dc1 * hw.wtga * dt_veg + errp + erre + HVAP * ecidif;
        qsat(t_veg, at(S.forc_pbot, co), qsatl, el, qsatldT);
        taf = hw.wtg0 * t_grnd + hw.wta0 * thm + hw.wtl0 * t_veg + hw.wtstem0 * t_stem;
        qaf = mw.wtlq0 * qsatl + mw.wtgq0 * qg + forc_q * mw.wtaq0;
        const double dth = thm - taf;
        const double dqh = forc_q - qaf;
        delq = mw.wtalq * qg - mw.wtlq0 * qsatl - mw.wtaq0 * forc_q;
        const double tstar = temp1 * dth;
        const double qstar = temp2 * dqh;
        const double forc_th = at(S.forc_th, co), thv = at(S.thv, co);
        const double thvstar = tstar * (1.0 + 0.61 * forc_q) + 0.61 * forc_th * qstar;
        const double zldis = KC(ZL), ur = KC(UR);
        double zeta = zldis * VKC * GRAV * thvstar / ((ustar * ustar) * thv);
        if (zeta >= 0.0) {
            zeta = fmin90(P.zetamaxstable, fmax90(zeta, 0.01));
            um = fmax90(ur, 0.1);
        } else {
            zeta = fmax90(-100.0, fmin90(zeta, -0.01));
            double wc;
            if (ustar * thvstar > 0.0) wc = 0.0;
            else wc = beta * cm_pow_tab(-GRAV * ustar * thvstar * zii / thv, 0.333, lt);
            um = sqrt(ur * ur + wc * wc);
        }
        const double obuold = itlef > 0 ? obu : 0.0;
        obu = zldis / zeta;
        if (obuold * obu < 0.0) nmozsgn = nmozsgn + 1;
        if (nmozsgn >= 4) obu = zldis / (-0.01);

        gs_mol_c = sh.gs_mol;
        fm_c = fv.fm;
        itlef = itlef + 1;
        bool converged = false;
        double num_iter = 0.0;
        if (itlef > itmin) {
            const double dele = fabs(efe - efeb);
            efeb = efe;
            const double det = fmax90(del, del2);
            num_iter = (double)itlef;
            converged = det < dtmin && dele < dlemin;
        }
        if (last) {
            at(W.t_veg, wo) = tlbef;
            at(W.del, wo) = dt_veg;
            at(W.efeb, wo) = rpp;
            at(W.qsatldT, wo) = wtgq;
            at(W.qaf, wo) = eflx_sh_veg;
            at(W.delq, wo) = qflx_evap_veg;
            at(W.gs_mol, wo) = qflx_tran_veg;
            at(S.um, po) = um;
            at(S.obu, po) = obu;
            at(S.zeta, po) = zeta;
            at(S.num_iter, po) = num_iter;
        }
        if (converged || itlef > sw.itmax) break;
#undef KC
#undef OPAQUE
    }
    if (bad) report_error(err, p, ENDRUN);
    return false;
}

// The fluxes and outputs of one patch that has finished its iteration.
template <bool PHS, class PRM, class COL, class CAN, class WRK>
__device__ __forceinline__ void canopy_finish_patch(const CView &V, const CSwitch &sw, const PRM &P,
                                                    const double *__restrict__ pft, const COL &col, const CAN &S,
                                                    int i0, int p, double dtime, const WRK &W, const double *lt)
{
    if (W.itlef[i0] < 0.0) return;
    const long pp = V.p1(p);
    const int c = S.column[pp];
    const int g = S.gridcell[pp];
    const int ivt = S.itype[pp];
    const long cc = V.c1(c), gg = V.g1(g);
    const double elai = S.elai[pp], esai = S.esai[pp], htop = S.htop[pp];
    const double emv = S.emv[pp], emg = col.emg[cc], thm = S.thm[pp];
    const double forc_pbot = S.forc_pbot[cc], forc_q = S.forc_q[cc], forc_rho = S.forc_rho[cc];
    const double qg = S.qg[cc], t_grnd = col.t_grnd[cc];
    const double fu = S.forc_u[gg], fvv = S.forc_v[gg];
    const double sabv = S.sabv[pp], dleaf = PF(F_DLEAF);
    const double liqcan0 = S.liqcan[pp], snocan0 = S.snocan[pp];
    Biomass B;
    biomass(sw, P, pft, ivt, elai, esai, htop, B);
    if (sw.biomass) {
        S.leaf_biomass[pp] = B.leaf_biomass;
        S.stem_biomass[pp] = B.stem_biomass;
    }
    const double fr = B.frac_rad_abs_by_stem, cp_leaf = B.cp_leaf, cp_stem = B.cp_stem, stem_biomass = B.stem_biomass;
    const double tl_ini = S.t_veg[pp];
    double t_stem = S.t_stem[pp];
    const double ts_ini = t_stem;

    // ---- diagnostics of the last FrictionVelocity call
    const double displa = S.displa[pp], z0mv = S.z0mv[pp];
    const double hu = S.forc_hgt_u[gg] + z0mv + displa;
    const double ur = fmax90(P.wind_min, sqrt(fu * fu + fvv * fvv));
    const double um = W.um[i0];
    FV fv;
    fv.ustar = W.nmozsgn[i0];
    fv.fm = W.fm[i0];
    friction_velocity_diag(hu, displa, z0mv, z0mv, z0mv, W.obu[i0], ur, um, fv, lt);

    // ---- the last pass again, from what it left
    const double temp1 = W.qsatl[i0], temp2 = W.el[i0];
    const double tlbef = W.t_veg[i0], dt_veg = W.del[i0];
    const double t_veg = tlbef + dt_veg;
    const double wtgq = W.qsatldT[i0], rah2 = W.taf[i0], btran = W.btran[i0];
    const double ram1 = 1.0 / (fv.ustar * fv.ustar / um);
    const double rah1 = 1.0 / (temp1 * fv.ustar);
    const double raw1 = 1.0 / (temp2 * fv.ustar);
    const double uaf = um * sqrt(1.0 / (ram1 * um));
    const double cf = P.cv / (sqrt(uaf) * sqrt(dleaf));
    const double rb = 1.0 / (cf * uaf);
    const HeatWeights hw = heat_weights(rah1, rb, rah2, B.sa_leaf, B.sa_stem, B.rstem);
    const MoistureWeights mw = moisture_weights((double)S.frac_veg_nosno[pp], elai + esai, raw1, rb, W.efeb[i0], wtgq);
    double qsatl, el, qsatldT;
    qsat(t_veg, forc_pbot, qsatl, el, qsatldT);
    const double taf = hw.wtg0 * t_grnd + hw.wta0 * thm + hw.wtl0 * t_veg + hw.wtstem0 * ts_ini;
    const double qaf = mw.wtlq0 * qsatl + mw.wtgq0 * qg + forc_q * mw.wtaq0;
    const double dth = thm - taf;
    const double dqh = forc_q - qaf;
    const double delq = mw.wtalq * qg - mw.wtlq0 * qsatl - mw.wtaq0 * forc_q;
    const double eflx_sh_veg = W.qaf[i0];
    double eflx_sh_stem = forc_rho * CPAIR * hw.wtstem
                          * ((hw.wta0 + hw.wtg0 + hw.wtl0) * ts_ini - hw.wtg0 * t_grnd - hw.wta0 * thm
                             - hw.wtl0 * tlbef);
    eflx_sh_stem = eflx_sh_stem + forc_rho * CPAIR * hw.wtstem * (-hw.wtl0 * dt_veg);
    const double qflx_evap_veg = W.delq[i0], qflx_tran_veg = W.gs_mol[i0];
    const double lw_stem = B.sa_internal * emv * SB * p4(ts_ini);
    const double lw_leaf = B.sa_internal * emv * SB * p3(tlbef) * (tlbef + 4.0 * dt_veg);

    // ---- radiation terms (:945-1002)
    const double forc_lwrad = col.forc_lwrad[cc];
    const double air = emv * (1.0 + (1.0 - emv) * (1.0 - emg)) * forc_lwrad;
    const double bir = -(2.0 - emv * (1.0 - emg)) * emv * SB;
    const double cir = emv * emg * SB;
    const int snl = col.snl[cc];
    const double frac_sno = col.frac_sno_eff[cc], frac_h2osfc = col.frac_h2osfc[cc];
    const double t_top = col.t_soisno[V.sno(c, snl + 1)], t_soi1 = col.t_soisno[V.sno(c, 1)];
    const double t_h2osfc = col.t_h2osfc[cc];
    const double lw_grnd = (frac_sno * p4(t_top) + (1.0 - frac_sno - frac_h2osfc) * p4(t_soi1)
                            + frac_h2osfc * p4(t_h2osfc));
    const double temp12m = fv.temp12m, temp22m = fv.temp22m;

    // ---- fluxes after the iteration (:1467-1615)
    const double errp = (1.0 - fr) * (sabv + air + bir * p3(tlbef) * (tlbef + 4.0 * dt_veg) + cir * lw_grnd)
           - lw_leaf + lw_stem - eflx_sh_veg - HVAP * qflx_evap_veg - ((t_veg - tl_ini) * cp_leaf / dtime);
    double dt_stem = 0.0;
    double dhsdt_canopy = 0.0;
    if (sw.biomass) {
        if (stem_biomass > 0.0) {
            dt_stem = (fr * (sabv + air + bir * p4(ts_ini) + cir * lw_grnd) - eflx_sh_stem + lw_leaf - lw_stem)
                      / (cp_stem / dtime - fr * bir * 4.0 * p3(ts_ini));
        } else {
            dt_stem = 0.0;
        }
        dhsdt_canopy = dt_stem * cp_stem / dtime + (t_veg - tl_ini) * cp_leaf / dtime;
        t_stem = t_stem + dt_stem;
    }
    const double delt = hw.wtal * t_grnd - hw.wtl0 * t_veg - hw.wta0 * thm - hw.wtstem0 * t_stem;
    S.taux[pp] = -forc_rho * fu / ram1;
    S.tauy[pp] = -forc_rho * fvv / ram1;
    S.eflx_sh_grnd[pp] = CPAIR * forc_rho * hw.wtg * delt;
    const double delt_snow = hw.wtal * t_top - hw.wtl0 * t_veg - hw.wta0 * thm - hw.wtstem0 * t_stem;
    const double delt_soil = hw.wtal * t_soi1 - hw.wtl0 * t_veg - hw.wta0 * thm - hw.wtstem0 * t_stem;
    const double delt_h2osfc = hw.wtal * t_h2osfc - hw.wtl0 * t_veg - hw.wta0 * thm - hw.wtstem0 * t_stem;
    S.eflx_sh_snow[pp] = CPAIR * forc_rho * hw.wtg * delt_snow;
    S.eflx_sh_soil[pp] = CPAIR * forc_rho * hw.wtg * delt_soil;
    S.eflx_sh_h2osfc[pp] = CPAIR * forc_rho * hw.wtg * delt_h2osfc;
    S.qflx_evap_soi[pp] = forc_rho * wtgq * delq;
    const double delq_snow = mw.wtalq * S.qg_snow[cc] - mw.wtlq0 * qsatl - mw.wtaq0 * forc_q;
    S.qflx_ev_snow[pp] = forc_rho * wtgq * delq_snow;
    const double delq_soil = mw.wtalq * S.qg_soil[cc] - mw.wtlq0 * qsatl - mw.wtaq0 * forc_q;
    S.qflx_ev_soil[pp] = forc_rho * wtgq * delq_soil;
    const double delq_h2osfc = mw.wtalq * S.qg_h2osfc[cc] - mw.wtlq0 * qsatl - mw.wtaq0 * forc_q;
    S.qflx_ev_h2osfc[pp] = forc_rho * wtgq * delq_h2osfc;
    const double t_ref2m = thm + temp1 * dth * (1.0 / temp12m - 1.0 / temp1);
    S.t_ref2m[pp] = t_ref2m;
    S.t_ref2m_r[pp] = t_ref2m;
    const double q_ref2m = forc_q + temp2 * dqh * (1.0 / temp22m - 1.0 / temp2);
    S.q_ref2m[pp] = q_ref2m;
    double e_ref2m;
    const double qsat_ref2m = qsat_only(t_ref2m, forc_pbot, e_ref2m);
    const double rh_ref2m = fmin90(100.0, q_ref2m / qsat_ref2m * 100.0);
    S.rh_ref2m[pp] = rh_ref2m;
    S.rh_ref2m_r[pp] = rh_ref2m;
    S.vpd_ref2m[pp] = e_ref2m * (1.0 - rh_ref2m / 100.0);
    S.dlrad[pp] = (1.0 - emv) * emg * forc_lwrad
                  + emv * emg * SB * p3(tlbef) * (tlbef + 4.0 * dt_veg) * (1.0 - fr)
                  + emv * emg * SB * p3(ts_ini) * (ts_ini + 4.0 * dt_stem) * fr;
    S.ulrad[pp] = ((1.0 - emg) * (1.0 - emv) * (1.0 - emv) * forc_lwrad
                   + emv * (1.0 + (1.0 - emg) * (1.0 - emv)) * SB * p3(tlbef) * (tlbef + 4.0 * dt_veg) * (1.0 - fr)
                   + emv * (1.0 + (1.0 - emg) * (1.0 - emv)) * SB * p3(ts_ini) * (ts_ini + 4.0 * dt_stem) * fr
                   + emg * (1.0 - emv) * SB * lw_grnd);
    S.t_skin[pp] = emv * t_veg + (1.0 - emv) * sqrt(sqrt(lw_grnd));
    const double cgrnds = S.cgrnds[pp] + CPAIR * forc_rho * hw.wtg * hw.wtal;
    const double cgrndl = S.cgrndl[pp] + forc_rho * wtgq * mw.wtalq * S.dqgdT[cc];
    S.cgrnds[pp] = cgrnds;
    S.cgrndl[pp] = cgrndl;
    S.cgrnd[pp] = cgrnds + cgrndl * col.htvp[cc];
    double snocan = snocan0, liqcan = liqcan0;
    const double snocan_baseline = snocan;
    if (t_veg > TFRZ) {
        if ((qflx_evap_veg - qflx_tran_veg) * dtime > liqcan)
            snocan = fmax90(0.0, snocan + liqcan + (qflx_tran_veg - qflx_evap_veg) * dtime);
        liqcan = fmax90(0.0, liqcan + (qflx_tran_veg - qflx_evap_veg) * dtime);
    } else if (t_veg <= TFRZ) {
        if ((qflx_evap_veg - qflx_tran_veg) * dtime > snocan)
            liqcan = liqcan + snocan + (qflx_tran_veg - qflx_evap_veg) * dtime;
        snocan = fmax90(0.0, snocan + (qflx_tran_veg - qflx_evap_veg) * dtime);
    }
    if (fabs(snocan) < 1.e-10 * fabs(snocan_baseline)) snocan = 0.0;
    S.snocan[pp] = snocan;
    S.liqcan[pp] = liqcan;

    // ---- remaining outputs
    if (PHS) S.btran[pp] = btran;       // (otherwise the set-up's)
    S.ustar[pp] = fv.ustar;
    S.ram1[pp] = ram1;
    S.rah1[pp] = rah1;
    S.raw1[pp] = raw1;
    S.rah2[pp] = rah2;
    S.raw2[pp] = rah2;
    S.uaf[pp] = uaf;
    S.rb1[pp] = rb;
    S.taf[pp] = taf;
    S.qaf[pp] = qaf;
    S.eflx_sh_stem[pp] = eflx_sh_stem;
    S.eflx_sh_veg[pp] = eflx_sh_veg;
    S.qflx_evap_veg[pp] = qflx_evap_veg;
    S.qflx_tran_veg[pp] = qflx_tran_veg;
    S.dhsdt_canopy[pp] = dhsdt_canopy;
    S.t_veg[pp] = t_veg;
    S.t_stem[pp] = t_stem;
    S.u10[pp] = fv.u10;
    S.u10_clm[pp] = fv.u10_clm;
    S.va[pp] = fv.va;
    S.fv[pp] = fv.fv;
    S.vds[pp] = fv.vds;
    S.dleaf_patch[pp] = dleaf;
    S.canopy_err[pp] = errp;
    // photosyns_inst
    PsnConst K;
    bool bad = false;       // the iteration has reported it
    psn_static(sw, pft, ivt, PHS ? 0.0 : btran, K, bad, PHS);
    S.c3flag[pp] = K.c3 ? 1 : 0;
    S.qe[pp] = K.qe;
    if (sw.stomatal == CTSM_STOMATA_BB1987) {
        S.bbb[pp] = K.bbb;
        S.mbb[pp] = K.mbb;
    }
    S.lnca[pp] = K.lnc;
}

// Values of the parameters alone, formed on the host (the same operations): the
// activation energies over rgas (tfrz + 25) and respiration's scaling at 25 C.
struct CanopyDerived {
    double kcha, koha, cpha, lmrha, vcmaxha, jmaxha, tpuha, lmrc;
};
static CanopyDerived canopy_derived(const ctsm_canopy_params &P)
{
    const double r25 = RGAS * 1.e-3 * (TFRZ + 25.0);
    return CanopyDerived{P.kcha / r25,    P.koha / r25,   P.cpha / r25, P.lmrha / r25, P.vcmaxha / r25,
                         P.jmaxha / r25, P.tpuha / r25, 1.0 + cm_exp((-P.lmrhd + P.lmrse * (TFRZ + 25.0)) / r25)};
}

// Everything one launch of the three kernels reads: a kernel's only argument.
struct RoundArgs {
    CView V;
    CSwitch sw;
    ctsm_canopy_params P;
    CanopyDerived D;
    const double *pft;
    ctsm_col_state col;
    ctsm_canopy_state S;
    int n, pfirst;                  // patches; the first one where there is no filter
    const int32_t *filter;
    double dtime;
    ErrWord *err;
    int round, budget;
    const int32_t *list_in, *cnt_in;
    int32_t *list_out, *cnt_out;
    CanopyWork W;
};
// the PHS form's argument: the same, then the PHS arrays
struct RoundArgsPhs {
    RoundArgs r;
    PhsArgs phs;
};
#define KARG __attribute__((address_space(4)))

// The arguments are read in place from the kernel-argument segment, each member
// where it is used: loaded all at once on entry, their few hundred uniform
// pointers would not fit the scalar registers and spill.
#define CANOPY_VIEW(A)                                                                                             \
    CView { (A)->V.begc, (A)->V.ldc, (A)->V.begp, (A)->V.ldp, (A)->V.begg, (A)->V.ldg, (A)->V.nlevsno,              \
            (A)->V.nlevsoi, (A)->V.nlevgrnd }
#define CANOPY_SWITCH(A)                                                                                           \
    CSwitch { (A)->sw.z0param, (A)->sw.stomatal, (A)->sw.soil_resis, (A)->sw.biomass, (A)->sw.undercanopy,          \
              (A)->sw.light_inhibit, (A)->sw.itmax }

// The set-up of every patch of the filter, one wave per block.
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) k_canopy_setup(RoundArgs)
{
    const KARG RoundArgs *A = (const KARG RoundArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    __shared__ SoilTerms terms[SOIL_RUNS * MAX_NLEVGRND];
    __shared__ int run_col[64];
    LOG_TABLE(logt);
    const int i0 = blockIdx.x * 64 + threadIdx.x;
    const bool active = i0 < A->n;
    const CView V = CANOPY_VIEW(A);
    const int p = !active ? V.begp : A->filter ? A->filter[i0] : A->pfirst + i0;
    int nruns;
    const int run = runs_of_wave(V, A->S, p, active, run_col, nruns);
    const int ivt = run >= 0 ? A->S.itype[V.p1(p)] : 0;
    for (int r0 = 0; r0 < nruns; r0 += SOIL_RUNS) {
        soil_terms_of_runs(V, A->col, A->S, run_col, r0, nruns, terms, logt);
        if (run >= r0 && run < r0 + SOIL_RUNS)
            A->W.btran[i0] = root_stress(V, A->S, A->pft, p, ivt, terms + (run - r0) * MAX_NLEVGRND);
    }
    if (!active) return;
    if (run < 0) {      // an index that addresses other arrays lies outside their allocations
        report_error(A->err, p, CTSM_E_ARG);
        A->W.itlef[i0] = -1.0;
        return;
    }
    const CSwitch sw = CANOPY_SWITCH(A);
    canopy_setup_patch(V, sw, A->P, A->pft, A->col, A->S, i0, p, A->err, A->W, logt);
}

// One round of the iteration over the patches still iterating (round 0: the
// whole filter), compacting those that continue into list_out with one atomic
// per wavefront.  Blocks are one wavefront, a patch per lane.  Round 0
// (STRIDE false) covers the filter with its grid; later rounds (STRIDE true)
// stride a capped grid over the round's count; there the segment pointer is made
// opaque on every pass, so its loads stay inside the pass instead of being
// hoisted in front of the loop.
// WAVES: the register budget the kernel is compiled for (waves per SIMD).  One wave
// needs 296 registers; the two-wave instance (256, and 176 B/lane of scratch) pays
// once a filter has a second wave for the SIMDs: launch_canopy has the rule.
// PHS: CanopyFluxes with plant hydraulic stress (argument RoundArgsPhs).
template <int WAVES, bool STRIDE, bool PHS = false>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES)))
k_canopy_round(typename std::conditional<PHS, RoundArgsPhs, RoundArgs>::type)
{
    const KARG RoundArgs *Ap = (const KARG RoundArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    __shared__ double consts[KC_N * 64];
    LOG_TABLE(logt);
    const int round = Ap->round;
    const int count = (round == 0) ? Ap->n : *Ap->cnt_in;
    const int lane = threadIdx.x;
    for (int base = blockIdx.x * 64; base < count; base += gridDim.x * 64) {
        const KARG RoundArgs *A = Ap;
        if (STRIDE) asm volatile("" : "+s"(A));
        const int idx = base + lane;
        bool cont = false;
        int i0 = (idx < count) ? ((round == 0) ? idx : A->list_in[idx]) : 0;
        if (idx < count) {
            const CView V = CANOPY_VIEW(A);
            const CSwitch sw = CANOPY_SWITCH(A);
            const int p = A->filter ? A->filter[i0] : A->pfirst + i0;
            if constexpr (PHS) {
                const KARG RoundArgsPhs *B = (const KARG RoundArgsPhs *)A;
                __shared__ double phs_soil[phs::SOIL_LDS * phs::SOIL_STRIDE];
                cont = canopy_iterate_patch<true>(V, sw, A->P, A->pft, A->col, A->S, i0, p, A->dtime, A->err,
                                                  A->budget, A->W, B->phs, A->D, logt, consts + lane, phs_soil + lane);
            } else {
                cont = canopy_iterate_patch<false>(V, sw, A->P, A->pft, A->col, A->S, i0, p, A->dtime, A->err,
                                                   A->budget, A->W, *A, A->D, logt, consts + lane, nullptr);
            }
        }
        const unsigned long long mask = __ballot(cont);
        if (mask) {
            const int leader = __ffsll((unsigned long long)mask) - 1;
            int pos = 0;
            if (lane == leader) pos = atomicAdd(A->cnt_out, __popcll(mask));
            pos = __shfl(pos, leader);
            if (cont) A->list_out[pos + __popcll(mask & ((1ull << lane) - 1ull))] = i0;
        }
        if (!STRIDE) break;
    }
}

// The outputs of every patch of the filter.
template <bool PHS>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) k_canopy_finish(RoundArgs)
{
    const KARG RoundArgs *A = (const KARG RoundArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    LOG_TABLE(logt);
    const int i0 = blockIdx.x * 64 + threadIdx.x;
    if (i0 >= A->n) return;
    const CView V = CANOPY_VIEW(A);
    const CSwitch sw = CANOPY_SWITCH(A);
    const int p = A->filter ? A->filter[i0] : A->pfirst + i0;
    canopy_finish_patch<PHS>(V, sw, A->P, A->pft, A->col, A->S, i0, p, A->dtime, A->W, logt);
}

__global__ void __launch_bounds__(64) k_zero_counts(int32_t *cnt, int n)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) cnt[i] = 0;
}
#undef PF

// photosyns_inst%TimeStepInit (PhotosynthesisMod.F90:1143-1201) and
// rb1(begp:endp) = 0 (CanopyFluxesMod.F90:830): every patch of the bounds,
// the n patches from begp or, where the bounds are the filter's own patches,
// the patches filter names.
__global__ void __launch_bounds__(256) k_canopy_init(int n, const int32_t *__restrict__ filter, int begp,
                                                     ctsm_canopy_state S)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= n) return;
    const long i = filter ? (long)(filter[f] - begp) : (long)f;
    S.psnsun[i] = 0.0; S.psnsun_wc[i] = 0.0; S.psnsun_wj[i] = 0.0; S.psnsun_wp[i] = 0.0;
    S.psnsha[i] = 0.0; S.psnsha_wc[i] = 0.0; S.psnsha_wj[i] = 0.0; S.psnsha_wp[i] = 0.0;
    S.fpsn[i] = 0.0; S.fpsn_wc[i] = 0.0; S.fpsn_wj[i] = 0.0; S.fpsn_wp[i] = 0.0;
    S.rb1[i] = 0.0;
}

// cgrnd / cgrnds / cgrndl = 0 before CanopyFluxes (BiogeophysPreFluxCalcsMod.F90:390-392)
__global__ void __launch_bounds__(256) k_zero_cgrnd(int n, const int32_t *__restrict__ filter, int begp,
                                                    ctsm_canopy_state S)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long pp = (long)((filter ? filter[i] : begp + i) - begp);
    S.cgrnd[pp] = 0.0;
    S.cgrnds[pp] = 0.0;
    S.cgrndl[pp] = 0.0;
}

// p2c_1d_filter of qflx_tran_veg (clm_driver.F90:1714-1716) and
// Compute_EffecRootFrac_And_VertTranSink_Default (SoilWaterPlantSinkMod.F90:332-424)
// for one column, reading its patches straight from HBM
__device__ __forceinline__ void root_sink_column(const CView &V, const ctsm_col_state &col,
                                                 const ctsm_canopy_state &S, int c, ErrWord *err)
{
    const long cc = V.c1(c);
    const int pi = col.patchi[cc], pf = col.patchf[cc];
    if (pf >= pi && (pi < V.begp || pf >= V.begp + V.ldp)) {   // patches outside the allocation
        report_error(err, c, CTSM_E_ARG);
        return;
    }
    // the p2c sum and the sink's normaliser are the same sum in the same order
    double tcol = 0.0;
    double r[MAX_NLEVSOI];
#pragma unroll
    for (int j = 0; j < MAX_NLEVSOI; ++j) r[j] = 0.0;
    for (int p = pi; p <= pf; ++p) {
        const long q = V.p1(p);
        if (!S.active[q]) continue;
        const double qt = S.qflx_tran_veg[q], w = S.wtcol[q];
        tcol = tcol + qt * w;
        // per level the patches are summed in ascending order, as the reference's j-outer loop does
#pragma unroll
        for (int j = 1; j <= MAX_NLEVSOI; ++j)
            if (j <= V.nlevsoi) r[j - 1] = r[j - 1] + S.rootr[V.soip(p, j)] * qt * w;
    }
    S.qflx_tran_veg_col[cc] = tcol;
#pragma unroll
    for (int j = 1; j <= MAX_NLEVSOI; ++j) {
        if (j > V.nlevsoi) continue;
        double rc = r[j - 1];
        if (tcol != 0.0) rc = rc / tcol;
        S.rootr_col[V.soi(c, j)] = rc;
        S.qflx_rootsoi_col[V.soi(c, j)] = rc * tcol;
    }
}

__global__ void __launch_bounds__(256) k_root_sink(CView V, ctsm_col_state col, ctsm_canopy_state S, int n,
                                                   const int32_t *__restrict__ filter, ErrWord *err)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    root_sink_column(V, col, S, filter ? filter[i] : V.begc + i, err);
}

// The same for consecutive columns (no filter) whose patches are consecutive:
// a block stages the patch range of RS_COLS columns in LDS (weights and
// activity once, then rootr RS_GROUPS levels at a time, every element read once
// and coalesced); thread group g sums level j0 + g of its column over the
// column's patches in ascending order from LDS -- the operations and their
// order are those of root_sink_column.  A block whose patches exceed the
// staging space takes root_sink_column.
constexpr int RS_COLS = 64;
constexpr int RS_GROUPS = 4;
constexpr int RS_CAP = 16 * RS_COLS;

__global__ void __launch_bounds__(RS_COLS *RS_GROUPS) k_root_sink_staged(CView V, ctsm_col_state col,
                                                                         ctsm_canopy_state S, int n, ErrWord *err)
{
    __shared__ double s_qt[RS_CAP], s_w[RS_CAP], s_row[RS_GROUPS][RS_CAP];
    __shared__ int32_t s_act[RS_CAP];
    __shared__ int s_lo, s_hi, s_bad;
    const int t = threadIdx.x;
    const int lane = t % RS_COLS, g = t / RS_COLS;
    const int i = blockIdx.x * RS_COLS + lane;
    const int c = V.begc + i;
    const long cc = V.c1(c);
    const bool live = i < n;
    int pi = 0, pf = -1;
    if (live) {
        pi = col.patchi[cc];
        pf = col.patchf[cc];
    }
    if (t == 0) { s_lo = INT_MAX; s_hi = INT_MIN; s_bad = 0; }
    __syncthreads();
    if (g == 0 && live && pf >= pi) {
        if (pi < V.begp || pf >= V.begp + V.ldp) atomicOr(&s_bad, 1);
        atomicMin(&s_lo, pi);
        atomicMax(&s_hi, pf);
    }
    __syncthreads();
    const int lo = s_lo, hi = s_hi;
    const int np = hi >= lo ? hi - lo + 1 : 0;
    if (s_bad || np > RS_CAP) {              // block-uniform
        if (g == 0 && live) root_sink_column(V, col, S, c, err);
        return;
    }
    for (int k = t; k < np; k += RS_COLS * RS_GROUPS) {
        const long q = V.p1(lo + k);
        s_qt[k] = S.qflx_tran_veg[q];
        s_w[k] = S.wtcol[q];
        s_act[k] = S.active[q];
    }
    __syncthreads();
    // every group forms its column's total (the same operations, so the same bits)
    double tcol = 0.0;
    for (int p = pi; p <= pf; ++p) {
        const int k = p - lo;
        if (!s_act[k]) continue;
        tcol = tcol + s_qt[k] * s_w[k];
    }
    if (g == 0 && live) S.qflx_tran_veg_col[cc] = tcol;
    for (int j0 = 1; j0 <= V.nlevsoi; j0 += RS_GROUPS) {
        __syncthreads();                     // the previous levels have been summed
        for (int r = 0; r < RS_GROUPS && j0 + r <= V.nlevsoi; ++r)
            for (int k = t; k < np; k += RS_COLS * RS_GROUPS) s_row[r][k] = S.rootr[V.soip(lo + k, j0 + r)];
        __syncthreads();
        const int j = j0 + g;
        if (!live || j > V.nlevsoi) continue;
        double r = 0.0;
        for (int p = pi; p <= pf; ++p) {
            const int k = p - lo;
            if (!s_act[k]) continue;
            r = r + s_row[g][k] * s_qt[k] * s_w[k];
        }
        double rc = r;
        if (tcol != 0.0) rc = rc / tcol;
        S.rootr_col[V.soi(c, j)] = rc;
        S.qflx_rootsoi_col[V.soi(c, j)] = rc * tcol;
    }
}

}  // namespace canopy

constexpr int SIMDS = 1024;      // 256 CUs

// Iterations of round r >= 1: round_its twice, then twice as many each time.  The
// late rounds hold a few thousand patches at most, whose waves fit the chip at once:
// packing them again gains nothing there and costs a launch and a cold start:
// 20,000 columns 3391 us in 13 rounds of 3, 3133 us in 6 of 3, 3, 6, 12, 24.
static int canopy_round_budget(int r, int round_its)
{
    return r <= 2 ? round_its : (int)std::min<long>((long)round_its << std::min(r - 2, 30), INT_MAX);
}

// Rounds after the first one: enough to take a patch from first_its
// iterations to itmax + 1.
static int canopy_later_rounds(int itmax, int first_its, int round_its)
{
    int r = 0;
    for (long left = (long)itmax + 1 - first_its; left > 0; left -= canopy_round_budget(r, round_its)) ++r;
    return r;
}

// Work buffer: N_WORK_FIELDS doubles per patch of the filter and, where the
// iteration runs in rounds, two patch lists and one counter per round.
size_t canopy_work_bytes(int n, int itmax, int first_its, int round_its)
{
    using namespace canopy;
    if (n <= 0) return 0;
    const int R = canopy_later_rounds(itmax, first_its, round_its);
    const size_t w = (size_t)N_WORK_FIELDS * n * sizeof(double);
    return R == 0 ? w : w + 2 * (size_t)n * sizeof(int32_t) + (size_t)(R + 1) * sizeof(int32_t);
}

// Patches a work buffer of `bytes` takes per pass where the iteration runs
// without rounds (launch_canopy then goes over a longer filter in parts); 0 where
// it runs in rounds, which take the whole filter at once.
int canopy_one_pass_patches(size_t bytes, int itmax, int first_its, int round_its)
{
    using namespace canopy;
    if (canopy_later_rounds(itmax, first_its, round_its) != 0) return 0;
    const size_t m = bytes / (N_WORK_FIELDS * sizeof(double)) / 64 * 64;
    return m > (size_t)INT_MAX ? INT_MAX : (int)m;
}

// work: canopy_work_bytes(n, ...) or, without rounds, room for `part` patches
// (part = 0: for all).
void launch_canopy(hipStream_t st, const ctsm_layout &L, const ctsm_config &cfg, const ctsm_canopy_params &prm,
                   const double *pft_dev, const ctsm_col_state &col, const ctsm_canopy_state &can, int n,
                   const int32_t *filter, double dtime, ErrWord *err, void *work, int part, int first_its,
                   int round_its, bool zero_cgrnd, int waves, bool bounds_are_filter, const ctsm_phs_state *phs_q,
                   const ctsm_phs_canopy_state *phs_h, const double *phs_table)
{
    using namespace canopy;
    const GptlRange range("canflux");
    const bool hydrstress = phs_h != nullptr;
    CView V{L.begc_alloc, L.ldc, L.begp_alloc, L.ldp, L.begg_alloc, L.ldg, cfg.nlevsno, cfg.nlevsoi, cfg.nlevgrnd};
    CSwitch sw{cfg.z0param_method, cfg.stomatalcond_method, cfg.soil_resis_method, cfg.use_biomass_heat_storage,
               cfg.use_undercanopy_stability, cfg.light_inhibit, cfg.itmax_canopy_fluxes};
    if (bounds_are_filter && filter) {
        if (n > 0)
            hipLaunchKernelGGL(k_canopy_init, dim3((n + 255) / 256), dim3(256), 0, st, n, filter, L.begp_alloc, can);
    } else if (L.ldp > 0) {
        hipLaunchKernelGGL(k_canopy_init, dim3((L.ldp + 255) / 256), dim3(256), 0, st, L.ldp, nullptr, 0, can);
    }
    if (n <= 0) return;
    if (zero_cgrnd)
        hipLaunchKernelGGL(k_zero_cgrnd, dim3((n + 255) / 256), dim3(256), 0, st, n, filter, L.begp_alloc, can);
    int R = canopy_later_rounds(cfg.itmax_canopy_fluxes, first_its, round_its);
    if (part <= 0 || part > n) part = n;
    for (int done = 0; done < n; done += part) {
        const int m = n - done < part ? n - done : part;
        const int blocks = (m + 63) / 64;
        RoundArgs a{V, sw, prm, canopy_derived(prm), pft_dev, col, can, m, L.begp_alloc + done, filter ? filter + done : nullptr, dtime, err,
                    0, 0, nullptr, nullptr, nullptr, nullptr, CanopyWork{}};
        // The two-wave instance from the first block that has no SIMD to itself.  65,536
        // columns (8,704 waves): 3380 us with one wave per SIMD, 3150 us with two; 762
        // waves: 1469 and 1566 us.  The later rounds, with the rest as it is, one wave and
        // two: 20,000 columns (2,656 blocks) 1688 and 1796 us, 40,000 (5,313) 2273 and
        // 2316, 65,536 (8,704) 2989 and 3048, 262,144 (34,816) 8903 and 8692.
        const bool two = waves > 1 && blocks > SIMDS, two_later = waves > 1 && blocks > 4 * SIMDS;
        auto first_kernel = two ? k_canopy_round<2, false> : k_canopy_round<1, false>;
        auto later_kernel = two_later ? k_canopy_round<2, true> : k_canopy_round<1, true>;
        double *w = (double *)work;
        auto field = [&](int k) { return w + (size_t)k * m; };
        a.W = CanopyWork{field(0), field(1), field(2),  field(3),  field(4),  field(5),  field(6),  field(7),
                         field(8), field(9), field(10), field(11), field(12), field(13), field(14), field(15)};
        hipLaunchKernelGGL(k_canopy_setup, dim3(blocks), dim3(64), 0, st, a);
        {
            const GptlRange iter_range("can_iter");
            // the PHS form: one instance, built for one wave per SIMD
            RoundArgsPhs b{};
            if (hydrstress) b.phs = PhsArgs{*phs_q, *phs_h, phs_table, cfg.nlevsoi, cfg.modifyphoto_and_lmr_forcrop};
            auto launch = [&](bool later, int grid) {
                if (hydrstress) {
                    b.r = a;
                    if (later) hipLaunchKernelGGL((k_canopy_round<1, true, true>), dim3(grid), dim3(64), 0, st, b);
                    else hipLaunchKernelGGL((k_canopy_round<1, false, true>), dim3(grid), dim3(64), 0, st, b);
                } else if (later) {
                    hipLaunchKernelGGL(later_kernel, dim3(grid), dim3(64), 0, st, a);
                } else {
                    hipLaunchKernelGGL(first_kernel, dim3(grid), dim3(64), 0, st, a);
                }
            };
            if (R == 0) {
                // one pass: every patch finishes (converged or itmax reached) in round 0
                a.budget = cfg.itmax_canopy_fluxes + 1;
                launch(false, blocks);
            } else {
                int32_t *list[2] = {(int32_t *)(w + (size_t)N_WORK_FIELDS * m), nullptr};
                list[1] = list[0] + m;
                int32_t *cnt = list[1] + m;
                hipLaunchKernelGGL(k_zero_counts, dim3(1), dim3(64), 0, st, cnt, R + 1);
                // Where every wave has a SIMD to itself there is nothing to pack the
                // survivors for but the lanes, and one later round takes them to the end:
                // 35,000 patches (544 waves) 1125 us against 1231 us in the rounds below,
                // 1088 waves 1309 and 1379, 2176 waves 1691 and 1621.
                const bool alone = blocks <= SIMDS;
                if (alone) R = std::min(R, 1);
                // later rounds stride over the patches still iterating with a grid that
                // keeps every wave slot of the chip busy
                const int later_blocks = blocks < 8192 ? blocks : 8192;
                for (int r = 0; r <= R; ++r) {
                    a.round = r;
                    a.budget = r == 0 ? first_its : alone ? cfg.itmax_canopy_fluxes + 1 : canopy_round_budget(r, round_its);
                    a.list_in = list[(r + 1) & 1];
                    a.cnt_in = r ? cnt + r - 1 : nullptr;
                    a.list_out = list[r & 1];
                    a.cnt_out = cnt + r;
                    launch(r > 0, r == 0 ? blocks : later_blocks);
                }
            }
        }
        if (hydrstress) hipLaunchKernelGGL(k_canopy_finish<true>, dim3(blocks), dim3(64), 0, st, a);
        else hipLaunchKernelGGL(k_canopy_finish<false>, dim3(blocks), dim3(64), 0, st, a);
    }
}

void launch_root_sink(hipStream_t st, const ctsm_layout &L, const ctsm_config &cfg, const ctsm_col_state &col,
                      const ctsm_canopy_state &can, int n, const int32_t *filter, ErrWord *err)
{
    const GptlRange range("hydro_without_drainage");
    using namespace canopy;
    if (n <= 0) return;
    CView V{L.begc_alloc, L.ldc, L.begp_alloc, L.ldp, L.begg_alloc, L.ldg, cfg.nlevsno, cfg.nlevsoi, cfg.nlevgrnd};
    if (filter)
        hipLaunchKernelGGL(k_root_sink, dim3((n + 255) / 256), dim3(256), 0, st, V, col, can, n, filter, err);
    else
        hipLaunchKernelGGL(k_root_sink_staged, dim3((n + RS_COLS - 1) / RS_COLS), dim3(RS_COLS * RS_GROUPS), 0, st, V,
                           col, can, n, err);
}

}  // namespace ctsm
