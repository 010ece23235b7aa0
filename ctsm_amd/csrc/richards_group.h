// richards_group.h -- moisture-form Richards solve with G lanes per column.
//
// The same arithmetic as soilwater_moisture_form (SoilWaterMovementMod.F90:
// 976-1440) and as the one-lane form in soilwater_dev.h, laid out for gfx950:
// a column's layers are split over G consecutive lanes (lane g of the group
// owns layers g*K .. g*K+K-1, K = 20/G), so
//   - the Clapp-Hornberger properties (two x**y per layer) and the flux rows
//     of a trial are computed by G lanes at once;
//   - the LAPACK dgtsv elimination, which is sequential in the layer index,
//     runs as G stages: lane s eliminates its rows, then the partly
//     eliminated row moves to lane s+1 (DPP);
//   - the back substitution runs the stages in reverse, carrying the two
//     solution values below;
//   - the error estimate max is reduced over the group, so every lane of the
//     group takes the same accept / halve / double decision.
// A lane keeps ~K*13 doubles instead of 20*13, and several waves share a SIMD.
// Values are bit-identical to the one-lane form.
// Bound by FP64 issue: vector instructions take 63 % of the SIMDs' cycles (1,048,576
// columns, three waves per SIMD); the HBM traffic, seven times the columns' own through
// spilled registers and the trials' diagnostics, runs at 3.0 TB/s.  The serial stages
// run with one lane of a group, so what can leave them has: the error estimate's two
// divisions a row, the diagonal's reciprocals, the row interchange's selects (a branch
// that few rows take).  The properties are straight-line over the lane's layers,
// divisors used several times are inverted once, log's table is in LDS.  262,144
// uneven columns: 5.31 ms before, 3.42 ms so with 8 lanes; 7.12 and 3.82 ms with 4.
// G = 0 takes the group size at run time (argument gsz: 2, 4 or 8 lanes of K
// layers each), so one kernel can give each wavefront the group size its
// columns' depth needs.
#pragma once
#include <type_traits>

#include "common.h"
#include "watertable_bc.h"

namespace ctsm {

__device__ __forceinline__ double gshfl(double v, int src, int width)
{
    return __shfl(v, src, width);
}

// The value of another lane of the group through a DPP move: two vector instructions
// where __shfl is two LDS permutes and their wait.  Groups are at most 8 lanes and
// aligned, so they lie inside a 16-lane DPP row.  A lane at the group's end gets its
// row neighbour's value or zero, which nothing uses.
template <int CTRL>
__device__ __forceinline__ double group_move(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double from_next(double v) { return group_move<0x101>(v); }   // row_shl:1
__device__ __forceinline__ double from_prev(double v) { return group_move<0x111>(v); }   // row_shr:1

// the maximum over the group's GS lanes, in every lane
__device__ __forceinline__ double group_max(double v, int GS)
{
    if (GS > 1) v = fmax90(v, group_move<0xb1>(v));     // quad_perm 1 0 3 2
    if (GS > 2) v = fmax90(v, group_move<0x4e>(v));     // quad_perm 2 3 0 1
    if (GS > 4) v = fmax90(v, group_move<0x141>(v));    // row_half_mirror: the other quad
    return v;
}

// whether v is 2^lo .. 2^hi
__device__ __forceinline__ bool within(double v, int lo, int hi)
{
    return (unsigned)__double2hiint(v) - ((unsigned)(1023 + lo) << 20) < ((unsigned)(hi - lo) << 20);
}
// whether `here` holds on any lane of the group
__device__ __forceinline__ bool any_of_group(bool here, int GS)
{
    const unsigned long long m = __ballot(here);
    return m && ((m >> (__lane_id() & ~(GS - 1))) & ((1ull << GS) - 1)) != 0;
}

// The solve with reciprocals (D = Recip) gives up, with the column as it was, where an
// operand of its divisions might leave the range they are exact in; the solve with
// divisions (D = Plain) takes any.  Ranges of the layers' constants that hold every
// operand but the substitution's to it, with s in 0.01 .. 1:
//   hk   0 or 2^-419 .. 2^20     (hkc s^(2b+3))
//   dsm  2^-9 .. 2^212           (b suc s^-b / (s ws))
//   the flux derivatives' numerators 0 or 2^-529 .. 2^232, a row's entries dl 0 or from
//   2^-682, its diagonal up to 2^290, so dl / d 0 or from 2^-972.
// Real soils are far inside; a NaN is outside.
constexpr int RICHARDS_RANGE = 6;
__device__ __forceinline__ bool ordinary_layer(double dz, double den, double ws, double bsw, double suc, double hkc)
{
    return within(dz, -10, 20) && within(den, -10, 20) && within(ws, -10, 1) && within(bsw, -4, 5) && bsw <= 24.0 &&
           within(suc, -4, 30) && (within(hkc, -80, 20) || hkc == 0.0);
}
__device__ __forceinline__ bool ordinary_steps(const Params &P, double dtime)
{
    return within(dtime, -20, 30) && P.dtmin >= 0x1.0p-20 && P.verySmall >= 0x1.0p-60;
}

// WT: the water-table bottom boundary (watertable_bc.h), a separate
// instantiation so the flux / zero-flux kernels keep their registers.
// lt: log's table in LDS.
template <class D, int G, bool WT, int K>
__device__ __forceinline__ int richards_group_by(const View &V, const Params &P, const ctsm_col_state &S, int c,
                                                 double dtime, int g, const double *lt, int gsz)
{
    constexpr bool RANGED = std::is_same<D, Recip>::value;
    const int GS = (G > 0) ? G : gsz;       // lanes in the group
    const int nl = S.nbedrock[V.c1(c)];
    if (nl < 2 || nl > MAX_NLEVSOI || nl > GS * K) return 1;

    // the layers of the lane; a layer below the column's last holds ordinary values,
    // which run through the trials without effect
    D mdz[K], ws[K], den[K];
    double bsw[K], hkc[K], suc[K], sink[K], liq[K];
    double Ud[K], Udu[K], Udl[K], Ub[K], f1[K];
    const double infl = S.qflx_infl[V.c1(c)];
    // watsat of the first layer of the next lane (for the interface below our last layer)
    D ws_nl = divisor<D>(1.0);
    bool outside = RANGED && !ordinary_steps(P, dtime);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int j = g * K + k;            // 0-based layer
        double dzk = 1.0, wsk = 1.0, denk = 1.0;
        bsw[k] = hkc[k] = suc[k] = 1.0;
        sink[k] = 0.0;
        liq[k] = 0.5;
        if (j < nl) {
            const int jj = j + 1;
            dzk = M_TO_MM * S.dz[V.sno(c, jj)];
            wsk = S.watsat[V.soi(c, jj)];
            bsw[k] = S.bsw[V.soi(c, jj)];
            suc[k] = S.sucsat[V.soi(c, jj)];
            sink[k] = S.qflx_rootsoi[V.soi(c, jj)];
            liq[k] = S.h2osoi_liq[V.sno(c, jj)];
            const double ic = S.icefrac[V.soi(c, jj)];
            double icei;
            if (j == nl - 1) {
                icei = ic;
            } else {
                icei = 0.5 * (ic + S.icefrac[V.soi(c, jj + 1)]);
                denk = M_TO_MM * (S.z[V.sno(c, jj + 1)] - S.z[V.sno(c, jj)]);
            }
            hkc[k] = cm_pow_tab(10.0, -(P.e_ice * icei), lt) * S.hksat[V.soi(c, jj)];
        }
        if (RANGED && !ordinary_layer(dzk, denk, wsk, bsw[k], suc[k], hkc[k])) outside = true;
        mdz[k] = divisor<D>(dzk);
        ws[k] = divisor<D>(wsk);
        den[k] = divisor<D>(denk);
    }
    {
        const int jn = (g + 1) * K;
        if (jn < nl) ws_nl = divisor<D>(S.watsat[V.soi(c, jn + 1)]);
    }
    if (RANGED && any_of_group(outside, GS)) return RICHARDS_RANGE;

    const bool zero_flux_bottom = (P.lower_bc == CTSM_BC_ZERO_FLUX);
    constexpr bool wt_bottom = WT;
    int jwt = 0;
    double zwt = 0.0, z_bot = 0.0, q_ka = 0.0, q_smp = 0.0;
    if (wt_bottom) {
        if (nl != V.nlevsoi || !S.zwt || !S.smpmin) return RICHARDS_BAD_COLUMN;
        jwt = watertable_layer(V, S, c);
        zwt = S.zwt[V.c1(c)];
        z_bot = S.z[V.sno(c, nl)];
    }
    const int bot_lane = (nl - 1) / K;
    int nsub = 0;
    // qcharge: the sum of the lane that holds the bottom layer
    double dtsub = dtime, dtdone = 0.0, qcharge = 0.0;
    int status = 0;

    for (;;) {
        nsub = nsub + 1;
        if (nsub > MAX_TRIALS) { status = 3; break; }
        const bool candidate = fabs(dtime - (dtdone + dtsub)) < P.verySmall;

        // ---- forward: properties, fluxes and rows of the owned layers.  No branch on
        //      the layer: the powers and divisions of all the lane's layers run
        //      through each other.
        double s2[K], smp[K], dsm[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const double vwc = fmax90(liq[k], 1.0e-6) / mdz[k];
            s2[k] = fmin90(vwc / ws[k], 1.0);
            s2[k] = fmax90(0.01, s2[k]);
            smp[k] = -(suc[k] * cm_pow_tab(s2[k], -bsw[k], lt));
            dsm[k] = (-(bsw[k] * smp[k]) / s2[k]) / ws[k];
        }
        // the next lane's first layer, for the interface below our last
        const double s2_nx = from_next(s2[0]), smp_nx = from_next(smp[0]), dsm_nx = from_next(dsm[0]);
        double hk_bot = 0.0, dhkdw_bot = 0.0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int j = g * K + k;
            const bool bottom = (j >= nl - 1);
            const double s2n = k + 1 < K ? s2[k + 1 < K ? k + 1 : k] : s2_nx;
            const double smpn = k + 1 < K ? smp[k + 1 < K ? k + 1 : k] : smp_nx;
            const double dsmn = k + 1 < K ? dsm[k + 1 < K ? k + 1 : k] : dsm_nx;
            const D wsn = k + 1 < K ? ws[k + 1 < K ? k + 1 : k] : ws_nl;
            double s1 = bottom ? s2[k] : 0.5 * (s2[k] + s2n);
            s1 = fmin90(s1, 1.0);
            s1 = fmax90(0.01, s1);
            const double e = 2.0 * bsw[k] + 3.0;
            const double hk = hkc[k] * cm_pow_tab(s1, e, lt);
            const double dhkdw = e * hk / s1;
            const double dhkds1 = 0.5 * dhkdw / ws[k];
            const double dhkds2 = 0.5 * dhkdw / wsn;
            const double num = smpn - smp[k];
            double qout = -(hk * num / den[k]) + hk;
            double dqodw1 = (hk * dsm[k] - dhkds1 * num) / den[k] + dhkds1;
            double dqodw2 = (-(hk * dsmn) - dhkds2 * num) / den[k] + dhkds2;
            if (bottom) {
                double hkb = hk, dhkb = dhkdw;
                if (zero_flux_bottom) { qout = 0.0; dqodw1 = 0.0; }
                else if (wt_bottom) {
                    if (jwt < V.nlevsoi) { qout = 0.0; dqodw1 = 0.0; }
                    else watertable_bottom_flux(hk, dhkdw, smp[k], dsm[k], ws[k].b, zwt, z_bot, qout, dqodw1);
                    // the sub-step's drainage is qout + dqodw1 * dwat
                    hkb = qout;
                    dhkb = dqodw1;
                }
                else { qout = hk; dqodw1 = dhkdw / ws[k]; }
                dqodw2 = 0.0;
                if (j == nl - 1) { hk_bot = hkb; dhkdw_bot = dhkb; }
            }
            if (candidate && j < nl) {
                if (wt_bottom) {
                    // what compute_qcharge reads of the last trial
                    if (j == jwt) q_ka = watertable_ka(fmax90(liq[k], 1.0e-6) / mdz[k], ws[k].b, hkc[k], bsw[k]);
                    if (j == (jwt > 1 ? jwt : 1) - 1) q_smp = smp[k];
                }
                S.smp_l[V.soi(c, j + 1)] = smp[k];
                S.hk_l[V.soi(c, j + 1)] = hk;
                S.qout[V.soi(c, j + 1)] = qout;
            }
            // this layer's outgoing flux terms; the row needs the incoming ones, which
            // belong to the layer above (filled in below)
            Ud[k] = qout; Udu[k] = dqodw1; Udl[k] = dqodw2;
        }
        // rows (a in Udl, b in Ud, c in Udu, r in Ub) and start-of-step net flux f1; the
        // incoming flux of our first layer is the previous lane's last outgoing one
        {
            const double qin_p = from_prev(Ud[K - 1]), dqidw0_p = from_prev(Udu[K - 1]), dqidw1_p = from_prev(Udl[K - 1]);
            double qin = (g == 0) ? infl : qin_p;
            double dqidw0 = (g == 0) ? 0.0 : dqidw0_p;
            double dqidw1 = (g == 0) ? 0.0 : dqidw1_p;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int j = g * K + k;
                const double qout = Ud[k], dqodw1 = Udu[k], dqodw2 = Udl[k], dtdz = dtsub / mdz[k];
                if (candidate && j < nl) S.qin[V.soi(c, j + 1)] = qin;
                const double fluxNet = qin - qout - sink[k];
                f1[k] = fluxNet;
                // (rows below the last are 0 1 0 | 0: they leave the last row as it is
                // and solve to 0)
                const bool in = j < nl;
                Ub[k] = in ? -(fluxNet * dtdz) : 0.0;                           // r
                Udl[k] = in ? dqidw0 * dtdz : 0.0;                              // a (unused for j = 0)
                Ud[k] = in ? -1.0 - (-dqidw1 + dqodw1) * dtdz : 1.0;            // b
                Udu[k] = j < nl - 1 ? -(dqodw2 * dtdz) : 0.0;                   // c
                qin = qout; dqidw0 = dqodw1; dqidw1 = dqodw2;
            }
        }
        // first row of the next lane (a, b, c, r) for our last elimination step
        // (moved by every lane, then cleared in the last one, which has no next row)
        double a_nx = from_next(Udl[0]);
        if (g == GS - 1) a_nx = 0.0;
        const double b_nx = from_next(Ud[0]), c_nx = from_next(Udu[0]), r_nx = from_next(Ub[0]);

        // ---- dgtsv elimination in G stages; (cd, cdu, cb) is the current, partly
        //      eliminated row.  Rows are rarely interchanged: those lanes redo the row.
        double cd = Ud[0], cdu = Udu[0], cb = Ub[0];
        bool singular = false;
#pragma unroll
        for (int s = 0; s < GS; ++s) {
            if (g == s) {
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int j = g * K + k;
                    if (!RANGED && j >= nl - 1) {
                        // a NaN or an infinity would pass from the last row to those below
                        if (j > nl - 1) continue;
                        Ud[k] = cd; Udu[k] = 0.0; Udl[k] = 0.0; Ub[k] = cb;
                        if (cd == 0.0) singular = true;
                        continue;
                    }
                    const double dl = k + 1 < K ? Udl[k + 1 < K ? k + 1 : k] : a_nx;
                    const double nd = k + 1 < K ? Ud[k + 1 < K ? k + 1 : k] : b_nx;
                    const double ndu = k + 1 < K ? Udu[k + 1 < K ? k + 1 : k] : c_nx;
                    const double nb = k + 1 < K ? Ub[k + 1 < K ? k + 1 : k] : r_nx;
                    const double fact = dl / divisor<D>(cd);
                    Ud[k] = cd; Udu[k] = cdu; Udl[k] = 0.0; Ub[k] = cb;
                    double td = nd - fact * cdu, tdu = ndu, tb = nb - fact * cb;
                    if (!(fabs(cd) > fabs(dl))) {
                        if (fabs(cd) >= fabs(dl)) {
                            // also the last row, whose dl is 0
                            if (cd == 0.0) singular = true;
                        } else {
                            const double fact_i = cd / dl;
                            Ud[k] = dl; Udu[k] = nd; Ub[k] = nb;
                            td = cdu - fact_i * nd;
                            tb = cb - fact_i * nb;
                            if (j + 1 != nl - 1) { Udl[k] = ndu; tdu = -fact_i * ndu; }
                        }
                    }
                    cd = td; cdu = tdu; cb = tb;
                }
            }
            if (s + 1 < GS) {
                cd = from_prev(cd);
                cdu = from_prev(cdu);
                cb = from_prev(cb);
            }
        }

        // ---- back substitution in reverse stages (the reciprocals of the diagonal
        //      beforehand, outside the chain), then the error estimate
        D d[K];
#pragma unroll
        for (int k = 0; k < K; ++k) d[k] = divisor<D>(Ud[k]);
        double x1 = 0.0, x2 = 0.0;
#pragma unroll
        for (int s = GS - 1; s >= 0; --s) {
            if (g == s) {
#pragma unroll
                for (int k = K - 1; k >= 0; --k) {
                    double r = Ub[k] - Udu[k] * x1 - Udl[k] * x2;
                    if (!RANGED) {
                        // and from the rows below the last to it
                        const int j = g * K + k;
                        if (j == nl - 1) r = Ub[k];
                        if (j == nl - 2) r = Ub[k] - Udu[k] * x1;
                    }
                    const double x = r / d[k];
                    Ub[k] = x;
                    x2 = x1;
                    x1 = x;
                }
            }
            if (s > 0) {
                x1 = from_next(x1);
                x2 = from_next(x2);
            }
        }
        if (RANGED) {
            // the numerators of the substitution, and what the water content can become
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (!(fabs(Ub[k] * Ud[k]) >= 0x1.0p-900 && fabs(Ub[k]) < 0x1.0p+200) && Ub[k] != 0.0) outside = true;
        }
        // any lane singular -> the whole column fails
        if (any_of_group(singular || outside, GS)) {
            if (!RANGED || any_of_group(singular, GS)) { status = 2; break; }
            return RICHARDS_RANGE;
        }
        double emax = 0.0, dwat_bot = 0.0;
        bool top_nan = false;
#pragma unroll
        for (int k = K - 1; k >= 0; --k) {
            const int j = g * K + k;
            const double x = Ub[k], dtdz = dtsub / mdz[k];
            const double ev = fabs(f1[k] - x / dtdz) * dtsub * 0.5;
            if (j == nl - 1) dwat_bot = x;
            if (j < nl && ev > emax) emax = ev;
            if (j == 0) top_nan = ev != ev;
        }
        // group max of the error estimate (each owned layer's value; empty lanes hold 0 <=
        // any).  As in the reference's maxval from the first layer on, a NaN there stays
        // and one below it does not count; the solve with reciprocals meets none.
        double errorMax = group_max(emax, GS);
        if (!RANGED && any_of_group(top_nan, GS)) errorMax = NAN;
        if (errorMax > P.xTolerUpper && dtsub > P.dtmin) {
            dtsub = fmax90(dtsub / 2.0, P.dtmin);
            continue;
        }
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (g * K + k < nl) liq[k] = liq[k] + Ub[k] * mdz[k].b;
        const double qcTemp = zero_flux_bottom ? 0.0 : hk_bot + dhkdw_bot * dwat_bot;
        qcharge = qcharge + qcTemp * (dtsub / dtime);
        dtdone = dtdone + dtsub;
        if (fabs(dtime - dtdone) < P.verySmall) break;
        if (errorMax < P.xTolerLower) dtsub = dtsub * 2.0;
        dtsub = fmin90(dtsub, dtime - dtdone);
    }
    if (status) return status;

    if (wt_bottom && jwt < V.nlevsoi) {
        const double ka = gshfl(q_ka, jwt / K, GS);
        const double smp_w = gshfl(q_smp, ((jwt > 1 ? jwt : 1) - 1) / K, GS);
        qcharge = watertable_qcharge(V, S, c, jwt, ka, smp_w, dtime);
    }
    if (g == bot_lane) {
        S.num_substeps[V.c1(c)] = (double)nsub;
        S.qcharge[V.c1(c)] = qcharge;
    }
    // over-saturated layers push water upward (:1405-1409), bottom lane first
    double carry = 0.0;
#pragma unroll
    for (int s = GS - 1; s >= 0; --s) {
        if (g == s) {
#pragma unroll
            for (int k = K - 1; k >= 0; --k) {
                const int j = g * K + k;
                if (j < nl) {
                    const double w = liq[k] + carry;
                    if (j == 0) {
                        liq[k] = w;
                    } else {
                        const double cap = S.eff_porosity[V.soi(c, j + 1)] * M_TO_MM * S.dz[V.sno(c, j + 1)];
                        carry = fmax90(w - cap, 0.0);
                        liq[k] = fmin90(cap, w);
                    }
                }
            }
        }
        carry = from_next(carry);
    }
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (g * K + k < nl) S.h2osoi_liq[V.sno(c, g * K + k + 1)] = liq[k];
    return 0;
}

template <int G, bool WT = false, int K = (MAX_NLEVSOI + (G > 0 ? G : 1) - 1) / (G > 0 ? G : 1)>
__device__ __forceinline__ int richards_group(const View &V, const Params &P, const ctsm_col_state &S, int c,
                                              double dtime, int g, const double *lt, int gsz = G)
{
    int rc = richards_group_by<Recip, G, WT, K>(V, P, S, c, dtime, g, lt, gsz);
    if (rc == RICHARDS_RANGE) rc = richards_group_by<Plain, G, WT, K>(V, P, S, c, dtime, g, lt, gsz);
    return rc;
}

}  // namespace ctsm
