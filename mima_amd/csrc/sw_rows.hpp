// SW gas optics as weighted table rows and the clear-sky layer optics, for
// kernels whose lane is one column and holds several g-points in registers (as
// lw_rows.hpp for the longwave).
//
// taumol_sw's optical depths (rrtmg_sw_taumol.f90) are linear in their table
// values with weights that do not depend on the g-point.
//
// Contraction is off here, and multiply-adds are written out: a column's result
// must not depend on the kernel that the size of the call selects.
#pragma once
#include <hip/hip_runtime.h>

#include "rrtmg_device.hpp"
#include "rrtmg_types.hpp"
#include "sw_optics.hpp"

namespace rrtmg {

#pragma clang fp contract(off)

// The rows of one (layer, column) of band JB: gas(offset, row, weight) for the
// gas optical depth, ray(offset, row, weight) for the Rayleigh one; returns what
// both lack, the parts without g-dependence.  Rows are 1-based as the
// reference's indices; the band formulas and their lines are those of sw_gas.
template <typename Real>
struct SwFlat {
    Real taug, taur;
};
template <int JB, typename Real, typename FG, typename FR>
__device__ __forceinline__ SwFlat<Real> sw_rows(const SwBand &B, const SwLayer<Real> &c, bool lower, FG &&gas, FR &&ray)
{
    constexpr int NA = SW_NSPA[JB - 16], NB = SW_NSPB[JB - 16];
    const int ind0 = lower ? ((c.jp - 1) * 5 + (c.jt - 1)) * NA : ((c.jp - 13) * 5 + (c.jt - 1)) * NB;
    const int ind1 = lower ? (c.jp * 5 + (c.jt1 - 1)) * NA : ((c.jp - 12) * 5 + (c.jt1 - 1)) * NB;
    SwFlat<Real> flat{(Real)0, (Real)0};
    auto pair = [&](int off, int row, int step, Real m, Real f) {
        const Real mf = m * f;
        gas(off, row, m - mf);
        gas(off, row + step, mf);
    };
    auto four = [&](int off, Real m) {
        gas(off, ind0 + 1, m * c.fac00);
        gas(off, ind0 + 2, m * c.fac10);
        gas(off, ind1 + 1, m * c.fac01);
        gas(off, ind1 + 2, m * c.fac11);
    };
    // (eta, T, p) interpolation of a pair of species; s1: rows per temperature
    auto eight = [&](int off, Real cola, Real colb, Real rat, Real mult, int s1) {
        Real comb, fs;
        int js;
        sw_eta<Real>(cola, colb, rat, mult, comb, js, fs);
        pair(off, ind0 + js, 1, comb * c.fac00, fs);
        pair(off, ind0 + js + s1, 1, comb * c.fac10, fs);
        pair(off, ind1 + js, 1, comb * c.fac01, fs);
        pair(off, ind1 + js + s1, 1, comb * c.fac11, fs);
    };
    auto foreign = [&]() { pair(B.forref, c.indf, 1, c.colh2o * c.forfac, c.forfrac); };
    auto cont = [&]() {
        pair(B.selfref, c.inds, 1, c.colh2o * c.selffac, c.selffrac);
        foreign();
    };
    if constexpr (JB == 23 || JB == 25 || JB == 26 || JB == 27)
        ray(B.raylg, 1, c.colmol);
    else if constexpr (JB != 24)
        flat.taur = c.colmol * (Real)B.rayl;
    if constexpr (JB == 16 || JB == 18 || JB == 19) {
        constexpr double rat = JB == 16 ? 252.131 : JB == 18 ? 38.9589 : 5.49281;
        const Real other = JB == 19 ? c.colco2 : c.colch4;
        if (lower) {
            eight(B.absa, c.colh2o, other, (Real)rat, (Real)8, 9);
            cont();
        } else {
            four(B.absb, other);
        }
    } else if constexpr (JB == 17 || JB == 21) {
        constexpr double rat = JB == 17 ? 0.364641 : 0.0045321;
        if (lower) {
            eight(B.absa, c.colh2o, c.colco2, (Real)rat, (Real)8, 9);
            cont();
        } else {
            eight(B.absb, c.colh2o, c.colco2, (Real)rat, (Real)4, 5);
            foreign();
        }
    } else if constexpr (JB == 20) {
        if (lower) {
            four(B.absa, c.colh2o);
            cont();
        } else {
            four(B.absb, c.colh2o);
            foreign();
        }
        gas(B.absch4, 1, c.colch4);
    } else if constexpr (JB == 22) {
        flat.taug = fdiv((Real)4.35e-4 * c.colo2, (Real)(350.0 * 2.0));
        if (lower) {
            eight(B.absa, c.colh2o, c.colo2, (Real)(1.6 * 0.022708), (Real)8, 9);
            cont();
        } else {
            four(B.absb, c.colo2 * (Real)1.6);
        }
    } else if constexpr (JB == 23) {
        if (lower) {
            four(B.absa, c.colh2o * (Real)1.029);
            cont();
        }
    } else if constexpr (JB == 24) {
        if (lower) {
            Real comb, fs;
            int js;
            sw_eta<Real>(c.colh2o, c.colo2, (Real)0.124692, (Real)8, comb, js, fs);
            const Real mf = c.colmol * fs;
            ray(B.rayla, js, c.colmol - mf);
            ray(B.rayla, js + 1, mf);
            eight(B.absa, c.colh2o, c.colo2, (Real)0.124692, (Real)8, 9);
            gas(B.abso3a, 1, c.colo3);
            cont();
        } else {
            ray(B.raylb, 1, c.colmol);
            four(B.absb, c.colo2);
            gas(B.abso3b, 1, c.colo3);
        }
    } else if constexpr (JB == 25) {
        if (lower) {
            four(B.absa, c.colh2o);
            gas(B.abso3a, 1, c.colo3);
        } else {
            gas(B.abso3b, 1, c.colo3);
        }
    } else if constexpr (JB == 27) {
        four(lower ? B.absa : B.absb, c.colo3);
    } else if constexpr (JB == 28) {
        if (lower)
            eight(B.absa, c.colo3, c.colo2, (Real)6.67029e-07, (Real)8, 9);
        else
            eight(B.absb, c.colo3, c.colo2, (Real)6.67029e-07, (Real)4, 5);
    } else if constexpr (JB == 29) {
        if (lower) {
            four(B.absa, c.colh2o);
            cont();
            gas(B.absco2, 1, c.colco2);
        } else {
            four(B.absb, c.colco2);
            gas(B.absh2o, 1, c.colh2o);
        }
    }
    return flat;
}

// exp(-x): series below 0.06, table entry above
__device__ __forceinline__ float sw_beam(float x, const float *__restrict__ tbl)
{
    const float e = at32(tbl, (unsigned)tbl_index(x));
    return x <= 0.06f ? fmaf(0.5f * x, x, 1.f - x) : e;
}

// PIFM two-stream layer of a clear sky (rrtmg_sw_reftra.f90:127-303 with
// asymmetry 0, so gamma3 = gamma4 = 1/2 and za1 = za2) and its direct-beam
// transmittance; imu: 1 / mu.  FP32 as reftra in sw_optics.hpp arranges it:
// the eigenvalue from 1 - w, numerators and denominator multiplied by zem1,
// divisions as products with the reciprocal; k: the eigenvalue.  FP64 keeps the
// reference's expressions (tbl NULL: the function the table holds).
template <typename Real>
struct SwOptics {
    Real r, rd, t, td, dbt;
};
__device__ __forceinline__ SwOptics<float> sw_two_stream(float tau, float w, float k, float mu, float imu,
                                                        const float *__restrict__ tbl)
{
    SwOptics<float> o;
    const float g1 = fmaf(w, -1.25f, 2.f), g2 = 0.75f * w;
    o.dbt = sw_beam(fminf(tau * imu, 500.f), tbl);
    if (w >= 0.9999995f) {
        const float za1 = fmaf(g1, mu, -0.5f), zgt = g1 * tau;
        const float rz = fdiv(1.f, 1.f + zgt);
        const bool thin = o.dbt == 1.f;
        o.r = thin ? 0.f : fmaf(-za1, 1.f - o.dbt, zgt) * rz;
        o.rd = thin ? 0.f : zgt * rz;
        o.t = 1.f - o.r;
        o.td = 1.f - o.rd;
        return o;
    }
    const float a = 0.5f * (g1 + g2), hk = 0.5f * k, k2 = 2.f * k;
    const float kp = fmaf(k, mu, 1.f), km = fmaf(-k, mu, 1.f), apk = a + hk, amk = a - hk, am = a * mu;
    const float zkg = k + g1, kmg = k - g1, pp = kp * km;
    const float e1 = sw_beam(fminf(k * tau, 500.f), tbl), e2 = o.dbt, ee = e1 * e1;
    const float d = fmaf(kmg, ee, zkg);  // zdend's denominator; zdenr zem1 = pp d
    const float den = pp * d, lim = 1.e-08f * e1;
    const bool tiny = den >= -lim && den <= lim;
    const float wr = w * fdiv(1.f, den);
    const float nr = fmaf(-k2 * (0.5f - am), e2 * e1, fmaf(-kp * amk, ee, km * apk));
    const float nt = fmaf(e2, fmaf(-km * amk, ee, kp * apk), -k2 * (0.5f + am) * e1);
    o.r = tiny ? 1.e-08f : nr * wr;
    o.t = tiny ? e2 : fmaf(-nt, wr, e2);
    const float rd = fdiv(1.f, d);
    o.rd = g2 * (1.f - ee) * rd;
    o.td = k2 * e1 * rd;
    return o;
}
__device__ __forceinline__ SwOptics<double> sw_two_stream(double tau, double w, double, double mu, double,
                                                         const double *__restrict__ tbl)
{
    SwOptics<double> o;
    const double eps = 1.e-08;
    const double g1 = (8.0 - w * 5.0) * 0.25, g2 = 3.0 * w * 0.25;
    auto beam = [&](double x) {
        if (!tbl) return tbl_exp(x, tbl);
        return x <= 0.06 ? 1.0 - x + 0.5 * x * x : at32(tbl, (unsigned)tbl_index(x));
    };
    const double e2 = beam(fmin(tau / mu, 500.0));
    o.dbt = e2;
    if (w >= 0.9999995) {
        const double za1 = g1 * mu - 0.5, zgt = g1 * tau;
        const bool thin = e2 == 1.0;
        o.r = thin ? 0.0 : (zgt - za1 * (1.0 - e2)) / (1.0 + zgt);
        o.rd = thin ? 0.0 : zgt / (1.0 + zgt);
        o.t = 1.0 - o.r;
        o.td = 1.0 - o.rd;
        return o;
    }
    const double a = g1 * 0.5 + g2 * 0.5, k = sqrt(g1 * g1 - g2 * g2);
    const double rp = k * mu, kp = 1.0 + rp, km = 1.0 - rp, k2 = 2.0 * k, pp = 1.0 - rp * rp, zkg = k + g1;
    const double e1 = beam(fmin(k * tau, 500.0));
    const double ep1 = 1.0 / e1, ep2 = 1.0 / e2;
    const double den = pp * zkg * ep1 + pp * (k - g1) * e1;
    if (den >= -eps && den <= eps) {
        o.r = eps;
        o.t = e2;
    } else {
        o.r = w * (km * (a + k * 0.5) * ep1 - kp * (a - k * 0.5) * e1 - k2 * (0.5 - a * mu) * e2) / den;
        o.t = e2 - e2 * w * (kp * (a + k * 0.5) * ep1 - km * (a - k * 0.5) * e1 - k2 * (0.5 + a * mu) * ep2) / den;
    }
    const double ee = e1 * e1, beta = (g1 - k) / zkg, dend = 1.0 / ((1.0 - beta * ee) * zkg);
    o.rd = g2 * (1.0 - ee) * dend;
    o.td = k2 * e1 * dend;
    return o;
}

// The clear-sky optics of one (layer, g-point).  FP32 takes reftra in FP64
// where |1 - k mu| < 0.01 w: there the direct-beam quotient, whose numerator and
// denominator vanish at k mu = 1 with absolute errors of the FP32 epsilon, is off
// by more than 6e-6 once multiplied by the single-scattering albedo w (an
// absorbing g-point, k near 2, sits at k mu = 1 through whole columns of
// mu = 1/2, and scatters nothing).
template <typename Real>
__device__ __forceinline__ SwOptics<Real> sw_clear_layer(Real taug, Real taur, Real mu, Real imu,
                                                         const Real *__restrict__ tbl)
{
    const Real tau = taur + taug;
    if constexpr (sizeof(Real) == 4) {
        const Real rt = fdiv((Real)1, tau);
        const Real w = taur * rt, omw = taug * rt;
        // k = sqrt(2 (1 - w) (gamma1 + gamma2)), free of the cancellation of
        // gamma1^2 - gamma2^2
        const Real k = __builtin_amdgcn_sqrtf(omw * fmaf(w, -1.f, 4.f));
        SwOptics<Real> o = sw_two_stream(tau, w, k, mu, imu, tbl);
        if (fabs(fmaf(-k, mu, 1.f)) < (Real)0.01 * w) {
            const LayerOptics<float> x = reftra_island(taug, taur, mu, tbl);
            o.r = x.r;
            o.rd = x.rd;
            o.t = x.t;
            o.td = x.td;
        }
        return o;
    } else {
        return sw_two_stream(tau, taur / tau, (Real)0, mu, imu, tbl);
    }
}

#pragma clang fp contract(fast)

}  // namespace rrtmg
