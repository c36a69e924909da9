// Backward band body of the clear-sky LW path (two sweeps, lw_vjp.hip) and its
// loaders, shared by the LW backward band kernels and the fused LW+SW
// forward+backward kernel (fused.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "lw_optics.hpp"
#include "lw_rows.hpp"
#include "lw_unit.hpp"
#include "mdual.hpp"
#include "rrtmg_device.hpp"

namespace rrtmg {

// a layer's coefficients with the derivatives each can have (LW_DMASK)
template <typename Real>
struct LwLayerD {
#define LWD(f, F) typename MField<Real, LW_DMASK[F]>::type f
#define LWD_FIELDS(X)                                                                                              \
    X(fac00, LWF_FAC00); X(fac01, LWF_FAC01); X(fac10, LWF_FAC10); X(fac11, LWF_FAC11);                            \
    X(colh2o, LWF_COLH2O); X(colco2, LWF_COLCO2); X(colo3, LWF_COLO3); X(coln2o, LWF_COLN2O);                      \
    X(colco, LWF_COLCO); X(colch4, LWF_COLCH4); X(colo2, LWF_COLO2); X(colbrd, LWF_COLBRD);                        \
    X(selffac, LWF_SELFFAC); X(selffrac, LWF_SELFFRAC); X(forfac, LWF_FORFAC); X(forfrac, LWF_FORFRAC);            \
    X(minorfrac, LWF_MINORFRAC); X(scaleminor, LWF_SCALEMINOR); X(scaleminorn2, LWF_SCALEMINORN2);                 \
    X(coldry, LWF_COLDRY); X(pavel, LWF_PAVEL); X(wx1, LWF_WX1); X(wx2, LWF_WX2); X(wx3, LWF_WX3);                 \
    X(wx4, LWF_WX4)
    LWD_FIELDS(LWD);
#undef LWD
    Real tlayfrac;  // its derivative is 1
    int jp, jt, jt1, inds, indf, indm, indlay;
};

// the field's derivatives, from der_offset on in the layer's groups of four
template <unsigned M, typename Real, typename G>
__device__ __forceinline__ auto lw_field_d(Real v, const G *g, int o)
{
    if constexpr (M == 0) {
        return v;
    } else {
        MDual<Real, M> r;
        r.v = v;
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (M >> k & 1u) {
                r.d[k] = g[o / 4].x[o % 4];
                ++o;
            }
        return r;
    }
}

// a layer's groups of four in the prep's two buffers, as loaded; groups a band
// does not use are not loaded
template <typename Real>
struct LwGroupsD {
    struct alignas(16) Group {
        Real x[4];
    };
    Group v[LWF_GROUPS], d[LWD_GROUPS];
    int ipk;
    __device__ __forceinline__ void load(const Real *__restrict__ dco, const Real *__restrict__ dde,
                                         const int *__restrict__ pk, int lay, int col, int ncol)
    {
        const Group *vb = (const Group *)dco + (size_t)lay * LWF_GROUPS * ncol;
        const Group *db = (const Group *)dde + (size_t)lay * LWD_GROUPS * ncol;
#pragma unroll
        for (int k = 0; k < LWF_GROUPS; ++k)
            v[k] = *(const Group *)((const char *)(vb + (size_t)k * ncol) + (LaneOffset<Real>)col * sizeof(Group));
#pragma unroll
        for (int k = 0; k < LWD_GROUPS; ++k)
            d[k] = *(const Group *)((const char *)(db + (size_t)k * ncol) + (LaneOffset<Real>)col * sizeof(Group));
        ipk = at32(pk, (unsigned)(lay * ncol + col));
    }
    __device__ __forceinline__ void unpack(LwLayerD<Real> &c) const
    {
#define LDD(f, F) c.f = lw_field_d<LW_DMASK[F], Real>(v[(F) / 4].x[(F) % 4], d, der_offset(LW_DMASK, F))
        LWD_FIELDS(LDD);
#undef LDD
        c.tlayfrac = v[LWF_TLAYFRAC / 4].x[LWF_TLAYFRAC % 4];
        c.jp = unpack_jp(ipk);
        c.jt = unpack_jt(ipk);
        c.jt1 = unpack_jt1(ipk);
        c.inds = unpack_inds(ipk);
        c.indf = unpack_indf(ipk);
        c.indm = unpack_indm(ipk);
        c.indlay = unpack_indlay(ipk);
    }
};
#undef LWD_FIELDS

// contraction off, as in lw_rows.hpp
#pragma clang fp contract(off)

// sums over the lanes of a band, valid on the first one of each column
template <int BAND, int N, typename Real>
__device__ __forceinline__ void lw_lane_sums(Real (&v)[N])
{
    constexpr int LPC = LwLanes<BAND>::LPC;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        if constexpr (LPC == 2) v[i] = v[i] + __shfl_down(v[i], 1);
        if constexpr (LPC == 3) v[i] = v[i] + (__shfl_down(v[i], 1) + __shfl_down(v[i], 2));
        if constexpr (LPC == 4) {
            v[i] = v[i] + __shfl_down(v[i], 1);
            v[i] = v[i] + __shfl_down(v[i], 2);
        }
    }
}

// d/dtau of the transmittance 1 - exp(-tau) and of the tau transition function
// (lw_rt_exact).  FP32: exp(-tau) from the hardware's exp2 with the product's
// rounding error added back; the transition function's derivative, below 1.5,
// from its series (sum (2n-1) 2 B_2n tau^(2n-2) / (2n)!, B the Bernoulli
// numbers; the first term left out is 3e-9), above from
// 2/tau^2 - 2 e/(1 - e)^2, which loses digits to cancellation below.
template <typename Real>
struct LwDRT {
    Real datr, dtf;
};
__device__ __forceinline__ LwDRT<double> lw_drt(double od)
{
    const LwRT<double> x = lw_rt_exact(od, true);
    return {x.datr, x.dtf};
}
__device__ __forceinline__ LwDRT<float> lw_drt(float od)
{
    const float log2e = 1.44269502f, log2e_lo = 1.92596303e-8f;
    const float t = od * log2e, lo = fma(od, log2e, -t) + od * log2e_lo;
    const float e0 = __builtin_amdgcn_exp2f(-t), e = fma(-0.693147181f * lo, e0, e0);
    const float x2 = od * od;
    float s = fma(3.4795e-10f, x2, -1.162518e-8f);
    s = fma(s, x2, (float)(1. / 2661120.));
    s = fma(s, x2, (float)(-1. / 86400.));
    s = fma(s, x2, (float)(1. / 3024.));
    s = fma(s, x2, (float)(-1. / 120.));
    s = fma(s, x2, (float)(1. / 6.));
    const float io = __builtin_amdgcn_rcpf(od), q = __builtin_amdgcn_rcpf(1.f - e);
    return {e, od < 1.5f ? s : 2.f * fma(io, io, -(e * q) * q)};
}

// Backward of one unit of a wave (its forward is that of u, and so are the band
// fluxes, where w.bflux is given).
//
// Gradient with respect to a layer: the optical depth of g-point g is
// sum_r W_r K_r[g] (lw_rows), so sum_g a_g dtau_g/dx = sum_r dW_r/dx (sum_g a_g
// K_r[g]): the weights' derivatives are formed once for the lane's g-points
// (Gather).
template <int BAND, typename Real>
struct LwVjpUnit {
    using Unit = LwUnit<BAND, Real>;
    static constexpr int GC = Unit::GC, NG = Unit::NG;
    using Vec = GVec<GC, Real>;
    const Unit u;
    const LwVjpWork &w;
    Real *gpart, *glev, *gsc;
    const Real *cu, *cd;
    size_t n2;
    Real cband;
    __device__ __forceinline__ LwVjpUnit(const Unit &u_, const LwVjpWork &w_) : u(u_), w(w_)
    {
        const size_t ncol = u.in.ncol, n3 = (size_t)(u.in.nlay + 1) * ncol;
        n2 = (size_t)u.in.nlay * ncol;
        gpart = (Real *)w.gpart + (size_t)(BAND - 1) * 3 * n2;
        glev = (Real *)w.glev + (size_t)(BAND - 1) * n3;
        gsc = (Real *)w.gsc + (size_t)(BAND - 1) * 2 * ncol;
        cu = (const Real *)w.cot;
        cd = cu + n3;
        // radiance cotangents of this band: flux = fluxfac * sum_b 0.5 delwave_b sum_g rad
        cband = (Real)(2.0 * asin(1.0) * 2.e4 * 0.5 * u.B.delwave);
    }
    __device__ __forceinline__ Real ru(int k) const { return at32(cu, (unsigned)(k * u.in.ncol + u.col)) * cband; }
    __device__ __forceinline__ Real rd(int k) const { return at32(cd, (unsigned)(k * u.in.ncol + u.col)) * cband; }
    // g-points past the band's end (dummies of its last lane) have no adjoints
    __device__ __forceinline__ Real live(int j, Real x) const { return NG % GC == 0 || u.g0 + j < NG ? x : (Real)0; }
    __device__ __forceinline__ Real plkslope(int i) const { return at32(u.plk, (unsigned)i) - at32(u.plk, (unsigned)(i - 1)); }
    // What the rows of a layer add to its gradients g: an interpolation's
    // derivative takes the difference of its rows, not the difference of their
    // sums, which are many times larger (lw_rows).  S: sum over the lane's
    // g-points of the adjoint times the row; a: the adjoints.
    struct Gather {
        using Whole = void;
        const Real *ktab, *ktab_b;
        const int g0;
        const Real (&a)[GC];
        Real (&g)[3];
        template <int K>
        __device__ __forceinline__ void row(Real (&k)[GC], std::integral_constant<int, K>, int off, int r) const
        {
            load_row<NG>(k, K == LW_ABSB ? ktab_b : ktab, (unsigned)(off + (r - 1) * NG + g0));
        }
        __device__ __forceinline__ Real dot(const Real (&k)[GC]) const
        {
            Real t = (Real)0;
#pragma unroll
            for (int j = 0; j < GC; ++j) t = fma(a[j], k[j], t);
            return t;
        }
        __device__ __forceinline__ Real dot(const Real (&k)[GC], const Real (&l)[GC]) const  // of k - l
        {
            Real t = (Real)0;
#pragma unroll
            for (int j = 0; j < GC; ++j) t = fma(a[j], k[j] - l[j], t);
            return t;
        }
        template <int K, typename W>
        __device__ __forceinline__ void operator()(std::integral_constant<int, K> where, int off, int r, const W &m) const
        {
            Real k[GC];
            row(k, where, off, r);
            md_gather(g, dot(k), m);
        }
        template <int K, typename W, typename F>
        __device__ __forceinline__ void operator()(std::integral_constant<int, K> where, int off, int r, int step, const W &m, const F &f) const
        {
            Real k0[GC], k1[GC];
            row(k0, where, off, r);
            row(k1, where, off, r + step);
            const Real s0 = dot(k0), s1 = dot(k1, k0);
            md_gather(g, fma(val(f), s1, s0), m);
            md_gather(g, val(m) * s1, f);
        }
        template <int K, typename W, typename F>
        __device__ __forceinline__ void operator()(std::integral_constant<int, K> where, int off, int r, const W &m, const F &w0, const F &,
                                                   const F &w2) const
        {
            Real k0[GC], k1[GC], k2[GC];
            row(k0, where, off, r);
            row(k1, where, off, r + 1);
            row(k2, where, off, r + 2);
            const Real s1 = dot(k1), s0 = dot(k0, k1), s2 = dot(k2, k1);
            md_gather(g, fma(val(w0), s0, fma(val(w2), s2, s1)), m);
            md_gather(g, val(m) * s0, w0);
            md_gather(g, val(m) * s2, w2);
        }
        template <int K, typename W, typename M, typename F>
        __device__ __forceinline__ void operator()(std::integral_constant<int, K> where, int off, int r, int neta, const W &m, const M &mf,
                                                   const F &fs, int) const
        {
            Real k0[GC], k1[GC], l0[GC], l1[GC];
            row(k0, where, off, r);
            row(k1, where, off, r + 1);
            row(l0, where, off, r + neta);
            row(l1, where, off, r + neta + 1);
            const Real s0 = dot(k0), s1 = dot(k1, k0), d0 = dot(l0, k0), t1 = dot(l1, l0);
            const Real low = fma(val(fs), s1, s0), up = fma(val(fs), t1 - s1, d0);
            md_gather(g, fma(val(mf), up, low), m);
            md_gather(g, val(m) * up, mf);
            md_gather(g, val(m) * fma(val(mf), t1 - s1, s1), fs);
        }
        // the Planck fraction's rows
        __device__ __forceinline__ void operator()(int, int, Real) const {}
        template <typename F>
        __device__ __forceinline__ void operator()(int off, int r, int step, const F &f) const
        {
            Real k0[GC], k1[GC];
            row(k0, LwOther{}, off, r);
            row(k1, LwOther{}, off, r + step);
            md_gather(g, dot(k1, k0), f);
        }
    };
    // a layer's local part: what one layer adds to the gradients, and the
    // sweeps past it
    struct Local {
        Real g[3];           // T, q, O3 of the layer, over the lane's g-points
        Real dn, up, sec;    // levels below and above; sum a_od od
    };
    // p: the layer; od: optical depths; r, ar: downward radiances entering the layer and
    // adjoints of the upward ones leaving it; rad, a: upward radiances entering
    // it and adjoints of the downward ones leaving it, then those past it; af:
    // the surface's adjoints of the lowest layer's Planck fractions, 0 elsewhere
    __device__ __forceinline__ void load(LwGroupsD<Real> &p, int lev) const
    {
        p.load((const Real *)w.dcoef, (const Real *)w.dder, w.ipk, lev - 1, u.col, u.in.ncol);
    }
    __device__ __forceinline__ Local local(int lev, const LwGroupsD<Real> &p, const Vec &od, const Vec &r, const Vec &ar, const Vec &af,
                                           Real plev_dn, Real plev_up, Real (&rad)[GC], Real (&a)[GC]) const
    {
        LwLayerD<Real> c;
        p.unpack(c);
        const bool lower = lev <= u.laytrop;
        Real fr[GC], a_tg[GC], a_pf[GC];
#pragma unroll
        for (int j = 0; j < GC; ++j) fr[j] = (Real)0;
        lw_fracs<BAND, Real>(u.B, u.cst, c, lower, [&](int off, int rr, const auto &wt) {
            Real k[GC];
            load_row<NG>(k, u.ktab, (unsigned)(off + (rr - 1) * NG + u.g0));
#pragma unroll
            for (int j = 0; j < GC; ++j) fr[j] = fma(val(wt), k[j], fr[j]);
        });
        const Real slope = plkslope(c.indlay), blay = fma(c.tlayfrac, slope, at32(u.plk, (unsigned)(c.indlay - 1)));
        const Real dpdn = plev_dn - blay, dpup = plev_up - blay;
        const Real ct = lev < u.in.nlay ? rd(lev) : (Real)0;
        Local o{};
        Real a_blay = (Real)0;
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            Real atr, tf;
            u.transmit(od.x[j], atr, tf);
            // the derivatives of the smooth functions that the series and the
            // tables stand for, 1 - exp(-tau) and the transition function
            const LwDRT<Real> x = lw_drt(od.x[j]);
            const Real sdn = fma(tf, dpdn, blay), sup = fma(tf, dpup, blay);
            const Real bbd = fr[j] * sdn, bbu = fr[j] * sup;
            const Real a_bbd = a[j] * atr, a_bbu = ar.x[j] * atr;
            const Real a_atr = fma(a[j], bbd - r.x[j], ar.x[j] * (bbu - rad[j]));
            rad[j] = fma(bbu - rad[j], atr, rad[j]);
            a[j] = fma(-a[j], atr, a[j]) + live(j, ct);
            a_pf[j] = fma(a_bbd, sdn, fma(a_bbu, sup, af.x[j]));
            const Real a_tf = fr[j] * fma(a_bbd, dpdn, a_bbu * dpup);
            a_blay = fma(fr[j] * ((Real)1 - tf), a_bbd + a_bbu, a_blay);
            o.dn = fma(a_bbd * fr[j], tf, o.dn);
            o.up = fma(a_bbu * fr[j], tf, o.up);
            const Real a_od = od.x[j] > (Real)0 ? fma(a_atr, x.datr, a_tf * x.dtf) : (Real)0;
            o.sec = fma(a_od, od.x[j], o.sec);
            a_tg[j] = a_od * u.secdiff;
            if constexpr (BAND == 4 || BAND == 7) a_tg[j] = a_tg[j] * lw_gfactor<BAND, Real>(u.g0 + j, lower);
        }
        o.g[0] = a_blay * slope;
        lw_rows<BAND, Real>(u.B, u.cst, c, lower, Gather{u.ktab, u.ktab_b, u.g0, a_tg, o.g});
        lw_fracs<BAND, Real>(u.B, u.cst, c, lower, Gather{u.ktab, u.ktab, u.g0, a_pf, o.g});
        return o;
    }
    // surface: rad and a of the downward sweep into those of the upward one;
    // a_tb, af: the adjoints of the surface temperature and the Planck fractions
    __device__ __forceinline__ void surface(const Real (&fr)[GC], Real (&rad)[GC], Real (&a)[GC], Real &a_tb,
                                            Vec &af) const
    {
        const double tbound = u.w.colscal[(size_t)u.in.ncol + u.col];
        const Real semiss = (Real)u.in.emis[(size_t)(BAND - 1) * u.in.ncol + u.col];
        const Real dplankbnd = semiss * plkslope(clampi((int)(tbound - 159.0), 1, 180)), c0 = rd(0);
        const Real emit = u.plankbnd();
        u.surface(fr, rad);
        a_tb = (Real)0;
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            af.x[j] = a[j] * emit;
            a_tb = fma(a[j] * fr[j], dplankbnd, a_tb);
            a[j] = fma(a[j], (Real)1 - semiss, live(j, c0));
        }
    }
    __device__ __forceinline__ void store_layer(const Local &o, int lev) const
    {
        Real v[3] = {o.g[0], o.g[1], o.g[2]};
        lw_lane_sums<BAND>(v);
        if (u.first) {
            const unsigned ix = (unsigned)((lev - 1) * u.in.ncol + u.col);
            at32(gpart, ix) = v[0];
            at32(gpart + n2, ix) = v[1];
            at32(gpart + 2 * n2, ix) = v[2];
        }
    }
    // gradient of level k from the layers above and below it
    __device__ __forceinline__ void store_level(Real x, int k) const
    {
        const unsigned ix = (unsigned)(k * u.in.ncol + u.col);
        Real v[1] = {x * plkslope(at32(w.ilev, ix))};
        lw_lane_sums<BAND>(v);
        if (u.first) at32(glev, ix) = v[0];
    }
    __device__ __forceinline__ void store_column(Real a_tb, Real a_sec) const
    {
        Real v[2] = {a_tb, a_sec};
        lw_lane_sums<BAND>(v);
        if (u.first) {
            // a_sec holds sum a_od od = secdiff sum a_od tau
            gsc[u.col] = v[0];
            gsc[u.in.ncol + u.col] = v[1] / u.secdiff * u.dsecdiff();
        }
    }
};

// One unit by one wave.  Both sweeps of the forward have an adjoint that runs
// the other way, and neither adjoint needs the forward's radiances but for the
// local terms, so two sweeps do: top-down, the downward radiance and the
// adjoint of the upward one; bottom-up, the upward radiance and the adjoint of
// the downward one, with all local terms.  row: the wave's scratch,
// [nlay][3][64][GC]: optical depths, incoming downward radiances, adjoints of
// the upward radiances.
template <int BAND, typename Real>
__device__ __forceinline__ void lw_vjp_band_body(const LwVjpUnit<BAND, Real> q, int lane, Real *__restrict__ row)
{
    constexpr int GC = LwVjpUnit<BAND, Real>::GC;
    using Vec = GVec<GC, Real>;
    const auto &u = q.u;
    const bool flux = q.w.bflux;
    const int nlay = u.in.nlay;
    auto at = [&](int lev, int k) -> Vec & { return at32((Vec *)row, (unsigned)(((lev - 1) * 3 + k) * 64 + lane)); };
    Real rad[GC], a[GC], a_tb;  // radiances, the other direction's adjoints
    Vec af;
    {
        LwLayer<Real> c;
        Real fr[GC];
        const Real top = q.ru(nlay);
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            rad[j] = (Real)0;
            a[j] = q.live(j, top);
        }
        if (flux) u.store(rad, nlay, 0);
        for (int lev = nlay; lev >= 1; --lev) {
            u.load(c, lev);
            Vec od, r, s;
            u.depths(c, lev, od.x);
            u.fracs(c, lev, fr);
            const Real blay = u.planklay(c), dplankdn = u.planklev(lev - 1) - blay, ct = q.ru(lev - 1);
#pragma unroll
            for (int j = 0; j < GC; ++j) {
                Real atr, tf;
                u.transmit(od.x[j], atr, tf);
                r.x[j] = rad[j];
                s.x[j] = a[j];
                const Real bbd = fr[j] * fma(tf, dplankdn, blay);
                rad[j] = fma(bbd - rad[j], atr, rad[j]);
                a[j] = fma(-a[j], atr, a[j]) + q.live(j, ct);
            }
            at(lev, 0) = od;
            at(lev, 1) = r;
            at(lev, 2) = s;
            if (flux) u.store(rad, lev - 1, 0);
        }
        q.surface(fr, rad, a, a_tb, af);
    }
    if (flux) u.store(rad, 0, 1);
    Real a_sec = (Real)0, up = (Real)0, plev = u.planklev(0);
    for (int lev = 1; lev <= nlay; ++lev) {
        // (loaded here, before the layer's work; a layer ahead, their registers
        // spill: 8192 x 40 1.01 -> 1.10 ms)
        const Vec od = at(lev, 0), r = at(lev, 1), s = at(lev, 2);
        LwGroupsD<Real> p;
        q.load(p, lev);
        const Real plev_up = u.planklev(lev);
        const auto o = q.local(lev, p, od, r, s, af, plev, plev_up, rad, a);
        plev = plev_up;
#pragma unroll
        for (int j = 0; j < GC; ++j) af.x[j] = (Real)0;
        if (flux) u.store(rad, lev, 1);
        q.store_layer(o, lev);
        q.store_level(up + o.dn, lev - 1);
        up = o.up;
        a_sec = a_sec + o.sec;
    }
    q.store_level(up, nlay);
    q.store_column(a_tb, a_sec);
}

// One unit by a workgroup of WAVES waves, for calls too small to fill the chip
// with waves: the layers' optics and local terms are shared out among the waves
// and one wave runs the two sweeps between them.  row: the workgroup's scratch,
// [nlay][6][64][GC] (optical depth, transmittance, the two sources, which the
// incoming radiances replace, and the two adjoints), [nlay][3][64] (levels below
// and above, sum a_od od of each layer) and [64][GC] (the surface's adjoints of
// the Planck fractions).
template <int WAVES, int BAND, typename Real>
__device__ __forceinline__ void lw_vjp_band_layers(const LwVjpUnit<BAND, Real> q, int wave, int lane,
                                                   Real *__restrict__ row)
{
    constexpr int GC = LwVjpUnit<BAND, Real>::GC;
    using Vec = GVec<GC, Real>;
    const auto &u = q.u;
    const int nlay = u.in.nlay;
    auto at = [&](int lev, int k) -> Vec & { return at32((Vec *)row, (unsigned)(((lev - 1) * 6 + k) * 64 + lane)); };
    Real *sums = row + (size_t)nlay * 6 * 64 * GC;
    auto sum = [&](int lev, int k) -> Real & { return at32(sums, (unsigned)(((lev - 1) * 3 + k) * 64 + lane)); };
    for (int lev = nlay - wave; lev >= 1; lev -= WAVES) {
        LwLayer<Real> c;
        u.load(c, lev);
        Vec od, atr, bbd, bbu;
        Real fr[GC];
        u.depths(c, lev, od.x);
        u.fracs(c, lev, fr);
        const Real blay = u.planklay(c), dn = u.planklev(lev - 1) - blay, up = u.planklev(lev) - blay;
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            Real tf;
            u.transmit(od.x[j], atr.x[j], tf);
            bbd.x[j] = fr[j] * fma(tf, dn, blay);
            bbu.x[j] = fr[j] * fma(tf, up, blay);
        }
        at(lev, 0) = od;
        at(lev, 1) = atr;
        at(lev, 2) = bbd;
        at(lev, 3) = bbu;
    }
    __syncthreads();
    Real a_tb = (Real)0;
    if (wave == 0) {
        Real rad[GC], a[GC];
        const Real top = q.ru(nlay);
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            rad[j] = (Real)0;
            a[j] = q.live(j, top);
        }
        // through the sources k, read four layers ahead; the incoming radiances
        // replace them, the adjoints go to k + 2
        auto sweep = [&](int first, int step, int k) {
            Vec tr[4], src[4];
            Real ct[4];
            auto fetch = [&](int i, int lev) {
                tr[i] = at(lev, 1);
                src[i] = at(lev, k);
                ct[i] = step < 0 ? q.ru(lev - 1) : lev < nlay ? q.rd(lev) : (Real)0;
            };
#pragma unroll
            for (int i = 0; i < 4; ++i) fetch(i, clampi(first + i * step, 1, nlay));
            for (int n = 0; n < nlay; n += 4)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (n + i >= nlay) break;
                    const int lev = first + (n + i) * step;
                    Vec r, s;
#pragma unroll
                    for (int j = 0; j < GC; ++j) {
                        r.x[j] = rad[j];
                        s.x[j] = a[j];
                        rad[j] = fma(src[i].x[j] - rad[j], tr[i].x[j], rad[j]);
                        a[j] = fma(-a[j], tr[i].x[j], a[j]) + q.live(j, ct[i]);
                    }
                    fetch(i, clampi(lev + 4 * step, 1, nlay));
                    at(lev, k) = r;
                    at(lev, k + 2) = s;
                }
        };
        sweep(nlay, -1, 2);
        LwLayer<Real> c;
        Real fr[GC];
        u.load(c, 1);
        u.fracs(c, 1, fr);
        Vec af;
        q.surface(fr, rad, a, a_tb, af);
        *(Vec *)(sums + (size_t)3 * nlay * 64 + lane * GC) = af;
        sweep(1, 1, 3);
    }
    __syncthreads();
    for (int lev = 1 + wave; lev <= nlay; lev += WAVES) {
        Vec rad = at(lev, 3), a = at(lev, 5);
        if (q.w.bflux) {  // the fluxes: those entering the layer, and those leaving the outermost ones
            u.store(at(lev, 2).x, lev, 0);
            u.store(rad.x, lev - 1, 1);
        }
        const Vec od = at(lev, 0), r = at(lev, 2), s = at(lev, 4);
        Vec af{};
        if (lev == 1) af = *(const Vec *)(sums + (size_t)3 * nlay * 64 + lane * GC);
        LwGroupsD<Real> p;
        q.load(p, lev);
        const auto o = q.local(lev, p, od, r, s, af, u.planklev(lev - 1), u.planklev(lev), rad.x, a.x);
        if (q.w.bflux && lev == nlay) u.store(rad.x, nlay, 1);
        if (q.w.bflux && lev == 1) {
            LwLayer<Real> c;
            Real fr[GC], rad0[GC];
            u.load(c, 1);
            u.fracs(c, 1, fr);
            const Real blay = u.planklay(c), dn = u.planklev(0) - blay;
#pragma unroll
            for (int j = 0; j < GC; ++j) {
                Real atr, tf;
                u.transmit(od.x[j], atr, tf);
                rad0[j] = fma(fr[j] * fma(tf, dn, blay) - r.x[j], atr, r.x[j]);
            }
            u.store(rad0, 0, 0);
        }
        q.store_layer(o, lev);
        sum(lev, 0) = o.dn;
        sum(lev, 1) = o.up;
        sum(lev, 2) = o.sec;
    }
    __syncthreads();
    for (int k = wave; k <= nlay; k += WAVES)
        q.store_level(k == 0 ? sum(1, 0) : k == nlay ? sum(nlay, 1) : sum(k, 1) + sum(k + 1, 0), k);
    if (wave == 0) {
        Real a_sec = (Real)0;
        for (int lev = 1; lev <= nlay; ++lev) a_sec = a_sec + sum(lev, 2);
        q.store_column(a_tb, a_sec);
    }
    __syncthreads();
}

#pragma clang fp contract(fast)

// the forward's view of the backward's workspace
__device__ __forceinline__ LwWork lw_vjp_forward(const LwVjpWork &w)
{
    LwWork f;
    f.coef = w.dcoef;
    f.tlev = w.tlev;
    f.ipk = w.ipk;
    f.ilev = w.ilev;
    f.laytrop = w.laytrop;
    f.colscal = w.colscal;
    f.bflux = w.bflux;
    return f;
}

// what the LW backward body reads and writes, for the call below
struct LwUnitArgs {
    int ncol, nlay, plk_off;
    gptr<const double> emis, tauaer;  // tauaer NULL: no aerosol
    gptr<const double> colscal;
    gptr<const float> dcoef, dder, tlev, cot, tab;
    gptr<const int> ipk, ilev, laytrop;
    gptr<const LwConst> cst;
    gptr<float> gpart, glev, gsc, bflux;  // bflux NULL: no forward fluxes
};
__device__ __forceinline__ LwUnitArgs lw_unit_args(const ColumnInputs &in, const LwVjpWork &w, int plk_off,
                                                   const float *tab, const LwConst *cst)
{
    LwUnitArgs a;
    a.ncol = in.ncol;
    a.nlay = in.nlay;
    a.plk_off = plk_off;
    a.emis = (gptr<const double>)in.emis;
    a.tauaer = (gptr<const double>)in.tauaer;
    a.colscal = (gptr<const double>)w.colscal;
    a.dcoef = (gptr<const float>)w.dcoef;
    a.dder = (gptr<const float>)w.dder;
    a.tlev = (gptr<const float>)w.tlev;
    a.cot = (gptr<const float>)w.cot;
    a.tab = (gptr<const float>)tab;
    a.ipk = (gptr<const int>)w.ipk;
    a.ilev = (gptr<const int>)w.ilev;
    a.laytrop = (gptr<const int>)w.laytrop;
    a.cst = (gptr<const LwConst>)cst;
    a.gpart = (gptr<float>)w.gpart;
    a.glev = (gptr<float>)w.glev;
    a.gsc = (gptr<float>)w.gsc;
    a.bflux = (gptr<float>)w.bflux;
    return a;
}

// The FP32 body with its tables in LDS, of the LW LDS-table backward kernel and
// of the fused kernel (a function call of its own: 0.97 ms against 0.95 at
// 8192 x 40, 5.6 against 5.1 at 32768 x 60).  et: the (exp, tfn)
// pairs; ktab: the band's k-tables; row: the wave's scratch row; columns c0 on,
// below cend.
template <int BAND>
__device__ __forceinline__ void lw_vjp_unit(const LwUnitArgs &a, const LwBand &B, lptr<const ExpTfn<float>> et,
                                         lptr<const float> ktab, int c0, int cend, int lane, gptr<float> row)
{
    ColumnInputs in{};
    in.ncol = a.ncol;
    in.nlay = a.nlay;
    in.emis = (const double *)a.emis;
    in.tauaer = (const double *)a.tauaer;
    LwVjpWork w;
    w.colscal = (double *)(const double *)a.colscal;
    w.dcoef = (void *)(const float *)a.dcoef;
    w.dder = (void *)(const float *)a.dder;
    w.tlev = (void *)(const float *)a.tlev;
    w.cot = (void *)(const float *)a.cot;
    w.ipk = (int *)(const int *)a.ipk;
    w.ilev = (int *)(const int *)a.ilev;
    w.laytrop = (int *)(const int *)a.laytrop;
    w.gpart = (void *)(float *)a.gpart;
    w.glev = (void *)(float *)a.glev;
    w.gsc = (void *)(float *)a.gsc;
    w.bflux = (void *)(float *)a.bflux;
    const LwWork f = lw_vjp_forward(w);
    const float *tab = (const float *)a.tab, *kt = (const float *)ktab;
    const LwUnit<BAND, float> u(in, f, B, kt, BAND >= 3 && BAND <= 5 ? tab : kt, tab, (const ExpTfn<float> *)et,
                                a.plk_off, (const LwConst *)a.cst, c0, cend, lane);
    lw_vjp_band_body(LwVjpUnit<BAND, float>(u, w), lane, (float *)row);
}
// that of band b (0-based)
__device__ __forceinline__ void lw_vjp_unit_of(const LwUnitArgs &a, const LwBand *bands, int b,
                                               lptr<const ExpTfn<float>> et, lptr<const float> ktab, int c0, int cend,
                                               int lane, gptr<float> row)
{
#define BODY(bb)                                                                    \
    case bb - 1:                                                                    \
        lw_vjp_unit<bb>(a, bands[bb - 1], et, ktab, c0, cend, lane, row);           \
        break;
    switch (b) {
        BODY(1) BODY(2) BODY(3) BODY(4) BODY(5) BODY(6) BODY(7) BODY(8)
        BODY(9) BODY(10) BODY(11) BODY(12) BODY(13) BODY(14) BODY(15) BODY(16)
    }
#undef BODY
}

}  // namespace rrtmg
