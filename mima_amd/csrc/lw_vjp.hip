// Backward (vector-Jacobian product) of the clear-sky LW path on gfx950:
// given cotangents of uflx, dflx (levels) and hr (layers), the gradients with
// respect to layer temperature, level temperature, water vapour, ozone and
// surface temperature.  No counterpart in the reference, whose only
// derivative is the idrv = 1 surface-Planck term dF/dTs
// (rrtmg_lw_rtrnmr.f90:629-746); the forward being differentiated is
// rrtmg_lw (rrtmg_lw_rad.nomcica.f90:80) as the forward kernels implement it.
//
// Kernels:
//  * prep (one thread per (layer, column)): inatm + setcoef in FP64 dual
//    numbers seeded with (tlay, h2o, o3) of each layer, writing every
//    per-layer coefficient's value (the forward's record) and its nonzero
//    derivatives (a second record, LW_DMASK); level Planck indices; and the per-level
//    radiance cotangents after folding the heating-rate cotangent into the
//    fluxes; then a per-column kernel for laytrop, the column water and
//    dry-air totals, precipitable water and surface temperature.
//  * band (lane = up to four g-points of a column, as in the forward): top-down,
//    the downward radiances and the adjoints of the upward ones; bottom-up, the
//    upward radiances, the adjoints of the downward ones and the layers' local
//    terms.  The optical depths are kept between the sweeps; the gas optics'
//    derivatives come from the weights of their table rows (lw_vjp_body.hpp),
//    those of transmittance and source are analytic (for table lookups, those
//    of the functions the tables tabulate).  What bounds it is VALU work: with a
//    lane per g-point, four sweeps and every derivative carried by every
//    coefficient it took 1746 us at 8192 x 40 in FP32 (32768 x 60: 10.1 ms),
//    now 946 (5.05); FP64 4096 x 40 2.80 -> 1.40 ms.  The prep stores groups of
//    four fields, a wave's side by side: 121 -> 38 us.
//  * finish (one thread per (layer, column)): sums over bands in FP64 and
//    the precipitable-water chain of the diffusivity angle.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "lw_optics.hpp"
#include "lw_vjp_body.hpp"
#include "rrtmg_device.hpp"

namespace rrtmg {

using D3 = Dual<double, 3>;


// ---------------------------------------------------------------------------
// prep: the forward prep's arithmetic (lw.hip, rrtmg_lw_rad.nomcica.f90:729-852,
// rrtmg_lw_setcoef.f90:150-413) on dual numbers, one thread per (layer,
// column): the layer's coefficients with their derivatives, the Planck index
// of the level above it (and of the surface level), and the radiance
// cotangents of its lower level (and of the top level)
template <typename Real>
__global__ __launch_bounds__(256) void lw_vjp_prep_kernel(ColumnInputs in, VjpCot cot, LwVjpWork w,
                                                          const LwConst *__restrict__ cst, double heatfac)
{
    const int ncol = in.ncol, nlay = in.nlay;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)nlay * ncol) return;
    const int lay = (int)(i / ncol), col = (int)(i - (size_t)lay * ncol);
    Real *tlevf = (Real *)w.tlev;
    const double amd = 28.9660, amw = 18.0160, amdw = 1.607793, amdo = 0.603428;
    const double avogad = 6.02214199e+23, grav = 9.8066;
    const double stpfac = 296.0 / 1013.0;
    // the values and the derivatives of the (layer, column)
    Real rec[LWF_STRIDE], der[LW_DSTRIDE];
#pragma unroll
    for (int f = LWF_COUNT; f < LWF_STRIDE; ++f) rec[f] = (Real)0;
#pragma unroll
    for (int f = der_offset(LW_DMASK, LWF_COUNT); f < LW_DSTRIDE; ++f) der[f] = (Real)0;
    auto put = [&](auto field, const D3 &x) {
        constexpr int F = decltype(field)::value, O = der_offset(LW_DMASK, F);
        constexpr unsigned m = LW_DMASK[F];
        rec[F] = (Real)x.v;
        if constexpr ((m & 1u) != 0) der[O] = (Real)x.d[0];
        if constexpr ((m & 2u) != 0) der[O + dmask_count(m & 1u)] = (Real)x.d[1];
        if constexpr ((m & 4u) != 0) der[O + dmask_count(m & 3u)] = (Real)x.d[2];
    };
    if (lay == 0) {
        double tz0 = in.tlev[col];
        int i0 = clampi((int)(tz0 - 159.0), 1, 180);
        w.ilev[col] = i0;
        tlevf[col] = (Real)(tz0 - 159.0 - (double)i0);
    }
    {
        const size_t ix = (size_t)lay * ncol + col;
        const double pavel = in.play[ix];
        const D3 tavel = D3::seed(in.tlay[ix], 0);
        const D3 h2o = D3::seed(in.h2o[ix], 1);
        const D3 o3 = D3::seed(in.o3[ix], 2);
        const double pz0 = in.plev[ix], pz1 = in.plev[ix + ncol];
        D3 wkl1 = (h2o / (1.0 - h2o)) * amdw;
        const double wkl2 = in.co2[ix], wkl4 = in.n2o[ix], wkl6 = in.ch4[ix], wkl7 = in.o2[ix];
        const D3 wkl3 = o3 * amdo;
        const D3 amm = (1.0 - wkl1) * amd + wkl1 * amw;
        const D3 coldry = ((pz0 - pz1) * 1.e3 * avogad) / (1.e2 * grav * amm * (1.0 + wkl1));
        D3 summol(0.0);
        summol = summol + wkl2;
        summol = summol + wkl3;
        summol = summol + wkl4;
        summol = summol + 0.0;
        summol = summol + wkl6;
        summol = summol + wkl7;
        const D3 wbrodl = coldry * (1.0 - summol);
        wkl1 = coldry * wkl1;
        const D3 wx1 = coldry * in.ccl4[ix] * 1.e-20, wx2 = coldry * in.cfc11[ix] * 1.e-20;
        const D3 wx3 = coldry * in.cfc12[ix] * 1.e-20, wx4 = coldry * in.cfc22[ix] * 1.e-20;

        const int indlay = clampi((int)(tavel.v - 159.0), 1, 180);
        const D3 tlayfrac = tavel - 159.0 - (double)indlay;
        const double tz = in.tlev[ix + ncol];
        const int indlev = clampi((int)(tz - 159.0), 1, 180);
        w.ilev[ix + ncol] = indlev;
        tlevf[ix + ncol] = (Real)(tz - 159.0 - (double)indlev);

        const double plog = log(pavel);
        const int jp = clampi((int)(36.0 - 5 * (plog + 0.04)), 1, 58);
        const double fp = 5.0 * (cst->preflog[jp - 1] - plog);
        const D3 dt0 = (tavel - cst->tref[jp - 1]) / 15.0;
        const int jt = clampi((int)(3.0 + dt0.v), 1, 4);
        const D3 ft = dt0 - (double)(jt - 3);
        const D3 dt1 = (tavel - cst->tref[jp]) / 15.0;
        const int jt1 = clampi((int)(3.0 + dt1.v), 1, 4);
        const D3 ft1 = dt1 - (double)(jt1 - 3);
        const D3 water = wkl1 / coldry;
        const D3 scalefac = pavel * stpfac / tavel;
        const D3 forfac = scalefac / (1. + water);
        D3 forfrac, selffac = water * forfac, selffrac(0.0);
        int indfor, indself = 0;
        if (plog > 4.56) {
            D3 factor = (332.0 - tavel) / 36.0;
            indfor = clampi((int)factor.v, 1, 2);
            forfrac = factor - (double)indfor;
            factor = (tavel - 188.0) / 7.2;
            indself = clampi((int)factor.v - 7, 1, 9);
            selffrac = factor - (double)(indself + 7);
        } else {
            const D3 factor = (tavel - 188.0) / 36.0;
            indfor = 3;
            forfrac = factor - 1.0;
        }
        const D3 scaleminor = pavel / tavel;
        const D3 scaleminorn2 = (pavel / tavel) * (wbrodl / (coldry + wkl1));
        const D3 factor = (tavel - 180.8) / 7.2;
        const int indminor = clampi((int)factor.v, 1, 18);
        const D3 minorfrac = factor - (double)indminor;
        const D3 colh2o = 1.e-20 * wkl1;
        D3 colco2 = 1.e-20 * (coldry * wkl2);
        D3 colo3 = 1.e-20 * (coldry * wkl3);
        D3 coln2o = 1.e-20 * (coldry * wkl4);
        D3 colco(0.0);
        D3 colch4 = 1.e-20 * (coldry * wkl6);
        const D3 colo2 = 1.e-20 * (coldry * wkl7);
        if (colco2.v == 0.0) colco2 = 1.e-32 * coldry;
        if (colo3.v == 0.0) colo3 = 1.e-32 * coldry;
        if (coln2o.v == 0.0) coln2o = 1.e-32 * coldry;
        if (colco.v == 0.0) colco = 1.e-32 * coldry;
        if (colch4.v == 0.0) colch4 = 1.e-32 * coldry;
        const D3 colbrd = 1.e-20 * wbrodl;
        const double compfp = 1. - fp;
        put(std::integral_constant<int, LWF_FAC10>{}, compfp * ft);
        put(std::integral_constant<int, LWF_FAC00>{}, compfp * (1.0 - ft));
        put(std::integral_constant<int, LWF_FAC11>{}, fp * ft1);
        put(std::integral_constant<int, LWF_FAC01>{}, fp * (1.0 - ft1));
        put(std::integral_constant<int, LWF_COLH2O>{}, colh2o);
        put(std::integral_constant<int, LWF_COLCO2>{}, colco2);
        put(std::integral_constant<int, LWF_COLO3>{}, colo3);
        put(std::integral_constant<int, LWF_COLN2O>{}, coln2o);
        put(std::integral_constant<int, LWF_COLCO>{}, colco);
        put(std::integral_constant<int, LWF_COLCH4>{}, colch4);
        put(std::integral_constant<int, LWF_COLO2>{}, colo2);
        put(std::integral_constant<int, LWF_COLBRD>{}, colbrd);
        put(std::integral_constant<int, LWF_SELFFAC>{}, colh2o * selffac);
        put(std::integral_constant<int, LWF_SELFFRAC>{}, selffrac);
        put(std::integral_constant<int, LWF_FORFAC>{}, colh2o * forfac);
        put(std::integral_constant<int, LWF_FORFRAC>{}, forfrac);
        put(std::integral_constant<int, LWF_MINORFRAC>{}, minorfrac);
        put(std::integral_constant<int, LWF_SCALEMINOR>{}, scaleminor);
        put(std::integral_constant<int, LWF_SCALEMINORN2>{}, scaleminorn2);
        put(std::integral_constant<int, LWF_COLDRY>{}, coldry);
        put(std::integral_constant<int, LWF_PAVEL>{}, D3(pavel));
        put(std::integral_constant<int, LWF_WX1>{}, wx1);
        put(std::integral_constant<int, LWF_WX2>{}, wx2);
        put(std::integral_constant<int, LWF_WX3>{}, wx3);
        put(std::integral_constant<int, LWF_WX4>{}, wx4);
        put(std::integral_constant<int, LWF_TLAYFRAC>{}, tlayfrac);
        w.ipk[ix] = pack_lw(jp, jt, jt1, indself, indfor, indminor, indlay);
        // [lay][group][col][4]: a wave's store of a group is contiguous
        struct alignas(16) Group {
            Real x[4];
        };
        Group *gv = (Group *)w.dcoef + (size_t)lay * LWF_GROUPS * ncol + col;
        Group *gd = (Group *)w.dder + (size_t)lay * LWD_GROUPS * ncol + col;
#pragma unroll
        for (int k = 0; k < LWF_GROUPS; ++k)
            gv[(size_t)k * ncol] = {rec[4 * k], rec[4 * k + 1], rec[4 * k + 2], rec[4 * k + 3]};
#pragma unroll
        for (int k = 0; k < LWD_GROUPS; ++k)
            gd[(size_t)k * ncol] = {der[4 * k], der[4 * k + 1], der[4 * k + 2], der[4 * k + 3]};
    }

    // level radiance cotangents: fluxes' own cotangents plus the heating rate
    // hr(k) = heatfac (fnet(k) - fnet(k+1)) / (p(k) - p(k+1)), fnet = up - dn
    // (rrtmg_lw_rtrnmr.f90:767-772); this thread's level lay, and the top
    Real *cu = (Real *)w.cot, *cd = cu + (size_t)(nlay + 1) * ncol;
    for (int k = lay; k <= (lay == nlay - 1 ? nlay : lay); ++k) {
        const size_t ix = (size_t)k * ncol + col;
        double fbar = 0.0;
        if (cot.hr) {
            if (k < nlay) fbar += heatfac * cot.hr[ix] / (in.plev[ix] - in.plev[ix + ncol]);
            if (k > 0) fbar -= heatfac * cot.hr[ix - ncol] / (in.plev[ix - ncol] - in.plev[ix]);
        }
        cu[ix] = (Real)((cot.uflx ? cot.uflx[ix] : 0.0) + fbar);
        cd[ix] = (Real)((cot.dflx ? cot.dflx[ix] : 0.0) - fbar);
    }
}

// per-column part of the prep (lw_column_sums): laytrop, the column water and
// dry-air totals, precipitable water and surface temperature
__global__ __launch_bounds__(256) void lw_vjp_column_kernel(ColumnInputs in, LwVjpWork w)
{
    const int col = blockIdx.x * 64 + ((int)threadIdx.x & 63), ncol = in.ncol;
    const LwColumn r = lw_column_sums(in.plev, in.h2o, false, w.ipk, ncol, in.nlay, min(col, ncol - 1));
    if (threadIdx.x >= 64 || col >= ncol) return;
    const double amd = 28.9660, amw = 18.0160, grav = 9.8066;
    const double wvsh = (amw * r.wvttl) / (amd * r.amttl);
    w.laytrop[col] = r.laytrop;
    w.colscal[col] = wvsh * (1.e3 * in.plev[col]) / (1.e2 * grav);
    w.colscal[(size_t)ncol + col] = in.tsfc[col];
    w.colscal[(size_t)2 * ncol + col] = r.wvttl;
    w.colscal[(size_t)3 * ncol + col] = r.amttl;
}


// Tables in global memory: persistent workgroups of WAVES waves; work items (CPW
// columns of a band) from a counter, band by band, the bands with most work
// first.  One wave: lw_vjp_band_body; more: lw_vjp_band_layers.
template <typename Real, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(sizeof(Real) == 4 || WAVES > 4 ? 2 : 1)))
void lw_vjp_band_kernel(ColumnInputs in, LwVjpWork w, const LwBand *__restrict__ bands, size_t row_elems, int et_off,
                        int plk_off, const Real *__restrict__ tab, const LwConst *__restrict__ cst)
{
    __shared__ int s_item;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    const ExpTfn<Real> *et = et_off >= 0 ? (const ExpTfn<Real> *)(tab + et_off) : nullptr;
    Real *row = (Real *)w.dstate + (size_t)blockIdx.x * row_elems;
    const LwWork f = lw_vjp_forward(w);
    for (;;) {
        int item = __builtin_amdgcn_readfirstlane(next_item(w.items, &s_item));
#define BODY(b)                                                                                                  \
    {                                                                                                            \
        const int n = (in.ncol + lw_cpw(b) - 1) / lw_cpw(b);                                                     \
        if (item < n) {                                                                                          \
            const LwVjpUnit<b, Real> q(                                                                          \
                LwUnit<b, Real>(in, f, bands[b - 1], tab, tab, tab, et, plk_off, cst, item * lw_cpw(b), in.ncol, lane), w); \
            if constexpr (WAVES == 1) lw_vjp_band_body(q, lane, row);                                            \
            else lw_vjp_band_layers<WAVES>(q, wave, lane, row);                                                  \
            continue;                                                                                            \
        }                                                                                                        \
        item -= n;                                                                                               \
    }
        BODY(5) BODY(3) BODY(4) BODY(7) BODY(9) BODY(13) BODY(12) BODY(8)
        BODY(1) BODY(6) BODY(15) BODY(16) BODY(11) BODY(2) BODY(10) BODY(14)
#undef BODY
        return;
    }
}

// FP32 kernel of the large calls, scheduled as the forward's lw_band_lds_kernel
// (persistent workgroups with the (exp, tfn) pairs and one band's k-tables in
// LDS; work items from the XCDs' counters) with LWV_WGW waves, each of which
// takes every LWV_WGW-th of an item's 16 units.
__global__ __launch_bounds__(64 * LWV_WGW) void lw_vjp_band_lds_kernel(ColumnInputs in, LwVjpWork w,
                                                                       const LwBand *__restrict__ bands,
                                                                       LwLdsPlan plan, int et_off, int plk_off,
                                                                       const float *__restrict__ tab,
                                                                       const LwConst *__restrict__ cst)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    ExpTfn<float> *et = (ExpTfn<float> *)smem_raw;
    float *ktab = (float *)(smem_raw + LW_ET_VECS * 16);
    for (int i = threadIdx.x; i < LW_ET_VECS; i += 64 * LWV_WGW)
        ((uint4 *)smem_raw)[i] = ((const uint4 *)(tab + et_off))[i];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    float *row = (float *)w.dstate +
                 ((size_t)blockIdx.x * LWV_WGW + wave) * lw_vjp_row_bytes(in.nlay, 1, LWV_LDS);
    const int ntiles = (in.ncol + LW_TILE - 1) / LW_TILE;
    const LwUnitArgs ua = lw_unit_args(in, w, plk_off, tab, cst);
    __shared__ int s_item;
    int loaded = -1, queue = 0;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_item = lw_claim_tile_item(w.items, ntiles, queue);
        __syncthreads();
        const int item = __builtin_amdgcn_readfirstlane(s_item);
        if (item < 0) return;
        const int tile = item / LW_TILE_ITEMS;
        const LwTileSlot slot = LW_TILE_SLOTS.s[item - tile * LW_TILE_ITEMS];
        const int b = slot.band - 1;
        if (b != loaded) {
            lw_copy_tables(ktab, tab, plan, b);
            __syncthreads();
            loaded = b;
        }
        const int cend = min((tile + 1) * LW_TILE, in.ncol);
        for (int k = wave; k < 16; k += LWV_WGW) {
            const int c0 = tile * LW_TILE + (slot.part * 16 + k) * slot.cpw;
            if (c0 >= cend) break;
            lw_vjp_unit_of(ua, bands, b, (lptr<const ExpTfn<float>>)et, (lptr<const float>)ktab, c0, cend, lane,
                           (gptr<float>)row);
        }
    }
}

// finish: band sums and the precipitable-water chain of the diffusivity
// angle (pwvcm depends on the water vapour of every layer), one thread per
// (layer, column); the thread of layer 0 also writes the surface gradient and
// that of the top layer the top level's
template <typename Real>
__global__ __launch_bounds__(256) void lw_vjp_finish_kernel(ColumnInputs in, LwVjpWork w, LwGrad out)
{
    const int ncol = in.ncol, nlay = in.nlay;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)nlay * ncol) return;
    const int lay = (int)(i / ncol), col = (int)(i - (size_t)lay * ncol);
    const size_t n2 = (size_t)nlay * ncol, n3 = (size_t)(nlay + 1) * ncol;
    const Real *gpart = (const Real *)w.gpart, *glev = (const Real *)w.glev, *gsc = (const Real *)w.gsc;
    double a_pw = 0.0, gts = 0.0;
    for (int b = 0; b < 16; ++b) {
        gts += (double)gsc[(size_t)b * 2 * ncol + col];
        a_pw += (double)gsc[(size_t)b * 2 * ncol + ncol + col];
    }
    if (lay == 0) out.tsfc[col] = gts;
    for (int k = lay; k <= (lay == nlay - 1 ? nlay : lay); ++k) {
        double s = 0.0;
        for (int b = 0; b < 16; ++b) s += (double)glev[(size_t)b * n3 + (size_t)k * ncol + col];
        out.tlev[(size_t)k * ncol + col] = s;
    }
    // pwvcm = (amw wvttl / (amd amttl)) 1e3 plev(0) / (1e2 grav), wvttl = sum
    // coldry wkl1, amttl = sum coldry (1 + wkl1) (rrtmg_lw_rad.nomcica.f90:845-852)
    const double amd = 28.9660, amw = 18.0160, amdw = 1.607793, avogad = 6.02214199e+23, grav = 9.8066;
    using D1 = Dual<double, 1>;
    const double wvttl = w.colscal[(size_t)2 * ncol + col], amttl = w.colscal[(size_t)3 * ncol + col];
    const double cpw = (amw / amd) * (1.e3 * in.plev[col]) / (1.e2 * grav);
    const size_t ix = (size_t)lay * ncol + col;
    const D1 h = D1::seed(in.h2o[ix], 0);
    const double pz0 = in.plev[ix], pz1 = in.plev[ix + ncol];
    const D1 wkl1 = (h / (1.0 - h)) * amdw;
    const D1 amm = (1.0 - wkl1) * amd + wkl1 * amw;
    const D1 coldry = ((pz0 - pz1) * 1.e3 * avogad) / (1.e2 * grav * amm * (1.0 + wkl1));
    const D1 wv = coldry * wkl1, am = coldry + coldry * wkl1;
    const double dpw = cpw * (wv.d[0] * amttl - wvttl * am.d[0]) / (amttl * amttl);
    double gt = 0.0, gq = 0.0, go = 0.0;
    for (int b = 0; b < 16; ++b) {
        const Real *gp = gpart + (size_t)b * 3 * n2;
        gt += (double)gp[ix];
        gq += (double)gp[n2 + ix];
        go += (double)gp[2 * n2 + ix];
    }
    out.tlay[ix] = gt;
    out.h2o[ix] = gq + a_pw * dpw;
    out.o3[ix] = go;
}

template <typename Real>
static void launch_lw_vjp_prep_t(const ColumnInputs &in, const VjpCot &cot, const LwVjpWork &w,
                                 const LwDevTables &t, hipStream_t s)
{
    const int nb = (in.ncol + 63) / 64;
    const int nbl = (int)(((size_t)in.nlay * in.ncol + 255) / 256);
    hipLaunchKernelGGL(lw_vjp_prep_kernel<Real>, dim3(nbl), dim3(256), 0, s, in, cot, w, t.cst, t.heatfac);
    hipLaunchKernelGGL(lw_vjp_column_kernel, dim3(nb), dim3(256), 0, s, in, w);
}

template <typename Real>
static void launch_lw_vjp_band_t(const ColumnInputs &in, const LwVjpWork &w, const LwDevTables &t, bool smooth,
                                 hipStream_t s)
{
    hipLaunchKernelGGL(reset_items_kernel, dim3(1), dim3(8), 0, s, w.items);
    if constexpr (sizeof(Real) == 4) {
        if (w.kind == LWV_LDS) {
            hipLaunchKernelGGL(lw_vjp_band_lds_kernel, dim3(w.chunk), dim3(64 * LWV_WGW), (size_t)t.plan.fwd_lds_bytes,
                               s, in, w, t.bands_fwd, t.plan, t.desc.et_tbl, t.desc.totplnk, (const float *)t.tab,
                               t.cst);
            return;
        }
    }
    const size_t row = lw_vjp_row_bytes(in.nlay, 1, w.kind);
    const int et_off = smooth ? -1 : t.desc.et_tbl;
#define LAUNCH(WAVES)                                                                                             \
    hipLaunchKernelGGL((lw_vjp_band_kernel<Real, WAVES>), dim3(w.chunk), dim3(64 * WAVES), 0, s, in, w, t.bands, row, \
                       et_off, t.desc.totplnk, (const Real *)t.tab, t.cst)
    if (w.kind == LWV_GROUP4) LAUNCH(4);
    if constexpr (sizeof(Real) == 4) {
        if (w.kind == LWV_GROUP8) LAUNCH(8);
    } else {
        if (w.kind == LWV_WAVE) LAUNCH(1);
    }
#undef LAUNCH
}

template <typename Real>
static hipError_t launch_lw_vjp_finish_t(const ColumnInputs &in, const LwGrad &out, const LwVjpWork &w,
                                         const LwDevTables &t, hipStream_t s, const LwOutputs *fwd, int mode)
{
    const int nbl = (int)(((size_t)in.nlay * in.ncol + 255) / 256);
    hipLaunchKernelGGL(lw_vjp_finish_kernel<Real>, dim3(nbl), dim3(256), 0, s, in, w, out);
    if (fwd) {
        const hipError_t e = launch_lw_finish(in, *fwd, w.bflux, t, mode, s);
        if (e != hipSuccess) return e;
    }
    return hipGetLastError();
}

hipError_t launch_lw_vjp(const ColumnInputs &in, const VjpCot &cot, const LwGrad &out, const LwVjpWork &w,
                         const LwDevTables &t, int mode, hipStream_t s, hipEvent_t *ev, const LwOutputs *fwd)
{
    if (fwd && !w.bflux) return hipErrorInvalidValue;
    if (ev) (void)hipEventRecord(ev[0], s);
    hipError_t e = launch_lw_vjp_prep(in, cot, w, t, mode, s);
    if (e != hipSuccess) return e;
    if (ev) (void)hipEventRecord(ev[1], s);
    e = launch_lw_vjp_band(in, w, t, mode, s);
    if (e != hipSuccess) return e;
    if (ev) (void)hipEventRecord(ev[2], s);
    e = launch_lw_vjp_finish(in, out, w, t, mode, s, fwd);
    if (ev) (void)hipEventRecord(ev[3], s);
    return e;
}

hipError_t launch_lw_vjp_prep(const ColumnInputs &in, const VjpCot &cot, const LwVjpWork &w, const LwDevTables &t,
                              int mode, hipStream_t s)
{
    if (mode == 1) launch_lw_vjp_prep_t<float>(in, cot, w, t, s);
    else launch_lw_vjp_prep_t<double>(in, cot, w, t, s);
    return hipGetLastError();
}

hipError_t launch_lw_vjp_band(const ColumnInputs &in, const LwVjpWork &w, const LwDevTables &t, int mode,
                              hipStream_t s)
{
    if (mode == 1) launch_lw_vjp_band_t<float>(in, w, t, false, s);
    else launch_lw_vjp_band_t<double>(in, w, t, mode == 2, s);
    return hipGetLastError();
}

hipError_t launch_lw_vjp_finish(const ColumnInputs &in, const LwGrad &out, const LwVjpWork &w, const LwDevTables &t,
                                int mode, hipStream_t s, const LwOutputs *fwd)
{
    if (fwd && !w.bflux) return hipErrorInvalidValue;
    return mode == 1 ? launch_lw_vjp_finish_t<float>(in, out, w, t, s, fwd, mode)
                     : launch_lw_vjp_finish_t<double>(in, out, w, t, s, fwd, mode);
}

}  // namespace rrtmg
