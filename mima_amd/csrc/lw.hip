// Longwave RRTMG on gfx950: prep (inatm + setcoef), band kernel (taumol +
// rtrnmr per g-point) and finish (band sums, fluxfac, heating).  Reference:
// rrtmg_lw/gcm_model/src/ of MiMA's RRTMG_LW (file:line cited per function).
//
// Band kernels: a lane holds up to four g-points of one column, LPC adjacent
// lanes a band, CPW columns a wave (LwLanes).  The gas optics are weighted table
// rows (lw_rows.hpp), so what does not depend on the g-point (coefficients,
// species parameters, weights, Planck values) is formed once for four
// g-points, a table row is one 16-byte load, and the g-sum is three additions
// and at most two shuffles.  With one g-point per lane the same work took twice
// the instructions (32768 columns x 40 layers: 2.16 ms -> 1.11 ms in FP32,
// 8192 x 40 in FP64: 1.35 -> 0.83 ms).
//
// Three kernels, by the size of the call (lw_fwd_kind); a column's result is
// the same bits in each:
// * lw_band_lds_kernel, large FP32 calls: what bounds it is LDS and L1
//   bandwidth (every optical depth takes about 18 table values), so the (exp,
//   transition function) pairs, 80 KB, and the k-tables of the workgroup's band
//   are in LDS; VALU 50% of its time.
// * lw_band_kernel, a wave per unit, large FP64 calls: the FP64 pairs alone
//   take 160 KB of LDS, the k-tables come from L1 and L2.
// * lw_band_kernel, a workgroup per unit with its waves sharing the layers,
//   calls below 4096 columns: too few waves to hide a layer's chain of
//   dependent loads (128 x 40: 137 -> 56 us).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "lw_optics.hpp"
#include "lw_rows.hpp"
#include "lw_unit.hpp"
#include "rrtmg_device.hpp"

namespace rrtmg {

// ---------------------------------------------------------------------------
// prep: FP64 (rrtmg_lw_rad.nomcica.f90:729-852 and rrtmg_lw_setcoef.f90:150-413),
// one thread per (layer, column): the layer's coefficients in the band
// kernel's precision, its integer table indices and the Planck index of the
// level above it (and of the surface level)
template <typename Real>
__global__ __launch_bounds__(256) void lw_prep_kernel(ColumnInputs in, LwWork w, const LwConst *__restrict__ cst)
{
    const int ncol = in.ncol, nlay = in.nlay;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t n = (size_t)nlay * ncol;
    const int lay = (int)(i / ncol), col = (int)(i - (size_t)lay * ncol);
    Real *tlevf = (Real *)w.tlev;
    const double amd = 28.9660, amw = 18.0160, amdw = 1.607793, amdo = 0.603428;
    const double avogad = 6.02214199e+23, grav = 9.8066;
    const double stpfac = 296.0 / 1013.0;
    // level 0 Planck index (setcoef: indlev0, t0frac)
    if (i < n && lay == 0) {
        double tz0 = in.tlev[col];
        int i0 = clampi((int)(tz0 - 159.0), 1, 180);
        w.ilev[col] = i0;
        tlevf[col] = (Real)(tz0 - 159.0 - (double)i0);
    }
    if (i < n) {
        const size_t ix = (size_t)lay * ncol + col;
        double pavel = in.play[ix], tavel = in.tlay[ix];
        double pz0 = in.plev[ix], pz1 = in.plev[ix + ncol];
        double h2o = in.h2o[ix];
        // MiMA's driver passes specific humidity and an O3 mass mixing
        // ratio (rrtmg_lw_rad.nomcica.f90:775-778); the McICA driver's inatm
        // takes volume mixing ratios (rrtmg_lw_rad.f90:778, 784)
        double wkl1 = in.vmr ? h2o : (h2o / (1.0 - h2o)) * amdw;
        double wkl2 = in.co2[ix], wkl3 = in.vmr ? in.o3[ix] : in.o3[ix] * amdo, wkl4 = in.n2o[ix], wkl6 = in.ch4[ix],
               wkl7 = in.o2[ix];
        double amm = (1.0 - wkl1) * amd + wkl1 * amw;
        double coldry = (pz0 - pz1) * 1.e3 * avogad / (1.e2 * grav * amm * (1.0 + wkl1));
        double summol = 0.0;
        summol = summol + wkl2;
        summol = summol + wkl3;
        summol = summol + wkl4;
        summol = summol + 0.0;
        summol = summol + wkl6;
        summol = summol + wkl7;
        double wbrodl = coldry * (1.0 - summol);
        wkl1 = coldry * wkl1;
        double wx1 = coldry * in.ccl4[ix] * 1.e-20, wx2 = coldry * in.cfc11[ix] * 1.e-20;
        double wx3 = coldry * in.cfc12[ix] * 1.e-20, wx4 = coldry * in.cfc22[ix] * 1.e-20;

        // Planck interpolation indices of the layer and of its top level
        int indlay = clampi((int)(tavel - 159.0), 1, 180);
        double tlayfrac = tavel - 159.0 - (double)indlay;
        double tz = in.tlev[ix + ncol];
        int indlev = clampi((int)(tz - 159.0), 1, 180);
        w.ilev[ix + ncol] = indlev;
        tlevf[ix + ncol] = (Real)(tz - 159.0 - (double)indlev);

        double plog = log(pavel);
        int jp = clampi((int)(36.0 - 5 * (plog + 0.04)), 1, 58);
        double fp = 5.0 * (cst->preflog[jp - 1] - plog);
        double dt0 = (tavel - cst->tref[jp - 1]) / 15.0;
        int jt = clampi((int)(3.0 + dt0), 1, 4);
        double ft = dt0 - (double)(jt - 3);
        double dt1 = (tavel - cst->tref[jp]) / 15.0;
        int jt1 = clampi((int)(3.0 + dt1), 1, 4);
        double ft1 = dt1 - (double)(jt1 - 3);
        double water = wkl1 / coldry;
        double scalefac = pavel * stpfac / tavel;
        double forfac = scalefac / (1. + water), forfrac, selffac = water * forfac, selffrac = 0.0;
        int indfor, indself = 0;
        if (plog > 4.56) {
            double factor = (332.0 - tavel) / 36.0;
            indfor = clampi((int)factor, 1, 2);
            forfrac = factor - (double)indfor;
            factor = (tavel - 188.0) / 7.2;
            indself = clampi((int)factor - 7, 1, 9);
            selffrac = factor - (double)(indself + 7);
        } else {
            double factor = (tavel - 188.0) / 36.0;
            indfor = 3;
            forfrac = factor - 1.0;
        }
        double scaleminor = pavel / tavel;
        double scaleminorn2 = (pavel / tavel) * (wbrodl / (coldry + wkl1));
        double factor = (tavel - 180.8) / 7.2;
        int indminor = clampi((int)factor, 1, 18);
        double minorfrac = factor - (double)indminor;
        double colh2o = 1.e-20 * wkl1;
        double colco2 = 1.e-20 * (coldry * wkl2);
        double colo3 = 1.e-20 * (coldry * wkl3);
        double coln2o = 1.e-20 * (coldry * wkl4);
        double colco = 0.0;
        double colch4 = 1.e-20 * (coldry * wkl6);
        double colo2 = 1.e-20 * (coldry * wkl7);
        if (colco2 == 0.0) colco2 = 1.e-32 * coldry;
        if (colo3 == 0.0) colo3 = 1.e-32 * coldry;
        if (coln2o == 0.0) coln2o = 1.e-32 * coldry;
        if (colco == 0.0) colco = 1.e-32 * coldry;
        if (colch4 == 0.0) colch4 = 1.e-32 * coldry;
        double colbrd = 1.e-20 * wbrodl;
        double compfp = 1. - fp;
        Real rec[LWF_STRIDE];
        rec[LWF_FAC10] = (Real)(compfp * ft);
        rec[LWF_FAC00] = (Real)(compfp * (1.0 - ft));
        rec[LWF_FAC11] = (Real)(fp * ft1);
        rec[LWF_FAC01] = (Real)(fp * (1.0 - ft1));
        rec[LWF_COLH2O] = (Real)colh2o;
        rec[LWF_COLCO2] = (Real)colco2;
        rec[LWF_COLO3] = (Real)colo3;
        rec[LWF_COLN2O] = (Real)coln2o;
        rec[LWF_COLCO] = (Real)colco;
        rec[LWF_COLCH4] = (Real)colch4;
        rec[LWF_COLO2] = (Real)colo2;
        rec[LWF_COLBRD] = (Real)colbrd;
        rec[LWF_SELFFAC] = (Real)(colh2o * selffac);
        rec[LWF_SELFFRAC] = (Real)selffrac;
        rec[LWF_FORFAC] = (Real)(colh2o * forfac);
        rec[LWF_FORFRAC] = (Real)forfrac;
        rec[LWF_MINORFRAC] = (Real)minorfrac;
        rec[LWF_SCALEMINOR] = (Real)scaleminor;
        rec[LWF_SCALEMINORN2] = (Real)scaleminorn2;
        rec[LWF_COLDRY] = (Real)coldry;
        rec[LWF_PAVEL] = (Real)pavel;
        rec[LWF_WX1] = (Real)wx1;
        rec[LWF_WX2] = (Real)wx2;
        rec[LWF_WX3] = (Real)wx3;
        rec[LWF_WX4] = (Real)wx4;
        rec[LWF_TLAYFRAC] = (Real)tlayfrac;
        w.ipk[ix] = pack_lw(jp, jt, jt1, indself, indfor, indminor, indlay);
        for (int f = LWF_COUNT; f < LWF_STRIDE; ++f) rec[f] = (Real)0;
        // [lay][group][col][4]: a wave's store of a group is contiguous
        struct alignas(16) Group {
            Real x[4];
        };
        Group *g = (Group *)w.coef + (size_t)lay * LWF_GROUPS * ncol + col;
#pragma unroll
        for (int k = 0; k < LWF_GROUPS; ++k)
            g[(size_t)k * ncol] = {rec[4 * k], rec[4 * k + 1], rec[4 * k + 2], rec[4 * k + 3]};
    }
}

// per-column part of the prep (lw_column_sums): laytrop, precipitable water,
// surface temperature
__global__ __launch_bounds__(256) void lw_column_kernel(ColumnInputs in, LwWork w)
{
    const int col = blockIdx.x * 64 + ((int)threadIdx.x & 63), ncol = in.ncol;
    const LwColumn r = lw_column_sums(in.plev, in.h2o, in.vmr, w.ipk, ncol, in.nlay, min(col, ncol - 1));
    if (threadIdx.x >= 64 || col >= ncol) return;
    const double amd = 28.9660, amw = 18.0160, grav = 9.8066;
    const double wvsh = (amw * r.wvttl) / (amd * r.amttl);
    w.laytrop[col] = r.laytrop;
    w.colscal[col] = wvsh * (1.e3 * in.plev[col]) / (1.e2 * grav);
    w.colscal[(size_t)ncol + col] = in.tsfc[col];
}

// contraction off, as in lw_rows.hpp
#pragma clang fp contract(off)

// One unit by one wave (rrtmg_lw_rtrnmr.f90:483-716, clear sky): the downward
// sweep keeps each layer's optical depths in the wave's scratch row,
// [nlay][64][GC], for the upward one, which forms the sources again from them.
// (Keeping transmittance and source instead doubles the traffic of the rows,
// which leaves the caches: 1.27 ms against 1.14 at 32768 x 40.)
template <int BAND, typename Real>
__device__ __forceinline__ void lw_band_body(const LwUnit<BAND, Real> u, int lane, Real *__restrict__ row)
{
    constexpr int GC = LwUnit<BAND, Real>::GC;
    using Vec = GVec<GC, Real>;
    const int nlay = u.in.nlay;
    Real rad[GC], fr[GC];
    LwLayer<Real> c;
#pragma unroll
    for (int j = 0; j < GC; ++j) rad[j] = (Real)0;
    u.store(rad, nlay, 0);  // drad(nlayers) stays 0
    for (int lev = nlay; lev >= 1; --lev) {
        u.load(c, lev);
        Vec od;
        u.depths(c, lev, od.x);
        at32((Vec *)row, (unsigned)((lev - 1) * 64 + lane)) = od;
        u.fracs(c, lev, fr);
        const Real blay = u.planklay(c), dplankdn = u.planklev(lev - 1) - blay;
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            Real atr, tf;
            u.transmit(od.x[j], atr, tf);
            const Real bbd = fr[j] * fma(tf, dplankdn, blay);
            rad[j] = fma(bbd - rad[j], atr, rad[j]);
        }
        u.store(rad, lev - 1, 0);
    }
    u.surface(fr, rad);
    u.store(rad, 0, 1);
    // the optical depths are read two levels ahead
    Vec n1 = at32((const Vec *)row, (unsigned)lane), n2 = at32((const Vec *)row, (unsigned)(64 + lane));
    for (int lev = 1; lev <= nlay; ++lev) {
        const Vec od = n1;
        n1 = n2;
        if (lev + 1 < nlay) n2 = at32((const Vec *)row, (unsigned)((lev + 1) * 64 + lane));
        u.load(c, lev);
        u.fracs(c, lev, fr);
        const Real blay = u.planklay(c), dplankup = u.planklev(lev) - blay;
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            Real atr, tf;
            u.transmit(od.x[j], atr, tf);
            const Real bbu = fr[j] * fma(tf, dplankup, blay);
            rad[j] = fma(bbu - rad[j], atr, rad[j]);
        }
        u.store(rad, lev, 1);
    }
}

// One unit by a workgroup of LW_LWAVES waves, for calls too small to fill the
// chip with waves: the layers' optics, which do not depend on each other, are
// shared out among the waves (a layer takes some 4000 cycles of dependent loads
// whoever computes it), then one wave sweeps down and the next up through the
// stored transmittances and sources, leaving the radiances, and all form the
// sums.  row: the workgroup's scratch, [nlay][4][64][GC] (transmittance, downward
// source, upward source and then radiance, downward radiance) and one more [64][GC] (Planck fractions of the lowest layer).
template <int WAVES, int BAND, typename Real>
__device__ __forceinline__ void lw_band_layers(const LwUnit<BAND, Real> u, int wave, int lane, Real *__restrict__ row)
{
    constexpr int GC = LwUnit<BAND, Real>::GC;
    using Vec = GVec<GC, Real>;
    const int nlay = u.in.nlay;
    auto at = [&](int lev, int k) -> Vec & { return at32((Vec *)row, (unsigned)(((lev - 1) * 4 + k) * 64 + lane)); };
    for (int lev = nlay - wave; lev >= 1; lev -= WAVES) {
        LwLayer<Real> c;
        u.load(c, lev);
        Real od[GC], fr[GC];
        u.depths(c, lev, od);
        u.fracs(c, lev, fr);
        const Real blay = u.planklay(c), dn = u.planklev(lev - 1) - blay, up = u.planklev(lev) - blay;
        Vec atr, bbd, bbu, f;
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            Real tf;
            u.transmit(od[j], atr.x[j], tf);
            bbd.x[j] = fr[j] * fma(tf, dn, blay);
            bbu.x[j] = fr[j] * fma(tf, up, blay);
            f.x[j] = fr[j];
        }
        at(lev, 0) = atr;
        at(lev, 1) = bbd;
        at(lev, 2) = bbu;
        if (lev == 1) at(nlay + 1, 0) = f;
    }
    __syncthreads();
    // sweep through the sources k, read four layers ahead; the radiances go to
    // the places `to` (none if negative)
    auto sweep = [&](Real (&rad)[GC], int first, int step, int k, int to) {
        Vec a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int lev = clampi(first + i * step, 1, nlay);
            a[i] = at(lev, 0);
            b[i] = at(lev, k);
        }
        for (int n = 0; n < nlay; n += 4)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (n + i >= nlay) break;
                const int lev = first + (n + i) * step, next = clampi(lev + 4 * step, 1, nlay);
                Vec r;
#pragma unroll
                for (int j = 0; j < GC; ++j) r.x[j] = rad[j] = fma(b[i].x[j] - rad[j], a[i].x[j], rad[j]);
                a[i] = at(next, 0);
                b[i] = at(next, k);
                if (to >= 0) at(lev, to) = r;
            }
    };
    // wave 0 down, wave 1 up; the latter needs the downward radiance at the
    // surface where the surface reflects, and keeps no level of its own way down
    Real rad[GC];
#pragma unroll
    for (int j = 0; j < GC; ++j) rad[j] = (Real)0;
    if (wave == 0) {
        u.store(rad, nlay, 0);
        sweep(rad, nlay, -1, 1, 3);
    } else if (wave == 1) {
        sweep(rad, nlay, -1, 1, -1);
        const Vec f = at(nlay + 1, 0);
        u.surface(f.x, rad);
        u.store(rad, 0, 1);
        sweep(rad, 1, 1, 2, 2);
    }
    __syncthreads();
    for (int lev = 1 + wave; lev <= nlay; lev += WAVES) {
        u.store(at(lev, 3).x, lev - 1, 0);
        u.store(at(lev, 2).x, lev, 1);
    }
}

// Persistent workgroups of WAVES waves; work items (a band of CPW columns) from
// a global counter, band by band, the bands with most work first.  LAYERS: a
// workgroup takes an item (lw_band_layers), the (exp, tfn) pairs are read from
// L2; else each wave takes items of its own, with the pairs in LDS.
template <typename Real, int WAVES, bool LAYERS>
__global__ __launch_bounds__(64 * WAVES)
    __attribute__((amdgpu_waves_per_eu(2))) void lw_band_kernel(ColumnInputs in, LwWork w,
                                                                const LwBand *__restrict__ bands, size_t row_elems,
                                                                int et_off, int plk_off,
                                                                const Real *__restrict__ tab,
                                                                const LwConst *__restrict__ cst)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int s_item;
    const ExpTfn<Real> *et;
    if constexpr (LAYERS) {
        et = (const ExpTfn<Real> *)(tab + et_off);
    } else {
        if (et_off >= 0) {
            const uint4 *src = (const uint4 *)(tab + et_off);
            constexpr int n = (int)((2 * (NTBL + 1) * sizeof(Real) + 15) / 16);
            for (int i = threadIdx.x; i < n; i += 64 * WAVES) ((uint4 *)smem_raw)[i] = src[i];
        }
        __syncthreads();
        et = (const ExpTfn<Real> *)smem_raw;
    }
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    Real *row = (Real *)w.dstate + ((size_t)blockIdx.x * (LAYERS ? 1 : WAVES) + (LAYERS ? 0 : wave)) * row_elems;
    for (;;) {
        int item = 0;
        if constexpr (LAYERS) {
            item = __builtin_amdgcn_readfirstlane(next_item(w.items, &s_item));
        } else {
            if (lane == 0) item = atomicAdd(w.items, 1);
            item = __builtin_amdgcn_readfirstlane(item);
        }
        // the item's band and its first column
#define UNIT(b, e) LwUnit<b, Real>(in, w, bands[b - 1], tab, tab, tab, e, plk_off, cst, item * lw_cpw(b), in.ncol, lane)
#define BODY(b)                                                                                                  \
    {                                                                                                            \
        const int n = (in.ncol + lw_cpw(b) - 1) / lw_cpw(b);                                                     \
        if (item < n) {                                                                                          \
            if constexpr (LAYERS)                                                                                \
                lw_band_layers<WAVES>(UNIT(b, et), wave, lane, row);                                                  \
            else if (sizeof(Real) == 4 || et_off >= 0)                                                           \
                lw_band_body(UNIT(b, et), lane, row);                                                            \
            else if constexpr (sizeof(Real) == 8)                                                                \
                lw_band_body(UNIT(b, nullptr), lane, row);                                                       \
            continue;                                                                                            \
        }                                                                                                        \
        item -= n;                                                                                               \
    }
        BODY(5) BODY(3) BODY(4) BODY(7) BODY(9) BODY(13) BODY(12) BODY(8)
        BODY(1) BODY(6) BODY(15) BODY(16) BODY(11) BODY(2) BODY(10) BODY(14)
#undef BODY
#undef UNIT
        return;
    }
}

#pragma clang fp contract(fast)

// FP32 kernel of the large calls: persistent 16-wave workgroups, one per CU,
// with the (exp, tfn) pairs and one band's k-tables in LDS (absb of bands 3-5,
// 75 KB, stays global).  Work item = one band of a tile of LW_TILE columns
// (LwTileSlots), one unit of CPW columns per wave (lw_claim_tile_item).
__global__ __launch_bounds__(1024) void lw_band_lds_kernel(ColumnInputs in, LwWork w,
                                                           const LwBand *__restrict__ bands_lds, LwLdsPlan plan,
                                                           size_t row_elems, int et_off, int plk_off,
                                                           const float *__restrict__ tab,
                                                           const LwConst *__restrict__ cst)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    ExpTfn<float> *et = (ExpTfn<float> *)smem_raw;
    float *ktab = (float *)(smem_raw + LW_ET_VECS * 16);
    for (int i = threadIdx.x; i < LW_ET_VECS; i += 1024) ((uint4 *)smem_raw)[i] = ((const uint4 *)(tab + et_off))[i];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    float *row = (float *)w.dstate + ((size_t)blockIdx.x * 16 + wave) * row_elems;
    const int ntiles = (in.ncol + LW_TILE - 1) / LW_TILE;
    __shared__ int s_item;
    int loaded = -1, queue = 0;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_item = lw_claim_tile_item(w.items, ntiles, queue);
        __syncthreads();
        const int item = __builtin_amdgcn_readfirstlane(s_item);
        if (item < 0) return;
        const int tile = item / LW_TILE_ITEMS, k = item - tile * LW_TILE_ITEMS;
        const LwTileSlot slot = LW_TILE_SLOTS.s[k];
        const int b = slot.band - 1;
        if (b != loaded) {
            lw_copy_tables(ktab, tab, plan, b);
            __syncthreads();
            loaded = b;
        }
        const int c0 = tile * LW_TILE + (slot.part * 16 + wave) * slot.cpw, cend = min((tile + 1) * LW_TILE, in.ncol);
        if (c0 >= cend) continue;
#define BODY(bb)                                                                                                  \
    case bb - 1:                                                                                                  \
        lw_band_body(LwUnit<bb, float>(in, w, bands_lds[bb - 1], ktab, bb >= 3 && bb <= 5 ? tab : ktab, tab, et,   \
                                       plk_off, cst, c0, cend, lane),                                             \
                     lane, row);                                                                                  \
        break;
        switch (b) {
            BODY(1) BODY(2) BODY(3) BODY(4) BODY(5) BODY(6) BODY(7) BODY(8)
            BODY(9) BODY(10) BODY(11) BODY(12) BODY(13) BODY(14) BODY(15) BODY(16)
        }
#undef BODY
    }
}

// finish: band sums, fluxfac, net flux and heating (rrtmg_lw_rtrnmr.f90:719-777),
// one thread per (layer, column): the fluxes of the layer's lower level (and
// of the top level) and its heating rate from the net fluxes of both levels
template <typename Real>
__global__ __launch_bounds__(256) void lw_finish_kernel(ColumnInputs in, LwWork w, LwOutputs out,
                                                        const LwBand *__restrict__ bands, double heatfac)
{
    const int ncol = in.ncol, nlay = in.nlay;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)nlay * ncol) return;
    const int lay = (int)(i / ncol), col = (int)(i - (size_t)lay * ncol);
    const Real *bflux = (const Real *)w.bflux;
    const size_t bstride = (size_t)(nlay + 1) * ncol;
    const double fluxfac = 2.0 * asin(1.0) * 2.e4;
    double fnet[2];
    for (int j = 0; j < 2; ++j) {
        const int k = lay + j;
        double up = 0.0, dn = 0.0;
        for (int b = 0; b < 16; ++b) {
            double dw = bands[b].delwave;
            up = up + ((double)bflux[(size_t)b * 2 * bstride + (size_t)k * ncol + col] * 0.5) * dw;
            dn = dn + ((double)bflux[(size_t)b * 2 * bstride + bstride + (size_t)k * ncol + col] * 0.5) * dw;
        }
        up = up * fluxfac;
        dn = dn * fluxfac;
        if (j == 0 || lay == nlay - 1) {
            size_t ix = (size_t)k * ncol + col;
            out.uflx[ix] = up;
            out.dflx[ix] = dn;
            out.uflxc[ix] = up;
            out.dflxc[ix] = dn;
        }
        fnet[j] = up - dn;
    }
    size_t il = (size_t)lay * ncol + col;
    double h = heatfac * (fnet[0] - fnet[1]) / (in.plev[il] - in.plev[il + ncol]);
    out.hr[il] = h;
    out.hrc[il] = h;
}

template <typename Real>
static hipError_t launch_lw_t(const ColumnInputs &in, const LwOutputs &out, const LwWork &w, const LwDevTables &t,
                              double heatfac, bool smooth, hipStream_t s, hipEvent_t *ev)
{
    const int nb = (in.ncol + 63) / 64;
    const int nbl = (int)(((size_t)in.nlay * in.ncol + 255) / 256);
    if (ev) (void)hipEventRecord(ev[0], s);
    hipLaunchKernelGGL(lw_prep_kernel<Real>, dim3(nbl), dim3(256), 0, s, in, w, t.cst);
    hipLaunchKernelGGL(lw_column_kernel, dim3(nb), dim3(256), 0, s, in, w);
    if (ev) (void)hipEventRecord(ev[1], s);
    hipLaunchKernelGGL(reset_items_kernel, dim3(1), dim3(8), 0, s, w.items);
    const size_t row = lw_fwd_state_bytes(in.nlay, 1), et = (2 * (NTBL + 1) * sizeof(Real) + 15) / 16 * 16;
    const int et_off = smooth ? -1 : t.desc.et_tbl;
    if constexpr (sizeof(Real) == 4) {
        if (w.kind == 16)
            hipLaunchKernelGGL(lw_band_lds_kernel, dim3(w.chunk), dim3(1024), (size_t)t.plan.fwd_lds_bytes, s, in, w,
                               t.bands_fwd, t.plan, row, et_off, t.desc.totplnk, (const float *)t.tab, t.cst);
    }
    if constexpr (sizeof(Real) == 8) {
        if (w.kind == 8)
            hipLaunchKernelGGL((lw_band_kernel<Real, 8, false>), dim3(w.chunk), dim3(512), smooth ? 0 : et, s, in, w,
                               t.bands, row, et_off, t.desc.totplnk, (const Real *)t.tab, t.cst);
    }
    if (w.kind == 1)
        hipLaunchKernelGGL((lw_band_kernel<Real, 8, true>), dim3(w.chunk), dim3(512), 0, s, in, w, t.bands,
                           lw_fwd_layers_bytes(in.nlay, 1), et_off, t.desc.totplnk, (const Real *)t.tab, t.cst);
    if (w.kind == 2)
        hipLaunchKernelGGL((lw_band_kernel<Real, 4, true>), dim3(w.chunk), dim3(256), 0, s, in, w, t.bands,
                           lw_fwd_layers_bytes(in.nlay, 1), et_off, t.desc.totplnk, (const Real *)t.tab, t.cst);
    if (ev) (void)hipEventRecord(ev[2], s);
    hipLaunchKernelGGL(lw_finish_kernel<Real>, dim3(nbl), dim3(256), 0, s, in, w, out, t.bands, heatfac);
    if (ev) (void)hipEventRecord(ev[3], s);
    return hipGetLastError();
}

hipError_t launch_lw_prep(const ColumnInputs &in, const LwWork &w, const LwDevTables &t, int mode, hipStream_t s)
{
    const int nb = (in.ncol + 63) / 64;
    const int nbl = (int)(((size_t)in.nlay * in.ncol + 255) / 256);
    if (mode == 1)
        hipLaunchKernelGGL(lw_prep_kernel<float>, dim3(nbl), dim3(256), 0, s, in, w, t.cst);
    else
        hipLaunchKernelGGL(lw_prep_kernel<double>, dim3(nbl), dim3(256), 0, s, in, w, t.cst);
    hipLaunchKernelGGL(lw_column_kernel, dim3(nb), dim3(256), 0, s, in, w);
    return hipGetLastError();
}

hipError_t launch_lw_finish(const ColumnInputs &in, const LwOutputs &out, void *bflux, const LwDevTables &t,
                            int mode, hipStream_t s)
{
    const int nbl = (int)(((size_t)in.nlay * in.ncol + 255) / 256);
    LwWork w;
    w.bflux = bflux;
    if (mode == 1)
        hipLaunchKernelGGL(lw_finish_kernel<float>, dim3(nbl), dim3(256), 0, s, in, w, out, t.bands, t.heatfac);
    else
        hipLaunchKernelGGL(lw_finish_kernel<double>, dim3(nbl), dim3(256), 0, s, in, w, out, t.bands, t.heatfac);
    return hipGetLastError();
}

hipError_t launch_lw(const ColumnInputs &in, const LwOutputs &out, const LwWork &w, const LwDevTables &t, int mode,
                     hipStream_t s, hipEvent_t *ev)
{
    return mode == 1 ? launch_lw_t<float>(in, out, w, t, t.heatfac, false, s, ev)
                     : launch_lw_t<double>(in, out, w, t, t.heatfac, mode == 2, s, ev);
}

}  // namespace rrtmg
