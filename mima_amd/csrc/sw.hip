// Shortwave RRTMG on gfx950: prep (inatm_sw + setcoef_sw), band kernel
// (taumol_sw + spcvrt_sw + reftra_sw + vrtqdr_sw per g-point) and finish
// (band sums, net flux, heating).  Reference: rrtmg_sw/gcm_model/src/ of
// MiMA's RRTMG_SW (file:line cited per function).
//
// Band kernels: a lane holds four or two g-points of one day column, LPC adjacent
// lanes a band, CPW columns a wave (SwLanes); the day columns come from a list,
// so that the waves of a grid row half in the night are full.  The gas optics
// are weighted table rows (sw_rows.hpp).  Each lane runs the adding method for
// its g-points: a bottom-up sweep keeps the reflectances below every level, a
// top-down sweep forms the layers' optics again, carries the downward state and
// produces the level fluxes, which are summed over the band's g-points into
// per-band fluxes.  What bounds it is VALU issue, 57% of its time at 32768 x 40,
// most of it the two-stream layer, evaluated once per sweep, and the latency of
// its chain: 1.15 ms -> 0.92 ms there against one g-point per lane with shuffled
// sums and FP64 two-stream layers in four times as many g-points.
//
// Calls below 6144 columns share a unit's layers among the waves of a workgroup
// and keep the optics (2261 x 59: 356 -> 231 us, 128 x 40: 104 -> 42 us).  A
// column's result is the same bits in each kernel (sw_fwd_kind).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "rrtmg_device.hpp"
#include "sw_optics.hpp"
#include "sw_rows.hpp"

namespace rrtmg {

// ---------------------------------------------------------------------------
// prep: FP64 (rrtmg_sw_rad.nomcica.f90:933-1047 and rrtmg_sw_setcoef.f90:129-284),
// one thread per (layer, column): the layer's coefficients in the band
// kernel's precision and its integer table indices.  GROUPS: in groups of four
// fields, [lay][group][col][4], for lanes that hold a column; else a record per
// (layer, column) (store_records), for the cloudy kernel's, which hold a
// g-point of few columns a wave and read a record as one line (in groups it ran
// 8-12% slower).
template <typename Real, bool GROUPS>
__global__ __launch_bounds__(256) void sw_prep_kernel(ColumnInputs in, SwWork w, const double *__restrict__ preflog,
                                                      const double *__restrict__ tref)
{
    const int ncol = in.ncol, nlay = in.nlay;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t n = (size_t)nlay * ncol, iblk = (size_t)blockIdx.x * blockDim.x;
    const int lay = (int)(i / ncol), col = (int)(i - (size_t)lay * ncol);
    __shared__ __align__(16) Real srec[GROUPS ? 4 : 256 * SWF_STRIDE];
    const double amd = 28.9660, amw = 18.0160, amdw = 1.607793, amdo = 0.603428;
    const double avogad = 6.02214199e+23, grav = 9.8066;
    const double stpfac = 296.0 / 1013.0;
    if (i < n) {
        const size_t ix = (size_t)lay * ncol + col;
        double pavel = in.play[ix], tavel = in.tlay[ix];
        double pz0 = in.plev[ix], pz1 = in.plev[ix + ncol];
        double h2o = in.h2o[ix];
        // in.vmr: h2o and O3 as volume mixing ratios (the McICA driver's
        // inatm, rrtmg_sw_rad.f90:1015, 1021), else MiMA's specific
        // humidity and O3 mass mixing ratio (rrtmg_sw_rad.nomcica.f90:1004, 1007)
        double wkl1 = in.vmr ? h2o : (h2o / (1.0 - h2o)) * amdw;
        double amm = (1.0 - wkl1) * amd + wkl1 * amw;
        double coldry = (pz0 - pz1) * 1.e3 * avogad / (1.e2 * grav * amm * (1.0 + wkl1));
        double colh2o = 1.e-20 * (coldry * wkl1);
        double colco2 = 1.e-20 * (coldry * in.co2[ix]);
        double colo3 = 1.e-20 * (coldry * (in.vmr ? in.o3[ix] : in.o3[ix] * amdo));
        double colch4 = 1.e-20 * (coldry * in.ch4[ix]);
        double colo2 = 1.e-20 * (coldry * in.o2[ix]);
        double colmol = 1.e-20 * coldry + colh2o;
        if (colco2 == 0.0) colco2 = 1.e-32 * coldry;
        if (colch4 == 0.0) colch4 = 1.e-32 * coldry;
        if (colo2 == 0.0) colo2 = 1.e-32 * coldry;

        double plog = log(pavel);
        int jp = clampi((int)(36.0 - 5 * (plog + 0.04)), 1, 58);
        double fp = 5.0 * (preflog[jp - 1] - plog);
        double dt0 = (tavel - tref[jp - 1]) / 15.0;
        int jt = clampi((int)(3.0 + dt0), 1, 4);
        double ft = dt0 - (double)(jt - 3);
        double dt1 = (tavel - tref[jp]) / 15.0;
        int jt1 = clampi((int)(3.0 + dt1), 1, 4);
        double ft1 = dt1 - (double)(jt1 - 3);
        double water = (coldry * wkl1) / coldry;
        double scalefac = pavel * stpfac / tavel;
        double forfac, forfrac, selffac, selffrac;
        int indfor, indself;
        if (plog > 4.56) {
            forfac = scalefac / (1. + water);
            double factor = (332.0 - tavel) / 36.0;
            indfor = clampi((int)factor, 1, 2);
            forfrac = factor - (double)indfor;
            selffac = water * forfac;
            factor = (tavel - 188.0) / 7.2;
            indself = clampi((int)factor - 7, 1, 9);
            selffrac = factor - (double)(indself + 7);
        } else {
            forfac = scalefac / (1. + water);
            double factor = (tavel - 188.0) / 36.0;
            indfor = 3;
            forfrac = factor - 1.0;
            selffac = 0.0;
            selffrac = 0.0;
            indself = 0;
        }
        double compfp = 1.0 - fp;
        Real rec[SWF_STRIDE];
        rec[SWF_FAC10] = (Real)(compfp * ft);
        rec[SWF_FAC00] = (Real)(compfp * (1.0 - ft));
        rec[SWF_FAC11] = (Real)(fp * ft1);
        rec[SWF_FAC01] = (Real)(fp * (1.0 - ft1));
        rec[SWF_COLH2O] = (Real)colh2o;
        rec[SWF_COLCO2] = (Real)colco2;
        rec[SWF_COLO3] = (Real)colo3;
        rec[SWF_COLCH4] = (Real)colch4;
        rec[SWF_COLO2] = (Real)colo2;
        rec[SWF_COLMOL] = (Real)colmol;
        rec[SWF_SELFFAC] = (Real)selffac;
        rec[SWF_SELFFRAC] = (Real)selffrac;
        rec[SWF_FORFAC] = (Real)forfac;
        rec[SWF_FORFRAC] = (Real)forfrac;
        w.ipk[ix] = pack_sw(jp, jt, jt1, indself, indfor);
        for (int f = SWF_COUNT; f < SWF_STRIDE; ++f) rec[f] = (Real)0;
        if constexpr (GROUPS) {
            struct alignas(16) Group {
                Real x[4];
            };
            Group *g = (Group *)w.coef + (size_t)lay * SWF_GROUPS * ncol + col;
#pragma unroll
            for (int k = 0; k < SWF_GROUPS; ++k)
                g[(size_t)k * ncol] = {rec[4 * k], rec[4 * k + 1], rec[4 * k + 2], rec[4 * k + 3]};
        } else {
#pragma unroll
            for (int f = 0; f < SWF_STRIDE; ++f) srec[threadIdx.x * SWF_STRIDE + f] = rec[f];
        }
    }
    if constexpr (!GROUPS) {
        const int nrec = (int)(n - iblk < blockDim.x ? n - iblk : blockDim.x);
        store_records<Real, SWF_STRIDE>((Real *)w.coef + iblk * SWF_STRIDE, srec, nrec);
    }
}

// per-column part of the prep (sw_column_refs): laytrop, the solar-source
// reference layers and, where w.day is given, the list of day columns, which
// the band kernel's lanes are filled from (64 columns in order; the order of
// the blocks does not matter, columns being independent)
__global__ __launch_bounds__(256) void sw_column_kernel(ColumnInputs in, SwWork w)
{
    const int col0 = blockIdx.x * 64, lane = (int)threadIdx.x & 63, col = col0 + lane;
    if (w.day && threadIdx.x < 64) {
        const bool day = col < in.ncol && in.coszen[col] >= 1.e-10;
        const unsigned long long m = __builtin_amdgcn_ballot_w64(day);
        int base = 0;
        if (lane == 0 && m) base = atomicAdd(w.items + 1, __popcll(m));
        base = __builtin_amdgcn_readfirstlane(base);
        if (day) w.day[base + __popcll(m & ((1ull << lane) - 1))] = col;
    }
    sw_column_refs(w.ipk, in.ncol, in.nlay, col0, w.laytrop, w.laysolfr);
}

// contraction off, as in sw_rows.hpp
#pragma clang fp contract(off)

// Sum of a column's g-points on its first lane, in FP64 and rounded once: over
// pairs, then fours, then the rest, in the same order for either W.
template <int JB, int W, typename Real>
__device__ __forceinline__ Real band_sum(const Real (&v)[SwLanes<JB, W>::GC])
{
    using L = SwLanes<JB, W>;
    double s = (double)v[0] + (double)v[1];
    if constexpr (L::NG % 4 == 0) {
        constexpr int step = L::GC == 4 ? 1 : 2, fours = L::NG / 4;
        if constexpr (L::GC == 4)
            s = s + ((double)v[2] + (double)v[3]);
        else
            s = s + __shfl_down(s, 1);
        if constexpr (fours == 2) s = s + __shfl_down(s, step);
        if constexpr (fours == 3) s = s + (__shfl_down(s, step) + __shfl_down(s, 2 * step));
    } else if constexpr (L::NG == 6) {
        s = s + (__shfl_down(s, 1) + __shfl_down(s, 2));
    } else if constexpr (L::NG == 10) {
        const double r = __shfl_down(s, 4);
        s = s + __shfl_down(s, 1);
        s = s + __shfl_down(s, 2);
        s = s + r;
    }
    return (Real)s;
}

// What a wave needs of one band and the columns [c0, c0 + CPW) below cend of the
// day list (of all columns where there is none).  tab: the packed k-tables;
// tbl: the exp table (global or LDS), or NULL for the function itself.
template <int JB, int W, typename Real>
struct SwUnit {
    using L = SwLanes<JB, W>;
    static constexpr int NG = L::NG, GC = L::GC;
    const ColumnInputs &in;
    const SwWork &w;
    const SwBand &B;
    const Real *__restrict__ tab, *__restrict__ tbl;
    int g0, col, laytrop;
    bool day, first;  // first: the lane that stores the column's sums
    Real mu, imu, albp, albd, zinc[GC];
    __device__ __forceinline__ SwUnit(const ColumnInputs &in_, const SwWork &w_, const SwBand &B_, const Real *tab_,
                                      const Real *tbl_, int c0, int cend, int lane)
        : in(in_), w(w_), B(B_), tab(tab_), tbl(tbl_)
    {
        const int cl = lane / L::LPC;
        g0 = (lane - cl * L::LPC) * GC;
        const bool active = cl < L::CPW && c0 + cl < cend;
        col = active ? c0 + cl : cend - 1;
        if (w.day) col = w.day[col];
        day = in.coszen[col] >= 1.e-10;
        first = active && day && g0 == 0;
        laytrop = w.laytrop[col];
        mu = day ? (Real)in.coszen[col] : (Real)1;
        imu = fdiv((Real)1, mu);
        constexpr bool nir = JB <= 24 || JB == 29;  // rrtmg_sw_rad.nomcica.f90:567-577
        albp = (Real)(nir ? in.aldir[col] : in.asdir[col]);
        albd = (Real)(nir ? in.aldif[col] : in.asdif[col]);
        const int lsf = w.laysolfr[(size_t)(JB - 16) * in.ncol + col];
        SwLayer<Real> c;
        load(c, lsf);
#pragma unroll
        for (int j = 0; j < GC; ++j)
            zinc[j] = (Real)(in.adjflux * sw_sfluxzen(JB, B, Tab<Real>{tab, NG, g0 + j}, c, lsf <= laytrop) * (double)mu);
    }
    __device__ __forceinline__ void load(SwLayer<Real> &c, int lay) const
    {
        sw_load_groups(c, (const Real *)w.coef, w.ipk, lay - 1, col, in.ncol);
    }
    // gas and Rayleigh optical depths of layer lay
    __device__ __forceinline__ void depths(int lay, Real (&tg)[GC], Real (&tr)[GC]) const
    {
        SwLayer<Real> c;
        load(c, lay);
#pragma unroll
        for (int j = 0; j < GC; ++j) tg[j] = tr[j] = (Real)0;
        auto rows = [&](Real (&v)[GC], int off, int r, Real wt) {
            Real k[GC];
            load_row<NG>(k, tab, (unsigned)(off + (r - 1) * NG + g0));
#pragma unroll
            for (int j = 0; j < GC; ++j) v[j] = fma(wt, k[j], v[j]);
        };
        const SwFlat<Real> f =
            sw_rows<JB, Real>(B, c, lay <= laytrop, [&](int off, int r, Real wt) { rows(tg, off, r, wt); },
                              [&](int off, int r, Real wt) { rows(tr, off, r, wt); });
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            tg[j] = tg[j] + f.taug;
            tr[j] = tr[j] + f.taur;
        }
    }
    __device__ __forceinline__ SwOptics<Real> optics(Real tg, Real tr) const
    {
        return sw_clear_layer(tg, tr, mu, imu, tbl);
    }
    // one layer of the bottom-up sweep (rrtmg_sw_vrtqdr.f90:103-117): the
    // reflectances (pu, pud) of the atmosphere below its top
    static __device__ __forceinline__ void up(const SwOptics<Real> &l, Real &pu, Real &pud)
    {
        const Real z = fdiv((Real)1, fma(-pud, l.rd, (Real)1));
        const Real nu = fma(l.td * fma(l.t - l.dbt, pud, l.dbt * pu), z, l.r);
        pud = fma(l.td * l.td * pud, z, l.rd);
        pu = nu;
    }
    // one layer of the top-down sweep (:119-137)
    static __device__ __forceinline__ void down(const SwOptics<Real> &l, Real &tdn, Real &rdn, Real &beam)
    {
        const Real z = fdiv((Real)1, fma(-l.rd, rdn, (Real)1));
        tdn = fma(l.td * fma(beam * l.r, rdn, tdn - beam), z, beam * l.t);
        rdn = fma(l.td * l.td * rdn, z, l.rd);
        beam = l.dbt * beam;
    }
    // fluxes of the g-points at a level (:139-150), times the incoming flux
    __device__ __forceinline__ void flux(int j, Real pu, Real pud, Real tdn, Real rdn, Real beam, Real &fu, Real &fd) const
    {
        const Real z = fdiv((Real)1, fma(-rdn, pud, (Real)1)), dif = tdn - beam;
        fu = zinc[j] * (fma(dif, pud, beam * pu) * z);
        fd = zinc[j] * fma(fma(beam * pu, rdn, dif), z, beam);
    }
    __device__ __forceinline__ void store(const Real (&fu)[GC], const Real (&fd)[GC], int lev) const
    {
        const size_t bs = (size_t)(in.nlay + 1) * in.ncol;
        Real *bf = (Real *)w.bflux + (size_t)(JB - 16) * 2 * bs;
        const Real su = band_sum<JB, W>(fu), sd = band_sum<JB, W>(fd);
        if (first) {
            at32(bf, (unsigned)(lev * in.ncol + col)) = su;
            at32(bf + bs, (unsigned)(lev * in.ncol + col)) = sd;
        }
    }
};

// One unit by one wave (rrtmg_sw_spcvrt.f90:302-600 with
// rrtmg_sw_vrtqdr.f90:28-152, clear sky): the bottom-up sweep keeps the
// reflectances below every level in the wave's scratch row,
// [nlay + 1][2][64][GC], the top-down sweep forms the layers' optics again
// (keeping them too costs more in traffic than forming them).
template <int JB, int W, typename Real>
__device__ __forceinline__ void sw_band_body(const SwUnit<JB, W, Real> u, int lane, Real *__restrict__ row)
{
    constexpr int GC = SwUnit<JB, W, Real>::GC;
    using Vec = GVec<GC, Real>;
    const int nlay = u.in.nlay;
    auto at = [&](int lev, int k) -> Vec & { return at32((Vec *)row, (unsigned)((lev * 2 + k) * 64 + lane)); };
    Vec pu, pud;
#pragma unroll
    for (int j = 0; j < GC; ++j) {
        pu.x[j] = u.albp;
        pud.x[j] = u.albd;
    }
    at(0, 0) = pu;
    at(0, 1) = pud;
    for (int lay = 1; lay <= nlay; ++lay) {
        Real tg[GC], tr[GC];
        u.depths(lay, tg, tr);
#pragma unroll
        for (int j = 0; j < GC; ++j) u.up(u.optics(tg[j], tr[j]), pu.x[j], pud.x[j]);
        at(lay, 0) = pu;
        at(lay, 1) = pud;
    }
    Real tdn[GC], rdn[GC], beam[GC], fu[GC], fd[GC];
#pragma unroll
    for (int j = 0; j < GC; ++j) {
        tdn[j] = beam[j] = (Real)1;
        rdn[j] = (Real)0;
    }
    for (int lev = nlay; lev >= 0; --lev) {
        // the reflectances below the next level, read a layer ahead of their use
        Vec nu, nud;
        if (lev > 0) {
            nu = at(lev - 1, 0);
            nud = at(lev - 1, 1);
        }
#pragma unroll
        for (int j = 0; j < GC; ++j) u.flux(j, pu.x[j], pud.x[j], tdn[j], rdn[j], beam[j], fu[j], fd[j]);
        u.store(fu, fd, lev);
        if (lev == 0) break;
        Real tg[GC], tr[GC];
        u.depths(lev, tg, tr);
#pragma unroll
        for (int j = 0; j < GC; ++j) u.down(u.optics(tg[j], tr[j]), tdn[j], rdn[j], beam[j]);
        pu = nu;
        pud = nud;
    }
}

// One unit by a workgroup of WAVES waves, for calls too small to fill the chip
// with waves: the layers' optics are shared out among the waves and kept, one
// wave sweeps up and one down through them, and all form the fluxes.  row: the
// workgroup's scratch, [nlay + 1][10][64][GC]: optics of the layer below a
// level (r, rd, t, td, dbt), reflectances below it, and the downward state.
template <int WAVES, int JB, int W, typename Real>
__device__ __forceinline__ void sw_band_layers(const SwUnit<JB, W, Real> u, int wave, int lane, Real *__restrict__ row)
{
    constexpr int GC = SwUnit<JB, W, Real>::GC;
    using Vec = GVec<GC, Real>;
    const int nlay = u.in.nlay;
    auto at = [&](int lev, int k) -> Vec & { return at32((Vec *)row, (unsigned)((lev * 10 + k) * 64 + lane)); };
    for (int lay = 1 + wave; lay <= nlay; lay += WAVES) {
        Real tg[GC], tr[GC];
        u.depths(lay, tg, tr);
        Vec v[5];
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            const SwOptics<Real> o = u.optics(tg[j], tr[j]);
            v[0].x[j] = o.r;
            v[1].x[j] = o.rd;
            v[2].x[j] = o.t;
            v[3].x[j] = o.td;
            v[4].x[j] = o.dbt;
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) at(lay, k) = v[k];
    }
    __syncthreads();
    auto load = [&](Vec (&v)[5], int lay) {
#pragma unroll
        for (int k = 0; k < 5; ++k) v[k] = at(clampi(lay, 1, nlay), k);
    };
    auto layer = [](const Vec (&v)[5], int j) {
        return SwOptics<Real>{v[0].x[j], v[1].x[j], v[2].x[j], v[3].x[j], v[4].x[j]};
    };
    Vec n[2][5];
    if (wave == 0) {
        Vec pu, pud;
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            pu.x[j] = u.albp;
            pud.x[j] = u.albd;
        }
        at(0, 5) = pu;
        at(0, 6) = pud;
        load(n[0], 1);
        load(n[1], 2);
        for (int l0 = 1; l0 <= nlay; l0 += 2)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int lay = l0 + i;
                if (lay > nlay) break;
#pragma unroll
                for (int j = 0; j < GC; ++j) u.up(layer(n[i], j), pu.x[j], pud.x[j]);
                load(n[i], lay + 2);
                at(lay, 5) = pu;
                at(lay, 6) = pud;
            }
    } else if (wave == 1) {
        Vec tdn, rdn, beam;
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            tdn.x[j] = beam.x[j] = (Real)1;
            rdn.x[j] = (Real)0;
        }
        load(n[0], nlay);
        load(n[1], nlay - 1);
        for (int l0 = nlay; l0 >= 0; l0 -= 2)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int lev = l0 - i;
                if (lev < 0) break;
                at(lev, 7) = tdn;
                at(lev, 8) = rdn;
                at(lev, 9) = beam;
                if (lev == 0) break;
#pragma unroll
                for (int j = 0; j < GC; ++j) u.down(layer(n[i], j), tdn.x[j], rdn.x[j], beam.x[j]);
                load(n[i], lev - 2);
            }
    }
    __syncthreads();
    for (int lev = wave; lev <= nlay; lev += WAVES) {
        const Vec pu = at(lev, 5), pud = at(lev, 6), tdn = at(lev, 7), rdn = at(lev, 8), beam = at(lev, 9);
        Real fu[GC], fd[GC];
#pragma unroll
        for (int j = 0; j < GC; ++j) u.flux(j, pu.x[j], pud.x[j], tdn.x[j], rdn.x[j], beam.x[j], fu[j], fd[j]);
        u.store(fu, fd, lev);
    }
}
#pragma clang fp contract(fast)

// Persistent workgroups of WAVES waves; work items (a band of CPW day columns)
// from a global counter, band by band, the bands with most work first.  LAYERS:
// a workgroup takes an item (sw_band_layers), the exp table is read from L2;
// else each wave takes items of its own, with the table in LDS.
template <typename Real, int WAVES, int W, bool LAYERS>
__global__ __launch_bounds__(64 * WAVES)
    __attribute__((amdgpu_waves_per_eu(sizeof(Real) == 4 ? 4 : 2))) void sw_band_kernel(ColumnInputs in, SwWork w,
                                                                                       const SwBand *__restrict__ bands,
                                                                                       size_t row_elems, int nrows,
                                                                                       int exp_off,
                                                                                       const Real *__restrict__ tab)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int s_item;
    if constexpr (!LAYERS) {
        if (exp_off >= 0) {
            const uint4 *src = (const uint4 *)(tab + exp_off);
            constexpr int n = (int)(((NTBL + 1) * sizeof(Real) + 15) / 16);
            for (int i = threadIdx.x; i < n; i += 64 * WAVES) ((uint4 *)smem_raw)[i] = src[i];
        }
        __syncthreads();
    }
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    const int r = (int)blockIdx.x * (LAYERS ? 1 : WAVES) + (LAYERS ? 0 : wave);
    if (r >= nrows) return;  // uniform over the workgroup with LAYERS
    Real *row = (Real *)w.dstate + (size_t)r * row_elems;
    const int ncol = w.day ? w.items[1] : in.ncol;
    for (;;) {
        int item = 0;
        if constexpr (LAYERS) {
            item = __builtin_amdgcn_readfirstlane(next_item(w.items, &s_item));
        } else {
            if (lane == 0) item = atomicAdd(w.items, 1);
            item = __builtin_amdgcn_readfirstlane(item);
        }
        // the item's band and its first column
#define UNIT(b, e) SwUnit<b, W, Real>(in, w, bands[b - 16], tab, e, item * sw_cpw(b, W), ncol, lane)
#define BODY(b)                                                                                                  \
    {                                                                                                            \
        const int n = (ncol + sw_cpw(b, W) - 1) / sw_cpw(b, W);                                                  \
        if (item < n) {                                                                                          \
            if constexpr (LAYERS)                                                                                \
                sw_band_layers<WAVES>(UNIT(b, tab + exp_off), wave, lane, row);                                  \
            else if (sizeof(Real) == 4 || exp_off >= 0)                                                          \
                sw_band_body(UNIT(b, (const Real *)smem_raw), lane, row);                                        \
            else if constexpr (sizeof(Real) == 8)                                                                \
                sw_band_body(UNIT(b, nullptr), lane, row);                                                       \
            continue;                                                                                            \
        }                                                                                                        \
        item -= n;                                                                                               \
    }
        BODY(17) BODY(21) BODY(24) BODY(18) BODY(19) BODY(16) BODY(20) BODY(29)
        BODY(28) BODY(27) BODY(23) BODY(25) BODY(26) BODY(22)
#undef BODY
#undef UNIT
        return;
    }
}

// finish: band sums, net flux and heating (rrtmg_sw_rad.nomcica.f90:700-726),
// one thread per (layer, column): the fluxes of the layer's lower level (and
// of the top level) and its heating rate, zero in the top layer
template <typename Real>
__global__ __launch_bounds__(256) void sw_finish_kernel(ColumnInputs in, SwWork w, SwOutputs out, double heatfac)
{
    const int ncol = in.ncol, nlay = in.nlay;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)nlay * ncol) return;
    const int lay = (int)(i / ncol), col = (int)(i - (size_t)lay * ncol);
    const Real *bflux = (const Real *)w.bflux;
    const size_t bstride = (size_t)(nlay + 1) * ncol;
    const size_t il = (size_t)lay * ncol + col;
    if (in.coszen[col] < 1.e-10) {
        for (int k = lay; k <= (lay == nlay - 1 ? nlay : lay); ++k) {
            size_t ix = (size_t)k * ncol + col;
            out.uflx[ix] = 0.0;
            out.dflx[ix] = 0.0;
            out.uflxc[ix] = 0.0;
            out.dflxc[ix] = 0.0;
        }
        out.hr[il] = 0.0;
        out.hrc[il] = 0.0;
        return;
    }
    double net[2];
    for (int j = 0; j < 2; ++j) {
        const int k = lay + j;
        double up = 0.0, dn = 0.0;
        for (int b = 0; b < 14; ++b) {
            up += (double)bflux[(size_t)b * 2 * bstride + (size_t)k * ncol + col];
            dn += (double)bflux[(size_t)b * 2 * bstride + bstride + (size_t)k * ncol + col];
        }
        if (j == 0 || lay == nlay - 1) {
            size_t ix = (size_t)k * ncol + col;
            out.uflx[ix] = up;
            out.dflx[ix] = dn;
            out.uflxc[ix] = up;
            out.dflxc[ix] = dn;
        }
        net[j] = dn - up;
    }
    double pdp = in.plev[il] - in.plev[il + ncol];
    double h = (lay == nlay - 1) ? 0.0 : (net[1] - net[0]) * (heatfac / pdp);
    out.hr[il] = h;
    out.hrc[il] = h;
}

template <typename Real>
static hipError_t launch_sw_t(const ColumnInputs &in, const SwOutputs &out, const SwWork &w, const SwDevTables &t,
                              bool smooth, hipStream_t s, hipEvent_t *ev)
{
    const int nb = (in.ncol + 63) / 64;
    const int nbl = (int)(((size_t)in.nlay * in.ncol + 255) / 256);
    if (ev) (void)hipEventRecord(ev[0], s);
    hipLaunchKernelGGL(reset_items_kernel, dim3(1), dim3(2), 0, s, w.items);
    hipLaunchKernelGGL((sw_prep_kernel<Real, true>), dim3(nbl), dim3(256), 0, s, in, w, t.preflog, t.tref);
    hipLaunchKernelGGL(sw_column_kernel, dim3(nb), dim3(256), 0, s, in, w);
    if (ev) (void)hipEventRecord(ev[1], s);
    const size_t row = sw_fwd_rows_bytes(in.nlay, 1, w.kind);
    const int exp_off = smooth ? -1 : t.desc.exp_tbl;
    const size_t lds = smooth ? 0 : ((NTBL + 1) * sizeof(Real) + 15) / 16 * 16;
#define LAUNCH(WAVES, W, LAYERS, blocks, bytes)                                                                      \
    hipLaunchKernelGGL((sw_band_kernel<Real, WAVES, W, LAYERS>), dim3(blocks), dim3(64 * WAVES), bytes, s, in, w,    \
                       t.bands, row, w.rows, exp_off, (const Real *)t.tab)
    if (w.kind == SW_WAVE4) LAUNCH(8, 4, false, (w.rows + 7) / 8, lds);
    if (w.kind == SW_WAVE2) LAUNCH(8, 2, false, (w.rows + 7) / 8, lds);
    if (w.kind == SW_GROUP8) LAUNCH(8, 2, true, w.rows, 0);
    if (w.kind == SW_GROUP4) LAUNCH(4, 2, true, w.rows, 0);
#undef LAUNCH
    if (ev) (void)hipEventRecord(ev[2], s);
    hipLaunchKernelGGL(sw_finish_kernel<Real>, dim3(nbl), dim3(256), 0, s, in, w, out, t.heatfac);
    if (ev) (void)hipEventRecord(ev[3], s);
    return hipGetLastError();
}

hipError_t launch_sw_prep(const ColumnInputs &in, const SwWork &w, const SwDevTables &t, int mode, hipStream_t s)
{
    const int nb = (in.ncol + 63) / 64;
    const int nbl = (int)(((size_t)in.nlay * in.ncol + 255) / 256);
    if (mode == 1)
        hipLaunchKernelGGL((sw_prep_kernel<float, false>), dim3(nbl), dim3(256), 0, s, in, w, t.preflog, t.tref);
    else
        hipLaunchKernelGGL((sw_prep_kernel<double, false>), dim3(nbl), dim3(256), 0, s, in, w, t.preflog, t.tref);
    hipLaunchKernelGGL(sw_column_kernel, dim3(nb), dim3(256), 0, s, in, w);
    return hipGetLastError();
}

hipError_t launch_sw_finish(const ColumnInputs &in, const SwOutputs &out, void *bflux, const SwDevTables &t,
                            int mode, hipStream_t s)
{
    const int nbl = (int)(((size_t)in.nlay * in.ncol + 255) / 256);
    SwWork w;
    w.bflux = bflux;
    if (mode == 1)
        hipLaunchKernelGGL(sw_finish_kernel<float>, dim3(nbl), dim3(256), 0, s, in, w, out, t.heatfac);
    else
        hipLaunchKernelGGL(sw_finish_kernel<double>, dim3(nbl), dim3(256), 0, s, in, w, out, t.heatfac);
    return hipGetLastError();
}

hipError_t launch_sw(const ColumnInputs &in, const SwOutputs &out, const SwWork &w, const SwDevTables &t, int mode,
                     hipStream_t s, hipEvent_t *ev)
{
    return mode == 1 ? launch_sw_t<float>(in, out, w, t, false, s, ev)
                     : launch_sw_t<double>(in, out, w, t, mode == 2, s, ev);
}

}  // namespace rrtmg
