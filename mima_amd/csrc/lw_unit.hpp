// One band of a wave's columns in the LW band kernels, forward and backward: a
// lane holds LwLanes<BAND>::GC g-points of one column.
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "lw_optics.hpp"
#include "lw_rows.hpp"
#include "rrtmg_device.hpp"

namespace rrtmg {

[[maybe_unused]] static __constant__ constexpr LwTileSlots LW_TILE_SLOTS{};

// 16-byte vectors of the FP32 (exp, tfn) pairs, at the start of the LDS of the
// kernels that keep them and a band's k-tables there
constexpr int LW_ET_VECS = (int)((2 * (NTBL + 1) * sizeof(float) + 15) / 16);

// Item of a persistent kernel whose workgroups take the LW_TILE_ITEMS bands of
// tiles of LW_TILE columns: each XCD claims the tiles t = xcd (mod 8) from its
// own counter, so the bands that read a tile's coefficients share an L2, and
// takes other XCDs' items when its own are gone.  queue: the caller's, from 0;
// -1: none left.  One thread of the workgroup calls it.
__device__ __forceinline__ int lw_claim_tile_item(int *items, int ntiles, int &queue)
{
    for (; queue < 8; ++queue) {
        const int x = ((int)blockIdx.x + queue) & 7;
        const int n = ((ntiles - x + 7) >> 3) * LW_TILE_ITEMS;
        const int k = n > 0 ? atomicAdd(items + x, 1) : n;
        if (k < n) return (x + 8 * (k / LW_TILE_ITEMS)) * LW_TILE_ITEMS + k % LW_TILE_ITEMS;
    }
    return -1;
}
// a band's k-tables into LDS but for [cut0, cut1), absb where it stays global
__device__ __forceinline__ void lw_copy_tables(float *__restrict__ ktab, const float *__restrict__ tab,
                                               const LwLdsPlan &plan, int b)
{
    const int t0 = plan.tab0[b], n = plan.tab0[b + 1] - t0, c0 = plan.cut0[b], c1 = plan.cut1[b];
    for (int i = threadIdx.x; i < n / 4; i += blockDim.x)
        if (i < c0 / 4 || i >= c1 / 4)
            ((float4 *)ktab)[i < c0 / 4 ? i : i - (c1 - c0) / 4] = ((const float4 *)(tab + t0))[i];
    // what the dummies of a band's last lane read past the last row
    if (threadIdx.x == 0) ((float4 *)ktab)[(n - (c1 - c0)) / 4] = {0.f, 0.f, 0.f, 0.f};
}

// contraction off, as in lw_rows.hpp
#pragma clang fp contract(off)

// Sum of a column's g-points on its first lane: exact enough in FP64 (the sum
// is rounded once to FP32, and FP64 differs from the reference's order by its
// last digits only).
template <int BAND, typename Real>
__device__ __forceinline__ Real band_sum(const Real (&v)[LwLanes<BAND>::GC], int g0)
{
    using L = LwLanes<BAND>;
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < L::GC; ++j) {
        const bool in = L::NG % L::GC == 0 || g0 + j < L::NG;
        s = j == 0 ? (double)v[0] : in ? s + (double)v[j] : s;
    }
    if constexpr (L::LPC == 2) s = s + __shfl_down(s, 1);
    if constexpr (L::LPC == 3) s = s + (__shfl_down(s, 1) + __shfl_down(s, 2));
    if constexpr (L::LPC == 4) {
        s = s + __shfl_down(s, 1);
        s = s + __shfl_down(s, 2);
    }
    return (Real)s;
}

// (exp(-tau), tau transition function) entries of the 10000-interval tables
template <typename Real>
struct alignas(2 * sizeof(Real)) ExpTfn {
    Real e, t;
};

// What a wave needs of one band and CPW columns from column c0 on, below cend.
// ktab: the band's k-tables, at B's offsets (global, or a copy in LDS); ktab_b:
// those of the upper atmosphere's major species (absb); tab: the packed global
// buffer (Planck); et: the (exp, tfn) pairs (global or LDS), or NULL for the
// smooth functions.
template <int BAND, typename Real>
struct LwUnit {
    using L = LwLanes<BAND>;
    static constexpr int NG = L::NG, GC = L::GC;
    const ColumnInputs &in;
    const LwWork &w;
    const LwBand &B;
    const Real *__restrict__ ktab, *__restrict__ ktab_b, *__restrict__ plk;
    const ExpTfn<Real> *et;
    const LwConst *__restrict__ cst;
    int g0, col, laytrop;
    bool first;  // the lane that stores the column's sums
    Real secdiff;
    __device__ __forceinline__ LwUnit(const ColumnInputs &in_, const LwWork &w_, const LwBand &B_,
                                      const Real *ktab_, const Real *ktab_b_, const Real *tab,
                                      const ExpTfn<Real> *et_, int plk_off, const LwConst *cst_, int c0, int cend,
                                      int lane)
        : in(in_), w(w_), B(B_), ktab(ktab_), ktab_b(ktab_b_), plk(tab + plk_off + (BAND - 1) * 181), et(et_), cst(cst_)
    {
        const int cl = lane / L::LPC;
        g0 = (lane - cl * L::LPC) * GC;
        const bool active = cl < L::CPW && c0 + cl < cend;
        col = active ? c0 + cl : cend - 1;
        first = active && g0 == 0;
        laytrop = w.laytrop[col];
        // diffusivity secant (rrtmg_lw_rtrnmr.f90:272-280)
        double sd = 1.66;
        if (!(BAND == 1 || BAND == 4 || BAND >= 10)) {
            sd = B.a0 + B.a1 * exp(B.a2 * w.colscal[col]);
            if (sd > 1.80) sd = 1.80;
            if (sd < 1.50) sd = 1.50;
        }
        secdiff = (Real)sd;
    }
    __device__ __forceinline__ void load(LwLayer<Real> &c, int lev) const
    {
        lw_load_layer(c, (const Real *)w.coef, w.ipk, lev - 1, col, in.ncol, in.nlay);
    }
    __device__ __forceinline__ Real planklev(int lev) const
    {
        const int i = at32(w.ilev, (unsigned)(lev * in.ncol + col));
        const Real f = at32((const Real *)w.tlev, (unsigned)(lev * in.ncol + col));
        return fma(f, at32(plk, (unsigned)i) - at32(plk, (unsigned)(i - 1)), at32(plk, (unsigned)(i - 1)));
    }
    __device__ __forceinline__ Real planklay(const LwLayer<Real> &c) const
    {
        return fma(c.tlayfrac, at32(plk, (unsigned)c.indlay) - at32(plk, (unsigned)(c.indlay - 1)),
                   at32(plk, (unsigned)(c.indlay - 1)));
    }
    // optical depths on the diffusivity path of layer lev, from its record
    __device__ __forceinline__ void depths(const LwLayer<Real> &c, int lev, Real (&od)[GC]) const
    {
        const bool lower = lev <= laytrop;
#pragma unroll
        for (int j = 0; j < GC; ++j) od[j] = (Real)0;
        lw_rows<BAND, Real>(B, cst, c, lower, [&](auto where, int off, int r, Real wt) {
            Real k[GC];
            load_row<NG>(k, where == LW_ABSB ? ktab_b : ktab, (unsigned)(off + (r - 1) * NG + g0));
#pragma unroll
            for (int j = 0; j < GC; ++j) od[j] = fma(wt, k[j], od[j]);
        });
        const Real ta =
            in.tauaer ? (Real)in.tauaer[((size_t)(BAND - 1) * in.nlay + (lev - 1)) * in.ncol + col] : (Real)0;
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            if constexpr (BAND == 4 || BAND == 7) od[j] = od[j] * lw_gfactor<BAND, Real>(g0 + j, lower);
            od[j] = secdiff * (od[j] + ta);
            if (od[j] < (Real)0) od[j] = (Real)0;
        }
    }
    // Planck fractions of layer lev
    __device__ __forceinline__ void fracs(const LwLayer<Real> &c, int lev, Real (&fr)[GC]) const
    {
#pragma unroll
        for (int j = 0; j < GC; ++j) fr[j] = (Real)0;
        lw_fracs<BAND, Real>(B, cst, c, lev <= laytrop, [&](int off, int r, Real wt) {
            Real k[GC];
            load_row<NG>(k, ktab, (unsigned)(off + (r - 1) * NG + g0));
#pragma unroll
            for (int j = 0; j < GC; ++j) fr[j] = fma(wt, k[j], fr[j]);
        });
    }
    // transmittance and transition function of an optical depth
    __device__ __forceinline__ void transmit(Real od, Real &atr, Real &tf) const
    {
        if (!et) {  // smooth mode: the tabulated functions at every depth
            const LwRT<Real> rt = lw_rt_exact(od, false);
            atr = rt.atrans;
            tf = rt.tf;
        } else {
            const ExpTfn<Real> x = et[tbl_index(od)];
            const bool thin = od <= (Real)0.06;
            atr = thin ? fma((Real)-0.5 * od, od, od) : (Real)1 - x.e;
            tf = thin ? (Real)0.166667 * od : x.t;
        }
    }
    // d secdiff / d pwvcm, where the secant is not at a limit
    __device__ __forceinline__ Real dsecdiff() const
    {
        if (BAND == 1 || BAND == 4 || BAND >= 10) return (Real)0;
        const double e = exp(B.a2 * w.colscal[col]), sd = B.a0 + B.a1 * e;
        return sd > 1.80 || sd < 1.50 ? (Real)0 : (Real)(B.a1 * B.a2 * e);
    }
    // Planck function that the surface emits (rrtmg_lw_setcoef.f90:190-194), FP64
    __device__ __forceinline__ Real plankbnd() const
    {
        const double tbound = w.colscal[(size_t)in.ncol + col];
        const Real semiss = (Real)in.emis[(size_t)(BAND - 1) * in.ncol + col];
        const int i = clampi((int)(tbound - 159.0), 1, 180);
        const double f = tbound - 159.0 - (double)i;
        return (Real)((double)semiss * ((double)plk[i - 1] + f * ((double)plk[i] - (double)plk[i - 1])));
    }
    // surface emission and reflection: downward radiances into upward ones
    __device__ __forceinline__ void surface(const Real (&fr)[GC], Real (&rad)[GC]) const
    {
        const Real semiss = (Real)in.emis[(size_t)(BAND - 1) * in.ncol + col], emit = plankbnd();
#pragma unroll
        for (int j = 0; j < GC; ++j) rad[j] = fma(fr[j], emit, ((Real)1 - semiss) * rad[j]);
    }
    // band sum of the radiances at level lev (up: 1, down: 0)
    __device__ __forceinline__ void store(const Real (&rad)[GC], int lev, int up) const
    {
        Real *bf = (Real *)w.bflux + (size_t)(2 * (BAND - 1) + 1 - up) * (in.nlay + 1) * in.ncol;
        const Real s = band_sum<BAND>(rad, g0);
        if (first) at32(bf, (unsigned)(lev * in.ncol + col)) = s;
    }
};

#pragma clang fp contract(fast)

}  // namespace rrtmg
