// LW gas optics as weighted table rows, for kernels whose lane is one column
// and holds several g-points in registers.
//
// Every band formula of taumol (rrtmg_lw_taumol.f90) is linear in its table
// values, with weights that do not depend on the g-point: the optical depth
// of g-point g is sum_r W_r K[row_r][g], and the Planck fraction a sum of one
// or two rows of its own.  lw_rows calls term(table, offset, row, weight) for each
// row of the optical depth, lw_fracs frac(offset, row, weight) for each row of
// the Planck fraction; what a caller does per row (a multiply-add over its
// g-points, or the transposed product of a backward pass) is then the whole
// per-g-point cost of the gas optics, and the species parameters, indices and
// weights are formed once per (layer, column, band).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dual.hpp"
#include "lw_optics.hpp"
#include "rrtmg_device.hpp"
#include "rrtmg_types.hpp"

namespace rrtmg {

// Contraction is off here, and multiply-adds are written out: which of two
// products the compiler fuses into a sum differs between the kernels that
// instantiate a formula, and a column's result must not depend on the kernel
// that the size of the call selects.
#pragma clang fp contract(off)

// The three rows of the lower atmosphere's eta interpolation
// (rrtmg_lw_taumol.f90:550-668) from one base row: below 0.125 the cubic
// scheme on rows js, js+1, js+2, above 0.875 on js-1, js, js+1, between them
// linear on js, js+1, written here with a zero weight on js-1.
template <typename Real, typename V>
struct LwEta3 {
    int js;  // first of the three rows (1-based)
    V w0, w1, w2;
};
template <typename Real, typename V>
__device__ __forceinline__ LwEta3<Real, V> lw_eta3(const Eta<V> &e)
{
    const bool lo = val(e.specparm) < (Real)0.125, hi = val(e.specparm) > (Real)0.875;
    const V p = lo ? V(e.fs - (Real)1) : V(-e.fs);
    const V p2 = p * p, p4 = p2 * p2;
    const V k1 = (Real)1 - p - (Real)2 * p4, k2 = p + p4;
    LwEta3<Real, V> r;
    r.js = lo || e.js < 2 ? e.js : e.js - 1;  // js < 2 there only for NaN
    r.w0 = lo ? p4 : hi ? k2 : V((Real)0);
    r.w1 = lo || hi ? k1 : V((Real)1 - e.fs);
    r.w2 = lo ? k2 : hi ? p4 : e.fs;
    return r;
}

// which k-table a row belongs to: absb, or any other
using LwOther = std::integral_constant<int, 0>;
using LwAbsB = std::integral_constant<int, 1>;
constexpr int LW_ABSB = 1;

#define CHI(i, j) ((Real)at32(lw_cst<Real>(cst->chi_mls, cst->chi_mls_f), (unsigned)(((j)-1) * 7 + ((i)-1))))
#define RAT(NAME, e) ((Real)at32(lw_cst<Real>(cst->NAME, cst->NAME##_f), (unsigned)(e)))
#define CHIQ(a, b, j) ((Real)lw_cst<Real>(cst->chi_ratio, cst->chi_ratio_f)[lw_chi_ratio_k<a, b, j>()])

// A backward caller, whose gradient would lose digits to the sum of weight
// derivatives of opposite signs, takes the interpolations whole instead, by
// further overloads of term and frac: a pair of rows (table, offset, row, step,
// weight, fraction), three rows (table, offset, row, weight, three factors
// that add up to one), the four rows of a minor species (table, offset, row,
// rows per temperature, weight, temperature fraction, eta fraction, 0); frac
// (offset, row, step, fraction).  Its type has a member type Whole.
template <typename T, typename = void>
struct LwTakesWhole : std::false_type {};
template <typename T>
struct LwTakesWhole<T, std::void_t<typename T::Whole>> : std::true_type {};

// The rows of one (layer, column) of band BAND; the band formulas and their
// reference lines are those of lw_gas.  Rows are 1-based as the reference's
// indices.  The g-point factors of bands 4 and 7 aloft are lw_gfactor.
template <int BAND, typename Real, typename L, typename FT>
__device__ __forceinline__ void lw_rows(const LwBand &B, const LwConst *__restrict__ cst, const L &c,
                                        bool lower, FT &&term)
{
    constexpr int NA = LW_NSPA[BAND - 1], NB = LW_NSPB[BAND - 1];
    const int ind0 = lower ? ((c.jp - 1) * 5 + (c.jt - 1)) * NA : ((c.jp - 13) * 5 + (c.jt - 1)) * NB;
    const int ind1 = lower ? (c.jp * 5 + (c.jt1 - 1)) * NA : ((c.jp - 12) * 5 + (c.jt1 - 1)) * NB;
    const int jp = c.jp;
    auto pair = [&](auto k, int off, int row, int step, const auto &m, const auto &f) {  // m ((1-f) K[row] + f K[row+step])
        if constexpr (LwTakesWhole<std::decay_t<FT>>::value) {
            term(k, off, row, step, m, f);
        } else {
            const auto mf = m * f;
            term(k, off, row, m - mf);
            term(k, off, row + step, mf);
        }
    };
    // m (k.w0 K[row] + k.w1 K[row+1] + k.w2 K[row+2])
    auto three = [&](int off, int row, const auto &m, const auto &k) {
        if constexpr (LwTakesWhole<std::decay_t<FT>>::value) {
            term(LwOther{}, off, row, m, k.w0, k.w1, k.w2);
        } else {
            term(LwOther{}, off, row, m * k.w0);
            term(LwOther{}, off, row + 1, m * k.w1);
            term(LwOther{}, off, row + 2, m * k.w2);
        }
    };
    auto four = [&](auto k, int off, const auto &m) {
        term(k, off, ind0 + 1, m * c.fac00);
        term(k, off, ind0 + 2, m * c.fac10);
        term(k, off, ind1 + 1, m * c.fac01);
        term(k, off, ind1 + 2, m * c.fac11);
    };
    auto self = [&](const auto &m) { pair(LwOther{}, B.selfref, c.inds, 1, m, c.selffrac); };
    auto foreign = [&](const auto &m) { pair(LwOther{}, B.forref, c.indf, 1, m, c.forfrac); };
    auto minor1 = [&](int off, const auto &m) { pair(LwOther{}, off, c.indm, 1, m, c.minorfrac); };
    auto minor2 = [&](int off, int neta, const auto &e, const auto &m) {
        const int r = e.js + neta * (c.indm - 1);
        if constexpr (LwTakesWhole<std::decay_t<FT>>::value) {
            term(LwOther{}, off, r, neta, m, c.minorfrac, e.fs, 0);
        } else {
            const auto hi = m * c.minorfrac;
            pair(LwOther{}, off, r, 1, m - hi, e.fs);
            pair(LwOther{}, off, r + neta, 1, hi, e.fs);
        }
    };
    auto major3 = [&](int off, const auto &e, int ind, const auto &fa, const auto &fb) {
        const auto k = lw_eta3<Real>(e);
        const auto a = e.speccomb * fa;
        const auto b = e.speccomb * fb;
        const int r = ind + k.js;
        three(off, r, a, k);
        three(off, r + 9, b, k);
    };
    auto major_b = [&](int off, const auto &e, int ind, const auto &fa, const auto &fb) {
        pair(LwAbsB{}, off, ind + e.js, 1, e.speccomb * fa, e.fs);
        pair(LwAbsB{}, off, ind + e.js + 5, 1, e.speccomb * fb, e.fs);
    };
    auto binary_lo = [&](const auto &e, const auto &e1) {
        major3(B.absa, e, ind0, c.fac00, c.fac10);
        major3(B.absa, e1, ind1, c.fac01, c.fac11);
    };
    auto binary_hi = [&](const auto &e, const auto &e1) {
        major_b(B.absb, e, ind0, c.fac00, c.fac10);
        major_b(B.absb, e1, ind1, c.fac01, c.fac11);
    };
    auto cont = [&]() {  // self and foreign continuum of the lower atmosphere
        self(c.selffac);
        foreign(c.forfac);
    };
    if constexpr (BAND == 1) {
        if (lower) {
            const Real cr = c.pavel < (Real)250 ? (Real)1 - fdiv((Real)0.15 * ((Real)250 - c.pavel), (Real)154.4) : (Real)1;
            four(LwOther{}, B.absa, cr * c.colh2o);
            self(cr * c.selffac);
            foreign(cr * c.forfac);
            minor1(B.ka_mn2, cr * c.colbrd * c.scaleminorn2);
        } else {
            const Real cr = (Real)1 - (Real)0.15 * fdiv(c.pavel, (Real)95.6);
            four(LwAbsB{}, B.absb, cr * c.colh2o);
            foreign(cr * c.forfac);
            minor1(B.kb_mn2, cr * c.colbrd * c.scaleminorn2);
        }
    } else if constexpr (BAND == 2) {
        if (lower) {
            const Real cr = (Real)1 - fdiv((Real).05 * (c.pavel - (Real)100), (Real)900);
            four(LwOther{}, B.absa, cr * c.colh2o);
            self(cr * c.selffac);
            foreign(cr * c.forfac);
        } else {
            four(LwAbsB{}, B.absb, c.colh2o);
            foreign(c.forfac);
        }
    } else if constexpr (BAND == 3) {
        const auto adj = lw_adjcol(c.coln2o, c.coldry, CHI(4, jp + 1), (Real)1.5, (Real)0.5, (Real)0.65);
        if (lower) {
            binary_lo(lw_eta(c.colh2o, c.colco2, RAT(rat_h2oco2, jp), (Real)8),
                      lw_eta(c.colh2o, c.colco2, RAT(rat_h2oco2, jp + 1), (Real)8));
            cont();
            minor2(B.ka_mn2o, 9, lw_eta(c.colh2o, c.colco2, CHIQ(1, 2, 3), (Real)8), adj);
        } else {
            const auto em = lw_eta(c.colh2o, c.colco2, CHIQ(1, 2, 13), (Real)4);
            binary_hi(lw_eta(c.colh2o, c.colco2, RAT(rat_h2oco2, jp), (Real)4),
                      lw_eta(c.colh2o, c.colco2, RAT(rat_h2oco2, jp + 1), (Real)4));
            foreign(c.forfac);
            minor2(B.kb_mn2o, 5, em, adj);
        }
    } else if constexpr (BAND == 4 || BAND == 5) {
        if (lower) {
            binary_lo(lw_eta(c.colh2o, c.colco2, RAT(rat_h2oco2, jp), (Real)8),
                      lw_eta(c.colh2o, c.colco2, RAT(rat_h2oco2, jp + 1), (Real)8));
            cont();
            if constexpr (BAND == 5) {
                minor2(B.ka_mo3, 9, lw_eta(c.colh2o, c.colco2, CHIQ(1, 2, 7), (Real)8), c.colo3);
                term(LwOther{}, B.ccl4, 1, c.wx1);
            } else {
            }
        } else {
            binary_hi(lw_eta(c.colo3, c.colco2, RAT(rat_o3co2, jp), (Real)4),
                      lw_eta(c.colo3, c.colco2, RAT(rat_o3co2, jp + 1), (Real)4));
            if constexpr (BAND == 5) {
                term(LwOther{}, B.ccl4, 1, c.wx1);
            } else {
            }
        }
    } else if constexpr (BAND == 6) {
        if (lower) {
            four(LwOther{}, B.absa, c.colh2o);
            cont();
            minor1(B.ka_mco2, lw_adjcol(c.colco2, c.coldry, CHI(2, jp + 1), (Real)3, (Real)2, (Real)0.77));
        }
        term(LwOther{}, B.cfc11adj, 1, c.wx2);
        term(LwOther{}, B.cfc12, 1, c.wx3);
    } else if constexpr (BAND == 7) {
        if (lower) {
            const auto em = lw_eta(c.colh2o, c.colo3, CHIQ(1, 3, 3), (Real)8);
            binary_lo(lw_eta(c.colh2o, c.colo3, RAT(rat_h2oo3, jp), (Real)8),
                      lw_eta(c.colh2o, c.colo3, RAT(rat_h2oo3, jp + 1), (Real)8));
            cont();
            minor2(B.ka_mco2, 9, em, lw_adjcol(c.colco2, c.coldry, CHI(2, jp + 1), (Real)3, (Real)3, (Real)0.79));
        } else {
            four(LwAbsB{}, B.absb, c.colo3);
            minor1(B.kb_mco2, lw_adjcol(c.colco2, c.coldry, CHI(2, jp + 1), (Real)3, (Real)2, (Real)0.79));
        }
    } else if constexpr (BAND == 8) {
        const auto adj = lw_adjcol(c.colco2, c.coldry, CHI(2, jp + 1), (Real)3, (Real)2, (Real)0.65);
        if (lower) {
            four(LwOther{}, B.absa, c.colh2o);
            cont();
            minor1(B.ka_mco2, adj);
            minor1(B.ka_mo3, c.colo3);
            minor1(B.ka_mn2o, c.coln2o);
        } else {
            four(LwAbsB{}, B.absb, c.colo3);
            minor1(B.kb_mco2, adj);
            minor1(B.kb_mn2o, c.coln2o);
        }
        term(LwOther{}, B.cfc12, 1, c.wx3);
        term(LwOther{}, B.cfc22adj, 1, c.wx4);
    } else if constexpr (BAND == 9) {
        const auto adj = lw_adjcol(c.coln2o, c.coldry, CHI(4, jp + 1), (Real)1.5, (Real)0.5, (Real)0.65);
        if (lower) {
            binary_lo(lw_eta(c.colh2o, c.colch4, RAT(rat_h2och4, jp), (Real)8),
                      lw_eta(c.colh2o, c.colch4, RAT(rat_h2och4, jp + 1), (Real)8));
            cont();
            minor2(B.ka_mn2o, 9, lw_eta(c.colh2o, c.colch4, CHIQ(1, 6, 3), (Real)8), adj);
        } else {
            four(LwAbsB{}, B.absb, c.colch4);
            minor1(B.kb_mn2o, adj);
        }
    } else if constexpr (BAND == 10 || BAND == 11) {
        if (lower) {
            four(LwOther{}, B.absa, c.colh2o);
            cont();
            if constexpr (BAND == 11) minor1(B.ka_mo2, c.colo2 * c.scaleminor);
        } else {
            four(LwAbsB{}, B.absb, c.colh2o);
            foreign(c.forfac);
            if constexpr (BAND == 11) minor1(B.kb_mo2, c.colo2 * c.scaleminor);
        }
    } else if constexpr (BAND == 12) {
        if (lower) {
            binary_lo(lw_eta(c.colh2o, c.colco2, RAT(rat_h2oco2, jp), (Real)8),
                      lw_eta(c.colh2o, c.colco2, RAT(rat_h2oco2, jp + 1), (Real)8));
            cont();
        }
    } else if constexpr (BAND == 13) {
        if (lower) {
            binary_lo(lw_eta(c.colh2o, c.coln2o, RAT(rat_h2on2o, jp), (Real)8),
                      lw_eta(c.colh2o, c.coln2o, RAT(rat_h2on2o, jp + 1), (Real)8));
            cont();
            minor2(B.ka_mco2, 9, lw_eta(c.colh2o, c.coln2o, CHIQ(1, 4, 1), (Real)8),
                   lw_adjcol(c.colco2, c.coldry, (Real)3.55e-4, (Real)3, (Real)2, (Real)0.68));
            minor2(B.ka_mco, 9, lw_eta(c.colh2o, c.coln2o, CHIQ(1, 4, 3), (Real)8), c.colco);
        } else {
            minor1(B.kb_mo3, c.colo3);
        }
    } else if constexpr (BAND == 14) {
        if (lower) {
            four(LwOther{}, B.absa, c.colco2);
            cont();
        } else {
            four(LwAbsB{}, B.absb, c.colco2);
        }
    } else if constexpr (BAND == 15) {
        if (lower) {
            const auto em = lw_eta(c.coln2o, c.colco2, CHIQ(4, 2, 1), (Real)8);
            binary_lo(lw_eta(c.coln2o, c.colco2, RAT(rat_n2oco2, jp), (Real)8),
                      lw_eta(c.coln2o, c.colco2, RAT(rat_n2oco2, jp + 1), (Real)8));
            cont();
            minor2(B.ka_mn2, 9, em, c.colbrd * c.scaleminor);
        }
    } else {  // 16; aloft nspb(16) = 0, so both levels read rows 1 and 2
        if (lower) {
            binary_lo(lw_eta(c.colh2o, c.colch4, RAT(rat_h2och4, jp), (Real)8),
                      lw_eta(c.colh2o, c.colch4, RAT(rat_h2och4, jp + 1), (Real)8));
            cont();
        } else {
            four(LwAbsB{}, B.absb, c.colch4);
        }
    }
}

// The rows of the Planck fraction of one (layer, column) of band BAND: two of
// the band's species parameter at a reference level, or one.  Bands 12 and 15
// have none aloft (their optics are zero there).
template <int BAND, typename Real, typename L, typename FF>
__device__ __forceinline__ void lw_fracs(const LwBand &B, const LwConst *__restrict__ cst, const L &c,
                                         bool lower, FF &&frac)
{
    auto pfrac = [&](int off, const auto &e) {
        if constexpr (LwTakesWhole<std::decay_t<FF>>::value) {
            frac(off, e.js, 1, e.fs);
        } else {
            frac(off, e.js, (Real)1 - e.fs);
            frac(off, e.js + 1, e.fs);
        }
    };
    auto flat = [&](int off) { frac(off, 1, (Real)1); };
    (void)cst;
    if constexpr (BAND == 3) {
        if (lower)
            pfrac(B.fracrefa, lw_eta(c.colh2o, c.colco2, CHIQ(1, 2, 9), (Real)8));
        else
            pfrac(B.fracrefb, lw_eta(c.colh2o, c.colco2, CHIQ(1, 2, 13), (Real)4));
    } else if constexpr (BAND == 4) {
        if (lower)
            pfrac(B.fracrefa, lw_eta(c.colh2o, c.colco2, CHIQ(1, 2, 11), (Real)8));
        else
            pfrac(B.fracrefb, lw_eta(c.colo3, c.colco2, CHIQ(3, 2, 13), (Real)4));
    } else if constexpr (BAND == 5) {
        if (lower)
            pfrac(B.fracrefa, lw_eta(c.colh2o, c.colco2, CHIQ(1, 2, 5), (Real)8));
        else
            pfrac(B.fracrefb, lw_eta(c.colo3, c.colco2, CHIQ(3, 2, 43), (Real)4));
    } else if constexpr (BAND == 6) {
        flat(B.fracrefa);
    } else if constexpr (BAND == 7) {
        if (lower)
            pfrac(B.fracrefa, lw_eta(c.colh2o, c.colo3, CHIQ(1, 3, 3), (Real)8));
        else
            flat(B.fracrefb);
    } else if constexpr (BAND == 9) {
        if (lower)
            pfrac(B.fracrefa, lw_eta(c.colh2o, c.colch4, CHIQ(1, 6, 9), (Real)8));
        else
            flat(B.fracrefb);
    } else if constexpr (BAND == 12) {
        if (lower) pfrac(B.fracrefa, lw_eta(c.colh2o, c.colco2, CHIQ(1, 2, 10), (Real)8));
    } else if constexpr (BAND == 13) {
        if (lower)
            pfrac(B.fracrefa, lw_eta(c.colh2o, c.coln2o, CHIQ(1, 4, 5), (Real)8));
        else
            flat(B.fracrefb);
    } else if constexpr (BAND == 15) {
        if (lower) pfrac(B.fracrefa, lw_eta(c.coln2o, c.colco2, CHIQ(4, 2, 1), (Real)8));
    } else if constexpr (BAND == 16) {
        if (lower)
            pfrac(B.fracrefa, lw_eta(c.colh2o, c.colch4, CHIQ(1, 6, 6), (Real)8));
        else
            flat(B.fracrefb);
    } else {
        flat(lower ? B.fracrefa : B.fracrefb);
    }
}
#undef CHI
#undef RAT
#undef CHIQ

// the empirical factor of g-point g (0-based) of bands 4 and 7 aloft
// (rrtmg_lw_taumol.f90:1011-1017, 1646-1651)
template <int BAND, typename Real>
__device__ __forceinline__ Real lw_gfactor(int g, bool lower)
{
    Real m = (Real)1;
    if constexpr (BAND == 4)
        m = g < 7 ? (Real)1 : g == 7 ? (Real)0.92 : g == 8 ? (Real)0.88 : g == 9 ? (Real)1.07 : g == 10 ? (Real)1.1
          : g == 11 ? (Real)0.99 : g == 12 ? (Real)0.88 : (Real)0.943;
    if constexpr (BAND == 7)
        m = g < 5 || g > 10 ? (Real)1 : g == 5 ? (Real)0.92 : g == 6 ? (Real)0.88 : g == 7 ? (Real)1.07
          : g == 8 ? (Real)1.1 : g == 9 ? (Real)0.99 : (Real)0.855;
    return lower ? (Real)1 : m;
}

#pragma clang fp contract(fast)

}  // namespace rrtmg
