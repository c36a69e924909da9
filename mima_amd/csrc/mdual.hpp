// Forward-mode numbers whose zero derivatives are part of the type: MDual<F, M>
// carries a value and the derivatives with respect to layer temperature (bit 0
// of M), water vapour (bit 1) and ozone (bit 2) that M names; the others are
// zero and cost neither registers nor arithmetic (a floating-point product
// with a stored zero is not folded away: it may be a NaN).  An operation's
// result has the union of its operands' derivatives; plain numbers have none.
//
// Multiply-adds are written out and contraction is off, so that a formula has
// the same bits in every kernel that uses it.  Branches compare values.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rrtmg_device.hpp"

namespace rrtmg {

#pragma clang fp contract(off)

template <typename F, unsigned M>
struct MDual {
    static_assert(M != 0 && M < 8, "a plain number has no derivatives");
    F v;
    F d[3];  // d[k] is set only where bit k of M is
    __device__ __forceinline__ MDual() = default;
    __device__ __forceinline__ explicit MDual(F x) : v(x)
    {
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (M >> k & 1u) d[k] = (F)0;
    }
    __device__ __forceinline__ explicit operator int() const { return (int)v; }
};

// a field's number: plain where it has no derivatives
template <typename F, unsigned M>
struct MField {
    using type = MDual<F, M>;
};
template <typename F>
struct MField<F, 0> {
    using type = F;
};

template <typename F, unsigned M>
__device__ __forceinline__ F val(const MDual<F, M> &x)
{
    return x.v;
}

#define MD_EACH(mask) _Pragma("unroll") for (int k = 0; k < 3; ++k) if ((mask) >> k & 1u)
#define MD_T template <typename F, unsigned M>
#define MD_TT template <typename F, unsigned A, unsigned B>
#define MD_IN __device__ __forceinline__

MD_T MD_IN MDual<F, M> operator-(const MDual<F, M> &a)
{
    MDual<F, M> r;
    r.v = -a.v;
    MD_EACH(M) r.d[k] = -a.d[k];
    return r;
}
MD_TT MD_IN MDual<F, A | B> operator+(const MDual<F, A> &a, const MDual<F, B> &b)
{
    MDual<F, A | B> r;
    r.v = a.v + b.v;
    MD_EACH(A | B) r.d[k] = !(B >> k & 1u) ? a.d[k] : !(A >> k & 1u) ? b.d[k] : a.d[k] + b.d[k];
    return r;
}
MD_TT MD_IN MDual<F, A | B> operator-(const MDual<F, A> &a, const MDual<F, B> &b)
{
    MDual<F, A | B> r;
    r.v = a.v - b.v;
    MD_EACH(A | B) r.d[k] = !(B >> k & 1u) ? a.d[k] : !(A >> k & 1u) ? -b.d[k] : a.d[k] - b.d[k];
    return r;
}
MD_TT MD_IN MDual<F, A | B> operator*(const MDual<F, A> &a, const MDual<F, B> &b)
{
    MDual<F, A | B> r;
    r.v = a.v * b.v;
    MD_EACH(A | B)
        r.d[k] = !(B >> k & 1u) ? a.d[k] * b.v : !(A >> k & 1u) ? a.v * b.d[k] : fma(a.d[k], b.v, a.v * b.d[k]);
    return r;
}
MD_TT MD_IN MDual<F, A | B> fdiv(const MDual<F, A> &a, const MDual<F, B> &b)
{
    MDual<F, A | B> r;
    r.v = fdiv(a.v, b.v);
    const F ib = fdiv((F)1, b.v);
    MD_EACH(A | B)
        r.d[k] = (!(B >> k & 1u) ? a.d[k] : !(A >> k & 1u) ? -(r.v * b.d[k]) : fma(-r.v, b.d[k], a.d[k])) * ib;
    return r;
}
// with plain numbers
MD_T MD_IN MDual<F, M> operator+(const MDual<F, M> &a, F b)
{
    MDual<F, M> r = a;
    r.v = a.v + b;
    return r;
}
MD_T MD_IN MDual<F, M> operator+(F a, const MDual<F, M> &b) { return b + a; }
MD_T MD_IN MDual<F, M> operator-(const MDual<F, M> &a, F b)
{
    MDual<F, M> r = a;
    r.v = a.v - b;
    return r;
}
MD_T MD_IN MDual<F, M> operator-(F a, const MDual<F, M> &b)
{
    MDual<F, M> r;
    r.v = a - b.v;
    MD_EACH(M) r.d[k] = -b.d[k];
    return r;
}
MD_T MD_IN MDual<F, M> operator*(const MDual<F, M> &a, F b)
{
    MDual<F, M> r;
    r.v = a.v * b;
    MD_EACH(M) r.d[k] = a.d[k] * b;
    return r;
}
MD_T MD_IN MDual<F, M> operator*(F a, const MDual<F, M> &b) { return b * a; }
MD_T MD_IN MDual<F, M> fdiv(const MDual<F, M> &a, F b)
{
    MDual<F, M> r;
    r.v = fdiv(a.v, b);
    const F ib = fdiv((F)1, b);
    MD_EACH(M) r.d[k] = a.d[k] * ib;
    return r;
}
MD_T MD_IN MDual<F, M> pow(const MDual<F, M> &a, F e)
{
    MDual<F, M> r;
    r.v = ::pow(a.v, e);
    const F s = a.v != (F)0 ? fdiv(e * r.v, a.v) : (F)0;
    MD_EACH(M) r.d[k] = s * a.d[k];
    return r;
}
MD_T MD_IN bool operator<(const MDual<F, M> &a, F b) { return a.v < b; }
MD_T MD_IN bool operator>(const MDual<F, M> &a, F b) { return a.v > b; }
MD_T MD_IN bool operator>=(const MDual<F, M> &a, F b) { return a.v >= b; }

// g[k] += s dw/dx_k for the derivatives w has
template <typename F>
MD_IN void md_gather(F (&)[3], F, F)
{
}
MD_T MD_IN void md_gather(F (&g)[3], F s, const MDual<F, M> &w)
{
    MD_EACH(M) g[k] = fma(s, w.d[k], g[k]);
}

#undef MD_EACH
#undef MD_T
#undef MD_TT
#undef MD_IN

#pragma clang fp contract(fast)

}  // namespace rrtmg
