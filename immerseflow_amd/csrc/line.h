// Helpers of the zebra line SOR kernels (k_line_factor, k_line_sor, and the
// persistent k_line_pers).
#pragma once
#include "common.h"
#include "sor.h"

namespace iff {

template <typename T> __device__ __forceinline__ T fmaT(T a, T b, T c)
{
    if constexpr (sizeof(T) == 8)
        return __builtin_fma(a, b, c);
    else
        return __builtin_fmaf(a, b, c);
}

enum { kLfR, kLfNlr, kLfNcp, kLfH, kLfQ };  // per-cell factor planes (kLinePlanes)

template <typename T> struct LineMetric {
    const T *xp, *xm, *yp, *ym;
    __device__ LineMetric(const CaseDev &c)
    {
        if constexpr (sizeof(T) == 8) {
            xp = c.x.cp; xm = c.x.cm; yp = c.y.cp; ym = c.y.cm;
        } else {
            xp = c.xf.cp; xm = c.xf.cm; yp = c.yf.cp; ym = c.yf.cm;
        }
    }
    // row coefficients of a cell (x metric xpi, xmi of its column): l = -aW,
    // b = sa, u = -aE when solved
    __device__ static bool cell(unsigned f, T xpi, T xmi, T yN, T yS, T &l, T &b, T &u)
    {
        l = (T)0;
        b = (T)1;
        u = (T)0;
        if (!(f & F_FLUID)) return false;
        const T aE = (f & F_OPEN_E) ? xpi : (T)0;
        const T aW = (f & F_OPEN_W) ? xmi : (T)0;
        const T aN = (f & F_OPEN_N) ? yN : (T)0;
        const T aS = (f & F_OPEN_S) ? yS : (T)0;
        const T sa = (aE + aW) + (aN + aS);
        if (sa == (T)0) return false;
        l = -aW;
        b = sa;
        u = -aE;
        return true;
    }
};

template <typename T> __device__ __forceinline__ T shfl_up_t(T v, int d) { return __shfl_up(v, (unsigned)d, 64); }
template <typename T> __device__ __forceinline__ T shfl_down_t(T v, int d) { return __shfl_down(v, (unsigned)d, 64); }

}  // namespace iff
