// Finite-difference stencils of the BSSN path, evaluated on a tile staged in
// LDS. `s` points at the sample, `st` is the stride between neighbours along
// the axis, `a` the sample's index along the axis inside its padded block of
// extent `n`, `lo`/`hi` whether the block's low/high face on that axis is a
// domain boundary. Each expression keeps the term order of the reference
// stencil it restates, and floating-point contraction is off, so the sums
// round exactly as the reference's do (the right-hand sides of near-puncture
// data are small differences of these sums, so FMA rounding would show). One
// exception: ko_face multiplies its sums by reciprocals of the boundary
// divisors where the reference, and ko_edge, divide by them, which may differ
// in the last bit.
#pragma once

namespace dgr {

template <typename T>
struct Axis1 {  // deriv644 first derivative constants (derivs.cpp:2621-2623)
    T by12, by60;
    __device__ explicit Axis1(T h) {
#pragma clang fp contract(off)
        const T ih = T(1.0) / h;
        by12 = ih / T(12.0);
        by60 = ih / T(60.0);
    }
};

template <typename T>
struct Axis2 {  // deriv644 second derivative constants (derivs.cpp:2950-2952)
    T by12, by180;
    __device__ explicit Axis2(T h) {
#pragma clang fp contract(off)
        const T ih2 = T(1.0) / (h * h);
        by180 = ih2 / T(180.0);
        by12 = ih2 / T(12.0);
    }
};

template <typename T>
struct AxisKO {  // ko_deriv42 constants (derivs.cpp:966-972)
    T pre, smr3, smr2, smr1;
    __device__ explicit AxisKO(T h) {
#pragma clang fp contract(off)
        pre = T(-1.0) / T(64.0) / h;
        smr3 = T(59.0) / T(48.0) * T(64) * h;
        smr2 = T(43.0) / T(48.0) * T(64) * h;
        smr1 = T(49.0) / T(48.0) * T(64) * h;
    }
};

// deriv644_{x,y,z}: interior derivs.cpp:2646-2649, closures :2654-2697.
template <typename T>
__device__ __forceinline__ T d1(const T *s, int st, int a, int n, bool lo, bool hi,
                                const Axis1<T> &c) {
#pragma clang fp contract(off)
#define U(o) s[(o) * st]
    const int ie = n - 3;
    if (lo && a < 6) {
        if (a == 3) return (T(-25.0) * U(0) + T(48.0) * U(1) - T(36.0) * U(2) + T(16.0) * U(3) - T(3.0) * U(4)) * c.by12;
        if (a == 4) return (T(-3.0) * U(-1) - T(10.0) * U(0) + T(18.0) * U(1) - T(6.0) * U(2) + U(3)) * c.by12;
        return (+U(-2) - T(8.0) * U(-1) + T(8.0) * U(1) - U(2)) * c.by12;
    }
    if (hi && a >= ie - 3) {
        if (a == ie - 3) return (+U(-2) - T(8.0) * U(-1) + T(8.0) * U(1) - U(2)) * c.by12;
        if (a == ie - 2) return (-U(-3) + T(6.0) * U(-2) - T(18.0) * U(-1) + T(10.0) * U(0) + T(3.0) * U(1)) * c.by12;
        return (T(3.0) * U(-4) - T(16.0) * U(-3) + T(36.0) * U(-2) - T(48.0) * U(-1) + T(25.0) * U(0)) * c.by12;
    }
    return (-U(-3) + T(9.0) * U(-2) - T(45.0) * U(-1) + T(45.0) * U(1) - T(9.0) * U(2) + U(3)) * c.by60;
#undef U
}

// deriv644_{xx,yy,zz}: interior derivs.cpp:2975-2979, closures :2984-3047.
template <typename T>
__device__ __forceinline__ T d2(const T *s, int st, int a, int n, bool lo, bool hi,
                                const Axis2<T> &c) {
#pragma clang fp contract(off)
#define U(o) s[(o) * st]
    const int ie = n - 3;
    if (lo && a < 6) {
        if (a == 3) return (T(45.0) * U(0) - T(154.0) * U(1) + T(214.0) * U(2) - T(156.0) * U(3) + T(61.0) * U(4) - T(10.0) * U(5)) * c.by12;
        if (a == 4) return (T(10.0) * U(-1) - T(15.0) * U(0) - T(4.0) * U(1) + T(14.0) * U(2) - T(6.0) * U(3) + U(4)) * c.by12;
        return (-U(-2) + T(16.0) * U(-1) - T(30.0) * U(0) + T(16.0) * U(1) - U(2)) * c.by12;
    }
    if (hi && a >= ie - 3) {
        if (a == ie - 3) return (-U(-2) + T(16.0) * U(-1) - T(30.0) * U(0) + T(16.0) * U(1) - U(2)) * c.by12;
        if (a == ie - 2) return (U(-4) - T(6.0) * U(-3) + T(14.0) * U(-2) - T(4.0) * U(-1) - T(15.0) * U(0) + T(10.0) * U(1)) * c.by12;
        return (T(-10.0) * U(-5) + T(61.0) * U(-4) - T(156.0) * U(-3) + T(214.0) * U(-2) - T(154.0) * U(-1) + T(45.0) * U(0)) * c.by12;
    }
    return (T(2.0) * U(-3) - T(27.0) * U(-2) + T(270.0) * U(-1) - T(490.0) * U(0) + T(270.0) * U(1) - T(27.0) * U(2) + T(2.0) * U(3)) * c.by180;
#undef U
}

// ko_deriv42_{x,y,z}: interior derivs.cpp:988-993, closures :996-1056.
template <typename T>
__device__ __forceinline__ T ko(const T *s, int st, int a, int n, bool lo, bool hi,
                                const AxisKO<T> &c) {
#pragma clang fp contract(off)
#define U(o) s[(o) * st]
    const int ie = n - 3;
    if (lo && a < 6) {
        if (a == 3) return (U(3) - T(3.0) * U(2) + T(3.0) * U(1) - U(0)) / c.smr3;
        if (a == 4) return (U(3) - T(6.0) * U(2) + T(12.0) * U(1) - T(10.0) * U(0) + T(3.0) * U(-1)) / c.smr2;
        return (U(3) - T(6.0) * U(2) + T(15.0) * U(1) - T(19.0) * U(0) + T(12.0) * U(-1) - T(3.0) * U(-2)) / c.smr1;
    }
    if (hi && a >= ie - 3) {
        if (a == ie - 3) return (U(-3) - T(6.0) * U(-2) + T(15.0) * U(-1) - T(19.0) * U(0) + T(12.0) * U(1) - T(3.0) * U(2)) / c.smr1;
        if (a == ie - 2) return (U(-3) - T(6.0) * U(-2) + T(12.0) * U(-1) - T(10.0) * U(0) + T(3.0) * U(1)) / c.smr2;
        return (U(-3) - T(3.0) * U(-2) + T(3.0) * U(-1) - U(0)) / c.smr3;
    }
    return c.pre * (-U(-3) + T(6.0) * U(-2) - T(15.0) * U(-1) + T(20.0) * U(0) - T(15.0) * U(1) + T(6.0) * U(2) - U(3));
#undef U
}

// Stencil constants of one axis for a whole block, computed once with the
// same operations as Axis1/Axis2/AxisKO (so the values are identical).
template <typename T>
struct AxisConstsT {
    T d1_12, d1_60, d2_12, d2_180, ko_pre, ko_s3, ko_s2, ko_s1;
    T ko_r3, ko_r2, ko_r1;  // 1/ko_s3 ..: a division by a block constant is ~30 instructions in FP64
};
using AxisConsts = AxisConstsT<double>;

__host__ __device__ inline AxisConsts axis_consts(double h) {
#pragma clang fp contract(off)
    AxisConsts k;
    const double ih = 1.0 / h;
    k.d1_12 = ih / 12.0;
    k.d1_60 = ih / 60.0;
    const double ih2 = 1.0 / (h * h);
    k.d2_180 = ih2 / 180.0;
    k.d2_12 = ih2 / 12.0;
    k.ko_pre = -1.0 / 64.0 / h;
    k.ko_s3 = 59.0 / 48.0 * 64 * h;
    k.ko_s2 = 43.0 / 48.0 * 64 * h;
    k.ko_s1 = 49.0 / 48.0 * 64 * h;
    k.ko_r3 = 1.0 / k.ko_s3;
    k.ko_r2 = 1.0 / k.ko_s2;
    k.ko_r1 = 1.0 / k.ko_s1;
    return k;
}

// The same stencils with a compile-time stride ST, split into the interior
// formula and the face closure: *_edge returns the closure value where the
// point is one of the three nearest a flagged face (lo: a < 6, hi: a >= ie-3
// with ie = n-3) and `r` otherwise, so a caller whose tile touches no flagged
// face on this axis skips it altogether. Expressions as in d1/d2/ko above.
#define U(o) s[(o) * ST]
template <int ST, typename T>
__device__ __forceinline__ T d1_in(const T *s, T by60) {
#pragma clang fp contract(off)
    return (-U(-3) + T(9.0) * U(-2) - T(45.0) * U(-1) + T(45.0) * U(1) - T(9.0) * U(2) + U(3)) * by60;
}

template <int ST, typename T>
__device__ __forceinline__ T d1_edge(const T *s, T r, int a, int ie, bool lo, bool hi, T by12) {
#pragma clang fp contract(off)
    if (lo && a < 6) {
        if (a == 3) return (-T(25.0) * U(0) + T(48.0) * U(1) - T(36.0) * U(2) + T(16.0) * U(3) - T(3.0) * U(4)) * by12;
        if (a == 4) return (-T(3.0) * U(-1) - T(10.0) * U(0) + T(18.0) * U(1) - T(6.0) * U(2) + U(3)) * by12;
        return (+U(-2) - T(8.0) * U(-1) + T(8.0) * U(1) - U(2)) * by12;
    }
    if (hi && a >= ie - 3) {
        if (a == ie - 3) return (+U(-2) - T(8.0) * U(-1) + T(8.0) * U(1) - U(2)) * by12;
        if (a == ie - 2) return (-U(-3) + T(6.0) * U(-2) - T(18.0) * U(-1) + T(10.0) * U(0) + T(3.0) * U(1)) * by12;
        return (T(3.0) * U(-4) - T(16.0) * U(-3) + T(36.0) * U(-2) - T(48.0) * U(-1) + T(25.0) * U(0)) * by12;
    }
    return r;
}

template <int ST, typename T>
__device__ __forceinline__ T d2_in(const T *s, T by180) {
#pragma clang fp contract(off)
    return (T(2.0) * U(-3) - T(27.0) * U(-2) + T(270.0) * U(-1) - T(490.0) * U(0) + T(270.0) * U(1) - T(27.0) * U(2) + T(2.0) * U(3)) * by180;
}

template <int ST, typename T>
__device__ __forceinline__ T d2_edge(const T *s, T r, int a, int ie, bool lo, bool hi, T by12) {
#pragma clang fp contract(off)
    if (lo && a < 6) {
        if (a == 3) return (T(45.0) * U(0) - T(154.0) * U(1) + T(214.0) * U(2) - T(156.0) * U(3) + T(61.0) * U(4) - T(10.0) * U(5)) * by12;
        if (a == 4) return (T(10.0) * U(-1) - T(15.0) * U(0) - T(4.0) * U(1) + T(14.0) * U(2) - T(6.0) * U(3) + U(4)) * by12;
        return (-U(-2) + T(16.0) * U(-1) - T(30.0) * U(0) + T(16.0) * U(1) - U(2)) * by12;
    }
    if (hi && a >= ie - 3) {
        if (a == ie - 3) return (-U(-2) + T(16.0) * U(-1) - T(30.0) * U(0) + T(16.0) * U(1) - U(2)) * by12;
        if (a == ie - 2) return (U(-4) - T(6.0) * U(-3) + T(14.0) * U(-2) - T(4.0) * U(-1) - T(15.0) * U(0) + T(10.0) * U(1)) * by12;
        return (-T(10.0) * U(-5) + T(61.0) * U(-4) - T(156.0) * U(-3) + T(214.0) * U(-2) - T(154.0) * U(-1) + T(45.0) * U(0)) * by12;
    }
    return r;
}

template <int ST, typename T>
__device__ __forceinline__ T ko_in(const T *s, T pre) {
#pragma clang fp contract(off)
    return pre * (-U(-3) + T(6.0) * U(-2) - T(15.0) * U(-1) + T(20.0) * U(0) - T(15.0) * U(1) + T(6.0) * U(2) - U(3));
}

template <int ST, typename T, typename K>
__device__ __forceinline__ T ko_edge(const T *s, T r, int a, int ie, bool lo, bool hi, const K &k) {
#pragma clang fp contract(off)
    if (lo && a < 6) {
        if (a == 3) return (U(3) - T(3.0) * U(2) + T(3.0) * U(1) - U(0)) / T(k.ko_s3);
        if (a == 4) return (U(3) - T(6.0) * U(2) + T(12.0) * U(1) - T(10.0) * U(0) + T(3.0) * U(-1)) / T(k.ko_s2);
        return (U(3) - T(6.0) * U(2) + T(15.0) * U(1) - T(19.0) * U(0) + T(12.0) * U(-1) - T(3.0) * U(-2)) / T(k.ko_s1);
    }
    if (hi && a >= ie - 3) {
        if (a == ie - 3) return (U(-3) - T(6.0) * U(-2) + T(15.0) * U(-1) - T(19.0) * U(0) + T(12.0) * U(1) - T(3.0) * U(2)) / T(k.ko_s1);
        if (a == ie - 2) return (U(-3) - T(6.0) * U(-2) + T(12.0) * U(-1) - T(10.0) * U(0) + T(3.0) * U(1)) / T(k.ko_s2);
        return (U(-3) - T(3.0) * U(-2) + T(3.0) * U(-1) - U(0)) / T(k.ko_s3);
    }
    return r;
}
#undef U

// The interior formulas on taps already read: t[0..5] = U(-3) U(-2) U(-1) U(1)
// U(2) U(3), c = U(0). Same terms, same order.
struct Taps {
    double t[6];
};
template <int ST>
__device__ __forceinline__ Taps taps(const double *s) {
    return {{s[-3 * ST], s[-2 * ST], s[-ST], s[ST], s[2 * ST], s[3 * ST]}};
}
__device__ __forceinline__ double d1_of(const Taps &a, double by60) {
#pragma clang fp contract(off)
    return (-a.t[0] + 9.0 * a.t[1] - 45.0 * a.t[2] + 45.0 * a.t[3] - 9.0 * a.t[4] + a.t[5]) * by60;
}
__device__ __forceinline__ double d2_of(const Taps &a, double c, double by180) {
#pragma clang fp contract(off)
    return (2.0 * a.t[0] - 27.0 * a.t[1] + 270.0 * a.t[2] - 490.0 * c + 270.0 * a.t[3] - 27.0 * a.t[4] + 2.0 * a.t[5]) * by180;
}
// The closures of a flagged face on the six values next to it along the axis,
// e[0] on the face's node, for the point at distance l from the face (l > 2: r,
// the interior value). All three rows are evaluated and one selected: every
// lane reads the same six values' places, and no lane waits for another row's
// loads. HI: the high face (its rows sum in another order, as the reference's).
template <bool HI, int L>
__device__ __forceinline__ double d1_row(const double *e, double by12) {
#pragma clang fp contract(off)
    if constexpr (L == 0)
        return HI ? (3.0 * e[4] - 16.0 * e[3] + 36.0 * e[2] - 48.0 * e[1] + 25.0 * e[0]) * by12
                  : (-25.0 * e[0] + 48.0 * e[1] - 36.0 * e[2] + 16.0 * e[3] - 3.0 * e[4]) * by12;
    else if constexpr (L == 1)
        return HI ? (-e[4] + 6.0 * e[3] - 18.0 * e[2] + 10.0 * e[1] + 3.0 * e[0]) * by12
                  : (-3.0 * e[0] - 10.0 * e[1] + 18.0 * e[2] - 6.0 * e[3] + e[4]) * by12;
    else
        return HI ? (e[4] - 8.0 * e[3] + 8.0 * e[1] - e[0]) * by12 : (e[0] - 8.0 * e[1] + 8.0 * e[3] - e[4]) * by12;
}
template <bool HI>
__device__ __forceinline__ double d1_face(const double *e, double r, int l, double by12) {
    const double a = d1_row<HI, 0>(e, by12), b = d1_row<HI, 1>(e, by12), c = d1_row<HI, 2>(e, by12);
    return l == 0 ? a : l == 1 ? b : l == 2 ? c : r;
}
template <bool HI>
__device__ __forceinline__ double d2_face(const double *e, double r, int l, double by12) {
#pragma clang fp contract(off)
    const double a =
        HI ? (-10.0 * e[5] + 61.0 * e[4] - 156.0 * e[3] + 214.0 * e[2] - 154.0 * e[1] + 45.0 * e[0]) * by12
           : (45.0 * e[0] - 154.0 * e[1] + 214.0 * e[2] - 156.0 * e[3] + 61.0 * e[4] - 10.0 * e[5]) * by12;
    const double b = HI ? (e[5] - 6.0 * e[4] + 14.0 * e[3] - 4.0 * e[2] - 15.0 * e[1] + 10.0 * e[0]) * by12
                        : (10.0 * e[0] - 15.0 * e[1] - 4.0 * e[2] + 14.0 * e[3] - 6.0 * e[4] + e[5]) * by12;
    const double c = HI ? (-e[4] + 16.0 * e[3] - 30.0 * e[2] + 16.0 * e[1] - e[0]) * by12
                        : (-e[0] + 16.0 * e[1] - 30.0 * e[2] + 16.0 * e[3] - e[4]) * by12;
    return l == 0 ? a : l == 1 ? b : l == 2 ? c : r;
}
// (by reciprocals, for a division is ~30 instructions in FP64: the right-hand side
// of 200 ragged blocks, 28% of them flagged, is 2.3e-13 from
// values computed apart with either, that of one 19^3 block 1.9e-13)
template <typename K>
__device__ __forceinline__ double ko_face(const double *e, double r, int l, const K &k) {
#pragma clang fp contract(off)
    const double a = (e[3] - 3.0 * e[2] + 3.0 * e[1] - e[0]) * k.ko_r3;
    const double b = (e[4] - 6.0 * e[3] + 12.0 * e[2] - 10.0 * e[1] + 3.0 * e[0]) * k.ko_r2;
    const double c = (e[5] - 6.0 * e[4] + 15.0 * e[3] - 19.0 * e[2] + 12.0 * e[1] - 3.0 * e[0]) * k.ko_r1;
    return l == 0 ? a : l == 1 ? b : l == 2 ? c : r;
}
__device__ __forceinline__ double ko_of(const Taps &a, double c, double pre) {
#pragma clang fp contract(off)
    return pre * (-a.t[0] + 6.0 * a.t[1] - 15.0 * a.t[2] + 20.0 * c - 15.0 * a.t[3] + 6.0 * a.t[4] - a.t[5]);
}

}  // namespace dgr
