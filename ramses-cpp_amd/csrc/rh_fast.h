// rh_fast.h -- the Godunov update's arithmetic for ordinary states, as the
// kernels of rh_godunov.hip run it: the operations of rh_physics.h on the
// same operands in the same order, so every value is the same, with the
// steps left out that cannot matter for a state in range.
//
// In range (prim below checks every state a cell's update reads; a wave with a
// state outside takes the general code) means finite and far from overflow and
// underflow, so that
//   * a quotient needs neither the scaling nor the fix-up of the IEEE
//     division sequence: a reciprocal refined to the last bit (4 instructions)
//     and a product corrected by its exact remainder (3); quotients by one
//     divisor share its reciprocal;
//   * a square root needs no scaling (11 instructions instead of 18);
//   * no operand of a minimum or maximum is a NaN, so v_min/v_max replace
//     compare-and-select pairs (3 instructions for a double);
//   * halving and quartering are exact, so a product with a power of two can
//     be joined to the following sum by an fma without changing its value.
//
// Frame.  A cell's line along a dimension is read in the frame that points
// from the neighbour across the oct face (X, with X2 beyond it) through the
// cell (C) to its sibling in the oct (S): for a cell on the oct's upper side
// the axis is reversed and the normal velocity changes sign.  Every operation
// of the scheme commutes with that reflection (differences, products and
// quotients change sign exactly, minima and maxima change places), except the
// choice of a side where the contact speed is exactly zero, which the solvers
// take from `mir`.  So all lanes run the same code on the same operands and no
// operand is selected by the cell's place in its oct.  Components are in the
// rotated order of the reference's trace: density, normal velocity, the two
// tangential velocities, pressure.
#pragma once
#include "rh_physics.h"

namespace rh {
namespace fast {

// Votes of a wave, in a form the compiler knows to be the same in every lane,
// so that branches on them keep nothing alive for the path not taken.
RH_DEV bool any_lane(bool b) { return __builtin_amdgcn_ballot_w64(b) != 0; }
RH_DEV bool all_lanes(bool b) { return __builtin_amdgcn_ballot_w64(!b) == 0; }

RH_DEV double mn(double a, double b) { return __builtin_fmin(a, b); }
RH_DEV double mx(double a, double b) { return __builtin_fmax(a, b); }
RH_DEV float mn(float a, float b) { return __builtin_fminf(a, b); }
RH_DEV float mx(float a, float b) { return __builtin_fmaxf(a, b); }
RH_DEV double fm(double a, double b, double c) { return __builtin_fma(a, b, c); }
RH_DEV float fm(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
// smax(a, 0) that keeps a NaN in FP32 (in range FP64 has none).
RH_DEV double nonneg(double a) { return mx(a, 0.0); }
RH_DEV float nonneg(float a) { return smax(a, 0.0f); }
RH_DEV double signed_as(double a, double s) { return __builtin_copysign(a, s); }
RH_DEV float signed_as(float a, float s) { return __builtin_copysignf(a, s); }

// Reciprocal (the hardware's, good to 2^-24, times 1 + e + e^2 with its error
// e: 2^-72 before the last rounding), and a quotient by a divisor whose
// reciprocal is known (float: the hardware reciprocal, as dv()).
//
// Markstein's theorem (IBM J. Res. Dev. 34, 1990): the product corrected by its
// exact remainder is the correctly rounded quotient where the reciprocal is the
// correctly rounded one.  unit_quot's is, for every divisor but a significand of
// all ones, and for that one too where the hardware's is not below it (gfx950
// returns the correctly rounded reciprocal itself there).  So quotients by a
// cell's density, whose reciprocal prim takes from unit_quot, round as IEEE
// division does.  recip's alone misses the last bit for one divisor in 2^17; a
// quotient by such a divisor differs from IEEE's only next to a midpoint of two
// doubles, for a handful of its 2^52 dividends.
RH_DEV double recip(double b) {
    const double y = __builtin_amdgcn_rcp(b);
    const double e = fm(-b, y, 1.0);
    return fm(y, fm(e, e, e), y);
}
RH_DEV float recip(float b) { return __builtin_amdgcn_rcpf(b); }
RH_DEV double quot(double a, double b, double y) {
    const double q = a * y;
    const double r = fm(-b, q, a);
    return fm(r, y, q);
}
RH_DEV float quot(float a, float, float y) { return a * y; }
// 1/b with b's reciprocal y as above.
RH_DEV double unit_quot(double b, double y) { return fm(fm(-b, y, 1.0), y, y); }
RH_DEV float unit_quot(float, float y) { return y; }

// Square root of a value of at least 1e-20: a Newton step for half the
// reciprocal root h (from the hardware's, good to 2^-24, to 2^-47), then the
// root 2x*h corrected twice by its exact remainder times h, as Markstein's
// quotients are: the first leaves it within an ulp, the second within 2^-47 ulp
// of the root before it is rounded.  A root lies that close to a midpoint of
// two doubles only for some 1,400 significands; for those, and for 2 10^10
// others, gfx950 gives the correctly rounded root.
RH_DEV double root(double x) {
    const double g = 0.5 * __builtin_amdgcn_rsq(x), xx = x + x;
    const double h = fm(g, fm(-(xx * g), g, 0.5), g);
    double s = xx * h;
    s = fm(fm(-s, s, x), h, s);
    return fm(fm(-s, s, x), h, s);
}
RH_DEV float root(float x) { return __builtin_amdgcn_sqrtf(x); }

// a with its sign changed where bit 31 of s is set.
RH_DEV double flip(double a, int s) { return __hiloint2double(__double2hiint(a) ^ s, __double2loint(a)); }
RH_DEV float flip(float a, int s) { return __int_as_float(__float_as_int(a) ^ s); }

// Constants of a launch in the compute type.
template <typename T> struct Consts {
    T gamma, gm1, smalle, smallp;
    T y_gm1;    // recip(gm1) (double) or 1/gm1 (float), for the internal energy p/(gm1)
    T dx, hdx;  // cell width and half of it
    T inv;      // 1/dx where exact (double), else recip(dx)
    T hdt;      // half the time step
};
RH_DEV double e_int(double p, const Consts<double>& k) { return quot(p, k.gm1, k.y_gm1); }
RH_DEV float e_int(float p, const Consts<float>& k) { return p * k.y_gm1; }

// Bounds of a state in range (prim).  Within them, and with dt/dx <= 2^20, dt >=
// 2^-100, dx in [2^-60, 2^60] and gamma - 1 in [2^-10, 64], no FP64 intermediate
// of the update exceeds 1e290 and none that is rounded falls below the normal
// numbers where that could show; the smallest difference of two velocities is
// 2^-453, so products of two differences do not vanish.  FP32 has less room: its
// lower bound is higher, products that vanish are handled by kept, and fluxes
// that overflow are caught by watch.
constexpr double RANGE_HI = 0x1p50;
constexpr double RANGE_LO = 1e-10;
constexpr float RANGE_LO_F = 0x1p-20f;
constexpr int RANGE_EXP = -400;   // of a velocity other than 0
constexpr int TINY_EXP_F = -45;  // of an FP32 velocity that kept looks after

// Conservative -> primitive (the operations of ctoprim); y = 1/density.
// ok is cleared when the state is out of range: below the floors (density and
// internal specific energy t of at least RANGE_LO or RANGE_LO_F; then no floor
// of ctoprim or of the trace's sound speed applies either), too large (s covers
// the density, t and twice the kinetic specific energy; a NaN or an infinity in
// any component reaches s), or with a velocity that is tiny but not 0 (frexp's
// exponent of 0 is 0, so a zero velocity passes).  tiny is set for an FP32
// velocity whose differences' products may vanish.
RH_DEV void prim(const double u[5], double q[5], double& y, const Consts<double>& k, bool& ok, bool&) {
    y = unit_quot(u[0], recip(u[0]));
    q[0] = u[0];
    q[1] = u[1] * y;
    q[2] = u[2] * y;
    q[3] = u[3] * y;
    const double v2 = (q[1] * q[1] + q[2] * q[2]) + q[3] * q[3];
    const double t = fm(-0.5, v2, u[4] * y);
    q[4] = k.gm1 * u[0] * t;
    const double s = (v2 + t) + u[0];
    const int least = min(min(__builtin_amdgcn_frexp_exp(q[1]), __builtin_amdgcn_frexp_exp(q[2])),
                          __builtin_amdgcn_frexp_exp(q[3]));
    ok = ok & (s < RANGE_HI) & (mn(u[0], t) >= RANGE_LO) & (least > RANGE_EXP);
}
RH_DEV void prim(const double ud[5], float q[5], float& y, const Consts<float>& k, bool& ok, bool& tiny) {
    float u[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) u[i] = (float)ud[i];
    y = recip(u[0]);
    q[0] = u[0];
    q[1] = u[1] * y;
    q[2] = u[2] * y;
    q[3] = u[3] * y;
    const float v2 = (q[1] * q[1] + q[2] * q[2]) + q[3] * q[3];
    const float t = fm(-0.5f, v2, u[4] * y);
    q[4] = k.gm1 * u[0] * t;
    const float s = (v2 + t) + u[0];
    const int least = min(min(__builtin_amdgcn_frexp_expf(q[1]), __builtin_amdgcn_frexp_expf(q[2])),
                          __builtin_amdgcn_frexp_expf(q[3]));
    ok = ok & (s < (float)RANGE_HI) & (mn(u[0], t) >= RANGE_LO_F);
    tiny = tiny | (least <= TINY_EXP_F);
}

// Sound speed squared of a trace (its floors: see prim).
template <typename T> RH_DEV T trace_c2(T r, T p, T y, const Consts<T>& k) { return quot(k.gamma * p, r, y); }

// minmod(a, b): the smaller of two differences of one sign, else 0.
RH_DEV double minmod(double a, double b) { return mx(mn(a, b), mn(mx(a, b), 0.0)); }
RH_DEV float minmod(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, 0.0f); }

// The limiters return 0 where the product of the two differences rounds to 0,
// which in FP32 happens ahead of every front, where velocities fall off by
// orders of magnitude from cell to cell (shock tubes of 16^3 to 64^3: in up to
// 20 % of the waves at one step).  Waves with such velocities take the second
// difference b through this: 0 where the product vanishes (left to the general
// form, 96 tubes take 0.575 ms per step instead of 0.504).  Slopes too small
// for the face states' exact factors are left to the general form; of
// velocities near FP32's smallest a quarter of their source term may differ
// from the general form's by that smallest number.
RH_DEV float kept(float a, float b, float lo, bool& ok) {
    const float p = a * b;
    ok = ok & ((p <= 0.0f) | (mn(sabs(a), sabs(b)) >= lo));
    return p != 0.0f ? b : 0.0f;
}
template <typename T> RH_DEV void keep(const T a[5], T b[5], const Consts<T>& k, bool tiny, bool& ok) {
    if constexpr (sizeof(T) == 4) {
        if (__builtin_expect(any_lane(tiny), 0)) {
            const float lo = 0x1p-122f * mx(1.0f, k.dx);
#pragma unroll
            for (int i = 1; i < 4; ++i) b[i] = kept(a[i], b[i], lo, ok);
        }
    }
}

// Difference limited as limiter() does (slope types 0-3 and 6-8); mm =
// minmod(a, b).  Types 4 and 5 are not symmetric under the reflection.
template <typename T> RH_DEV T limited(T a, T b, T mm, int slope_type, bool density) {
    if (slope_type == 1) return mm;
    const T c = T(0.5) * (a + b);
    if (slope_type == 2 || slope_type == 3) return signed_as(mn(sabs(mm + mm), sabs(c)), mm);
    if (slope_type == 8) return signed_as(mn(T(1.5) * sabs(mm), sabs(c)), mm);
    if (slope_type == 6) return density ? c : T(0.0);
    if (slope_type == 7) return mm != T(0.0) ? signed_as(dv(T(2.0) * sabs(a) * sabs(b), sabs(a) + sabs(b)), mm) : T(0.0);
    return T(0.0);
}
// The same for ghost_limiter().
template <typename T> RH_DEV T ghost_limited(T a, T b, T mm, int interpol_type) {
    if (interpol_type == 1) return T(0.5) * mm;
    if (interpol_type == 2) return signed_as(mn(sabs(mm), T(0.25) * sabs(a + b)), mm);
    if (interpol_type == 3) return mm != T(0.0) ? T(0.25) * (a + b) : T(0.0);
    return T(0.0);
}

// Half-step source terms B = hdt*src of density, normal velocity and pressure
// (trace_core), from their slopes.
template <typename T>
RH_DEV void half_sources(const T q[5], T y, T c2, T dr, T du, T dp, const Consts<T>& k, T B[3]) {
    B[0] = k.hdt * (-q[1] * dr - du * q[0]);
    B[1] = k.hdt * (-q[1] * du - quot(dp, q[0], y));
    B[2] = k.hdt * (-q[1] * dp - du * q[0] * c2);
}

// One face state of a cell: q + s*A (+ B on density, normal velocity and
// pressure), A given as the factor times the vector h it is exact in.  least
// keeps the smallest face density: the trace's density floor (the cell's own
// density below 1e-10) is left to the general form.
template <typename T>
RH_DEV void face(const T q[5], const T h[5], T f, const T B[3], T fb, T out[5], T& least) {
    out[0] = fm(fb, B[0], fm(f, h[0], q[0]));
    out[1] = fm(fb, B[1], fm(f, h[1], q[1]));
    out[2] = fm(f, h[2], q[2]);
    out[3] = fm(f, h[3], q[3]);
    out[4] = fm(fb, B[2], fm(f, h[4], q[4]));
    least = mn(least, out[0]);
}

// Slopes of a cell in a form its face states are built from: own state on
// the upper (lower) face = q +- fo*ho + Bo, ghost = q +- fg*hg + fbg*Bg with
// the factors of Factors<SHARED, EXACT>.
// SHARED (slope_type 1 and interpol_type 1): the ghost's difference is half
// the own one and is taken over twice the width, so its slope is a quarter of
// the own slope, its step to the face half and its sources a quarter, all
// exactly; one set of slopes serves both.
// EXACT (dx a power of two): hdx*(L/dx) is exactly L/2.
template <typename T, bool SHARED> struct Slopes {
    T ho[5], Bo[3];
    T hg[SHARED ? 1 : 5], Bg[SHARED ? 1 : 3];
};
template <typename T, bool SHARED, bool EXACT>
RH_DEV void slopes(const T q[5], const T a[5], const T b[5], T y, T c2, int slope_type, int interpol_type,
                   const Consts<T>& k, Slopes<T, SHARED>& s) {
    T dq[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        const T mm = minmod(a[i], b[i]);
        const T L = SHARED ? mm : limited(a[i], b[i], mm, slope_type, i == 0);
        if constexpr (EXACT) {
            s.ho[i] = L;
            dq[i] = L * k.inv;
        } else {
            dq[i] = quot(L, k.dx, k.inv);
            s.ho[i] = k.hdx * dq[i];
        }
    }
    half_sources(q, y, c2, dq[0], dq[1], dq[4], k, s.Bo);
    if constexpr (!SHARED) {
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const T mm = minmod(a[i], b[i]);
            const T L = ghost_limited(a[i], b[i], mm, interpol_type);
            if constexpr (EXACT) {
                s.hg[i] = L;
                dq[i] = L * (T(0.5) * k.inv);
            } else {
                dq[i] = T(0.5) * quot(L, k.dx, k.inv);
                s.hg[i] = k.dx * dq[i];
            }
        }
        half_sources(q, y, c2, dq[0], dq[1], dq[4], k, s.Bg);
    }
}
// up: +1 for the face towards S, -1 for the face towards X.
template <typename T, bool SHARED, bool EXACT>
RH_DEV void own_face(const T q[5], const Slopes<T, SHARED>& s, T up, T out[5], T& least) {
    face(q, s.ho, up * (EXACT ? T(0.5) : T(1.0)), s.Bo, T(1.0), out, least);
}
template <typename T, bool SHARED, bool EXACT>
RH_DEV void ghost_face(const T q[5], const Slopes<T, SHARED>& s, T up, T out[5], T& least) {
    if constexpr (SHARED) face(q, s.ho, up * (EXACT ? T(0.25) : T(0.5)), s.Bo, T(0.25), out, least);
    else face(q, s.hg, up * (EXACT ? T(0.5) : T(1.0)), s.Bg, T(1.0), out, least);
}

// Physical flux and total energy of a face state.
template <typename T> RH_DEV void flux_of(const T q[5], T f[5], T& mu, T& E, const Consts<T>& k) {
    mu = q[0] * q[1];
    E = fm(T(0.5), q[0] * ((q[1] * q[1] + q[2] * q[2]) + q[3] * q[3]), e_int(q[4], k));
    f[0] = mu;
    f[1] = mu * q[1] + q[4];
    f[2] = mu * q[2];
    f[3] = mu * q[3];
    f[4] = (E + q[4]) * q[1];
}
template <typename T> RH_DEV T face_c2(const T q[5], const Consts<T>& k) {
    return quot(k.gamma * q[4], q[0], recip(q[0]));
}

// The range of the states does not keep FP32 products from overflowing (ar*p
// from densities of about 2^30 with sound speeds of 2^20, and sooner where a
// long time step takes the face states beyond the cells').  The general solver
// may return something finite there -- HLLC a physical flux where this one
// multiplies an infinite star term by 0 -- and its minima and maxima treat a
// NaN differently, so fluxes that are not finite are left to it: seen gathers
// the fluxes and stays infinite or NaN once one is.
RH_DEV void watch(const double*, double&) {}
RH_DEV void watch(const float F[5], float& seen) { seen = fm(F[0], F[1], fm(F[2], F[3], seen)) + F[4]; }
RH_DEV bool finite(double) { return true; }
RH_DEV bool finite(float seen) { return sabs(seen) < __builtin_inff(); }

// riemann_hllc.  Its floors on densities, pressures, sound speeds and the
// contact speed are left to the general form: ok is cleared where one would
// apply (a pressure below density*smallp has a squared sound speed of at most
// 1e-20).  Only the larger sound speed is used and the square root is
// monotone, so one root serves.  The side of the contact, and the side whose
// physical flux is the answer where both signals run one way, are one choice;
// there the star term is multiplied by 0 instead of branching.
template <typename T> RH_DEV void hllc(const T l[5], const T r[5], T F[5], const Consts<T>& k, bool mir, bool& ok) {
    const T c2l = face_c2(l, k), c2r = face_c2(r, k);
    const T c = root(mx(c2l, c2r));
    const T sl = mn(l[1], r[1]) - c, sr = mx(l[1], r[1]) + c;
    const T al = l[0] * (l[1] - sl), ar = r[0] * (sr - r[1]);
    const T div = ar + al;
    const T yd = recip(div);
    const T us = quot((ar * r[1] + al * l[1]) + (l[4] - r[4]), div, yd);
    const T ps = nonneg(quot((ar * l[4] + al * r[4]) + al * ar * (l[1] - r[1]), div, yd));
    ok = ok & (mn(c2l, c2r) >= T(2e-20)) & (sabs(us) <= T(1e6));
    const bool pass_l = sl > T(0.0), pass_r = sr < T(0.0);
    const bool left = pass_l | (!pass_r & ((us > T(0.0)) | (mir & (us == T(0.0)))));
    T q[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) q[i] = left ? l[i] : r[i];
    const T sk = left ? sl : sr;
    const int away = left ? 0 : (int)0x80000000;  // den is negative on the left side, positive on the right
    const T den = flip(mn(flip(sk - us, away), T(-1e-10)), away);
    const T ye = recip(den);
    const T dsu = sk - q[1];
    const T rs = quot(q[0] * dsu, den, ye);
    T f[5], mu, E;
    flux_of(q, f, mu, E, k);
    const T Es = quot((dsu * E - q[4] * q[1]) + ps * us, den, ye);
    const T s = (pass_l | pass_r) ? T(0.0) : sk;
    F[0] = f[0] + s * (rs - q[0]);
    F[1] = f[1] + s * (rs * us - mu);
    F[2] = f[2] + s * (rs * q[2] - q[0] * q[2]);
    F[3] = f[3] + s * (rs * q[3] - q[0] * q[3]);
    F[4] = f[4] + s * (Es - E);
    const bool cold = (div < T(1e-5)) & !pass_l & !pass_r;
    if (__builtin_expect(any_lane(cold), 0)) {
        T fl[5], fr[5];
        flux_of(l, fl, mu, E, k);
        flux_of(r, fr, mu, E, k);
#pragma unroll
        for (int i = 0; i < 5; ++i) F[i] = cold ? T(0.5) * (fl[i] + fr[i]) : F[i];
    }
}

// riemann_llf and riemann_hll (whose signals are at least 2e-10 apart here).
template <typename T> RH_DEV void llf(const T l[5], const T r[5], T F[5], const Consts<T>& k) {
    T fl[5], fr[5], ml, mr, El, Er;
    flux_of(l, fl, ml, El, k);
    flux_of(r, fr, mr, Er, k);
    const T cl = root(mx(face_c2(l, k), T(1e-20))), cr = root(mx(face_c2(r, k), T(1e-20)));
    const T am = T(0.5) * mx(sabs(l[1]) + cl, sabs(r[1]) + cr);
    F[0] = T(0.5) * (fl[0] + fr[0]) - am * (r[0] - l[0]);
    F[1] = T(0.5) * (fl[1] + fr[1]) - am * (mr - ml);
    F[2] = T(0.5) * (fl[2] + fr[2]) - am * (r[0] * r[2] - l[0] * l[2]);
    F[3] = T(0.5) * (fl[3] + fr[3]) - am * (r[0] * r[3] - l[0] * l[3]);
    F[4] = T(0.5) * (fl[4] + fr[4]) - am * (Er - El);
}
template <typename T> RH_DEV void hll(const T l[5], const T r[5], T F[5], const Consts<T>& k) {
    T fl[5], fr[5], ml, mr, El, Er;
    flux_of(l, fl, ml, El, k);
    flux_of(r, fr, mr, Er, k);
    const T cl = root(mx(face_c2(l, k), T(1e-20))), cr = root(mx(face_c2(r, k), T(1e-20)));
    const T sl = mn(T(0.0), mn(l[1] - cl, r[1] - cr)), sr = mx(T(0.0), mx(l[1] + cl, r[1] + cr));
    const T w = sr - sl, i = unit_quot(w, recip(w)), ss = sr * sl;
    F[0] = ((sr * fl[0] - sl * fr[0]) + ss * (r[0] - l[0])) * i;
    F[1] = ((sr * fl[1] - sl * fr[1]) + ss * (mr - ml)) * i;
    F[2] = ((sr * fl[2] - sl * fr[2]) + ss * (r[0] * r[2] - l[0] * l[2])) * i;
    F[3] = ((sr * fl[3] - sl * fr[3]) + ss * (r[0] * r[3] - l[0] * l[3])) * i;
    F[4] = ((sr * fl[4] - sl * fr[4]) + ss * (Er - El)) * i;
}

// riemann_acoustic: few runs use it, so it keeps the general divisions; only
// the side taken at a zero contact speed depends on the frame.
RH_DEV void acoustic(const double l[5], const double r[5], double F[5], const Consts<double>& k, bool mir) {
    riemann_acoustic(l, r, F, Gas<double>{k.gamma, k.gm1, k.smalle, k.smallp, 0.0}, mir);
}
RH_DEV void acoustic(const float l[5], const float r[5], float F[5], const Consts<float>& k, bool mir) {
    riemann_acoustic_f(l, r, F, Gas<float>{k.gamma, k.gm1, k.smalle, k.smallp, k.y_gm1}, mir);
}

template <int R, typename T>
RH_DEV void riemann(const T l[5], const T r[5], T F[5], const Consts<T>& k, bool mir, bool& ok) {
    if constexpr (R == 2) hllc(l, r, F, k, mir, ok);
    else if constexpr (R == 1) hll(l, r, F, k);
    else if constexpr (R == 4) acoustic(l, r, F, k, mir);
    else llf(l, r, F, k);
}

}  // namespace fast
}  // namespace rh
