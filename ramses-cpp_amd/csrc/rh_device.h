// rh_device.h -- device helpers shared by the kernel files: cell indexing,
// state loads, the Courant candidate, ordered keys, the own update of a cell.
#pragma once
#include "rh_kernels.h"
#include "rh_physics.h"

namespace rh {
namespace {

RH_DEV void load_u(const double* __restrict__ u, int ncell, int icell, double out[5]) {
    const size_t i = (size_t)icell - 1;
#pragma unroll
    for (int iv = 0; iv < 5; ++iv) out[iv] = u[(size_t)iv * ncell + i];
}

RH_DEV int cell_id(const MeshDev& m, int igrid, int ic0) { return m.ncoarse + ic0 * m.ngridmax + igrid; }

// Index of cell ic0 among the four cells on an oct face normal to d.
RH_DEV int face_slot(int ic0, int d) { return ((ic0 >> (d + 1)) << d) | (ic0 & ((1 << d) - 1)); }

template <typename T> RH_DEV void copy5(const T a[5], T b[5]) {
#pragma unroll
    for (int i = 0; i < 5; ++i) b[i] = a[i];
}

// NaN-skipping minimum: a NaN candidate never replaces the running value,
// as with std::min(dt_max, dt_cand) in the reference loop.
RH_DEV double min_skip_nan(double a, double b) { return (b < a) ? b : a; }

// A lane's own NaN must not stand for its partners' values either.
RH_DEV double wave_min(double v) {
    v = min_skip_nan(__builtin_inf(), v);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        double o = __shfl_xor(v, off, 64);
        v = min_skip_nan(v, o);
    }
    return v;
}

// Courant candidate of one leaf cell, HydroSolver.cpp:878-977.
RH_DEV double courant_cand_u(const MeshDev& m, const double u[5], int id, double dx, double gamma,
                             double courant_factor) {
    double d = smax(u[0], 1e-10), v2 = 0.0;
    for (int i = 1; i <= 3; ++i) {
        double v = u[i] / d;
        v2 = v2 + v * v;
    }
    // The reference subtracts a non-thermal energy of 0 and adds a
    // non-thermal sound speed of 0/d: both leave every value unchanged (c2
    // is at least 1e-20 or NaN, and d is NaN only where the velocities and
    // so the result are), so they are left out.
    double pr = smax((u[4] - 0.5 * d * v2) * (gamma - 1.0), d * 1e-10);
    pr = smin(pr, d * 1e2);
    double c2 = smax(gamma * pr / smax(d, 1e-10), 1e-20);
    double cs = ssqrt(smax(c2, 1e-10));
    double u_wave = 3 * cs;
    for (int i = 1; i <= 3; ++i) u_wave = u_wave + sabs(u[i] / d);
    if (!m.f) {
        // No gravity: a_grav = 0, so alpha = max(0 * dx / u_wave^2, 1e-4) =
        // 1e-4 wherever u_wave is a number (it is at least 3e-5); where it
        // is NaN the result is NaN either way.
        const double s1 = ssqrt(1.0 + 2.0 * courant_factor * 1e-4) - 1.0;
        return (dx / u_wave) * s1 / 1e-4;
    }
    double a_grav = 0.0;
    for (int i = 1; i <= 3; ++i) a_grav = a_grav + sabs(m.f[(size_t)(i - 1) * m.ncell + id - 1]);
    double alpha = a_grav * dx / (u_wave * u_wave);
    alpha = smax(alpha, 0.0001);
    return (dx / u_wave) * (ssqrt(1.0 + 2.0 * courant_factor * alpha) - 1.0) / alpha;
}

// Block minimum over an NT-thread block (NT a multiple of 64).
template <int NT> RH_DEV void block_min_n(double cand, double* part) {
    __shared__ double s_min[NT / 64];
    const int t = threadIdx.x;
    cand = wave_min(cand);
    if ((t & 63) == 0) s_min[t >> 6] = cand;
    __syncthreads();
    if (t == 0) {
        double v = s_min[0];
        for (int w = 1; w < NT / 64; ++w) v = min_skip_nan(v, s_min[w]);
        part[blockIdx.x] = v;
    }
}

// Ordered 64-bit key of a double: unsigned comparison of keys orders them as
// the doubles (-0 before +0), and NaN maps to the largest key, so a minimum
// over keys never picks a NaN candidate -- the reference's std::min loop
// skips them too.  The minimum of a set is order-independent, so atomics
// give a deterministic result.
RH_DEV unsigned long long dt_key(double v) {
    if (v != v) return ~0ull;
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
RH_DEV double key_dt(unsigned long long k) {
    const unsigned long long b = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    return __longlong_as_double((long long)b);
}

// Time step and cell width of oct p: the kernel arguments for a single mesh,
// its box's entries for an ensemble.
RH_DEV void step_of(const LevelDev& lv, int p, const double* d_dt, double& dt, double& dx, double& inv_dx) {
    if (lv.obox) {
        const int bx = lv.obox[p];
        dt = d_dt[bx];
        dx = lv.box_len[bx];
        inv_dx = lv.box_len[lv.nbox + bx];
    } else {
        dt = *d_dt;
    }
}

struct Nbr {
    int cell;  // 1-based cell index (<= 0: boundary)
    int pos;   // oct position in the level list, or -1 for a record
    int ic0;   // cell within that oct
    int rec;   // record index when pos < 0
};

template <typename TC> RH_DEV void narrow(const double a[5], TC b[5]) {
#pragma unroll
    for (int i = 0; i < 5; ++i) b[i] = (TC)a[i];
}

// Primitive state of a cell for the slopes, traces and Riemann problems:
// FP64 ctoprim in the FP64 form; in the mixed form the conservative state is
// narrowed to FP32 and converted there.
template <typename TC>
RH_DEV void face_prim(const double u[5], TC q[5], const Gas<double>& gd, const Gas<TC>& gc) {
    if constexpr (sizeof(TC) == 8) {
        ctoprim(u, q, gd);
    } else {
        TC uc[5];
        narrow(u, uc);
        ctoprim(uc, q, gc);
    }
}

// One face's Riemann problem: the FP64 form calls the bit-faithful solver on
// double states; the mixed form solves it in FP32 (its flux is widened to
// FP64 where it enters the update or a reflux).  ql/qr are rotated; F comes
// back rotated.
template <int RIEMANN, bool MIXED, typename TC>
RH_DEV void solve_face(const TC ql[5], const TC qr[5], TC F[5], const Gas<TC>& gc, const Gas<double>& gd) {
    if constexpr (MIXED) riemann_f<RIEMANN>(ql, qr, F, gc);
    else riemann<RIEMANN>(ql, qr, F, gd);
}

// A leaf cell's own update and clamps, HydroSolver.cpp:489-547.
RH_DEV void own_update(double u[5], const double fs[5], double dtdx, const GasParams& gp) {
#pragma unroll
    for (int iv = 0; iv < 5; ++iv) u[iv] = u[iv] + dtdx * fs[iv];
    double d_curr = sclamp(u[0], 1e-10, 1e6);
    u[0] = d_curr;
    for (int i = 1; i <= 3; ++i) u[i] = sclamp(u[i], -d_curr * 10.0, d_curr * 10.0);
    double v2_curr = 0.0;
    for (int i = 1; i <= 3; ++i) {
        double v = u[i] / d_curr;
        v2_curr = v2_curr + v * v;
    }
    double ei_curr = u[4] - 0.5 * d_curr * v2_curr;
    if (ei_curr < d_curr * 1e-10 / gp.gm1) {
        double e_non = 0;
        u[4] = d_curr * 1e-10 / gp.gm1 + 0.5 * d_curr * v2_curr + e_non;
    }
    u[4] = smin(u[4], d_curr * 1e8);
}

constexpr long long KMAX = 0x7fffffffffffffffLL;

// Keys of the six incoming contributions of cell ic0 of oct p, from the
// tables (face slot f; -1: none): the sibling's when it is a leaf, X's when
// its oct is a same-level neighbour and X a leaf.
RH_DEV void incoming_keys(const LevelDev& lv, int p, int ic0, int lm, long long kin[6]) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const bool par = (ic0 >> d) & 1;
        const int icS = ic0 ^ (1 << d);
        const long long kS = ((lm >> icS) & 1) ? ((long long)p * 8 + icS) * 8 + (par ? 2 * d + 1 : 2 * d) : -1;
        const int E = lv.nbo[(size_t)(2 * d + (par ? 1 : 0)) * lv.noct + p];
        long long kX = -1;
        if (E >= 0 && ((lv.leaf[E] >> icS) & 1)) kX = ((long long)E * 8 + icS) * 8 + (par ? 2 * d : 2 * d + 1);
        kin[2 * d] = par ? kS : kX;
        kin[2 * d + 1] = par ? kX : kS;
    }
}

template <typename T> RH_DEV void shfl5(const T in[5], T out[5], int mask) {
#pragma unroll
    for (int i = 0; i < 5; ++i) out[i] = __shfl_xor(in[i], mask, 64);
}
template <typename T> RH_DEV void sel5(bool c, const T a[5], const T b[5], T out[5]) {
#pragma unroll
    for (int i = 0; i < 5; ++i) out[i] = c ? a[i] : b[i];
}

// Workgroup index -> oct range, XCD-aware.  The dispatcher deals
// workgroups round-robin to the 8 XCDs, each with its own L2, so workgroup
// x runs on XCD x % 8.  Renumbering gives each XCD one contiguous share of
// the list (XCD k takes ranges k*q.. in order, q = n/8, the first n%8 XCDs
// one more), so octs that are neighbours in the list's Morton order, whose
// cells each other's line gathers read, share an L2 instead of every
// neighbour pair fetching the same lines from HBM on two XCDs.  A bijection
// of [0, n) for any n.
RH_DEV int xcd_block(int x, int n) {
    const int xcd = x & 7, idx = x >> 3, q = n >> 3, r = n & 7;
    return xcd < r ? xcd * (q + 1) + idx : r * (q + 1) + (xcd - r) * q + idx;
}

}  // namespace
}  // namespace rh
