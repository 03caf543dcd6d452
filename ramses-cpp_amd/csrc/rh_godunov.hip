// rh_godunov.hip -- the Godunov update for ordinary states, one Riemann solver
// per translation unit (RH_RIEMANN).
//
//   k_step_oct    one wave per 8 octs, the three dimensions one after another
//   k_step_dims   three waves per 8 octs, one dimension each
//
// The eight cells of an oct sit in eight adjacent lanes, a lane's sibling
// along dimension d is lane ^ (1 << d).  Both kernels run dim_pass, which
// computes one dimension of a cell's update in the frame of rh_fast.h, and for
// the waves in which some state is out of that frame's range the general form
// (general_dim).
//
// Bound: the vector ALU, 78-79 % (FP64) and 65-69 % (mixed) busy at the
// 1.8-2.2 GHz that these launches run at.  An HLLC/MinMod update executes 2,552
// VALU instructions per cell in the FP64 form and 2,050 in the mixed form, and
// 149 more for the next step's Courant candidate (the kernels of rh_hydro.hip,
// which select each operand by a cell's place in its oct, round every division
// separately and trace own and ghost states apart: 5,747 and 3,779, and
// 180-195); HBM traffic is a quarter of what the memory delivers.  At 2^21
// octs (256^3 cells) a launch takes 1.69-1.75 ms in the FP64 form and 1.45-1.47
// ms in the mixed form, against 3.48 and 2.09 ms; at 512 octs 9.4 and 9.2 us
// against 12.8 and 12.1 us (k_step_dims).
// Registers: three waves per SIMD (168 per lane).  Two waves took 2.04 ms
// against 1.90 (FP64, an earlier order of the code), four waves 1.61 against
// 1.49 (mixed, 24 bytes spilled): a spill is written through to memory for
// every wave, so what the ordinary update keeps per lane is arranged to need
// none (the general form's 180-220 bytes are touched by its waves only).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rh_device.h"
#include "rh_fast.h"
#include "rh_godunov.h"

namespace rh {

namespace {

// Waves per SIMD asked for (registers per lane: 168 / 128 at 3 / 4).  The mixed
// k_step_dims needs 120 with its general form out of line; at three waves that
// took 163 and the launch 1.95 ms at 2^21 octs instead of 1.78.
constexpr int OCT_WAVES = 3, DIMS_WAVES = 3, DIMS_WAVES_F = 4;

using fast::all_lanes;
using fast::any_lane;
using fast::Consts;
using fast::flip;
using fast::Slopes;

// ---------------------------------------------------------------------------
// General form of a wave's update: any finite or non-finite state, any mesh,
// octs of several boxes, each lane with its own time step and cell width.  The
// routines of rh_physics.h in the reference's orientation, the eight cells of
// an oct in eight lanes as in the ordinary form: per dimension four traces and
// three Riemann problems a cell.  It is reached by waves that hold a state out
// of range (ahead of a blast's front, where velocities fall off towards 0; cold
// gas in the mixed form) or an oct that is its own neighbour.
// Bound: a launch waits for its slowest wave, so what counts is the length of
// one wave's instruction stream, and where many waves come here, spills, which
// are written to memory.  k_step_dims has each of its waves do its own
// dimension.  One such wave in a launch of 512 octs adds 8 us in the FP64 form
// and 6 in the mixed form, in one of 32,768 octs 20 and 7; with every wave
// here 2^18 octs take 0.70 and 0.26 ms.  (One lane per cell, recomputing the
// face problems one after another from LDS, added 87 and 71 us, 82 and 67, and
// took 1.55 and 1.12 ms: 64^3 blasts ran at 112 instead of 56 us per step.)

template <typename T> using SharedRows = __attribute__((address_space(3))) T*;
template <typename T, int N> RH_DEV SharedRows<T> shared_rows(T (*w)[N]) { return (SharedRows<T>)&w[0][0]; }

// The launch's arguments, read again: kept in registers through the ordinary
// form they would cost it some.
RH_DEV const void* launch_args() { return (const void*)__builtin_amdgcn_kernarg_segment_ptr(); }
RH_DEV StepArgs args_at(const void* p) {
    typedef const __attribute__((address_space(4))) char* Kernarg;
    const unsigned long long v = (unsigned long long)p;
    const unsigned long long u = ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
                                 (unsigned)__builtin_amdgcn_readfirstlane((int)v);
    StepArgs a;
    __builtin_memcpy(&a, (const void*)(Kernarg)u, sizeof(a));
    return a;
}

// A value that is the same in every lane, in scalar registers.
RH_DEV double uniform(double x) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)),
                            __builtin_amdgcn_readfirstlane(__double2loint(x)));
}
RH_DEV float uniform(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }

// Five rows of a lane's column.
template <typename T> RH_DEV void put_rows(SharedRows<T> w, int t, const T v[5]) {
#pragma unroll
    for (int i = 0; i < 5; ++i) w[i * 64 + t] = v[i];
}
template <typename T> RH_DEV void get_rows(SharedRows<T> w, int t, T v[5]) {
#pragma unroll
    for (int i = 0; i < 5; ++i) v[i] = w[i * 64 + t];
}

// A lane's cell.
struct GeneralCell {
    int p, ic0, lm, cC;
    bool leaf;
};
// The step of its box.
template <typename T> struct GeneralStep {
    double dtdx;
    T dt, dx, inv;  // inv: 1/dx where exact
};
// In the FP64 form nothing is moved across.
template <bool MIXED> RH_DEV void phase() {
    if constexpr (!MIXED) __builtin_amdgcn_sched_barrier(0);
}
template <typename T>
RH_DEV void general_prim(const StepArgs& a, const Gas<T>& gc, int icell, T q[5]) {
    const Gas<double> gd{a.gp.gamma, a.gp.gm1, a.gp.smalle, a.gp.smallp, 1.0 / a.gp.gm1};
    double u[5];
    load_u(a.m.uold, a.m.ncell, icell, u);
    face_prim(u, q, gd, gc);
}
RH_DEV GeneralCell general_cell(const StepArgs& a, int praw, int t) {
    GeneralCell c;
    c.ic0 = t & 7;
    c.p = min(praw, a.lv.noct - 1);
    c.lm = a.lv.leaf[c.p];
    c.leaf = praw < a.lv.noct && ((c.lm >> c.ic0) & 1);
    c.cC = cell_id(a.m, a.lv.grid[c.p], c.ic0);
    return c;
}
template <typename T> RH_DEV GeneralStep<T> general_step(const StepArgs& a, int p, double dt, double dx) {
    double inv_dx = a.inv_dx;
    if (a.lv.obox) step_of(a.lv, p, a.d_dt, dt, dx, inv_dx);
    return {dt / dx, (T)dt, (T)dx, (T)inv_dx};
}
template <typename T> RH_DEV Gas<T> general_gas(const StepArgs& a) {
    return {(T)a.gp.gamma, (T)a.gp.gm1, (T)a.gp.smalle, (T)a.gp.smallp, (T)(1.0 / a.gp.gm1)};
}

// One dimension: the cell's own fluxes through the oct's face (Fe) and towards
// its sibling (Fi), and the flux X computes through the oct's face (Fx);
// rotated order, zero where there is none.  w: five rows for what does not fit
// the registers.
template <int R, bool MIXED, bool EXACT, bool SHARED, typename T>
RH_DEV void general_dim(const StepArgs& a, const Gas<T>& gc, const GeneralCell& c, GeneralStep<T> g, int d,
                        SharedRows<T> w, int t, T Fe[5], T Fi[5], T Fx[5]) {
    const MeshDev& m = a.m;
    const LevelDev& lv = a.lv;
    const int st = SHARED ? 1 : a.gp.slope_type, it = SHARED ? 1 : a.gp.interpol_type;
    const Gas<double> gd{a.gp.gamma, a.gp.gm1, a.gp.smalle, a.gp.smallp, 1.0 / a.gp.gm1};
    // Nothing made of them is kept from one dimension to the next.
    if constexpr (!MIXED) asm volatile("" : "+v"(g.dt), "+v"(g.dx));
    const Len<T, EXACT> len{g.dx, g.inv};
    // trace() of a cell's own (over dx) or ghost state (over twice that).
    auto traced = [&](const T q[5], const T dq[5], T hdx, T qm[5], T qp[5]) {
        const T r = smax(q[0], T(1e-10));
        trace_core(q, dq, r, q[1], cs2(r, smax(q[4], r * T(1e-20)), gc), hdx, T(0.5) * g.dt, qm, qp);
    };
    const int b = 1 << d;
    const bool par = (c.ic0 >> d) & 1;
    const int icS = c.ic0 ^ b;
    const int E = lv.nbo[(size_t)(2 * d + (par ? 1 : 0)) * lv.noct + c.p];
    int4 rc = make_int4(0, 0, 0, 0);
    int X, X2 = 0, cC = c.cC;
    if (E >= 0) {
        const int gE = lv.grid[E];
        X = cell_id(m, gE, icS);
        if ((lv.leaf[E] >> icS) & 1) X2 = cell_id(m, gE, c.ic0);
    } else {
        rc = lv.rec[-1 - E];
        X = rc.x;
    }
    // The FP64 form's phases are kept apart: scheduled into one another they need
    // more registers than there are, and every spill is written to memory.
    T q[5], x[5];
    general_prim(a, gc, c.cC, q);
    copy5(q, x);
    if (X > 0) general_prim(a, gc, X, x);
    rotate(q, d);
    rotate(x, d);
    phase<MIXED>();
    // The cell's ghost and own states: towards X (gx, ox) and towards the
    // sibling (l, z, of which the sibling's own ghost state comes here).
    T ox[5], gx[5], l[5], r[5], z[5], mi[5], pl[5];
    {
        T s[5], dq[5];
        shfl5(q, s, b);
        sel5(par, s, x, l);
        sel5(par, x, s, r);
        ghost_slopes(l, q, r, it, coarse(len), dq);
        phase<MIXED>();
        traced(q, dq, g.dx, mi, pl);
        sel5(par, mi, pl, gx);
        if constexpr (!MIXED) put_rows(w, t, gx);
        sel5(par, pl, mi, z);
        phase<MIXED>();
        own_slopes(l, q, r, st, g.dt, len, dq);
        phase<MIXED>();
        traced(q, dq, T(0.5) * g.dx, mi, pl);
        sel5(par, mi, pl, ox);
        sel5(par, pl, mi, s);
        shfl5(z, z, b);
        sel5(par, z, s, l);
        sel5(par, s, z, r);
    }
    phase<MIXED>();
    solve_face<R, MIXED>(l, r, Fi, gc, gd);
    phase<MIXED>();
    const bool sib_leaf = (c.lm >> icS) & 1;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        Fi[i] = sib_leaf ? Fi[i] : T(0);
        Fe[i] = Fx[i] = T(0);
    }

    // The neighbour's states on the oct's face: z its ghost state, x its own.
    const bool refined = rc.w & REC_REFINED_DEV, bound = rc.w & REC_BOUNDARY_DEV;
    if (E >= 0 ? X2 <= 0 : refined) return;
    if constexpr (!MIXED) {
        // Read again: kept through the solve they would be spilled.
        asm volatile("" : "+v"(X), "+v"(cC)::"memory");
        if (!bound) {
            general_prim(a, gc, X > 0 ? X : cC, x);
            rotate(x, d);
        }
        if (E >= 0) {
            general_prim(a, gc, cC, q);
            rotate(q, d);
        }
    }
    if (E >= 0) {
        T dq[5];
        general_prim(a, gc, X2, r);
        rotate(r, d);
        sel5(par, q, r, l);
        sel5(par, r, q, r);
        phase<MIXED>();
        ghost_slopes(l, x, r, it, coarse(len), dq);
        phase<MIXED>();
        traced(x, dq, g.dx, mi, pl);
        sel5(par, pl, mi, z);
        phase<MIXED>();
        own_slopes(l, x, r, st, g.dt, len, dq);
        phase<MIXED>();
        traced(x, dq, T(0.5) * g.dx, mi, pl);
        sel5(par, pl, mi, x);
    } else if (bound) {
        // The cell's own state with the normal momentum reversed, traced
        // without slopes.
        double u[5];
        load_u(m.uold, m.ncell, cC, u);
#pragma unroll
        for (int i = 1; i <= 3; ++i)
            if (i == 1 + d) u[i] = u[i] * -1.0;
        T dq[5] = {T(0), T(0), T(0), T(0), T(0)};
        face_prim(u, q, gd, gc);
        rotate(q, d);
        traced(q, dq, T(0.5) * g.dx, mi, pl);
        sel5(par, pl, mi, z);
    } else {
        // A coarser cell, between its own neighbours.
        copy5(x, l);
        copy5(x, r);
        if (rc.y > 0) {
            general_prim(a, gc, rc.y, l);
            rotate(l, d);
        }
        if (rc.z > 0) {
            general_prim(a, gc, rc.z, r);
            rotate(r, d);
        }
        T dq[5];
        ghost_slopes(l, x, r, it, coarse(len), dq);
        traced(x, dq, g.dx, mi, pl);
        sel5(par, pl, mi, z);
    }
    phase<MIXED>();
    sel5(par, ox, z, l);
    sel5(par, z, ox, r);
    solve_face<R, MIXED>(l, r, Fe, gc, gd);
    phase<MIXED>();
    if (E >= 0) {
        if constexpr (!MIXED) get_rows(w, t, gx);
        sel5(par, gx, x, l);
        sel5(par, x, gx, r);
        solve_face<R, MIXED>(l, r, Fx, gc, gd);
    } else if (!bound && c.leaf) {
        const int slot = lv.rec_slot[-1 - E] + face_slot(c.ic0, d);
        const double sg = par ? -1.0 : 1.0;
        T F[5];
        rotated(Fe, F, d);
#pragma unroll
        for (int iv = 0; iv < 5; ++iv) lv.slot_r[(size_t)slot * 5 + iv] = g.dtdx * sg * F[iv] * 0.125;
    }
    phase<MIXED>();
}

// Contribution rows as the ordinary form keeps them (see contribution()): what
// is added to the cell, the mixed form's without its factor.
RH_DEV double general_row(double F, double dtdx, bool minus) { return dtdx * (minus ? -F : F) * 0.125; }
RH_DEV float general_row(float F, double, bool minus) { return minus ? -F : F; }
RH_DEV double general_added(double w, double) { return w; }
RH_DEV double general_added(float w, double dtdx) { return dtdx * (double)w * 0.125; }
template <typename T>
RH_DEV void general_rows(const T F[5], int d, double dtdx, bool minus, T out[5]) {
    rotated(F, out, d);
#pragma unroll
    for (int iv = 0; iv < 5; ++iv) out[iv] = general_row(out[iv], dtdx, minus);
}

// The ordered accumulation of a cell: its own update takes its place among the
// contributions by their keys.  w: rows 5d+iv from X of dimension d, rows
// 15+5d+iv from S of dimensions 0 and 1; ws2 those of dimension 2.
template <typename T>
RH_DEV void general_apply(const StepArgs& a, const GeneralCell& c, double dtdx, double u[5], const double fs[5], const T ws2[5],
                          SharedRows<T> w, int t) {
    long long kin[6];
    incoming_keys(a.lv, c.p, c.ic0, c.lm, kin);
    const long long KOWN = ((long long)c.p * 8 + c.ic0) * 8 + 6;
    int done = 0;
#pragma unroll 1
    for (int step = 0; step < 7; ++step) {
        long long best = (done & 64) ? KMAX : KOWN;
        int f = (done & 64) ? 7 : 6;
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            const bool take = !((done >> j) & 1) && kin[j] >= 0 && kin[j] < best;
            best = take ? kin[j] : best;
            f = take ? j : f;
        }
        if (f == 7) break;
        done |= 1 << f;
        if (f == 6) {
            own_update(u, fs, dtdx, a.gp);
        } else {
            // Face f of the cell is the one across which X lies where its
            // side is the cell's side of the oct.
            const int d = f >> 1;
            const bool from_x = (f & 1) == ((c.ic0 >> d) & 1), in_regs = f >= 4 && !from_x;
            const int row = from_x ? 5 * d : 15 + 5 * (d & 1);
#pragma unroll
            for (int iv = 0; iv < 5; ++iv) {
                const T v = w[(row + iv) * 64 + t];
                u[iv] = u[iv] + general_added(in_regs ? ws2[iv] : v, dtdx);
            }
        }
    }
}

template <bool MIXED> using StepType = std::conditional_t<MIXED, float, double>;

// The whole update of a wave: the new state of its cells.  praw: the lane's
// oct; w: 25 rows.
template <int R, bool MIXED, bool EXACT, bool SHARED>
RH_DEV void general_wave(const void* args, SharedRows<StepType<MIXED>> w, int praw, int t, double dt, double dx,
                         double u[5]) {
    using T = StepType<MIXED>;
    const StepArgs a = args_at(args);
    const Gas<T> gc = general_gas<T>(a);
    const GeneralCell c = general_cell(a, praw, t);
    const GeneralStep<T> g = general_step<T>(a, c.p, dt, dx);
    double fs[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    T ws[5];
    // As in k_godunov_oct: three copies of the dimension's code lose more in
    // instruction fetch than the constant rotations gain in the FP64 form
    // of HLLC only.
    constexpr int DIM_UNROLL = (MIXED || R != 2) ? 3 : 1;
#pragma unroll DIM_UNROLL
    for (int d = 0; d < 3; ++d) {
        T Fe[5], Fi[5], Fx[5], row[5];
        general_dim<R, MIXED, EXACT, SHARED>(a, gc, c, g, d, w + 5 * d * 64, t, Fe, Fi, Fx);
        const bool par = (c.ic0 >> d) & 1;
        general_rows(Fx, d, g.dtdx, par, row);
        put_rows(w + 5 * d * 64, t, row);
        shfl5(Fi, row, 1 << d);
        general_rows(row, d, g.dtdx, !par, ws);
        if (d < 2) put_rows(w + (15 + 5 * d) * 64, t, ws);
        rotate(Fe, d);
        rotate(Fi, d);
#pragma unroll
        for (int iv = 0; iv < 5; ++iv) {
            fs[iv] = fs[iv] + (double)(par ? Fi[iv] : Fe[iv]);
            fs[iv] = fs[iv] - (double)(par ? Fe[iv] : Fi[iv]);
        }
    }
    load_u(a.pre, a.m.ncell, c.cC, u);
    if (c.leaf) general_apply(a, c, g.dtdx, u, fs, ws, w, t);
}

// One dimension for k_step_dims, with the results where dim_pass leaves its
// own: contributions in rows 5d and 15+5d of w, own fluxes in the cell's frame
// (rh_fast.h) in rows 0-4 and 5-9 of o.
template <int R, bool MIXED, bool EXACT, bool SHARED>
__device__ __attribute__((noinline)) void general_one_dim(const void* args, SharedRows<StepType<MIXED>> w,
                                                          SharedRows<StepType<MIXED>> o, int d, int praw, int t,
                                                          double dt, double dx) {
    using T = StepType<MIXED>;
    const StepArgs a = args_at(args);
    d = __builtin_amdgcn_readfirstlane(d);
    const Gas<T> gc = general_gas<T>(a);
    const GeneralCell c = general_cell(a, praw, t);
    const GeneralStep<T> g = general_step<T>(a, c.p, dt, dx);
    T Fe[5], Fi[5], Fx[5], row[5];
    general_dim<R, MIXED, EXACT, SHARED>(a, gc, c, g, d, w + 5 * d * 64, t, Fe, Fi, Fx);
    const bool par = (c.ic0 >> d) & 1;
    general_rows(Fx, d, g.dtdx, par, row);
    put_rows(w + 5 * d * 64, t, row);
    shfl5(Fi, Fx, 1 << d);
    general_rows(Fx, d, g.dtdx, !par, row);
    put_rows(w + (15 + 5 * d) * 64, t, row);
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        Fe[i] = par && i != 1 ? -Fe[i] : Fe[i];
        Fi[i] = par && i != 1 ? -Fi[i] : Fi[i];
    }
    put_rows(o, t, Fe);
    put_rows(o + 5 * 64, t, Fi);
}
// The accumulation for k_step_dims (row 25: those of S of dimension 2).
struct State5 {
    double u[5];
};
template <bool MIXED>
__device__ __attribute__((noinline)) State5 general_sum(const void* args, SharedRows<StepType<MIXED>> w, State5 fs,
                                                        int praw, int t, double dt, double dx) {
    using T = StepType<MIXED>;
    const StepArgs a = args_at(args);
    const GeneralCell c = general_cell(a, praw, t);
    State5 s;
    const GeneralStep<T> g = general_step<T>(a, c.p, dt, dx);
    T ws2[5];
    get_rows(w + 25 * 64, t, ws2);
    load_u(a.pre, a.m.ncell, c.cC, s.u);
    if (c.leaf) general_apply(a, c, g.dtdx, s.u, fs.u, ws2, w, t);
    return s;
}

// ---------------------------------------------------------------------------

// Element i of an array at a byte offset that fits 32 bits (step_kernels_take):
// the base stays in scalar registers and the lane's part of the address is one
// 32-bit value, shared by the five components of a state.  The empty asm keeps
// the compiler from adding the two up in 64 bits per component.
template <typename E> using GlobalPtr = __attribute__((address_space(1))) E*;
template <typename E> RH_DEV GlobalPtr<E> scalar_base(E* p) {
    GlobalPtr<E> g = (GlobalPtr<E>)p;
    asm("" : "+s"(g));
    return g;
}
template <typename E> RH_DEV E at(const E* base, unsigned i) {
    return *(GlobalPtr<const E>)((GlobalPtr<const char>)scalar_base(base) + i * (unsigned)sizeof(E));
}
RH_DEV void load5(const MeshDev& m, const double* u, int icell, double out[5]) {
    const unsigned off = ((unsigned)icell - 1u) * 8u;
#pragma unroll
    for (int iv = 0; iv < 5; ++iv)
        out[iv] = *(GlobalPtr<const double>)((GlobalPtr<const char>)scalar_base(u + (size_t)iv * m.ncell) + off);
}
RH_DEV void store5(const MeshDev& m, double* u, int icell, const double v[5]) {
    const unsigned off = ((unsigned)icell - 1u) * 8u;
#pragma unroll
    for (int iv = 0; iv < 5; ++iv)
        *(GlobalPtr<double>)((GlobalPtr<char>)scalar_base(u + (size_t)iv * m.ncell) + off) = v[iv];
}

// Value of lane ^ (1 << D), through the LDS crossbar without an address.
template <int D> RH_DEV int across_lanes(int x) { return __builtin_amdgcn_ds_swizzle(x, ((1 << D) << 10) | 0x1f); }
template <int D> RH_DEV float sib(float x) { return __int_as_float(across_lanes<D>(__float_as_int(x))); }
template <int D> RH_DEV double sib(double x) {
    return __hiloint2double(across_lanes<D>(__double2hiint(x)), across_lanes<D>(__double2loint(x)));
}

// Component of a global state at position i of the rotated order.
template <int D> constexpr int rot(int i) {
    return i == 1 ? 1 + D : i == 2 ? (D == 1 ? 1 : 2) : i == 3 ? (D == 2 ? 1 : 3) : i;
}

// A cell's own fluxes of one dimension, in its frame and rotated order: Fe
// through the oct's face, Fi towards its sibling.
template <typename T> struct DimFlux {
    T Fe[5], Fi[5];
};

// A wave's cells and constants.
template <typename T> struct Cell {
    int p, ic0, lm, cC;
    bool leaf, tiny;  // tiny: see fast::prim
    T q[5], y, c2;  // primitives in global order, 1/density, trace_c2
};

// A contribution to a cell is -((dtdx*sign)*F)*0.125 with the neighbour's flux
// F in the global frame, added to the cell: k8*F in the cell's frame (k8 =
// dtdx/8; the normal momentum's sign as given by s).  The FP64 form passes on
// the product, the mixed form the FP32 flux, widened and multiplied where it
// is added.
RH_DEV double contribution(double F, double k8, int s) { return flip(k8, s) * F; }
RH_DEV float contribution(float F, double, int s) { return flip(F, s); }
RH_DEV double added(double w, double) { return w; }
RH_DEV double added(float w, double k8) { return k8 * (double)w; }

// A cell's neighbours across its oct's face along a dimension: the oct E there
// (or a record code), the cells X and X2 whose states the line reads, and
// whether X computes a flux through the shared face.
struct Across {
    int E, X, X2;
    bool flux_x;
};
template <int D, typename T> RH_DEV int oct_across(const LevelDev& lv, const Cell<T>& c) {
    return at(lv.nbo, (2u * D + ((c.ic0 >> D) & 1u)) * (unsigned)lv.noct + (unsigned)c.p);
}
template <int D, typename T> RH_DEV Across across(const MeshDev& m, const LevelDev& lv, const Cell<T>& c, int E) {
    Across n{E, c.cC, c.cC, false};
    if (E >= 0) {
        const int g = at(lv.grid, E), icS = c.ic0 ^ (1 << D);
        n.X = cell_id(m, g, icS);
        n.X2 = cell_id(m, g, c.ic0);
        n.flux_x = (at(lv.leaf, E) >> icS) & 1;
    } else {
        // A boundary reads the cell's own state, a missing neighbour of a
        // coarser cell the coarser cell's.
        const int4 rc = lv.rec[-1 - E];
        const int far = ((c.ic0 >> D) & 1) ? rc.z : rc.y;
        if (rc.x > 0) n.X = rc.x;
        n.X2 = far > 0 ? far : n.X;
    }
    return n;
}

// One dimension of a cell's update: its own fluxes, the contributions of X
// (into rows 5D+iv of s_x) and of S (ws).  u, w: the states of X and X2.  The
// external face comes first: what it needs of X is then dead, which keeps the
// registers below 168 (three waves per SIMD); next() issues the loads of the
// next dimension's states after the last solve (before it they cost 20 more
// registers and the kernel spills; without it, 1.83 ms against 1.77).
template <int R, typename T, bool EXACT, bool SHARED, int D, typename Next>
RH_DEV void dim_pass(const MeshDev& m, const LevelDev& lv, int slope_type, int interpol_type, const Consts<T>& k,
                     const Cell<T>& c, const Across& n, double u[5], const double w[5], double k8, bool& ok,
                     DimFlux<T>& out, T ws[5], T (*s_x)[64], int t, Next next) {
    const bool par = (c.ic0 >> D) & 1;
    const int sbit = par ? (int)0x80000000 : 0;
    const int E = n.E;
    const bool special = any_lane(!n.flux_x);  // records or refined neighbours in this wave
    int4 rc = make_int4(0, 0, 0, 0);
    if (special && E < 0) rc = lv.rec[-1 - E];
    const bool coarse = E < 0 && !(rc.w & (REC_REFINED_DEV | REC_BOUNDARY_DEV));
    ok = ok & (E != c.p);

    // The line C, S, X, X2 in the cell's frame; differences towards S.
    T q[5], x[5], dl[5], dr[5], dx[5], g[5], yX, y2;
#pragma unroll
    for (int i = 0; i < 5; ++i) q[i] = c.q[rot<D>(i)];
    q[1] = flip(q[1], sbit);
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        T s = sib<D>(q[i]);
        if (i == 1) s = -s;
        dr[i] = s - q[i];
    }
    bool tiny = c.tiny;
    fast::prim(u, g, yX, k, ok, tiny);
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        x[i] = g[rot<D>(i)];
        if (i == 1) x[i] = flip(x[i], sbit);
        dl[i] = q[i] - x[i];
    }
    fast::prim(w, g, y2, k, ok, tiny);
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        T z = g[rot<D>(i)];
        if (i == 1) z = flip(z, sbit);
        dx[i] = x[i] - z;
    }
    // A wave with a state out of range has nothing to gain from the rest.
    if (__builtin_expect(!all_lanes(ok), 0)) return;
    Slopes<T, SHARED> sc;
    fast::keep(dl, dr, k, tiny, ok);
    fast::slopes<T, SHARED, EXACT>(q, dl, dr, c.y, c.c2, slope_type, interpol_type, k, sc);

    // X's states on the shared face, from X2, X and C (a coarser X's from its
    // own neighbours; a boundary's is the cell's with the normal velocity
    // reversed, without slopes).
    T gx[5], om[5], l[5], F[5], least = q[0];
    if (__builtin_expect(special, 0)) {
        if (__builtin_expect(any_lane(coarse), 0)) {
            int far = par ? rc.y : rc.z;
            if (!coarse || far <= 0) far = n.X;
            load5(m, m.uold, far, u);
            fast::prim(u, g, y2, k, ok, tiny);
#pragma unroll
            for (int i = 0; i < 5; ++i) {
                T z = g[rot<D>(i)];
                if (i == 1) z = flip(z, sbit);
                dl[i] = coarse ? z - x[i] : dl[i];
            }
        }
    }
    {
        Slopes<T, SHARED> sx;
        fast::keep(dl, dx, k, tiny, ok);
        fast::slopes<T, SHARED, EXACT>(x, dx, dl, yX, fast::trace_c2(x[0], x[4], yX, k), slope_type, interpol_type, k, sx);
        fast::ghost_face<T, SHARED, EXACT>(x, sx, T(1.0), gx, least);
        fast::own_face<T, SHARED, EXACT>(x, sx, T(1.0), om, least);
    }
    if (__builtin_expect(special, 0)) {
        const bool bound = E < 0 && (rc.w & REC_BOUNDARY_DEV);
#pragma unroll
        for (int i = 0; i < 5; ++i) gx[i] = bound ? (i == 1 ? -q[i] : q[i]) : gx[i];
    }

    // X's own flux through the shared face.
    fast::ghost_face<T, SHARED, EXACT>(q, sc, T(-1.0), l, least);
    fast::riemann<R>(om, l, F, k, par, ok);
    T seen = T(0);
    fast::watch(F, seen);  // the cell's own fluxes: applies_to
    ok = ok & fast::finite(seen);
#pragma unroll
    for (int i = 0; i < 5; ++i) s_x[5 * D + rot<D>(i)][t] = contribution(F[i], k8, i == 1 ? sbit : 0);
    // The cell's own.
    fast::own_face<T, SHARED, EXACT>(q, sc, T(-1.0), l, least);
    fast::riemann<R>(gx, l, out.Fe, k, par, ok);
    if (__builtin_expect(special, 0)) {
        const bool none = E >= 0 ? !n.flux_x : (rc.w & REC_REFINED_DEV) != 0;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            out.Fe[i] = none ? T(0) : out.Fe[i];
            if (!n.flux_x) s_x[5 * D + i][t] = T(0);
        }
        if (coarse && c.leaf) {
            const int slot = lv.rec_slot[-1 - E] + face_slot(c.ic0, D);
#pragma unroll
            for (int i = 0; i < 5; ++i)
                lv.slot_r[(size_t)slot * 5 + rot<D>(i)] = flip(k8, i == 1 ? sbit : 0) * (double)out.Fe[i];
        }
    }

    // Towards the sibling: the ghost state it sees on the shared face travels
    // to it, its own comes here; then the fluxes change places.
    T gs[5];
    fast::ghost_face<T, SHARED, EXACT>(q, sc, T(1.0), gs, least);
#pragma unroll
    for (int i = 0; i < 5; ++i) gs[i] = sib<D>(gs[i]);
    gs[1] = -gs[1];
    fast::own_face<T, SHARED, EXACT>(q, sc, T(1.0), l, least);
    ok = ok & (least >= T(1e-10));
    fast::riemann<R>(l, gs, out.Fi, k, par, ok);
    next();
#pragma unroll
    for (int i = 0; i < 5; ++i) F[i] = sib<D>(out.Fi[i]);
    if (__builtin_expect(!all_lanes(c.lm == 0xff), 0)) {
        // A refined sibling: no flux through the face from either side.
        const bool sib_leaf = (c.lm >> (c.ic0 ^ (1 << D))) & 1;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            out.Fi[i] = sib_leaf ? out.Fi[i] : T(0);
            F[i] = sib_leaf ? F[i] : T(0);
        }
    }
#pragma unroll
    for (int i = 0; i < 5; ++i) ws[rot<D>(i)] = contribution(F[i], k8, i == 1 ? ~sbit & (int)0x80000000 : 0);
}

// Adds a dimension's own fluxes as the reference's face loop does: the minus
// face, then minus the plus face, in global order.
template <int D, typename T> RH_DEV void add_own(double fs[5], const DimFlux<T>& f, bool par) {
    if (par) {
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const double e = (double)f.Fe[i], n = (double)f.Fi[i];
            double& s = fs[rot<D>(i)];
            s = i == 1 ? (s + n) - e : (s - n) + e;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            double& s = fs[rot<D>(i)];
            s = (s + (double)f.Fe[i]) - (double)f.Fi[i];
        }
    }
}

// own_update() for finite values (applies_to() votes on the state it starts
// from; what is added to it is bounded by the range of the states).
RH_DEV void own_update_fast(double u[5], const double fs[5], double dtdx, const GasParams& gp, double y_gm1) {
#pragma unroll
    for (int iv = 0; iv < 5; ++iv) u[iv] = u[iv] + dtdx * fs[iv];
    const double d = fast::mn(fast::mx(u[0], 1e-10), 1e6);
    u[0] = d;
    const double lim = d * 10.0, y = fast::recip(d);
    double v2 = 0.0;
#pragma unroll
    for (int i = 1; i <= 3; ++i) {
        u[i] = fast::mn(fast::mx(u[i], -lim), lim);
        const double v = fast::quot(u[i], d, y);
        v2 = v2 + v * v;
    }
    const double dv2 = d * v2, least = fast::quot(d * 1e-10, gp.gm1, y_gm1);
    if (__builtin_fma(-0.5, dv2, u[4]) < least) u[4] = __builtin_fma(0.5, dv2, least);
    u[4] = fast::mn(u[4], d * 1e8);
}
// Whether the state an update starts from is finite and no larger than 2^100
// (it is uold's, already in range, except where a caller has changed unew),
// and in the mixed form what its fluxes add to it too (fast::watch).
template <typename T> RH_DEV bool applies_to(const double u[5], const double fs[5]) {
    double s = ((fabs(u[0]) + fabs(u[1])) + (fabs(u[2]) + fabs(u[3]))) + fabs(u[4]);
    if constexpr (sizeof(T) == 4) s += ((fabs(fs[0]) + fabs(fs[1])) + (fabs(fs[2]) + fabs(fs[3]))) + fabs(fs[4]);
    return s < 0x1p100;
}

// Wave speed sum of the Courant candidate, courant_cand_u() up to u_wave, for
// a level without gravity; an out-of-range state takes the general divisions.
RH_DEV double wave_speed(const double u[5], double gamma) {
    const double d = smax(u[0], 1e-10);
    const double s = (__builtin_fabs(u[1]) + __builtin_fabs(u[2])) + (__builtin_fabs(u[3]) + __builtin_fabs(u[4]));
    double v[3], v2 = 0.0, c2;
    if (all_lanes(s + d < 0x1p100)) {
        const double y = fast::recip(d);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            v[i] = fast::quot(u[1 + i], d, y);
            v2 = v2 + v[i] * v[i];
        }
        double pr = fast::mx(__builtin_fma(-0.5, d * v2, u[4]) * (gamma - 1.0), d * 1e-10);
        pr = fast::mn(pr, d * 1e2);
        c2 = fast::mx(fast::quot(gamma * pr, d, y), 1e-10);
        c2 = fast::root(c2);
    } else {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            v[i] = u[1 + i] / d;
            v2 = v2 + v[i] * v[i];
        }
        double pr = smax((u[4] - 0.5 * d * v2) * (gamma - 1.0), d * 1e-10);
        pr = smin(pr, d * 1e2);
        c2 = smax(gamma * pr / smax(d, 1e-10), 1e-20);
        c2 = ssqrt(smax(c2, 1e-10));
    }
    double w = 3 * c2;
#pragma unroll
    for (int i = 0; i < 3; ++i) w = w + sabs(v[i]);
    return w;
}

// A wave's time step, cell width and constants, held in scalar registers.  All
// its octs must be of one box; false when they are not, or when the time step
// or the cell width is out of range.
template <typename T>
RH_DEV bool constants(const StepArgs& a, int p, double& dt, double& dx, Consts<T>& k) {
    bool ok = true;
    double inv_dx = a.inv_dx;
    dx = a.dx;
    if (a.lv.obox) {
        const int mine = a.lv.obox[p], box = __builtin_amdgcn_readfirstlane(mine);
        ok = mine == box;
        dt = a.d_dt[box];
        dx = a.lv.box_len[box];
        inv_dx = a.lv.box_len[a.lv.nbox + box];
    } else {
        dt = a.d_dt ? *a.d_dt : a.dt;
        if (a.slots.in) {
            unsigned long long key = a.slots.in[(threadIdx.x & (COURANT_SLOTS - 1)) * COURANT_STRIDE];
#pragma unroll
            for (int off = COURANT_SLOTS / 2; off > 0; off >>= 1) key = min(key, (unsigned long long)__shfl_xor(key, off, 64));
            dt = key_dt(key);
        }
        if (blockIdx.x == 0) {
            if (a.slots.in && threadIdx.x == 0) *a.slots.dt_out = dt;
            if (a.slots.clear && threadIdx.x < COURANT_SLOTS)
                a.slots.clear[threadIdx.x * COURANT_STRIDE] = dt_key(a.slots.dt_init);
        }
    }
    dt = uniform(dt);
    dx = uniform(dx);
    k.gamma = (T)a.gp.gamma;
    k.gm1 = (T)a.gp.gm1;
    k.smalle = (T)a.gp.smalle;
    k.smallp = (T)a.gp.smallp;
    k.dx = uniform((T)dx);
    k.hdx = uniform(T(0.5) * k.dx);
    k.hdt = uniform(T(0.5) * (T)dt);
    const double dtdx = uniform(dt / dx);
    if constexpr (sizeof(T) == 8) {
        k.y_gm1 = uniform(fast::recip(a.gp.gm1));
        k.inv = uniform(inv_dx != 0.0 ? inv_dx : fast::recip(dx));
        return ok && dt >= 0x1p-100 && dtdx <= 0x1p20 && dx >= 0x1p-60 && dx <= 0x1p60;
    } else {
        k.y_gm1 = uniform((T)(1.0 / a.gp.gm1));
        k.inv = uniform(fast::recip(k.dx));
        return ok && dt >= 0x1p-100 && dtdx <= 0x1p20 && dx >= 0x1p-40 && dx <= 0x1p40;
    }
}

// The ordered accumulation of a cell (processing order: position in the list,
// then cell, then face).  An oct's neighbours across its faces come wholly
// before or after it, so the order is: the X contributions of octs before
// it by position, the siblings with a lower cell index (highest dimension
// first), the cell itself, the siblings with a higher index, the X
// contributions of octs after it.  wx: this lane's contributions in LDS, rows
// 5d+iv from X of dimension d, rows 15+5d+iv from S of dimensions 0 and 1; ws2
// those of dimension 2; key: position of the oct across * 4 + dimension (a
// record's is negative and its contribution 0).
template <typename T>
RH_DEV void apply(double u[5], const double fs[5], const T ws2[5], const T (*wx)[64], const int key[3], int p, int ic0,
                  int t, double dtdx, const GasParams& gp, double y_gm1) {
    const double k8 = dtdx * 0.125;
    const int lo = min(min(key[0], key[1]), key[2]), hi = max(max(key[0], key[1]), key[2]);
    const int k3[3] = {lo, key[0] ^ key[1] ^ key[2] ^ lo ^ hi, hi};
    double x[3][5], ws[3][5];
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int iv = 0; iv < 5; ++iv) {
            x[j][iv] = added(wx[(k3[j] & 3) * 5 + iv][t], k8);
            ws[j][iv] = added(j < 2 ? wx[15 + 5 * j + iv][t] : ws2[iv], k8);
        }
#pragma unroll
    for (int j = 0; j < 3; ++j)
        if (k3[j] < 4 * p)
#pragma unroll
            for (int iv = 0; iv < 5; ++iv) u[iv] = u[iv] + x[j][iv];
#pragma unroll
    for (int d = 2; d >= 0; --d)
        if ((ic0 >> d) & 1)
#pragma unroll
            for (int iv = 0; iv < 5; ++iv) u[iv] = u[iv] + ws[d][iv];
    own_update_fast(u, fs, dtdx, gp, y_gm1);
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if (!((ic0 >> d) & 1))
#pragma unroll
            for (int iv = 0; iv < 5; ++iv) u[iv] = u[iv] + ws[d][iv];
#pragma unroll
    for (int j = 0; j < 3; ++j)
        if (k3[j] > 4 * p)
#pragma unroll
            for (int iv = 0; iv < 5; ++iv) u[iv] = u[iv] + x[j][iv];
}

// End of a cell's update: the new state into unew and, in the fused step, the
// next step's Courant candidate (the state set_uold would copy).  Without
// gravity a candidate falls monotonically with the cell's wave speed sum, each
// operation rounding monotonically, so the wave takes the largest sum and
// does the divisions once.
RH_DEV void finish(const MeshDev& m, const LevelDev& lv, const GasParams& gp, const double u[5], bool leaf, int cC, int p,
                   int pfirst, int t, double dx, const StepArgs& a) {
    double* const cpart = a.cpart;
    unsigned long long *const ckeys = a.ckeys, *const slots = a.slots.out;
    const double courant_factor = a.courant_factor;
    if (leaf) store5(m, m.unew, cC, u);
    if (!cpart && !ckeys && !slots) return;
    const double s1 = ssqrt(1.0 + 2.0 * courant_factor * 1e-4) - 1.0;
    const bool one_box = !ckeys || lv.obox[pfirst] == lv.obox[min(pfirst + 8, lv.noct) - 1];
    double cand = __builtin_inf();
    if (one_box && !m.f && s1 > 0.0) {
        double w = leaf ? wave_speed(u, gp.gamma) : 0.0;
        w = w > 0.0 ? w : 0.0;  // a NaN is skipped
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) w = fast::mx(w, __shfl_xor(w, off, 64));
        if (w > 0.0) cand = (dx / w) * s1 / 1e-4;
    } else {
        // dx is the width of the wave's first box; its others have their own.
        if (leaf) cand = courant_cand_u(m, u, cC, one_box ? dx : lv.box_len[lv.obox[p]], gp.gamma, courant_factor);
        if (one_box) cand = wave_min(cand);
    }
    if (cpart) {
        if (t == 0) cpart[blockIdx.x] = cand;
    } else if (slots) {
        if (t == 0) atomicMin(&slots[(blockIdx.x & (COURANT_SLOTS - 1)) * COURANT_STRIDE], dt_key(cand));
    } else if (one_box) {
        if (t == 0) atomicMin(&ckeys[lv.obox[pfirst]], dt_key(cand));
    } else if (cand != __builtin_inf()) {
        atomicMin(&ckeys[lv.obox[p]], dt_key(cand));
    }
}

// This wave's cells: 8 octs of the list, lanes past its end on the last oct.
// Their states are loaded before the time step is taken from the slots, so
// that the two waits overlap.
template <typename T>
RH_DEV void find_cell(const MeshDev& m, const LevelDev& lv, int praw, int t, Cell<T>& c, double u[5]) {
    c.ic0 = t & 7;
    c.p = min(praw, lv.noct - 1);
    c.lm = at(lv.leaf, c.p);
    c.leaf = praw < lv.noct && ((c.lm >> c.ic0) & 1);
    c.cC = cell_id(m, at(lv.grid, c.p), c.ic0);
    load5(m, m.uold, c.cC, u);
}
template <typename T> RH_DEV void take_cell(const double u[5], const Consts<T>& k, Cell<T>& c, bool& ok) {
    c.tiny = false;
    fast::prim(u, c.q, c.y, k, ok, c.tiny);
    c.c2 = fast::trace_c2(c.q[0], c.q[4], c.y, k);
}

template <int R, bool MIXED, bool EXACT, bool SHARED>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(OCT_WAVES, 8))) void k_step_oct(StepArgs a) {
    using T = typename std::conditional<MIXED, float, double>::type;
    __shared__ T s_x[25][64];
    const MeshDev& m = a.m;
    const LevelDev& lv = a.lv;
    const int t = threadIdx.x;
    const int praw = xcd_block(blockIdx.x, gridDim.x) * 8 + (t >> 3);
    double dt, dx;
    Consts<T> k;
    Cell<T> c;
    double u[5];
    find_cell(m, lv, praw, t, c, u);
    bool ok = constants(a, c.p, dt, dx, k);
    take_cell(u, k, c, ok);
    const double dtdx = uniform(dt / dx), k8 = uniform(dtdx * 0.125);
    if (__builtin_expect(all_lanes(ok), 1)) {
        const int E0 = oct_across<0>(lv, c), E1 = oct_across<1>(lv, c), E2 = oct_across<2>(lv, c);
        const Across n[3] = {across<0>(m, lv, c, E0), across<1>(m, lv, c, E1), across<2>(m, lv, c, E2)};
        double fs[5], w[5], un[5], wn[5];
        T ws[5];
        load5(m, m.uold, n[0].X, u);
        load5(m, m.uold, n[0].X2, w);
        auto pass = [&](auto dc) {
            constexpr int D = decltype(dc)::value;
            DimFlux<T> f;
            auto next = [&]() {
                if constexpr (D < 2) {
                    load5(m, m.uold, n[D + 1].X, un);
                    load5(m, m.uold, n[D + 1].X2, wn);
                } else {
                    load5(m, a.pre, c.cC, un);
                }
            };
            dim_pass<R, T, EXACT, SHARED, D>(m, lv, a.gp.slope_type, a.gp.interpol_type, k, c, n[D], u, w, k8, ok, f, ws,
                                             s_x, t, next);
            copy5(un, u);
            copy5(wn, w);
            const bool par = (c.ic0 >> D) & 1;
            if constexpr (D < 2)
#pragma unroll
                for (int iv = 0; iv < 5; ++iv) s_x[15 + 5 * D + iv][t] = ws[iv];
            if constexpr (D == 0) {
                // From 0 the order of the two faces does not matter.
#pragma unroll
                for (int i = 0; i < 5; ++i) {
                    const double v = (double)f.Fe[i] - (double)f.Fi[i];
                    fs[rot<D>(i)] = i == 1 ? flip(v, par ? (int)0x80000000 : 0) : v;
                }
            } else {
                add_own<D>(fs, f, par);
            }
        };
        pass(std::integral_constant<int, 0>{});
        if (__builtin_expect(all_lanes(ok), 1)) pass(std::integral_constant<int, 1>{});
        if (__builtin_expect(all_lanes(ok), 1)) pass(std::integral_constant<int, 2>{});
        const int key[3] = {n[0].E * 4, n[1].E * 4 + 1, n[2].E * 4 + 2};
        ok = ok & applies_to<T>(u, fs);
        if (__builtin_expect(all_lanes(ok), 1))
            apply(u, fs, ws, s_x, key, c.p, c.ic0, t, dtdx, a.gp, uniform(fast::recip(a.gp.gm1)));
    }
    if (__builtin_expect(!all_lanes(ok), 0)) {
        general_wave<R, MIXED, EXACT, SHARED>(launch_args(), shared_rows(s_x), praw, t, dt, dx, u);
    }
    finish(m, lv, a.gp, u, c.leaf, c.cC, c.p, praw - (t >> 3), t, dx, a);
}

template <int R, bool MIXED, bool EXACT, bool SHARED>
__global__ __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(MIXED ? DIMS_WAVES_F : DIMS_WAVES, 8))) void k_step_dims(StepArgs a) {
    using T = typename std::conditional<MIXED, float, double>::type;
    // Contributions of X and S per dimension, own fluxes for the first
    // wave, the oct across per dimension, range votes.
    __shared__ T s_x[30][64];
    __shared__ T s_o[30][64];
    __shared__ int s_key[2][64];
    __shared__ int s_bad[3];
    const MeshDev& m = a.m;
    const LevelDev& lv = a.lv;
    const int t = threadIdx.x & 63;
    const int d = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int praw = xcd_block(blockIdx.x, gridDim.x) * 8 + (t >> 3);
    double dt, dx;
    Consts<T> k;
    Cell<T> c;
    double u[5];
    find_cell(m, lv, praw, t, c, u);
    bool ok = constants(a, c.p, dt, dx, k);
    take_cell(u, k, c, ok);
    const double dtdx = uniform(dt / dx), k8 = uniform(dtdx * 0.125);
    double fs[5];
    int key0 = 0;
    // Rows of s_o: own fluxes of dimensions 1 and 2, then of dimension 0 where
    // they come from the general form.
    constexpr int OWN[3] = {20, 0, 10};
    auto own = [&](auto dc, DimFlux<T>& f) {
        constexpr int D = decltype(dc)::value;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            f.Fe[i] = s_o[OWN[D] + i][t];
            f.Fi[i] = s_o[OWN[D] + 5 + i][t];
        }
    };
    auto pass = [&](auto dc) {
        constexpr int D = decltype(dc)::value;
        DimFlux<T> f;
        if (__builtin_expect(all_lanes(ok), 1)) {
            T ws[5];
            double x[5], w[5];
            const Across n = across<D>(m, lv, c, oct_across<D>(lv, c));
            load5(m, m.uold, n.X, x);
            load5(m, m.uold, n.X2, w);
            dim_pass<R, T, EXACT, SHARED, D>(m, lv, a.gp.slope_type, a.gp.interpol_type, k, c, n, x, w, k8, ok, f, ws,
                                             s_x, t, [] {});
            const int kd = n.E * 4 + D;
            if constexpr (D == 0) key0 = kd;
            else s_key[D - 1][t] = kd;
#pragma unroll
            for (int i = 0; i < 5; ++i) {
                s_x[15 + 5 * D + i][t] = ws[i];
                if constexpr (D > 0) {
                    s_o[OWN[D] + i][t] = f.Fe[i];
                    s_o[OWN[D] + 5 + i][t] = f.Fi[i];
                }
            }
        }
        const bool bad = !all_lanes(ok);  // every lane votes
        if (t == 0) s_bad[D] = bad;
        if (__builtin_expect(bad, 0)) {
            general_one_dim<R, MIXED, EXACT, SHARED>(launch_args(), shared_rows(s_x), shared_rows(s_o + OWN[D]), D, praw,
                                                     t, dt, dx);
            if constexpr (D == 0) own(dc, f);
        }
        if constexpr (D == 0) {
            const bool par = c.ic0 & 1;
#pragma unroll
            for (int i = 0; i < 5; ++i) {
                const double v = (double)f.Fe[i] - (double)f.Fi[i];
                fs[i] = i == 1 ? flip(v, par ? (int)0x80000000 : 0) : v;
            }
        }
    };
    if (d == 0) pass(std::integral_constant<int, 0>{});
    else if (d == 1) pass(std::integral_constant<int, 1>{});
    else pass(std::integral_constant<int, 2>{});
    __syncthreads();
    if (d != 0) return;
    auto other = [&](auto dc) {
        constexpr int D = decltype(dc)::value;
        DimFlux<T> f;
        own(dc, f);
        add_own<D>(fs, f, (c.ic0 >> D) & 1);
    };
    other(std::integral_constant<int, 1>{});
    other(std::integral_constant<int, 2>{});
    load5(m, a.pre, c.cC, u);
    ok = applies_to<T>(u, fs) && !(s_bad[0] | s_bad[1] | s_bad[2]);
    if (__builtin_expect(all_lanes(ok), 1)) {
        T ws2[5];
#pragma unroll
        for (int iv = 0; iv < 5; ++iv) ws2[iv] = s_x[25 + iv][t];
        const int key[3] = {key0, s_key[0][t], s_key[1][t]};
        apply(u, fs, ws2, s_x, key, c.p, c.ic0, t, dtdx, a.gp, uniform(fast::recip(a.gp.gm1)));
    } else {
        State5 f;
        copy5(fs, f.u);
        const State5 s = general_sum<MIXED>(launch_args(), shared_rows(s_x), f, praw, t, dt, dx);
        copy5(s.u, u);
    }
    finish(m, lv, a.gp, u, c.leaf, c.cC, c.p, praw - (t >> 3), t, dx, a);
}

template <int R, bool MIXED, bool EXACT, bool SHARED>
void launch_as(bool dims, const StepArgs& a, hipStream_t stream) {
    const dim3 grid((a.lv.noct + 7) / 8);
    if (dims) hipLaunchKernelGGL((k_step_dims<R, MIXED, EXACT, SHARED>), grid, dim3(192), 0, stream, a);
    else hipLaunchKernelGGL((k_step_oct<R, MIXED, EXACT, SHARED>), grid, dim3(64), 0, stream, a);
}
template <int R, bool MIXED> void launch_prec(bool dims, const StepArgs& a, hipStream_t stream) {
    const bool shared = a.gp.slope_type == 1 && a.gp.interpol_type == 1;
    if (a.inv_dx != 0.0) {
        if (shared) launch_as<R, MIXED, true, true>(dims, a, stream);
        else launch_as<R, MIXED, true, false>(dims, a, stream);
    } else {
        if (shared) launch_as<R, MIXED, false, true>(dims, a, stream);
        else launch_as<R, MIXED, false, false>(dims, a, stream);
    }
}

}  // namespace

template <int R> void launch_step(bool mixed, bool dims, const StepArgs& a, hipStream_t stream) {
    if (mixed) launch_prec<R, true>(dims, a, stream);
    else launch_prec<R, false>(dims, a, stream);
}
template void launch_step<RH_RIEMANN>(bool, bool, const StepArgs&, hipStream_t);

}  // namespace rh
