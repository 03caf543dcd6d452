// rh_godunov.h -- launch of the Godunov update for ordinary states
// (rh_godunov.hip), one Riemann solver per translation unit.
#pragma once
#include "rh_kernels.h"

namespace rh {

// Arguments of one update launch.  dx, inv_dx: the level's cell width and its
// exact reciprocal or 0 (an ensemble reads both per box; inv_dx != 0 when
// every box has one); pre: the buffer the cells' state before the update is
// read from; cpart / ckeys / slots: where the next step's Courant candidates
// go, or null (launch_godunov's FusedCourant).
struct StepArgs {
    MeshDev m;
    LevelDev lv;
    GasParams gp;
    const double* d_dt;  // null: the time step is the slots' or dt (a single mesh)
    double dt;
    double dx, inv_dx;
    const double* pre;
    double* cpart;
    unsigned long long* ckeys;
    double courant_factor;
    CourantSlots slots;
};

// Whether the update runs in these kernels for a configuration: their slope
// limiters are those symmetric under a reversed axis (types 4 and 5, whose two
// sides are weighted by the sign of the velocity, are not), their range
// analysis holds for gamma - 1 in [2^-10, 64], and they address a state
// component, and the six neighbour tables of a level, by 32-bit byte offsets.
inline bool step_kernels_take(const GasParams& gp, int ncell) {
    return gp.slope_type != 4 && gp.slope_type != 5 && gp.gm1 >= 0x1p-10 && gp.gm1 <= 64.0 && ncell <= (1 << 29);
}

// dims: three waves per 8 octs, one per dimension; else one wave.
template <int R> void launch_step(bool mixed, bool dims, const StepArgs& a, hipStream_t stream);
extern template void launch_step<0>(bool, bool, const StepArgs&, hipStream_t);
extern template void launch_step<1>(bool, bool, const StepArgs&, hipStream_t);
extern template void launch_step<2>(bool, bool, const StepArgs&, hipStream_t);
extern template void launch_step<4>(bool, bool, const StepArgs&, hipStream_t);

}  // namespace rh
