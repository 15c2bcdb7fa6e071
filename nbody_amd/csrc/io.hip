// io.hip -- the particle state between the sorted device arrays and the
// caller's input-order arrays.  The permutation and the xyz interleaving run
// on the device, so that what crosses the bus is already in the caller's
// layout (the host loops over eight sorted arrays took ~20 of the 29 ms that
// a 1M-particle state took to read).
#include "common.h"
#include "launch.h"

namespace nbh {

// sorted state -> input order, xyz triples; any output may be null.  Scattered
// by id: a particle's three coordinates go out as one 24-byte run.
__global__ __launch_bounds__(256) void pack_state_kernel(State S, uint32_t n, double* __restrict__ pos,
                                                         double* __restrict__ vel, double* __restrict__ mass,
                                                         double* __restrict__ charge) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const size_t j = S.id[i];
    if (pos) {
        const double x = S.x[i], y = S.y[i], z = S.z[i];
        pos[3 * j] = x; pos[3 * j + 1] = y; pos[3 * j + 2] = z;
    }
    if (vel) {
        const double x = S.vx[i], y = S.vy[i], z = S.vz[i];
        vel[3 * j] = x; vel[3 * j + 1] = y; vel[3 * j + 2] = z;
    }
    if (mass) mass[j] = S.mass[i];
    if (charge) charge[j] = S.charge[i];
}

__global__ __launch_bounds__(256) void pack_forces_kernel(State S, uint32_t n, float* __restrict__ acc,
                                                          float* __restrict__ pot) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const size_t j = S.id[i];
    if (acc) {
        const float x = S.ax[i], y = S.ay[i], z = S.az[i];
        acc[3 * j] = x; acc[3 * j + 1] = y; acc[3 * j + 2] = z;
    }
    if (pot) pot[j] = S.pot[i];
}

// g = [gx | gy | gz | gm] in sorted order -> input order
__global__ __launch_bounds__(256) void pack_gradient_kernel(const double* __restrict__ g,
                                                            const uint32_t* __restrict__ id, uint32_t n,
                                                            double* __restrict__ gx, double* __restrict__ gm) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const size_t j = id[i];
    const double x = g[i], y = g[(size_t)n + i], z = g[2 * (size_t)n + i];
    gx[3 * j] = x; gx[3 * j + 1] = y; gx[3 * j + 2] = z;
    gm[j] = g[3 * (size_t)n + i];
}

// new positions and velocities (input order, xyz triples) into dst, which
// becomes input-ordered; masses and charges come from src, the current state
// in its sorted order.  *bad is set if a value is not finite.
__global__ __launch_bounds__(256) void unpack_state_kernel(State src, State dst, uint32_t n,
                                                           const double* __restrict__ pos,
                                                           const double* __restrict__ vel, uint32_t* bad) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t j = src.id[i];
    dst.mass[j] = src.mass[i];
    dst.charge[j] = src.charge[i];
    const double v[6] = {pos[3 * (size_t)i], pos[3 * (size_t)i + 1], pos[3 * (size_t)i + 2],
                         vel[3 * (size_t)i], vel[3 * (size_t)i + 1], vel[3 * (size_t)i + 2]};
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 6; ++k) ok &= isfinite(v[k]);
    if (!ok) *bad = 1u;
    dst.x[i] = v[0]; dst.y[i] = v[1]; dst.z[i] = v[2];
    dst.vx[i] = v[3]; dst.vy[i] = v[4]; dst.vz[i] = v[5];
    dst.id[i] = i;
}

// a new handle's state from the caller's arrays
__global__ __launch_bounds__(256) void init_state_kernel(State dst, uint32_t n, const double* __restrict__ pos,
                                                         const double* __restrict__ vel,
                                                         const double* __restrict__ mass,
                                                         const double* __restrict__ charge) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const size_t o = 3 * (size_t)i;
    dst.x[i] = pos[o]; dst.y[i] = pos[o + 1]; dst.z[i] = pos[o + 2];
    dst.vx[i] = vel[o]; dst.vy[i] = vel[o + 1]; dst.vz[i] = vel[o + 2];
    dst.mass[i] = mass[i];
    dst.charge[i] = charge[i];
    dst.ax[i] = dst.ay[i] = dst.az[i] = dst.pot[i] = 0.f;
    dst.id[i] = i;
}
void launch_init_state(const State& dst, uint32_t n, const double* pos, const double* vel, const double* mass,
                       const double* charge, hipStream_t st) {
    hipLaunchKernelGGL(init_state_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, st, dst, n, pos, vel, mass, charge);
}
void launch_pack_state(const State& S, uint32_t n, double* pos, double* vel, double* mass, double* charge,
                       hipStream_t st) {
    hipLaunchKernelGGL(pack_state_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, st, S, n, pos, vel, mass, charge);
}
void launch_pack_forces(const State& S, uint32_t n, float* acc, float* pot, hipStream_t st) {
    hipLaunchKernelGGL(pack_forces_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, st, S, n, acc, pot);
}
void launch_pack_gradient(const double* g, const uint32_t* id, uint32_t n, double* gx, double* gm, hipStream_t st) {
    hipLaunchKernelGGL(pack_gradient_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, st, g, id, n, gx, gm);
}
void launch_unpack_state(const State& src, const State& dst, uint32_t n, const double* pos, const double* vel,
                         uint32_t* bad, hipStream_t st) {
    hipLaunchKernelGGL(unpack_state_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, st, src, dst, n, pos, vel, bad);
}

}  // namespace nbh
