// courant_fine of one cell and the wave reductions of its partial results, and
// the reflux writes: shared by the brick kernels and the separate passes.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rh_godunov.h"
#include "rh_physics64.h"

namespace rh {

// Constants of courant_fine / cmpdt on one level.
struct CourantK {
    double dx, vol, gamma, smallr, smallc, courant_factor, smallp, gsum_dx;
    int ndim;
};

// The dt of a cell whose summed signal speed is ctot = sum_d(|v_d| + c)
// (cmpdt, hydro/godunov_utils.f90:228-337), or the level's initial bound
// dx/smallc where ctot is 0 (no leaf cell).  dt falls with rising ctot:
// ctot (1 + sqrt(1 + 2C max(g dx/ctot^2, 1e-4))) is the larger of
// ctot + sqrt(ctot^2 + 2C g dx) and ctot times a constant, so the smallest dt
// of a level is that of its largest ctot, and the square root and the
// division are taken once per reduction instead of once per cell.
__device__ __forceinline__ double signal_dt(double ctot, const CourantK &c)
{
#pragma clang fp contract(off)
    if (!(ctot > 0.0)) return c.dx / c.smallc;
    double grav = c.gsum_dx / (ctot * ctot);
    grav = grav > 0.0001 ? grav : 0.0001;
    const double gf = 1.0 + __builtin_sqrt(1.0 + 2.0 * c.courant_factor * grav);
    const double dtmax = c.courant_factor * c.dx / c.smallc;
    const double dtcell = 2.0 * c.courant_factor * c.dx / (ctot * gf);
    return dtmax < dtcell ? dtmax : dtcell;
}
__device__ __forceinline__ double wave_sum(double x)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}
__device__ __forceinline__ double wave_min(double x)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        double y = __shfl_xor(x, o, 64);
        x = y < x ? y : x;
    }
    return x;
}
__device__ __forceinline__ double wave_max(double x)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        double y = __shfl_xor(x, o, 64);
        x = y > x ? y : x;
    }
    return x;
}
// The same for a wave of which only lanes [0, nvalid) exist (the last wave of
// a workgroup whose size is not a multiple of 64): partners at or beyond
// nvalid are skipped.  Lane 0's partners in the round of offset o are lanes
// o..2o-1, whose partial results only gather lanes above them, so lane 0
// ends with the reduction over exactly the existing lanes.
__device__ __forceinline__ double wave_sum_n(double x, int nvalid)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double y = __shfl_xor(x, o, 64);
        if ((lane ^ o) < nvalid) x += y;
    }
    return x;
}
__device__ __forceinline__ double wave_min_n(double x, int nvalid)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double y = __shfl_xor(x, o, 64);
        if ((lane ^ o) < nvalid && y < x) x = y;
    }
    return x;
}
__device__ __forceinline__ double wave_max_n(double x, int nvalid)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double y = __shfl_xor(x, o, 64);
        if ((lane ^ o) < nvalid && y > x) x = y;
    }
    return x;
}

__device__ __forceinline__ CourantK make_courant_k(double dx, int ndim, double gamma, double smallr, double smallc2,
                                                   double courant_factor, const double g[3])
{
    CourantK c;
    c.dx = dx;
    c.vol = ndim == 1 ? dx : dx * dx * dx;
    c.gamma = gamma;
    c.smallr = smallr;
    c.smallc = __builtin_sqrt(smallc2);
    c.courant_factor = courant_factor;
    c.smallp = smallc2 / gamma;
    double gs = 0.0;
    for (int d = 0; d < ndim; d++) gs = gs + __builtin_fabs(g[d]);
    c.gsum_dx = gs * dx;
    c.ndim = ndim;
    return c;
}

// One leaf cell of courant_fine (hydro/courant_fine.f90:120-160): its share of
// the conservation sums, and its summed signal speed ctot (cmpdt), in FP64.
// ir = 1/r replaces the reference's three divisions by r, and with no magnetic
// field its c_f = sqrt(c2 + sqrt(c2^2)) with c2 = a^2/2 is sqrt(a^2).  About 50
// issue slots; with the dt and the sums formed per term it took 90.
// Contraction is spelled out, so that every kernel gets the same bits.
template <int ND>
__device__ __forceinline__ double courant_cell(const double u[5], const CourantK &c, double vol, double &mass,
                                               double &ekin, double &eint)
{
#pragma clang fp contract(off)
    const double r = tmax(u[0], c.smallr);
    const double ir = rcp_nr(r), hr = 0.5 * r;
    const double v[3] = {u[1] * ir, u[2] * ir, u[3] * ir};
    double e = u[4];
#pragma unroll
    for (int d = 0; d < 3; d++) e = __builtin_fma(-hr, v[d] * v[d], e);
    mass = __builtin_fma(u[0], vol, mass);
    ekin = __builtin_fma(u[4], vol, ekin);
    eint = __builtin_fma(e, vol, eint);
    const double pe = (c.gamma - 1.0) * e, pf = r * c.smallp;
    const double a2 = c.gamma * tmax(pe, pf) * ir;
    // a2 >= gamma smallp = smallc^2: the square root of the Riemann solvers
    // (floored where smallc^2 < 2^-900)
    const double cf = sqrt_pos(tmax(a2, 0x1p-900));
    double ctot = 0.0;
#pragma unroll
    for (int d = 0; d < ND; d++) ctot = ctot + __builtin_fabs(v[d]) + cf;
    return ctot;
}

// courant_fine of one cell for the mixed-precision kernel: the conservation
// sums and the pressure recovery p=(gamma-1)(E-rho v^2/2) in FP64, the signal
// speed and the cell's dt in FP32 (cmpdt's c_f = sqrt(c2+sqrt(c2^2)) with
// c2 = a^2/2 and no magnetic field is a), the dt rounded to FP64 for the
// min-reduction.
__device__ __forceinline__ void courant_cell_mixed(const double u[5], const CourantK &c, double &mass, double &ekin,
                                                   double &eint, double &dtmin)
{
    mass = mass + u[0] * c.vol;
    ekin = ekin + u[4] * c.vol;
    const double rr = u[0] > c.smallr ? u[0] : c.smallr;
    const double ir = rcp_nr(rr);
    const double ke = 0.5 * (u[1] * u[1] + u[2] * u[2] + u[3] * u[3]) * ir;
    eint = eint + (u[4] - ke) * c.vol;
    const double pe = (c.gamma - 1.0) * (u[4] - ke), pf = rr * c.smallp;
    const double p = pe > pf ? pe : pf;
    const float irf = (float)ir;
    const float cf = __builtin_amdgcn_sqrtf((float)(c.gamma * p) * irf);
    const float ctot = (__builtin_fabsf((float)u[1] * irf) + cf) + (__builtin_fabsf((float)u[2] * irf) + cf) +
                       (__builtin_fabsf((float)u[3] * irf) + cf);
    const float cfl = (float)c.courant_factor;
    float grav = (float)c.gsum_dx * __builtin_amdgcn_rcpf(ctot * ctot);
    grav = grav > 0.0001f ? grav : 0.0001f;
    const double dtmax = c.courant_factor * c.dx / c.smallc;
    const float dtcell = 2.0f * cfl * (float)c.dx *
                         __builtin_amdgcn_rcpf(ctot * (1.0f + __builtin_amdgcn_sqrtf(1.0f + 2.0f * cfl * grav)));
    const double d = dtmax < (double)dtcell ? dtmax : (double)dtcell;
    dtmin = d < dtmin ? d : dtmin;
}

template <typename T>
__device__ __forceinline__ HydroK<T> make_k(const double dt, double dx, double gamma, double smallr, double smallc2,
                                            double courant_factor, double smax_cap, int use_smax, int slope,
                                            int riemann)
{
    HydroK<T> k;
    k.gamma = T(gamma);
    k.smallr = T(smallr);
    k.smallc2 = T(smallc2 > 0x1p-900 ? smallc2 : 0x1p-900);
    k.smallp_trace = T(smallr * smallc2);
    k.smallp_riem = T(smallc2 / gamma);
    k.entho = T(1.0 / (gamma - 1.0));
    k.dtdx = T(dt / dx);
    k.smax_cap = T(use_smax ? smax_cap : courant_factor * dx / dt);
    k.slope_type = slope;
    k.riemann = riemann;
    return k;
}

// Coarse-fine refluxing, godfine1 (hydro/godunov_fine.f90:894-1052): a face
// between a cell of the level and an interpolated ghost cell sends -flux/2^ndim
// (ghost on the low side) or +flux/2^ndim (ghost on the high side) to the
// ghost's parent cell.  Three ways:
// - racc null: FP64 atomics into the parent cell of unew;
// - racc, rdet 0: FP64 atomics into the ghost's accumulator racc[5 g];
// either way the order of the contributions to one parent cell is not fixed
// (last-bit differences from run to run and from the serial reference);
// - racc, rdet 1 (deterministic mode): a plain store into the face's own slot
//   racc[5 (kReluxSlots g + slot)], slot = 4 side + sub (side: the ghost oct's
//   face, -x +x -y +y -z +z; sub: which of its 2^(ndim-1) cells), one writer
//   per slot; k_reflux_fold then adds the slots in slot order.
constexpr int kRefluxSlots = kRefluxSlotsPerGhost;
__device__ __forceinline__ void reflux_add(double *unew, const int32_t *ghost_parent, int ngridmax, int vghost,
                                           double sign, const double F[5], int ttd, double *racc = nullptr,
                                           int rdet = 0, int slot = 0, bool accumulate = false)
{
    const int gi = vghost - ngridmax - 1;
    if (racc) {
        const double w = 1.0 / (double)ttd;
        if (rdet) {
            // accumulate: the diffusion pass adds to the slot the Godunov launch wrote
            double *q = racc + 5 * ((size_t)gi * kRefluxSlots + slot);
#pragma unroll
            for (int n = 0; n < 5; n++) q[n] = accumulate ? q[n] + sign * (F[n] * w) : sign * (F[n] * w);
            return;
        }
#pragma unroll
        for (int n = 0; n < 5; n++) atomicAdd(racc + 5 * (size_t)gi + n, sign * (F[n] * w));
        return;
    }
    const int igrid = ghost_parent[2 * gi], icell = ghost_parent[2 * gi + 1];
    if (igrid <= 0) return;  // parent missing: rh_build_nbor reported it
    const double w = 1.0 / (double)ttd;
    double *p = unew + (size_t)(igrid - 1) * 5 * ttd + (icell - 1);
#pragma unroll
    for (int n = 0; n < 5; n++) atomicAdd(p + n * ttd, sign * (F[n] * w));
}

// The summed refluxes q (already weighted by 1/2^ndim, with their signs) of
// one ghost oct: into its accumulator, or into its parent cell of unew.
__device__ __forceinline__ void reflux_flush(double *unew, const int32_t *ghost_parent, int ngridmax, int vghost,
                                             const double q[5], int ttd, double *racc)
{
    const int gi = vghost - ngridmax - 1;
    if (racc) {
#pragma unroll
        for (int n = 0; n < 5; n++) atomicAdd(racc + 5 * (size_t)gi + n, q[n]);
        return;
    }
    const int igrid = ghost_parent[2 * gi], icell = ghost_parent[2 * gi + 1];
    if (igrid <= 0) return;
    double *p = unew + (size_t)(igrid - 1) * 5 * ttd + (icell - 1);
#pragma unroll
    for (int n = 0; n < 5; n++) atomicAdd(p + n * ttd, q[n]);
}

}  // namespace rh
