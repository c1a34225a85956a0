// The passes beside the 3D brick kernels: the 1D Godunov step, the Courant
// condition and its reductions, ghost octs, restriction, the coarse-fine reflux
// fold, artificial diffusion.
#include "rh_courant.h"
#include "rh_gather.h"
#include "rh_godunov.h"

namespace rh {

// ---------------------------------------------------------------------------
// 1D: one thread per cell; stencil of 5 cells from the 3-slot neighbour table.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) k_godunov1d(const God1Args a)
{
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= 2 * a.noct) return;
    const int o = a.head + (gid >> 1);  // 1-based oct
    const int i2 = gid & 1;
    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    const HydroK<T> k = make_k<T>(dt, a.dx, a.gamma, a.smallr, a.smallc2, a.courant_factor, a.smax_cap, a.use_smax,
                                  a.slope < 2 ? a.slope : 2, a.riemann);
    const double smalle = a.smallc2 / a.gamma / (a.gamma - 1.0);
    const double gdt[3] = {a.g * (dt * 0.5), 0.0, 0.0};
    const int32_t *nb = a.nbor + (size_t)(o - a.head) * 3;
    const int boxmin[3] = {a.boxmin, 0, 0}, boxmax[3] = {a.boxmax, 1, 1};
    const int btype[3][2] = {{a.btype[0], a.btype[1]}, {2, 2}, {2, 2}};
    T q[5][5];
    uint8_t rf[5];
    for (int d = -2; d <= 2; d++) {
        const int p = i2 + d;
        const int slot = (p + 2) >> 1;
        const int v = nb[slot];
        // key of that oct relative to the domain: self oct key is unknown here,
        // the slot tells the side (slot 0 = low, 2 = high)
        int okey[3] = {slot == 0 ? a.boxmin - 1 : (slot == 2 ? a.boxmax : a.boxmin), 0, 0};
        int c[3] = {p & 1, 0, 0};
        double u[5], qq[5];
        gather_cell(a.uold, a.refined, v, okey, 1, boxmin, boxmax, btype, c, u, rf[d + 2]);
        prim_from_cons(u, qq, a.smallr, smalle, a.gamma, gdt);
#pragma unroll
        for (int n = 0; n < 5; n++) q[d + 2][n] = T(qq[n]);
    }
    T qp[3][5], qm[3][5];
#pragma unroll
    for (int c = 1; c <= 3; c++) {
        T dq[5];
#pragma unroll
        for (int n = 0; n < 5; n++) dq[n] = k.slope_type ? slope_half(k.slope_type, q[c - 1][n], q[c][n], q[c + 1][n]) : T(0);
        const T inv_r = trcp(q[c][0]);
        if (k.slope_type > 0)
            dq[1] = vel_bound_half(dq[1], q[c - 1][0], q[c - 1][1], inv_r, q[c][1], q[c + 1][0], q[c + 1][1]);
        trace1(q[c], dq, qp[c - 1], qm[c - 1], k, inv_r);
    }
    T fl[5], fr[5];
    face_flux(0, qm[0], qp[1], fl, k);
    face_flux(0, qm[1], qp[2], fr, k);
    const bool zl = rf[1] || rf[2], zr = rf[2] || rf[3];
    const int ind = i2;
    const double *pb = a.ubase + (size_t)(o - 1) * 10 + ind;
    double *po = a.unew + (size_t)(o - 1) * 10 + ind;
    double FLs[5], FRs[5];
#pragma unroll
    for (int n = 0; n < 5; n++) {
        FLs[n] = zl ? 0.0 : (double(fl[n]) * dt) * a.inv_dx;
        FRs[n] = zr ? 0.0 : (double(fr[n]) * dt) * a.inv_dx;
        po[2 * n] = pb[2 * n] + (FLs[n] - FRs[n]);
    }
    if (a.reflux) {
        // the left neighbour cell lies in this oct (i2=1) or in slot 0; the right one in this oct or slot 2
        const int vl = i2 == 1 ? o : nb[0], vr = i2 == 0 ? o : nb[2];
        if (!zl && vl > a.ngridmax) reflux_add(a.unew, a.ghost_parent, a.ngridmax, vl, -1.0, FLs, 2, a.racc, a.rdet, 4);
        if (!zr && vr > a.ngridmax) reflux_add(a.unew, a.ghost_parent, a.ngridmax, vr, 1.0, FRs, 2, a.racc, a.rdet, 0);
    }
}

// ---------------------------------------------------------------------------
// Courant time step and conservation sums (courant_fine + cmpdt).
// ---------------------------------------------------------------------------
constexpr int kCourantThreads = 256;

// The block's partials {mass, ekin, eint, dt} in a fixed order; dt_of turns the
// block's largest signal speed into its dt.
template <typename F>
__device__ __forceinline__ void courant_block(double mass, double ekin, double eint, double sig, F dt_of,
                                              double *__restrict__ part)
{
    __shared__ double red[kCourantThreads / 64][4];
    mass = wave_sum(mass);
    ekin = wave_sum(ekin);
    eint = wave_sum(eint);
    sig = wave_max(sig);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    if (l == 0) {
        red[w][0] = mass;
        red[w][1] = ekin;
        red[w][2] = eint;
        red[w][3] = sig;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double s0 = 0, s1 = 0, s2 = 0, m = red[0][3];
        for (int i = 0; i < kCourantThreads / 64; i++) {
            s0 += red[i][0];
            s1 += red[i][1];
            s2 += red[i][2];
            m = red[i][3] > m ? red[i][3] : m;
        }
        part[4 * blockIdx.x + 0] = s0;
        part[4 * blockIdx.x + 1] = s1;
        part[4 * blockIdx.x + 2] = s2;
        part[4 * blockIdx.x + 3] = dt_of(m);
    }
}

template <int TTD>
__global__ void __launch_bounds__(kCourantThreads) k_courant(const double *__restrict__ uold,
                                                             const uint8_t *__restrict__ refined, int head, int noct,
                                                             const CourantK c, double *__restrict__ part)
{
    double mass = 0, ekin = 0, eint = 0, sig = 0;
    constexpr int ttd = TTD, stride = 5 * TTD;
    const long ncell = (long)noct * ttd;
    const long step = (long)gridDim.x * blockDim.x;
    // four cells per thread per round, their loads issued together
    constexpr int U = 4;
    for (long i0 = (long)blockIdx.x * blockDim.x + threadIdx.x; i0 < ncell; i0 += U * step) {
        double u[U][5];
        bool leaf[U];
#pragma unroll
        for (int k = 0; k < U; k++) {
            const long i = i0 + k * step;
            leaf[k] = false;
            if (i < ncell) {
                const long o = (long)(head - 1) + i / ttd;
                const int ind = (int)(i % ttd);
                const double *p = uold + o * stride + ind;
#pragma unroll
                for (int n = 0; n < 5; n++) u[k][n] = p[n * ttd];
                leaf[k] = !refined[o * 8 + ind];
            }
        }
#pragma unroll
        for (int k = 0; k < U; k++)
            if (leaf[k])
                sig = tmax(sig, courant_cell < TTD == 8 ? 3 : 1 > (u[k], c, c.vol, mass, ekin, eint));
    }
    courant_block(mass, ekin, eint, sig, [&](double x) { return signal_dt(x, c); }, part);
}

// courant_fine over octs of several levels: c0 carries the level-independent
// constants (c0.dx = finest dx, c0.gsum_dx = sum |g|), dx of an oct is
// boxlen*2^-lev (the same value the host computes as boxlen/2^lev).  Without
// gravity dt = dx / (signal speed) times a constant, and dx scales by powers
// of two, so the block reduces max ctot 2^lev (exact) and takes one dt of it;
// with gravity (and in FP32) each cell's dt is formed and -dt reduced.  MIXED:
// the signal speed and dt in FP32, as the mixed-precision kernels' fused
// reduction (courant_cell_mixed).
template <bool MIXED>
__global__ void __launch_bounds__(kCourantThreads) k_courant_ml(const double *__restrict__ uold,
                                                                const uint8_t *__restrict__ refined,
                                                                const int32_t *__restrict__ lev, int head, int noct,
                                                                const CourantK c0, double boxlen,
                                                                double *__restrict__ part)
{
    const bool percell = MIXED || c0.gsum_dx != 0.0;
    double mass = 0, ekin = 0, eint = 0, dtmin = c0.dx / c0.smallc, sig = 0.0;
    const long ncell = (long)noct * 8;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < ncell; i += (long)gridDim.x * blockDim.x) {
        const long o = (long)(head - 1) + i / 8;
        const int ind = (int)(i % 8);
        if (refined[o * 8 + ind]) continue;
        CourantK c = c0;
        const int l = lev[o];
        const double dx = __builtin_ldexp(boxlen, -l);
        c.dx = dx;
        c.vol = dx * dx * dx;
        c.gsum_dx = c0.gsum_dx * dx;
        const double *p = uold + o * 40 + ind;
        const double u[5] = {p[0], p[8], p[16], p[24], p[32]};
        if constexpr (MIXED) {
            courant_cell_mixed(u, c, mass, ekin, eint, dtmin);
        } else {
            const double ctot = courant_cell<3>(u, c, c.vol, mass, ekin, eint);
            if (percell)
                dtmin = tmin(dtmin, signal_dt(ctot, c));
            else
                sig = tmax(sig, __builtin_ldexp(ctot, l));
        }
    }
    courant_block(
        mass, ekin, eint, percell ? -dtmin : sig,
        [&](double x) {
            if (percell) return -x;
            if (!(x > 0.0)) return c0.dx / c0.smallc;  // no leaf cell
            CourantK c = c0;
            c.dx = boxlen;
            return signal_dt(x, c);
        },
        part);
}

// Block b of a grid of nb blocks renumbered so that the blocks the hardware
// sends to one XCD (b mod 8) take one contiguous range of [0, nb).
__device__ __forceinline__ int xcd_block(int b, int nb)
{
    const int x = b & 7, l = b >> 3, q = nb >> 3, r = nb & 7;
    return x * q + (x < r ? x : r) + l;
}

__global__ void k_zero(double *p, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = 0.0;
}

// Coarse-fine reflux fold: each ghost oct stands for one parent cell.  The
// accumulator is left zeroed for the next step (it starts zeroed); ghosts
// that received no flux leave their parent cell untouched, as the direct
// reflux of the per-level calls does.
// With nslot = kRefluxSlots (deterministic mode) each ghost has one slot per
// face of its oct, added to the parent cell one after another in slot order:
// the same sums on every run.
// One thread per ghost and variable: the fold is a chain of dependent gathers
// (order, accumulator, parent cell), so what counts is how many are in flight.
// 4.9 M cells on five levels: 26.0 -> 25.6 us; 1.1 M cells on four: 5.2 -> 4.9.
__global__ void __launch_bounds__(256) k_reflux_fold(double *unew, double *__restrict__ racc,
                                                     const int32_t *__restrict__ ghost_parent,
                                                     const int32_t *__restrict__ order, int nghost, int ttd, int nslot)
{
    // in parent-cell order (see k_refresh_ghosts)
    const int i = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const int t = i / 5, n = i - 5 * t;
    if (t >= nghost) return;
    const int g = order[t];
    double *rg = racc + 5 * (size_t)g * nslot + n;
    const int igrid = ghost_parent[2 * g], icell = ghost_parent[2 * g + 1];
    double *p = igrid > 0 ? unew + (size_t)(igrid - 1) * 5 * ttd + n * ttd + (icell - 1) : nullptr;
    double acc = 0.0;
    bool touched = false;
    for (int k = 0; k < nslot; k++) {
        const double f = rg[5 * k];
        if (f == 0.0) continue;
        rg[5 * k] = 0.0;
        if (!p) continue;  // parent in a boundary oct: the reference drops it with the cache oct
        if (!touched) acc = *p;
        touched = true;
        acc = acc + f;
    }
    if (touched) *p = acc;
}

// Fixed-order reduction of the per-block partials by one 256-thread block:
// out = {mass, ekin, eint, emag, dt}; dt_out (optional) receives dt for the
// next Godunov launch; t_acc (optional) accumulates the time (the old dt_out
// when acc_old, else the new dt).
__device__ __forceinline__ void courant_final_block(const double *__restrict__ part, int nblocks, double dtmax,
                                                    double *__restrict__ out, double *__restrict__ dt_out,
                                                    double *__restrict__ t_acc, int acc_old)
{
    __shared__ double red[4][4];
    double s0 = 0, s1 = 0, s2 = 0, m = dtmax;
    // One block's latency is all that this takes, so the loads go out together:
    // the old time and dt, needed last, first, and four rounds of partials at a
    // time (2048 partials 6.8 -> 5.0 us).
    const bool last = threadIdx.x == 0;
    const double t_old = last && t_acc ? *t_acc : 0.0, dt_old = last && dt_out ? *dt_out : 0.0;
    const double2 *p2 = reinterpret_cast<const double2 *>(part);
    constexpr int U = 4;
    for (int i0 = threadIdx.x; i0 < nblocks; i0 += U * 256) {
        double2 a[U], b[U];
#pragma unroll
        for (int k = 0; k < U; k++) {
            const int i = i0 + 256 * k < nblocks ? i0 + 256 * k : i0;
            a[k] = p2[2 * i];
            b[k] = p2[2 * i + 1];
        }
#pragma unroll
        for (int k = 0; k < U; k++)
            if (i0 + 256 * k < nblocks) {
                s0 += a[k].x;
                s1 += a[k].y;
                s2 += b[k].x;
                m = b[k].y < m ? b[k].y : m;
            }
    }
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    m = wave_min(m);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    if (l == 0) {
        red[w][0] = s0;
        red[w][1] = s1;
        red[w][2] = s2;
        red[w][3] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a0 = 0, a1 = 0, a2 = 0, mm = red[0][3];
        for (int i = 0; i < 4; i++) {
            a0 += red[i][0];
            a1 += red[i][1];
            a2 += red[i][2];
            mm = red[i][3] < mm ? red[i][3] : mm;
        }
        out[0] = a0;
        out[1] = a1;
        out[2] = a2;
        out[3] = 0.0;
        out[4] = mm;
        if (t_acc) *t_acc = t_old + ((acc_old && dt_out) ? dt_old : mm);
        if (dt_out) *dt_out = mm;
    }
}

__global__ void __launch_bounds__(256) k_courant_final(const double *__restrict__ part, int nblocks, double dtmax,
                                                       double *__restrict__ out, double *__restrict__ dt_out,
                                                       double *__restrict__ t_acc, int acc_old)
{
    courant_final_block(part, nblocks, dtmax, out, dt_out, t_acc, acc_old);
}

// The conservation sums of whole bricks, added in the order in which a work-list
// launch of uncut bricks adds them: FP64 per column of the brick, its cells along z
// (hw: the kernel's interior columns come first, see brick64_hw), mixed per cell
// index.  state: the state that the step wrote.
__global__ void __launch_bounds__(512) k_brick_sums(const GodArgs a, const double *__restrict__ state, int bx, int by,
                                                    int bz, int hw, int mixed, double *__restrict__ part)
{
    __shared__ double red[8][3];
    const int wx = bx + 2, wy = by + 2, bid = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
    const int32_t *win = a.win + (size_t)bid * wx * wy * (bz + 2);
    const int zr = a.zr ? a.zr[bid] : (bz - 1) << 16;
    const double gv[3] = {a.g[0], a.g[1], a.g[2]};
    const CourantK ck = make_courant_k(a.dx, 3, a.gamma, a.smallr, a.smallc2, a.courant_factor, gv);
    double mass = 0.0, ekin = 0.0, eint = 0.0, dt = 0.0;
    // cell (x, y, z) of the brick
    auto add = [&](int x, int y, int z) {
        const int v = win[((z >> 1) + 1) * (wx * wy) + ((y >> 1) + 1) * wx + (x >> 1) + 1];
        if (v < a.head || v >= a.head + a.noct || a.org[3 * bid] + (x >> 1) >= a.boxmax[0] ||
            a.org[3 * bid + 1] + (y >> 1) >= a.boxmax[1] || a.org[3 * bid + 2] + (z >> 1) >= a.boxmax[2])
            return;
        const int ind = (x & 1) + 2 * (y & 1) + 4 * (z & 1);
        if (a.refined[(size_t)(v - 1) * 8 + ind]) return;
        const double *p = state + (size_t)(v - 1) * 40 + ind;
        const double u[5] = {p[0], p[8], p[16], p[24], p[32]};
        if (mixed)
            courant_cell_mixed(u, ck, mass, ekin, eint, dt);
        else
            (void)courant_cell<3>(u, ck, ck.vol, mass, ekin, eint);
    };
    if (mixed) {
        for (int i = tid; i < bx * by * bz * 8; i += nt) {
            const int oc = i >> 3;
            const int oz = oc / (bx * by);
            if (oz >= (zr & 0xffff) && oz <= zr >> 16)
                add(2 * (oc % bx) + (i & 1), 2 * ((oc / bx) % by) + ((i >> 1) & 1), 2 * oz + ((i >> 2) & 1));
        }
    } else {
        const int x = hw ? tid % (2 * bx) : tid % (2 * bx + 2) - 1, y = hw ? tid / (2 * bx) : tid / (2 * bx + 2) - 1;
        if (x >= 0 && x < 2 * bx && y >= 0 && y < 2 * by)
            for (int z = 2 * (zr & 0xffff); z <= 2 * (zr >> 16) + 1; z++) add(x, y, z);
    }
    const int nv = nt - (tid & ~63) < 64 ? nt - (tid & ~63) : 64;
    mass = wave_sum_n(mass, nv);
    ekin = wave_sum_n(ekin, nv);
    eint = wave_sum_n(eint, nv);
    if ((tid & 63) == 0) {
        red[tid >> 6][0] = mass;
        red[tid >> 6][1] = ekin;
        red[tid >> 6][2] = eint;
    }
    __syncthreads();
    if (tid == 0) {
        double s[3] = {0, 0, 0};
        for (int i = 0; i < (nt + 63) / 64; i++)
            for (int k = 0; k < 3; k++) s[k] += red[i][k];
        for (int k = 0; k < 3; k++) part[4 * bid + k] = s[k];
        part[4 * bid + 3] = a.dx / ck.smallc;
    }
}

// One block per job of a batch: each job's own partials, in its fixed order.
__global__ void __launch_bounds__(256) k_courant_final_batch(const CourantJob *__restrict__ jobs)
{
    const CourantJob j = jobs[blockIdx.x];
    courant_final_block(j.part, j.nparts, j.dtmax, j.out, j.dt_inout, j.t_acc, 1);
}

// ---------------------------------------------------------------------------
// AMR: ghost octs (interpolated from the parent level) and restriction
// ---------------------------------------------------------------------------
__device__ __forceinline__ void cell_xc(int ndim, int ind, double xc[3])
{
    const int iz = (ind - 1) / 4, iy = (ind - 1 - 4 * iz) / 2, ix = ind - 1 - 2 * iy - 4 * iz;
    xc[0] = (double)ix - 0.5;
    xc[1] = ndim > 1 ? (double)iy - 0.5 : 0.0;
    xc[2] = ndim > 2 ? (double)iz - 0.5 : 0.0;
}

// One variable of interpol_hydro (hydro/interpol_hydro.f90:5-113) with the
// limiters of :610-752; a[j], j = 0 (central parent) and 1..2ndim
// (-x,+x,-y,+y,-z,+z).  ND is a compile-time constant so that every loop
// unrolls and the arrays stay in registers (a runtime ndim put them in scratch
// memory).
template <int ND>
__device__ __forceinline__ void interpol_var_dev(const double a[7], double u[8], int interpol_type)
{
    constexpr int ndim = ND, twondim = 2 * ND, ttd = 1 << ND;
    double w[3] = {0, 0, 0};
    if (interpol_type == 1) {
        #pragma unroll
        for (int d = 1; d <= ndim; d++) {
            const double dl = 0.5 * (a[2 * d] - a[0]), dr = 0.5 * (a[0] - a[2 * d - 1]);
            w[d - 1] = (dl * dr <= 0.0) ? 0.0 : fmin(fabs(dl), fabs(dr)) * dl / fabs(dl);
        }
    } else if (interpol_type == 2 || interpol_type == 3) {
        #pragma unroll
        for (int d = 1; d <= ndim; d++) w[d - 1] = 0.25 * (a[2 * d] - a[2 * d - 1]);
        if (interpol_type == 2) {
            double ac[8];
            #pragma unroll
            for (int c = 0; c < ttd; c++) ac[c] = a[0];
            #pragma unroll
            for (int d = 1; d <= ndim; d++)
                #pragma unroll
                for (int c = 1; c <= ttd; c++) {
                    double xc[3];
                    cell_xc(ndim, c, xc);
                    ac[c - 1] = ac[c - 1] + 2.0 * w[d - 1] * xc[d - 1];
                }
            double cmax = ac[0], cmin = ac[0], kmax = a[1], kmin = a[1];
            #pragma unroll
            for (int c = 1; c < ttd; c++) {
                cmax = fmax(cmax, ac[c]);
                cmin = fmin(cmin, ac[c]);
            }
            #pragma unroll
            for (int j = 2; j <= twondim; j++) {
                kmax = fmax(kmax, a[j]);
                kmin = fmin(kmin, a[j]);
            }
            double dk = a[0] - kmax, dc = a[0] - cmax;
            const double lmax = (dk * dc > 0.0) ? fmin(1.0, dk / dc) : 0.0;
            dk = a[0] - kmin;
            dc = a[0] - cmin;
            const double lmin = (dk * dc > 0.0) ? fmin(1.0, dk / dc) : 0.0;
            const double lim = fmin(lmin, lmax);
            #pragma unroll
            for (int d = 0; d < ndim; d++) w[d] = w[d] * lim;
        }
    }
    #pragma unroll
    for (int c = 1; c <= ttd; c++) {
        double xc[3];
        cell_xc(ndim, c, xc);
        double v = a[0];
        #pragma unroll
        for (int d = 1; d <= ndim; d++) v = v + w[d - 1] * xc[d - 1];
        u[c - 1] = v;
    }
}

// All five variables, u1[j][ivar].
template <int ND>
__device__ __forceinline__ void interpol_hydro_dev(double u1[7][5], double u2[8][5], int interpol_var, int interpol_type,
                                   double smallr)
{
    constexpr int twondim = 2 * ND, ttd = 1 << ND;
    if (interpol_var == 1)
        #pragma unroll
        for (int j = 0; j <= twondim; j++) {
            double ekin = 0.0;
            #pragma unroll
            for (int d = 1; d <= 3; d++) ekin = ekin + 0.5 * (u1[j][d] * u1[j][d]) / fmax(u1[j][0], smallr);
            u1[j][4] = u1[j][4] - ekin - 0.0;
        }
#pragma unroll
    for (int iv = 0; iv < 5; iv++) {
        double a[7], u[8];
        #pragma unroll
        for (int j = 0; j <= twondim; j++) a[j] = u1[j][iv];
        interpol_var_dev<ND>(a, u, interpol_type);
        #pragma unroll
        for (int c = 0; c < ttd; c++) u2[c][iv] = u[c];
    }
    if (interpol_var == 1)
        #pragma unroll
        for (int c = 0; c < ttd; c++) {
            double ekin = 0.0;
            #pragma unroll
            for (int d = 1; d <= 3; d++) ekin = ekin + 0.5 * (u2[c][d] * u2[c][d]) / fmax(u2[c][0], smallr);
            u2[c][4] = u2[c][4] + ekin + 0.0;
        }
}

template <int ND>
__global__ void __launch_bounds__(64) k_refresh_ghosts(const GhostArgs a)
{
    // ghosts in parent-cell order, a contiguous range of that order per XCD,
    // so that the parent octs a wave gathers meet in one L2
    const int t = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const bool valid = t < a.nghost;
    if constexpr (ND == 1) {
        if (!valid) return;
    }
    constexpr int ttd = 1 << ND, nslot = 2 * ND + 1;
    const int stride = ttd * 5;
    double u2[8][5];
    int g = -1;
    if (valid) {
        int k = 0;
        for (int j = 1; j < a.nseg; j++) k = t >= a.seg_t[j] ? j : k;
        const int pos = a.seg_o[k] + (t - a.seg_t[k]);
        g = a.order[pos] - a.gi0;
        const int boxmin[3] = {a.seg_box[k][0], a.seg_box[k][1], a.seg_box[k][2]};
        const int boxmax[3] = {a.seg_box[k][3], a.seg_box[k][4], a.seg_box[k][5]};
        double u1[7][5];
#pragma unroll
        for (int j = 0; j < nslot; j++) {
            const int code = a.src[(size_t)(2 * j) * a.src_ld + pos], ind = a.src[(size_t)(2 * j + 1) * a.src_ld + pos];
            // the source's oct key locates boundary ghosts only (code < 0)
            int okey[3] = {0, 0, 0};
            if (code < 0) {
                okey[0] = a.srckey[(g * 7 + j) * 3];
                okey[1] = a.srckey[(g * 7 + j) * 3 + 1];
                okey[2] = a.srckey[(g * 7 + j) * 3 + 2];
            }
            int c[3] = {(ind - 1) & 1, ((ind - 1) >> 1) & 1, ((ind - 1) >> 2) & 1};
            uint8_t rf;
            if constexpr (ND == 3) {
                // select-based flip: no runtime index into u1 (which would put it in scratch)
                const CellRef r =
                    cell_ref3(a.uold, a.refined, code, okey, boxmin, boxmax, reflexive_mask(a.btype), c);
                cell_load3(r, u1[j], rf);
                cell_flip(u1[j], r.flip);
            } else {
                gather_cell(a.uold, a.refined, code, okey, ND, boxmin, boxmax, a.btype, c, u1[j], rf);
            }
        }
        interpol_hydro_dev<ND>(u1, u2, a.interpol_var, a.interpol_type, a.smallr);
    } else {
#pragma unroll
        for (int c = 0; c < 8; c++)
#pragma unroll
            for (int n = 0; n < 5; n++) u2[c][n] = 0.0;
    }
    if constexpr (ND == 3) {
        // Stores staged through LDS one variable at a time: a ghost's variable
        // is one aligned 64-byte line, written by four lanes with 16 bytes
        // each, so a store instruction of the wave covers 16 whole lines
        // instead of touching 64 lines with 16 bytes each.
        __shared__ double2 sm[64 * 4];
        const int lane = threadIdx.x;
        int gq[4];
#pragma unroll
        for (int q = 0; q < 4; q++) gq[q] = __shfl(g, (q * 64 + lane) >> 2);
#pragma unroll
        for (int n = 0; n < 5; n++) {
            if (n) __syncthreads();
#pragma unroll
            for (int c = 0; c < 4; c++) sm[lane * 4 + c] = make_double2(u2[2 * c][n], u2[2 * c + 1][n]);
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (gq[q] >= 0) {
                    double2 *p2 = reinterpret_cast<double2 *>(a.uold + (size_t)(a.first - 1 + gq[q]) * stride);
                    p2[n * 4 + (lane & 3)] = sm[q * 64 + lane];
                }
        }
    } else {
        double *p = a.uold + (size_t)(a.first - 1 + g) * stride;
#pragma unroll
        for (int c = 0; c < ttd; c++)
#pragma unroll
            for (int n = 0; n < 5; n++) p[n * ttd + c] = u2[c][n];
    }
}

// k_refresh_ghosts<3> where the variables are interpolated independently
// (interpol_var = 0): 64 ghosts per block, one wave per variable.  The refresh
// is bound by the latency of its dependent gathers (order, source, cell); one
// thread per ghost held 35 values, two waves per SIMD, and a mesh's ghosts did
// not even fill those.  A thread per ghost and variable has a fifth of the
// loads, five times the threads and the registers for all of them at once.
// 4.9 M cells on five levels: 67.9 -> 57.7 us; 1.1 M cells on four: 10.5 -> 7.5.
__global__ void __launch_bounds__(320) k_refresh_ghosts_var(const GhostArgs a)
{
    // (ghosts in parent-cell order and staged stores: see k_refresh_ghosts)
    const int lane = threadIdx.x & 63, n = threadIdx.x >> 6;
    const int t = xcd_block(blockIdx.x, gridDim.x) * 64 + lane;
    int g = -1;
    double u[8];
    if (t < a.nghost) {
        int k = 0;
        for (int j = 1; j < a.nseg; j++) k = t >= a.seg_t[j] ? j : k;
        const int pos = a.seg_o[k] + (t - a.seg_t[k]);
        int code[7], ind[7];
        g = a.order[pos] - a.gi0;
#pragma unroll
        for (int j = 0; j < 7; j++) {
            code[j] = a.src[(size_t)(2 * j) * a.src_ld + pos];
            ind[j] = a.src[(size_t)(2 * j + 1) * a.src_ld + pos] - 1;
        }
        const int boxmin[3] = {a.seg_box[k][0], a.seg_box[k][1], a.seg_box[k][2]};
        const int boxmax[3] = {a.seg_box[k][3], a.seg_box[k][4], a.seg_box[k][5]};
        const int refl = reflexive_mask(a.btype);
        const double *p[7];
        bool neg[7];
#pragma unroll
        for (int j = 0; j < 7; j++) {
            p[j] = code[j] > 0 ? a.uold + (size_t)(code[j] - 1) * 40 + ind[j] + 8 * n : a.uold;
            neg[j] = false;
            if (code[j] < 0) {
                // the source's oct key locates boundary ghosts only
                const int *key = a.srckey + (g * 7 + j) * 3;
                const int okey[3] = {key[0], key[1], key[2]};
                const int c[3] = {ind[j] & 1, (ind[j] >> 1) & 1, (ind[j] >> 2) & 1};
                const CellRef r = cell_ref3(a.uold, a.refined, code[j], okey, boxmin, boxmax, refl, c);
                p[j] = r.p + 8 * n;
                neg[j] = r.flip >= 0 && r.flip == n - 1;
            }
        }
        double v[7];
#pragma unroll
        for (int j = 0; j < 7; j++) v[j] = *p[j];
#pragma unroll
        for (int j = 0; j < 7; j++) {
            v[j] = code[j] == 0 ? 0.0 : v[j];
            v[j] = neg[j] ? -v[j] : v[j];
        }
        interpol_var_dev<3>(v, u, a.interpol_type);
    } else {
#pragma unroll
        for (int c = 0; c < 8; c++) u[c] = 0.0;
    }
    __shared__ double2 sm[5][64 * 4];
#pragma unroll
    for (int c = 0; c < 4; c++) sm[n][lane * 4 + c] = make_double2(u[2 * c], u[2 * c + 1]);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int gq = __shfl(g, (q * 64 + lane) >> 2);
        if (gq >= 0)
            reinterpret_cast<double2 *>(a.uold + (size_t)(a.first - 1 + gq) * 40)[n * 4 + (lane & 3)] =
                sm[n][q * 64 + lane];
    }
}

hipError_t launch_refresh_ghosts(const GhostArgs &a, hipStream_t s)
{
    if (a.nghost <= 0) return hipSuccess;
    if (a.ndim == 3 && a.interpol_var == 0)
        hipLaunchKernelGGL(k_refresh_ghosts_var, dim3((a.nghost + 63) / 64), dim3(320), 0, s, a);
    else if (a.ndim == 3)
        hipLaunchKernelGGL(k_refresh_ghosts<3>, dim3((a.nghost + 63) / 64), dim3(64), 0, s, a);
    else
        hipLaunchKernelGGL(k_refresh_ghosts<1>, dim3((a.nghost + 63) / 64), dim3(64), 0, s, a);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256) k_upload(double *uold, const int32_t *father, int head, int noct, int ttd,
                                                int internal_energy, double smallr)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= noct) return;
    const int o = head - 1 + i;
    const int igrid = father[2 * i], icell = father[2 * i + 1];
    if (igrid <= 0) return;
    const double *c = uold + (size_t)o * 5 * ttd;
    double *p = uold + (size_t)(igrid - 1) * 5 * ttd + (icell - 1);
    for (int n = 0; n < 5; n++) {
        double avg = 0.0;
        for (int k = 0; k < ttd; k++) avg = avg + c[n * ttd + k];
        p[n * ttd] = avg / (double)ttd;
    }
    if (internal_energy) {
        double avg = 0.0;
        for (int k = 0; k < ttd; k++) {
            double ekin = 0.0;
            for (int d = 1; d <= 3; d++) ekin = ekin + 0.5 * (c[d * ttd + k] * c[d * ttd + k]) / fmax(c[k], smallr);
            avg = avg + c[4 * ttd + k] - ekin - 0.0 - 0.0;
        }
        double ekin = 0.0;
        for (int d = 1; d <= 3; d++) ekin = ekin + 0.5 * (p[d * ttd] * p[d * ttd]) / fmax(p[0], smallr);
        p[4 * ttd] = avg / (double)ttd + ekin + 0.0 + 0.0;
    }
}

// upload_fine with interpol_var = 0: one thread per (fine oct, variable),
// each averaging one contiguous 64-byte line of the oct.
__global__ void __launch_bounds__(256) k_upload_var(double *uold, const int32_t *__restrict__ father, int head,
                                                    int noct)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)noct * 5) return;
    const int io = (int)(i / 5), n = (int)(i % 5);
    const int igrid = father[2 * io], icell = father[2 * io + 1];
    if (igrid <= 0) return;
    // the oct's variable is one aligned 64-byte line: four 16-byte loads
    const double2 *c = reinterpret_cast<const double2 *>(uold + ((size_t)(head - 1 + io) * 5 + n) * 8);
    double avg = 0.0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const double2 v = c[k];
        avg = avg + v.x;
        avg = avg + v.y;
    }
    uold[((size_t)(igrid - 1) * 5 + n) * 8 + (icell - 1)] = avg / 8.0;
}

// Restriction of one level and its share of the Courant pass in one read of its
// octs (the batched AMR step; interpol_var = 0): per round a block takes 32 octs,
// a thread per cell, whose values go through LDS to a thread per oct and
// variable, which averages them in the cells' order as k_upload_var does.  Levels
// run finest first.  Leaf cells are no restriction's target, so a level's
// Courant share does not wait for the level's own restriction.  father null: the
// coarsest level, nothing to restrict to.  Both passes alone are bound by
// their reads: 4.9 M cells on five levels 71 us (four restrictions and a Courant
// pass) -> 67 us, 1.1 M cells on four, mixed precision, 29.3 -> 25.6 us.
template <bool MIXED>
__global__ void __launch_bounds__(kCourantThreads) k_upload_courant(double *uold, const uint8_t *__restrict__ refined,
                                                                    const int32_t *__restrict__ father, int head,
                                                                    int noct, int lev, const CourantK c0, double boxlen,
                                                                    double *__restrict__ part)
{
    __shared__ double sm[kCourantThreads / 8 * 5][9];
    const bool percell = MIXED || c0.gsum_dx != 0.0;
    double mass = 0, ekin = 0, eint = 0, dtmin = c0.dx / c0.smallc, sig = 0.0;
    CourantK c = c0;
    const double dx = __builtin_ldexp(boxlen, -lev);
    c.dx = dx;
    c.vol = dx * dx * dx;
    c.gsum_dx = c0.gsum_dx * dx;
    const int lo = threadIdx.x >> 3, ind = threadIdx.x & 7;
    const int t = threadIdx.x, io = t / 5, n5 = t - 5 * io;
    // the next round's loads are in flight while a round is worked on
    double un[5];
    bool leafn;
    int gridn, celln;
    auto load = [&](long o0) {
        const long o = o0 + lo < noct ? o0 + lo : noct - 1;
        const double *p = uold + (head - 1 + o) * 40 + ind;
#pragma unroll
        for (int n = 0; n < 5; n++) un[n] = p[8 * n];
        leafn = !refined[(head - 1 + o) * 8 + ind] && o0 + lo < noct;
        gridn = 0;
        celln = 0;
        if (father && io < 32 && o0 + io < noct) {
            gridn = father[2 * (o0 + io)];
            celln = father[2 * (o0 + io) + 1];
        }
    };
    const long step = (long)gridDim.x * 32;
    load((long)blockIdx.x * 32);
    for (long o0 = (long)blockIdx.x * 32; o0 < noct; o0 += step) {
        double u[5];
#pragma unroll
        for (int n = 0; n < 5; n++) u[n] = un[n];
        const bool leaf = leafn;
        const int igrid = gridn, icell = celln;
        if (o0 + step < noct) load(o0 + step);
        if (father) {
            __syncthreads();
#pragma unroll
            for (int n = 0; n < 5; n++) sm[lo * 5 + n][ind] = u[n];
            __syncthreads();
            if (igrid > 0) {
                double avg = 0.0;
#pragma unroll
                for (int k = 0; k < 8; k++) avg = avg + sm[t][k];
                uold[((size_t)(igrid - 1) * 5 + n5) * 8 + (icell - 1)] = avg / 8.0;
            }
        }
        if (!leaf) continue;
        if constexpr (MIXED) {
            courant_cell_mixed(u, c, mass, ekin, eint, dtmin);
        } else {
            const double ctot = courant_cell<3>(u, c, c.vol, mass, ekin, eint);
            if (percell)
                dtmin = tmin(dtmin, signal_dt(ctot, c));
            else
                sig = tmax(sig, __builtin_ldexp(ctot, lev));
        }
    }
    courant_block(
        mass, ekin, eint, percell ? -dtmin : sig,
        [&](double x) {
            if (percell) return -x;
            if (!(x > 0.0)) return c0.dx / c0.smallc;  // no leaf cell
            CourantK cb = c0;
            cb.dx = boxlen;
            return signal_dt(x, cb);
        },
        part);
}

hipError_t launch_upload(double *uold, const int32_t *father, int head, int noct, int ndim, int internal_energy,
                         double smallr, hipStream_t s)
{
    if (noct <= 0) return hipSuccess;
    if (ndim == 3 && !internal_energy) {
        const long n = (long)noct * 5;
        hipLaunchKernelGGL(k_upload_var, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, uold, father, head, noct);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_upload, dim3((noct + 255) / 256), dim3(256), 0, s, uold, father, head, noct, 1 << ndim,
                       internal_energy, smallr);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Artificial diffusion (difmag > 0): cmpdivu + cmpdiff, hydro/umuscl.f90:
// 2392-2540, called by unsplit at :273-283.  The diffusive flux of a face,
// dt * difmag * min(0, mean of the velocity divergence at its 2^(ndim-1)
// corner nodes) * (u_R - u_L), is linear in the update, so it runs as a pass
// after the Godunov launch: unew += (D_low - D_high) per dimension, D zeroed
// where either cell is refined (as the fluxes), refluxed into the parent cell
// across coarse-fine faces (as godfine1 refluxes flux + D).  Each cell
// computes its own faces; the two cells of a face compute the same D from the
// same values in the same order.
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(256) k_diffusion3d(const DiffArgs a)
{
#pragma clang fp contract(off)
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)a.noct * 8) return;
    const int o = a.head - 1 + (int)(i >> 3), ind = (int)(i & 7);
    const int c0[3] = {ind & 1, (ind >> 1) & 1, (ind >> 2) & 1};
    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    const double gdt[3] = {a.g[0] * (dt * 0.5), a.g[1] * (dt * 0.5), a.g[2] * (dt * 0.5)};
    const int32_t *nb = a.nbor + (size_t)(o - (a.head - 1)) * 27;
    // velocities (with ctoprim's gravity kick) of the 3x3x3 cells around the
    // cell, the conservative states of the cell and its 6 face neighbours,
    // the refined flags, and the oct index of the face neighbours
    double q[3][3][3][3];
    double uf[7][5];
    uint8_t rf[7];
    int vf[7];
    for (int dz = -1; dz <= 1; dz++)
        for (int dy = -1; dy <= 1; dy++)
            for (int dx = -1; dx <= 1; dx++) {
                const int cc[3] = {c0[0] + dx, c0[1] + dy, c0[2] + dz};
                int oo[3], cb[3];
                for (int d = 0; d < 3; d++) {
                    oo[d] = cc[d] >> 1;  // -1, 0 or 1
                    cb[d] = cc[d] & 1;
                }
                const int v = nb[(oo[0] + 1) + 3 * (oo[1] + 1) + 9 * (oo[2] + 1)];
                const int okey[3] = {a.ckey[3 * o] + oo[0], a.ckey[3 * o + 1] + oo[1], a.ckey[3 * o + 2] + oo[2]};
                const CellRef r = cell_ref3(a.uold, a.refined, v, okey, a.boxmin, a.boxmax, a.refl, cb);
                double u[5];
                uint8_t f;
                cell_load3(r, u, f);
                cell_flip(u, r.flip);
                const double rho = u[0] > a.smallr ? u[0] : a.smallr;
                const double ir = 1.0 / rho;
                for (int d = 0; d < 3; d++) q[dz + 1][dy + 1][dx + 1][d] = u[1 + d] * ir + gdt[d];
                const int nz = (dx != 0) + (dy != 0) + (dz != 0);
                if (nz <= 1) {
                    // 0: the cell; 1..6: -x +x -y +y -z +z
                    const int k = nz == 0 ? 0 : dx ? (dx < 0 ? 1 : 2) : dy ? (dy < 0 ? 3 : 4) : (dz < 0 ? 5 : 6);
                    for (int n = 0; n < 5; n++) uf[k][n] = u[n];
                    rf[k] = f;
                    vf[k] = v;
                }
            }
    // divergence at the node (x, y, z) in {0,1}^3 of the cell's corners,
    // cmpdivu's expression order (node (i,j,k) uses cells i-1..i, j-1..j, k-1..k)
    const double fact = 0.25 / a.dx;  // half**(ndim-1)/dx
    auto Q = [&](int x, int y, int z, int d) { return q[z + 1][y + 1][x + 1][d]; };
    double dv[2][2][2];
    for (int z = 0; z < 2; z++)
        for (int y = 0; y < 2; y++)
            for (int x = 0; x < 2; x++) {
                double ux = 0.0, vy = 0.0, wz = 0.0;
                ux = ux + fact * (Q(x, y, z, 0) - Q(x - 1, y, z, 0));
                ux = ux + fact * (Q(x, y - 1, z, 0) - Q(x - 1, y - 1, z, 0));
                vy = vy + fact * (Q(x, y, z, 1) - Q(x, y - 1, z, 1) + Q(x - 1, y, z, 1) - Q(x - 1, y - 1, z, 1));
                ux = ux + fact * (Q(x, y, z - 1, 0) - Q(x - 1, y, z - 1, 0) + Q(x, y - 1, z - 1, 0) -
                                  Q(x - 1, y - 1, z - 1, 0));
                vy = vy + fact * (Q(x, y, z - 1, 1) - Q(x, y - 1, z - 1, 1) + Q(x - 1, y, z - 1, 1) -
                                  Q(x - 1, y - 1, z - 1, 1));
                wz = wz + fact * (Q(x, y, z, 2) - Q(x, y, z - 1, 2) + Q(x, y - 1, z, 2) - Q(x, y - 1, z - 1, 2) +
                                  Q(x - 1, y, z, 2) - Q(x - 1, y, z - 1, 2) + Q(x - 1, y - 1, z, 2) -
                                  Q(x - 1, y - 1, z - 1, 2));
                dv[z][y][x] = ux + vy + wz;
            }
    const double f4 = 0.25;  // half**(ndim-1)
    const bool myref = a.refined[(size_t)o * 8 + ind] != 0;
    double un[5];
    for (int n = 0; n < 5; n++) un[n] = a.unew[(size_t)o * 40 + n * 8 + ind];
    for (int d = 0; d < 3; d++) {
        double D[2][5];
        for (int side = 0; side < 2; side++) {
            // face at the cell's low (side 0) or high (side 1) boundary of dimension d
            double div1;
            if (d == 0) {
                div1 = f4 * dv[0][0][side];
                div1 = div1 + f4 * dv[0][1][side];
                div1 = div1 + f4 * (dv[1][0][side] + dv[1][1][side]);
            } else if (d == 1) {
                div1 = 0.0;
                div1 = div1 + f4 * (dv[0][side][0] + dv[0][side][1]);
                div1 = div1 + f4 * (dv[1][side][0] + dv[1][side][1]);
            } else {
                div1 = f4 * (dv[side][0][0] + dv[side][0][1] + dv[side][1][0] + dv[side][1][1]);
            }
            div1 = a.difmag * (div1 < 0.0 ? div1 : 0.0);
            const int k = 1 + 2 * d + side;
            const bool z = myref || rf[k];
            for (int n = 0; n < 5; n++) {
                const double du = side == 0 ? uf[0][n] - uf[k][n] : uf[k][n] - uf[0][n];
                D[side][n] = z ? 0.0 : dt * div1 * du;
            }
            // coarse-fine face: the neighbour is an interpolated ghost oct
            if (a.reflux && !z && vf[k] > a.ngridmax) {
                const int sub = d == 0 ? ((ind >> 1) & 1) + 2 * ((ind >> 2) & 1)
                              : d == 1 ? (ind & 1) + 2 * ((ind >> 2) & 1)
                                       : (ind & 1) + 2 * ((ind >> 1) & 1);
                // ghost on the low side sends -D/8 (its high face slot), on the high side +D/8
                reflux_add(a.unew, a.ghost_parent, a.ngridmax, vf[k], side == 0 ? -1.0 : 1.0, D[side], 8, a.racc,
                           a.rdet, side == 0 ? 4 * (2 * d + 1) + sub : 4 * (2 * d) + sub, a.rdet != 0);
            }
        }
        for (int n = 0; n < 5; n++) un[n] = un[n] + (D[0][n] - D[1][n]);
    }
    for (int n = 0; n < 5; n++) a.unew[(size_t)o * 40 + n * 8 + ind] = un[n];
}

hipError_t launch_diffusion3d(const DiffArgs &a, hipStream_t s)
{
    const long n = (long)a.noct * 8;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_diffusion3d, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_godunov1d(const God1Args &a, int prec, hipStream_t s)
{
    const int n = 2 * a.noct;
    if (n <= 0) return hipSuccess;
    const int nb = (n + 255) / 256;
    if (prec == 0)
        hipLaunchKernelGGL((k_godunov1d<double>), dim3(nb), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((k_godunov1d<float>), dim3(nb), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_courant_reduce(const double *partials, int nparts, double dtmax, double *out, double *dt_inout,
                                 double *t_acc, hipStream_t s)
{
    hipLaunchKernelGGL(k_courant_final, dim3(1), dim3(256), 0, s, partials, nparts, dtmax, out, dt_inout, t_acc, 1);
    return hipGetLastError();
}

hipError_t launch_brick_sums(const GodArgs &a, const double *state, int bx, int by, int bz, int prec, double *partials,
                             double *out, hipStream_t s)
{
    const int nt = (2 * bx + 2) * (2 * by + 2), ni = 4 * bx * by;
    const int hw = prec == 0 && a.slope != 3 && ni % 64 == 0 && nt - ni <= 64;
    if (a.nbricks <= 0 || nt > 512) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_brick_sums, dim3(a.nbricks), dim3(nt), 0, s, a, state, bx, by, bz, hw, prec, partials);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_courant_final, dim3(1), dim3(256), 0, s, partials, a.nbricks, a.dx / __builtin_sqrt(a.smallc2),
                       out, nullptr, nullptr, 0);
    return hipGetLastError();
}

hipError_t launch_courant_reduce_batch(const CourantJob *jobs, int njobs, hipStream_t s)
{
    if (njobs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_courant_final_batch, dim3(njobs), dim3(256), 0, s, jobs);
    return hipGetLastError();
}

// The level-independent constants of a Courant pass over several levels.
static CourantK courant_ml_k(double dx_finest, double gamma, double smallr, double smallc, double courant_factor,
                             const double g[3])
{
    CourantK c;
    c.dx = dx_finest;
    c.vol = 0.0;
    c.gamma = gamma;
    c.smallr = smallr;
    c.smallc = smallc;
    c.courant_factor = courant_factor;
    c.smallp = (smallc * smallc) / gamma;
    double gs = 0.0;
    for (int d = 0; d < 3; d++) gs = gs + __builtin_fabs(g[d]);
    c.gsum_dx = gs;  // times dx per oct in the kernel
    c.ndim = 3;
    return c;
}

hipError_t launch_courant_ml(const double *uold, const uint8_t *refined, const int32_t *lev, int head, int noct,
                             double boxlen, double dx_finest, double gamma, double smallr, double smallc,
                             double courant_factor, const double g[3], double *partials, int max_blocks, double *out,
                             double *dt_out, hipStream_t s, double *t_acc, bool mixed)
{
    const CourantK c = courant_ml_k(dx_finest, gamma, smallr, smallc, courant_factor, g);
    const long ncell = (long)noct * 8;
    int nb = (int)((ncell + kCourantThreads - 1) / kCourantThreads);
    nb = nb < max_blocks ? nb : max_blocks;
    nb = nb < 1 ? 1 : nb;
    if (mixed)
        hipLaunchKernelGGL(k_courant_ml<true>, dim3(nb), dim3(kCourantThreads), 0, s, uold, refined, lev, head, noct, c,
                           boxlen, partials);
    else
        hipLaunchKernelGGL(k_courant_ml<false>, dim3(nb), dim3(kCourantThreads), 0, s, uold, refined, lev, head, noct,
                           c, boxlen, partials);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_courant_final, dim3(1), dim3(256), 0, s, partials, nb, dx_finest / smallc, out, dt_out,
                       t_acc, 1);
    return hipGetLastError();
}

hipError_t launch_upload_courant(double *uold, const uint8_t *refined, const UploadLevel *lv, int nlev, double boxlen,
                                 double dx_finest, double gamma, double smallr, double smallc, double courant_factor,
                                 const double g[3], double *partials, int max_parts, double *out, double *dt_out,
                                 hipStream_t s, double *t_acc, bool mixed)
{
    const CourantK c = courant_ml_k(dx_finest, gamma, smallr, smallc, courant_factor, g);
    int first = 0;
    for (int i = nlev - 1; i >= 0; i--) {
        // as many blocks as an even share of the partials allows
        const int cap = max_parts / nlev > 1 ? max_parts / nlev : 1;
        int nb = (lv[i].noct + 31) / 32;
        nb = nb < cap ? nb : cap;
        if (nb < 1) continue;
        if (mixed)
            hipLaunchKernelGGL(k_upload_courant<true>, dim3(nb), dim3(kCourantThreads), 0, s, uold, refined,
                               lv[i].father, lv[i].head, lv[i].noct, lv[i].level, c, boxlen, partials + 4 * first);
        else
            hipLaunchKernelGGL(k_upload_courant<false>, dim3(nb), dim3(kCourantThreads), 0, s, uold, refined,
                               lv[i].father, lv[i].head, lv[i].noct, lv[i].level, c, boxlen, partials + 4 * first);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        first += nb;
    }
    hipLaunchKernelGGL(k_courant_final, dim3(1), dim3(256), 0, s, partials, first, dx_finest / smallc, out, dt_out,
                       t_acc, 1);
    return hipGetLastError();
}

hipError_t launch_zero(double *p, long n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    long nb = (n + 255) / 256;
    nb = nb < 4096 ? nb : 4096;
    hipLaunchKernelGGL(k_zero, dim3((unsigned)nb), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

hipError_t launch_reflux_fold(double *unew, double *racc, const int32_t *ghost_parent, const int32_t *order,
                              int nghost, int ttd, hipStream_t s, int nslot)
{
    if (nghost <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_reflux_fold, dim3((unsigned)((5l * nghost + 255) / 256)), dim3(256), 0, s, unew, racc, ghost_parent, order,
                       nghost, ttd, nslot);
    return hipGetLastError();
}

hipError_t launch_courant(const double *uold, const uint8_t *refined, int head, int noct, int ndim, double dx,
                          double gamma, double smallr, double smallc, double courant_factor, const double g[3],
                          double *partials, int max_blocks, double *out, double *dt_out, hipStream_t s,
                          double *t_acc)
{
    CourantK c;
    c.dx = dx;
    c.vol = ndim == 1 ? dx : dx * dx * dx;
    c.gamma = gamma;
    c.smallr = smallr;
    c.smallc = smallc;
    c.courant_factor = courant_factor;
    c.smallp = (smallc * smallc) / gamma;
    double gs = 0.0;
    for (int d = 0; d < ndim; d++) gs = gs + __builtin_fabs(g[d]);
    c.gsum_dx = gs * dx;
    c.ndim = ndim;
    const int ttd = 1 << ndim;
    const long ncell = (long)noct * ttd;
    int nb = (int)((ncell + kCourantThreads - 1) / kCourantThreads);
    if (nb > max_blocks) nb = max_blocks;
    if (nb < 1) nb = 1;
    if (ttd == 8)
        hipLaunchKernelGGL(k_courant<8>, dim3(nb), dim3(kCourantThreads), 0, s, uold, refined, head, noct, c, partials);
    else
        hipLaunchKernelGGL(k_courant<2>, dim3(nb), dim3(kCourantThreads), 0, s, uold, refined, head, noct, c, partials);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_courant_final, dim3(1), dim3(256), 0, s, partials, nb, dx / smallc, out, dt_out, t_acc, 0);
    return hipGetLastError();
}

}  // namespace rh
