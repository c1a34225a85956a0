// Device-resident steps of a small 1D level in one workgroup (FP64).
//
// A 1D level of up to kTubeCells cells takes next to no time to compute, so a
// step launched as Courant pass, its final reduction and the update is the
// latency of three dependent launches (15 us).  Here one workgroup holds the
// level: the state stays in registers, primitives, left states and fluxes pass
// through LDS, and all steps of a call run in one launch with three barriers
// each.  What bounds a step is its dependent chain (conversion, dt reduction,
// slopes, Riemann solve), at 1024 cells also the issue of one CU.  Measured,
// MinMod + HLLC, 2000 steps a call: 64 cells 13.4 -> 1.5 us per step, 512 14.3 ->
// 2.4, 1024 14.4 -> 3.8.  Beyond, with four cells per thread, it spilled and took 16
// us, no less than the launches (14.6).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rh_courant.h"
#include "rh_godunov.h"

namespace rh {

// trace1d (trace1 of rh_physics.h) with its FMAs written out.
__device__ __forceinline__ void trace1_64(const double q[5], const double h[5], double qp[5], double qm[5],
                                          const HydroK<double> &k, double inv_r)
{
#pragma clang fp contract(off)
    const double r = q[0], u = q[1], p = q[4];
    const double s[5] = {tfma(-h[1], r, -u * h[0]), tfma(-inv_r, h[4], -u * h[1]), -u * h[2], -u * h[3],
                         tfma(-(h[1] * k.gamma), p, -u * h[4])};
#pragma unroll
    for (int n = 0; n < 5; n++) {
        const double ws = tfma(s[n], k.dtdx, q[n]);
        qp[n] = ws - h[n];
        qm[n] = ws + h[n];
    }
    if (qp[0] < k.smallr) qp[0] = r;
    if (qp[4] < k.smallp_trace) qp[4] = p;
    if (qm[0] < k.smallr) qm[0] = r;
    if (qm[4] < k.smallp_trace) qm[4] = p;
}

// Largest of the wave's non-negative values, in every lane: 0 is the value of
// lanes a shift leaves without a source.
template <int CTRL, int ROWMASK> __device__ __forceinline__ double dpp_max(double x)
{
    const int64_t b = __builtin_bit_cast(int64_t, x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWMASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWMASK, 0xf, false);
    return tmax(x, __builtin_bit_cast(double, ((int64_t)hi << 32) | (uint32_t)lo));
}
__device__ __forceinline__ double wave_max_dpp(double x)
{
    x = dpp_max<0x111, 0xf>(x);  // row_shr:1, 2, 4, 8
    x = dpp_max<0x112, 0xf>(x);
    x = dpp_max<0x114, 0xf>(x);
    x = dpp_max<0x118, 0xf>(x);
    x = dpp_max<0x142, 0xa>(x);  // row_bcast:15 into rows 1 and 3
    x = dpp_max<0x143, 0xc>(x);  // row_bcast:31 into rows 2 and 3
    const int64_t b = __builtin_bit_cast(int64_t, x);
    const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __builtin_bit_cast(double, ((int64_t)hi << 32) | (uint32_t)lo);
}

struct TubeArgs {
    God1Args g;        // uold, unew: the level's arrays (both receive the final state)
    int nsteps;
    int sums;          // write the sums and dt of the last step to out, dt_dev
    double dt_fixed;   // > 0: the dt of every step
    double *out, *dt_dev, *t_dev;
};

// Cells of a level held by one workgroup: K per thread of up to 512 threads, and
// one wave more whose first two lanes hold the ghost cells beyond the ends of
// the level (in the cells' own waves their extra states and the last face's
// solve lengthened every step).  120 bytes of LDS per cell.
constexpr int kTubeThreads = 512, kTubeCells = 1024;

template <int RS, int K> __global__ void __launch_bounds__(kTubeThreads + 64) k_tube(const TubeArgs t)
{
#pragma clang fp contract(off)
    const God1Args &a = t.g;
    extern __shared__ double lds[];
    __shared__ double red[2][16], red3[3][16];
    __shared__ int endcell[2];
    constexpr int ld = K * kTubeThreads + 2;  // entries ld-2, ld-1: beyond the ends
    const int n = 2 * a.noct, nt = blockDim.x - 64, tid = threadIdx.x, nw = nt >> 6;
    double *sq = lds, *sm = lds + 5 * ld, *sf = lds + 10 * ld;  // primitives, left states, low-face fluxes
    const double gm1 = a.gamma - 1.0, smalle = a.smallc2 / a.gamma / gm1;
    const double gv[3] = {a.g, 0.0, 0.0}, gz[3] = {0.0, 0.0, 0.0};
    const CourantK ck = make_courant_k(a.dx, 1, a.gamma, a.smallr, a.smallc2, a.courant_factor, gv);
    HydroK<double> k = make_k<double>(1.0, a.dx, a.gamma, a.smallr, a.smallc2, a.courant_factor, a.smax_cap, a.use_smax,
                                      a.slope < 2 ? a.slope : 2, a.riemann);
    if constexpr (RS == 3) k.smallp_riem = hllc_floor(k);
    // signal_dt without gravity, its constants taken out of the steps
    const double dtn = 2.0 * ck.courant_factor * ck.dx, gf = 1.0 + __builtin_sqrt(1.0 + 2.0 * ck.courant_factor * 0.0001);
    const double dtcap = ck.courant_factor * ck.dx / ck.smallc, dtmax = a.dx / ck.smallc;
    const bool courant = t.dt_fixed <= 0.0;
    const bool end = tid >= nt;  // the wave of the level's ends
    if (tid < 2) endcell[tid] = -1;
    __syncthreads();

    // this thread's cells: state; neighbours' entries in sq (a ghost cell reads
    // the cell it copies, the velocity negated where nl / nr is set), in sm and
    // in sf
    double u[K][5];
    int lq[K], rq[K], lm[K], rf[K];
    bool have[K], leaf[K], zl[K], zr[K], nl[K], nr[K];
#pragma unroll
    for (int j = 0; j < K; j++) {
        const int c = tid + j * nt;
        have[j] = !end && c < n;
        const int li = have[j] ? c >> 1 : 0, i2 = c & 1, self = have[j] ? c : 0;
        const int v = a.nbor[(size_t)li * 3 + (i2 ? 2 : 0)];  // the oct on the cell's outer side
        const double *p = a.uold + (size_t)(a.head - 1 + li) * 10 + i2;
#pragma unroll
        for (int m = 0; m < 5; m++) u[j][m] = p[2 * m];
        const uint8_t *rfl = a.refined + (size_t)(a.head - 1 + li) * 8;
        // an oct of the level, or a boundary ghost of the oct -v, whose inner
        // cell copies that oct's outer cell
        const int w = (v > 0 ? v : -v) - a.head;
        const bool ok = w >= 0 && w < a.noct;
        const int outer = ok ? 2 * w + (v > 0 ? 1 - i2 : i2) : self;
        const bool rn = ok && a.refined[(size_t)(a.head - 1 + w) * 8 + (v > 0 ? 1 - i2 : i2)] != 0;
        const bool neg = v < 0 && a.btype[i2] == 1;
        lq[j] = i2 ? self - 1 : outer;
        rq[j] = i2 ? outer : self + 1;
        if (!have[j]) lq[j] = rq[j] = 0;
        lm[j] = i2 == 0 && v < 0 ? ld - 2 : lq[j];
        rf[j] = i2 == 1 && v < 0 ? ld - 1 : rq[j];
        nl[j] = i2 == 0 && neg;
        nr[j] = i2 == 1 && neg;
        leaf[j] = have[j] && !rfl[i2];
        zl[j] = rfl[i2] || (i2 ? rfl[0] != 0 : rn);
        zr[j] = rfl[i2] || (i2 ? rn : rfl[1] != 0);
        if (have[j] && v < 0) endcell[i2] = c;
    }
    __syncthreads();
    // end wave: lane 0 the low, lane 1 the high end (side = lane)
    const int side = tid & 1, ec = end && (tid & 63) < 2 ? endcell[side] : -1;
    const bool mirror = a.btype[side] == 1;
    // the two ghost cells copy the end cell, or mirror it and the one inside
    const int e1 = ec >= 0 ? ec : 0, e2 = mirror && ec >= 0 ? (ec ^ 1) : e1;

    double dt = t.dt_fixed, time = 0.0;
    for (int s = 0; s < t.nsteps; s++) {
        // ---- primitives, largest signal speed ----
        double q[K][5], ir[K], sig = 0.0;
        if (!end) {
#pragma unroll
            for (int j = 0; j < K; j++) {
                ir[j] = prim64(u[j], q[j], a.smallr, smalle, gm1, gz);
                // the signal speed of cmpdt from the primitives at hand
                const double x = fabs_(q[j][1]) + sound_speed64(a.gamma * q[j][4], q[j][0]);
                sig = leaf[j] ? tmax(sig, x) : sig;
                if (have[j])
#pragma unroll
                    for (int m = 0; m < 5; m++) sq[m * ld + tid + j * nt] = q[j][m];
            }
            if (courant) {
                sig = wave_max_dpp(sig);
                if ((tid & 63) == 0) red[s & 1][tid >> 6] = sig;
            }
        }
        __syncthreads();
        if (courant) {
            const int l = tid & 63;
            sig = wave_max_dpp(l < nw ? red[s & 1][l] : 0.0);
            dt = ck.gsum_dx != 0.0 ? signal_dt(sig, ck) : tmin(dtn / (sig * gf), dtcap);
            dt = sig > 0.0 ? tmin(dt, dtmax) : dtmax;
        }
        time += dt;
        const double c = dt * a.inv_dx, gk = a.g * (dt * 0.5);
        k.dtdx = c;
        if (RS != 3) k.smax_cap = a.use_smax ? a.smax_cap : a.courant_factor * a.dx * rcp_h(dt);
        // halved slopes of a cell from its neighbours' primitives (the gravity
        // kick is the same in all cells), then the two face states
        auto trace = [&](const double qm1[5], const double q0[5], const double qp1[5], double ir0, double qp[5],
                         double qm[5]) __attribute__((always_inline)) {
            double h[5] = {0, 0, 0, 0, 0};
            if (k.slope_type) {
#pragma unroll
                for (int m = 0; m < 5; m++) h[m] = slope64(k.slope_type, q0[m] - qm1[m], qp1[m] - q0[m]);
                h[1] = vel_bound64(h[1], qm1[0], q0[1] - qm1[1], ir0, qp1[0], qp1[1] - q0[1]);
            }
            const double qk[5] = {q0[0], q0[1] + gk, q0[2], q0[3], q0[4]};
            trace1_64(qk, h, qp, qm, k, ir0);
        };
        double qp[K][5];
        if (!end) {
#pragma unroll
            for (int j = 0; j < K; j++) {
                double l[5], r[5], qm[5];
#pragma unroll
                for (int m = 0; m < 5; m++) {
                    l[m] = sq[m * ld + lq[j]];
                    r[m] = sq[m * ld + rq[j]];
                }
                l[1] = nl[j] ? -l[1] : l[1];
                r[1] = nr[j] ? -r[1] : r[1];
                trace(l, q[j], r, ir[j], qp[j], qm);
                if (have[j])
#pragma unroll
                    for (int m = 0; m < 5; m++) sm[m * ld + tid + j * nt] = qm[m];
            }
        } else if (ec >= 0) {
            double g1[5], g2[5], x[5], qm[5];
#pragma unroll
            for (int m = 0; m < 5; m++) {
                x[m] = sq[m * ld + ec];
                g1[m] = sq[m * ld + e1];
                g2[m] = sq[m * ld + e2];
            }
            g1[1] = mirror ? -g1[1] : g1[1];
            g2[1] = mirror ? -g2[1] : g2[1];
            double lo[5], hi[5];
#pragma unroll
            for (int m = 0; m < 5; m++) {
                lo[m] = side == 0 ? g2[m] : x[m];
                hi[m] = side == 0 ? x[m] : g2[m];
            }
            trace(lo, g1, hi, rcp_h(g1[0]), qp[0], qm);
            if (side == 0)
#pragma unroll
                for (int m = 0; m < 5; m++) sm[m * ld + ld - 2] = qm[m];
        }
        __syncthreads();
        double fl[K][5];
        if (!end) {
#pragma unroll
            for (int j = 0; j < K; j++) {
                double l[5];
#pragma unroll
                for (int m = 0; m < 5; m++) l[m] = sm[m * ld + lm[j]];
                face64<RS>(0, l, qp[j], fl[j], k);
                if (have[j])
#pragma unroll
                    for (int m = 0; m < 5; m++) sf[m * ld + tid + j * nt] = fl[j][m];
            }
        } else if (ec >= 0 && side == 1) {
            double l[5], f[5];
#pragma unroll
            for (int m = 0; m < 5; m++) l[m] = sm[m * ld + ec];
            face64<RS>(0, l, qp[0], f, k);
#pragma unroll
            for (int m = 0; m < 5; m++) sf[m * ld + ld - 1] = f[m];
        }
        if (t.sums && s == t.nsteps - 1) {
            // the conservation sums of the state before the last step
            double m = 0, e = 0, ei = 0;
#pragma unroll
            for (int j = 0; j < K; j++)
                if (leaf[j]) (void)courant_cell<1>(u[j], ck, ck.vol, m, e, ei);
            const double v3[3] = {wave_sum(m), wave_sum(e), wave_sum(ei)};
            if (!end && (tid & 63) == 0)
#pragma unroll
                for (int i = 0; i < 3; i++) red3[i][tid >> 6] = v3[i];
        }
        __syncthreads();
        if (!end)
#pragma unroll
            for (int j = 0; j < K; j++)
#pragma unroll
                for (int m = 0; m < 5; m++)
                    u[j][m] = tfma(c, (zl[j] ? 0.0 : fl[j][m]) - (zr[j] ? 0.0 : sf[m * ld + rf[j]]), u[j][m]);
    }
    if (!end)
#pragma unroll
        for (int j = 0; j < K; j++)
            if (have[j]) {
                const int cell = tid + j * nt;
                const size_t o = (size_t)(a.head - 1 + (cell >> 1)) * 10 + (cell & 1);
#pragma unroll
                for (int m = 0; m < 5; m++) {
                    const_cast<double *>(a.uold)[o + 2 * m] = u[j][m];
                    a.unew[o + 2 * m] = u[j][m];
                }
            }
    if (tid == 0) {
        *t.t_dev += time;
        if (t.sums) {
            for (int i = 0; i < 3; i++) {
                double x = 0;
                for (int w = 0; w < nw; w++) x += red3[i][w];
                t.out[i] = x;
            }
            t.out[3] = 0.0;
            t.out[4] = dt;
            *t.dt_dev = dt;
        }
    }
}

bool tube_fits(const God1Args &a)
{
    // a level that fills its box: no cell lacks a neighbour inside it, and at
    // most its two ends lie beyond
    return 2 * a.noct <= kTubeCells && a.noct == a.boxmax - a.boxmin && !a.reflux;
}

hipError_t launch_tube(const God1Args &a, int nsteps, double dt_fixed, double *out, double *dt_dev, double *t_dev,
                       hipStream_t s)
{
    const int n = 2 * a.noct;
    if (n <= 0 || nsteps <= 0) return hipSuccess;
    const bool two = n > kTubeThreads;
    const int nt = 64 + (two ? kTubeThreads : (n + 63) & ~63);
    const size_t bytes = (size_t)15 * ((two ? 2 : 1) * kTubeThreads + 2) * sizeof(double);
    auto run = [&](auto kernel) -> hipError_t {
        // beyond the 64 KB a launch may ask for by default
        hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return e;
        // launches of bounded length
        constexpr int kChunk = 4096;
        for (int k = 0; k < nsteps; k += kChunk) {
            const int m = nsteps - k < kChunk ? nsteps - k : kChunk;
            const TubeArgs t{a, m, dt_fixed <= 0.0 && k + m == nsteps, dt_fixed, out, dt_dev, t_dev};
            hipLaunchKernelGGL(kernel, dim3(1), dim3(nt), bytes, s, t);
        }
        return hipGetLastError();
    };
#define RH_TUBE(RS) (two ? run(k_tube<RS, 2>) : run(k_tube<RS, 1>))
    return a.riemann == 3 ? RH_TUBE(3) : a.riemann == 2 ? RH_TUBE(2) : RH_TUBE(1);
#undef RH_TUBE
}

}  // namespace rh
