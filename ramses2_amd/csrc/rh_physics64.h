// FP64 physics of the brick kernels: the routines of rh_physics.h in forms that
// take fewer instructions.  The FP64 kernels are bound by the issue of their
// vector instructions, so each routine here is written for its count of issue
// slots and the length of its dependent chain; the results agree with the
// reference's expressions to rounding.  (The mixed-precision kernels use
// rh_physics.h: their FP32 results depend on every rounding.)
//
// Contraction is off and every FMA written out: the compiler otherwise contracts
// the same expression differently from one copy of the code to the next (a
// peeled first iteration, another brick shape), and a plane's bits would depend
// on where a march begins.
#pragma once
#include "rh_physics.h"

namespace rh {

__device__ __forceinline__ double tfma(double a, double b, double c) { return __builtin_fma(a, b, c); }

// Maximum and minimum of values that a load or another block of code produced:
// the instruction alone.  fmax and fmin quiet such an operand first (it could be
// a signalling NaN), one more instruction each, 113 in the two planes of a 3D HLLC
// march; of a quiet NaN and a number both forms give the number.  The 256^3 kernel takes
// 646 us with fmax and fmin throughout, 637 with these, 8x6x8 bricks at 128^3 98.7
// and 97.9.  Not for operands of cross-lane moves, for which the compiler counts
// wait states.
__device__ __forceinline__ double vmax(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// the same with a value uniform in the wave
__device__ __forceinline__ double vmax_u(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "s"(b));
    return r;
}
__device__ __forceinline__ double vmin(double a, double b)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// max(a, 0) and min(a, 0)
__device__ __forceinline__ double vmax0(double a)
{
    double r;
    asm("v_max_f64 %0, %1, 0" : "=v"(r) : "v"(a));
    return r;
}
__device__ __forceinline__ double vmin0(double a)
{
    double r;
    asm("v_min_f64 %0, %1, 0" : "=v"(r) : "v"(a));
    return r;
}
// max(|a|, |b|) and min(|a|, b)
__device__ __forceinline__ double vmax_abs(double a, double b)
{
    double r;
    asm("v_max_f64 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double vmin_abs(double a, double b)
{
    double r;
    asm("v_min_f64 %0, |%1|, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// 1/b from the hardware reciprocal (about 2^-24) refined by one third-order
// step, r (1 + e + e^2) with e = 1 - b r: three dependent FMAs instead of the
// four of two Newton steps (rcp_nr), the remaining error e^3 far below an ulp, so
// the result is off by its last rounding only.
__device__ __forceinline__ double rcp_h(double b)
{
    const double r = __builtin_amdgcn_rcp(b);
    const double e = __builtin_fma(-b, r, 1.0);
    return __builtin_fma(r, __builtin_fma(e, e, e), r);
}
// 1/sqrt(x) for x in [2^-1020, 2^1020]: the hardware reciprocal square root
// refined by one third-order step, y (1 + e/2 + 3 e^2/8) with e = 1 - x y^2
// (five dependent operations; the remaining error is of the order of e^3).
__device__ __forceinline__ double rsq_pos(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double e = __builtin_fma(-(x * y), y, 1.0);
    return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}
// max(sqrt(g na/da), sqrt(g nb/db)) for positive operands without a division: the
// larger quotient is found by cross multiplication, and sqrt(n/d) = n/sqrt(n d)
// takes one refined reciprocal square root.  Two sound speeds of a face cost
// 19 issue slots this way against 35 as two refined reciprocals and a square
// root.  The products are floored where sqrt would leave the normal range.
__device__ __forceinline__ double sqrt_quot_max(double na, double da, double nb, double db, double g)
{
    const bool a = na * db > nb * da;
    const double n = g * (a ? na : nb), d = a ? da : db;
    return n * rsq_pos(__builtin_fmax(n * d, 0x1p-1020));
}
// sqrt(n/d): a sound speed from gamma*P and rho
__device__ __forceinline__ double sound_speed64(double n, double d)
{
    return n * rsq_pos(__builtin_fmax(n * d, 0x1p-1020));
}

// ctoprim (prim_from_cons) of one cell: m = rho v gives the kinetic energy as
// m.v/2, three operations fewer.  Returns 1/rho, which the predictor of the
// same cell uses again.
__device__ __forceinline__ double prim64(const double u[5], double q[5], double smallr, double smalle, double gm1,
                                         const double gdt_half[3])
{
#pragma clang fp contract(off)
    const double r = tmax(u[0], smallr);
    const double ir = rcp_h(r);
    const double vx = u[1] * ir, vy = u[2] * ir, vz = u[3] * ir;
    const double s = __builtin_fma(u[3], vz, __builtin_fma(u[2], vy, u[1] * vx));
    q[0] = r;
    q[1] = vx + gdt_half[0];
    q[2] = vy + gdt_half[1];
    q[3] = vz + gdt_half[2];
    q[4] = gm1 * tmax(__builtin_fma(-0.5, s, u[4]), smalle * r);
    return ir;
}

// uslope (slope_half) from the differences a = q0-qm1 and b = qp1-q0, halved:
// MinMod is half the median of a, b and 0; MonCen is the centred slope clamped
// to [min(max(a,b),0), max(min(a,b),0)], an interval that is [0, min] or
// [max, 0] where a and b agree in sign and only 0 where they do not.  min and
// max are exact, so the values are those of slope_half, one or two
// instructions sooner.
__device__ __forceinline__ double slope64(int st, double a, double b)
{
    const double lo = vmin(a, b), hi = vmax(a, b);
    if (st == 1) return 0.5 * vmax(lo, vmin0(hi));
    const double c = (a + b) * 0.25;  // dcen/2
    return vmax(vmin(c, vmax0(lo)), vmin0(hi));
}
// vel_bound_half from the same differences
__device__ __forceinline__ double vel_bound64(double dqh, double rl, double a, double inv_r0, double rr, double b)
{
    const double lim = tmin(rl * fabs_(a), rr * fabs_(b)) * inv_r0;
    return tcopysign(vmin_abs(dqh, lim), dqh);
}

// trace3d, hydro/umuscl.f90:860-1466, hydro part for one cell.
// q: cell primitives; dqh[d][n]: halved slopes (the reference's 0.5*dq).
// Outputs qp[d][n] (right state at the left interface) and qm[d][n] (left
// state at the right interface).  hr, hp: max |dqh[d][0]| and max |dqh[d][4]|.
__device__ __forceinline__ void trace64(const double q[5], const double dqh[3][5], double qp[3][5], double qm[3][5],
                                        const HydroK<double> &k, double inv_r, double hr, double hp)
{
#pragma clang fp contract(off)
    using T = double;
    T r = q[0], u = q[1], v = q[2], w = q[3], p = q[4];
    T drx = dqh[0][0], dux = dqh[0][1], dvx = dqh[0][2], dwx = dqh[0][3], dpx = dqh[0][4];
    T dry = dqh[1][0], duy = dqh[1][1], dvy = dqh[1][2], dwy = dqh[1][3], dpy = dqh[1][4];
    T drz = dqh[2][0], duz = dqh[2][1], dvz = dqh[2][2], dwz = dqh[2][3], dpz = dqh[2][4];
    T divv = dux + dvy + dwz;
    // -(v . grad) of each variable
    auto adv = [&](T dx, T dy, T dz) { return tfma(-w, dz, tfma(-v, dy, -u * dx)); };
    T ws[5];
    ws[0] = tfma(tfma(-r, divv, adv(drx, dry, drz)), k.dtdx, r);
    ws[1] = tfma(tfma(-inv_r, dpx, adv(dux, duy, duz)), k.dtdx, u);
    ws[2] = tfma(tfma(-inv_r, dpy, adv(dvx, dvy, dvz)), k.dtdx, v);
    ws[3] = tfma(tfma(-inv_r, dpz, adv(dwx, dwy, dwz)), k.dtdx, w);
    ws[4] = tfma(tfma(-(divv * k.gamma), p, adv(dpx, dpy, dpz)), k.dtdx, p);
#pragma unroll
    for (int d = 0; d < 3; d++) {
#pragma unroll
        for (int n = 0; n < 5; n++) {
            T h = dqh[d][n];
            qp[d][n] = ws[n] - h;
            qm[d][n] = ws[n] + h;
        }
    }
    // The floors (a state below smallr or smallp falls back to the cell's
    // value) rarely bite.  The smallest of the six states is ws - max|h|
    // (rounding is monotonic, so the test is exact): a wave without a floored
    // state skips the 12 compares and 24 selects.
    if (__builtin_expect(ws[0] - hr < k.smallr || ws[4] - hp < k.smallp_trace, 0)) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            if (qp[d][0] < k.smallr) qp[d][0] = r;
            if (qp[d][4] < k.smallp_trace) qp[d][4] = p;
            if (qm[d][0] < k.smallr) qm[d][0] = r;
            if (qm[d][4] < k.smallp_trace) qm[d][4] = p;
        }
    }
}

// riemann_hllc, hydro/godunov_utils.f90:638-857 (mass, momenta, energy fluxes).
// Only the star state and the energy of the side that is sampled are formed;
// the sampled values are those of the reference, which forms both.  The states
// come from trace64, whose densities are at least smallr, and with the pressure
// floor (hllc_floor) no sound speed is below smallc, so those two floors of the
// reference's are not repeated but for the right density, which turns a lost state
// there into one whose sound speed is no NaN (sqrt_quot_max takes the right one
// where the comparison is false): the upwind side of a supersonic face is then
// selected whatever the other holds.  Selecting the side's state costs the 256^3 kernel
// 1.4% against forming it by the star formulas (653 -> 663 us).
__device__ __forceinline__ void hllc64(const double ql[5], const double qr[5], double f[5], const HydroK<double> &k)
{
#pragma clang fp contract(off)
    using T = double;
    const T half = T(0.5);
    T rl = ql[0];
    T ul = ql[1], vl = ql[2], wl = ql[3];
    T Pl = vmax(ql[4], rl * k.smallp_riem);
    T rr = vmax_u(qr[0], k.smallr);
    T ur = qr[1], vr = qr[2], wr = qr[3];
    T Pr = vmax(qr[4], rr * k.smallp_riem);
    // max(sqrt(a), sqrt(b)) = sqrt(max(a, b)): one root for the two sound speeds
    T cmax = sqrt_quot_max(Pl, rl, Pr, rr, k.gamma);
    T SL = vmin(ul, ur) - cmax;
    T SR = vmax(ul, ur) + cmax;
    T dl = ul - SL, dr = SR - ur;
    T rcl = rl * dl, rcr = rr * dr;
    T den = tfma(rr, dr, rcl);
    T num = (Pl - Pr) + tfma(rcr, ur, rcl * ul);
    // The reference samples, in this order: SL > 0 -> left state; ustar > 0
    // -> left star state; SR > 0 -> right star state; else right state.  The
    // side whose values are used is left exactly when SL > 0 or ustar > 0,
    // and the star state is taken when SL <= 0 and (ustar > 0 or SR > 0); in
    // both star cases the side is the reference's ustar > 0.  So one select
    // of the side's values and one of four values (state or star) give the
    // reference's result (its chain costs three selects per value), and the
    // total energy is formed for that side only.
    //
    // The side's state has to be selected: the star state's formulas return it
    // too when given the side's own velocity and pressure, but only to a rounding of
    // S - us, which loses a factor |u|/c, and all of it where the sound speed is
    // below half an ulp of the velocity.  There den and num can be 0 and the star
    // state NaN, which the selects discard.  ustar = num/den has the sign of num
    // where den > 0, and is no positive number where den = 0.
    const bool sl_pos = SL > T(0), us_pos = num > T(0) && den > T(0);
    const bool left = sl_pos || us_pos;
    const bool star = !sl_pos && (us_pos || SR > T(0));
    T S = left ? SL : SR;
    T rs = left ? rl : rr, us = left ? ul : ur, Ps = left ? Pl : Pr;
    T vo = left ? vl : vr, wo = left ? wl : wr;
    T es = tfma(half * rs, tfma(wo, wo, tfma(us, us, vo * vo)), Ps * k.entho);
    T ds = S - us;
    // 1/den and 1/(S - ustar) = den/(S den - num) from one reciprocal: the
    // hardware one takes four issue slots, and the two would depend on each other
    T t = tfma(S, den, -num);
    T ri = rcp_h(den * t);
    T inv_den = ri * t, inv_sd = (ri * den) * den;
    T un = num * inv_den;
    T Pn = tfma(rcl * rcr, ul - ur, tfma(rcr, Pl, rcl * Pr)) * inv_den;
    T uo = star ? un : us, Po = star ? Pn : Ps;
    T ro = star ? rs * ds * inv_sd : rs;
    T eo = star ? tfma(Pn, un, tfma(ds, es, -(Ps * us))) * inv_sd : es;
    f[0] = ro * uo;
    f[1] = tfma(f[0], uo, Po);
    f[2] = f[0] * vo;
    f[3] = f[0] * wo;
    f[4] = (eo + Po) * uo;
}
// The pressure floor of hllc64: smallc^2/gamma, and where smallc is (nearly) 0 that
// of a sound speed of 2^-300, so that for gas at rest without pressure den and the
// product under the reciprocal, of the order of rho^2 c^3, stay in range.
__device__ __forceinline__ double hllc_floor(const HydroK<double> &k)
{
    return tmax(k.smallc2, 0x1p-600) / k.gamma;
}

// Conservative state and physical flux of one side (side_state).
__device__ __forceinline__ void side64(const double q[5], double entho, double u[5], double f[5])
{
#pragma clang fp contract(off)
    const double ke = tfma(q[3], q[3], tfma(q[2], q[2], q[1] * q[1]));
    u[0] = q[0];
    u[1] = q[0] * q[1];
    u[2] = q[0] * q[2];
    u[3] = q[0] * q[3];
    u[4] = tfma(0.5 * q[0], ke, q[4] * entho);
    f[0] = u[1];
    f[1] = tfma(q[1], u[1], q[4]);
    f[2] = q[1] * u[2];
    f[3] = q[1] * u[3];
    f[4] = q[1] * (u[4] + q[4]);
}

// riemann_llf, hydro/godunov_utils.f90:338-485.
__device__ __forceinline__ void llf64(const double ql[5], const double qr[5], double f[5], const HydroK<double> &k)
{
#pragma clang fp contract(off)
    const double pl = vmax(ql[4], ql[0] * k.smallp_riem), pr = vmax(qr[4], qr[0] * k.smallp_riem);
    const double cl = sound_speed64(k.gamma * pl, ql[0]), cr = sound_speed64(k.gamma * pr, qr[0]);
    const double cmax = tmin(tmax(fabs_(ql[1]) + cl, fabs_(qr[1]) + cr), k.smax_cap);
    double uL[5], uR[5], fL[5], fR[5];
    side64(ql, k.entho, uL, fL);
    side64(qr, k.entho, uR, fR);
#pragma unroll
    for (int n = 0; n < 5; n++) f[n] = 0.5 * tfma(-cmax, uR[n] - uL[n], fL[n] + fR[n]);
}

// riemann_hll, hydro/godunov_utils.f90:486-637.
__device__ __forceinline__ void hll64(const double ql[5], const double qr[5], double f[5], const HydroK<double> &k)
{
#pragma clang fp contract(off)
    const double ul = ql[1], ur = qr[1];
    const double pl = vmax(ql[4], ql[0] * k.smallp_riem), pr = vmax(qr[4], qr[0] * k.smallp_riem);
    const double cmax = sqrt_quot_max(pl, ql[0], pr, qr[0], k.gamma);
    const double SL = tmax(tmin(vmin(ul, ur) - cmax, 0.0), -k.smax_cap);
    const double SR = tmin(tmax(vmax(ul, ur) + cmax, 0.0), k.smax_cap);
    double uL[5], uR[5], fL[5], fR[5];
    side64(ql, k.entho, uL, fL);
    side64(qr, k.entho, uR, fR);
    const double inv = rcp_h(SR - SL), ss = SR * SL;  // SR - SL >= 2c > 0, the same for all five
#pragma unroll
    for (int n = 0; n < 5; n++) f[n] = tfma(ss, uR[n] - uL[n], tfma(SR, fL[n], -(SL * fR[n]))) * inv;
}

// cmpflxm for the solver RS (1 LLF, 2 HLL, 3 HLLC) with states already rotated
// to the face normal: (rho, u_n, u_t1, u_t2, p).
template <int RS> __device__ __forceinline__ void solve64(const double a[5], const double b[5], double g[5], const HydroK<double> &k)
{
    if constexpr (RS == 3)
        hllc64(a, b, g, k);
    else if constexpr (RS == 2)
        hll64(a, b, g, k);
    else
        llf64(a, b, g, k);
}
template <int RS>
__device__ __forceinline__ void face64(int idim, const double ql[5], const double qr[5], double f[5],
                                       const HydroK<double> &k)
{
    const int ln = idim + 1, lt1 = idim == 0 ? 2 : 1, lt2 = idim == 2 ? 2 : 3;
    const double a[5] = {ql[0], ql[ln], ql[lt1], ql[lt2], ql[4]};
    const double b[5] = {qr[0], qr[ln], qr[lt1], qr[lt2], qr[4]};
    double g[5];
    solve64<RS>(a, b, g, k);
    f[0] = g[0];
    f[ln] = g[1];
    f[lt1] = g[2];
    f[lt2] = g[3];
    f[4] = g[4];
}

}  // namespace rh
