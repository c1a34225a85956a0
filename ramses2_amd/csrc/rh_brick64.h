// FP64 brick kernel of the 3D Godunov update (slopes 0-2, one Riemann solver
// per instance; the 27-point slope and the mixed precision run brick_body of
// rh_godunov.hip).
//
// One workgroup per oct brick, one thread per column of the brick's cells plus
// one halo cell, marching along z.  Per plane tt there are two phases, each
// ended by a barrier:
//   A: the update of plane tt-1 from the x and y fluxes (the column's own low faces
//      in registers, its high faces in LDS), tt-2 final and stored; the own cell
//      of plane tt+1 converted to primitives, the loads of plane tt+2 issued;
//      slopes and Hancock predictor of plane tt, its left x and y states to LDS;
//   B: primitives of plane tt+1 to LDS (every slope of plane tt has read the
//      plane by now, so one plane is kept), and the Riemann problems of plane tt,
//      the x and y fluxes to LDS, the z fluxes into the update of plane tt-1.
// The states and the fluxes have buffers of their own: two barriers per plane
// instead of four when the fluxes overwrite the states, and the update's LDS
// latency overlaps the conversion and the slopes.
//
// The kernel is bound by the issue of its vector instructions at two waves per
// SIMD, so what counts is instructions per plane.  Where the 4 BX BY interior
// columns fill whole waves and the halo ring fits one more (8x6, 4x4 bricks),
// interior and halo waves run loops of their own (the role is uniform in a
// wave, both loops pass the same barriers): the interior loop has no ring
// loads, no divergent tests, and solves its three faces in straight line; the
// halo loop solves one face per lane, converts the ring and updates nothing.
// Measured in turn on one card against the one-body kernel this replaced (four
// barriers, every thread testing its role, the expressions of rh_physics.h), with
// the Courant reduction: 256^3 in 8x6x16 bricks 858 -> 668 us (25.1 G
// cell-updates/s, 2.0 TB/s of the 80 algorithmic bytes per cell; reading the column's
// own low faces back from LDS and two reciprocals per HLLC face cost another 3%),
// 128^3 in 8x6x8 bricks 135 -> 99 us, 90^3 MinMod + LLF (a run-time solver choice
// before) 107 -> 59 us.
#pragma once
#include <type_traits>

#include "rh_courant.h"
#include "rh_gather.h"

namespace rh {

// Waves per SIMD the kernel is built for: at three (168 VGPRs) it spills.
constexpr int kBrick64Waves = 2;

template <int BX, int BY> constexpr bool brick64_hw()
{
    return (4 * BX * BY) % 64 == 0 && (2 * BX + 2) * (2 * BY + 2) - 4 * BX * BY <= 64;
}

// LDS of one workgroup.  sacc (coarse-fine refluxes summed per window oct, one
// atomic per ghost oct at the end) is added where the workgroups of two waves
// per SIMD still fit the 160 KB of a CU with it.
template <int BX, int BY, int BZ, bool GEN> struct Brick64Core {
    static constexpr int CX = 2 * BX + 2, CY = 2 * BY + 2, NT = CX * CY, NI = 4 * BX * BY;
    static constexpr int NP = (2 * BX + 4) * (2 * BY + 4), NW = (BX + 2) * (BY + 2) * (BZ + 2);
    static constexpr int NFX = 2 * BY * (2 * BX + 1), NFY = 2 * BX * (2 * BY + 1);
    int32_t swin[NW];
    double sq[5][NP];                  // primitives of one plane
    double qx[5][NFX], qy[5][NFY];     // left states by face
    double fx[5][NFX], fy[5][NFY];     // fluxes by face
    double sun[5][NI];                 // new state of the lower plane of an oct layer
    double sub[GEN ? 1 : 2][5][GEN ? 1 : NI];  // conserved state of the last two planes (the update's base)
    uint8_t sref[GEN ? NW : 1];                // refined cells of each window oct (bit: cell)
};
template <int BX, int BY, int BZ, bool GEN> struct Brick64Lds : Brick64Core<BX, BY, BZ, GEN> {
    using Core = Brick64Core<BX, BY, BZ, GEN>;
    static constexpr int WGS = 4 * kBrick64Waves / ((Core::NT + 63) / 64) > 0 ? 4 * kBrick64Waves / ((Core::NT + 63) / 64) : 1;
    static constexpr bool RA =
        GEN && Core::NW <= 512 && sizeof(Core) + (size_t)Core::NW * 40 <= (size_t)160 * 1024 / WGS;
    double sacc[RA ? Core::NW : 1][5];
};

// The march over the z layers [zlo, zhi] of brick bid.  Courant partials go to
// cpart[4*pslot].  A: GodArgs, as a kernel argument or in the constant address
// space (a work-list descriptor).  KIND: which inputs the instance takes, see
// BrickKind.
template <int BX, int BY, int BZ, int RS, int KIND, typename A>
__device__ __forceinline__ void brick64(A &a, const int bid, const int zlo, const int zhi, const int pslot,
                                        Brick64Lds<BX, BY, BZ, KIND != kBrickUniform> &sm)
{
#pragma clang fp contract(off)
    constexpr bool GEN = KIND != kBrickUniform;
    // Phase A, whose LDS reads wait most, runs at a raised wave priority, so that
    // the CU's other workgroup fills its gaps with solves instead of delaying
    // it, where two workgroups (of four waves) share a CU: 8x6x16 at 256^3 646 -> 629
    // us, 8x6x8 at 128^3 104 -> 100, 7x7x8 at 128^3 135 -> 129.  With four workgroups
    // of two waves the raised ones starve the others (4x4x8 at 128^3 125 -> 136 us);
    // where one fills the CU there is none to yield to (256^3 without and with it:
    // 15x7x8 833 and 837 us, 15x7x16 788 and 782).
    constexpr bool kPrioA = Brick64Lds<BX, BY, BZ, GEN>::WGS == 2;
    constexpr int CX = 2 * BX + 2, CY = 2 * BY + 2, NT = CX * CY, NI = 4 * BX * BY;
    constexpr int PX = 2 * BX + 4;
    constexpr int WX = BX + 2, WY = BY + 2, NW = WX * WY * (BZ + 2);
    constexpr bool HW = brick64_hw<BX, BY>(), RA = Brick64Lds<BX, BY, BZ, GEN>::RA;
    const int tid = threadIdx.x;
    const bool rlds = RA && a.reflux && !a.rdet;
    if (RA && rlds)
        for (int i = tid; i < NW * 5; i += NT) (&sm.sacc[0][0])[i] = 0.0;
    const int ox0 = a.org[3 * bid + 0], oy0 = a.org[3 * bid + 1], oz0 = a.org[3 * bid + 2];
    const int tlo = 2 * zlo, thi = 2 * zhi + 1;

    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    HydroK<double> k = make_k<double>(dt, a.dx, a.gamma, a.smallr, a.smallc2, a.courant_factor, a.smax_cap,
                                      a.use_smax, a.slope, a.riemann);
    if constexpr (RS == 3) k.smallp_riem = hllc_floor(k);
    const double gm1 = a.gamma - 1.0, smalle = a.smallc2 / a.gamma / gm1;
    double gvec[3] = {0.0, 0.0, 0.0}, gdt[3] = {0.0, 0.0, 0.0};
    if constexpr (GEN)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            gvec[d] = a.g[d];
            gdt[d] = a.g[d] * (dt * 0.5);
        }
    // The fluxes stay unscaled; the update adds dt/dx times each difference of
    // the two faces of a dimension with one FMA, both cells of a face reading
    // the same flux, so the update conserves.  The reference's (F dt)/dx
    // (hydro/umuscl.f90:135-220) is formed only for the coarse reflux.
    const double dtdx = dt * a.inv_dx, dtdx8 = 0.125 * dtdx;
    const int boxmin[3] = {a.boxmin[0], a.boxmin[1], a.boxmin[2]};
    const int boxmax[3] = {a.boxmax[0], a.boxmax[1], a.boxmax[2]};
    const bool bnd = KIND == kBrickBounded && a.bnd != 0, reflux = GEN && a.reflux != 0;
    int refl = 0;
    if constexpr (GEN)
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int sd = 0; sd < 2; sd++) refl |= (a.btype[d][sd] == 1) << (2 * d + sd);
    const CourantK ck = make_courant_k(a.dx, 3, a.gamma, a.smallr, a.smallc2, a.courant_factor, gvec);
    const bool courant = a.courant != 0;
    double c_mass = 0.0, c_ekin = 0.0, c_eint = 0.0, c_sig = 0.0;
    // The window, and the refined cells of its octs as one byte each: the flags
    // of a face's cells are then two LDS bytes away, and a brick without any
    // refined cell skips them (a flag per cell, fetched, staged and read with
    // the plane's primitives, cost a refined mesh 6%).
    bool mine = false;
    for (int i = tid; i < NW; i += NT) {
        const int v = a.win[(size_t)bid * NW + i];
        sm.swin[i] = v;
        if constexpr (GEN) {
            int m = 0;
            if (a.any_ref && v > 0) {
                const uint64_t f = *(const uint64_t *)(a.refined + (size_t)(v - 1) * 8);
#pragma unroll
                for (int ind = 0; ind < 8; ind++) m |= ((f >> (8 * ind)) & 0xff) != 0 ? 1 << ind : 0;
            } else if (bnd && a.any_ref && v < 0) {
                const int okey[3] = {ox0 + i % WX - 1, oy0 + i / WX % WY - 1, oz0 + i / (WX * WY) - 1};
                for (int ind = 0; ind < 8; ind++) {
                    const int c[3] = {ind & 1, (ind >> 1) & 1, ind >> 2};
                    const uint8_t *rf = cell_ref3(a.uold, a.refined, v, okey, boxmin, boxmax, refl, c).rf;
                    if (rf && *rf) m |= 1 << ind;
                }
            }
            sm.sref[GEN ? i : 0] = (uint8_t)m;
            mine = mine || m != 0;
        }
    }
    const bool anyref = GEN && __syncthreads_or(mine);
    if (!GEN) __syncthreads();

    // ROLE 1: a column of the brick's interior; 2: a column of the halo ring;
    // 0: either, tested per thread (shapes whose interior does not fill waves)
    auto run = [&](auto role) __attribute__((always_inline)) {
        constexpr int ROLE = decltype(role)::value;
        int cx, cy;
        if constexpr (ROLE == 1) {
            cx = tid % (2 * BX);
            cy = tid / (2 * BX);
        } else if constexpr (ROLE == 2) {
            const int h = tid - NI;
            if (h < 2 * CX) {
                cx = (h < CX ? h : h - CX) - 1;
                cy = h < CX ? -1 : 2 * BY;
            } else {
                const int g = h - 2 * CX;
                cx = g < 2 * BY ? -1 : 2 * BX;
                cy = g < 2 * BY ? g : g - 2 * BY;
            }
        } else {
            cx = tid % CX - 1;
            cy = tid / CX - 1;
        }
        const bool inx = ROLE == 1 || (cx >= 0 && cx < 2 * BX), iny = ROLE == 1 || (cy >= 0 && cy < 2 * BY);
        const bool interior = ROLE == 1 || (ROLE == 0 && inx && iny);
        // faces: the column's low x and y faces are solved by it, its left
        // states belong to its high faces
        const bool do_fx = ROLE == 1 || (iny && cx >= 0), do_fy = ROLE == 1 || (inx && cy >= 0);
        const bool has_qx = ROLE == 1 || (iny && cx < 2 * BX), has_qy = ROLE == 1 || (inx && cy < 2 * BY);
        const int pc = (cy + 2) * PX + (cx + 2);
        // x face f of row cy: the first 2BX faces row by row, then the last
        // faces of all rows (the rows of a wave stay 2BX doubles apart)
        const int ixl = (ROLE != 1 && cx == 2 * BX) ? NI + cy : cy * (2 * BX) + cx;
        const int ixh = cx == 2 * BX - 1 ? NI + cy : cy * (2 * BX) + cx + 1;
        const int iyl = cy * (2 * BX) + cx, iyh = iyl + 2 * BX;
        const int icol = cy * (2 * BX) + cx;  // interior only
        const int wcol = ((cy + 2) >> 1) * WX + ((cx + 2) >> 1), icell = (cx & 1) + 2 * (cy & 1);

        // ring of cells around the column region: its corners are read by no
        // slope that feeds a face, and (ROLE 2) neither are the two cells next
        // to each corner
        constexpr int NRING = ROLE == 2 ? 4 * (BX + BY) : ROLE == 0 ? 2 * (CX + CY) : 0;
        const int r = ROLE == 2 ? tid - NI : tid;
        const bool ring = ROLE != 1 && r < NRING;
        int rx = 0, ry = 0;
        if (ring) {
            constexpr int EX = ROLE == 2 ? 2 * BX : CX, EY = ROLE == 2 ? 2 * BY : CY, E0 = ROLE == 2 ? 0 : -1;
            if (r < 2 * EX) {
                rx = (r < EX ? r : r - EX) + E0;
                ry = r < EX ? -2 : 2 * BY + 1;
            } else {
                const int g = r - 2 * EX;
                rx = g < EY ? -2 : 2 * BX + 1;
                ry = (g < EY ? g : g - EY) + E0;
            }
        }
        const int pr = (ry + 2) * PX + (rx + 2);

        auto fetch = [&](int px, int py, int tz, double u[5], int &fl) __attribute__((always_inline)) {
            const int ox = (px + 2) >> 1, oy = (py + 2) >> 1, oz = (tz + 2) >> 1;
            const int v = sm.swin[(oz * WY + oy) * WX + ox];
            fl = -1;
            if (!bnd) {
                // no boundary ghosts: an oct, or none (then nothing that the
                // cell feeds is stored, and any cell's values do)
                const size_t o = (size_t)(v > 1 ? v - 1 : 0);
                const int ind = (px & 1) + 2 * (py & 1) + 4 * (tz & 1);
                const double *p = a.uold + o * 40 + ind;
#pragma unroll
                for (int n = 0; n < 5; n++) u[n] = p[8 * n];
                return;
            }
            const int okey[3] = {ox0 + ox - 1, oy0 + oy - 1, oz0 + oz - 1};
            const int c[3] = {px & 1, py & 1, tz & 1};
            CellRef cr = cell_ref3(a.uold, a.refined, v, okey, boxmin, boxmax, refl, c);
            cr.rf = nullptr;
            uint8_t rf;
            cell_load3(cr, u, rf);
            fl = cr.flip;
        };

        double u_o[5], u_r[5];
        int fl_o = -1, fl_r = -1;
        auto convert = [&](double u[5], int fl, double q[5]) __attribute__((always_inline)) {
            if (bnd && fl >= 0) cell_flip(u, fl);  // reflexive ghosts only: skipped by waves without any
            return prim64(u, q, a.smallr, smalle, gm1, gdt);
        };
        auto put = [&](const double q[5], int i) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < 5; n++) sm.sq[n][i] = q[n];
        };

        // own column: primitives of plane tt, their difference from plane tt-1
        // (the upper difference of the plane before), density of plane tt-1,
        // 1/rho of plane tt
        double q0[5], dzm[5], rho_m, ir0;
        {
            double q[5];
            fetch(cx, cy, tlo - 2, u_o, fl_o);
            convert(u_o, fl_o, q);
            fetch(cx, cy, tlo - 1, u_o, fl_o);
            if (ring) fetch(rx, ry, tlo - 1, u_r, fl_r);
            ir0 = convert(u_o, fl_o, q0);
            rho_m = q[0];
#pragma unroll
            for (int n = 0; n < 5; n++) dzm[n] = q0[n] - q[n];
            put(q0, pc);
            if (ring) {
                convert(u_r, fl_r, q);
                put(q, pr);
            }
            fetch(cx, cy, tlo, u_o, fl_o);
            if (ring) fetch(rx, ry, tlo, u_r, fl_r);
        }
        __syncthreads();

        double qmz[5] = {0, 0, 0, 0, 0};   // left state of the low z face of plane tt
        double fz[5] = {0, 0, 0, 0, 0};    // flux of the low z face of plane tt-1, after its solve that of plane tt
        double fxo[5] = {0, 0, 0, 0, 0};   // fluxes of the low x and y faces of plane tt-1
        double fyo[5] = {0, 0, 0, 0, 0};
        // plane tt-1 without its z faces, after the solve of its high one its new
        // state.  The two z fluxes are subtracted before they are added, as those of
        // x and y: equal fluxes (a planar flow's pressure) then cancel exactly.
        double pp[5] = {0, 0, 0, 0, 0};
        double ub[5] = {0, 0, 0, 0, 0};    // the update's base of plane tt-1 (GEN)
        bool ref1 = false, ref2 = false;   // refined flags of planes tt-1 and tt-2

        // plane tf of the column is final: its new state pp to unew
        auto finish = [&](int tf, const bool upper) __attribute__((always_inline)) {
            const int v = sm.swin[((tf + 2) >> 1) * (WX * WY) + wcol];
            const bool own = v >= a.head && v < a.head + a.noct && ox0 + (cx >> 1) < boxmax[0] &&
                             oy0 + (cy >> 1) < boxmax[1] && oz0 + (tf >> 1) < boxmax[2];
            if (!own) return;
            // the two planes of an oct fill each 64-byte line of unew: the
            // lower plane's values wait in LDS and both are stored together
            if (upper) {
                double *po = a.unew + (size_t)(v - 1) * 40 + icell;
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    po[8 * n] = sm.sun[n][icol];
                    po[8 * n + 4] = pp[n];
                }
            } else {
#pragma unroll
                for (int n = 0; n < 5; n++) sm.sun[n][icol] = pp[n];
            }
            if (courant && !ref2) c_sig = tmax(c_sig, courant_cell<3>(pp, ck, ck.vol, c_mass, c_ekin, c_eint));
        };

        auto wi = [&](int x, int y, int z) __attribute__((always_inline)) {
            return (((z + 2) >> 1) * WY + ((y + 2) >> 1)) * WX + ((x + 2) >> 1);
        };
        auto refined = [&](int x, int y, int z) __attribute__((always_inline)) {
            return ((sm.sref[GEN ? wi(x, y, z) : 0] >> ((x & 1) + 2 * (y & 1) + 4 * (z & 1))) & 1) != 0;
        };
        // a face next to a refined cell has no flux of this level; most waves
        // have none and skip the ten selects
        auto refzero = [&](bool z, double f[5]) __attribute__((always_inline)) {
            if (__any(z))
#pragma unroll
                for (int n = 0; n < 5; n++) f[n] = z ? 0.0 : f[n];
        };
        // Coarse-fine refluxes.  The cells of an oct face share one ghost oct,
        // so an x or y face adds the fluxes of both planes of the oct layer at
        // the upper one (the lower plane's still in LDS where this thread
        // stores its own next), and a z face can meet a ghost only below an
        // even plane: a third of the tests and half of the atomics of adding
        // every face by itself.
        auto owned = [&](int x, int y, int z, int v) __attribute__((always_inline)) {
            return x >= 0 && x < 2 * BX && y >= 0 && y < 2 * BY && z >= tlo && z <= thi && v >= a.head &&
                   v < a.head + a.noct && ox0 + (x >> 1) < boxmax[0] && oy0 + (y >> 1) < boxmax[1] &&
                   oz0 + (z >> 1) < boxmax[2];
        };
        // F into the ghost oct v of window slot i: summed in LDS, or straight
        // to the accumulator / parent cell
        auto radd = [&](int i, int v, double sign, const double F[5], int slot) __attribute__((always_inline)) {
            if (RA && rlds) {
                const double w = sign * dtdx8;
#pragma unroll
                for (int n = 0; n < 5; n++) atomicAdd(&sm.sacc[RA ? i : 0][n], F[n] * w);
            } else {
                double G[5];
#pragma unroll
                for (int n = 0; n < 5; n++) G[n] = F[n] * dtdx;
                reflux_add(a.unew, a.ghost_parent, a.ngridmax, v, sign, G, 8, a.racc, a.rdet, slot);
            }
        };
        // the low x (y) face of the column, plane tt odd: f of this plane, the
        // plane below's at fb (stride st)
        auto reflux_xy = [&](int tt, const bool dy, const double *fb, int st, const double f[5]) __attribute__((always_inline)) {
            const int xl = dy ? cx : cx - 1, yl = dy ? cy - 1 : cy;
            const int il = wi(xl, yl, tt), ih = wi(cx, cy, tt), vl = sm.swin[il], vh = sm.swin[ih];
            const bool gl = vl > a.ngridmax;
            if (gl == (vh > a.ngridmax)) return;
            if (!(gl ? owned(cx, cy, tt, vh) : owned(xl, yl, tt, vl))) return;
            const int i = gl ? il : ih, v = gl ? vl : vh;
            const double sign = gl ? -1.0 : 1.0;
            const int slot = (dy ? 8 + (cx & 1) : (cy & 1)) + (gl ? 4 : 0);
            double F[5];
#pragma unroll
            for (int n = 0; n < 5; n++) F[n] = fb[n * st];
            if (!a.rdet) {
#pragma unroll
                for (int n = 0; n < 5; n++) F[n] = F[n] + f[n];
            } else {
                radd(i, v, sign, f, slot + 2);
            }
            radd(i, v, sign, F, slot);
        };
        // the low z face, plane tt even
        auto reflux_z = [&](int tt, const double f[5]) __attribute__((always_inline)) {
            const int il = wi(cx, cy, tt - 1), ih = wi(cx, cy, tt), vl = sm.swin[il], vh = sm.swin[ih];
            const bool gl = vl > a.ngridmax;
            if (gl == (vh > a.ngridmax)) return;
            if (!(gl ? owned(cx, cy, tt, vh) : owned(cx, cy, tt - 1, vl))) return;
            radd(gl ? il : ih, gl ? vl : vh, gl ? -1.0 : 1.0, f, (gl ? 20 : 16) + (cx & 1) + 2 * (cy & 1));
        };

        // one plane; par = tt & 1
        auto plane = [&](const int tt, const int par) __attribute__((always_inline)) {
            // ---- A: update of plane tt-1, plane tt-2 stored ----
            if constexpr (kPrioA) __builtin_amdgcn_s_setprio(1);
            if (interior && tt > tlo) {
                double part[5];
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    const double u = GEN ? ub[n] : sm.sub[GEN ? 0 : par ^ 1][n][GEN ? 0 : icol];
                    part[n] = tfma(dtdx, fyo[n] - sm.fy[n][iyh], tfma(dtdx, fxo[n] - sm.fx[n][ixh], u));
                }
                if (tt - 2 >= tlo) finish(tt - 2, par != 0);
#pragma unroll
                for (int n = 0; n < 5; n++) pp[n] = part[n];
            }
            // ---- the own cell of plane tt+1 ----
            double qp[5];
            if constexpr (!GEN) {
                if (interior)
#pragma unroll
                    for (int n = 0; n < 5; n++) sm.sub[GEN ? 0 : par ^ 1][n][GEN ? 0 : icol] = u_o[n];
            }
            const double irp = convert(u_o, fl_o, qp);
            // the next loads below the conversion that consumes the current ones, so that both use the same registers
            __builtin_amdgcn_sched_barrier(0);
            fetch(cx, cy, tt < thi ? tt + 2 : thi + 2, u_o, fl_o);
            // ---- T: slopes and predictor of plane tt ----
            double dq[3][5], hr = 0.0, hp = 0.0;
            auto slopes = [&](const int sl) __attribute__((always_inline)) {
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    dq[0][n] = slope64(sl, q0[n] - sm.sq[n][pc - 1], sm.sq[n][pc + 1] - q0[n]);
                    dq[1][n] = slope64(sl, q0[n] - sm.sq[n][pc - PX], sm.sq[n][pc + PX] - q0[n]);
                    dq[2][n] = slope64(sl, dzm[n], qp[n] - q0[n]);
                }
                hr = vmax_abs(vmax_abs(dq[0][0], dq[1][0]), dq[2][0]);
                hp = vmax_abs(vmax_abs(dq[0][4], dq[1][4]), dq[2][4]);
                dq[0][1] = vel_bound64(dq[0][1], sm.sq[0][pc - 1], q0[1] - sm.sq[1][pc - 1], ir0, sm.sq[0][pc + 1],
                                       sm.sq[1][pc + 1] - q0[1]);
                dq[1][2] = vel_bound64(dq[1][2], sm.sq[0][pc - PX], q0[2] - sm.sq[2][pc - PX], ir0,
                                       sm.sq[0][pc + PX], sm.sq[2][pc + PX] - q0[2]);
                dq[2][3] = vel_bound64(dq[2][3], rho_m, dzm[3], ir0, qp[0], qp[3] - q0[3]);
            };
            if (k.slope_type == 1)
                slopes(1);
            else if (k.slope_type != 0)
                slopes(2);
            else
#pragma unroll
                for (int n = 0; n < 5; n++) dq[0][n] = dq[1][n] = dq[2][n] = 0.0;
            double qr[3][5], ql[3][5];
            trace64(q0, dq, qr, ql, k, ir0, hr, hp);
            if (has_qx)
#pragma unroll
                for (int n = 0; n < 5; n++) sm.qx[n][ixh] = ql[0][n];
            if (has_qy)
#pragma unroll
                for (int n = 0; n < 5; n++) sm.qy[n][iyh] = ql[1][n];
            const bool myref = anyref && refined(cx, cy, tt);
            if constexpr (kPrioA) __builtin_amdgcn_s_setprio(0);
            __syncthreads();
            // ---- B: primitives of plane tt+1 to LDS ----
            put(qp, pc);
            if (ring) {
                double q[5];
                convert(u_r, fl_r, q);
                put(q, pr);
                __builtin_amdgcn_sched_barrier(0);
                fetch(rx, ry, tt < thi ? tt + 2 : thi + 1, u_r, fl_r);
            }
            // ---- F: the low x, y and z faces of plane tt ----
            const bool xy = tt >= tlo && tt <= thi;
            double (&f_x)[5] = fxo, (&f_y)[5] = fyo;
            if (ROLE == 2) {
                // the right column's x face or the top row's y face: one pass,
                // the direction chosen per lane
                if (xy && (do_fx || do_fy)) {
                    const bool dy = do_fy;
                    double l[5], g[5];
#pragma unroll
                    for (int n = 0; n < 5; n++) l[n] = dy ? sm.qy[n][iyl] : sm.qx[n][ixl];
                    const double l5[5] = {l[0], dy ? l[2] : l[1], dy ? l[1] : l[2], l[3], l[4]};
                    const double r5[5] = {dy ? qr[1][0] : qr[0][0], dy ? qr[1][2] : qr[0][1], dy ? qr[1][1] : qr[0][2],
                                          dy ? qr[1][3] : qr[0][3], dy ? qr[1][4] : qr[0][4]};
                    solve64<RS>(l5, r5, g, k);
                    double f[5] = {g[0], dy ? g[2] : g[1], dy ? g[1] : g[2], g[3], g[4]};
                    if (anyref) refzero(myref || (dy ? refined(cx, cy - 1, tt) : refined(cx - 1, cy, tt)), f);
                    double *fb = dy ? &sm.fy[0][iyl] : &sm.fx[0][ixl];
                    const int st = dy ? Brick64Lds<BX, BY, BZ, GEN>::NFY : Brick64Lds<BX, BY, BZ, GEN>::NFX;
                    if (reflux && par == 1) reflux_xy(tt, dy, fb, st, f);
#pragma unroll
                    for (int n = 0; n < 5; n++) {
                        fb[n * st] = f[n];
                        f_x[n] = f_y[n] = f[n];
                    }
                }
            } else if (xy) {
                if (do_fx) {
                    double l[5];
#pragma unroll
                    for (int n = 0; n < 5; n++) l[n] = sm.qx[n][ixl];
                    face64<RS>(0, l, qr[0], f_x, k);
                    if (anyref) refzero(myref || refined(cx - 1, cy, tt), f_x);
                    if (reflux && par == 1)
                        reflux_xy(tt, false, &sm.fx[0][ixl], Brick64Lds<BX, BY, BZ, GEN>::NFX, f_x);
#pragma unroll
                    for (int n = 0; n < 5; n++) sm.fx[n][ixl] = f_x[n];
                }
                if (do_fy) {
                    double l[5];
#pragma unroll
                    for (int n = 0; n < 5; n++) l[n] = sm.qy[n][iyl];
                    face64<RS>(1, l, qr[1], f_y, k);
                    if (anyref) refzero(myref || refined(cx, cy - 1, tt), f_y);
                    if (reflux && par == 1)
                        reflux_xy(tt, true, &sm.fy[0][iyl], Brick64Lds<BX, BY, BZ, GEN>::NFY, f_y);
#pragma unroll
                    for (int n = 0; n < 5; n++) sm.fy[n][iyl] = f_y[n];
                }
            }
            if (ROLE != 2 && interior && tt >= tlo) {
                double f[5];
                face64<RS>(2, qmz, qr[2], f, k);
                if (anyref) refzero(myref || ref1, f);
                if (reflux && par == 0) reflux_z(tt, f);
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    pp[n] = tfma(dtdx, fz[n] - f[n], pp[n]);
                    fz[n] = f[n];
                }
            }
            if constexpr (GEN) {
                // the base of this plane's update (unew for the drop-in call,
                // uold for the device-resident steps)
                if (interior && xy) {
                    const int v = sm.swin[((tt + 2) >> 1) * (WX * WY) + wcol];
                    const double *pb = a.ubase + (size_t)(v > 1 ? v - 1 : 0) * 40 + icell + 4 * par;
#pragma unroll
                    for (int n = 0; n < 5; n++) ub[n] = pb[8 * n];
                }
            }
            __syncthreads();
            rho_m = q0[0];
            ir0 = irp;
#pragma unroll
            for (int n = 0; n < 5; n++) {
                qmz[n] = ql[2][n];
                dzm[n] = qp[n] - q0[n];
                q0[n] = qp[n];
            }
            ref2 = ref1;
            ref1 = myref;
        };
        // planes tlo-1 .. thi+1, two per trip (tlo is even, thi odd): the parity
        // is a constant and the values carried from plane to plane are renamed
        for (int tt = tlo - 1; tt <= thi; tt += 2) {
            plane(tt, 1);
            plane(tt + 1, 0);
        }
        if (interior) finish(thi, true);
    };
    // (a part of a brick may hold no layer)
    if (zlo <= zhi) {
        if constexpr (HW) {
            if (__builtin_amdgcn_readfirstlane(tid) < NI)
                run(std::integral_constant<int, 1>());
            else
                run(std::integral_constant<int, 2>());
        } else {
            run(std::integral_constant<int, 0>());
        }
    }

    if (RA && rlds) {
        // one atomic per ghost oct of the window and conserved variable
        __syncthreads();
        for (int i = tid; i < NW; i += NT) {
            const int v = sm.swin[i];
            if (v <= a.ngridmax) continue;
            double q[5];
            bool any = false;
#pragma unroll
            for (int n = 0; n < 5; n++) {
                q[n] = sm.sacc[RA ? i : 0][n];
                any = any || q[n] != 0.0;
            }
            if (any) reflux_flush(a.unew, a.ghost_parent, a.ngridmax, v, q, 8, a.racc);
        }
    }
    if (courant) {
        // the brick's partials of courant_fine in a fixed reduction order; the
        // last wave may be partial (NT need not be a multiple of 64)
        const int nv = NT - (tid & ~63) < 64 ? NT - (tid & ~63) : 64;
        c_mass = wave_sum_n(c_mass, nv);
        c_ekin = wave_sum_n(c_ekin, nv);
        c_eint = wave_sum_n(c_eint, nv);
        c_sig = wave_max_n(c_sig, nv);
        __syncthreads();
        double *red = &sm.sq[0][0];
        const int w = tid >> 6;
        if ((tid & 63) == 0) {
            red[4 * w + 0] = c_mass;
            red[4 * w + 1] = c_ekin;
            red[4 * w + 2] = c_eint;
            red[4 * w + 3] = c_sig;
        }
        __syncthreads();
        if (tid == 0) {
            double m = 0, e = 0, ei = 0, s = red[3];
            for (int i = 0; i < (NT + 63) / 64; i++) {
                m += red[4 * i];
                e += red[4 * i + 1];
                ei += red[4 * i + 2];
                s = tmax(s, red[4 * i + 3]);
            }
            a.cpart[4 * pslot + 0] = m;
            a.cpart[4 * pslot + 1] = e;
            a.cpart[4 * pslot + 2] = ei;
            a.cpart[4 * pslot + 3] = signal_dt(s, ck);
        }
    }
}

}  // namespace rh
