// gfx950 kernels of the fine-level Godunov hydro step.
//
// 3D: one workgroup per oct brick (BX*BY*BZ octs = 2BX x 2BY x 2BZ cells).
// FP64 with the one-dimensional slopes runs brick64 (rh_brick64.h); brick_body
// below is the mixed-precision kernel, and the FP64 one of the 27-point slope.
// The workgroup marches through the brick along z, one cell plane per
// iteration.  One thread owns one cell column of the (2BX+2) x (2BY+2) trace
// region (the brick's cells plus one cell of halo).  Per plane:
//   P: gather plane t of the (2BX+4) x (2BY+4) primitive region from uold
//      through the brick window (hash-resolved oct indices, boundary ghosts
//      synthesised on the fly), convert to primitives in FP64, keep a ring of
//      two planes in LDS (three for the 27-point slope), the next plane's
//      values already in flight (prefetched a plane ahead);
//   T: slopes (uslope) and Hancock predictor (trace3d) of plane t-1, once per
//      cell; left states of x/y faces go to LDS, z states stay in registers;
//   F: each column solves the Riemann problem on its own low x, y and z face
//      (cmpflxm), so every face is solved once; refined faces get zero flux;
//   U: conservative update u + (dt/dx)(F(i) - F(i+1)), dimension by dimension
//      in the order of godfine1 (hydro/godunov_fine.f90:737-816), written to
//      unew; the courant_fine sums and dt of the new state are reduced from
//      registers as it is stored.
// The FP32 results depend on every rounding, down to which of two products the
// compiler contracts into an FMA, so the FP32 instances are left as they are
// where the FP64 ones moved on.
// No MFMA: the work is divides, square roots and compares, not a contraction.
//
// NaNs are honoured here: the mixed solver can lose a state (two floored cells
// that move apart leave its denominator 0 in FP32), and a cell that is NaN must
// drop out of the dt as it does in the reference, whose compares it fails.
// (With -fno-honor-nans the 256^3 kernel took 535 instead of 546 us, and a level
// whose cells were all lost returned courant_factor times its dt.)
#include <type_traits>

#include "rh_courant.h"
#include "rh_gather.h"
#include "rh_godunov.h"
#include "rh_launch.h"

namespace rh {

// Positivity-preserving 27-point slope (slope_type 3, umuscl.f90:2207-2270)
// for variable n of the cell at ring index (s0, pc), returned halved like
// slope_half: the centred differences are formed as (q+ - q-)/4 = dfx/2, so
// the sum dff and the products slop*dfx/2 are the reference's values halved
// exactly.
template <typename T, int PX, int NP>
__device__ __forceinline__ void slope27(const T (*sq)[5][NP], int sm, int s0, int sp, int n, int pc, T dq3[3])

{
    const T qc = sq[s0][n][pc];
    T vmin = T(0), vmax = T(0);
    bool first = true;
    const int sl[3] = {sm, s0, sp};
#pragma unroll
    for (int kk = 0; kk < 3; kk++)
#pragma unroll
        for (int jj = -1; jj <= 1; jj++)
#pragma unroll
            for (int ii = -1; ii <= 1; ii++) {
                T df = sq[sl[kk]][n][pc + ii + jj * PX] - qc;
                if (first) {
                    vmin = vmax = df;
                    first = false;
                } else {
                    vmin = tmin(vmin, df);
                    vmax = tmax(vmax, df);
                }
            }
    T dfx = T(0.25) * (sq[s0][n][pc + 1] - sq[s0][n][pc - 1]);
    T dfy = T(0.25) * (sq[s0][n][pc + PX] - sq[s0][n][pc - PX]);
    T dfz = T(0.25) * (sq[sp][n][pc] - sq[sm][n][pc]);
    T dff = fabs_(dfx) + fabs_(dfy) + fabs_(dfz);
    T slop = dff > T(0) ? tmin(T(1), tdiv(tmin(fabs_(vmin), fabs_(vmax)), dff)) : T(1);
    dq3[0] = slop * dfx;
    dq3[1] = slop * dfy;
    dq3[2] = slop * dfz;
}

// Loads of the next plane's P-phase cells issued a plane ahead (the FP32
// per-level kernel; it runs at two waves per SIMD with them, measured 4% faster
// at 256^3 than at three without, while the work-list kernel keeps four waves
// per SIMD).
// The z march unrolled by two planes.
#ifndef RH_MARCH_UNROLL2
#define RH_MARCH_UNROLL2 0
#endif
// Levels periodic in every dimension gather through a path without the
// boundary-ghost synthesis (a uniform branch per launch).
#ifndef RH_FAST_FETCH
#define RH_FAST_FETCH 1
#endif
#ifndef RH_PREFETCH_F32
#define RH_PREFETCH_F32 1
#endif

// unew stored one oct layer (two z-planes) at a time, in whole 64-byte lines
// (pair_writes).
#ifndef RH_PAIR_WRITES
#define RH_PAIR_WRITES 1
#endif
// Whole-line stores: the FP32 per-level kernel and the FP32 specialised
// work-list kernel (serving): the mixed kernel 0.624 -> 0.581 ms at 256^3,
// serving's mixed capacity +7%; the FP32 general work-list kernel (AMR)
// measured 7.6% slower with them and stores each half as it comes.
template <typename T, bool WL, bool GEN> constexpr bool pair_writes()
{
    return RH_PAIR_WRITES && (sizeof(T) == 8 || !WL || !GEN);
}
// Refluxes summed in LDS per window oct before one atomic per ghost oct and
// variable (instead of one per fine face), for bricks whose window has at
// most this many octs (4x4x4 bricks: 216 window octs, 8.6 KB of FP64 sums).
#ifndef RH_REFLUX_LDS_MAX
#define RH_REFLUX_LDS_MAX 512
#endif
// The update's base values (the cell's uold) taken from the P phase's loads
// through LDS instead of a second global load at the update, where the
// update adds to uold (device-resident steps).
#ifndef RH_UB_LDS
#define RH_UB_LDS 1
#endif
// The FP32 per-level kernel's Courant reduction in the update phase (as the
// FP64 kernel does) instead of re-reading the brick after the march: it costs
// the kernel a wave per SIMD, which the uniform level step recovers (step
// 0.93 -> 0.87 ms at 256^3) and the work-list kernel of the AMR and serving
// steps does not (AMR mixed step 5% slower), so the latter keeps the re-read.
#ifndef RH_COURANT_IN_UPDATE_F32
#define RH_COURANT_IN_UPDATE_F32 1
#endif

// The FP32 per-level kernel of 8x6x16 bricks runs at three waves per SIMD:
// it fits in 168 VGPRs without spilling when the update's base values are
// loaded at the update (1.5% faster than two waves with them loaded before the
// slopes, and 4.6% faster than two waves with them loaded at the update).  The
// other FP32 shapes spill at three waves and keep two, with the early loads.
template <int BX, int BY, int BZ, typename T, bool WL>
constexpr bool f32_three_waves()
{
    return sizeof(T) == 4 && !WL && BX == 8 && BY == 6 && BZ == 16;
}

// Minimum waves per SIMD requested from the register allocator for the brick
// kernels (occupancy vs. register spills; chosen by measurement).
#ifndef RH_BRICK_MIN_WAVES_F32
#define RH_BRICK_MIN_WAVES_F32 2
#endif
#ifndef RH_BRICK_MIN_WAVES
#define RH_BRICK_MIN_WAVES 2
#endif

// Waves per SIMD a brick kernel runs at (its launch bound): the FP32
// work-list kernel at four, at most 128 VGPRs (the AMR 4x4x4 kernel spills 4
// of its 131 for it, and the mixed AMR step is 9% faster: 0.670 -> 0.612 ms).
template <int BX, int BY, int BZ, typename T, bool WL> constexpr int brick_waves()
{
    return sizeof(T) == 8 ? RH_BRICK_MIN_WAVES
                          : (WL ? 4 : (f32_three_waves<BX, BY, BZ, T, WL>() ? 3 : RH_BRICK_MIN_WAVES_F32));
}

// Halo-wave thread order: the 4 BX BY interior columns fill whole waves and
// the halo columns fit one more (8x6 bricks, 192 + 60 threads; 4x4, 64 + 36).
template <int BX, int BY, int RS, int NS> constexpr bool brick_hw()
{
    return (4 * BX * BY) % 64 == 0 && (2 * BX + 2) * (2 * BY + 2) - 4 * BX * BY <= 64 && RS == 3 && NS == 2;
}

// The next-plane prefetch: the HLLC variants of the FP32 per-level kernel, with
// a thread for every cell of the P-phase ring.
template <int BX, int BY, typename T, int RS, int NS, bool WL> constexpr bool brick_prefetch()
{
    constexpr int CX = 2 * BX + 2, CY = 2 * BY + 2, NT = CX * CY, NI = 4 * BX * BY;
    constexpr bool HW = brick_hw<BX, BY, RS, NS>();
    constexpr int NRING = HW ? 4 * (BX + BY) : 2 * (CX + CY);
    return sizeof(T) == 4 && RH_PREFETCH_F32 && !WL && RS == 3 && NS == 2 &&
           (HW ? NRING <= NT - NI : NRING <= NT);
}

// LDS of one brick workgroup.  NS primitive planes are kept: 2 when the slopes
// need only face neighbours (the z neighbours of a column sit in registers),
// 3 for the 27-point slope of slope_type 3.
// SEP: face fluxes get their own buffer (sff) instead of overwriting the
// face states in sf, which saves one barrier per plane.  Measured: no gain
// (256^3 FP64 and mixed within 1%), so off by default; the barriers are not
// what limits the kernel.
template <int BX, int BY, int BZ, typename T, int NS, bool SEP, bool PWT> struct BrickSmemCore {
    static constexpr int CX = 2 * BX + 2, CY = 2 * BY + 2, NT = CX * CY;
    static constexpr int PX = 2 * BX + 4, PY = 2 * BY + 4, NP = PX * PY;
    static constexpr int WX = BX + 2, WY = BY + 2, WZ = BZ + 2, NW = WX * WY * WZ;
    int32_t swin[NW];
    T sq[NS][5][NP];
    uint8_t sref[NS][NP];
    T sf[2][5][NT];
    T sff[SEP ? 2 : 1][5][SEP ? NT : 1];
    // new state of the lower z-plane of the oct layer, per interior column
    // (RH_PAIR_WRITES)
    static constexpr bool PW = PWT;
    double sun[PW ? 5 : 1][PW ? 4 * BX * BY : 1];
};
// The optional buffers are added only while the workgroups the kernel's
// waves per SIMD call for (WPS) still fit the 160 KB of LDS of a CU, so that
// they never cost occupancy:
// - sacc (RA): the coarse-fine refluxes of the brick summed per window oct,
//   flushed once per ghost oct at the end (windows of at most
//   RH_REFLUX_LDS_MAX octs);
// - sub (UBL, kernels with the next-plane prefetch, UBOK): the conserved
//   state of each interior column's cell on the last two planes, kept from
//   the P phase's loads as the update's base values.
template <int BX, int BY, int BZ, typename T, int NS, bool SEP, int WPS, bool UBOK, bool PWT>
struct BrickSmem : BrickSmemCore<BX, BY, BZ, T, NS, SEP, PWT> {
    using Core = BrickSmemCore<BX, BY, BZ, T, NS, SEP, PWT>;
    static constexpr int NW = Core::NW, NT = Core::NT;
    static constexpr int WGS = (4 * WPS) / ((NT + 63) / 64) > 0 ? (4 * WPS) / ((NT + 63) / 64) : 1;
    static constexpr size_t LIM = (size_t)160 * 1024 / WGS;
    static constexpr bool RA = NW <= RH_REFLUX_LDS_MAX && sizeof(Core) + (size_t)NW * 40 <= LIM;
    static constexpr size_t RAB = RA ? (size_t)NW * 40 : 40;
    static constexpr bool UBL =
        UBOK && RH_UB_LDS && NT <= 256 && sizeof(Core) + RAB + (size_t)80 * 4 * BX * BY <= LIM;
    double sacc[RA ? NW : 1][5];
    double sub[UBL ? 2 : 1][5][UBL ? 4 * BX * BY : 1];
};

// Separate flux buffer where the LDS allows it: the two-plane ring (the
// 27-point slope's three planes are the big ones) within the 160 KB of a CU.
#ifndef RH_SEP_FLUX
#define RH_SEP_FLUX 0
#endif
template <int BX, int BY, int BZ, typename T, int NS> constexpr bool sep_flux()
{
    return RH_SEP_FLUX && NS == 2 && sizeof(BrickSmemCore<BX, BY, BZ, T, NS, true, false>) <= 160 * 1024;
}

// The LDS of the per-level (WL = false) or work-list kernel.  The base
// values through LDS (UBL) pay in the FP32 kernel, whose three waves per SIMD
// leave no registers to load them early (a load at the update waits, by the
// in-order memory counter, for the next-plane prefetch issued before it): at
// 256^3 the mixed kernel 0.666 -> 0.618 ms.
template <int BX, int BY, int BZ, typename T, int RS, int NS, bool WL, bool GEN>
using BrickLds = BrickSmem<BX, BY, BZ, T, NS, sep_flux<BX, BY, BZ, T, NS>(), brick_waves<BX, BY, BZ, T, WL>(),
                           brick_prefetch<BX, BY, T, RS, NS, WL>(),
                           pair_writes<T, WL, GEN>()>;

__device__ __forceinline__ int ring_slot2(int t) { return t & 1; }
__device__ __forceinline__ int ring_slot3(int t) { return (t + 3) % 3; }

// One brick: the body shared by the per-level kernel and the work-list kernel.
// RS = 3 compiles HLLC in; NS is the depth of the primitive ring.
// A is GodArgs (a kernel argument) or GodArgs in the constant address space
// (a work-list descriptor): both are read-only for the kernel's lifetime, so
// the compiler reloads their fields with scalar loads instead of holding them.
// GEN = false compiles the body for a level that is periodic in every
// dimension, has no refined cell and no coarse-fine faces (every uniform
// level): without the boundary-ghost gather, the refined-face zeroing and the
// reflux code.  The launch checks the level.
template <int BX, int BY, int BZ, typename T, int RS, int NS, bool WL, bool GEN = true, typename A>
__device__ __forceinline__ void brick_body(A &a, const int bid, BrickLds<BX, BY, BZ, T, RS, NS, WL, GEN> &sm,
                                           const int zlo, const int zhi, const int pslot)
{
    constexpr int CX = 2 * BX + 2, CY = 2 * BY + 2, NT = CX * CY;
    constexpr int PX = 2 * BX + 4, PY = 2 * BY + 4, NP = PX * PY;
    constexpr int WX = BX + 2, WY = BY + 2, WZ = BZ + 2, NW = WX * WY * WZ;
    int32_t *swin = sm.swin;
    auto &sq = sm.sq;
    auto &sref = sm.sref;
    auto &sf = sm.sf;
    constexpr bool SEP = sep_flux<BX, BY, BZ, T, NS>();
    T(*fb)[5][NT];
    if constexpr (SEP)
        fb = sm.sff;
    else
        fb = sm.sf;
    (void)CY;
    const int tid = threadIdx.x;
    for (int i = tid; i < NW; i += NT) swin[i] = a.win[(size_t)bid * NW + i];
    // refluxes summed in LDS (atomic mode only: the deterministic mode keeps
    // one slot per fine face)
    constexpr bool RA = std::remove_reference_t<decltype(sm)>::RA;
    const bool rlds = RA && GEN && a.reflux && !a.rdet;
    if (rlds)
        for (int i = tid; i < NW * 5; i += NT) (&sm.sacc[0][0])[i] = 0.0;
    const int ox0 = a.org[3 * bid + 0], oy0 = a.org[3 * bid + 1], oz0 = a.org[3 * bid + 2];
    // cell planes [tlo, thi] (the z layers of this part that hold octs of the
    // level); the march covers them plus two halo planes on each side
    const int tlo = 2 * zlo, thi = 2 * zhi + 1;

    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    const HydroK<T> k = make_k<T>(dt, a.dx, a.gamma, a.smallr, a.smallc2, a.courant_factor, a.smax_cap, a.use_smax,
                                  a.slope, a.riemann);
    const double smalle = a.smallc2 / a.gamma / (a.gamma - 1.0);
    const double dtxhalf = dt * 0.5;
    const double gdt[3] = {a.g[0] * dtxhalf, a.g[1] * dtxhalf, a.g[2] * dtxhalf};
    const double inv_dx = a.inv_dx;
    // The face fluxes stay unscaled (in LDS and in registers); the update
    // adds dt/dx times each difference of the two faces of a dimension with
    // one FMA, u + (dt/dx)(F(i) - F(i+1)), both cells of a face reading the
    // same flux, so the update conserves.  The reference stores (F dt)/dx per
    // face (hydro/umuscl.f90:135-220); that product, in its order for FP64,
    // is formed only for the coarse reflux.
    const double dtdx64 = dt * inv_dx;
    auto fscale = [&](double f) -> double { return sizeof(T) == 4 ? f * dtdx64 : (f * dt) * inv_dx; };
    const int boxmin[3] = {a.boxmin[0], a.boxmin[1], a.boxmin[2]};
    const int boxmax[3] = {a.boxmax[0], a.boxmax[1], a.boxmax[2]};
    const bool anyref = GEN && a.any_ref != 0;  // refined flags are all 0 when not
    int refl = 0;
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int sd = 0; sd < 2; sd++) refl |= (a.btype[d][sd] == 1) << (2 * d + sd);
    const double gvec[3] = {a.g[0], a.g[1], a.g[2]};
    __syncthreads();

    // Column of this thread.  Row-major over the (2BX+2)(2BY+2) columns, or,
    // when the 4 BX BY interior columns fill whole waves and the halo columns
    // fit one more (HW: 8x6 bricks, 192 + 60 threads; 4x4, 64 + 36), interior columns
    // first and the halo ring last, so that the halo wave, which needs at most
    // one face per column and no update, runs one solver pass instead of three
    // and skips the update; it takes the P-phase ring instead.
    constexpr int NI = 4 * BX * BY;
    constexpr bool HW = brick_hw<BX, BY, RS, NS>();
    int cx, cy;
    if constexpr (HW) {
        if (tid < NI) {
            cx = tid % (2 * BX);
            cy = tid / (2 * BX);
        } else {
            const int h = tid - NI;
            if (h < CX) {
                cx = h - 1;
                cy = -1;
            } else if (h < 2 * CX) {
                cx = h - CX - 1;
                cy = 2 * BY;
            } else if (h < 2 * CX + 2 * BY) {
                cx = -1;
                cy = h - 2 * CX;
            } else {
                cx = 2 * BX;
                cy = h - 2 * CX - 2 * BY;
            }
        }
    } else {
        cx = tid % CX - 1;
        cy = tid / CX - 1;
    }
    // index of this column in the face-state and flux buffers (row-major)
    const int col = (cy + 1) * CX + (cx + 1);
    const int pc = (cy + 2) * PX + (cx + 2);
    const bool interior = cx >= 0 && cx < 2 * BX && cy >= 0 && cy < 2 * BY;
    const bool do_fx = cx >= 0 && cx <= 2 * BX && cy >= 0 && cy < 2 * BY;
    const bool do_fy = cy >= 0 && cy <= 2 * BY && cx >= 0 && cx < 2 * BX;

    T qmz_prev[5] = {T(0), T(0), T(0), T(0), T(0)};
    uint8_t ref_prev = 0;
    T fz_prev[5] = {T(0), T(0), T(0), T(0), T(0)};  // z-face fluxes in the solver's precision
    double part_prev[5] = {0, 0, 0, 0, 0};
    // own column primitives of planes tt-1 and tt (used when NS == 2)
    T qcol_m[5] = {T(0), T(0), T(0), T(0), T(0)}, qcol_0[5] = {T(0), T(0), T(0), T(0), T(0)};


    // P-phase cells of this thread: its own column's cell, and for the first
    // NRING threads one cell of the ring around the column region.  Their
    // loads are issued one plane ahead (u_o, u_r) and converted the next plane.
    // The ring leaves out its four corner cells, which no slope reads (the
    // 27-point stencil reaches them only from the corner columns, whose
    // states feed no face): 2(CX+CY) cells, one wave for the 7x7 brick.
    // With HW the ring is the halo wave's and leaves out the two cells next to
    // each corner as well, which only the corner columns read with the
    // one-dimensional slopes of this variant: 4(BX+BY) cells.
    constexpr int NRING = HW ? 4 * (BX + BY) : 2 * (CX + CY);
    const int r = HW ? tid - NI : tid;
    const bool ring = r >= 0 && r < NRING;
    int ring_i = 0;
    if (ring) {
        int rx, ry;
        if constexpr (HW) {
            if (r < 2 * BX) {
                rx = r;
                ry = -2;
            } else if (r < 4 * BX) {
                rx = r - 2 * BX;
                ry = 2 * BY + 1;
            } else if (r < 4 * BX + 2 * BY) {
                rx = -2;
                ry = r - 4 * BX;
            } else {
                rx = 2 * BX + 1;
                ry = r - 4 * BX - 2 * BY;
            }
        } else if (r < CX) {
            rx = r - 1;
            ry = -2;
        } else if (r < 2 * CX) {
            rx = r - CX - 1;
            ry = 2 * BY + 1;
        } else if (r < 2 * CX + CY) {
            rx = -2;
            ry = r - 2 * CX - 1;
        } else {
            rx = 2 * BX + 1;
            ry = r - 2 * CX - CY - 1;
        }
        ring_i = (ry + 2) * PX + (rx + 2);
    }
    const bool bnd = GEN && (RH_FAST_FETCH ? a.bnd != 0 : true);
    auto fetch = [&](int i, int tz, double u[5], uint8_t &rf, int &fl) {
        const int px = i % PX - 2, py = i / PX - 2;
        const int ox = (px + 2) >> 1, oy = (py + 2) >> 1, oz = (tz + 2) >> 1;
        const int v = swin[(oz * WY + oy) * WX + ox];
        const int c[3] = {px & 1, py & 1, tz & 1};
        if (!bnd) {
            // no boundary ghosts: an oct (v > 0) or none (v == 0)
            const int ind = c[0] + 2 * c[1] + 4 * c[2];
            CellRef r;
            r.p = v > 0 ? a.uold + (size_t)(v - 1) * 40 + ind : nullptr;
            r.rf = anyref && v > 0 ? a.refined + (size_t)(v - 1) * 8 + ind : nullptr;
            cell_load3(r, u, rf);
            fl = -1;
            return;
        }
        const int okey[3] = {ox0 + ox - 1, oy0 + oy - 1, oz0 + oz - 1};
        CellRef r = cell_ref3(a.uold, a.refined, v, okey, boxmin, boxmax, refl, c);
        if (!anyref) r.rf = nullptr;
        cell_load3(r, u, rf);
        fl = r.flip;
    };
    // prefetch a plane ahead (load latency hidden) in the HLLC variants of the
    // FP32 per-level kernel, which drops to two waves per SIMD with it and is
    // faster for it; the work-list kernel and the other variants load at use,
    // as they would spill or lose waves (it also needs a thread for every
    // ring cell)
    constexpr bool PF = brick_prefetch<BX, BY, T, RS, NS, WL>();
    double u_o[5], u_r[5];
    uint8_t rf_o, rf_r = 0;
    int fl_o, fl_r = -1;
    // the update's base values from the P phase (through LDS) when the update
    // adds to uold; the own column's cell of plane t is u_o in the P phase
    constexpr bool UBL = std::remove_reference_t<decltype(sm)>::UBL && PF;
    const bool ubl = UBL && (!GEN || a.ubase == a.uold);  // the specialised body is launched with ubase == uold
    const int icol = interior ? cy * (2 * BX) + cx : 0;
    if (PF) {
        fetch(pc, tlo - 2, u_o, rf_o, fl_o);
        if (ring) fetch(ring_i, tlo - 2, u_r, rf_r, fl_r);
    }

    // ---- P: primitives of plane t into ring slot st, own column to qcol_p ----
    auto p_phase = [&](const int t, const int st, T qcol_p[5]) {
        if constexpr (!PF) {
            for (int i = tid; i < NP; i += NT) {
                const int px = i % PX - 2, py = i / PX - 2;
                const int ox = (px + 2) >> 1, oy = (py + 2) >> 1, oz = (t + 2) >> 1;
                const int v = swin[(oz * WY + oy) * WX + ox];
                int okey[3] = {ox0 + ox - 1, oy0 + oy - 1, oz0 + oz - 1};
                int c[3] = {px & 1, py & 1, t & 1};
                double u[5], q[5];
                uint8_t rf;
                gather_cell_m(a.uold, a.refined, v, okey, 3, boxmin, boxmax, refl, c, u, rf);
                prim_from_cons<sizeof(T) == 4>(u, q, a.smallr, smalle, a.gamma, gdt);
#pragma unroll
                for (int n = 0; n < 5; n++) sq[st][n][i] = T(q[n]);
                sref[st][i] = rf;
            }
            __syncthreads();
#pragma unroll
            for (int n = 0; n < 5; n++) qcol_p[n] = sq[st][n][pc];
        } else {
            double q[5];
            if (bnd && fl_o >= 0) cell_flip(u_o, fl_o);  // reflexive ghosts only: skipped by waves without any
            if (ubl && interior)
#pragma unroll
                for (int n = 0; n < 5; n++) sm.sub[UBL ? (t & 1) : 0][n][UBL ? icol : 0] = u_o[n];
            prim_from_cons<sizeof(T) == 4>(u_o, q, a.smallr, smalle, a.gamma, gdt);
#pragma unroll
            for (int n = 0; n < 5; n++) {
                qcol_p[n] = T(q[n]);
                sq[st][n][pc] = qcol_p[n];
            }
            sref[st][pc] = rf_o;
            if (ring) {
                if (bnd && fl_r >= 0) cell_flip(u_r, fl_r);
                prim_from_cons<sizeof(T) == 4>(u_r, q, a.smallr, smalle, a.gamma, gdt);
#pragma unroll
                for (int n = 0; n < 5; n++) sq[st][n][ring_i] = T(q[n]);
                sref[st][ring_i] = rf_r;
            }
            // unconditional (the last plane re-reads itself): a load under a
            // branch makes the compiler copy the loop-carried registers at the
            // loop latch, which waits for the loads (and the update's stores)
            const int tn = t < thi + 2 ? t + 1 : t;
            // keep the next plane's loads below the conversions that consume
            // the current values, so that both use the same registers
            __builtin_amdgcn_sched_barrier(0);
            fetch(pc, tn, u_o, rf_o, fl_o);
            if (ring) fetch(ring_i, tn, u_r, rf_r, fl_r);
            __syncthreads();
        }
    };
    auto rotate = [&](const T qcol_p[5]) {
#pragma unroll
        for (int n = 0; n < 5; n++) {
            qcol_m[n] = qcol_0[n];
            qcol_0[n] = qcol_p[n];
        }
    };
    // the two planes below the first output plane only fill the ring; peeled,
    // so that the march has one loop body and latch (a skipped body makes the
    // compiler copy every loop-carried register at the latch, waiting for the
    // prefetch loads and the update's stores)
    for (int t = tlo - 2; t < tlo; ++t) {
        T qcol_p[5];
        p_phase(t, NS == 3 ? ring_slot3(t) : ring_slot2(t), qcol_p);
        rotate(qcol_p);
    }
    // courant_fine of the state written (the dt of the next step), when asked
    // for: taken from each leaf cell's new state as it is stored; the FP32
    // work-list kernel re-reads the brick's cells after the march
    // (RH_COURANT_IN_UPDATE_F32)
    constexpr bool CU = sizeof(T) == 8 || (RH_COURANT_IN_UPDATE_F32 && !WL);
    const CourantK ck = make_courant_k(a.dx, 3, a.gamma, a.smallr, a.smallc2, a.courant_factor, gvec);
    // c_dt: the smallest dt (FP32), the largest summed signal speed (FP64)
    double c_mass = 0.0, c_ekin = 0.0, c_eint = 0.0, c_dt = sizeof(T) == 8 ? 0.0 : a.dx / ck.smallc;
    // one plane of the march; par = t & 1 (the ring slot of plane t when NS == 2)
    auto march = [&](const int t, const int par) __attribute__((always_inline)) {
        const int st = NS == 3 ? ring_slot3(t) : par;
        T qcol_p[5];
        p_phase(t, st, qcol_p);
        // ---- T: slopes and predictor of plane tt = t-1 ----
        const int tt = t - 1;
        const bool plane_out = tt >= tlo && tt <= thi;
        // the values the update of plane tt adds to: with the prefetch (same
        // register budget), loaded here so that the T and F phases cover
        // their latency, else (and in the three-wave FP32 kernel) at the update
        constexpr bool UB_EARLY = PF && !f32_three_waves<BX, BY, BZ, T, WL>();
        double ub[5];
        if constexpr (UB_EARLY) {
            if (!ubl && interior && plane_out) {
                const int ox = (cx >> 1) + 1, oy = (cy >> 1) + 1, oz = (tt >> 1) + 1;
                const int v = swin[(oz * WY + oy) * WX + ox];
                const int ind = (cx & 1) + 2 * (cy & 1) + 4 * (tt & 1);
                const double *pb = a.ubase + (size_t)(v > 0 ? v - 1 : 0) * 40 + ind;
#pragma unroll
                for (int n = 0; n < 5; n++) ub[n] = pb[8 * n];
            }
        }
        const int s0 = NS == 3 ? ring_slot3(t - 1) : par ^ 1;
        const int smm = NS == 3 ? ring_slot3(t - 2) : 0;
        T q0[5], dq[3][5];
#pragma unroll
        for (int n = 0; n < 5; n++) q0[n] = qcol_0[n];
        if (NS == 3 && k.slope_type == 3) {
#pragma unroll
            for (int n = 0; n < 5; n++) {
                T d3[3];
                slope27<T, PX, NP>(sq, smm, s0, st, n, pc, d3);
                dq[0][n] = d3[0];
                dq[1][n] = d3[1];
                dq[2][n] = d3[2];
            }
        } else {
            // one uniform branch on the slope type for all 15 slopes
            auto slopes = [&](const int sl) {
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    dq[0][n] = slope_half(sl, sq[s0][n][pc - 1], q0[n], sq[s0][n][pc + 1]);
                    dq[1][n] = slope_half(sl, sq[s0][n][pc - PX], q0[n], sq[s0][n][pc + PX]);
                    dq[2][n] = slope_half(sl, qcol_m[n], q0[n], qcol_p[n]);
                }
            };
            if (k.slope_type == 1)
                slopes(1);
            else if (k.slope_type != 0)
                slopes(2);
            else
#pragma unroll
                for (int n = 0; n < 5; n++) dq[0][n] = dq[1][n] = dq[2][n] = T(0);
        }
        const T inv_r0 = trcp(q0[0]);
        if (k.slope_type > 0) {
            dq[0][1] = vel_bound_half(dq[0][1], sq[s0][0][pc - 1], sq[s0][1][pc - 1], inv_r0, q0[1],
                                      sq[s0][0][pc + 1], sq[s0][1][pc + 1]);
            dq[1][2] = vel_bound_half(dq[1][2], sq[s0][0][pc - PX], sq[s0][2][pc - PX], inv_r0, q0[2],
                                      sq[s0][0][pc + PX], sq[s0][2][pc + PX]);
            dq[2][3] = vel_bound_half(dq[2][3], qcol_m[0], qcol_m[3], inv_r0, q0[3], qcol_p[0], qcol_p[3]);
        }
        T qp[3][5], qm[3][5];
        trace3(q0, dq, qp, qm, k, inv_r0);
        const uint8_t myref = anyref ? sref[s0][pc] : 0;
#pragma unroll
        for (int n = 0; n < 5; n++) {
            sf[0][n][col] = qm[0][n];
            sf[1][n][col] = qm[1][n];
        }
        __syncthreads();
        // ---- F: Riemann problems on the low x, y, z faces of this column ----
        T fx[5], fy[5];
        T fz[5] = {T(0), T(0), T(0), T(0), T(0)};
        const bool wfx = do_fx && plane_out, wfy = do_fy && plane_out;
        if (HW && tid >= NI) {
            // halo wave: the right column's x face or the top row's y face,
            // one solver pass with the direction chosen per lane
            if (wfx || wfy) {
                const bool dy = wfy;
                const int nb = dy ? col - CX : col - 1;
                T ql[5], qr[5], a5[5], b5[5], g[5];
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    ql[n] = dy ? sf[1][n][nb] : sf[0][n][nb];
                    qr[n] = dy ? qp[1][n] : qp[0][n];
                }
                a5[0] = ql[0], a5[1] = dy ? ql[2] : ql[1], a5[2] = dy ? ql[1] : ql[2], a5[3] = ql[3], a5[4] = ql[4];
                b5[0] = qr[0], b5[1] = dy ? qr[2] : qr[1], b5[2] = dy ? qr[1] : qr[2], b5[3] = qr[3], b5[4] = qr[4];
                riemann_hllc(a5, b5, g, k);
                T f[5] = {g[0], dy ? g[2] : g[1], dy ? g[1] : g[2], g[3], g[4]};
                if (anyref) {
                    const bool z = myref || sref[s0][dy ? pc - PX : pc - 1];
#pragma unroll
                    for (int n = 0; n < 5; n++) f[n] = z ? T(0) : f[n];
                }
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    fx[n] = f[n];
                    fy[n] = f[n];
                }
            }
        } else {
            if (wfx) {
                T ql[5];
#pragma unroll
                for (int n = 0; n < 5; n++) ql[n] = sf[0][n][col - 1];
                face_flux<RS>(0, ql, qp[0], fx, k);
                if (anyref) {
                    const bool z = myref || sref[s0][pc - 1];
#pragma unroll
                    for (int n = 0; n < 5; n++) fx[n] = z ? T(0) : fx[n];
                }
            }
            if (wfy) {
                T ql[5];
#pragma unroll
                for (int n = 0; n < 5; n++) ql[n] = sf[1][n][col - CX];
                face_flux<RS>(1, ql, qp[1], fy, k);
                if (anyref) {
                    const bool z = myref || sref[s0][pc - PX];
#pragma unroll
                    for (int n = 0; n < 5; n++) fy[n] = z ? T(0) : fy[n];
                }
            }
        }
        if (interior && tt >= tlo && tt <= thi + 1) {
            T f[5];
            face_flux<RS>(2, qmz_prev, qp[2], f, k);
#pragma unroll
            for (int n = 0; n < 5; n++) fz[n] = f[n];
            if (anyref) {
                const bool z = myref || ref_prev;
#pragma unroll
                for (int n = 0; n < 5; n++) fz[n] = z ? T(0) : fz[n];
            }
        }
        if (GEN && a.reflux) {
            // window slot of a cell of the trace region
            auto wi = [&](int x, int y, int z) { return (((z + 2) >> 1) * WY + ((y + 2) >> 1)) * WX + ((x + 2) >> 1); };
            // one fine face's reflux into the ghost oct of window slot i:
            // summed in LDS, or straight to the accumulator / parent cell
            auto radd = [&](int i, int v, double sign, const double F[5], int slot) {
                if (RA && rlds) {
#pragma unroll
                    for (int n = 0; n < 5; n++) atomicAdd(&sm.sacc[RA ? i : 0][n], sign * (F[n] * 0.125));
                } else {
                    reflux_add(a.unew, a.ghost_parent, a.ngridmax, v, sign, F, 8, a.racc, a.rdet, slot);
                }
            };
            auto owned = [&](int x, int y, int z, int v) {
                return x >= 0 && x < 2 * BX && y >= 0 && y < 2 * BY && z >= tlo && z <= thi && v >= a.head &&
                       v < a.head + a.noct && ox0 + (x >> 1) < boxmax[0] && oy0 + (y >> 1) < boxmax[1] &&
                       oz0 + (z >> 1) < boxmax[2];
            };
            double F[5];
            if (wfx && !(myref || sref[s0][pc - 1])) {
                const int il = wi(cx - 1, cy, tt), ih = wi(cx, cy, tt), vl = swin[il], vh = swin[ih];
#pragma unroll
                for (int n = 0; n < 5; n++) F[n] = fscale(double(fx[n]));
                const int sub = (cy & 1) + 2 * (tt & 1);
                if (vl > a.ngridmax && owned(cx, cy, tt, vh)) radd(il, vl, -1.0, F, 4 + sub);
                if (vh > a.ngridmax && owned(cx - 1, cy, tt, vl)) radd(ih, vh, 1.0, F, sub);
            }
            if (wfy && !(myref || sref[s0][pc - PX])) {
                const int il = wi(cx, cy - 1, tt), ih = wi(cx, cy, tt), vl = swin[il], vh = swin[ih];
#pragma unroll
                for (int n = 0; n < 5; n++) F[n] = fscale(double(fy[n]));
                const int sub = (cx & 1) + 2 * (tt & 1);
                if (vl > a.ngridmax && owned(cx, cy, tt, vh)) radd(il, vl, -1.0, F, 12 + sub);
                if (vh > a.ngridmax && owned(cx, cy - 1, tt, vl)) radd(ih, vh, 1.0, F, 8 + sub);
            }
            if (interior && tt >= tlo && tt <= thi + 1 && !(myref || ref_prev)) {
                const int il = wi(cx, cy, tt - 1), ih = wi(cx, cy, tt), vl = swin[il], vh = swin[ih];
#pragma unroll
                for (int n = 0; n < 5; n++) F[n] = fscale(double(fz[n]));
                const int sub = (cx & 1) + 2 * (cy & 1);
                if (vl > a.ngridmax && owned(cx, cy, tt, vh)) radd(il, vl, -1.0, F, 20 + sub);
                if (vh > a.ngridmax && owned(cx, cy, tt - 1, vl)) radd(ih, vh, 1.0, F, 16 + sub);
            }
        }
        if constexpr (!SEP) __syncthreads();  // the fluxes overwrite the face states in sf
        if (wfx)
#pragma unroll
            for (int n = 0; n < 5; n++) fb[0][n][col] = fx[n];
        if (wfy)
#pragma unroll
            for (int n = 0; n < 5; n++) fb[1][n][col] = fy[n];
        __syncthreads();
        // ---- U: conservative update ----
        if (interior) {
            double part[5] = {0, 0, 0, 0, 0};
            if (plane_out) {
                if (ubl) {
#pragma unroll
                    for (int n = 0; n < 5; n++) ub[n] = sm.sub[UBL ? (tt & 1) : 0][n][UBL ? icol : 0];
                } else if constexpr (!UB_EARLY) {
                    const int ox = (cx >> 1) + 1, oy = (cy >> 1) + 1, oz = (tt >> 1) + 1;
                    const int v = swin[(oz * WY + oy) * WX + ox];
                    const int ind = (cx & 1) + 2 * (cy & 1) + 4 * (tt & 1);
                    const double *pb = a.ubase + (size_t)(v > 0 ? v - 1 : 0) * 40 + ind;
#pragma unroll
                    for (int n = 0; n < 5; n++) ub[n] = pb[8 * n];
                }
#pragma unroll
                for (int n = 0; n < 5; n++) {
                    const double fl = fb[0][n][col], fr = fb[0][n][col + 1];
                    const double gl = fb[1][n][col], gr = fb[1][n][col + CX];
                    part[n] = __builtin_fma(dtdx64, gl - gr, __builtin_fma(dtdx64, fl - fr, ub[n]));
                }
            }
            const int tf = tt - 1;
            if (tf >= tlo && tf <= thi) {
                const int ox = (cx >> 1) + 1, oy = (cy >> 1) + 1, oz = (tf >> 1) + 1;
                const int v = swin[(oz * WY + oy) * WX + ox];
                const bool own = v >= a.head && v < a.head + a.noct && ox0 + ox - 1 < boxmax[0] &&
                                 oy0 + oy - 1 < boxmax[1] && oz0 + oz - 1 < boxmax[2];
                if (own) {
                    const int ind = (cx & 1) + 2 * (cy & 1) + 4 * (tf & 1);
                    double *po = a.unew + (size_t)(v - 1) * 40 + ind;
                    double un[5];
#pragma unroll
                    for (int n = 0; n < 5; n++)
                        un[n] = __builtin_fma(dtdx64, double(fz_prev[n]) - double(fz[n]), part_prev[n]);
                    if constexpr (std::remove_reference_t<decltype(sm)>::PW) {
                        // the two z-planes of an oct fill each 64-byte line of
                        // unew: the lower plane's values wait in LDS (the
                        // thread's own slot) and both halves are stored
                        // together with the upper plane
                        const int ic = cy * (2 * BX) + cx;
                        if (tf & 1) {
#pragma unroll
                            for (int n = 0; n < 5; n++) {
                                po[8 * n - 4] = sm.sun[n][ic];
                                po[8 * n] = un[n];
                            }
                        } else {
#pragma unroll
                            for (int n = 0; n < 5; n++) sm.sun[n][ic] = un[n];
                        }
                    } else {
#pragma unroll
                        for (int n = 0; n < 5; n++) po[8 * n] = un[n];
                    }
                    if (CU && a.courant && !ref_prev) {
                        if constexpr (sizeof(T) == 4)
                            courant_cell_mixed(un, ck, c_mass, c_ekin, c_eint, c_dt);
                        else
                            c_dt = tmax(c_dt, courant_cell<3>(un, ck, ck.vol, c_mass, c_ekin, c_eint));
                    }
                }
            }
#pragma unroll
            for (int n = 0; n < 5; n++) {
                part_prev[n] = part[n];
                fz_prev[n] = fz[n];
            }
        }
#pragma unroll
        for (int n = 0; n < 5; n++) qmz_prev[n] = qm[2][n];
        ref_prev = myref;
        rotate(qcol_p);
    };
    if constexpr (RH_MARCH_UNROLL2 && NS == 2) {
        // two planes per trip (the trip count 2(zhi - zlo + 2) is even): the
        // ring slots are constants and the registers carried from plane to
        // plane are renamed instead of copied
        for (int t = tlo; t <= thi + 2; t += 2) {
            march(t, 0);
            march(t + 1, 1);
        }
    } else {
        for (int t = tlo; t <= thi + 2; ++t) march(t, t & 1);
    }
    if (RA && rlds) {
        // one atomic per ghost oct of the window and conserved variable
        __syncthreads();
        for (int i = tid; i < NW; i += NT) {
            const int v = swin[i];
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
    if (a.courant) {
        // the brick's partials of courant_fine in a fixed reduction order
        // (FP64); the FP32 kernel first re-reads its own leaf cells from unew
        // while still in cache
        __syncthreads();
        for (int i = tid; !CU && i < BX * BY * BZ * 8; i += NT) {
            const int oc = i >> 3, ind = i & 7;
            const int ox = oc % BX + 1, oy = (oc / BX) % BY + 1, oz = oc / (BX * BY) + 1;
            if (oz <= zlo || oz > zhi + 1) continue;  // another part's layers
            const int v = swin[(oz * WY + oy) * WX + ox];
            const bool own = v >= a.head && v < a.head + a.noct && ox0 + ox - 1 < boxmax[0] &&
                             oy0 + oy - 1 < boxmax[1] && oz0 + oz - 1 < boxmax[2];
            if (!own || a.refined[(size_t)(v - 1) * 8 + ind]) continue;
            const double *pu = a.unew + (size_t)(v - 1) * 40 + ind;
            const double un[5] = {pu[0], pu[8], pu[16], pu[24], pu[32]};
            courant_cell_mixed(un, ck, c_mass, c_ekin, c_eint, c_dt);
        }
        // lanes of this wave that exist (NT need not be a multiple of 64)
        const int nv = NT - (tid & ~63) < 64 ? NT - (tid & ~63) : 64;
        c_mass = wave_sum_n(c_mass, nv);
        c_ekin = wave_sum_n(c_ekin, nv);
        c_eint = wave_sum_n(c_eint, nv);
        c_dt = sizeof(T) == 8 ? wave_max_n(c_dt, nv) : wave_min_n(c_dt, nv);
        __syncthreads();
        double *red = (double *)&sf[0][0][0];
        const int w = tid >> 6;
        if ((tid & 63) == 0) {
            red[4 * w + 0] = c_mass;
            red[4 * w + 1] = c_ekin;
            red[4 * w + 2] = c_eint;
            red[4 * w + 3] = c_dt;
        }
        __syncthreads();
        if (tid == 0) {
            double m = 0, e = 0, ei = 0, d = red[3];
            for (int i = 0; i < (NT + 63) / 64; i++) {
                m += red[4 * i];
                e += red[4 * i + 1];
                ei += red[4 * i + 2];
                if constexpr (sizeof(T) == 8)
                    d = tmax(red[4 * i + 3], d);
                else
                    d = red[4 * i + 3] < d ? red[4 * i + 3] : d;
            }
            if constexpr (sizeof(T) == 8) d = signal_dt(d, ck);
            a.cpart[4 * pslot + 0] = m;
            a.cpart[4 * pslot + 1] = e;
            a.cpart[4 * pslot + 2] = ei;
            a.cpart[4 * pslot + 3] = d;
        }
    }
}

template <int BX, int BY, int BZ, typename T, int RS, int NS, bool GEN = true>
__global__ void __launch_bounds__((2 * BX + 2) * (2 * BY + 2),
                                  (sizeof(T) == 8                              ? RH_BRICK_MIN_WAVES
                                   : f32_three_waves<BX, BY, BZ, T, false>() ? 3
                                                                             : RH_BRICK_MIN_WAVES_F32))
    k_godunov3d(const GodArgs a)
{
    __shared__ BrickLds<BX, BY, BZ, T, RS, NS, false, GEN> sm;
    int bid, zlo, zhi, pslot;
    if (!level_item(a, BZ, bid, zlo, zhi, pslot)) return;
    brick_body<BX, BY, BZ, T, RS, NS, false, GEN>(a, bid, sm, zlo, zhi, pslot);
}

// Work-list kernel: work item i = (descriptor, brick), where a descriptor
// carries the arrays and parameters of one level of one mesh, so bricks of
// several levels and of several jobs share one launch.  The items are split
// into 8 contiguous ranges, one per XCD: workgroups are placed on the XCDs
// round-robin by workgroup id, so workgroup b runs item range[b % 8] + b / 8
// on XCD b % 8, and neighbouring bricks (which share halo octs) meet in that
// XCD's L2.  One workgroup per item: the hardware dispatcher is the queue.  (A
// persistent loop over an atomic counter holds its loop state and the
// reloaded descriptor in registers and measured 160 instead of 125 VGPRs for
// the FP32 HLLC kernel, one wave per SIMD less.)
typedef const __attribute__((address_space(4))) GodArgs ConstGodArgs;

template <int BX, int BY, int BZ, typename T, int RS, int NS, bool GEN = true>
__global__ void __launch_bounds__((2 * BX + 2) * (2 * BY + 2), (brick_waves<BX, BY, BZ, T, true>()))
    k_godunov3d_wl(const WorkList w)
{
    __shared__ BrickLds<BX, BY, BZ, T, RS, NS, true, GEN> sm;
    const int x = blockIdx.x & 7, l = blockIdx.x >> 3;
    const int i = w.range[x] + l;
    if (i >= w.range[x + 1]) return;
    const int4 it = w.items[i];
    const int di = __builtin_amdgcn_readfirstlane(it.x), bi = __builtin_amdgcn_readfirstlane(it.y);
    const int part = __builtin_amdgcn_readfirstlane(it.z), n = __builtin_amdgcn_readfirstlane(it.w);
    auto &a = ((ConstGodArgs *)w.descs)[di];
    int zlo, zhi;
    part_layers(a.zr ? a.zr[bi] : ((BZ - 1) << 16), part, n, zlo, zhi);
    brick_body<BX, BY, BZ, T, RS, NS, true, GEN>(a, bi, sm, zlo, zhi, bi * n + part);
}


// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
// (a build for one workload may name fewer)
#ifndef RH_BRICK_SHAPES
#define RH_BRICK_SHAPES(X) \
    X(7, 7, 8)             \
    X(7, 7, 16)            \
    X(8, 6, 8)             \
    X(8, 6, 16)            \
    X(4, 4, 4)             \
    X(4, 4, 8)             \
    X(15, 7, 8)            \
    X(15, 7, 16)           \
    X(7, 7, 4)             \
    X(3, 3, 4)             \
    X(3, 3, 8)             \
    X(1, 1, 1)
#endif

bool brick_shape_supported(int bx, int by, int bz)
{
#define RH_CHECK_SHAPE(A, B, C) \
    if (bx == A && by == B && bz == C) return true;
    RH_BRICK_SHAPES(RH_CHECK_SHAPE)
#undef RH_CHECK_SHAPE
    return false;
}

int g_specialized = 1;

// The objects of rh_brick64.hip, one per set of brick shapes
#define RH_SETS(X) X(0) X(1) X(2) X(3) X(4) X(5)
#define RH_DECL(N)                                                                                               \
    bool brick64_level_##N(const GodArgs &a, int bx, int by, int bz, int kind, hipStream_t s, hipEvent_t e0,      \
                           hipEvent_t e1, int *nparts);                                                          \
    bool brick64_list_##N(const WorkList &w, int nblocks, int bx, int by, int bz, int riemann, int kind, hipStream_t s);
RH_SETS(RH_DECL)
#undef RH_DECL

hipError_t launch_brick64(const GodArgs &a, int bx, int by, int bz, int kind, hipStream_t s, hipEvent_t e0,
                          hipEvent_t e1, int *nparts)
{
#define RH_TRY(N) \
    if (brick64_level_##N(a, bx, by, bz, kind, s, e0, e1, nparts)) return hipGetLastError();
    RH_SETS(RH_TRY)
#undef RH_TRY
    return hipErrorInvalidValue;
}

hipError_t launch_brick64_wl(const WorkList &w, int nblocks, int bx, int by, int bz, int riemann, int kind,
                             hipStream_t s)
{
#define RH_TRY(N) \
    if (brick64_list_##N(w, nblocks, bx, by, bz, riemann, kind, s)) return hipGetLastError();
    RH_SETS(RH_TRY)
#undef RH_TRY
    return hipErrorInvalidValue;
}

hipError_t launch_godunov3d(const GodArgs &a, int bx, int by, int bz, int prec, hipStream_t s, hipEvent_t e0,
                            hipEvent_t e1, int *nparts)
{
    if (nparts) *nparts = a.nbricks > 0 ? a.nbricks : 0;
    if (a.nbricks <= 0) return hipSuccess;
    if (prec == 0 && a.slope != 3)
        return launch_brick64(a, bx, by, bz, g_specialized ? brick_kind(a) : kBrickBounded, s, e0, e1, nparts);
    // the specialised mixed-precision body: periodic in every dimension, no
    // refined cells, no refluxes, the update added to uold
    const bool gen = a.bnd || a.any_ref || a.reflux || a.ubase != a.uold || !g_specialized;
#define RH_LAUNCH_SHAPE(A, B, C)                                                                         \
    if (bx == A && by == B && bz == C) {                                                                 \
        constexpr int nt = (2 * A + 2) * (2 * B + 2);                                                     \
        const int wv = prec == 0 ? RH_BRICK_MIN_WAVES : brick_waves<A, B, C, float, false>();            \
        if (a.slope == 3) {                                                                              \
            if (prec == 0)                                                                               \
                launch_brick(k_godunov3d<A, B, C, double, 0, 3>, nt, C, wv, a, s, e0, e1, nparts);              \
            else                                                                                         \
                launch_brick(k_godunov3d<A, B, C, float, 0, 3>, nt, C, wv, a, s, e0, e1, nparts);               \
        } else if (a.riemann == 3 && !gen) {                                                             \
            launch_brick(k_godunov3d<A, B, C, float, 3, 2, false>, nt, C, wv, a, s, e0, e1, nparts);            \
        } else if (a.riemann == 3) {                                                                     \
            launch_brick(k_godunov3d<A, B, C, float, 3, 2>, nt, C, wv, a, s, e0, e1, nparts);                   \
        } else {                                                                                         \
            launch_brick(k_godunov3d<A, B, C, float, 0, 2>, nt, C, wv, a, s, e0, e1, nparts);                   \
        }                                                                                                \
        return hipGetLastError();                                                                        \
    }
    RH_BRICK_SHAPES(RH_LAUNCH_SHAPE)
#undef RH_LAUNCH_SHAPE
    return hipErrorInvalidValue;
}

int worklist_zsplit(long nbricks, int bx, int by, int bz, int prec)
{
    return zsplit_for(nbricks, bz, (2 * bx + 2) * (2 * by + 2), prec == 0 ? 2 : 4);
}

hipError_t launch_godunov3d_wl(const WorkList &w, int bx, int by, int bz, int slope, int riemann,
                               int prec, hipStream_t s, int kind)
{
    if (w.range[8] <= 0) return hipSuccess;
    if (!g_specialized) kind = kBrickBounded;
    const bool gen = kind != kBrickUniform;
    int maxr = 0;
    for (int r = 0; r < 8; r++) maxr = w.range[r + 1] - w.range[r] > maxr ? w.range[r + 1] - w.range[r] : maxr;
    const int nblocks = 8 * maxr;
    if (prec == 0 && slope != 3) return launch_brick64_wl(w, nblocks, bx, by, bz, riemann, kind, s);
#define RH_LAUNCH_WL(A, B, C)                                                                            \
    if (bx == A && by == B && bz == C) {                                                                 \
        constexpr int nt = (2 * A + 2) * (2 * B + 2);                                                     \
        const dim3 g(nblocks), b(nt);                                                                    \
        if (slope == 3) {                                                                                \
            if (prec == 0)                                                                               \
                hipLaunchKernelGGL((k_godunov3d_wl<A, B, C, double, 0, 3>), g, b, 0, s, w);              \
            else                                                                                         \
                hipLaunchKernelGGL((k_godunov3d_wl<A, B, C, float, 0, 3>), g, b, 0, s, w);               \
        } else if (riemann == 3 && !gen) {                                                               \
            hipLaunchKernelGGL((k_godunov3d_wl<A, B, C, float, 3, 2, false>), g, b, 0, s, w);            \
        } else if (riemann == 3) {                                                                       \
            hipLaunchKernelGGL((k_godunov3d_wl<A, B, C, float, 3, 2>), g, b, 0, s, w);                   \
        } else {                                                                                         \
            hipLaunchKernelGGL((k_godunov3d_wl<A, B, C, float, 0, 2>), g, b, 0, s, w);                   \
        }                                                                                                \
        return hipGetLastError();                                                                        \
    }
    RH_BRICK_SHAPES(RH_LAUNCH_WL)
#undef RH_LAUNCH_WL
    return hipErrorInvalidValue;
}

}  // namespace rh
