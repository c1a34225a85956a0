// Refinement flags of a level from its current state: hydro_flag
// (hydro/hydro_flag.f90:7-159) with the density and pressure gradient
// criteria of hydro_refine (hydro/godunov_utils.f90:6-227), one thread per
// cell, into a device-resident flag1 array, and the flag1 helpers of the
// reference's Metal bridge (metal/metal_interface.f90:225-241 and around).
//
// For each cell and each of its 2*ndim face neighbours, the neighbour cell
// (key at level l+1, periodic directions wrapped) is read from the level-l
// oct that holds it, or, when that oct is not one of the level's own, from
// the cell of level l-1 that holds it; keys outside the box read the
// boundary oct built from the reference oct inside (init_bound_refine).
// The three values of each direction (left, cell, right) go through
// hydro_refine's arithmetic in its order, with no FMA contraction, so that
// the flags agree with the reference's cell for cell.
#include <hip/hip_runtime.h>

#include "../../include/ramses2_hip.h"
#include "../../include/ramses2_hip_ext.h"
#include "rh_gather.h"
#include "rh_mesh.h"
#include "rh_state.h"

namespace rh {

struct FlagArgs {
    const double *uold;
    const uint8_t *refined;
    int32_t *flag1;      // [ngridmax][8]
    const int32_t *ckey; // [ngrid][3]
    int head, noct;
    ResolveCtx fine, coarse;  // levels l and l-1 (coarse.nx == 0: none)
    int cmin[3], cmax[3];     // box at level l+1 (cell keys)
    int periodic[3];
    int refl;                 // reflexive faces (bit 2*dim+side)
    double gamma, smallr, err_d, err_p, floor_d, floor_p;
    int *counter;             // [1] a neighbour's cell missing
};

// Density and pressure of a cell as hydro_refine forms them from a
// conservative state, in the reference's order.
__device__ __forceinline__ void cell_dp(const FlagArgs &a, const double u[5], double &r, double &p)
{
#pragma clang fp contract(off)
    r = u[0] > a.smallr ? u[0] : a.smallr;
    double ekin = 0.0;
#pragma unroll
    for (int d = 1; d <= 3; d++) {
        const double v = u[d] / r;
        ekin = ekin + 0.5 * r * (v * v);
    }
    p = (a.gamma - 1.0) * (u[4] - ekin);
}

// hydro_refine's density and pressure tests for one direction (densities and
// pressures of the left cell, the cell and the right cell), in the reference's
// order.
__device__ __forceinline__ bool refine_dp(const FlagArgs &a, double rg, double pg, double rm, double pm, double rd,
                                          double pd)
{
#pragma clang fp contract(off)
    bool ok = false;
    if (a.err_d >= 0.0) {
        const double x = __builtin_fabs((rd - rm) / (rd + rm + a.floor_d));
        const double y = __builtin_fabs((rm - rg) / (rm + rg + a.floor_d));
        ok = ok || 2.0 * (x > y ? x : y) > a.err_d;
    }
    if (a.err_p >= 0.0) {
        const double x = __builtin_fabs((pd - pm) / (pd + pm + a.floor_p));
        const double y = __builtin_fabs((pm - pg) / (pm + pg + a.floor_p));
        ok = ok || 2.0 * (x > y ? x : y) > a.err_p;
    }
    return ok;
}

// Eight lanes per oct, one per cell.  The pass is bound by the latency of its
// dependent gathers (key, hash table, cell), so the lanes share them: six of
// them look up one neighbour oct each (a lookup per cell and neighbour was
// eight times as many), and of a cell's six neighbours the three in its own oct
// give their density and pressure through the lanes, so four cells are read and
// divided per lane instead of seven.  No count is kept (one address that every
// flagged cell added to).  96 -> 26 us per level on average, 297 k octs on five
// levels.
__global__ void __launch_bounds__(256) k_hydro_flag(const FlagArgs a)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)a.noct * 8) return;  // (whole octs: the eight lanes of one leave together)
    const int o = a.head - 1 + (int)(i >> 3), ind = (int)(i & 7), oct0 = threadIdx.x & 56;
    const int ck[3] = {a.ckey[3 * o], a.ckey[3 * o + 1], a.ckey[3 * o + 2]};
    // the neighbour cell across side sd of the oct in dimension d: the key kp of
    // its oct, its place c there
    auto beyond = [&](int d, int sd, int kp[3], int c[3]) {
#pragma unroll
        for (int e = 0; e < 3; e++) {
            int kn = 2 * ck[e] + ((ind >> e) & 1);
            if (e == d) {
                kn = 2 * ck[e] + (sd ? 2 : -1);
                if (a.periodic[e]) {
                    if (kn < a.cmin[e]) kn = a.cmax[e] - 1;
                    if (kn >= a.cmax[e]) kn = a.cmin[e];
                }
            }
            kp[e] = kn >> 1;
            c[e] = kn & 1;
        }
    };
    // lane 2d + sd of the oct: the oct there, or the one of level l-1 that holds
    // the neighbour cells where it is not one of the level's own; 0: neither
    int nb = 0, up = 0;
    if (ind < 6) {
        int kp[3], c[3];
        beyond(ind >> 1, ind & 1, kp, c);
        nb = resolve_oct(a.fine, kp[0], kp[1], kp[2]);
        if (nb > a.fine.ngridmax || nb == 0) {
            up = 1;
            nb = a.coarse.nx ? resolve_oct(a.coarse, kp[0] >> 1, kp[1] >> 1, kp[2] >> 1) : 0;
            if (nb > a.coarse.ngridmax) nb = 0;
        }
    }
    double um[5], r0, p0;
#pragma unroll
    for (int n = 0; n < 5; n++) um[n] = a.uold[(size_t)o * 40 + n * 8 + ind];
    cell_dp(a, um, r0, p0);
    bool ok = false, missing = false;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const int sd = (ind >> d) & 1;
        const int v = __shfl(nb, oct0 + 2 * d + sd), u = __shfl(up, oct0 + 2 * d + sd);
        const double rs = __shfl_xor(r0, 1 << d), ps = __shfl_xor(p0, 1 << d);
        int kp[3], c[3];
        beyond(d, sd, kp, c);
        if (u)
#pragma unroll
            for (int e = 0; e < 3; e++) {
                c[e] = kp[e] & 1;
                kp[e] >>= 1;
            }
        missing = missing || v == 0;
        const CellRef cr = cell_ref3(a.uold, a.refined, v, kp, u ? a.coarse.boxmin : a.fine.boxmin,
                                     u ? a.coarse.boxmax : a.fine.boxmax, a.refl, c);
        double un[5], rn, pn;
#pragma unroll
        for (int n = 0; n < 5; n++) un[n] = cr.p ? cr.p[8 * n] : 0.0;
        cell_dp(a, un, rn, pn);  // (a reflexive ghost's momentum sign drops out)
        ok = refine_dp(a, sd ? rs : rn, sd ? ps : pn, r0, p0, sd ? rn : rs, sd ? pn : ps) || ok;
    }
    if (missing)
        atomicOr(&a.counter[1], 1);
    else if (ok)
        a.flag1[(size_t)o * 8 + ind] = 1;
}

__global__ void k_fill_flag1(int32_t *flag1, long first, long n, int32_t v)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flag1[first + i] = v;
}

// Nonzero flags of n/8 octs (n is a multiple of 8), one atomic per block of a
// grid of at most kCountBlocks: device-scope additions to one address take
// about 40 ns each, one after another (a sum per wave: 40 us, now 3.8).
constexpr int kCountBlocks = 128;
__global__ void __launch_bounds__(256) k_count_flag1(const int4 *__restrict__ flag, long n4, int *count)
{
    int v = 0;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (long)gridDim.x * blockDim.x) {
        const int4 f = flag[i];
        v += (f.x != 0) + (f.y != 0) + (f.z != 0) + (f.w != 0);
    }
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __shared__ int w[4];
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
    __syncthreads();
    v = w[0] + w[1] + w[2] + w[3];
    if (threadIdx.x == 0 && v) atomicAdd(count, v);
}

}  // namespace rh

using namespace rh;

namespace {

int efail(int code, const std::string &msg)
{
    set_error(msg);
    return code;
}

int ensure_flag1()
{
    State &s = st();
    if (!s.inited || !s.uold) return efail(RH_ERR_STATE, "library not initialised / mesh not allocated");
    if (s.ndim != 3) return efail(RH_ERR_ARG, "refinement flags are computed for 3D meshes");
    if (!s.flag1) {
        const size_t n = (size_t)s.ngridmax * 8;
        RH_HIP_CHECK(dmalloc((void **)&s.flag1, n * sizeof(int32_t)));
        hipLaunchKernelGGL(k_fill_flag1, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s.stream, s.flag1, 0l,
                           (long)n, 0);
        RH_HIP_CHECK(hipGetLastError());
    }
    return 0;
}

int oct_range(int head_idx, int num_octs)
{
    const State &s = st();
    if (head_idx < 1 || num_octs < 0 || (int64_t)head_idx - 1 + num_octs > s.ngridmax)
        return efail(RH_ERR_ARG, "oct range out of bounds (flags cover octs 1..ngridmax)");
    return 0;
}

ResolveCtx level_ctx(int l)
{
    const State &s = st();
    ResolveCtx c;
    c.keys = s.hkeys;
    c.vals = s.hvals;
    c.cap = (uint64_t)s.hash_cap;
    c.koff = s.key_off[l - 1];
    c.nx = s.ckey_max[l - 1];
    c.ndim = s.ndim;
    c.ngridmax = s.ngridmax;
    for (int d = 0; d < 3; d++) {
        c.boxmin[d] = s.box_min[3 * (l - 1) + d];
        c.boxmax[d] = s.box_max[3 * (l - 1) + d];
        c.periodic[d] = s.periodic[d];
    }
    return c;
}

}  // namespace

extern "C" {

int rh_reset_flag1(int head_idx, int num_octs)
{
    if (int r = ensure_flag1()) return r;
    if (int r = oct_range(head_idx, num_octs)) return r;
    State &s = st();
    if (num_octs == 0) return 0;
    const long n = (long)num_octs * 8;
    hipLaunchKernelGGL(k_fill_flag1, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s.stream, s.flag1,
                       (long)(head_idx - 1) * 8, n, 0);
    RH_HIP_CHECK(hipGetLastError());
    return 0;
}

int rh_hydro_flag(int head_idx, int num_octs, double gamma, double smallr, double smallc2, double err_grad_d,
                  double err_grad_p, double floor_d, double floor_p)
{
    (void)smallc2;
    if (int r = ensure_flag1()) return r;
    if (int r = oct_range(head_idx, num_octs)) return r;
    State &s = st();
    if (num_octs == 0) return 0;
    if (err_grad_d == -1.0 && err_grad_p == -1.0) return 0;  // no gradient criterion (hydro_flag.f90:49-62)
    if (!(gamma > 1.0)) return efail(RH_ERR_ARG, "rh_hydro_flag: gamma must exceed 1");
    const int l = s.h_lev[head_idx - 1];
    if (l < 1 || l > s.nlevelmax) return efail(RH_ERR_MESH, "oct level outside the level parameters");
    for (int i = head_idx - 1; i < head_idx - 1 + num_octs; i++)
        if (s.h_lev[i] != l) return efail(RH_ERR_MESH, "octs of the range are not all on one level");
    FlagArgs a;
    a.uold = s.uold;
    a.refined = s.refined;
    a.flag1 = s.flag1;
    a.ckey = s.ckey;
    a.head = head_idx;
    a.noct = num_octs;
    a.fine = level_ctx(l);
    if (l > 1)
        a.coarse = level_ctx(l - 1);
    else
        a.coarse.nx = 0;
    for (int d = 0; d < 3; d++) {
        a.cmin[d] = s.box_min[3 * l + d];  // box of level l+1
        a.cmax[d] = s.box_max[3 * l + d];
        a.periodic[d] = s.periodic[d];
    }
    a.refl = 0;
    for (int d = 0; d < 3; d++)
        for (int sd = 0; sd < 2; sd++) a.refl |= (s.btype[d][sd] == 1) << (2 * d + sd);
    a.gamma = gamma;
    a.smallr = smallr;
    a.err_d = err_grad_d;
    a.err_p = err_grad_p;
    a.floor_d = floor_d;
    a.floor_p = floor_p;
    a.counter = s.d_counter;
    RH_HIP_CHECK(hipMemsetAsync(s.d_counter, 0, 2 * sizeof(int), s.stream));
    const long n = (long)num_octs * 8;
    hipLaunchKernelGGL(k_hydro_flag, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s.stream, a);
    RH_HIP_CHECK(hipGetLastError());
    int hc[2] = {0, 0};
    RH_HIP_CHECK(hipMemcpyAsync(hc, s.d_counter, 2 * sizeof(int), hipMemcpyDeviceToHost, s.stream));
    RH_HIP_CHECK(hipStreamSynchronize(s.stream));
    if (hc[1]) return efail(RH_ERR_MESH, "hydro_flag: a neighbour cell has no parent cell on the coarser level");
    return 0;
}

int rh_count_flag1(int head_idx, int num_octs, int32_t *count)
{
    if (int r = ensure_flag1()) return r;
    if (int r = oct_range(head_idx, num_octs)) return r;
    if (!count) return efail(RH_ERR_ARG, "rh_count_flag1: null count");
    State &s = st();
    *count = 0;
    if (num_octs == 0) return 0;
    const long n = (long)num_octs * 8;
    RH_HIP_CHECK(hipMemsetAsync(s.d_counter, 0, sizeof(int), s.stream));
    const long n4 = n / 4, nb = (n4 + 255) / 256;
    hipLaunchKernelGGL(k_count_flag1, dim3((unsigned)(nb < kCountBlocks ? nb : kCountBlocks)), dim3(256), 0, s.stream,
                       (const int4 *)(s.flag1 + (size_t)(head_idx - 1) * 8), n4, s.d_counter);
    RH_HIP_CHECK(hipGetLastError());
    int c = 0;
    RH_HIP_CHECK(hipMemcpyAsync(&c, s.d_counter, sizeof(int), hipMemcpyDeviceToHost, s.stream));
    RH_HIP_CHECK(hipStreamSynchronize(s.stream));
    *count = c;
    return 0;
}

int rh_upload_flag1(const int32_t *flag1, int ngridmax)
{
    if (int r = ensure_flag1()) return r;
    State &s = st();
    if (!flag1 || ngridmax != s.ngridmax) return efail(RH_ERR_ARG, "rh_upload_flag1: flag1(8, ngridmax) expected");
    RH_HIP_CHECK(hipMemcpyAsync(s.flag1, flag1, (size_t)ngridmax * 8 * sizeof(int32_t), hipMemcpyHostToDevice,
                                s.stream));
    RH_HIP_CHECK(hipStreamSynchronize(s.stream));
    return 0;
}

int rh_get_flag1(int head_idx, int num_octs, int32_t *flag1)
{
    if (int r = ensure_flag1()) return r;
    if (int r = oct_range(head_idx, num_octs)) return r;
    if (num_octs == 0) return 0;
    if (!flag1) return efail(RH_ERR_ARG, "rh_get_flag1: null flag1");
    State &s = st();
    RH_HIP_CHECK(hipMemcpyAsync(flag1, s.flag1 + (size_t)(head_idx - 1) * 8, (size_t)num_octs * 8 * sizeof(int32_t),
                                hipMemcpyDeviceToHost, s.stream));
    RH_HIP_CHECK(hipStreamSynchronize(s.stream));
    return 0;
}

int rh_transfer_flag1_host(int32_t *flag1, int ngridmax)
{
    if (int r = ensure_flag1()) return r;
    State &s = st();
    if (!flag1 || ngridmax != s.ngridmax) return efail(RH_ERR_ARG, "rh_transfer_flag1_host: flag1(8, ngridmax) expected");
    RH_HIP_CHECK(hipMemcpyAsync(flag1, s.flag1, (size_t)ngridmax * 8 * sizeof(int32_t), hipMemcpyDeviceToHost,
                                s.stream));
    RH_HIP_CHECK(hipStreamSynchronize(s.stream));
    return 0;
}

}  // extern "C"
