// Launch helpers of the brick kernels: the compiled shapes, launches with
// events, the half-brick split of a launch's last round, and the block to work
// item map of the per-level kernels.
#pragma once
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <map>

#include "rh_godunov.h"

namespace rh {

// Kernel launch, optionally with start/stop events tracked by the dispatch
// itself (hipExtLaunchKernelGGL): timing without separate event packets on
// the stream between the kernels of a step.
template <typename K, typename... Args>
static void launch_ev(K kernel, dim3 g, dim3 b, hipStream_t s, hipEvent_t e0, hipEvent_t e1, Args... args)
{
    if (e0 || e1)
        hipExtLaunchKernelGGL(kernel, g, b, 0, s, e0, e1, 0, args...);
    else
        hipLaunchKernelGGL(kernel, g, b, 0, s, args...);
}

// Compute units of the current device.
inline int device_cus()
{
    static int ncu = 0;
    if (!ncu) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1)
            return 256;
        ncu = n;
    }
    return ncu;
}

// Half-brick split of the final round (GodArgs::nsplit).  With equal work
// per brick, q bricks per XCD on `slots` concurrent workgroups per XCD run in
// ceil(q / slots) rounds; when the last round holds rem = q mod slots <=
// slots/2 bricks, running those rem bricks as 2 rem half-bricks ends the
// launch about half a round earlier (e.g. 352 bricks per XCD on 64 slots:
// 5.53 instead of 6 rounds, by a list-scheduling model).
#ifndef RH_TAIL_SPLIT
#define RH_TAIL_SPLIT 1
#endif
template <typename K> static int tail_split(K kernel, int nthreads, const GodArgs &a)
{
    if (!RH_TAIL_SPLIT || !a.xcd_remap || a.reflux) return 0;
    static std::map<const void *, int> occ_cache;
    const int cus_per_xcd = device_cus() / 8 > 0 ? device_cus() / 8 : 1;
    auto it = occ_cache.find((const void *)kernel);
    int occ;
    if (it == occ_cache.end()) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, nthreads, 0) != hipSuccess) occ = 0;
        occ_cache[(const void *)kernel] = occ;
    } else {
        occ = it->second;
    }
    const int slots = occ * cus_per_xcd, q = a.nbricks >> 3;
    if (slots <= 1 || q <= 0) return 0;
    const int rem = q % slots;
    return rem > 0 && 2 * rem <= slots ? rem : 0;
}

// zsplit_parts on the current device
inline int zsplit_for(long nbricks, int bz, int nt, int waves)
{
    return zsplit_parts(nbricks, bz, nt, waves, device_cus());
}
// z layers [zlo, zhi] of part `part` of n of a brick whose layers are zr (zlo |
// zhi << 16; may be empty: zlo > zhi)
__device__ __forceinline__ void part_layers(int zr, int part, int n, int &zlo, int &zhi)
{
    const int lo = zr & 0xffff, len = (zr >> 16) - lo + 1;
    zlo = lo + len * part / n;
    zhi = lo + len * (part + 1) / n - 1;
}

template <typename K>
static void launch_brick(K kernel, int nt, int bz, int waves, const GodArgs &a0, hipStream_t s, hipEvent_t e0,
                         hipEvent_t e1, int *nparts)
{
    GodArgs a = a0;
    a.zsplit = a.xcd_remap ? zsplit_for(a.nbricks, bz, nt, waves) : 1;
    a.nsplit = a.zsplit > 1 ? 0 : tail_split(kernel, nt, a);
    const int q = a.nbricks >> 3, r = a.nbricks & 7;
    const dim3 g(a.nsplit ? 8 * (q + (r ? 1 : 0) + a.nsplit) : a.nbricks * a.zsplit), b(nt);
    if (nparts) *nparts = a.nbricks * a.zsplit + 8 * a.nsplit;
    launch_ev(kernel, g, b, s, e0, e1, a);
}

// The work item of workgroup blockIdx.x of a per-level launch: brick bid, part
// `part` of n of its z layers (of bz) and its slot among the Courant partials;
// false where the workgroup has none.  Consecutive items go to the same XCD, so
// that the bricks' shared halo octs meet in that XCD's L2.
__device__ __forceinline__ bool level_item(const GodArgs &a, int bz, int &bid, int &zlo, int &zhi, int &pslot)
{
    bid = blockIdx.x;
    int part = 0, n = 1;
    pslot = bid;
    if (a.xcd_remap && a.nsplit == 0) {
        const int nb = gridDim.x, x = bid & 7, l = bid >> 3;
        const int q = nb >> 3, r = nb & 7;
        pslot = x * q + (x < r ? x : r) + l;
        n = a.zsplit;
        bid = pslot / n;
        part = pslot - bid * n;
    } else if (a.xcd_remap) {
        // the last nsplit bricks of each XCD's range run as two work items,
        // one per half of the brick's z layers, so that the final round of
        // workgroups on the XCD is half as long
        const int x = blockIdx.x & 7, l = blockIdx.x >> 3;
        const int q = a.nbricks >> 3, r = a.nbricks & 7, m = a.nsplit;
        const int start = x * q + (x < r ? x : r), count = q + (x < r ? 1 : 0);
        if (l >= count + m) return false;
        if (l < count - m) {
            bid = start + l;
            pslot = bid;
        } else {
            const int j = l - (count - m);
            bid = start + count - m + (j >> 1);
            n = 2;
            part = j & 1;
            // Courant partial of the upper half: after the nbricks whole-brick slots
            pslot = part == 0 ? bid : a.nbricks + x * m + (j >> 1);
        }
    }
    if (bid >= a.nbricks) return false;
    part_layers(a.zr ? a.zr[bid] : ((bz - 1) << 16), part, n, zlo, zhi);
    return true;
}

}  // namespace rh
