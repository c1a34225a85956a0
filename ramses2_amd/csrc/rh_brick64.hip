// FP64 brick kernels: the instances of brick64 and their launches.  Compiled
// once per set of brick shapes (RH_SET), so that the sets build in parallel.
//
// Compiled with NaNs honoured: a level that has lost its state still has a dt (the
// bound that the cells without a NaN give), and the solvers may form a NaN on the
// side of a select that is not taken.  What that costs in quieted operands of
// fmax and fmin is avoided by vmax and vmin of rh_physics64.h.
//
// The scheduler is told to look for instruction-level parallelism: the kernel
// runs at two waves per SIMD whatever its registers (its LDS and 210-250 VGPRs),
// so the default's care for occupancy only lengthens its dependent chains
// (256^3 650 -> 641 us, 128^3 105.5 -> 103 us).
#include "rh_brick64.h"
#include "rh_launch.h"

#ifndef RH_SET
#error "RH_SET selects the brick shapes of this object"
#endif
#define RH_CAT2(a, b) a##b
#define RH_CAT(a, b) RH_CAT2(a, b)
#if RH_SET == 0
#define RH_SHAPES(X) X(7, 7, 8) X(7, 7, 16)
#elif RH_SET == 1
#define RH_SHAPES(X) X(8, 6, 8) X(8, 6, 16)
#elif RH_SET == 2
#define RH_SHAPES(X) X(4, 4, 4) X(4, 4, 8)
#elif RH_SET == 3
#define RH_SHAPES(X) X(15, 7, 8) X(15, 7, 16)
#elif RH_SET == 4
#define RH_SHAPES(X) X(7, 7, 4) X(3, 3, 4)
#else
#define RH_SHAPES(X) X(3, 3, 8) X(1, 1, 1)
#endif

namespace rh {

template <int BX, int BY, int BZ, int RS, int KIND>
__global__ void __launch_bounds__((2 * BX + 2) * (2 * BY + 2), kBrick64Waves) k_brick64(const GodArgs a)
{
    __shared__ Brick64Lds<BX, BY, BZ, KIND != kBrickUniform> sm;
    int bid, zlo, zhi, pslot;
    if (!level_item(a, BZ, bid, zlo, zhi, pslot)) return;
    brick64<BX, BY, BZ, RS, KIND>(a, bid, zlo, zhi, pslot, sm);
}

// Work-list form, see k_godunov3d_wl: workgroup b runs item range[b % 8] + b / 8.
typedef const __attribute__((address_space(4))) GodArgs ConstGodArgs;

template <int BX, int BY, int BZ, int RS, int KIND>
__global__ void __launch_bounds__((2 * BX + 2) * (2 * BY + 2), kBrick64Waves) k_brick64_wl(const WorkList w)
{
    __shared__ Brick64Lds<BX, BY, BZ, KIND != kBrickUniform> sm;
    const int x = blockIdx.x & 7, l = blockIdx.x >> 3;
    const int i = w.range[x] + l;
    if (i >= w.range[x + 1]) return;
    const int4 it = w.items[i];
    const int di = __builtin_amdgcn_readfirstlane(it.x), bid = __builtin_amdgcn_readfirstlane(it.y);
    const int part = __builtin_amdgcn_readfirstlane(it.z), n = __builtin_amdgcn_readfirstlane(it.w);
    auto &a = ((ConstGodArgs *)w.descs)[di];
    int zlo, zhi;
    part_layers(a.zr ? a.zr[bid] : ((BZ - 1) << 16), part, n, zlo, zhi);
    brick64<BX, BY, BZ, RS, KIND>(a, bid, zlo, zhi, bid * n + part, sm);
}

template <int BX, int BY, int BZ, int RS>
static void level_launch(const GodArgs &a, int kind, hipStream_t s, hipEvent_t e0, hipEvent_t e1, int *nparts)
{
    constexpr int nt = (2 * BX + 2) * (2 * BY + 2);
    if (kind == kBrickUniform)
        launch_brick(k_brick64<BX, BY, BZ, RS, kBrickUniform>, nt, BZ, kBrick64Waves, a, s, e0, e1, nparts);
    else if (kind == kBrickPeriodic)
        launch_brick(k_brick64<BX, BY, BZ, RS, kBrickPeriodic>, nt, BZ, kBrick64Waves, a, s, e0, e1, nparts);
    else
        launch_brick(k_brick64<BX, BY, BZ, RS, kBrickBounded>, nt, BZ, kBrick64Waves, a, s, e0, e1, nparts);
}

template <int BX, int BY, int BZ, int RS>
static void list_launch(const WorkList &w, int nblocks, int kind, hipStream_t s)
{
    const dim3 g(nblocks), b((2 * BX + 2) * (2 * BY + 2));
    if (kind == kBrickUniform)
        hipLaunchKernelGGL((k_brick64_wl<BX, BY, BZ, RS, kBrickUniform>), g, b, 0, s, w);
    else if (kind == kBrickPeriodic)
        hipLaunchKernelGGL((k_brick64_wl<BX, BY, BZ, RS, kBrickPeriodic>), g, b, 0, s, w);
    else
        hipLaunchKernelGGL((k_brick64_wl<BX, BY, BZ, RS, kBrickBounded>), g, b, 0, s, w);
}

// The launches of this object's shapes; false for a shape of another set.
bool RH_CAT(brick64_level_, RH_SET)(const GodArgs &a, int bx, int by, int bz, int kind, hipStream_t s, hipEvent_t e0,
                                    hipEvent_t e1, int *nparts)
{
#define RH_ONE(A, B, C)                                                \
    if (bx == A && by == B && bz == C) {                               \
        if (a.riemann == 3)                                            \
            level_launch<A, B, C, 3>(a, kind, s, e0, e1, nparts);       \
        else if (a.riemann == 2)                                       \
            level_launch<A, B, C, 2>(a, kind, s, e0, e1, nparts);       \
        else                                                           \
            level_launch<A, B, C, 1>(a, kind, s, e0, e1, nparts);       \
        return true;                                                   \
    }
    RH_SHAPES(RH_ONE)
#undef RH_ONE
    return false;
}

bool RH_CAT(brick64_list_, RH_SET)(const WorkList &w, int nblocks, int bx, int by, int bz, int riemann, int kind,
                                   hipStream_t s)
{
#define RH_ONE(A, B, C)                                                \
    if (bx == A && by == B && bz == C) {                               \
        if (riemann == 3)                                              \
            list_launch<A, B, C, 3>(w, nblocks, kind, s);               \
        else if (riemann == 2)                                         \
            list_launch<A, B, C, 2>(w, nblocks, kind, s);               \
        else                                                           \
            list_launch<A, B, C, 1>(w, nblocks, kind, s);               \
        return true;                                                   \
    }
    RH_SHAPES(RH_ONE)
#undef RH_ONE
    return false;
}

}  // namespace rh
