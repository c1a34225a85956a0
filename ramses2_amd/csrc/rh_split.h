// How many parts along z a launch cuts its bricks into: host arithmetic only.
#pragma once

namespace rh {

// Entries (4 doubles each) of a context's Courant-partial buffer from the start; a
// launch whose bricks are cut writes one per part and never more than these
// (whole bricks: ensure_partials).
constexpr int kMinPartials = 4096;

// Parts along z of each brick of a launch of nbricks bricks of bz oct layers
// and nt threads at `waves` waves per SIMD, on ncu compute units.  A brick marches
// its planes one after another (2.4 us each where it has the CU to itself, 3.5 us
// at two waves per SIMD), so a launch of fewer bricks than the chip holds takes the
// time of one brick, however few they are.  Cutting each brick into n parts
// shortens the march to 2 ceil(bz/n) + 3 planes, at three halo planes more per
// part; n minimises the modelled time while all parts still run at once.
// Bricks of 8x6x8: 32^3 cells in FP64 (12 bricks, 96 parts) 46.8 -> 14.8 us,
// 64^3 (96 bricks, 384 parts) 31.2 -> 29.2 us, mixed 33.5 -> 27 us; mixed 32^3 in
// 4x4x4 bricks 19.4 -> 14.9 us.  Once the whole bricks fill the chip the parts'
// extra planes cost more than the shorter march gains, and they stay whole.
inline int zsplit_parts(long nbricks, int bz, int nt, int waves, int ncu)
{
    const int wg = (nt + 63) / 64;
    const int percu = 4 * waves / wg > 0 ? 4 * waves / wg : 1;
    const long room = (long)percu * ncu < kMinPartials ? (long)percu * ncu : kMinPartials;
    int best = 1;
    double cost = 0;
    for (int n = 1; n <= bz && nbricks * n <= room; n++) {
        const long c = (nbricks * n + ncu - 1) / ncu;   // workgroups per CU
        const double w = c * wg / 4.0;                   // waves per SIMD
        const double t = (2 * ((bz + n - 1) / n) + 3) * (0.54 + 0.46 * (w > 1 ? w : 1.0));
        if (n == 1 || t < 0.97 * cost) {
            best = n;
            cost = t;
        }
    }
    return best;
}

}  // namespace rh
