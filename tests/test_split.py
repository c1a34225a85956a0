"""Parts along z of a launch (rh_split.h, host arithmetic compiled here): for every
brick shape, waves per SIMD and size of chip, a cut launch writes no more Courant
partials than a context has from the start, and all its parts run at once; whole
bricks need one each."""
import os
import subprocess

from ramses2_amd.build import CSRC

SRC = r"""
#include <stdio.h>
#include "rh_split.h"
int main()
{
    const int shapes[][3] = {{7, 7, 8}, {7, 7, 16}, {8, 6, 8}, {8, 6, 16}, {4, 4, 4}, {4, 4, 8}, {15, 7, 8},
                             {15, 7, 16}, {7, 7, 4}, {3, 3, 4}, {3, 3, 8}, {1, 1, 1}};
    const int cus[] = {1, 38, 80, 256, 304, 512, 1024};
    long bad = 0, cut = 0;
    for (auto &b : shapes)
        for (int waves = 1; waves <= 4; waves++)
            for (int ncu : cus)
                for (long nb = 1; nb <= 6000; nb++) {
                    const int nt = (2 * b[0] + 2) * (2 * b[1] + 2), wg = (nt + 63) / 64;
                    const int n = rh::zsplit_parts(nb, b[2], nt, waves, ncu);
                    const int percu = 4 * waves / wg > 0 ? 4 * waves / wg : 1;
                    if (n < 1 || n > b[2] || (n > 1 && (nb * n > rh::kMinPartials || nb * n > (long)percu * ncu)))
                        bad++;
                    cut += n > 1;
                }
    printf("%ld %ld\n", bad, cut);
    return 0;
}
"""


def test_parts_fit_the_partials(tmp_path):
    src, exe = tmp_path / "split.cpp", tmp_path / "split"
    src.write_text(SRC)
    cxx = os.environ.get("CXX", "g++")
    subprocess.run([cxx, "-O1", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    bad, cut = map(int, subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split())
    assert bad == 0
    assert cut > 1000
