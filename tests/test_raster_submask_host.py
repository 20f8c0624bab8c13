"""CPU check of the sub-block mask of all sub-blocks of a tile at once
(csrc/ubs_raster.h, subblock_mask_exact) against the test of one rectangle at
a time and against the pixels themselves: no pixel whose fp32 sigma the blend
accepts lies in a sub-block the mask leaves out, and the mask keeps at most 2 %
more sub-blocks than the per-rectangle test (their margins differ by 1e-5 of
the form's terms over a tile, which widens an ellipse's reach by less than a
hundredth of a pixel but for needles)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#pragma clang fp contract(off)
#include "ubs_raster.h"
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
template <int SB>
void run(int n, int seed) {
    std::mt19937_64 rng(seed);
    std::uniform_real_distribution<double> U(0, 1);
    long long ours = 0, each = 0, bad = 0;
    const double lo = log(4e-4), hi = log(3.3);
    for (int k = 0; k < n; ++k) {
        const double l1 = exp(lo + U(rng) * (hi - lo)), l2 = exp(lo + U(rng) * (hi - lo));
        // rotated, axis-aligned (b = 0 or -0) and circular ones; centres on and off the pixel grid
        const double th = k % 5 ? U(rng) * M_PI : 0, cs = cos(th), sn = sin(th), l3 = k % 7 ? l2 : l1;
        const float a = (float)(l1 * cs * cs + l3 * sn * sn), c = (float)(l1 * sn * sn + l3 * cs * cs);
        const float b = (float)((l1 - l3) * cs * sn);
        float mx = (float)(U(rng) * 2000 - 40), my = (float)(U(rng) * 1100 - 40);
        if (k % 3 == 0) { mx = floorf(mx) + 0.5f; my = floorf(my); }
        const float det = a * c - b * b;
        if (!(det > 0)) continue;
        const float hx = sqrtf(c / det) * 1.001f + 1e-3f, hy = sqrtf(a / det) * 1.001f + 1e-3f;
        const int T = 8 * SB;
        for (int ty = (int)floorf((my - hy) / T); ty <= (int)floorf((my + hy) / T); ++ty)
            for (int tx = (int)floorf((mx - hx) / T); tx <= (int)floorf((mx + hx) / T); ++tx) {
                const float x0 = (float)(tx * T), y0 = (float)(ty * T);
                const uint32_t m = ubs::subblock_mask_exact<SB>(mx, my, a, b, c, hx, hy, x0, y0);
                const uint32_t box = ubs::subblock_mask<SB>(mx, my, hx, hy, x0, y0);
                for (int s = 0; s < SB * SB; ++s) {
                    const float lx = x0 + (float)(s % SB * 8) + 0.5f, ly = y0 + (float)(s / SB * 8) + 0.5f;
                    if ((box >> s) & 1u)
                        each += ubs::ellipse_meets_rect(mx, my, a, b, c, lx, lx + 7.f, ly, ly + 7.f);
                    if ((m >> s) & 1u) { ++ours; continue; }
                    for (int l = 0; l < 64; ++l) {
                        const float dx = mx - (lx + (float)(l & 7)), dy = my - (ly + (float)(l >> 3));
                        const float q = fmaf(2.f * b * dx, dy, fmaf(a * dx, dx, (c * dy) * dy));
                        if (q >= 0.f && q < 1.f) ++bad;
                    }
                }
            }
    }
    printf("%lld %lld %lld\n", ours, each, bad);
}
// a conic that is no ellipse keeps what the box test says: everything, or nothing
template <int SB>
int odd() {
    const float inf = INFINITY;
    const uint32_t all = (uint32_t)((1ull << (SB * SB)) - 1);
    return ubs::subblock_mask_exact<SB>(3, 3, 1, 2, 1, inf, inf, 0, 0) == all &&
           ubs::subblock_mask_exact<SB>(3, 3, -1, 0, -1, NAN, NAN, 0, 0) == 0 &&
           ubs::subblock_mask_exact<SB>(NAN, 3, 1, 0, 1, 1, 1, 0, 0) == 0;
}
int main(int argc, char **argv) {
    const int n = atoi(argv[1]), seed = atoi(argv[2]);
    run<1>(n, seed); run<2>(n, seed); run<4>(n, seed);
    printf("%d\n", odd<1>() && odd<2>() && odd<4>());
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")
def test_tile_mask_against_one_rectangle_at_a_time(tmp_path):
    src, exe = tmp_path / "drv.cpp", tmp_path / "drv"
    src.write_text(DRIVER)
    subprocess.run(["hipcc", "--cuda-host-only", "-O2", "-std=c++17", "-ffp-contract=off",
                    "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "universal-beta-splatting_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    for seed in (1, 2):
        out = subprocess.run([str(exe), "40000", str(seed)], check=True, capture_output=True, text=True,
                             timeout=300).stdout.split("\n")
        for line in out[:3]:
            ours, each, bad = map(int, line.split())
            assert bad == 0, f"{bad} accepted pixels in sub-blocks left out"
            assert ours <= 1.02 * each, (ours, each)
        assert out[3] == "1"
