"""CPU checks of the direct placement's task plan (csrc/ubs_isect.h) and its
workspace: no patch has more tasks than its table of counts holds, whatever part
of the pairs reaches it; scenes of few pairs get a workspace of their own size on
any grid; the limits of the grid."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include "ubs_isect.h"
#include <cstdio>
#include <random>
#include <vector>
using namespace ubs;
int main() {
    std::mt19937_64 rng(3);
    std::vector<uint32_t> blocks;
    for (uint32_t b = 1; b <= 3000; ++b) blocks.push_back(b);
    for (uint32_t b = 3000; b < (1u << 21); b = b * 21 / 20 + 1) blocks.push_back(b);
    blocks.push_back(1u << 21);
    long long checked = 0, raised = 0;
    for (uint32_t b : blocks) {
        const uint32_t most = bins_most_tasks(b);
        const uint64_t pairs = std::min<uint64_t>(1024ull * b, (1ull << 31) - 1);
        for (int k = 0; k < 40; ++k) {
            const uint32_t total = k == 0 ? (uint32_t)pairs : k == 1 ? 0u : (uint32_t)(rng() % (pairs + 1) >> (k % 5));
            const uint32_t aim = bins_task_aim(total, most), floor = bins_block_floor(aim);
            const uint64_t work = (uint64_t)total + (uint64_t)floor * b;
            if (work >= 1ull << 32) return 1;      // the kernel's sums have 32 bits
            if (work / aim + 1 > most) return 2;   // more tasks than rows of counts
            if (aim / floor > 60) return 3;        // a task of more than 61 blocks
            if (b < 448 && aim != kTaskPairs) return 4;
            raised += aim != kTaskPairs;
            ++checked;
        }
    }
    printf("%lld %lld\n", checked, raised);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")
def test_tasks_fit_their_table(tmp_path):
    src, exe = tmp_path / "drv.cpp", tmp_path / "drv"
    src.write_text(DRIVER)
    subprocess.run(["hipcc", "--cuda-host-only", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "universal-beta-splatting_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.returncode
    checked, raised = map(int, out.stdout.split())
    assert checked > 100000 and raised > 1000


def test_workspace_follows_the_pairs():
    from gsplat.cuda._backend import lib

    size = lib().ubs_isect_bins_workspace_bytes
    patches = 16 * 32  # 512 x 512 tiles
    # 2 KB of counts a task, at most 2.3 tasks per 1024 pairs and 2 more; a bit a pair and patch; 16 bytes a pair
    for n in (1, 1000, 10_000, 200_000, 450_000):
        blocks = -(-n // 1024)
        most = patches * 2048 * (2.3 * blocks + 2) + patches * blocks * (128 + 4 + 10) + 16 * n + 1100 * 1024 + patches * 20
        assert 0 < size(1, n, 512, 512) <= most, (n, size(1, n, 512, 512), most)
    assert size(1, 10_000, 512, 512) < 30 << 20
    assert size(1, 10_000, 512, 513) == 0 and size(1, 10_000, 513, 512) == 0  # 513 rows or columns: a patch more
    assert size(2, 10_000, 512, 256) > 0 and size(2, 10_000, 512, 257) == 0
    assert size(1, 10_000, 65536, 1) == 0


def test_the_placement_is_taken_where_it_is_faster():
    """The rule at sizes measured on both ways (us placed / sorted beside them)."""
    from gsplat.cuda._backend import lib

    pays = lib().ubs_isect_bins_pays
    for C, N, tw, th, n, want in (
            (1, 1_000_000, 120, 68, 5_783_480, 1),     # 267 / 399
            (1, 1_000_000, 120, 68, 57_081, 1),        # 221 / 251
            (2, 1_000_000, 120, 68, 117_066, 1),       # 292 / 296
            (4, 1_000_000, 120, 68, 23_131_325, 1),    # 819 / 1084
            (4, 1_000_000, 120, 68, 230_382, 0),       # 492 / 443
            (8, 1_000_000, 120, 68, 46_244_700, 1),    # 1834 / 2295
            (8, 1_000_000, 120, 68, 461_549, 0),       # 1028 / 746
            (8, 100_000, 120, 68, 4_623_075, 1),       # 381 / 420
            (8, 100_000, 120, 68, 46_389, 0),          # 319 / 255
            (2, 1_000_000, 240, 135, 11_639_522, 1),   # 608 / 714
            (2, 1_000_000, 240, 135, 115_285, 0),      # 425 / 312
            (1, 10_000, 512, 512, 58_877, 0),          # 530 / 214
            (1, 10_000, 512, 512, 616, 1),             # 530 / 1303
            (1, 1_000_000, 512, 512, 5_853_432, 0),    # 872 / 465
            (1, 1_000_000, 256, 256, 5_832_977, 1),    # 410 / 460
            (1, 1_000_000, 1, 1, 1_000_000, 0),        # 430 / 249
            (1, 100_000, 2, 2, 274_376, 0),            # 211 / 182
            (1, 1_000_000, 8, 8, 4_968_502, 1),        # 272 / 326
            (1, 1_000_000, 120, 68, 0, 1)):
        assert pays(C, N, tw, th, n) == want, (C, N, tw, th, n)
        assert pays(C, N, tw, th, -1) in (want, 2)
    assert pays(1, 1_000_000, 120, 68, -1) == 1 and pays(1, 1_000_000, 512, 512, -1) == 2
    assert pays(1, 1_000_000, 512, 513, 10 ** 9) == 0 and pays(1, 0, 120, 68, 0) == 0  # past the limits, no pairs
