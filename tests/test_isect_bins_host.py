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
