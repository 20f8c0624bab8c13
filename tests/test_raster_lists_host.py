"""CPU check of the blend kernels' positions in a tile's list (csrc/ubs_raster.h)
against 64-bit arithmetic, with lists that end at the largest index accepted,
2^31 - 1: a 32-bit sum past it turned negative, and the position passed for one
inside the list."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include "ubs_raster.h"
#include <cstdio>
int main() {
    long long checked = 0;
    const int64_t top = 0x7fffffff;
    const int64_t lengths[] = {0, 1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1023, 1025, 3000, top};
    const int batches[] = {64, 256, 1024};
    for (int64_t end : {top, top - 1, top - 300, (int64_t)5000})
        for (int64_t len : lengths)
            for (int bs : batches) {
                const int64_t start = end - len < 0 ? 0 : end - len, n = end - start;
                const int64_t nb = (n + bs - 1) / bs;
                if (ubs::list_batches((int32_t)start, (int32_t)end, bs) != nb) return 1;
                for (int64_t b = nb > 4 ? nb - 4 : 0; b <= nb; ++b) {
                    const int64_t at = b < nb ? start + b * bs : end;
                    for (int ahead : {0, 1, 63, bs - 1, bs, bs + 1, 2 * bs - 1}) {
                        if (ubs::list_has((int32_t)at, ahead, (int32_t)end) != (at + ahead < end)) return 2;
                        ++checked;
                    }
                    if (b == nb) continue;
                    for (int64_t last : {at, at + 1, at + bs - 1, at + bs, end - 1}) {
                        if (last < at || last >= end) continue;
                        const int64_t want = last < at + bs - 1 ? last : at + bs - 1;
                        if (ubs::list_batch_last((int32_t)at, (int32_t)last, bs) != want) return 3;
                        ++checked;
                    }
                }
            }
    printf("%lld\n", checked);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")
def test_list_positions_up_to_the_largest_index(tmp_path):
    src, exe = tmp_path / "drv.cpp", tmp_path / "drv"
    src.write_text(DRIVER)
    subprocess.run(["hipcc", "--cuda-host-only", "-O2", "-std=c++17", "-ftrapv", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "universal-beta-splatting_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.returncode
    assert int(out.stdout) > 1000
