"""Blend forward, work left out: a sub-block whose pixels are all done, or all
outside the image, evaluates none of the tile's further batches.  The steps are
counted by the counting build of the same kernel (libubs_probe.so)."""
import ctypes
import os

import numpy as np
import pytest
import torch

from gsplat.cuda import _wrapper as W

pytestmark = pytest.mark.gpu


def cu(a):
    return torch.tensor(np.ascontiguousarray(a), device="cuda")


@pytest.mark.parametrize("case", ["half_done", "outside"])
def test_done_waves_take_no_steps(device, case):
    path = os.path.join(os.path.dirname(W.lib().path), "libubs_probe.so")
    probe = ctypes.CDLL(path).ubs_probe_raster_fwd_stats
    vp, u32 = ctypes.c_void_p, ctypes.c_uint32
    probe.argtypes = [u32, u32, ctypes.c_int64] + [vp] * 5 + [u32] * 4 + [vp] * 9
    W_, H_ = (16, 16) if case == "half_done" else (8, 8)
    n, front = 3000, 8
    m2 = np.full((1, n, 2), 8.0, np.float32)
    cn = np.tile(np.array([1e-6, 0, 1e-6], np.float32), (1, n, 1))
    op = np.full((1, n), 1e-3, np.float32)
    be = np.full((1, n), 1.0, np.float32)
    if case == "half_done":  # opaque over the left half (its edge at x = 8)
        m2[0, :front], op[0, :front], be[0, :front] = (-992.0, 8.0), 0.95, 0.01
    col = np.full((1, n, 3), 0.5, np.float32)
    ins = [cu(a) for a in (m2, cn, col, op, be)]
    off, flat = cu(np.zeros((1, 1, 1), np.int32)), cu(np.arange(n, dtype=np.int32))
    rc, ra = torch.empty((1, H_, W_, 3), device="cuda"), torch.empty((1, H_, W_, 1), device="cuda")
    last = torch.empty((1, H_, W_), dtype=torch.int32, device="cuda")
    Tf = torch.empty((1, H_, W_), device="cuda")
    ws = torch.empty((int(W.lib().ubs_rasterize_workspace_bytes(1, n, 1)),), dtype=torch.uint8, device="cuda")
    stats = torch.zeros(5, dtype=torch.int64, device="cuda")
    p = W.ptr
    assert probe(1, n, n, p(ins[0]), p(ins[1]), p(ins[2]), p(ins[3]), p(ins[4]), W_, H_, 1, 1, p(off), p(flat), p(rc),
                 p(ra), p(last), p(Tf), p(ws), p(stats), W.stream_of(rc)) == 0
    want = W.raster_fwd_raw(*ins, None, None, W_, H_, 16, off, flat)
    for a, b in zip((rc, ra, last, Tf), want):
        assert torch.equal(a, b)
    steps, live = int(stats[0]), int((Tf.amax(dim=(0, 1)) > 1e-2).sum()) // 8  # columns of 8 pixels still blending
    assert live == 1
    waves = 2 if case == "half_done" else 1
    assert waves * (n - front) <= steps <= waves * n + 2 * (front + 2), steps
