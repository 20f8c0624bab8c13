"""Blend of primitives so thin that the determinant of their conic is near FP32's
largest values (2^125 to past 2^128): a line of pixels through their centre, over
the edge between two 8x8 sub-blocks.  No pixel of the line may be culled.

Tolerance: alpha to a few ulp of hardware log2 / exp2, 1e-5 relative."""
import numpy as np
import pytest
import torch

from gsplat.cuda import _wrapper as W

from util import rel_l2

pytestmark = pytest.mark.gpu


def cu(a):
    return torch.tensor(np.ascontiguousarray(a), device="cuda")


@pytest.mark.parametrize("power", [60, 125, 126, 127])
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("ts", [8, 16, 32])
def test_lines_of_pixels(device, power, axis, ts):
    S = 32
    m2 = np.full((1, 1, 2), 4.5, np.float32)
    m2[0, 0, axis] = 8.0
    cn = np.zeros((1, 1, 3), np.float32)
    cn[0, 0, 0 if axis == 0 else 2] = 1.5  # sigma = 1.5 d^2 along the line: pixels at +-0.5
    cn[0, 0, 2 if axis == 0 else 0] = 2.0 ** power
    op, be, col = np.full((1, 1), 0.5, np.float32), np.full((1, 1), 2.0, np.float32), np.ones((1, 1, 3), np.float32)
    n = S // ts
    off = np.arange(n * n, dtype=np.int32).reshape(1, n, n)
    flat = np.zeros(n * n, np.int32)
    ins = [cu(a) for a in (m2, cn, col, op, be)]
    fwd = W._raster_fwd(*ins, None, None, S, S, ts, cu(off), cu(flat), False, keep_masks=True)
    want = np.zeros((S, S))
    line = 0.5 * np.clip(1.0 - 1.5 * (np.arange(S) + 0.5 - 8.0) ** 2, 0, None) ** 2
    if axis == 0:
        want[4] = line
    else:
        want[:, 4] = line
    assert (want > 0).sum() == 2
    assert np.allclose(fwd[1].cpu().numpy()[0, :, :, 0], want, rtol=1e-5, atol=0)
    vrc = cu(np.ones((1, S, S, 3), np.float32))
    vra = cu(np.zeros((1, S, S, 1), np.float32))
    args = (*ins, None, None, S, S, ts, cu(off), cu(flat), fwd[1], fwd[2], fwd[3], vrc, vra)
    for g in (W.raster_bwd_raw(*args), W.raster_bwd_raw(*args, fwd_workspace=fwd[5], entry_masks=fwd[6])):
        assert rel_l2(g[2].cpu().numpy(), np.full((1, 1, 3), want.sum())) < 1e-5
