"""Blend backward with the FP64 recovery of transmittance: every primitive's T, of
both that a lane holds, comes from the FP64 product.

All primitives are centred on one pixel's centre, where alpha is the opacity to
the bit, a power of two, and only that pixel has a gradient (of 1 for the one
channel).  The colour gradient is then alpha T, an exact product, and T =
T_final / prod (1 - alpha) over the primitives from this one back.  Tolerance: the
one rounding of T to FP32, 2^-24 relative, and 1e-9 for the FP64 scan."""
import numpy as np
import pytest
import torch

from gsplat.cuda import _wrapper as W

pytestmark = pytest.mark.gpu


def cu(a):
    return torch.tensor(np.ascontiguousarray(a), device="cuda")


@pytest.mark.parametrize("n", [16, 33, 64, 97])
@pytest.mark.parametrize("size", [8, 7])  # (7: pixels outside the image, the general tests)
def test_every_transmittance_from_fp64(device, n, size):
    g = np.random.Generator(np.random.PCG64(n))
    m2 = np.full((1, n, 2), 3.5, np.float32)
    cn = np.tile(np.array([0.01, 0.0, 0.01], np.float32), (1, n, 1))
    op = (2.0 ** -g.integers(5, 9, (1, n))).astype(np.float32)
    be = np.full((1, n), 2.0, np.float32)
    col = g.uniform(0, 1, (1, n, 1)).astype(np.float32)
    off, flat = np.zeros((1, 1, 1), np.int32), np.arange(n, dtype=np.int32)
    vrc = np.zeros((1, size, size, 1), np.float32)
    vrc[0, 3, 3] = 1.0
    ins = [cu(a) for a in (m2, cn, col, op, be)]
    _, ra, last, Tf = W.raster_fwd_raw(*ins, None, None, size, size, 8, cu(off), cu(flat))
    W.set_backward_fp64_transmittance(True)
    try:
        got = W.raster_bwd_raw(*ins, None, None, size, size, 8, cu(off), cu(flat), ra, last, Tf, cu(vrc),
                               cu(np.zeros_like(vrc)))[2]
    finally:
        W.set_backward_fp64_transmittance(False)
    a = op[0].astype(np.float64)
    T = float(Tf[0, 3, 3]) / np.cumprod((1.0 - a)[::-1])[::-1]
    err = np.abs(got.cpu().numpy()[0, :, 0] / (a * T) - 1.0)
    assert err.max() < 2.0 ** -24 + 1e-9, err.max()
