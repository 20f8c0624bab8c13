"""Blend backward where a stack of opaque primitives lies just past the image's
edge, in an 8x8 sub-block whose inside pixels still blend what is behind it.
Nothing stops the blend at a pixel outside the image, so the product of
1 / (1 - alpha) over the stack passes FP32's range there (32 alphas of 0.95: 4e41);
no gradient may know of it.

Tolerance as in the other tests of this kernel (2e-3 relative L2): the pixels
inside blend a wide faint primitive or two, and the stack's own gradients are
zero."""
import numpy as np
import pytest
import torch

from gsplat.cuda import _wrapper as W
from oracle import ubs_oracle as O

from util import rel_l2

pytestmark = pytest.mark.gpu


def cu(a):
    return torch.tensor(np.ascontiguousarray(a), device="cuda")


@pytest.mark.parametrize("channels,ts", [(3, 16), (1, 8), (4, 32), (8, 16), (11, 8)])
@pytest.mark.parametrize("opacity,beta", [(0.95, 0.1), (0.997, 0.5), (0.998, 4.0)])
@pytest.mark.parametrize("edge", ["right", "bottom"])
def test_opaque_stack_past_the_edge(device, channels, ts, opacity, beta, edge):
    W_, H_, n = 41, 19, 40
    g = np.random.Generator(np.random.PCG64(channels))
    centre = (44.5, 9.5) if edge == "right" else (20.5, 21.5)  # a pixel's centre
    m2 = np.tile(np.array(centre, np.float32), (1, n + 2, 1))
    m2[0, :n] += g.uniform(-0.05, 0.05, (n, 2)).astype(np.float32)
    cn = np.tile(np.array([1 / 4.0, 0, 1 / 4.0], np.float32), (1, n + 2, 1))  # radius 2: no pixel inside
    op = np.full((1, n + 2), opacity, np.float32)
    be = np.full((1, n + 2), beta, np.float32)
    m2[0, n:] = (20.0, 9.0)  # behind it, two wide faint primitives over the whole image
    cn[0, n:] = (1 / 60.0 ** 2, 0, 1 / 60.0 ** 2)
    op[0, n:], be[0, n:] = 0.2, 2.0
    col = g.uniform(0, 1, (1, n + 2, channels)).astype(np.float32)
    tw, th = -(-W_ // ts), -(-H_ // ts)
    off = np.arange(tw * th, dtype=np.int32).reshape(1, th, tw) * (n + 2)
    flat = np.tile(np.arange(n + 2, dtype=np.int32), tw * th)
    ins = [cu(a) for a in (m2, cn, col, op, be)]
    d = np.float64
    vrc = g.normal(0, 1, (1, H_, W_, channels)).astype(np.float32)
    vra = g.normal(0, 1, (1, H_, W_, 1)).astype(np.float32)
    fwd = W._raster_fwd(*ins, None, None, W_, H_, ts, cu(off), cu(flat), False, keep_masks=True)
    _, ra, last, Tf, _, ws, masks = fwd
    _, wa, wl = O.raster_fwd(*(a.astype(d) for a in (m2, cn, col, op, be)), W_, H_, ts, off, flat)
    want = O.raster_bwd(*(a.astype(d) for a in (m2, cn, col, op, be)), W_, H_, ts, off, flat, wa, wl, vrc.astype(d),
                        vra.astype(d), T_final=1.0 - wa[..., 0])
    args = (*ins, None, None, W_, H_, ts, cu(off), cu(flat), ra, last, Tf, cu(vrc), cu(vra))
    for got in (W.raster_bwd_raw(*args), W.raster_bwd_raw(*args, fwd_workspace=ws, entry_masks=masks)):
        for a, b, name in zip(got, want, ("v_means2d", "v_conics", "v_colors", "v_opac", "v_betas")):
            a = a.cpu().numpy()
            assert np.isfinite(a).all(), name
            assert not a[0, :n].any(), name
            assert rel_l2(a, b) < 2e-3, (name, rel_l2(a, b))
