"""Blend forward at the edges of its lists: every way an entry may be evaluated
(alpha below its clamp, at the clamp, or only by the general code: negative or
huge opacity, negative beta, a conic with a zero entry), alone and mixed; list
lengths around a step, a wave and a batch; pixels that end inside a step; all
tile sizes and colour layouts.

Tolerance: an alpha is off by beta |log2(1 - sigma)| 2^-22 plus a few ulp, under
5e-6 relative where its weight is not negligible; weights sum to at most one, so
colours in [0, 1] move by at most n times that in the worst order and by its
square root in practice: 1e-4 absolute at n = 300 covers it.  Behind an alpha
near its clamp the error of 1 - alpha counts up to 1e3-fold, with T below 1e-3
by then.  last_ids are exact where FP32 and FP64 take the same branches.
"""
import numpy as np
import pytest
import torch

from gsplat.cuda import _wrapper as W
from oracle import ubs_oracle as O

pytestmark = pytest.mark.gpu


def _case(n, W_, H_, channels, mode, ts, seed):
    g = np.random.Generator(np.random.PCG64(seed))
    m2 = g.uniform((0, 0), (W_, H_), (1, n, 2)).astype(np.float32)
    s = g.uniform(3.0, 12.0, (n, 2))
    t = g.uniform(0, np.pi, n)
    R = np.stack([np.cos(t), -np.sin(t), np.sin(t), np.cos(t)], 1).reshape(n, 2, 2)
    ci = np.linalg.inv(R @ (s[:, :, None] ** 2 * np.eye(2)) @ R.transpose(0, 2, 1))
    cn = np.stack([ci[:, 0, 0], ci[:, 0, 1], ci[:, 1, 1]], 1)[None].astype(np.float32)
    op = g.uniform(0.02, 0.2, (1, n)).astype(np.float32)
    be = (4 * np.exp(g.normal(0, 0.5, (1, n)))).astype(np.float32)
    pick = g.integers(0, n, max(1, n // 16))
    if mode in ("clamp", "all"):
        op[0, pick] = 0.9995
        be[0, pick] = 0.3
    if mode in ("general", "all"):
        i = (pick + 1) % n
        op[0, i[0::4]] = -0.05        # T rises again
        op[0, i[1::4]] = 3e30
        be[0, i[2::4]] = -0.5
        cn[0, i[3::4], :2] = 0.0      # a band across the image
    col = g.uniform(0, 1, (1, n, channels)).astype(np.float32)
    tw, th = -(-W_ // ts), -(-H_ // ts)
    off = np.arange(tw * th, dtype=np.int32).reshape(1, th, tw) * n
    flat = np.tile(np.arange(n, dtype=np.int32), tw * th)
    return m2, cn, col, op, be, off, flat


@pytest.mark.parametrize("mode", ["plain", "clamp", "general", "all"])
@pytest.mark.parametrize("n,channels,ts", [(1, 3, 16), (2, 3, 16), (3, 1, 16), (63, 2, 16), (65, 4, 16), (64, 3, 8),
                                           (67, 8, 8), (255, 3, 16), (257, 3, 16), (300, 3, 32), (300, 8, 16)])
def test_blend_forward_list_edges(device, n, channels, ts, mode):
    W_, H_ = 43, 21  # ragged: outside pixels in every tile of the last row and column
    m2, cn, col, op, be, off, flat = _case(n, W_, H_, channels, mode, ts, 10 * n + channels)
    rc, ra, last, Tf = W.raster_fwd_raw(*(torch.tensor(a, device="cuda") for a in (m2, cn, col, op, be)), None, None,
                                        W_, H_, ts, torch.tensor(off, device="cuda"),
                                        torch.tensor(flat, device="cuda"))
    d = np.float64
    wc, wa, wl, mT, mS = O.raster_fwd(*(a.astype(d) for a in (m2, cn, col, op, be)), W_, H_, ts, off, flat,
                                      margins=True)
    safe = (mT > 1e-3) & (mS > 1e-6)  # pixels whose branches FP32 and FP64 take alike
    assert safe.mean() > 0.5
    assert np.array_equal(last.cpu().numpy()[safe], wl[safe])
    assert np.abs(rc.cpu().numpy() - wc)[safe].max() < 1e-4
    assert np.abs(ra.cpu().numpy() - wa)[safe].max() < 1e-4
    assert np.abs((1.0 - Tf.cpu().numpy())[..., None] - wa)[safe].max() < 1e-4
