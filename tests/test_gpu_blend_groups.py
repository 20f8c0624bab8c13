"""Blend backward at the edges of its groups: lists of every length around 16
and 32 primitives per 8x8 sub-block (a lane holds one or two), groups that
take the general tests (alpha at its clamp, beta below one, pixels that end
early) between plain ones, and the sub-block masks the forward keeps against
the tests the backward makes itself.

Tolerance: the FP32 recovery of T over at most 129 divisors is off by at most
129 x 2^-22 = 3e-5 relative, and alphas at the 0.999 clamp multiply rounding by
up to 1000 in the terms behind them; 2e-3 relative L2, as in the other tests of
this kernel.
"""
import numpy as np
import pytest
import torch

from gsplat.cuda import _wrapper as W
from oracle import ubs_oracle as O

from util import rel_l2

pytestmark = pytest.mark.gpu


def cu(a):
    return torch.tensor(np.ascontiguousarray(a), device="cuda")


def _case(n, W_, H_, channels, mode, ts, seed):
    """n primitives over the whole W_ x H_ image, in depth order."""
    g = np.random.Generator(np.random.PCG64(seed))
    m2 = g.uniform((0, 0), (W_, H_), (1, n, 2)).astype(np.float32)
    s = g.uniform(6.0, 30.0, (n, 2))
    t = g.uniform(0, np.pi, n)
    R = np.stack([np.cos(t), -np.sin(t), np.sin(t), np.cos(t)], 1).reshape(n, 2, 2)
    ci = np.linalg.inv(R @ (s[:, :, None] ** 2 * np.eye(2)) @ R.transpose(0, 2, 1))
    cn = np.stack([ci[:, 0, 0], ci[:, 0, 1], ci[:, 1, 1]], 1)[None].astype(np.float32)
    op = g.uniform(0.02, 0.3, (1, n)).astype(np.float32)
    be = (4 * np.exp(g.normal(0, 0.5, (1, n)))).astype(np.float32)
    if mode == "mixed":  # some alphas clamped, some betas below one, some pixels ending early
        op[0, g.integers(0, n, max(1, n // 9))] = 0.9995
        be[0, g.integers(0, n, max(1, n // 7))] = 0.4
    col = g.uniform(0, 1, (1, n, channels)).astype(np.float32)
    tw, th = -(-W_ // ts), -(-H_ // ts)
    off = np.arange(tw * th, dtype=np.int32).reshape(1, th, tw) * n
    flat = np.tile(np.arange(n, dtype=np.int32), tw * th)
    return m2, cn, col, op, be, off, flat, g


@pytest.mark.parametrize("mode", ["plain", "mixed"])
@pytest.mark.parametrize("n,channels,ts", [(1, 3, 16), (15, 3, 16), (16, 3, 16), (17, 3, 16), (31, 1, 16), (32, 3, 8),
                                           (33, 4, 16), (48, 2, 16), (49, 3, 32), (65, 8, 16), (80, 16, 8),
                                           (97, 33, 16), (129, 3, 16)])
def test_blend_backward_group_edges(device, n, channels, ts, mode):
    W_, H_ = 41, 19  # ragged in both directions, outside pixels in every tile of the last row and column
    m2, cn, col, op, be, off, flat, g = _case(n, W_, H_, channels, mode, ts, 100 * n + channels)
    ins = [cu(a) for a in (m2, cn, col, op, be)]
    rc, ra, last, Tf = W.raster_fwd_raw(*ins, None, None, W_, H_, ts, cu(off), cu(flat))
    d = np.float64
    _, wa, wl, mT, mS = O.raster_fwd(*(a.astype(d) for a in (m2, cn, col, op, be)), W_, H_, ts, off, flat,
                                     margins=True)
    safe = (mT > 1e-3) & (mS > 1e-6)  # pixels whose branches FP32 and FP64 take alike
    vrc = (g.normal(0, 1, (1, H_, W_, channels)) * safe[..., None]).astype(np.float32)
    vra = (g.normal(0, 1, (1, H_, W_, 1)) * safe[..., None]).astype(np.float32)
    got = W.raster_bwd_raw(*ins, None, None, W_, H_, ts, cu(off), cu(flat), ra, last, Tf, cu(vrc), cu(vra))
    want = O.raster_bwd(*(a.astype(d) for a in (m2, cn, col, op, be)), W_, H_, ts, off, flat, wa, wl, vrc.astype(d),
                        vra.astype(d), T_final=1.0 - wa[..., 0])
    for a, b, name in zip(got, want, ("v_means2d", "v_conics", "v_colors", "v_opac", "v_betas")):
        assert rel_l2(a.cpu().numpy(), b) < 2e-3, (name, rel_l2(a.cpu().numpy(), b))


@pytest.mark.parametrize("channels,ts,ckpt", [(3, 16, False), (3, 16, True), (1, 8, False), (4, 32, True),
                                              (11, 16, False)])
def test_blend_backward_masks_kept_by_the_forward(device, channels, ts, ckpt):
    """The masks are conservative and the same test, so the gradients agree to
    the rounding of the atomics' order."""
    n, W_, H_ = 700, 75, 52
    g = np.random.Generator(np.random.PCG64(ts + channels))
    m2, cn, col, op, be, off, flat, g = _case(n, W_, H_, channels, "mixed", ts, ts + channels)
    cn = cn * 9.0  # radii of 2 to 10 pixels: most entries miss most sub-blocks
    ins = [cu(a) for a in (m2, cn, col, op, be)]
    fwd = W._raster_fwd(*ins, None, None, W_, H_, ts, cu(off), cu(flat), ckpt, keep_masks=True)
    rc, ra, last, Tf, T_ckpt, ws, masks = fwd
    assert masks is not None and (T_ckpt is not None) == ckpt
    ref = W.raster_fwd_raw(*ins, None, None, W_, H_, ts, cu(off), cu(flat))
    for a, b in zip((rc, ra, last, Tf), ref):
        assert torch.equal(a, b)
    vrc, vra = (cu(g.normal(0, 1, tuple(t.shape)).astype(np.float32)) for t in (rc, ra))
    args = (*ins, None, None, W_, H_, ts, cu(off), cu(flat), ra, last, Tf, vrc, vra)
    own = W.raster_bwd_raw(*args, T_ckpt=T_ckpt, fwd_workspace=ws)
    kept = W.raster_bwd_raw(*args, T_ckpt=T_ckpt, fwd_workspace=ws, entry_masks=masks)
    for a, b, name in zip(own, kept, ("v_means2d", "v_conics", "v_colors", "v_opac", "v_betas")):
        assert rel_l2(b.cpu().numpy(), a.cpu().numpy().astype(np.float64)) < 1e-6, name
