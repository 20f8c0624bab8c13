"""Blend of lists that end at the largest intersection index accepted, 2^31 - 2,
against the same lists at the front of their array.  Images are the same bits and
last ids the same places; gradients agree to the rounding of the atomics' order."""
import numpy as np
import pytest
import torch

from gsplat.cuda import _wrapper as W

from util import rel_l2

pytestmark = pytest.mark.gpu


def cu(a):
    return torch.tensor(np.ascontiguousarray(a), device="cuda")


@pytest.mark.parametrize("ckpt", [False, True])
def test_lists_at_the_largest_index(device, ckpt):
    W_, H_, ts, per, tiles = 32, 16, 16, 700, 2
    g = np.random.Generator(np.random.PCG64(8))
    m2 = g.uniform((0, 0), (W_, H_), (1, per, 2)).astype(np.float32)
    r = g.uniform(2.0, 9.0, (1, per))
    cn = np.stack([r ** -2, 0 * r, r ** -2], 2).astype(np.float32)
    op = g.uniform(0.02, 0.2, (1, per)).astype(np.float32)
    be = g.uniform(1, 6, (1, per)).astype(np.float32)
    col = g.uniform(0, 1, (1, per, 3)).astype(np.float32)
    ins = [cu(a) for a in (m2, cn, col, op, be)]
    flat = cu(np.tile(np.arange(per, dtype=np.int32), tiles))
    vrc = cu(g.normal(0, 1, (1, H_, W_, 3)).astype(np.float32))
    vra = cu(g.normal(0, 1, (1, H_, W_, 1)).astype(np.float32))

    def run(first, ids):
        off = cu(np.array([[[first, first + per]]], np.int32))
        rc, ra, last, Tf, T_ckpt, ws, masks = W._raster_fwd(*ins, None, None, W_, H_, ts, off, ids, ckpt,
                                                            keep_masks=True)
        args = (*ins, None, None, W_, H_, ts, off, ids, ra, last, Tf, vrc, vra)
        own = W.raster_bwd_raw(*args, T_ckpt=T_ckpt)
        kept = W.raster_bwd_raw(*args, T_ckpt=T_ckpt, fwd_workspace=ws, entry_masks=masks)
        return (rc, ra, Tf, last - first), own, kept

    n = 2 ** 31 - 1
    if torch.cuda.mem_get_info()[0] < 48 * 2 ** 30:
        pytest.skip("not enough free GPU memory for 2^31 list entries")
    want = run(0, flat)
    assert int(want[0][3].min()) > 0  # every pixel has a contributor (0 would also stand for none)
    ids = torch.empty((n,), dtype=torch.int32, device="cuda")
    ids[n - tiles * per:] = flat
    got = run(n - tiles * per, ids)
    for a, b in zip(got[0], want[0]):
        assert torch.equal(a, b)
    for gg, ww in zip(got[1:], want[1:]):
        for a, b, name in zip(gg, ww, ("v_means2d", "v_conics", "v_colors", "v_opac", "v_betas")):
            assert rel_l2(a.cpu().numpy(), b.cpu().numpy().astype(np.float64)) < 1e-6, name
