"""Projection backward on needles: 2-D ellipses about a hundred pixels long and
half a pixel wide, with conic gradients as the blend gives them (moments of the
pixels along the needle).  What the covariance gradient takes from such a gradient
is its part across the needle, a 10^-4 of its entries: taken in FP32 that part
carries rounding of 10^-3, and the last bit of a conic gradient moves it as much.

Tolerance: with the conic's own gradient exact, what is left is the FP32 products
with the Jacobian and the rotation, four sums of two or three terms an entry, each
within 4 roundings of terms that are at most ten times the result: 10 x 16 x
2^-24 = 1e-5 relative to the primitive's gradient."""
import numpy as np
import pytest
import torch

from gsplat.cuda import _wrapper as W
from oracle import ubs_oracle as O

pytestmark = pytest.mark.gpu


def cu(a):
    return torch.tensor(np.ascontiguousarray(a), device="cuda")


@pytest.mark.parametrize("layout", ["triu6", "full33"])
def test_conic_gradient_across_needles(device, layout):
    N, W_, H_, f = 600, 640, 480, 500.0
    g = np.random.Generator(np.random.PCG64(4))
    z = g.uniform(3.0, 5.0, N)
    means = np.stack([g.uniform(-0.5, 0.5, N) * z, g.uniform(-0.4, 0.4, N) * z, z], 1).astype(np.float32)
    t = g.uniform(0, np.pi, N)
    u = np.stack([np.cos(t), np.sin(t), np.zeros(N)], 1)
    s1 = g.uniform(0.3, 0.9, N)  # 40 to 140 pixels along, the blur's half pixel across
    cov = (s1[:, None, None] ** 2 * u[:, :, None] * u[:, None, :] + 1e-8 * np.eye(3)).astype(np.float32)
    iu = np.triu_indices(3)
    cov6 = np.ascontiguousarray(cov[:, iu[0], iu[1]])
    vm = np.eye(4, dtype=np.float32)[None]
    K = np.array([[[f, 0, W_ / 2], [0, f, H_ / 2], [0, 0, 1]]], np.float32)
    fwd = cu(cov6 if layout == "triu6" else cov)
    lay = 0 if layout == "triu6" else 1
    radii, _, depths, conics, _ = W.projection_fwd_raw(cu(means), fwd, None, None, cu(vm), cu(K), W_, H_, 0.3, 0.01,
                                                       1e10, 0.0, False, False, lay)
    cn = conics.cpu().numpy().astype(np.float64)
    assert (radii > 0).all()
    # the blend's conic gradient: sum of s d d^T over pixels on the needle
    P = np.stack([cn[0, :, 0], cn[0, :, 1], cn[0, :, 1], cn[0, :, 2]], 1).reshape(N, 2, 2)
    lam, E = np.linalg.eigh(P)
    along, across = E[:, :, 0], E[:, :, 1]
    n = 200
    d = (g.uniform(-0.9, 0.9, (N, n, 1)) * (along * lam[:, :1] ** -0.5)[:, None]
         + g.uniform(-0.9, 0.9, (N, n, 1)) * (across * lam[:, 1:] ** -0.5)[:, None])
    M = np.einsum("np,npi,npj->nij", g.normal(0.2, 1, (N, n)), d, d)
    vcn = np.stack([M[:, 0, 0], 2 * M[:, 0, 1], M[:, 1, 1]], 1)[None].astype(np.float32)
    zero2, zero1 = np.zeros((1, N, 2), np.float32), np.zeros((1, N), np.float32)
    got = W.projection_bwd_raw(cu(means), fwd, None, None, cu(vm), cu(K), W_, H_, 0.3, False, radii, conics, None,
                               cu(zero2), cu(zero1), cu(vcn), None, False, lay)[1].cpu().numpy().astype(np.float64)
    w = np.float64
    want = O.proj_bwd(means.astype(w), cov6.astype(w), None, None, vm.astype(w), K.astype(w), W_, H_, 0.3,
                      radii.cpu().numpy(), cn, None, zero2.astype(w), zero1.astype(w), vcn.astype(w))[1]
    if layout == "full33":
        assert not got[:, [1, 2, 2], [0, 0, 1]].any()
        got = got[:, iu[0], iu[1]]
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() < 1e-5, (err.max(), np.median(err))
