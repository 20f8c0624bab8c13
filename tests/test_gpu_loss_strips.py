"""Image loss by streaming strips at its edges: rows of W C values around one and
two column blocks of 256, heights around a chunk (11 rows) and a strip (12 output
rows of 2 chunks, 23 of 3, 78 of 8), one to four channels, images batched so
that longer strips are taken, and five channels (the tile kernels).

Tolerances, as in the other tests of this loss: relative 2e-5 (fp32 separable
window vs the fp64 2-D window); gradient relative L2 2e-4 (fp32 sums of 121
products per map)."""
import numpy as np
import pytest
import torch

from gsplat import loss as Lmod
from oracle import ubs_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [
    (1, 1, 1, 1), (1, 11, 85, 3), (1, 12, 86, 3), (2, 13, 256, 1), (1, 24, 257, 1), (1, 25, 64, 4), (1, 23, 129, 4),
    (1, 6, 171, 3), (2, 37, 128, 2), (200, 70, 9, 3), (710, 80, 2, 2), (1, 20, 30, 5)])
@pytest.mark.parametrize("lam", [0.2, 1.0])
def test_streamed_loss_matches_oracle(device, shape, lam):
    rng = np.random.Generator(np.random.PCG64(sum(shape)))
    x = rng.uniform(0, 1, shape).astype(np.float32)
    y = np.clip(x + rng.normal(0, 0.2, shape), 0, 1).astype(np.float32)
    want_loss, want_grad = O.image_loss(x.astype(np.float64), y.astype(np.float64), lam)
    tx = torch.tensor(x, device=device, requires_grad=True)
    got = Lmod.image_loss(tx, torch.tensor(y, device=device), lam)
    got.backward()
    assert abs(float(got) - want_loss) <= 2e-5 * abs(want_loss) + 1e-7, (float(got), want_loss)
    g = tx.grad.cpu().numpy()
    err = float(np.linalg.norm(g - want_grad) / max(np.linalg.norm(want_grad), 1e-30))
    assert err < 2e-4, err
