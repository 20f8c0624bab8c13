"""Image loss of rows so wide that a value's byte offset in its row leaves 32
bits.  The widest rows accepted against a narrow image: all but the end of the row
is zero in both images, so the gradient there is the narrow image's, scaled by the
numbers of values.  Rows past it, whose tiles no launch holds, are refused.

Tolerance: gradient relative L2 2e-4, as in the other tests of this loss."""
import numpy as np
import pytest
import torch

from gsplat import loss as Lmod

pytestmark = pytest.mark.gpu


def _zeros(w, c):
    if torch.cuda.mem_get_info()[0] < 64 * 2 ** 30:
        pytest.skip("not enough free GPU memory for rows of 2^30 values")
    return torch.zeros((1, 1, w, c), device="cuda"), torch.zeros((1, 1, w, c), device="cuda")


@pytest.mark.parametrize("c", [1, 3])
def test_widest_rows(device, c):
    w, k = ((1 << 30) - 4097) // c, 300
    g = np.random.Generator(np.random.PCG64(c))
    a = torch.tensor(g.uniform(0, 1, (1, 1, k, c)).astype(np.float32), device="cuda")
    b = torch.tensor(g.uniform(0, 1, (1, 1, k, c)).astype(np.float32), device="cuda")
    grads = []
    for x, y in (_zeros(w, c), _zeros(1000, c)):
        x[:, :, -k:], y[:, :, -k:] = a, b
        x.requires_grad_(True)
        Lmod.image_loss(x, y, 0.2).backward()
        assert not x.grad[:, :, :-k - 10].any()
        grads.append(x.grad[:, :, -k - 10:].double() * x.numel())
        del x, y
    assert float((grads[0] - grads[1]).norm() / grads[1].norm()) < 2e-4


@pytest.mark.parametrize("w,c", [((1 << 30) + 4096, 1), ((1 << 29), 3)])
def test_wider_rows_are_refused(device, w, c):
    x, y = _zeros(w, c)
    with pytest.raises(RuntimeError, match="too large"):
        Lmod.image_loss(x, y, 0.2)
