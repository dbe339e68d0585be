"""AdafacLO on tensors whose tables of first-layer terms pass 4 GB: the same tensor with its dims in another order takes the linear
pass, which addresses an element's entries by themselves, and has to come out the same."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _step(p, g):
    import pylo_amd
    from pylo_amd.models import MetaMLP

    torch.manual_seed(2)
    param = torch.nn.Parameter(p)
    opt = pylo_amd.AdafacLO_CUDA([param], lr=1.0, network=MetaMLP(39, 32, 1))
    param.grad = g
    opt.step()
    return param.detach()


def _compare(shape, order, scale):
    """One step on `shape` and on its permutation; gradients are N(0, 1) times `scale`, which broadcasts and varies over the
    entries that tables hold, so that another entry's terms would show.  Updates of the two passes (fp32 accuracy, 32 hidden
    units) differ by some 1e-6 of the largest; 1e-4 is far above that and far below the difference between entries."""
    torch.cuda.empty_cache()
    gen = torch.Generator(device="cuda").manual_seed(3)
    g = torch.randn(shape, generator=gen, device="cuda").mul_(scale)
    zero = torch.zeros(shape, device="cuda")
    a = _step(zero.clone(), g)
    b = _step(zero.permute(order).contiguous(), g.permute(order).contiguous())
    back = [order.index(i) for i in range(len(order))]
    top = float(a.abs().max())
    assert top > 0.0
    worst = float(b.permute(back).sub_(a).abs_().max())
    assert worst <= 1e-4 * top, (worst, top)


def test_row_terms_of_many_trailing_dims():
    """0.55 G elements, 64 rows of 69 MB of terms each (64 x 16 x 14^5)."""
    scale = torch.logspace(-5, 0, 64, device="cuda").view(64, 1, 1, 1, 1, 1, 1)
    _compare((64, 16, 14, 14, 14, 14, 14), [2, 3, 4, 5, 6, 0, 1], scale)
