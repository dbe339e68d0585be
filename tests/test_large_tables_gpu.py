"""Tensors whose tables of first-layer terms pass 4 GB, where a byte offset into them does not fit 32 bits: entries beyond that
bound are given the gradients of entries below it, and their elements have to come out the same, bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _step(name, shape, copy):
    """One step on gradients that differ from entry to entry, `copy` applied to them; parameters start at zero."""
    import pylo_amd
    from pylo_amd.models import CELO2MLP, MetaMLP

    torch.cuda.empty_cache()
    torch.manual_seed(2)
    param = torch.nn.Parameter(torch.zeros(shape, device="cuda"))
    if name == "AdafacLO":
        opt = pylo_amd.AdafacLO_CUDA([param], lr=1.0, network=MetaMLP(39, 32, 1))
    else:
        opt = pylo_amd.ELO_CELO2_CUDA([param], lr=1.0, network=CELO2MLP(), hf_key=None, orthogonalize=False)
    gen = torch.Generator(device="cuda").manual_seed(3)
    param.grad = torch.randn(shape, generator=gen, device="cuda")
    copy(param.grad)
    opt.step()
    return param.detach()


def test_row_terms_of_many_trailing_dims():
    """0.55 G elements, 64 rows of 69 MB of terms each."""
    def copy(g):
        g[63].copy_(g[31])

    p = _step("AdafacLO", (64, 16, 14, 14, 14, 14, 14), copy)
    assert float(p[63].abs().max()) > 0.0 and torch.equal(p[63], p[31])


# 128 and 32 bytes of terms an entry; as columns (walked a row at a time) and as rows (elements in storage order)
@pytest.mark.parametrize("name,entries,low", [("AdafacLO", 40_000_000, 2 ** 25), ("ELO_CELO2", 150_000_000, 2 ** 27)])
@pytest.mark.parametrize("columns", [True, False])
def test_terms_of_many_entries(name, entries, low, columns):
    over = entries - low

    def cut(x, first):
        return x[:, first:first + over] if columns else x[first:first + over]

    p = _step(name, (2, entries) if columns else (entries, 2), lambda g: cut(g, low).copy_(cut(g, low // 2)))
    assert float(cut(p, low).abs().max()) > 0.0 and torch.equal(cut(p, low), cut(p, low // 2))
