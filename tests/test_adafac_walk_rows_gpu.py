"""The number of rows that a wave of the AdafacLO walks takes follows from the size of the plan and changes no result."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# one row, one past and one short of 16, 32 and 64 rows, several tasks, convolution kernels, other factored dims
SHAPES = [(1, 64), (17, 128), (33, 64), (63, 192), (64, 64), (65, 128), (129, 320), (130, 64, 3, 3), (31, 64, 1, 1), (66, 7, 64)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name", ["AdafacLO_CUDA", "ELO_CUDA"])
@pytest.mark.parametrize("filler", [34_000_000, 70_000_001])     # 32 and 64 rows; 16 with 3 M elements
def test_rows_of_a_wave(name, filler, dtype):
    import pylo_amd
    from pylo_amd.models import MetaMLP

    def run(extra):
        torch.manual_seed(2)
        kw = dict(network=MetaMLP(39, 32, 1), **({"hf_key": None} if name == "ELO_CUDA" else {}))
        gen = torch.Generator().manual_seed(7)
        params = [torch.nn.Parameter((0.05 * torch.randn(s, generator=gen)).to(dtype).cuda()) for s in SHAPES]
        params.append(torch.nn.Parameter(torch.zeros(extra, dtype=dtype, device="cuda")))
        opt = getattr(pylo_amd, name)(params, **kw)
        for _ in range(2):
            for p, s in zip(params, SHAPES):
                p.grad = (1e-2 * torch.randn(s, generator=gen)).to(dtype).cuda()
            params[-1].grad = torch.zeros_like(params[-1])
            opt.step()
        return params[:-1], [opt.state[p] for p in params[:-1]]

    a, sa = run(3_000_000)
    b, sb = run(filler)
    for p, q, s, t in zip(a, b, sa, sb):
        assert torch.equal(p, q), p.shape
        for key in ("exp_avg", "exp_avg_sq", "exp_avg_sq_r", "exp_avg_sq_c"):
            assert torch.equal(s[key], t[key]), (p.shape, key)
