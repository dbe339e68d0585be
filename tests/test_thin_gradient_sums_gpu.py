"""Sums of g^2 of matrices with few rows or few columns (``p0_wide``, ``p0_tall``), at the edges of their tiles and of the rule
that picks them, and ``k_v0a`` with a thread an entry (plans of more than 4096 blocks of 64 entries): whole steps against the
oracle, with gradients beyond the clamp (the exact pass) and rows of zeros among them.
"""

import copy

import pytest
import torch

from golden_io import max_err

pytestmark = pytest.mark.gpu

REL, ABS = 1e-5, 1e-6
EDGES = [(1, 65), (1, 257), (16, 260), (16, 1025), (17, 300), (2, 4100), (129, 1), (128, 16), (1025, 16), (1030, 17), (2050, 7), (1, 1)]
MANY = [(3, 65536), (2, 65540), (65600, 2), (4, 65537), (66000, 1), (5, 777)]


def _grads(shapes, gen, scale):
    out = [torch.randn(s, generator=gen, device="cuda") * scale for s in shapes]
    out[0].view(-1)[-1] = 40.0
    out[3][0].zero_()
    return out


@pytest.mark.parametrize("shapes", [EDGES, MANY], ids=["edges", "many"])
@pytest.mark.parametrize("clip", [dict(clip_grad=False), dict(clip_grad=True, grad_clip_val=0.5, clip_norm=1e9), dict(clip_grad=True)],
                         ids=["plain", "exact", "norm"])
def test_elo_celo2(shapes, clip):
    from oracle import pylo_oracle as O
    from pylo_amd import ELO_CELO2_CUDA
    from pylo_amd.models import CELO2MLP

    torch.manual_seed(5)
    net = CELO2MLP()
    cfg = dict(lr=1e-3, orthogonalize=False, **clip)
    gen = torch.Generator(device="cuda").manual_seed(6)
    init = [torch.randn(s, generator=gen, device="cuda") * 0.05 for s in shapes]
    ref = [v.double() for v in init]
    gpu = [torch.nn.Parameter(v.clone()) for v in init]
    orc = O.EloCelo2Oracle(ref, net.state_dict(), device="cuda", **cfg).double_()
    opt = ELO_CELO2_CUDA(gpu, network=net, hf_key=None, **cfg)
    for t in range(3):
        grads = _grads(shapes, gen, 0.3)
        for p, g in zip(gpu, grads):
            p.grad = g.clone()
        orc.step([g.double() for g in grads])
        opt.step()
        for i, (p, r) in enumerate(zip(gpu, ref)):
            assert max_err(p, r, REL, ABS) <= 1.0, (t, shapes[i])


@pytest.mark.parametrize("shapes", [EDGES, MANY], ids=["edges", "many"])
def test_velo(shapes):
    from oracle import pylo_oracle as O
    from pylo_amd import VeLO_CUDA
    from pylo_amd.models import VeLOMLP, VeLORNN

    torch.manual_seed(3)
    rnn, mlp = VeLORNN(lstm_hidden_size=64, param_inits=64), VeLOMLP(param_inits=64)
    gen = torch.Generator(device="cuda").manual_seed(7)
    init = [torch.randn(s, generator=gen, device="cuda") * 0.3 for s in shapes]
    cpu = [v.cpu() for v in init]
    gpu = [torch.nn.Parameter(v.clone()) for v in init]
    kw = dict(lr=1e-2, num_steps=50)
    orc = O.VeloOracle(cpu, rnn.state_dict(), mlp.state_dict(), **kw)
    opt = VeLO_CUDA(gpu, rnn=copy.deepcopy(rnn), mlp=copy.deepcopy(mlp), **kw)
    for t in range(3):
        grads = _grads(shapes, gen, 0.3)
        for p, g in zip(gpu, grads):
            p.grad = g.clone()
        orc.step([g.cpu() for g in grads], torch.tensor(1.5 - 0.2 * t))
        opt.step(torch.tensor(1.5 - 0.2 * t, device="cuda"))
        for i, p in enumerate(gpu):
            assert max_err(p, cpu[i], REL, ABS) <= 1.0, (t, shapes[i])
