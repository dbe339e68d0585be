"""The state of parameters that are stored in 16 or 64 bits: long enough that a buffer of the wrong type would be left."""

import copy

import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16, torch.float64]


@pytest.mark.parametrize("dtype", DTYPES)
def test_celo2_moments_of_stored_vectors(dtype):
    """Moments and updated parameters of AdamW tensors against a float32 run on the widened values: the arithmetic is the same,
    so the moments agree bit for bit and the parameters up to the rounding into the storage type."""
    from pylo_amd import CELO2_CUDA
    from pylo_amd.models import CELO2MLP

    gen = torch.Generator().manual_seed(5)
    shapes = [(70001,), (4096,), (301, 64)]
    init = [(0.05 * torch.randn(s, generator=gen)).to(dtype).cuda() for s in shapes]
    torch.manual_seed(1)
    net = CELO2MLP()
    stored = [torch.nn.Parameter(v.clone()) for v in init]
    wide = [torch.nn.Parameter(v.float()) for v in init]
    a, b = ([{"params": ps[:2]}, {"params": ps[2:], "is_embedding": True}] for ps in (stored, wide))
    oa, ob = CELO2_CUDA(a, lr=1e-3, network=net, hf_key=None), CELO2_CUDA(b, lr=1e-3, network=copy.deepcopy(net), hf_key=None)
    for t in range(3):
        for p, q, s in zip(stored, wide, shapes):
            p.grad = (1e-2 * torch.randn(s, generator=gen)).to(dtype).cuda()
            q.grad = p.grad.float()
            q.data.copy_(p.data)
        oa.step()
        ob.step()
        for p, q in zip(stored, wide):
            for key in ("exp_avg", "exp_avg_sq"):
                assert oa.state[p][key].dtype == torch.float32
                assert torch.equal(oa.state[p][key], ob.state[q][key]), (t, key)
            assert torch.equal(p.data, q.data.to(dtype)), t


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float64])
@pytest.mark.parametrize("name", ["ELO_CELO2_CUDA", "CELO2_CUDA", "VeLO_CUDA", "AdafacLO_CUDA", "ELO_CUDA"])
def test_checkpoint_of_stored_parameters(name, dtype):
    """A run continued from a state dict is the run itself, bit for bit, and its accumulators stay float32."""
    import pylo_amd
    from pylo_amd.models import CELO2MLP, MetaMLP, VeLOMLP, VeLORNN

    def make(init):
        torch.manual_seed(1)
        params = [torch.nn.Parameter(v.clone()) for v in init]
        kw = {"VeLO_CUDA": lambda: dict(lr=1.0, num_steps=100, rnn=VeLORNN(), mlp=VeLOMLP()),
              "AdafacLO_CUDA": lambda: dict(lr=1.0, network=MetaMLP(39, 32, 1)),
              "ELO_CUDA": lambda: dict(lr=1e-3, network=MetaMLP(39, 32, 1), hf_key=None)}.get(
                  name, lambda: dict(lr=1e-3, network=CELO2MLP(), hf_key=None))()
        return params, getattr(pylo_amd, name)(params, **kw)

    gen = torch.Generator().manual_seed(6)
    shapes = [(301, 256), (20001,), (40, 12, 3, 3)]
    init = [(0.05 * torch.randn(s, generator=gen)).to(dtype).cuda() for s in shapes]
    args = (torch.tensor(2.0, device="cuda"),) if name == "VeLO_CUDA" else ()

    def run(params, opt, seed):
        g = torch.Generator().manual_seed(seed)
        for p, s in zip(params, shapes):
            p.grad = (1e-2 * torch.randn(s, generator=g)).to(dtype).cuda()
        opt.step(*args)

    a, oa = make(init)
    run(a, oa, 1)
    run(a, oa, 2)
    saved, at = copy.deepcopy(oa.state_dict()), [p.detach().clone() for p in a]
    run(a, oa, 3)
    b, ob = make(at)
    ob.load_state_dict(saved)
    for p in b:
        for key, t in ob.state[p].items():
            assert key == "step" or not torch.is_tensor(t) or t.dtype == torch.float32, key
    run(b, ob, 3)
    for p, q in zip(a, b):
        assert torch.equal(p, q)
        for key, t in oa.state[p].items():
            assert not torch.is_tensor(t) or torch.equal(t, ob.state[q][key]), key
