"""AdafacLO's apply pass in storage order (tensors that no column-resident walk takes) with the element MLP on the
matrix pipe: one step at the edges of its groups of 64 elements, blocks of 256 and trips, against the oracle in fp64.

The bound: its operands' three bfloat16 planes are the fp32 numbers, so an error is that of an fp32 sum in another order,
no larger than one and a half times the largest that the fp32 oracle and the all-VALU kernel show on the same tensor
(each the largest of up to some hundred thousand), or than half a spacing of the result where these have almost none."""

import copy

import pytest
import torch

pytestmark = pytest.mark.gpu

SETS = {
    "vectors": [(1,), (63,), (64,), (65,), (255,), (257,), (1000,)],
    "matrices": [(1, 1), (1, 3), (65, 1), (3, 65), (5, 127), (33, 130), (130, 33)],
    "n-d": [(3, 5, 7), (2, 3, 4, 5), (6, 4, 3, 3), (5, 1, 9, 2)],
    "several trips": [(517, 1031), (300007,), (9, 70, 501)],
}


@pytest.mark.parametrize("which", list(SETS))
def test_adafac_linear_apply_against_fp64(which, monkeypatch):
    from oracle import pylo_oracle as O
    from pylo_amd import AdafacLO_CUDA
    from pylo_amd.models import MetaMLP

    torch.manual_seed(5)
    net = MetaMLP(39, 32, 1)
    shapes = SETS[which]
    gen = torch.Generator().manual_seed(12)
    init = [torch.randn(s, generator=gen) * 0.01 for s in shapes]    # small against the step
    grads = [torch.randn(s, generator=gen) * (10.0 ** (-(i % 4))) for i, s in enumerate(shapes)]
    ref64 = [v.double().cuda() for v in init]
    ref32 = [v.clone().cuda() for v in init]
    kw = dict(lr=1.0, step_mult=1.0, exp_mult=0.1)
    O.AdafacOracle(ref64, net.state_dict(), device="cuda", **kw).double_().step([g.double().cuda() for g in grads])
    O.AdafacOracle(ref32, net.state_dict(), device="cuda", **kw).step([g.cuda() for g in grads])
    outs = {}
    for name in ("0", "1"):
        monkeypatch.setenv("PYLO_MI355_VALU_MLP", name)
        gpu = [torch.nn.Parameter(v.clone().cuda()) for v in init]
        opt = AdafacLO_CUDA(gpu, network=copy.deepcopy(net), **kw)
        for p, g in zip(gpu, grads):
            p.grad = g.cuda()
        opt.step()
        torch.cuda.synchronize()
        outs[name] = [p.detach().double() for p in gpu]
    for i, s in enumerate(shapes):
        own = float((ref32[i].double() - ref64[i]).abs().max())
        valu = float((outs["1"][i] - ref64[i]).abs().max())
        err = float((outs["0"][i] - ref64[i]).abs().max())
        size = float((ref64[i] - init[i].double().cuda()).abs().max())
        print(s, "largest step", size, "fp32 oracle", own, "vector pipe", valu, "matrix pipe", err)
        assert err <= max(1.5 * max(own, valu), 2.0 ** -25 * size), (s, err, own, valu)
