"""The element passes of small plans are cut into smaller blocks (fewer rows a wave task, fewer trips a chunk): three
steps of every family at each of the five cuts, against the oracle in fp64, at the suite's bar (rel 1e-5 / abs 1e-6)."""

import copy

import pytest
import torch

from golden_io import max_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [100, 900, 2000, 3501, 6001])     # 16, 8, 4, 2 parts and whole blocks
@pytest.mark.parametrize("family", ["elo_celo2", "velo", "adafac"])
def test_every_cut_against_the_oracle(family, rows):
    _three_steps(family, [(rows, 256), (rows, 130), (1000,), (33, 128)], rows)


# The same with tensors of more than two dims: convolution kernels walked as matrices or by slices, channels last to first.
@pytest.mark.parametrize("rows", [10, 100, 400, 900])     # 16, 8, 2 parts and whole blocks
@pytest.mark.parametrize("family", ["elo_celo2", "velo", "adafac"])
def test_every_cut_with_more_than_two_dims(family, rows):
    _three_steps(family, [(rows, 64, 3, 3), (3, 5, rows, 7), (rows, 128, 9), (1, 1, 64), (rows,)], rows)


def _three_steps(family, shapes, rows):
    from oracle import pylo_oracle as O
    from pylo_amd import ELO_CELO2_CUDA, AdafacLO_CUDA, VeLO_CUDA
    from pylo_amd.models import CELO2MLP, MetaMLP, VeLOMLP, VeLORNN

    torch.manual_seed(rows)
    gen = torch.Generator(device="cuda").manual_seed(rows)
    init = [torch.randn(s, generator=gen, device="cuda") * 0.05 for s in shapes]
    ref = [v.double() for v in init]
    gpu = [torch.nn.Parameter(v.clone()) for v in init]
    if family == "elo_celo2":
        net = CELO2MLP()
        kw = dict(lr=1e-3, orthogonalize=False, adam_lr_mult=20.0)
        orc = O.EloCelo2Oracle(ref, net.state_dict(), device="cuda", **kw).double_()
        opt = ELO_CELO2_CUDA(gpu, network=net, hf_key=None, **kw)
    elif family == "velo":
        rnn, mlp = VeLORNN(lstm_hidden_size=64, param_inits=32), VeLOMLP(param_inits=32)
        kw = dict(lr=1e-2, num_steps=100)
        orc = O.VeloOracle(ref, rnn.state_dict(), mlp.state_dict(), device="cuda", **kw).double_()
        opt = VeLO_CUDA(gpu, rnn=copy.deepcopy(rnn), mlp=copy.deepcopy(mlp), **kw)
    else:
        net = MetaMLP(39, 32, 1)
        kw = dict(lr=1.0)
        orc = O.AdafacOracle(ref, net.state_dict(), device="cuda", **kw).double_()
        opt = AdafacLO_CUDA(gpu, network=copy.deepcopy(net), **kw)
    for t in range(3):
        grads = [torch.randn(s, generator=gen, device="cuda") * 10.0 ** -i for i, s in enumerate(shapes)]
        for p, g in zip(gpu, grads):
            p.grad = g
        args = (torch.tensor(2.0 - 0.3 * t, device="cuda"),) if family == "velo" else ()
        orc.step([g.double() for g in grads], *[a.double() for a in args])
        opt.step(*args)
        for i, p in enumerate(gpu):
            assert max_err(p, ref[i], 1e-5, 1e-6) <= 1.0, (family, rows, t, i)
