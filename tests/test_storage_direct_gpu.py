"""2-D tensors of 16-bit storage that the passes of VeLO, ELO-CELO2 and AdafacLO read and write in place (no fp32 staging).

Checked against the float32 step of the same class on the widened values: accumulators to rel 1e-5 / abs 1e-6, the
parameter as that step's value rounded into the type, to one spacing (a float32 difference of an ulp can fall on the other
side of a rounding boundary).  Shapes: rows of one and of several 128-column tasks, one row, one more than a task's rows,
plans with nothing to stage, with staged neighbours and with float32 ones."""

import pytest
import torch

from golden_io import max_err
from test_storage_types_gpu import _spacing

pytestmark = pytest.mark.gpu

SETS = [
    [(1, 128)],
    [(33, 128), (257, 384), (5, 1024)],
    [(64, 256), (130, 36), (96,), (16, 128), (128, 3, 2)],
]


def _run(cls, params, grads, loss):
    from pylo_amd import ELO_CELO2_CUDA, AdafacLO_CUDA, VeLO_CUDA
    from pylo_amd.models import CELO2MLP, MetaMLP, VeLOMLP, VeLORNN

    torch.manual_seed(1)
    for p, g in zip(params, grads):
        p.grad = g
    if cls == "VeLO":
        opt = VeLO_CUDA(params, lr=1.0, num_steps=100, weight_decay=0.01, rnn=VeLORNN(), mlp=VeLOMLP())
        opt.step(loss)
    elif cls.startswith("AdafacLO"):
        opt = AdafacLO_CUDA(params, lr=1.0, weight_decay=0.01, max_grad_norm=0.5 if "clipped" in cls else None,
                            network=MetaMLP(39, 32, 1))
        opt.step()
    else:
        opt = ELO_CELO2_CUDA(params, lr=1e-2, weight_decay=0.01, clip_grad=cls == "ELO_CELO2 clipped", clip_norm=1.0,
                             network=CELO2MLP(), hf_key=None)
        opt.step()
    return opt


@pytest.mark.parametrize("cls", ["VeLO", "ELO_CELO2", "ELO_CELO2 clipped", "AdafacLO", "AdafacLO clipped"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shapes", SETS)
@pytest.mark.parametrize("mixed", [False, True])
def test_step_in_place_matches_float32(shapes, dtype, mixed, cls):
    gen = torch.Generator().manual_seed(3)
    dts = [torch.float32 if mixed and i == len(shapes) - 1 and i > 0 else dtype for i in range(len(shapes))]
    init = [(torch.randn(s, generator=gen) * 0.3).to(dt) for s, dt in zip(shapes, dts)]
    grads = [(torch.randn(s, generator=gen) * 0.1).to(dt) for s, dt in zip(shapes, dts)]
    p16 = [torch.nn.Parameter(v.clone().cuda()) for v in init]
    p32 = [torch.nn.Parameter(v.float().cuda()) for v in init]
    loss = torch.tensor(2.0, device="cuda")
    o16 = _run(cls, p16, [g.cuda() for g in grads], loss)
    o32 = _run(cls, p32, [g.float().cuda() for g in grads], loss)
    torch.cuda.synchronize()
    for a, b, s, dt in zip(p16, p32, shapes, dts):
        for k in (k for k, v in o32.state[b].items() if torch.is_tensor(v) and v.is_cuda and k != "rank_onehot"):
            assert max_err(o16.state[a][k], o32.state[b][k].cpu(), 1e-5, 1e-6) <= 1.0, (s, k)
        got, want = a.detach().cpu(), b.detach().cpu()
        if dt == torch.float32:
            assert max_err(got, want, 1e-5, 1e-6) <= 1.0, s
        else:
            assert float(((got.double() - want.to(dt).double()).abs() / _spacing(want, dt)).max()) <= 1.0, s
            assert not torch.equal(got, init[[id(x) for x in p16].index(id(a))]), s
