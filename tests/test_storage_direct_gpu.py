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
    from pylo_amd import ELO_CELO2_CUDA, ELO_CUDA, AdafacLO_CUDA, VeLO_CUDA
    from pylo_amd.models import CELO2MLP, MetaMLP, VeLOMLP, VeLORNN

    torch.manual_seed(1)
    for p, g in zip(params, grads):
        p.grad = g
    if cls == "VeLO":
        opt = VeLO_CUDA(params, lr=1.0, num_steps=100, weight_decay=0.01, rnn=VeLORNN(), mlp=VeLOMLP())
        opt.step(loss)
    elif cls.startswith("ELO ") or cls == "ELO":
        opt = ELO_CUDA(params, lr=1e-2, weight_decay=0.01, clip_grad="clipped" in cls, clip_norm=0.5, network=MetaMLP(39, 32, 1),
                       hf_key=None)
        opt.step()
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
    _compare(o16, o32, p16, p32, init)


def _compare(o16, o32, p16, p32, init):
    for a, b, v in zip(p16, p32, init):
        s, dt = tuple(v.shape), v.dtype
        for k in (k for k, v in o32.state[b].items() if torch.is_tensor(v) and v.is_cuda and k != "rank_onehot"):
            assert max_err(o16.state[a][k], o32.state[b][k].cpu(), 1e-5, 1e-6) <= 1.0, (s, k)
        got, want = a.detach().cpu(), b.detach().cpu()
        if dt == torch.float32:
            assert max_err(got, want, 1e-5, 1e-6) <= 1.0, s
        else:
            assert float(((got.double() - want.to(dt).double()).abs() / _spacing(want, dt)).max()) <= 1.0, s
            assert not torch.equal(got, v), s


# Plans above 2.1 M elements, whose passes are not cut finer (instantiations of their own): tasks of sixteen rows, a last
# one of fewer, a staged neighbour, and a tensor too large to be kept in the cache between its statistics and its apply.
@pytest.mark.parametrize("cls", ["VeLO", "ELO_CELO2", "ELO_CELO2 clipped", "AdafacLO", "ELO clipped"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shapes", [[(4099, 768), (130, 36)], [(12801, 640), (256, 128)]])
def test_plans_that_are_not_cut(shapes, dtype, cls):
    gen = torch.Generator(device="cuda").manual_seed(4)
    init = [(torch.randn(s, generator=gen, device="cuda") * 0.3).to(dtype) for s in shapes]
    grads = [(torch.randn(s, generator=gen, device="cuda") * 0.1).to(dtype) for s in shapes]
    p16 = [torch.nn.Parameter(v.clone()) for v in init]
    p32 = [torch.nn.Parameter(v.float()) for v in init]
    loss = torch.tensor(2.0, device="cuda")
    o16 = _run(cls, p16, grads, loss)
    o32 = _run(cls, p32, [g.float() for g in grads], loss)
    torch.cuda.synchronize()
    _compare(o16, o32, p16, p32, [v.cpu() for v in init])


# ELO replaces NaN and infinite gradients after clipping (torch.nan_to_num): elements that are only known after the norm
# is, and that send the gradient sums through their second pass.
@pytest.mark.parametrize("cls", ["ELO", "ELO clipped"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("odd", [float("nan"), float("inf"), 0.0])
def test_elo_in_place_with_gradients_that_are_replaced(dtype, cls, odd):
    gen = torch.Generator(device="cuda").manual_seed(5)
    shapes = [(33, 128), (257, 384), (130, 36)]
    init = [(torch.randn(s, generator=gen, device="cuda") * 0.3).to(dtype) for s in shapes]
    grads = [(torch.randn(s, generator=gen, device="cuda") * 0.1).to(dtype) for s in shapes]
    if odd != 0.0:
        grads[1][200, 17] = odd
    p16 = [torch.nn.Parameter(v.clone()) for v in init]
    p32 = [torch.nn.Parameter(v.float()) for v in init]
    o16 = _run(cls, p16, grads, None)
    o32 = _run(cls, p32, [g.float() for g in grads], None)
    torch.cuda.synchronize()
    for a, b in zip(p16, p32):
        for k in (k for k, v in o32.state[b].items() if torch.is_tensor(v) and v.is_cuda):
            x, y = o16.state[a][k], o32.state[b][k].cpu()
            assert torch.equal(x.isfinite().cpu(), y.isfinite())
            assert max_err(x.nan_to_num(0.0, 0.0, 0.0), y.nan_to_num(0.0, 0.0, 0.0), 1e-5, 1e-6) <= 1.0, k
        got, want = a.detach().cpu(), b.detach().cpu().to(dtype)
        assert torch.equal(got.isfinite(), want.isfinite())
        fin = got.isfinite()
        assert float(((got[fin].double() - want[fin].double()).abs() / _spacing(want[fin].float(), dtype)).max()) <= 1.0
