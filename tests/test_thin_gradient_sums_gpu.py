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
FAC = 2e-6      # accumulators after three steps: at most eleven roundings of 2^-24 each
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
            for key in ("fac_r", "fac_c"):
                assert max_err(opt.state[p][key], orc.state[i][key], FAC, 1e-30) <= 1.0, (t, shapes[i], key)


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
            for key in ("fac_vec_row", "fac_vec_col"):
                assert max_err(opt.state[p][key], orc.state[i][key], REL, 1e-30) <= 1.0, (t, shapes[i], key)


@pytest.mark.parametrize("clip", [True, False])
def test_elo_with_nan_and_infinity(clip):
    """NaNs become zeros before they are squared (the exact pass, which they ask for); with clipping a NaN makes the global norm one and
    the scale 1, an infinity makes the scale 0."""
    from oracle import pylo_oracle as O
    from pylo_amd import ELO_CUDA
    from pylo_amd.models import MetaMLP

    torch.manual_seed(9)
    net = MetaMLP(39, 32, 1)
    gen = torch.Generator().manual_seed(30)
    cpu = [torch.randn(s, generator=gen) * 0.3 for s in EDGES]
    gpu = [torch.nn.Parameter(v.clone().cuda()) for v in cpu]
    cfg = dict(lr=1e-2, clip_grad=clip, clip_norm=3.0)
    orc = O.EloOracle(cpu, net.state_dict(), **cfg)
    opt = ELO_CUDA(gpu, network=copy.deepcopy(net), hf_key=None, **cfg)
    for t in range(4):
        grads = [torch.randn(s, generator=gen) for s in EDGES]
        if t == 1:
            for g in grads[:-1]:
                g.view(-1)[[0, g.numel() // 2, g.numel() - 1]] = float("nan")
        if t == 2 and clip:
            grads[1].view(-1)[256] = float("inf")
            grads[8][1024, 15] = -float("inf")
        for p, g in zip(gpu, grads):
            p.grad = g.cuda()
        orc.step(grads)
        opt.step()
        for i, p in enumerate(gpu):
            st, so = opt.state[p], orc.state[i]
            assert max_err(p, cpu[i], REL, ABS) <= 1.0, (t, EDGES[i])
            for key, was in (("exp_avg_sq_r", "exp_avg_sq_r"), ("exp_avg_sq_c", "exp_avg_sq_c")):
                assert bool(torch.isfinite(so[was]).all())
                assert max_err(st[key], so[was], REL, 1e-30) <= 1.0, (t, EDGES[i], key)


def _own(m):
    """Sizes of the partial sums that a thread adds m <= 16 squares up in: fours in pairs, then the fours in pairs."""
    fours = [min(4, m - i) for i in range(0, m, 4)]
    sizes = [k for f in fours for k in ([2] * (f > 1) + [2] * (f > 3) + [f] * (f > 2))]
    return sizes + [sum(fours[i:i + 2]) for i in (0, 2) if len(fours) > i + 1] + [m] * (len(fours) > 2)


def _bound(n, sizes):
    """RMS of the relative error, in 2^-24, of a mean of n squares of normal numbers that is then multiplied by a weight: a rounding
    has an RMS of 0.425 (values spread over their logarithm), two of them on the result, one on each square (fourth moment 3), one
    on each partial sum of k squares, whose share of the whole has the second moment (k / n)^2 (1 + 2 / k) / (1 + 2 / n)."""
    return 0.425 * (2 + 3 / n + sum((k / n) ** 2 * (1 + 2 / k) / (1 + 2 / n) for k in sizes)) ** 0.5


@pytest.mark.parametrize("m,n", [(16, 1024), (16, 4096), (7, 333), (13, 5001), (3, 1030)])
@pytest.mark.parametrize("tall", [False, True])
def test_means_of_squares(tall, m, n):
    """fac_r and fac_c after one step from zero, (1 - decay) times the means of g^2, against fp64: no more roundings than sums in
    pairs have.  Sums over the long side are fp32 up to 64 squares and double from there on."""
    from pylo_amd import ELO_CELO2_CUDA
    from pylo_amd.models import CELO2MLP

    torch.manual_seed(0)
    gen = torch.Generator(device="cuda").manual_seed(m * n)
    params = [torch.nn.Parameter(torch.randn((n, m) if tall else (m, n), generator=gen, device="cuda")) for _ in range(120)]
    for p in params:
        p.grad = torch.randn(p.shape, generator=gen, device="cuda") * 2.0 ** torch.rand(1, generator=gen, device="cuda")
    opt = ELO_CELO2_CUDA(params, network=CELO2MLP(), hf_key=None, clip_grad=False, orthogonalize=False)
    opt.step()
    err = {0: [], 1: []}
    for p in params:
        for key in ("fac_r", "fac_c"):
            fac = opt.state[p][key].double()
            dim = 1 if fac.shape[1] == 1 else 2              # summed over
            want = (p.grad.double() ** 2).mean(dim - 1, keepdim=True) * (1 - opt.beta_fac.float()).double().view(3, 1, 1)
            rel = (fac - want) / want
            assert float(rel.abs().max()) <= 8 * 2.0 ** -24
            err[int((dim == 1) == tall)].append(float(rel.pow(2).mean()))
    long_sizes = [k for k in (2, 4, 8, 16, 32, 64) for _ in range(n // k)]
    for over_long, bound in ((1, _bound(n, long_sizes)), (0, _bound(m, _own(m)))):
        e = err[over_long]
        got = (sum(e) / len(e)) ** 0.5 * 2 ** 24
        print(over_long, got, bound)
        assert got <= 1.1 * bound, (over_long, got, bound)      # a tenth: from 360 sums (m = 3) on
