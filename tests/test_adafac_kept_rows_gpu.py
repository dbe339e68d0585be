"""Steps of AdafacLO / ELO that keep the argument table's rows against steps that fill the table anew: bit-identical whatever happens
between them, the counters one per parameter and the same objects throughout."""

import copy

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(40, 64), (64,), (7, 3, 3, 3), (5, 9), ()]


def _between(t, opt):
    ps = [p for g in opt.param_groups for p in g["params"]]
    st = [opt.state[p] for p in ps]
    if t == 2:
        opt.param_groups[0]["lr"] = 0.3
    elif t == 3:
        ps[1].grad = None                                # sits a step out: its counter lags from here on
    elif t == 5:
        st[0]["step"].fill_(40.0)
    elif t == 6:
        st[2]["step"] = torch.tensor(3.0, dtype=torch.float64)
    elif t == 7:
        st[0]["exp_avg"] = st[0]["exp_avg"] * 0.5
    elif t == 8:
        ps[3].data = ps[3].data * 1.5
    elif t == 9:
        ps[0].grad = ps[0].grad.t().contiguous().t()     # dense, not contiguous
    elif t == 10:
        opt.load_state_dict(copy.deepcopy(opt.state_dict()))
    elif t == 11:
        opt.param_groups[0]["lr"] = torch.tensor(0.2)
    elif t == 12:
        opt.param_groups[0]["lr"].mul_(2.0)
        st[4]["exp_avg"].data = st[4]["exp_avg"].data * 0.5
    elif t == 13:
        extra = torch.nn.Parameter(torch.full((6, 6), 0.25, device="cuda"))
        extra.grad = torch.full_like(extra, 0.01)
        opt.add_param_group({"params": [extra]})


@pytest.mark.parametrize("family", ["adafac", "adafac own norms", "elo"])
def test_kept_rows(family):
    from pylo_amd import ELO_CUDA, AdafacLO_CUDA
    from pylo_amd.models import MetaMLP

    torch.manual_seed(4)
    net = MetaMLP(39, 32, 1)
    init = [torch.randn(s, device="cuda") for s in SHAPES]
    runs = []
    for kept in (True, False):
        params = [torch.nn.Parameter(v.clone()) for v in init]
        if family == "elo":
            opt = ELO_CUDA(params, lr=1e-2, network=copy.deepcopy(net), hf_key=None, clip_grad=True)
        else:
            opt = AdafacLO_CUDA(params, lr=0.5, network=copy.deepcopy(net), max_grad_norm=1.0 if "own" in family else None)
        gen = torch.Generator(device="cuda").manual_seed(5)
        took = 0
        for t in range(17):
            for p in params:
                p.grad = torch.randn(p.shape, generator=gen, device="cuda") * 0.1
            if t:
                _between(t, opt)
            if not kept:
                opt._fast = None
            if t == 1:
                counters = [opt.state[p]["step"] for p in params]
            before = opt._fast
            opt.step()
            took += before is not None and opt._fast is before
            if t == 1:
                assert all(a is opt.state[p]["step"] for a, p in zip(counters, params))
        assert took >= (6 if kept else 0) and (kept or took == 0)
        ps = [p for g in opt.param_groups for p in g["params"]]
        runs.append([p.detach() for p in ps] + [opt.state[p][k] for p in ps for k in ("step", "exp_avg", "exp_avg_sq", "exp_avg_sq_r")])
    assert all(torch.equal(a, b) for a, b in zip(*runs))
