"""Accumulators are float32 whatever type the parameters are stored in: the kernels read and write four bytes an element."""

import pytest
import torch

DTYPES = [torch.float32, torch.bfloat16, torch.float16, torch.float64]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("adam", [True, False])
@pytest.mark.parametrize("shape", [(70001,), (33, 17)])
def test_celo2_state_is_float32(dtype, adam, shape):
    from pylo_amd import CELO2_CUDA

    opt = object.__new__(CELO2_CUDA)
    opt.device, opt.n_mom, opt.n_fac = torch.device("cpu"), 3, 3
    state = {}
    opt._init_state(state, torch.nn.Parameter(torch.zeros(shape, dtype=dtype)), adam)
    tensors = [t for t in state.values() if torch.is_tensor(t)]
    assert tensors and all(t.dtype == torch.float32 for t in tensors)


@pytest.mark.parametrize("dtype", DTYPES)
def test_loaded_state_is_float32_and_unrounded(dtype):
    from pylo_amd import _lib

    def make():
        p = torch.nn.Parameter(torch.zeros(7, 5, dtype=dtype))
        q = torch.nn.Parameter(torch.zeros(3, dtype=dtype))
        return torch.optim.SGD([{"params": [p]}, {"params": [q]}], lr=0.1), p, q

    a, p, q = make()
    a.state[p].update(mom=torch.randn(3, 7, 5), rms=1e-9 * torch.rand(7, 5), step=torch.tensor(3.0, dtype=torch.float64), adam_step=2)
    b, p2, q2 = make()
    sd = a.state_dict()
    b.load_state_dict(sd)
    _lib.keep_float32_state(b, sd)
    assert torch.equal(b.state[p2]["mom"], a.state[p]["mom"]) and b.state[p2]["mom"].dtype == torch.float32
    assert torch.equal(b.state[p2]["rms"], a.state[p]["rms"]) and b.state[p2]["rms"].dtype == torch.float32
    assert b.state[p2]["step"].dtype == torch.float64 and b.state[p2]["adam_step"] == 2
    assert not b.state.get(q2)
    # accumulators that were saved in the parameter's type are widened
    sd["state"][0]["mom"] = sd["state"][0]["mom"].to(dtype)
    b.load_state_dict(sd)
    _lib.keep_float32_state(b, sd)
    assert torch.equal(b.state[p2]["mom"], a.state[p]["mom"].to(dtype).float())


@pytest.mark.parametrize("dtype", [t for t in DTYPES if t != torch.float32])
def test_loaded_state_is_a_copy(dtype):
    """Steps write accumulators in place: neither the dict nor the optimizer that it came from may see it, and a second load
    from the same dict starts where the first did."""
    from pylo_amd import _lib

    def make():
        p = torch.nn.Parameter(torch.zeros(7, 5, dtype=dtype))
        return torch.optim.SGD([p], lr=0.1), p

    a, p = make()
    a.state[p].update(mom=torch.randn(3, 7, 5), rms=torch.rand(7, 5), step=3)
    kept = {k: v.clone() for k, v in a.state[p].items() if torch.is_tensor(v)}
    sd = a.state_dict()
    for _ in range(2):
        b, q = make()
        b.load_state_dict(sd)
        _lib.keep_float32_state(b, sd)
        for k, v in kept.items():
            assert torch.equal(b.state[q][k], v)
            b.state[q][k].add_(1.0)
            assert torch.equal(a.state[p][k], v) and torch.equal(sd["state"][0][k], v)


@pytest.mark.parametrize("dtype", DTYPES)
def test_tensors_of_two_names_stay_one(dtype):
    """AdafacLO keeps the second moments of a vector under two names."""
    from pylo_amd import _lib

    p, q = (torch.nn.Parameter(torch.zeros(7, 5, dtype=dtype)) for _ in range(2))
    a, b = torch.optim.SGD([p], lr=0.1), torch.optim.SGD([q], lr=0.1)
    a.state[p].update(mom=torch.randn(3, 7, 5), rms=torch.rand(7, 5))
    a.state[p]["exp_avg"] = a.state[p]["mom"]
    sd = a.state_dict()
    b.load_state_dict(sd)
    _lib.keep_float32_state(b, sd)
    assert b.state[q]["exp_avg"] is b.state[q]["mom"] and b.state[q]["rms"] is not b.state[q]["mom"]


@pytest.mark.parametrize("dtype", DTYPES)
def test_hooks_of_loading_are_heard(dtype):
    """What a hook before the load puts into the dict, or returns in its place, is what is loaded; what one after it does to the
    state stays."""
    from pylo_amd import AdafacLO_CUDA

    def make():
        opt = object.__new__(AdafacLO_CUDA)
        p = torch.nn.Parameter(torch.zeros(7, 5, dtype=dtype))
        torch.optim.Optimizer.__init__(opt, [p], {"lr": 0.1})
        opt.capturable = False
        opt.sync_step_counters = lambda: None
        return opt, p

    a, p = make()
    a.state[p].update(mom=torch.randn(3, 7, 5), rms=torch.rand(7, 5), step=3)
    b, q = make()

    def doubled(_, sd):
        return {**sd, "state": {0: {**sd["state"][0], "mom": 2.0 * sd["state"][0]["mom"]}}}

    def cleared(opt):
        opt.state[q]["rms"].zero_()

    b.register_load_state_dict_pre_hook(doubled)
    b.register_load_state_dict_post_hook(cleared)
    b.load_state_dict(a.state_dict())
    assert torch.equal(b.state[q]["mom"], 2.0 * a.state[p]["mom"])
    assert b.state[q]["rms"].dtype == torch.float32 and not b.state[q]["rms"].any()
