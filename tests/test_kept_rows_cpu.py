"""Steps that keep argument-table rows from the step before, against the table that the optimizer's parameters, groups and state ask for
at that moment, whatever a program does to them between two steps.  The library call is a stand-in that keeps the table it is
given: no kernel runs, so the parameters may lie on the CPU (``_Param`` says otherwise)."""

import contextlib
import copy
import types
import weakref

import pytest
import torch


class _Param(torch.nn.Parameter):
    is_cuda = property(lambda self: True)


class _Plan:
    def __init__(self, kind, shapes, flags, device):
        from pylo_amd import _lib
        import numpy as np

        self.args, self.tables, self.finished, self.told = np.zeros(len(shapes), dtype=_lib.ARGS_DTYPE), [], [], 0

    def adafac_step(self, decays, net, step, stream, args=None):
        table = self.args.copy()
        if step >= 0:
            table["bc1"] = step       # the counter of every tensor
        self.tables.append(table)

    def celo2_step(self, decays, mlp, stream, args=None):
        self.tables.append(self.args.copy())

    def celo2_orthogonalize_finish(self, args, coeffs, iters, eps, stream):
        self.finished.append(args.copy())

    def velo_step(self, decays, nets, step, stream, args=None):
        self.tables.append(self.args.copy())

    def orthogonalize_supported(self, i):
        return 1

    def statistics_stale(self):
        return 0

    def invalidate_statistics(self):
        self.told += 1

    def close(self):
        pass


@pytest.fixture(autouse=True)
def _no_gpu(monkeypatch):
    from pylo_amd import _lib

    monkeypatch.setattr(_lib, "Plan", _Plan)
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: types.SimpleNamespace(cuda_stream=0))


SHAPES = [(6, 5), (6, 5), (4,), (3, 2, 2), (7, 3)]


def _make(family, cut=3):
    import pylo_amd as P
    from pylo_amd.models import CELO2MLP, MetaMLP, VeLOMLP, VeLORNN

    torch.manual_seed(0)
    ps = [_Param(torch.randn(s)) for s in SHAPES]
    groups = [dict(params=ps[:cut], lr=0.5), dict(params=ps[cut:], lr=0.25)]
    if family == "adafac":
        return P.AdafacLO_CUDA(groups, network=MetaMLP(39, 32, 1))
    if family == "elo":
        return P.ELO_CUDA(groups, network=MetaMLP(39, 32, 1), hf_key=None, clip_grad=True)
    if family == "velo":
        return P.VeLO_CUDA(groups, rnn=VeLORNN(lstm_hidden_size=64, param_inits=4), mlp=VeLOMLP(param_inits=4), num_steps=100)
    cls = P.CELO2_CUDA if family == "celo2" else P.ELO_CELO2_CUDA
    return cls(groups, network=CELO2MLP(), hf_key=None)


def _params(opt):
    return [p for g in opt.param_groups for p in g["params"]]


def _address(t):
    return t.data_ptr() if t is not None and t.numel() else 0


def _check(family, opt, before):
    table = opt._plan.tables[-1]
    rows = [(gi, g, p) for gi, g in enumerate(opt.param_groups) for p in g["params"]]
    assert len(table) == len(rows)
    for i, (gi, group, p) in enumerate(rows):
        row, st = table[i], opt.state[p]
        assert row["grad"] == p.grad.data_ptr() and row["param"] == p.data_ptr(), i
        if family in ("adafac", "elo"):
            assert row["mom"] == st["exp_avg"].data_ptr() and row["rms"] == st["exp_avg_sq"].data_ptr(), i
            r, c = ("fac_v", None) if p.dim() < 2 else ("fac_r", "fac_c")
            assert row[r] == st["exp_avg_sq_r"].data_ptr() and (c is None or row[c] == st["exp_avg_sq_c"].data_ptr()), i
            assert float(st["step"]) == before[i] + 1 and row["bc1"] == before[i], (i, float(st["step"]), row["bc1"], before[i])
            assert row["lr"] == group["lr"], i
        elif family == "velo":
            assert row["mom"] == st["mom"].data_ptr() and row["rms"] == st["rms"].data_ptr(), i
            assert [row[k] for k in ("fac_r", "fac_c", "fac_v")] == [_address(st[k]) for k in ("fac_vec_row", "fac_vec_col", "fac_vec_v")], i
            assert row["lr"] == group["lr"] and row["group"] == gi, i
        else:
            adam = p.dim() < 2
            keys = ("exp_avg", "exp_avg_sq") if adam and family == "celo2" else ("mom", "rms")
            assert [row["mom"], row["rms"]] == [st[k].data_ptr() for k in keys], i
            if adam:
                assert row["lr"] == pytest.approx(group["adam_lr_mult"] * group["lr"]), i
            else:
                assert [row["fac_r"], row["fac_c"]] == [st["fac_r"].data_ptr(), st["fac_c"].data_ptr()], i
                fin = opt._plan.finished[-1][i]
                assert fin["lr"] == pytest.approx(group["lr"]) and fin["param"] == p.data_ptr() and fin["step_out"], i


def _step(family, opt):
    for p in _params(opt):
        p.grad = torch.randn(p.shape)
    before = [float(opt.state[p].get("step", 0)) if p in opt.state else 0.0 for p in _params(opt)]
    loss = torch.tensor(1.0)
    opt.step(loss)
    _check(family, opt, before)


def _copied(opt, i):
    opt.state[_params(opt)[i]] = copy.deepcopy(opt.state[_params(opt)[i]])


def _move(opt):
    a, b = opt.param_groups[:2]
    b["params"].insert(0, a["params"].pop())


def _split(opt):
    g = opt.param_groups[0]
    tail, g["params"] = g["params"][1:], g["params"][:1]
    opt.add_param_group(dict({k: v for k, v in g.items() if k != "params"}, params=tail, lr=0.125))
    opt.param_groups.insert(1, opt.param_groups.pop())


def _merge(opt):
    opt.param_groups[0]["params"] += opt.param_groups[1]["params"]
    del opt.param_groups[1]


def _swapped(opt):
    st, (p, q) = opt.state, _params(opt)[:2]
    st[p], st[q] = st[q], st[p]


EVENTS = {
    "nothing": lambda opt: None,
    "one state copied": lambda opt: _copied(opt, 1),
    "every state copied": lambda opt: [_copied(opt, i) for i in range(len(SHAPES))],
    "two states swapped": _swapped,
    "moved between groups": _move,
    "matrices moved": lambda opt: [_move(opt) for _ in range(2)],
    "group split": _split,
    "groups merged": _merge,
    "learning rate": lambda opt: opt.param_groups[1].update(lr=0.0625),
}
FAMILIES = ["adafac", "elo", "velo", "elo_celo2", "celo2"]


@pytest.mark.parametrize("event", EVENTS)
@pytest.mark.parametrize("family", FAMILIES)
def test_rows_follow_what_changed(family, event):
    if family == "velo" and event == "two states swapped":
        pytest.skip("refused: each state carries its parameter's place in the LSTM")
    opt = _make(family)
    for _ in range(3):
        _step(family, opt)
    assert opt._fast is not None
    EVENTS[event](opt)
    for _ in range(3):
        _step(family, opt)


@pytest.mark.parametrize("family", ["adafac", "elo"])
def test_replaced_accumulators_are_freed(family):
    opt = _make(family)
    for _ in range(3):
        _step(family, opt)
    st = opt.state[_params(opt)[0]]
    gone = [weakref.ref(st[k]) for k in ("exp_avg", "exp_avg_sq")]
    st["exp_avg"], st["exp_avg_sq"] = st["exp_avg"].clone(), st["exp_avg_sq"].clone()
    assert all(r() is None for r in gone)
    _step(family, opt)


@pytest.mark.parametrize("family", ["adafac", "elo"])
def test_counters_stay_where_they_are(family):
    """Views, and what shares a counter's memory, follow it; two parameters that share one advance it twice a step."""
    opt = _make(family)
    _step(family, opt)
    opt.state[_params(opt)[4]]["step"] = torch.tensor(7.0, dtype=torch.float64).share_memory_()
    steps = [opt.state[p]["step"] for p in _params(opt)]
    views = [(t.detach(), t.numpy(), t.data_ptr()) for t in steps]
    for _ in range(3):
        _step(family, opt)
    assert opt._fast is not None
    for i, (t, (view, array, at)) in enumerate(zip(steps, views)):
        want = 10.0 if i == 4 else 4.0
        assert opt.state[_params(opt)[i]]["step"] is t and t.data_ptr() == at
        assert float(t) == float(view) == float(array) == want and t.untyped_storage().nbytes() == 8, i
    assert steps[4].is_shared()
    opt.state[_params(opt)[0]]["step"] = steps[3]
    for n in range(1, 4):
        for p in _params(opt):
            p.grad = torch.randn(p.shape)
        opt.step()
        assert float(steps[3]) == 4.0 + 2 * n
        assert opt._plan.tables[-1]["bc1"][0] == 2.0 + 2 * n and opt._plan.tables[-1]["bc1"][3] == 3.0 + 2 * n


@pytest.mark.parametrize("odd", [2.0, torch.tensor(2.0)], ids=["number", "float32"])
def test_counters_of_another_kind(odd):
    """... are taken as before, and the others' are left alone."""
    opt = _make("adafac")
    _step("adafac", opt)
    opt.state[_params(opt)[3]]["step"] = odd
    at = [opt.state[p]["step"].data_ptr() for p in _params(opt)[:3]]
    for _ in range(3):
        _step("adafac", opt)
    assert opt._fast is None and float(opt.state[_params(opt)[3]]["step"]) == 5.0
    assert at == [opt.state[p]["step"].data_ptr() for p in _params(opt)[:3]]


@pytest.mark.parametrize("family", ["adafac", "elo"])
def test_rows_do_not_outlive_a_capturable_step(family, monkeypatch):
    """... which fills the table anew: the groups' scalars in it are those of that step."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    opt = _make(family)
    for _ in range(3):
        _step(family, opt)
    opt.capturable, opt.param_groups[0]["lr"] = True, 0.1
    opt.step()
    opt.capturable, opt.param_groups[0]["lr"] = False, 0.5
    _step(family, opt)


@pytest.mark.parametrize("event", ["matrices moved", "group split", "groups merged"])
@pytest.mark.parametrize("family", ["elo_celo2", "celo2"])
def test_groups_change_without_kept_rows(family, event):
    """Raw steps of one shape share a buffer that is finished group by group, whatever group each tensor is in now."""
    opt = _make(family)
    for _ in range(2):
        _step(family, opt)
    EVENTS[event](opt)
    for _ in range(2):
        opt._fast = None
        _step(family, opt)


def test_velo_frozen_parameters_do_not_hide_a_move():
    """Frozen parameters have no row: the groups' lists keep their lengths while a row goes from one group to the other."""
    opt = _make("velo")
    a, b = opt.param_groups
    frozen = [_Param(torch.zeros(2)).requires_grad_(False) for _ in range(2)]
    a["params"].append(frozen[0])
    b["params"].append(frozen[1])
    rows = [p for p in _params(opt) if p.requires_grad]

    def step():
        for p in rows:
            p.grad = torch.randn(p.shape)
        opt.step(torch.tensor(1.0))
        table = opt._plan.tables[-1]
        assert [p.data_ptr() for p in rows] == table["param"].tolist()
        assert [gi for gi, g in enumerate(opt.param_groups) for p in g["params"] if p.requires_grad] == table["group"].tolist()

    for _ in range(3):
        step()
    assert opt._fast is not None
    b["params"].insert(0, a["params"].pop(2))
    a["params"].append(b["params"].pop())
    for _ in range(2):
        step()


@pytest.mark.parametrize("family", FAMILIES)
def test_sparse_gradients_are_refused(family):
    opt = _make(family)
    for _ in range(3):
        _step(family, opt)
    n, p = len(opt._plan.tables), _params(opt)[4]
    p.grad = torch.eye(7, 3).to_sparse()
    with pytest.raises((RuntimeError, TypeError), match="[Ss]parse|dense"):
        opt.step(torch.tensor(1.0))
    assert len(opt._plan.tables) == n
    p.grad = None
    if family == "velo":
        with pytest.raises(RuntimeError, match="needs a gradient"):
            opt.step(torch.tensor(1.0))
    else:
        opt.step()
        assert opt._plan.tables[-1]["grad"][4] == 0
    for _ in range(3):
        _step(family, opt)


@pytest.mark.parametrize("family", ["adafac", "elo", "elo_celo2", "celo2"])
def test_cleared_states_start_again(family):
    opt = _make(family)
    for _ in range(3):
        _step(family, opt)
    for p in _params(opt)[1:3]:
        opt.state[p] = {}
    for _ in range(2):
        _step(family, opt)
    key = "exp_avg_sq" if family in ("adafac", "elo") else "rms"
    assert key in opt.state[_params(opt)[1]]


@pytest.mark.parametrize("family", ["elo_celo2", "celo2"])
def test_another_group_in_its_place(family):
    opt = _make(family)
    for _ in range(3):
        _step(family, opt)
    opt.param_groups[1] = dict(opt.param_groups[1], lr=0.0625, param_scale_mult=True)
    for _ in range(2):
        _step(family, opt)


@pytest.mark.parametrize("family", FAMILIES)
def test_another_parameter_in_its_place(family):
    opt = _make(family)
    for _ in range(3):
        _step(family, opt)
    old = opt.param_groups[0]["params"][1]
    new = _Param(old.detach() * 2)
    opt.state[new] = opt.state.pop(old)
    opt.param_groups[0]["params"][1] = new
    for _ in range(2):
        _step(family, opt)


@pytest.mark.parametrize("family", FAMILIES)
def test_a_parameter_of_another_size(family):
    """Rows made for the old size would send the kernels past the end of the new tensors."""
    opt = _make(family)
    for _ in range(3):
        _step(family, opt)
    p, plan = _params(opt)[0], opt._plan
    p.grad = None
    p.data = torch.randn(2, 5)
    _step(family, opt)
    assert opt._plan is not plan


@pytest.mark.parametrize("family", FAMILIES)
def test_parameters_of_another_type(family):
    opt = _make(family)
    for old, new in ((torch.float32, torch.bfloat16), (torch.bfloat16, torch.float16), (torch.float16, torch.float32)):
        for dtype in (old, old, old, new):
            for p in _params(opt):
                p.grad = None
                p.data = p.data.to(dtype)
            before, plan = [float(opt.state[p].get("step", 0)) if p in opt.state else 0.0 for p in _params(opt)], opt._plan
            for p in _params(opt):
                p.grad = torch.randn(p.shape, dtype=dtype)
            opt.step(torch.tensor(1.0))
            _check(family, opt, before)
            assert (opt._plan is not plan) == (plan is None or dtype is new)
