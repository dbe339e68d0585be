"""Short slices of tensors with more than two dims on the fused ELO-CELO2 call (k_celo2_slices_wave): whole slices packed into
waves, one lane an element.  Raw steps and accumulators against the oracle, parameters re-synchronised after every step."""

import pytest
import torch

from golden_io import max_err
from test_celo2_gpu import ABS, REL, _check_states, _mk, _net, _pair, step_keeping_raw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [
    # a slice an element, nine elements (3 x 3), and lengths that leave lanes of a wave idle, end inside a wave or fill half of one
    [(40, 24, 1, 1), (5, 7, 1, 1), (24, 40, 3, 3), (13, 9, 3, 3), (1, 2, 1, 1)],
    [(12, 10, 2, 1), (9, 8, 5, 1), (16, 12, 4, 4), (12, 14, 5, 5), (33, 34, 1, 31), (33, 35, 8, 4), (40, 36, 7, 3)],
    # factored dims that are dims of the slice: channels differ inside an entry's run
    [(2, 3, 5, 5), (3, 2, 4, 7), (16, 1, 5, 1), (6, 4, 6)],
    # three trips of a wave, several blocks a tensor, next to a matrix and a vector
    [(300, 260, 3, 3), (520, 500, 1, 1), (64, 130), (300,)],
    # eight trips, the most a wave takes, in every launch; blocks that end in the middle of their trips.  A million slices of one
    # element: their gradients are of one sign, because f / sqrt(1e-9 + f^2) turns an error of 2^-24 in a momentum that has
    # cancelled to a 3e-5th of its own scale into one of 2e-3, and of so many some do
    [(1030, 1030, 1, 1), (515, 515, 3, 3), (200, 190, 5, 1), (1500, 2, 3, 4), (700, 1, 5, 1)],
])
@pytest.mark.parametrize("clip", [True, False])
def test_packed_slices_match_oracle(shapes, clip):
    net = _net()
    init, gen = _mk(shapes, 7)
    orc, opt, cpu, gpu = _pair(shapes, init, net, dict(lr=1e-3, exp_mult=0.01, clip_grad=clip, orthogonalize=False))
    for t in range(3):
        grads = [torch.randn(s, generator=gen) * 10.0 ** (-i % 3) for i, s in enumerate(shapes)]
        if shapes[0][0] * shapes[0][1] > 10 ** 6:
            grads = [g.abs_().add_(0.1) for g in grads]
        raw = {}
        for p, g in zip(gpu, grads):
            p.grad = g.cuda()
        orc.step(grads, keep_raw=raw)
        kept = step_keeping_raw(opt)
        torch.cuda.synchronize()
        _check_states(opt, orc, gpu, t)
        for i, r in raw.items():
            e = max_err(kept[i], r, REL, ABS)
            assert e <= 1.0, ("raw step", t, i, shapes[i], e)
        for pc, pg in zip(cpu, gpu):
            pg.data.copy_(pc)


def test_clipping_turned_on_and_off():
    """One plan whose steps take the sums of kernels before the norm is known and after it in turn: a step's order of launches
    follows from its own arguments, whatever the step before left."""
    net = _net()
    shapes = [(40, 24, 3, 3), (64, 40), (24, 40, 1, 1), (300,), (130, 64)]
    init, gen = _mk(shapes, 8)
    orc, opt, cpu, gpu = _pair(shapes, init, net, dict(lr=1e-3, exp_mult=0.01, clip_grad=True, orthogonalize=False))
    for t, clip in enumerate([True, False, False, True, False, True, True]):
        orc.h["clip_grad"] = opt.param_groups[0]["clip_grad"] = clip
        grads = [torch.randn(s, generator=gen) * 10.0 ** (-i % 3) for i, s in enumerate(shapes)]
        raw = {}
        for p, g in zip(gpu, grads):
            p.grad = g.cuda()
        orc.step(grads, keep_raw=raw)
        kept = step_keeping_raw(opt)
        torch.cuda.synchronize()
        _check_states(opt, orc, gpu, t)
        for i, r in raw.items():
            e = max_err(kept[i], r, REL, ABS)
            assert e <= 1.0, ("raw step", t, i, shapes[i], e)
        for pc, pg in zip(cpu, gpu):
            pg.data.copy_(pc)
