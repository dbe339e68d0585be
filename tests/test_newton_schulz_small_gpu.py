"""Small matrices (smaller dim at most 128) that one launch takes from the raw step to the parameter: every class of
sizes at its edges, matrices of one block and of several that meet, against the literal formula in fp64.

The bound is that of the tiled products' tests: no further from fp64 than 1.5 times what the formula in fp32 torch
products is, plus 5e-5 of the result's unit RMS (the operands' two fp16 planes and the pairing of iterations)."""

import numpy as np
import pytest
import torch

from test_newton_schulz_gpu import _orthogonalise_direct, _reference_direct

pytestmark = pytest.mark.gpu

SETS = {
    "up to 32": [(1, 1), (1, 7), (7, 1), (31, 33), (32, 32), (5, 128), (129, 5), (32, 1025), (3000, 17), (1, 30000), (16, 65536), (17, 32769)],
    "up to 64": [(33, 33), (33, 128), (129, 40), (64, 64), (64, 2048), (4099, 37), (37, 8191), (32768, 33)],
    "past the limits": [(65537, 5), (32769, 33), (8193, 96), (70, 8200)],       # the tiled products', with no small ones
    "four long ones": [(64, 32768), (25000, 49), (63, 24577), (30001, 64)],     # one to three of these are the tiled products'
    "sixteen long ones": [(128, 8192), (8192, 127), (1025, 128), (128, 4099), (2148, 100), (5754, 72), (7820, 65), (3000, 96)] * 2,
    "beside a higher class": [(16, 65536), (64, 8192), (65, 65), (3, 9)],       # lifted, and too long to be
    "beside larger ones": [(10, 512), (512, 300), (100, 300), (31, 33)],        # in the larger ones' launches
    "up to 128": [(65, 65), (65, 128), (129, 100), (128, 128), (784, 128), (128, 4096), (1027, 127), (96, 257), (8193, 80)],
}


@pytest.mark.parametrize("iters", [1, 2, 5])
@pytest.mark.parametrize("which", list(SETS))
def test_small_matrices_against_fp64(which, iters):
    gen = torch.Generator(device="cuda").manual_seed(iters)
    mats = [torch.randn(s, generator=gen, device="cuda") * 10.0 ** (-(i % 5)) for i, s in enumerate(SETS[which])]
    got = _orthogonalise_direct(mats, iters)
    again = _orthogonalise_direct(mats, iters)
    prev = torch.backends.cuda.matmul.allow_tf32
    torch.backends.cuda.matmul.allow_tf32 = False
    try:
        for x, y, z in zip(mats, got, again):
            want = _reference_direct(x, iters)
            e = float((y.double() - want).abs().max())
            e32 = float((_reference_direct(x, iters, dtype=torch.float32).double() - want).abs().max())
            print(tuple(x.shape), iters, e, e32)
            assert torch.equal(y, z), tuple(x.shape)
            assert e <= 1.5 * e32 + 5e-5, (tuple(x.shape), e, e32)
    finally:
        torch.backends.cuda.matmul.allow_tf32 = prev


@pytest.mark.parametrize("counts", [(24, 30, 20), (80, 100, 60)])
def test_many_that_meet_and_repeated_calls(counts):
    """Matrices of several blocks: all of them running at once, and more of them than a launch holds at a time (longer
    slabs, blocks that start when others end).  A plan used again and again, a NaN that stays in its matrix, and a call that
    only normalises and applies."""
    from pylo_amd import _lib

    a, b, c = counts
    n = a + b + c
    shapes = [(128, 784)] * a + [(60, 1500)] * b + [(3, 5000)] * c + [(128, 784), (200, 300)]
    gen = torch.Generator(device="cuda").manual_seed(1)
    mats = [torch.randn(s, generator=gen, device="cuda") for s in shapes]
    mats[5][3, 700] = float("nan")
    plan = _lib.Plan(_lib.KIND_CELO2, shapes, [0] * len(shapes), torch.device("cuda:0"))
    fin = np.zeros(len(mats), dtype=_lib.ARGS_DTYPE)
    want = None
    for call in range(4):
        steps = [x.clone() for x in mats]
        params = [torch.zeros_like(x) for x in mats]
        for i in range(len(mats)):
            fin["grad"][i], fin["param"][i], fin["step_out"][i] = 1, params[i].data_ptr(), steps[i].data_ptr()
            fin["lr"][i], fin["weight_decay"][i], fin["step_mult"][i] = -1.0, 0.0, 1.0
            fin["flags"][i] = _lib.ARG_ORTHOGONALIZE if call < 3 else 0
        plan.celo2_orthogonalize_finish(fin, (3.4445, -4.775, 2.0315), 5, 1e-8, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.isnan(params[5]).all()
        if call == 0:
            want = params
            for i in (0, a - 1, a, a + b - 1, a + b, n - 1, n + 1):
                assert float((params[i].double() - _reference_direct(mats[i])).abs().max()) <= 2e-4, i
            assert float((params[n].double() - _reference_direct(mats[n])).abs().max()) <= 2e-4
        elif call < 3:
            assert all(torch.equal(x, y) for i, (x, y) in enumerate(zip(params, want)) if i != 5)
        else:
            for i, x in enumerate(mats):
                if i != 5:
                    r = x.double() * torch.rsqrt(1e-9 + x.double().pow(2).mean())
                    assert float((params[i].double() - r).abs().max()) <= 1e-5, i
    plan.close()


@pytest.mark.parametrize("square", [1.0 + 1.4e-5, 1.0 + 2.9e-6, 1.21])
def test_sums_of_squares_of_long_matrices(square):
    """Equal entries, whose roundings all fall to the same side: the normaliser of a call that only applies the step.
    Sums of at most 32 squares run in fp32, so the mean square is off by at most 31 * 2^-24 of itself and the
    normaliser by half of that; the normaliser, the squares and the result are rounded by 2^-23 each at the most."""
    from pylo_amd import _lib

    shapes = [(16, 65536), (65536, 3), (64, 32768), (128, 4096), (8192, 128), (32, 1025)]
    mats = [torch.full(s, square ** 0.5, device="cuda") for s in shapes]
    plan = _lib.Plan(_lib.KIND_CELO2, shapes, [0] * len(shapes), torch.device("cuda:0"))
    fin = np.zeros(len(mats), dtype=_lib.ARGS_DTYPE)
    params = [torch.zeros_like(x) for x in mats]
    for i in range(len(mats)):
        fin["grad"][i], fin["param"][i], fin["step_out"][i] = 1, params[i].data_ptr(), mats[i].data_ptr()
        fin["lr"][i], fin["weight_decay"][i], fin["step_mult"][i] = -1.0, 0.0, 1.0
    want = [float(x.double().mul(torch.rsqrt(1e-9 + x.double().pow(2).mean()))[0, 0]) for x in mats]
    plan.celo2_orthogonalize_finish(fin, (3.4445, -4.775, 2.0315), 5, 1e-8, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for s, p, w in zip(shapes, params, want):
        off = float((p.double() / w - 1.0).abs().max())
        print(s, off)
        assert off <= 31 * 2.0 ** -25 + 3 * 2.0 ** -23, (s, off)
    plan.close()


@pytest.mark.parametrize("shape,offset,refused", [((128, 128), 4, True), ((2, 128, 128), 8, True), ((3, 4), 8, True), ((7, 9), 4, False)])
def test_alignment_of_the_finishing_call(shape, offset, refused):
    """Steps and parameters of whole groups of four elements are 16-byte aligned, others 4-byte: what the finishing pass
    of every other matrix asks for.  A refused call launches nothing."""
    from pylo_amd import _lib

    n = int(np.prod(shape))
    raw = torch.randn(n + 8, device="cuda")
    step = raw[offset // 4:offset // 4 + n]
    param = torch.zeros(n, device="cuda")
    plan = _lib.Plan(_lib.KIND_CELO2, [shape], [0], torch.device("cuda:0"))
    fin = np.zeros(1, dtype=_lib.ARGS_DTYPE)
    fin["grad"][0], fin["param"][0], fin["step_out"][0] = 1, param.data_ptr(), step.data_ptr()
    fin["lr"][0], fin["step_mult"][0] = -1.0, 1.0
    args = (fin, (3.4445, -4.775, 2.0315), 5, 1e-8, torch.cuda.current_stream().cuda_stream)
    if refused:
        with pytest.raises(RuntimeError, match="misaligned"):
            plan.celo2_orthogonalize_finish(*args)
        torch.cuda.synchronize()
        assert not param.any()
    else:
        plan.celo2_orthogonalize_finish(*args)
        x = step.double()
        assert float((param.double() - x * torch.rsqrt(1e-9 + x.pow(2).mean())).abs().max()) <= 1e-5
    plan.close()


def test_slices_aside():
    """Tensors of more than two dims whose slices are small matrices, with no larger one in the plan."""
    gen = torch.Generator(device="cuda").manual_seed(2)
    mats = [torch.randn(s, generator=gen, device="cuda") for s in [(2, 128, 128), (3, 64, 300), (2, 2, 100, 201), (1, 8100, 40)]]
    for x, y in zip(mats, _orthogonalise_direct(mats)):
        for xs, ys in zip(x.reshape(-1, *x.shape[-2:]), y.reshape(-1, *x.shape[-2:])):
            want = _reference_direct(xs)
            e32 = float((_reference_direct(xs, dtype=torch.float32).double() - want).abs().max())
            assert float((ys.double() - want).abs().max()) <= 1.5 * e32 + 5e-5, tuple(x.shape)
