"""Matrices with a smaller dim of at most 32 (k_ns_thin): folded ones, both tile counts, blocks that meet, storage types, calls that
only normalise, against the formula in fp64.

Bound: the result is an fp64 product rounded to fp32 (2^-24 of itself), times the normaliser (v_rsq_f32 of a rounded mean: 2^-23 +
2^-25), rounded, subtracted from zero: six roundings of 2^-24 cover it."""

import numpy as np
import pytest
import torch

from test_newton_schulz_gpu import _orthogonalise_direct, _reference_direct

pytestmark = pytest.mark.gpu
COEFFS = tuple(float(np.float32(c)) for c in (3.4445, -4.775, 2.0315))     # the call takes floats

SHAPES = [(m, n) for m in (1, 2, 3, 4, 5, 8, 9, 16) for n in (m, 63, 64 * 16 + 1, 20011)] + \
         [(m, n) for m in (17, 31, 32) for n in (m, 257, 4097)] + [(1, 65535), (16, 65536), (32, 32768)]


@pytest.mark.parametrize("iters", [1, 5])
@pytest.mark.parametrize("tall", [False, True])
def test_thin_matrices_against_fp64(tall, iters):
    gen = torch.Generator(device="cuda").manual_seed(iters)
    shapes = [(n, m) if tall else (m, n) for m, n in SHAPES]
    mats = [torch.randn(s, generator=gen, device="cuda") * 10.0 ** (-(i % 5)) for i, s in enumerate(shapes)]
    mats += [torch.zeros(shapes[5], device="cuda")]
    got, again = _orthogonalise_direct(mats, iters), _orthogonalise_direct(mats, iters)
    for x, y, z in zip(mats, got, again):
        assert torch.equal(y, z), tuple(x.shape)
        want = _reference_direct(x, iters, coeffs=COEFFS)
        off = float(((y.double() - want).abs() - 6 * 2.0 ** -24 * want.abs()).max())
        assert off <= 1e-9, (tuple(x.shape), off)


def _deficient(kind, m, n, gen):
    x = torch.randn((m, n), generator=gen, device="cuda")
    if kind == "constant":
        x = torch.full((m, n), 0.01, device="cuda")
    elif kind == "rank 1":
        x = torch.randn((m, 1), generator=gen, device="cuda") * torch.randn((1, n), generator=gen, device="cuda")
    elif kind == "twin rows":
        x[1::2] = x[0::2][: m // 2].clone()
    return x


@pytest.mark.parametrize("iters", [6, 7, 8, 12, 20])
@pytest.mark.parametrize("tall", [False, True])
def test_iterations_beyond_one_run(tall, iters):
    """More iterations than one Gram matrix in fp64 is good for, on matrices with and without a null space, folded, cut, and neither.
    Bound on the error's RMS over the result's: runs round X to fp32 where the formula in fp32 rounds X, A and A A after every
    iteration, so a quarter of that formula's error, and eight roundings of the result where that one is small."""
    gen = torch.Generator(device="cuda").manual_seed(iters)
    sizes = [(1, 65536), (4, 300), (4, 20011), (8, 64), (16, 16), (16, 40000), (17, 64), (32, 500), (32, 32768)]
    kinds = [(k, m, n) for m, n in sizes for k in ("gaussian", "constant", "rank 1", "twin rows")]
    mats = [_deficient(k, m, n, gen) for k, m, n in kinds]
    mats = [x.t().contiguous() for x in mats] if tall else mats
    for kind, x, got in zip(kinds, mats, _orthogonalise_direct(mats, iters)):
        want = _reference_direct(x, iters, coeffs=COEFFS)
        y = (x.t() if tall else x).cpu()
        y = y / (y.double().norm().float() + 1e-8)
        for _ in range(iters):
            a = y @ y.t()
            y = COEFFS[0] * y + (COEFFS[1] * a + COEFFS[2] * (a @ a)) @ y
        y = (y / y.double().pow(2).mean().sqrt().float()).double()
        y = (y.t() if tall else y).to(want.device)
        off = float((got.double() - want).pow(2).mean().sqrt())
        fp32 = float((y - want).pow(2).mean().sqrt())
        assert off <= 8 * 2.0 ** -24 + fp32 / 4, (kind, off, fp32)


@pytest.mark.parametrize("iters", [5, 8])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
def test_nan_and_infinity_stay_in_their_matrix(bad, iters):
    """... and reach every element of it, as in the formula; in folded and cut matrices, in the first and the last column."""
    gen = torch.Generator(device="cuda").manual_seed(8)
    shapes = [(1, 3000), (3000, 1), (4, 20011), (9, 40), (16, 65536), (32, 257), (4097, 31), (32, 32768), (32, 32)]
    mats = [torch.randn(s, generator=gen, device="cuda") for s in shapes]
    clean = _orthogonalise_direct(mats, iters)
    hit = mats[0::2]
    for i, x in enumerate(hit):
        x.view(-1)[0 if i % 2 else -1] = bad
    for i, (was, now) in enumerate(zip(clean, _orthogonalise_direct(mats, iters))):
        assert torch.isfinite(was).all()
        assert torch.isnan(now).all() if i % 2 == 0 else torch.equal(was, now), shapes[i]


def test_all_classes_next_to_slices_and_one_group_of_tiles():
    """Small matrices of every class on two streams, next to slices of tensors with more dims and to larger matrices of one group:
    three streams beside the caller's, twice over the same buffers, against the formula in fp64."""
    from test_slice_finish_gpu import _formula

    gen = torch.Generator(device="cuda").manual_seed(12)
    shapes = [(1024, 1024)] * 2 + [(40, 3, 3, 3), (7, 16, 16), (2, 64, 128), (5, 4, 1, 1)]
    for i in range(20):
        shapes += [(16 - i % 4, 700 + i), (900 + i, 17 + i % 15), (33 + i, 800), (700, 65 + 3 * i)]
    mats = [torch.randn(s, generator=gen, device="cuda") for s in shapes]
    first, second = _orthogonalise_direct(mats), _orthogonalise_direct(mats)
    for x, y, z in zip(mats, first, second):
        assert torch.equal(y, z), tuple(x.shape)
        off = float((y.double() - _formula(x, 5)).abs().max())      # the result has unit RMS
        # larger matrices: the level that their own tests hold them to on Gaussian input
        assert off <= (2e-4 if min(x.shape[-2:]) > 32 else 2e-5), (tuple(x.shape), off)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_normalise_only_and_storage(dtype):
    """Without the flag the step is applied as it stands; parameters in their own type; each at rel 6 x 2^-24 plus its spacing."""
    from pylo_amd import _lib

    flag = _lib.STORE_FLAG[dtype]
    gen = torch.Generator(device="cuda").manual_seed(3)
    mats = [torch.randn(s, generator=gen, device="cuda") for s in [(3, 5000), (5000, 3), (1, 777), (20, 900), (900, 20), (16, 16)]]
    shapes = [tuple(x.shape) for x in mats]
    plan = _lib.Plan(_lib.KIND_CELO2, shapes, [flag] * len(shapes), torch.device("cuda:0"))
    for orth in (True, False):
        steps, params = [x.clone() for x in mats], [torch.ones_like(x).to(dtype) for x in mats]
        fin = np.zeros(len(mats), dtype=_lib.ARGS_DTYPE)
        for i in range(len(mats)):
            fin["grad"][i], fin["param"][i], fin["step_out"][i] = 1, params[i].data_ptr(), steps[i].data_ptr()
            fin["lr"][i], fin["weight_decay"][i], fin["step_mult"][i] = -0.5, 0.25, 2.0
            fin["flags"][i] = _lib.ARG_ORTHOGONALIZE if orth else 0
        plan.celo2_orthogonalize_finish(fin, (3.4445, -4.775, 2.0315), 5, 1e-8, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        for x, p in zip(mats, params):
            r = _reference_direct(x, 5, coeffs=COEFFS) if orth else x.double() * torch.rsqrt(1e-9 + x.double().pow(2).mean())
            want = 1.0 + 0.5 * (2.0 * r + 0.25)
            half = 2.0 ** (-24 if dtype == torch.float32 else -8)
            off = float(((p.double() - want).abs() - 8 * 2.0 ** -24 * (1 + r.abs()) - 1.01 * half * want.abs()).max())
            assert off <= 1e-9, (tuple(x.shape), orth, off)
    plan.close()
