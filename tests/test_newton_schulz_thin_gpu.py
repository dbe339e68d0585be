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
