"""The tiled Newton-Schulz products at the edges of their blocks (16 x 16), sub-tiles (32 x 32) and tiles (128, 256): operand
planes are written in whole blocks through a transposing LDS read, the fp32 A lies as the accumulators of the tile that
computes it, and the padding of the planes, which nobody clears between calls, has to stay zero."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

COEFFS = (3.4445, -4.775, 2.0315)
SHAPES = [(129, 129), (129, 145), (143, 384), (144, 257), (145, 2049), (160, 161), (255, 256), (256, 272), (257, 500),
          (271, 271), (384, 400), (2050, 131), (769, 254), (300, 147), (8209, 130), (130, 8201)]


def _fp64(x):
    c0, c1, c2 = COEFFS
    x = x.double()
    t = x.shape[0] > x.shape[1]
    x = x.T if t else x
    x = x / (x.norm() + 1e-8)
    for _ in range(5):
        a = x @ x.T
        x = (c0 * torch.eye(a.shape[0], dtype=x.dtype, device=x.device) + c1 * a + c2 * (a @ a)) @ x
    x = x.T if t else x
    return x * torch.rsqrt(1e-9 + x.pow(2).mean())


@pytest.mark.parametrize("part", range(4))
@pytest.mark.parametrize("plan_of", ["few", "many", "batches"])
def test_blocks_tiles_and_padding(part, plan_of, monkeypatch):
    """Tiles of 64 x 64 (a plan of few tile jobs), of 128 x 128 and 128 x 256 (next to two large matrices), and batches of
    matrices that share their workspace.  Three calls of one plan: random steps, a NaN in every second matrix, random steps again.  The result is held to 2e-4 of its
    RMS (fp32 products sit at 2e-5 .. 5e-5), the third call's too: a product of padding with a NaN is a NaN, and what of it
    reached the planes' padding would be read by every later call."""
    from pylo_amd import _lib

    monkeypatch.setenv("PYLO_MI355_NS_SMALL", "0")
    if plan_of == "batches":
        monkeypatch.setenv("PYLO_MI355_NS_WORKSPACE_MB", "4")
    shapes = SHAPES[part::4] + ([(2304, 2304)] * 2 if plan_of == "many" else [])
    plan = _lib.Plan(_lib.KIND_CELO2, shapes, [0] * len(shapes), torch.device("cuda:0"))
    gen = torch.Generator(device="cuda").manual_seed(part)
    for call in range(3):
        steps = [torch.randn(s, generator=gen, device="cuda") for s in shapes]
        if call == 1:
            for i, x in enumerate(steps):
                if i % 2 == 0:
                    x[-1, -1] = float("nan")
        params = [torch.zeros_like(x) for x in steps]
        raw = [x.clone() for x in steps]
        fin = np.zeros(len(shapes), dtype=_lib.ARGS_DTYPE)
        for i in range(len(shapes)):
            fin["grad"][i], fin["param"][i], fin["step_out"][i] = 1, params[i].data_ptr(), steps[i].data_ptr()
            fin["lr"][i], fin["weight_decay"][i], fin["step_mult"][i] = -1.0, 0.0, 1.0
            fin["flags"][i] = _lib.ARG_ORTHOGONALIZE
        plan.celo2_orthogonalize_finish(fin, COEFFS, 5, 1e-8, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        for i, p in enumerate(params):
            if call == 1 and i % 2 == 0:
                assert torch.isnan(p).all(), shapes[i]
                continue
            want = _fp64(raw[i])
            err = float((p.double() - want).abs().max() / want.pow(2).mean().sqrt())
            assert err <= 2e-4, (call, shapes[i], err)
    plan.close()
