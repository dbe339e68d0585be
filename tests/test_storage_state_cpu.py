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
