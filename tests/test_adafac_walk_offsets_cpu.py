"""The offsets that a wave of AdafacLO's walk over convolution kernels keeps in 32 bits, seen in the workspace that a plan asks
for (no GPU needed): rows a task x 128 bytes of first-layer terms x trailing dims have to stay below 2^32."""

import ctypes as C
import math

import pytest

from pylo_amd import _lib


def _bytes(shape):
    lib = _lib.load()
    arr = (_lib.TensorShape * 1)()
    arr[0].ndim = len(shape)
    for d, v in enumerate(shape):
        arr[0].shape[d] = v
    n = C.c_size_t()
    assert lib.pylo_mi355_plan_workspace_bytes(_lib.KIND_ADAFAC, arr, 1, C.byref(n)) == 0
    return n.value


def _tasks_of_a_column(shape, monkeypatch):
    """From the walk's blocks of four tasks (16 bytes each) against the blocks of 4096 elements of the linear pass that takes the
    tensor with the fp32 instructions.  Tables are rounded up to 256 bytes, i.e. known to some sixteen blocks."""
    monkeypatch.delenv("PYLO_MI355_ADAFAC_F32", raising=False)
    walk = _bytes(shape)
    monkeypatch.setenv("PYLO_MI355_ADAFAC_F32", "1")
    linear = _bytes(shape)
    per, columns = math.prod(shape[2:]), math.prod(shape[1:])
    blocks = (walk - linear) / 16 + math.prod(shape) / 4096
    return round(4 * blocks / (columns / 64)), per


# the fourth and the fifth wrapped with 64 rows a task
@pytest.mark.parametrize("shape,rows", [
    ((8192, 512, 3, 3, 3), 64),
    ((256, 16, 8, 8, 8, 8, 8), 64),
    ((128, 16, 12, 12, 12, 12, 12), 64),
    ((64, 16, 14, 14, 14, 14, 14), 31),
    ((16, 16, 15, 14, 14, 14, 14, 8), 3),
])
def test_row_terms_of_a_task_fit_32_bits(shape, rows, monkeypatch):
    tasks, per = _tasks_of_a_column(shape, monkeypatch)
    assert rows * 128 * per <= 2 ** 32
    assert tasks == -(-shape[0] // rows)
