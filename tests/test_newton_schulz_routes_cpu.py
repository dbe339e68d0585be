"""Which launches take a plan's small matrices, seen in the workspace that a plan asks for (no GPU needed).

A matrix that goes through the tiled products has operand planes and tile tables there, one that goes aside (k_ns_small.h)
partial sums: 2 x blocks x (32, 64 or 128)^2 floats, the edge being that of the class it runs in."""

import ctypes as C

import pytest

from pylo_amd import _lib


def _bytes(shapes):
    lib = _lib.load()
    arr = (_lib.TensorShape * len(shapes))()
    for i, s in enumerate(shapes):
        arr[i].ndim = len(s)
        for d, v in enumerate(s):
            arr[i].shape[d] = v
    n = C.c_size_t()
    assert lib.pylo_mi355_plan_workspace_bytes(_lib.KIND_CELO2, arr, len(shapes), C.byref(n)) == 0
    return n.value


def _decoder(width, kv, layers):
    return [(width, width), (width, kv), (width, kv), (width, width), (width, 3 * width)] * layers


# few small matrices next to one group of larger ones ride with them: the plan is the one that has no small launches
@pytest.mark.parametrize("shapes", [
    [(1024, 784), (1024, 1024), (10, 1024)],
    [(384, 784), (384, 384), (10, 384)],
    [(512, 512)] + [(16, 1024), (1024, 16)] * 8,
    _decoder(256, 32, 3),
], ids=["classifier 1024", "classifier 384", "adapters beside one matrix", "decoder 256"])
def test_small_matrices_ride_with_larger_ones(shapes, monkeypatch):
    monkeypatch.delenv("PYLO_MI355_NS_SMALL", raising=False)
    default = _bytes(shapes)
    monkeypatch.setenv("PYLO_MI355_NS_SMALL", "0")
    assert default == _bytes(shapes)


# no larger ones, many small ones, or larger ones with launches that fill the chip: aside
@pytest.mark.parametrize("shapes", [
    [(128, 784), (128, 128), (10, 128)],
    [(512, 512)] + [(60, 100)] * 600,
    [(1024, 1024)] * 4 + [(16, 1024), (1024, 16)] * 8,
    _decoder(512, 64, 8),
], ids=["classifier 128", "many", "adapters beside four matrices", "decoder 512"])
def test_small_matrices_aside(shapes, monkeypatch):
    monkeypatch.delenv("PYLO_MI355_NS_SMALL", raising=False)
    default = _bytes(shapes)
    monkeypatch.setenv("PYLO_MI355_NS_SMALL", "0")
    assert default != _bytes(shapes)


@pytest.mark.parametrize("name,value", [("PYLO_MI355_NS_CHAINS", "3,2"), ("PYLO_MI355_NS_ADAPTIVE", "1")])
def test_other_chain_lengths_reach_small_matrices(name, value, monkeypatch):
    """Chains other than pairs and singles are the tiled products': a plan made while the environment asks for them has no
    small launches."""
    shapes = [(128, 784), (128, 128), (10, 128)]
    monkeypatch.setenv(name, value)
    asked = _bytes(shapes)
    monkeypatch.setenv("PYLO_MI355_NS_SMALL", "0")
    assert asked == _bytes(shapes)


@pytest.mark.parametrize("longs", [[(16, 65536)], [(65536, 9)], [(16, 65536)] * 20])
def test_long_thin_matrices_keep_their_class(longs):
    """Next to one 100 x 100 their blocks and partial sums are those that they have without it (64 x 32^2 floats, twice; the
    largest class would give them 8 x 128^2)."""
    assert _bytes(longs + [(100, 100)]) - _bytes(longs) <= _bytes([(100, 100)])


# long matrices with a smaller dim above 32: few of them go to tiles, many stay with the one-launch kernel
@pytest.mark.parametrize("shape,few,many", [((128, 2048), 15, 16), ((4096, 100), 1, 16), ((72, 8192), 15, 200),
                                            ((64, 32768), 3, 4), ((25000, 49), 1, 64)])
def test_long_matrices_go_to_tiles_while_they_are_few(shape, few, many, monkeypatch):
    monkeypatch.delenv("PYLO_MI355_NS_SMALL", raising=False)
    default = [_bytes([shape] * c) for c in (few, many)]
    monkeypatch.setenv("PYLO_MI355_NS_SMALL", "0")
    tiled = [_bytes([shape] * c) for c in (few, many)]
    assert default[0] == tiled[0] and default[1] != tiled[1]


def test_long_matrices_end_under_the_launch_of_many_others(monkeypatch):
    """One of 2000 x 128 next to eight and to eighty of 128 x 128: as the other launch and this one need, apart or together."""
    monkeypatch.delenv("PYLO_MI355_NS_SMALL", raising=False)
    few, many = ([(128, 128)] * c for c in (8, 80))
    alone = _bytes([(2000, 128)])
    together = 2 * 8 * 128 * 128 * 4              # its partial sums: eight blocks
    assert _bytes(few + [(2000, 128)]) - _bytes(few) > 0.9 * alone
    assert abs(_bytes(many + [(2000, 128)]) - _bytes(many) - together) < 0.9 * (alone - together)


@pytest.mark.parametrize("shape", [(128, 1024), (72, 5700), (100, 2100), (64, 24000), (48, 32768), (17, 30000), (16, 65536)])
def test_others_never_do(shape, monkeypatch):
    monkeypatch.delenv("PYLO_MI355_NS_SMALL", raising=False)
    default = _bytes([shape])
    monkeypatch.setenv("PYLO_MI355_NS_SMALL", "0")
    assert default != _bytes([shape])
