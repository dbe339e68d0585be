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
