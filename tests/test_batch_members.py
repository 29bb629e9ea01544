"""Members of a batch are HTensors like any other: their class, equality, copies and fields."""
import copy
import dataclasses

import numpy as np
import pytest

import ht_tensor_learning_using_gpu_tensor_cores_amd as ht
from ht_tensor_learning_using_gpu_tensor_cores_amd import engine

DIMS, RANKS = [5, 6, 7], [1, 2, 2, 2, 2]


def plain(packed, err):
    tr = ht.tree.first_vs_rest_3d()
    layout = ht.output_layout(DIMS, tr, RANKS, False)
    r = ht.HTensor(dims=DIMS, tree=tr, ranks=RANKS, packed=packed, rel_err=err)
    engine._unpack(r, layout)
    return r


@pytest.fixture
def packed():
    n = ht.output_layout(DIMS, ht.tree.first_vs_rest_3d(), RANKS, False)[3]
    return np.arange(n, dtype=np.float32)


def members(packed, calls):
    def make(b):
        calls.append(b)
        return vars(plain(packed, 0.25))
    return engine._lazy_members([0.25, 0.5], make)


def test_class_and_equality(packed):
    calls = []
    a, b = members(packed, calls)
    assert type(a) is ht.HTensor and a.rel_err == 0.25 and calls == []
    ref = plain(packed, 0.25)
    ref.U, ref.B, ref.sv = a.U, a.B, a.sv
    b.dims = [5, 6, 8]
    assert a == ref and ref == a and a != b
    assert b.ranks == RANKS and calls == [0, 1]  # made once each
    assert vars(a).keys() == vars(ref).keys()
    assert [f.name for f in dataclasses.fields(a)] == list(vars(ref))


@pytest.mark.parametrize("read_first", [False, True])
def test_copies_hold_the_fields(packed, read_first):
    a = members(packed, [])[0]
    if read_first:
        a.packed
    shallow, deep = copy.copy(a), copy.deepcopy(a)
    assert shallow.packed is a.packed and type(shallow) is ht.HTensor
    assert deep.packed is not a.packed and np.array_equal(deep.packed, a.packed)
    deep.packed[0] = -1.0
    assert a.packed[0] == 0.0
    assert vars(deep).keys() == vars(a).keys() == vars(plain(packed, 0.0)).keys()


def test_set_fields_stay_and_unknown_ones_fail(packed):
    a = members(packed, [])[0]
    a.stats = {"mine": 1}
    a.dims = "set before"
    assert a.ranks == RANKS and a.stats == {"mine": 1} and a.dims == "set before" and a.rel_err == 0.25
    with pytest.raises(AttributeError, match="HTensor.*nothing"):
        a.nothing
    with pytest.raises(AttributeError):
        plain(packed, 0.0).nothing
