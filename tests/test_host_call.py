"""Host side of the native calls, without a GPU: the pass over the row offsets against numpy, and what a matrix keeps for them."""
import ctypes
import types

import numpy as np
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from rode_amd import RoDeCSR, _lib, rode_sddmm_hip


@pytest.mark.parametrize("rows", [0, 1, 7, 65535, 65536, 65537, 200_001])  # (sums are taken per 65536 rows)
def test_row_stats(rows):
    rng = np.random.default_rng(rows)
    lens = np.minimum(rng.lognormal(2, 2.5, rows), 5000).astype(np.int64)
    ro = np.concatenate([[3], 3 + np.cumsum(lens)])
    aligned = lens + (ro[:-1] & 3)
    blocked = aligned >= 32
    want = (lens.max(initial=0), aligned.min() if rows else 0, aligned.max() if rows else 0, blocked.sum(),
            (((aligned + 511) >> 9) * blocked).sum(), (blocked & (aligned <= 512)).sum(), (blocked & (aligned <= 1024)).sum(),
            (lens * (aligned >= 500)).sum())
    for kind in (np.int32, np.int64):
        assert _lib.host_call().row_stats(torch.from_numpy(ro.astype(kind)), 500) == tuple(int(v) for v in want)
    with pytest.raises(ValueError):
        _lib.host_call().row_stats(torch.zeros(3), 500)


@pytest.mark.parametrize("kind", ["fake", "vmap", "sparse", "subclass"])
def test_row_stats_of_other_tensors(kind):
    """No tensor of its kind ends in an abort or a read of memory that is not there."""
    ro = torch.tensor([0, 3, 5], dtype=torch.int32)
    got = []

    def call(t):
        if kind == "subclass":  # its elements are where a tensor's are
            got.append(_lib.host_call().row_stats(t, 5)[:3] == (3, 3, 5))
        else:
            with pytest.raises(ValueError):
                _lib.host_call().row_stats(t, 5)
            got.append(True)
        return t

    if kind == "fake":
        call(FakeTensorMode().from_tensor(ro))
    elif kind == "vmap":
        torch.vmap(call)(ro.expand(2, 3))
    else:
        call(ro.to_sparse() if kind == "sparse" else ro.as_subclass(type("Subclass", (torch.Tensor,), {})))
    assert got == [True]


def _stand_in(plan=None):
    csr = object.__new__(RoDeCSR)
    csr.plan, csr.config, csr.columns_local, csr.nnz, csr._shared = plan, {"seg_length": 512}, False, 1, {}
    return csr


def test_two_first_calls_get_one_plans_struct(monkeypatch):
    """Another thread's first call runs from start to end while this one builds its struct."""
    csr, build, other = _stand_in(), rode_sddmm_hip.plans_struct, []

    def interrupted(*args, **kwargs):
        if not other:
            other.append(None)
            other[0] = csr.plans_address()
        return build(*args, **kwargs)

    monkeypatch.setattr(rode_sddmm_hip, "plans_struct", interrupted)
    address = csr.plans_address()
    assert address == other[0] == ctypes.addressof(csr.call_plans()) == csr.plans_address()
    held = address.plans  # the struct lives as long as its address is held, whatever the matrix keeps
    csr._shared.clear()
    assert ctypes.addressof(held) == address and held.seg_length == 512


def test_two_first_calls_get_one_hub_workspace(monkeypatch):
    plan, other = rode_sddmm_hip.HubPlan(torch.zeros(16, dtype=torch.int32), [1, 1, 32, 1, 1, 0, 0, 0]), []

    def size(header, n, elem_bytes):
        if not other:
            other.append(None)
            other[0] = plan.workspace(n, elem_bytes)
        return 64

    monkeypatch.setattr(_lib, "load", lambda: types.SimpleNamespace(rode_hip_hub_workspace_bytes=size))
    assert plan.workspace(32, 4) is other[0] is plan.workspace(32, 4)
    csr = _stand_in(plan)
    assert csr.plans_address(32).plans.hub_workspace == other[0].data_ptr() and csr.plans_address() != csr.plans_address(32)


@pytest.mark.parametrize("n", [32, 128, 256, 1024])
@pytest.mark.parametrize("elem", [4, 8])
def test_hub_workspace_is_bounded(n, elem):
    """The partial rows of an SpMM with all rows of a hub plan take up to eight dense operands (of 4 or 8 bytes an element); with more a
    call takes the long rows, which are few."""
    lib, slabs, longs = _lib.load(), 128, 300

    def size(rows, mean):
        header = (ctypes.c_int * 8)(rows, slabs, 512, 1, rows, longs, rows * mean, longs * 9000)
        return lib.rode_hip_hub_workspace_bytes(ctypes.addressof(header), n, elem)

    operand, few = slabs * 2048 * n * elem, size(599, 1200)  # (fewer than 600 rows: the long ones)
    assert 0 < few <= longs * slabs * n * elem
    for rows in (600, 8000, 16500, 40000, 100_000, 200_000):
        assert few < size(rows, 4000) <= 8 * operand or size(rows, 4000) == few
    assert size(600, 4000) > few and size(2_000_000, 1000) == few


def test_matrix_kept_without_its_longest_row():
    """A matrix that a program has pickled holds the statistics of its rows, not what later versions read off them."""
    import pickle
    csr = _stand_in()
    csr._stats = (300, 1, 303, 7, 7, 7, 7, 0)
    assert "longest_row" not in pickle.loads(pickle.dumps(csr)).__dict__
    assert pickle.loads(pickle.dumps(csr)).longest_row == 303
