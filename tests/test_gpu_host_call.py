"""The native host calls behind rode_sddmm and rode_spmm: the same results as the module's functions, and everything
that is not the ordinary call still reaches the Python layer."""
import threading

import numpy as np
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from rode_amd import RoDeCSR, _lib, rode_sddmm, rode_sddmm_hip, rode_spmm, sparse_attention

pytestmark = pytest.mark.gpu


def _matrix(m, n, k, seed=0):
    rng = np.random.default_rng(seed)
    lens = np.minimum(rng.integers(0, 70, size=m), n)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, size=v, replace=False)) for v in lens] + [np.zeros(0)]).astype(np.int32)
    return RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col), torch.from_numpy(rng.standard_normal(len(col)).astype(np.float32)),
                   "cuda", m, n, k)


@pytest.mark.parametrize("m,n,k,half", [(1, 40, 32, False), (257, 300, 64, True), (1000, 77, 20, False)])
def test_native_call_equals_the_module_functions(m, n, k, half):
    a = _matrix(m, n, k)
    kind = torch.float16 if half else torch.float32
    lhs, rhs = torch.randn(m, k, device="cuda").to(kind), torch.randn(n, k, device="cuda").to(kind)
    if k % (8 if half else 4) == 0:
        args = (a.block_indices, a.residue_indices, a.st_offsets, a.m1, a.m2, a.row_offsets, a.column_indices, a.values, a.m, a.n)
        got = _lib.host_call().sddmm(*args, k, lhs, rhs, a.plans_address(), rode_sddmm_hip._stream_handle(a.device))
        want = rode_sddmm_hip.sddmm_forward(*args, lhs, rhs, k, plan=a.plan)
        assert got is not None and torch.equal(got, want) and torch.equal(rode_sddmm(a, lhs, rhs), want)
        got, want = rode_spmm(a, rhs), rode_sddmm_hip.spmm_forward(*args, rhs, plan=a.plan)
        torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-5)


def test_other_calls_reach_the_python_layer():
    a = _matrix(64, 50, 32)
    lhs, rhs = torch.randn(64, 32, device="cuda"), torch.randn(50, 32, device="cuda")
    want = rode_sddmm(a, lhs, rhs)
    torch.testing.assert_close(rode_sddmm(a, lhs.t().contiguous().t(), rhs), want)  # not contiguous
    assert rode_sddmm(a, lhs.clone().requires_grad_(), rhs).grad_fn is not None
    assert rode_spmm(a, rhs.clone().requires_grad_()).grad_fn is not None
    with torch.no_grad():
        assert rode_spmm(a, rhs.clone().requires_grad_()).grad_fn is None
    with pytest.raises(ValueError, match="lhs_matrix shape"):
        rode_sddmm(a, rhs, lhs)
    with pytest.raises(AssertionError, match="must be on"):
        rode_sddmm(a, lhs.cpu(), rhs)
    with pytest.raises(AssertionError, match="rhs must be"):
        rode_sddmm(a, lhs, rhs.half())
    with pytest.raises(ValueError, match="dense width"):
        rode_spmm(a, torch.randn(50, 30, device="cuda"))
    with pytest.raises(ValueError, match="dense shape"):
        rode_spmm(a, torch.randn(50, device="cuda"))
    torch.testing.assert_close(rode_sddmm(a.with_values(2 * a.values), lhs, rhs), 2 * want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = rode_sddmm(a, lhs, rhs)
    side.synchronize()
    assert torch.equal(got, want)


@pytest.mark.parametrize("op", ["sddmm", "spmm", "attention"])
@pytest.mark.parametrize("kind", ["fake", "vmap", "jvp", "sparse", "subclass", "fake mode", "other dtype"])
@pytest.mark.filterwarnings("ignore:Accessing the data pointer of FakeTensor", "ignore:Sparse CSR tensor support")
def test_operands_that_are_no_plain_tensors(op, kind):
    """Refused with an exception (or, a mere subclass, taken): none ends in an abort or reaches a kernel without memory."""
    a = _matrix(64, 64, 32)
    x, y = torch.randn(64, 32, device="cuda"), torch.randn(64, 32, device="cuda")

    def call(t):
        if op == "sddmm":
            return rode_sddmm(a, x, t)
        return rode_spmm(a, t) if op == "spmm" else sparse_attention(a, x, x, t)

    want = call(y)
    if kind == "subclass":
        assert torch.equal(torch.Tensor(call(y.as_subclass(type("Subclass", (torch.Tensor,), {})))), want)
        return
    with pytest.raises((RuntimeError, AssertionError, ValueError)):
        if kind == "fake":
            call(FakeTensorMode().from_tensor(y))
        elif kind == "vmap":
            torch.vmap(call)(y.expand(2, 64, 32))
        elif kind == "jvp":
            torch.func.jvp(call, (y,), (y,))
        elif kind == "sparse":
            call(y.to_sparse_csr())
        elif kind == "fake mode":
            with FakeTensorMode(allow_non_fake_inputs=True):
                call(y)
        else:
            call(y.to(torch.complex64))
    assert torch.equal(call(y), want)


def test_two_threads_make_the_first_calls():
    x, y = torch.randn(300, 32, device="cuda"), torch.randn(300, 32, device="cuda")
    want = rode_sddmm(_matrix(300, 300, 32), x, y)
    for _ in range(20):
        a, start, got = _matrix(300, 300, 32), threading.Barrier(2), [None, None]

        def work(i):
            start.wait()
            got[i] = [rode_sddmm(a, x, y) for _ in range(3)]

        threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        assert all(torch.equal(g, want) for thread in got for g in thread)


class _Refuse(TorchDispatchMode):
    """The `at`-th tensor operation fails, as an allocation without memory does."""

    def __init__(self, at):
        super().__init__()
        self.left = at

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.left -= 1
        if self.left == 0:
            raise MemoryError("refused")
        return func(*args, **(kwargs or {}))


def test_decomposition_without_memory_leaves_nothing_running():
    m = 1_000_000  # (rows of 40: both lists have entries)
    ro = torch.arange(m + 1, dtype=torch.int32) * 40
    on_gpu, col = ro.cuda(), torch.arange(40 * m, dtype=torch.int32, device="cuda") // 40
    args = (ro, on_gpu, col, m, 512, rode_sddmm_hip._stream_handle(on_gpu.device))
    want = _lib.host_call().decompose(*args)
    assert want[5] is not None  # (with a plan)
    refused = 0
    while True:
        torch.cuda.synchronize()
        mode = _Refuse(refused + 1)
        with mode:
            try:
                got = _lib.host_call().decompose(*args)
            except MemoryError:
                refused += 1
                assert torch.cuda.current_stream().query()
                continue
        break
    assert refused >= 6 and mode.left == 1  # the lists, the scratch, the plan and the counts
    for a, b in zip(got, want):
        assert torch.equal(a, b) if isinstance(a, torch.Tensor) else a == b


def test_decomposition_of_sent_offsets_without_memory_leaves_nothing_running():
    """As `RoDeCSR` calls it: a copy of the offsets is on its way whatever fails."""
    m = 1_000_000  # (rows of 40: both lists have entries)
    ro = torch.arange(m + 1, dtype=torch.int32) * 40
    col = torch.arange(40 * m, dtype=torch.int32, device="cuda") // 40
    stream = rode_sddmm_hip._stream_handle(col.device)
    refused, results = 0, []
    while len(results) < 2:
        on_gpu = torch.full((m + 1,), -1, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        _lib.host_call().send_offsets(ro, on_gpu, 8, stream)
        mode = _Refuse(refused + 1 if not results else -1)
        with mode:
            try:
                results.append(_lib.host_call().decompose(ro, on_gpu, col, m, 512, stream, None))
            except MemoryError:
                refused += 1
                assert torch.cuda.current_stream().query()
        assert torch.equal(on_gpu.cpu(), ro)
    assert refused >= 5 and results[1][5] is not None  # the lists, the plan and the counts
    for a, b in zip(*results):
        assert torch.equal(a, b) if isinstance(a, torch.Tensor) else a == b


@pytest.mark.parametrize("upload", [False, True])
@pytest.mark.parametrize("m,n", [(1, 600), (127, 600), (128, 600), (129, 600), (33000, 33000)])
def test_decomposition_with_a_plan_equals_its_parts(m, n, upload):
    """The lists and the plan that one call makes (counts written by the last workgroup) against the separate entries,
    and the plan's numbers against a count of the columns inside each window.  Rows of at most 28 (31 from their aligned start), so that all
    of their nonzeros are in the residue list; every third run of 128 rows has its columns anywhere."""
    rng = np.random.default_rng(m + 7 * upload)
    lens = rng.integers(1, 29, m)
    ro = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    row = np.repeat(np.arange(m), lens)
    near = np.clip(row * n // m + rng.integers(-90, 90, len(row)), 0, n - 1)
    col = np.where(row // 128 % 3 == 1, rng.integers(0, n, len(row)), near).astype(np.int32)
    host, cols = torch.from_numpy(ro), torch.from_numpy(col).cuda()
    on_gpu = torch.full((m + 1,), -1, dtype=torch.int32, device="cuda") if upload else host.cuda()
    args = (host, on_gpu, cols, n, 512, rode_sddmm_hip._stream_handle(cols.device))
    blk, st, res, m1, m2, data, counts = _lib.host_call().decompose(*args, *([True] if upload else []))
    assert torch.equal(on_gpu.cpu(), host)
    parts = rode_sddmm_hip.preprocess_device(on_gpu, int(ro[-1]), 512, 32, 4)
    assert (m1, m2) == tuple(parts[3:]) and all(torch.equal(a, b) for a, b in zip((st, res), parts[1:3]))
    plan = rode_sddmm_hip.window_plan(res, m2, on_gpu, cols, n)
    assert counts == plan.counts and data[:4].tolist() == counts and torch.equal(data[4:4 + 4 * counts[0]], plan.data[4:4 + 4 * counts[0]])
    listed = data[4:4 + 4 * counts[0]].view(-1, 4).tolist()
    assert counts[0] == (m2 + 127) // 128 and counts[1] == sum(d[1] > 0 for d in listed)
    rows = res[:m2].cpu().numpy()
    for chunk, (first, count, slots, misses) in enumerate(listed):
        c = np.concatenate([col[ro[r]:ro[r + 1]] for r in rows[128 * chunk:128 * chunk + 128]])
        assert slots == len(c) and (count == 0 or misses == np.sum((c < first) | (c >= first + count)))
    assert m < 128 or counts[1] > 0
