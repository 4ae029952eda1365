"""GPU parity tests of the locality plan and the window kernels (chunks of the residue
list whose dense rows fit an LDS window): the planned entry points against the fp64 oracle
and against the same call without a plan, through the Python op (ctypes over the C ABI)."""
import numpy as np
import pytest
import torch

import oracle
from gpu_common import DEV, TOL_F16, TOL_F32, round_half, t
from rode_amd import RoDeCSR, rode_sddmm, rode_sddmm_hip, rode_spmm, workloads

pytestmark = pytest.mark.gpu


def banded(rows, cols, per_row, band, seed, far=0, long_every=0, long_len=0, empty_every=0):
    """Rows with `per_row` distinct columns inside a band around the diagonal, `far` more
    anywhere (outside the window), every `long_every`-th row `long_len` columns long (it gets
    block segments and a tail), every `empty_every`-th row empty."""
    rng = np.random.default_rng(seed)
    cols_of = []
    for r in range(rows):
        if empty_every and r % empty_every == empty_every - 1:
            cols_of.append(np.empty(0, dtype=np.int64))
            continue
        want = long_len if long_every and r % long_every == 0 else per_row
        centre = int(r * (cols - 1) / max(rows - 1, 1))
        lo, hi = max(0, centre - band // 2), min(cols, centre + band // 2)
        pick = rng.choice(np.arange(lo, hi), size=min(want, hi - lo), replace=False)
        if far:
            pick = np.concatenate([pick, rng.integers(0, cols, far)])
        cols_of.append(np.unique(pick))
    lens = np.array([len(c) for c in cols_of])
    row_ptr = np.zeros(rows + 1, dtype=np.int32)
    row_ptr[1:] = np.cumsum(lens)
    col = np.concatenate(cols_of).astype(np.int32)
    val = rng.uniform(-1, 1, len(col)).astype(np.float32)
    return row_ptr, col, val


def both(row_ptr, col, val, m, n, k):
    planned = RoDeCSR(t(row_ptr), t(col), t(val), DEV, m, n, k, locality=True)
    plain = RoDeCSR(t(row_ptr), t(col), t(val), DEV, m, n, k, locality=False)
    return planned, plain


def check_products(row_ptr, col, val, m, n, k, half=False, expect_plan=True):
    planned, plain = both(row_ptr, col, val, m, n, k)
    assert (planned.plan is not None) == expect_plan
    assert plain.plan is None
    rng = np.random.default_rng(17)
    B = rng.standard_normal((n, k)).astype(np.float32)
    L = rng.standard_normal((m, k)).astype(np.float32)
    dt = torch.float16 if half else torch.float32
    Bd, Ld = t(B).to(DEV, dt), t(L).to(DEV, dt)
    if half:
        B, L = round_half(B), round_half(L)
    tol = TOL_F16 if half else TOL_F32
    c64 = oracle.spmm_f64(row_ptr, col, val, B)
    l1 = np.maximum(np.abs(c64).sum(axis=1), 1e-30)
    o64, scale = oracle.sddmm_f64(row_ptr, col, val, L, B, with_abs=True)
    for csr in (planned, plain):
        C = rode_spmm(csr, Bd).cpu().numpy()
        assert np.max(np.abs(C - c64).max(axis=1) / l1) <= tol
        out = rode_sddmm(csr, Ld, Bd).cpu().numpy()
        # per element against the magnitude of the summed terms (strict for any row)
        assert np.max(np.abs(out - o64) / np.maximum(scale, 1e-30)) <= (2e-3 if half else 2e-6)
    return planned


def test_plan_of_a_banded_matrix_has_a_window_on_every_chunk():
    m, n, rp, col, val = workloads.config("c3_banded", 0.01)
    csr = RoDeCSR(t(rp), t(col), t(val), DEV, m, n, 128, locality=True)
    assert csr.m1 == 0 and csr.plan is not None
    d = csr.plan.descriptors()
    assert len(d) == (csr.m2 + 127) // 128 == csr.plan.counts[0] == csr.plan.counts[1]
    assert (d[:, 1] > 0).all() and (d[:, 1] <= 512).all()
    assert (d[:, 3] == 0).all()                            # every nonzero inside its chunk's window
    assert int(d[:, 2].sum()) == int(rp[-1])               # the residue list holds every nonzero here
    rows = np.arange(len(d)) * 128
    assert (d[:, 0] <= rows + 128).all() and (d[:, 0] + d[:, 1] >= rows - 128).all()  # windows follow the diagonal
    assert (d[:, 0] >= 0).all() and (d[:, 0] + d[:, 1] <= n).all()


def test_plan_of_scattered_columns_has_no_window():
    m, n, rp, col, val = workloads.config("c2_lognormal", 0.1)
    assert RoDeCSR(t(rp), t(col), t(val), DEV, m, n, 128, locality=True).plan is None
    # "auto" also drops a plan that covers too few chunks to be worth two more launches
    m, n, rp, col, val = workloads.config("c3_banded", 0.01)
    assert RoDeCSR(t(rp), t(col), t(val), DEV, m, n, 128).plan is None


@pytest.mark.parametrize("k,half", [(128, False), (64, False), (256, False), (200, False), (36, False), (128, True),
                                    (72, True), (32, False)])
def test_banded_matrix_planned_against_oracle(k, half):
    # 36 and 200: partial last tile; 32 fp32 / 64 fp16 and narrower: one tile, the plan is ignored by the kernels
    m, n, rp, col, val = workloads.config("c3_banded", 0.004)
    check_products(rp, col, val, m, n, k, half)


def test_rows_with_segments_tails_far_columns_and_empty_rows():
    # long rows (block segments + tails in the residue list, summed whole by the block kernel
    # under the whole-lists promise when there are many segments), columns outside the window,
    # empty rows with an unaligned start, a last chunk that is not full
    m = n = 3000
    rp, col, val = banded(m, n, 21, 200, seed=5, far=2, long_every=97, long_len=150, empty_every=13)
    csr = check_products(rp, col, val, m, n, 128)
    d = csr.plan.descriptors()
    win = d[d[:, 1] > 0]
    assert len(win) > 0 and (win[:, 3] > 0).any()           # some slots are outside their window
    check_products(rp, col, val, m, n, 64, half=False)
    check_products(rp, col, val, m, n, 128, half=True)


def test_window_clipped_at_the_matrix_edges_and_rectangular_operand():
    m, n = 2000, 700  # the band runs from column 0 to column n - 1
    rp, col, val = banded(m, n, 17, 300, seed=9)
    check_products(rp, col, val, m, n, 128)


def test_non_finite_dense_rows_stay_in_the_rows_that_reference_them():
    m = n = 1500
    rp, col, val = banded(m, n, 15, 120, seed=3, far=1)
    planned, plain = both(rp, col, val, m, n, 128)
    assert planned.plan is not None
    B = torch.randn(n, 128, device=DEV)
    bad = [0, 7, 640, n - 1]
    B[bad] = float("inf")
    touched = np.zeros(m, dtype=bool)
    rows = np.repeat(np.arange(m), np.diff(rp))
    touched[rows[np.isin(col, bad)]] = True
    for csr in (planned, plain):
        C = rode_spmm(csr, B).cpu().numpy()
        assert np.isfinite(C[~touched]).all()
        assert (~np.isfinite(C[touched])).any(axis=1).all()


def test_values_replaced_per_call_and_gradients_use_the_plan():
    m = n = 2048
    rp, col, val = banded(m, n, 19, 160, seed=11)
    planned, plain = both(rp, col, val, m, n, 64)
    assert planned.plan is not None and planned.with_values(planned.values * 2).plan is planned.plan
    L = torch.randn(m, 64, device=DEV, requires_grad=True)
    R = torch.randn(n, 64, device=DEV, requires_grad=True)
    outs = []
    for csr in (planned, plain):
        L.grad = R.grad = None
        s = rode_sddmm(csr, L, R)
        C = rode_spmm(csr, R, values=s)
        C.square().sum().backward()
        outs.append((s.detach().clone(), C.detach().clone(), L.grad.clone(), R.grad.clone()))
    for a, b in zip(*outs):
        assert torch.allclose(a, b, rtol=2e-4, atol=2e-4 * float(b.abs().max()))


def test_full_size_banded_configuration_planned():
    # configuration 3 at full size, K = 128: linearity and a row sample against the oracle
    m, n, rp, col, val = workloads.config("c3_banded", 1.0)
    csr = RoDeCSR(t(rp), t(col), t(val), DEV, m, n, 128)
    assert csr.plan is not None and csr.plan.counts[0] == csr.plan.counts[1]
    rng = np.random.default_rng(23)
    B = rng.standard_normal((n, 128)).astype(np.float32)
    L = rng.standard_normal((m, 128)).astype(np.float32)
    Bd, Ld = t(B).to(DEV), t(L).to(DEV)
    C = rode_spmm(csr, Bd)
    out = rode_sddmm(csr, Ld, Bd)
    sample = np.unique(np.concatenate([np.arange(0, 300), rng.integers(0, m, 400), np.arange(m - 300, m)]))
    idx = np.concatenate([np.arange(rp[r], rp[r + 1]) for r in sample])
    srp = np.zeros(len(sample) + 1, dtype=np.int32)
    srp[1:] = np.cumsum(rp[sample + 1] - rp[sample])
    c64 = oracle.spmm_f64(srp, col[idx], val[idx], B)
    l1 = np.maximum(np.abs(c64).sum(axis=1), 1e-30)
    assert np.max(np.abs(C[sample].cpu().numpy() - c64).max(axis=1) / l1) <= TOL_F32
    o64, scale = oracle.sddmm_f64(srp, col[idx], val[idx], L[sample], B, with_abs=True)
    assert np.max(np.abs(out.cpu().numpy()[idx] - o64) / np.maximum(scale, 1e-30)) <= 2e-6
    # linearity in the dense operand (exact property at any size)
    C2 = rode_spmm(csr, 2 * Bd)
    assert torch.equal(C2, 2 * C)


@pytest.mark.parametrize("width", [4_194_304, 6_300_008])  # (rows of 8 MiB, the widest the window kernel takes, and of 12.6 MB)
def test_very_wide_operand(width):
    """Windows of more than 4 GiB of dense rows: halves, 450 rows."""
    m, n = 128, 450
    rng = np.random.default_rng(11)
    col = np.concatenate([np.sort(rng.choice(n, 27, replace=False)) for _ in range(m)]).astype(np.int32)
    row_ptr = np.arange(0, 27 * m + 1, 27, dtype=np.int32)
    val = rng.uniform(-1, 1, len(col)).astype(np.float32)
    csr = RoDeCSR(t(row_ptr), t(col), t(val), DEV, m, n, 128, locality=True)
    assert csr.plan is not None and csr.plan.windowed == 1
    gen = torch.Generator(device=DEV).manual_seed(2)
    B = torch.randn(n, width, device=DEV, generator=gen, dtype=torch.float16)
    C = rode_spmm(csr, B)
    dense = torch.zeros(m, n, dtype=torch.float64, device=DEV)
    dense[torch.arange(m, device=DEV).repeat_interleave(27), csr.column_indices.long()] = csr.values.double()
    for at in (0, 8 * rng.integers(width // 8), width - 64):
        want = dense @ B[:, at:at + 64].double()
        assert (C[:, at:at + 64].double() - want).abs().max() <= 1e-5 * want.abs().max()


@pytest.mark.parametrize("per_row,chunks", [(9, 513), (14, 640), (27, 513)])
@pytest.mark.parametrize("k,dtype", [(128, torch.float32), (64, torch.float32), (128, torch.float16), (32, torch.float64)])
def test_calls_that_may_leave_the_plan_unused(per_row, chunks, k, dtype):
    """"auto" uses a plan where it pays, locality=True always: the same products, within the rounding of their order."""
    m = 128 * chunks - 5
    gen = torch.Generator(device=DEV).manual_seed(per_row)
    row = torch.arange(m, device=DEV)
    pick = torch.rand(m, 128, device=DEV, generator=gen).argsort(1)[:, :per_row].sort(1)[0]
    col = ((row - 64).clamp(0, m - 128)[:, None] + pick).flatten().int()
    ro, val = torch.arange(0, m * per_row + 1, per_row, dtype=torch.int32), torch.rand(m * per_row, device=DEV, generator=gen) - 0.5
    auto, always = (RoDeCSR(ro, col, val, DEV, m, m, k, locality=how) for how in ("auto", True))
    assert auto.plan.windowed == always.plan.windowed == chunks and auto.plan.nonzeros == auto.nnz and always.plan.nonzeros == 0
    B, L = (torch.randn(m, k, device=DEV, generator=gen).to(dtype) for _ in range(2))
    if dtype == torch.float64:
        a, b = (rode_sddmm_hip.spmm_forward(c.block_indices, c.residue_indices, c.st_offsets, c.m1, c.m2, c.row_offsets, c.column_indices,
                                            c.values.double(), m, m, B, plan=c.plan) for c in (auto, always))
        assert (a - b).abs().max() <= 1e-14 * b.abs().max()
        return
    for op in (lambda c: rode_spmm(c, B), lambda c: rode_sddmm(c, L, B)):
        a, b = op(auto), op(always)
        assert (a - b).abs().max() <= 2e-6 * b.abs().max()


@pytest.mark.parametrize("k,half", [(64, False), (128, False), (128, True)])
def test_sddmm_in_windows_is_as_exact_as_without(k, half):
    """2-norms of the errors against fp64. Of 442 368 products each is known to 1 / sqrt(2 * 442 368) = 0.1 %; a sum per tile of eight
    chunks rounds like the standard kernels' (0.05 to 1.8 % more), one chain over two or four tiles had 5 and 17 % more: the bound is 3 %."""
    m = 16384
    gen = torch.Generator(device=DEV).manual_seed(k)
    col = ((torch.arange(m, device=DEV) - 64).clamp(0, m - 128)[:, None] + torch.rand(m, 128, device=DEV, generator=gen).argsort(1)[:, :27].sort(1)[0])
    ro, val = torch.arange(0, 27 * m + 1, 27, dtype=torch.int32), torch.rand(27 * m, device=DEV, generator=gen) + 0.5
    L, B = (torch.randn(m, k, device=DEV, generator=gen).to(torch.float16 if half else torch.float32) for _ in range(2))
    want = val.double() * (L.double()[:, None] * B.double()[col]).sum(2).flatten()
    errors = []
    for how in (True, False):
        csr = RoDeCSR(ro, col.flatten().int(), val, DEV, m, m, k, locality=how)
        assert (csr.plan is not None) == how
        errors.append(((rode_sddmm(csr, L, B).double() - want).norm() / want.norm()).item())
    assert 0 < errors[0] <= 1.03 * errors[1]


def _strips(m, degree, seed):
    """Columns of m rows, `degree` ascending ones each: by chunks of 128 rows along the diagonal, some of them apart from their neighbours, before
    them, two columns further per row (windows of up to 511), without a window, and a column outside the window here and there."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    row = torch.arange(m, device=DEV)
    chunk, local = row // 128, row % 128
    kind = chunk % 11
    base = row - 100
    base = torch.where(kind == 4, base - 250, base)
    base = torch.where(kind == 6, (row + m // 2) % m, base)
    base = torch.where(kind == 8, chunk * 128 - 60 + 2 * local, base)
    base = base.clamp(0, m - 256)
    pick = torch.rand(m, 256, device=DEV, generator=gen).argsort(1)[:, :degree]
    col = base[:, None] + pick
    col[kind == 7] = torch.randint(0, m, (int((kind == 7).sum()), degree), device=DEV, generator=gen)
    far = (row % 50 == 3) & (kind != 7)
    col[far, 0] = torch.randint(0, m, (int(far.sum()),), device=DEV, generator=gen)
    return col.sort(1)[0]


@pytest.mark.parametrize("m", [128 * 2560 + 40, 128 * 700 - 3, 128 * 3])  # ten chunks a workgroup (the ring begins again several times), two or three, one at most
@pytest.mark.parametrize("dtype,k", [(torch.float32, 32), (torch.float32, 64), (torch.float32, 128), (torch.float32, 256), (torch.float16, 64),
                                     (torch.float16, 128), (torch.float16, 256), (torch.float64, 16), (torch.float64, 32), (torch.float64, 64)])
def test_rings_against_fp64(m, dtype, k):
    degree = 11
    col = _strips(m, degree, seed=k)
    gen = torch.Generator(device=DEV).manual_seed(k + 1)
    val = torch.rand(m * degree, device=DEV, generator=gen) + 0.5
    ro = torch.arange(0, m * degree + 1, degree, dtype=torch.int32)
    csr, plain = (RoDeCSR(ro, col.flatten().int(), val, DEV, m, m, k, locality=how) for how in (True, False))
    assert csr.plan is not None and csr.plan.windowed >= csr.plan.counts[0] * 3 // 4
    csr.plan.nonzeros = 31 * csr.m2  # (rows of 128 bytes want to know, and long rows to be worth it)
    B, L = (torch.randn(m, k, device=DEV, generator=gen, dtype=torch.float64).to(dtype) for _ in range(2))
    want = torch.zeros(m, k, device=DEV, dtype=torch.float64)
    for j in range(degree):
        want += val.view(m, degree)[:, j:j + 1].double() * B[col[:, j]].double()
    if dtype == torch.float64:
        got, other = (rode_sddmm_hip.spmm_forward(c.block_indices, c.residue_indices, c.st_offsets, c.m1, c.m2, c.row_offsets, c.column_indices,
                                                  c.values.double(), m, m, B, plan=c.plan) for c in (csr, plain))
        assert (got - want).abs().max() <= 1e-14 * want.abs().max()
        assert m < 128 * 2560 or not torch.equal(got, other)  # (a row's slots are added in the plan's order)
        return
    got, other = rode_spmm(csr, B), rode_spmm(plain, B)
    assert (got - want).abs().max() <= 2e-6 * want.abs().max()
    assert m < 128 * 2560 or not torch.equal(got, other)
    want = torch.stack([val.view(m, degree)[:, j].double() * (L.double() * B[col[:, j]].double()).sum(1) for j in range(degree)], 1).flatten()
    assert (rode_sddmm(csr, L, B) - want).abs().max() <= 2e-6 * want.abs().max()


@pytest.mark.parametrize("dtype,k", [(torch.float32, 32), (torch.float32, 64), (torch.float32, 128), (torch.float32, 48), (torch.float16, 64),
                                     (torch.float16, 128), (torch.float64, 16), (torch.float64, 32), (torch.float64, 20)])
def test_rows_with_no_column_in_their_window_are_not_reached_by_it(dtype, k):
    """Rows of 1 to 9 columns, none of them in their chunk's window, among rows of 21 that are: the positions that such a row does not fill
    are not to read a row of the window (the first one is infinite).  Rings and, for the other widths, windows."""
    one_line = k * torch.finfo(dtype).bits == 128 * 8  # (rows of 128 bytes take a plan only where it pays)
    m = 128 * (2560 if one_line else 12)
    gen = torch.Generator(device=DEV).manual_seed(k)
    row = torch.arange(m, device=DEV)
    lens = torch.where(row % 5 == 2, 1 + row // 5 % 9, 21)
    low = (row - 60).clamp(0, m - 120)
    low = torch.where(lens < 21, (low + m // 2) % (m - 120), low)
    col = low[:, None] + torch.rand(m, 120, device=DEV, generator=gen).argsort(1)[:, :21]
    col = torch.where(torch.arange(21, device=DEV) < lens[:, None], col, m).sort(1)[0]
    col = col[col < m].int()
    ro = torch.cat((torch.zeros(1, dtype=torch.int64, device=DEV), lens.cumsum(0))).int().cpu()
    csr = RoDeCSR(ro, col, torch.rand(col.numel(), device=DEV, generator=gen) + 0.5, DEV, m, m, k, locality=True)
    assert csr.plan is not None and csr.plan.windowed == csr.plan.counts[0] == m // 128
    csr.plan.nonzeros = 31 * csr.m2 if one_line else 0
    bad = torch.from_numpy(np.unique(csr.plan.descriptors()[:, 0])).to(DEV)
    B = torch.randn(m, k, device=DEV, dtype=torch.float64, generator=gen).to(dtype)
    B[bad.long()] = float("inf")
    if dtype == torch.float64:
        C = rode_sddmm_hip.spmm_forward(csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2, csr.row_offsets, csr.column_indices,
                                        csr.values.double(), m, m, B, plan=csr.plan)
    else:
        C = rode_spmm(csr, B)
    finite = torch.isfinite(C).all(1)
    touched = torch.zeros(m, dtype=torch.bool, device=DEV)
    touched[row.repeat_interleave(lens)[torch.isin(col, bad)]] = True
    assert (~touched & (lens < 21)).sum() > 100
    assert finite[~touched].all() and not finite[touched].any()


def _some_banded(m, degree, banded, seed):
    """`degree` ascending columns a row: of the 192 around the diagonal where `banded` (of every chunk of 128 rows) says so, else anywhere."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    row = torch.arange(m, device=DEV)
    near = (row - 96).clamp(0, m - 192)[:, None] + torch.rand(m, 192, device=DEV, generator=gen).argsort(1)[:, :degree]
    far = (torch.rand(m, degree, device=DEV, generator=gen) * (m // degree)).long() + torch.arange(degree, device=DEV) * (m // degree)
    col = torch.where(banded.to(DEV)[row // 128, None], near, far).sort(1)[0]
    ro = torch.arange(0, m * degree + 1, degree, dtype=torch.int32)
    return ro, col, torch.rand(m * degree, device=DEV, generator=gen) + 0.5


@pytest.mark.parametrize("dtype,k", [(torch.float32, 64), (torch.float32, 128), (torch.float16, 128), (torch.float64, 64)])
@pytest.mark.parametrize("kind", ["one run", "short runs", "few", "all but few"])
def test_rings_where_chunks_with_a_window_lie_together(kind, dtype, k):
    """1400 chunks, 175 of an XCD's share, dealt out to 32, 16 or 8 strips by their windows: all in three shares, in runs of 5 and 90 with 90 and 5 between,
    seven in all, all but seven."""
    chunks, degree = 1400, 9
    c = torch.arange(chunks)
    banded = {"one run": (c > 300) & (c < 777), "short runs": (c % 95 < 5) ^ (c > 700), "few": c % 200 == 150, "all but few": c % 200 != 150}[kind]
    m = 128 * chunks - 3
    ro, col, val = _some_banded(m, degree, banded, seed=k)
    csr = RoDeCSR(ro, col.flatten().int(), val, DEV, m, m, k, locality=True)
    assert csr.plan.windowed == int(banded.sum()) and csr.plan.nonzeros == 0
    gen = torch.Generator(device=DEV).manual_seed(k)
    B, L = (torch.randn(m, k, device=DEV, generator=gen, dtype=torch.float64).to(dtype) for _ in range(2))
    want = torch.zeros(m, k, device=DEV, dtype=torch.float64)
    for j in range(degree):
        want += val.view(m, degree)[:, j:j + 1].double() * B[col[:, j]].double()
    if dtype == torch.float64:
        got = rode_sddmm_hip.spmm_forward(csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2, csr.row_offsets, csr.column_indices,
                                          val.double(), m, m, B, plan=csr.plan)
        assert (got - want).abs().max() <= 1e-14 * want.abs().max()
        return
    assert (rode_spmm(csr, B) - want).abs().max() <= 2e-6 * want.abs().max()
    want = torch.stack([val.view(m, degree)[:, j].double() * (L.double() * B[col[:, j]].double()).sum(1) for j in range(degree)], 1).flatten()
    assert (rode_sddmm(csr, L, B) - want).abs().max() <= 2e-6 * want.abs().max()


def test_chunks_without_a_window_and_what_pays():
    """Six chunks in ten with a window, rows of 128 bytes: the standard kernels take all (they took 243 us for a million such rows, and 328 with the
    others by themselves). 704 chunks with one, SDDMM of 256-byte rows: too few for rings, but not for windows (21.4 us, standard kernels 30)."""
    m = 128 * 7813
    ro, col, val = _some_banded(m, 27, torch.arange(7813) % 10 < 6, seed=1)
    csr, plain = (RoDeCSR(ro, col.flatten().int(), val, DEV, m, m, 32, locality=how) for how in ("auto", False))
    assert csr.plan is not None and csr.plan.windowed * 10 <= 7 * csr.plan.counts[0]
    B, L = (torch.randn(m, 32, device=DEV) for _ in range(2))
    assert torch.equal(rode_spmm(csr, B), rode_spmm(plain, B)) and torch.equal(rode_sddmm(csr, L, B), rode_sddmm(plain, L, B))
    m = 128 * 704
    ro, col, val = _some_banded(m, 20, torch.ones(704, dtype=torch.bool), seed=2)
    csr, plain = (RoDeCSR(ro, col.flatten().int(), val, DEV, m, m, 64, locality=how) for how in ("auto", False))
    B, L = (torch.randn(m, 64, device=DEV) for _ in range(2))
    got, other = rode_sddmm(csr, L, B), rode_sddmm(plain, L, B)
    assert not torch.equal(got, other) and (got - other).abs().max() <= 2e-6 * other.abs().max()
