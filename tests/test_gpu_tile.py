"""Attention on the tiles of 16 rows (matrix cores) against fp64 on dense matrices."""
import ctypes

import numpy as np
import pytest
import torch

from rode_amd import RoDeCSR, _lib, sparse_attention
from rode_amd.autograd import _attention_backward_call, _attention_call

pytestmark = pytest.mark.gpu


def _mask(m, window, shift, extra, seed, short_rows=()):
    """Row r has the run [shift * r, shift * r + window) and `extra` random columns; short_rows keep three columns only
    (their tiles are none)."""
    rng = np.random.default_rng(seed)
    n = shift * m + window + 40
    rows = []
    for r in range(m):
        c = np.union1d(np.arange(shift * r, shift * r + window), rng.choice(n, extra, replace=False))
        rows.append(np.sort(rng.choice(c, 3, replace=False)) if r in short_rows else c)
    rp = np.concatenate([[0], np.cumsum([len(c) for c in rows])]).astype(np.int32)
    col = np.concatenate(rows).astype(np.int32)
    val = rng.uniform(0.5, 1.5, len(col)).astype(np.float32)
    csr = RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col), torch.from_numpy(val), "cuda", m, n, 64, locality=True)
    dense = torch.zeros(m, n, dtype=torch.float64)
    dense[np.repeat(np.arange(m), np.diff(rp)), col] = torch.from_numpy(val.astype(np.float64))
    return csr, dense.cuda()


def _reference(dense, q, k, v, scale):
    s = (q.double() @ k.double().t()) * dense * scale
    return torch.softmax(s.masked_fill(dense == 0, float("-inf")), dim=1) @ v.double()


def _heads(csr):
    return -(-1500000 // csr.nnz)  # (fewer nonzeros over all heads take other kernels)


CASES = [  # m, window, columns the window moves per row, random columns, width, half, scale
    (16, 64, 0, 0, 64, False, 0.3),      # one tile, nothing outside the run, whole steps only
    (75, 69, 1, 5, 64, True, 0.3),       # rows after the last tile, a cut-short last step
    (160, 260, 3, 70, 64, False, -0.3),  # more than 64 nonzeros outside a run, a negative scale
    (160, 260, 3, 70, 64, True, -0.3),
    (48, 97, 2, 20, 128, True, 0.2),
    (48, 97, 2, 20, 128, False, 0.2),
    (48, 130, 1, 16, 32, True, 0.4),
    (48, 130, 1, 16, 32, False, 0.4),
    (48, 400, 2, 130, 128, False, 0.1),  # three times 64 outside a run
    (48, 400, 2, 130, 32, True, 0.2),
]


@pytest.mark.parametrize("m,window,shift,extra,d,half,scale", CASES)
def test_tiles_against_fp64(m, window, shift, extra, d, half, scale):
    csr, dense = _mask(m, window, shift, extra, seed=m + window, short_rows=(40,) if m == 160 else ())
    assert csr.plan.counts[3] == m // 16 - (1 if m == 160 else 0)
    dt = torch.float16 if half else torch.float32
    g = torch.Generator(device="cuda").manual_seed(d)
    heads = _heads(csr)
    q, k, v = (torch.randn(r, d, device="cuda", generator=g).to(dt).expand(heads, r, d).contiguous() for r in (m, csr.n, csr.n))
    outs, all_scores, all_stats = _attention_call(csr, csr.values, q, k, v, scale, "scores")
    assert torch.equal(outs, sparse_attention(csr, q, k, v, scale=scale)) and torch.equal(outs, outs[:1].expand_as(outs))
    outs_p, all_probs, _ = _attention_call(csr, csr.values, q, k, v, scale, "probs")
    assert torch.equal(outs, outs_p)
    q, k, v, out, scores, stats, probs = (t[heads - 1] for t in (q, k, v, outs, all_scores, all_stats, all_probs))
    want = _reference(dense, q, k, v, scale)
    assert (out.double() - want).abs().max() <= 2e-5 * want.abs().max()
    rows = torch.repeat_interleave(torch.arange(m, device="cuda"), (csr.row_offsets[1:] - csr.row_offsets[:-1]).long())
    s = ((q.double() @ k.double().t()) * dense * scale)[rows, csr.column_indices.long()]
    assert (scores.double() - s).abs().max() <= 2e-5 * s.abs().max()
    assert (probs - torch.exp(scores - stats[rows, 0]) * stats[rows, 1]).abs().max() <= 2e-6


def _without_tiles(csr):
    """The same matrix whose plan says that it has no tiles: its groups go to the kernels for groups and rows."""
    args = [csr.row_offsets_cpu, csr.column_indices, csr.values, "cuda", csr.m, csr.n, 64]
    other = RoDeCSR(*args, locality=True)
    other.plan.counts[3] = other.plan._header[3] = 0
    return other


@pytest.mark.parametrize("sharp", [1.0, 8.0])
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_tiles_are_as_exact_as_the_other_kernels(d, half, sharp):
    """Errors against fp64 (2-norms), of the output and the gradients, not above those of the kernels on the vector ALUs.
    Both round every product and every sum once, in trees of the same depth; the 0.1 is for chance, in 65 K values and more."""
    m, scale, dt = 1024, sharp * d ** -0.5, torch.float16 if half else torch.float32
    csr, dense = _mask(m, 250, 1, 30, seed=d)
    assert csr.plan.counts[3] == m // 16
    heads = max(2, _heads(csr))
    gen = torch.Generator(device="cuda").manual_seed(d)
    q, k, v, g = (torch.randn(r, d, device="cuda", generator=gen) for r in (m, csr.n, csr.n, m))
    q, k, v = (t.to(dt) for t in (q, k, v))
    ins = [t.double().requires_grad_() for t in (q, k, v)]
    want = _reference(dense, *ins, scale)
    want = (want,) + torch.autograd.grad(want, ins, g.double())
    errors = []
    for c in (csr, _without_tiles(csr)):
        ins = [t.expand(heads, *t.shape).contiguous() for t in (q, k, v)]
        out, scores, stats = _attention_call(c, c.values, *ins, scale, "scores")
        got = (out,) + _attention_backward_call(c, c.transpose(with_values=False)[0], c.transposed_slots(), scores, stats,
                                                g.expand(heads, m, d).contiguous(), out, *ins, scale)
        errors.append([((a[0].double() - b).norm() / b.norm()).item() for a, b in zip(got, want)])
    print(*errors)
    for tiles, others in zip(*errors):
        assert 0 < tiles <= 1.1 * others


@pytest.mark.parametrize("half", [False, True])
def test_scores_without_range(half):
    """Infinite and largest scores, in a run and outside it, rows without a finite one: as on the other kernels."""
    m, d = 96, 64
    csr, dense = _mask(m, 100, 2, 30, seed=5)
    values = csr.values.clone()
    rows = torch.repeat_interleave(torch.arange(m, device="cuda"), (csr.row_offsets[1:] - csr.row_offsets[:-1]).long())
    inf, most = float("inf"), 0.9 * torch.finfo(torch.float32).max / 16  # (products of 16 below: log2(e) times the score has no range)
    for row, at, value in ((3, slice(None), -inf), (5, slice(0, 40), -inf), (20, slice(60, 61), most), (21, slice(60, 61), -most), (37, slice(7, 9), -16 * most),
                           (50, slice(129, 130), most), (52, slice(0, 1), most), (53, slice(0, 1), -inf), (70, slice(50, 51), inf)):
        picked = (rows == row).nonzero().flatten()
        values[picked[at]] = value
    csr = csr.with_values(values)
    csr._shared = {}
    other = RoDeCSR(csr.row_offsets_cpu, csr.column_indices, values, "cuda", m, csr.n, 64, locality=False)
    heads = _heads(csr)
    gen = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.rand(heads, r, d, device="cuda", generator=gen) for r in (m, csr.n, csr.n))
    q[:, [20, 21, 50, 52]] = 0.5
    k.fill_(0.5)
    if half:
        q, k, v = q.half(), k.half(), v.half()
    for scale in (0.125, 1.0):
        a, b = (_attention_call(c, c.values, q, k, v, scale, "scores") for c in (csr, other))
        assert not b[0][:, [3, 70]].isfinite().any() and b[0][:, [5, 20, 21, 37, 50, 52, 53]].isfinite().all()
        for x, y in zip(a, b):
            assert torch.equal(x.isnan(), y.isnan()) and torch.equal(x.isinf(), y.isinf())
            ok = y.isfinite()
            torch.testing.assert_close(x[ok], y[ok], rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("half", [False, True])
def test_non_finite_rows_of_v_stay_in_their_rows(half):
    """A column at either end of a tile's range is held by some of its rows only."""
    m, d = 96, 64
    csr, dense = _mask(m, 100, 2, 3, seed=5)
    assert csr.plan.counts[3] == m // 16
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn(r, d, device="cuda", generator=g) for r in (m, csr.n, csr.n))
    clean = _reference(dense, *((t.half() if half else t) for t in (q, k, v)), 0.2)
    bad = [1, 130, 2 * 47 + 99]
    v[bad] = float("inf")
    if half:
        q, k, v = q.half(), k.half(), v.half()
    out = sparse_attention(csr, *(t.expand(_heads(csr), *t.shape).contiguous() for t in (q, k, v)), scale=0.2)[63]
    touched = (dense[:, bad] != 0).any(dim=1)
    assert touched.any() and not touched.all()
    assert not torch.isfinite(out[touched]).all(dim=1).any()
    assert (out[~touched].double() - clean[~touched]).abs().max() <= 2e-5 * clean.abs().max()


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_every_head_has_operands_of_its_own(d, half):
    m, dt = 336, torch.float16 if half else torch.float32
    csr, dense = _mask(m, 300, 1, 40, seed=d, short_rows=(100,))
    assert csr.plan.counts[3] == m // 16 - 1
    heads, scale = _heads(csr), 0.2
    assert heads > 8
    gen = torch.Generator(device="cuda").manual_seed(d)
    q, k, v, g = (torch.randn(heads, r, d, device="cuda", generator=gen) for r in (m, csr.n, csr.n, m))
    ins = [t.to(dt).requires_grad_() for t in (q, k, v)]
    out = sparse_attention(csr, *ins, scale=scale)
    grads = torch.autograd.grad(out, ins, g)
    for h in (0, 1, heads // 2, heads - 1):
        one = [t[h].detach().double().requires_grad_() for t in ins]
        want = _reference(dense, *one, scale)
        assert (out[h].double() - want).abs().max() <= 2e-5 * want.abs().max()
        for a, b in zip(grads, torch.autograd.grad(want, one, g[h].double())):
            assert (a[h].double() - b).norm() <= (2e-3 if half else 1e-5) * b.norm()


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("scale", [0.0, -0.0, 1e-42])
def test_a_scale_of_zero_weighs_all_columns_alike(scale, half):
    m, d, dt = 48, 64, torch.float16 if half else torch.float32
    csr, dense = _mask(m, 97, 2, 20, seed=3)
    assert csr.plan.counts[3] == m // 16
    heads = _heads(csr)
    gen = torch.Generator(device="cuda").manual_seed(8)
    q, k, v, g = (torch.randn(r, d, device="cuda", generator=gen) for r in (m, csr.n, csr.n, m))
    ins = [t.to(dt).expand(heads, *t.shape).contiguous().requires_grad_() for t in (q, k, v)]
    out = sparse_attention(csr, *ins, scale=scale)
    grads = torch.autograd.grad(out, ins, g.expand(heads, m, d).contiguous())
    want = (dense != 0).double() @ v.to(dt).double() / (dense != 0).sum(1, keepdim=True)
    assert (out[heads - 1].double() - want).abs().max() <= 2e-5 * want.abs().max()
    mean = (dense != 0).double() / (dense != 0).sum(1, keepdim=True)
    want = mean.t().contiguous() @ g.double()
    assert (grads[2][heads - 1].double() - want).abs().max() <= (5e-3 if half else 1e-4) * want.abs().max()
    for t in grads[:2]:  # (their size is the scale's)
        assert t.abs().max() <= 1e-30


@pytest.mark.parametrize("m,window,shift,extra,d,half,scale", CASES)
def test_gradients_on_tiles_against_fp64(m, window, shift, extra, d, half, scale):
    csr, dense = _mask(m, window, shift, extra, seed=m + window, short_rows=(40,) if m == 160 else ())
    dt = torch.float16 if half else torch.float32
    gen = torch.Generator(device="cuda").manual_seed(d)
    heads = _heads(csr)
    q, k, v, g = (torch.randn(r, d, device="cuda", generator=gen) for r in (m, csr.n, csr.n, m))
    q, k, v = (t.to(dt) for t in (q, k, v))
    g[1] *= 1e-6  # (rows of very different gradients)
    ins = [t.double().requires_grad_() for t in (q, k, v)]
    want = torch.autograd.grad(_reference(dense, *ins, scale), ins, g.double())
    ins = [t.expand(heads, *t.shape).contiguous() for t in (q, k, v)]
    out, scores, stats = _attention_call(csr, csr.values, *ins, scale, "scores")
    got = _attention_backward_call(csr, csr.transpose(with_values=False)[0], csr.transposed_slots(), scores, stats,
                                   g.expand(heads, m, d).contiguous(), out, *ins, scale)
    of_g = g.double().abs().amax(1, keepdim=True)
    for a, b in zip(got, want):
        # (the kernels round g to halves for its products with halves: an error of g's size where one probability is nearly 1)
        size = b.abs().amax(1, keepdim=True) + (of_g if half and b is want[0] else 0.0) if b is want[0] else b.abs().max()
        assert ((a[heads - 1].double() - b).abs() / size).max() <= (5e-3 if half else 1e-4)


@pytest.mark.parametrize("half", [False, True])
def test_gradients_on_tiles_twice_held_column_and_inf(half):
    """A row that holds a column of its run twice (its slots in the transposed pattern are not the next row's), and a row of
    k that is not finite and that most rows of its tile do not hold: as without a plan."""
    m, d, dt = 256, 64, torch.float16 if half else torch.float32
    csr, _ = _mask(m, 130, 1, 12, seed=5)
    rp, col = csr.row_offsets.cpu().numpy(), csr.column_indices.cpu().numpy().copy()
    for row, at in ((21, 100), (40, 80)):  # the columns outside the run name one inside it
        c = col[rp[row]:rp[row + 1]]
        out = np.flatnonzero((c < row) | (c >= row + 130))
        c[out[0]] = row + at
    args = [torch.from_numpy(rp), torch.from_numpy(col), csr.values.cpu(), "cuda", m, csr.n, 64]
    tiled, plain = RoDeCSR(*args, locality=True), RoDeCSR(*args, locality=False)
    assert tiled.plan.counts[3] == m // 16 and plain.plan is None
    gen = torch.Generator(device="cuda").manual_seed(1)
    q, k, v, g = (torch.randn(48, r, d, device="cuda", generator=gen) for r in (m, csr.n, csr.n, m))
    k[:, 200, 3] = float("inf")
    res = []
    for c in (tiled, plain):
        ins = [t.to(dt).requires_grad_() for t in (q, k, v)]
        res.append(torch.autograd.grad(sparse_attention(c, *ins, scale=0.1), ins, g))
    for a, b in zip(*res):
        assert torch.equal(a.isfinite(), b.isfinite()) and b.isfinite().any() and not b.isfinite().all()
        ok = b.isfinite()
        assert (a[ok].float() - b[ok].float()).abs().max() <= (4e-3 if half else 2e-5) * b[ok].float().abs().max()


COLS = [  # columns of the mask, window, rows that the window moves per column, other rows, width, half
    (16, 64, 0, 0, 64, False),     # one tile, whole steps only, nothing outside the runs
    (75, 69, 1, 5, 64, True),      # columns after the last tile, a cut-short last step
    (320, 260, 3, 70, 64, False),  # a tile that is none, more nonzeros outside than are staged at a time, some columns with none
    (320, 260, 3, 70, 64, True),
    (48, 97, 2, 20, 128, True),
    (48, 400, 2, 130, 128, False),
    (48, 130, 1, 16, 32, True),
    (48, 130, 1, 65, 32, False),
]


@pytest.mark.parametrize("m,window,shift,extra,d,half", COLS)
def test_column_pass_on_tiles_against_fp64(m, window, shift, extra, d, half):
    """dv = P^T g and dk = dZ^T q on a pattern whose rows are the mask's columns, with weights of its own per head; then with
    rows of g and q that are not finite and that not all columns of a tile hold."""
    csr, _ = _mask(m, window, shift, extra, seed=m + window, short_rows=(40,) if m == 320 else ())
    if m == 320:  # (columns 33 and 34 lose what they hold outside their runs)
        rp, col = csr.row_offsets.cpu().numpy(), csr.column_indices.cpu().numpy()
        row = np.repeat(np.arange(m), np.diff(rp))
        keep = ~np.isin(row, (33, 34)) | ((col >= shift * row) & (col < shift * row + window))
        rp = np.concatenate([[0], np.cumsum(np.bincount(row[keep], minlength=m))]).astype(np.int32)
        csr = RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col[keep]), csr.values.cpu()[torch.from_numpy(keep)], "cuda", m, csr.n, 64, locality=True)
    assert csr.plan.counts[3] == m // 16 - (1 if m == 320 else 0)
    assert 5 * 4 * csr.plan.counts[3] >= 4 * csr.plan.counts[1]  # (with fewer in tiles other kernels take them)
    heads, dt = _heads(csr), torch.float16 if half else torch.float32
    gen = torch.Generator(device="cuda").manual_seed(d)
    g = torch.randn(heads, csr.n, d, device="cuda", generator=gen)
    q = torch.randn(heads, csr.n, d, device="cuda", generator=gen).to(dt)
    pairs = torch.randn(heads, csr.nnz, 2, device="cuda", generator=gen)
    rows = torch.repeat_interleave(torch.arange(m, device="cuda"), (csr.row_offsets[1:] - csr.row_offsets[:-1]).long())
    weights = torch.zeros(2, m, csr.n, device="cuda", dtype=torch.float64)
    held = weights[0] != 0
    held[rows, csr.column_indices.long()] = True

    def run():
        dk, dv = (torch.full((heads, m, d), float("nan"), device="cuda") for _ in range(2))
        _lib.check(_lib.load().rode_hip_attention_backward_cols(
            _lib.DENSE_CODE["f16" if half else "f32"], heads, csr.n, m, csr.nnz, d, csr.row_offsets.data_ptr(), csr.column_indices.data_ptr(),
            pairs.data_ptr(), g.data_ptr(), q.data_ptr(), dk.data_ptr(), dv.data_ptr(), ctypes.byref(csr.call_plans()), None), "cols")
        torch.cuda.synchronize()
        return dv, dk

    clean = run()
    for h in (0, heads // 2, heads - 1):
        for i, dense in ((0, g[h]), (1, q[h])):
            weights[i][rows, csr.column_indices.long()] = pairs[h, :, i].double()
            # every product and sum rounds once; a sum of n terms in trees of chains of 64 at most
            bound = 2.0 ** -24 * (64 + 12) * (weights[i].abs() @ dense.double().abs())
            assert ((clean[i][h].double() - weights[i] @ dense.double()).abs() <= bound + 1e-30).all()
    first = int(csr.column_indices[0])
    last = shift * (m - 1) + window - 1
    g[:, first], q[:, last] = float("inf"), float("nan")
    for i, (now, row) in enumerate(zip(run(), (first, last))):
        touched = held[:, row]
        assert touched.any()
        assert not now[:, touched].isfinite().all(dim=2).any()
        torch.testing.assert_close(now[:, ~touched], clean[i][:, ~touched], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_rows_with_very_different_numbers_outside_their_runs(d, half):
    """Four rows share a wave outside their runs, 16 lanes each, 64 nonzeros at a time: none beside many, and either side of
    16, 64 and 128.  Column 0, which only some rows hold, is not finite: a row that holds nothing there must not meet it."""
    m, window, dt = 64, 900, torch.float16 if half else torch.float32
    counts = [0, 130, 1, 16, 0, 0, 0, 0, 17, 15, 64, 65, 128, 129, 63, 3] + [0, 200, 0, 70, 2, 0, 0, 0, 0, 0, 0, 33, 80, 0, 31, 32] + list(range(50, 82))
    rng = np.random.default_rng(d)
    n = 1300
    cols = [np.sort(np.concatenate([np.arange(300 + r, 300 + r + window), rng.choice(298, k, replace=False)])) for r, k in enumerate(counts)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    col = np.concatenate(cols).astype(np.int32)
    csr = RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col), torch.ones(len(col)), "cuda", m, n, 64, locality=True)
    assert csr.plan.counts[3] == m // 16
    held = torch.zeros(m, n, dtype=torch.bool, device="cuda")
    held[torch.from_numpy(np.repeat(np.arange(m), np.diff(rp))).cuda(), csr.column_indices.long()] = True
    heads, scale = _heads(csr), d ** -0.5
    gen = torch.Generator(device="cuda").manual_seed(d)
    q, k, v, g = (torch.randn(r, d, device="cuda", generator=gen) for r in (m, n, n, m))
    q, k, v = (t.to(dt) for t in (q, k, v))
    ins = [t.double().requires_grad_() for t in (q, k, v)]
    want = _reference(held.double(), *ins, scale)
    want = (want,) + torch.autograd.grad(want, ins, g.double())
    ins = [t.expand(heads, *t.shape).contiguous().requires_grad_() for t in (q, k, v)]
    out = sparse_attention(csr, *ins, scale=scale)
    got = (out,) + torch.autograd.grad(out, ins, g.expand(heads, m, d).contiguous())
    for a, b in zip(got, want):
        assert (a[heads - 1].double() - b).norm() <= (2e-3 if half and b is not want[0] else 2e-6) * b.norm()
    k[0], v[0] = float("nan"), float("inf")
    ins = [t.expand(heads, *t.shape).contiguous().requires_grad_() for t in (q, k, v)]
    bad = sparse_attention(csr, *ins, scale=scale)
    dq, = torch.autograd.grad(bad, ins[:1], g.expand(heads, m, d).contiguous())
    touched = held[:, 0]
    assert touched.any() and not touched.all()
    for now, was in ((bad, out), (dq, got[1])):
        assert not now[:, touched].isfinite().all(dim=2).any()
        # (their tiles may be computed row by row now: either is within the bound above)
        assert (now[:, ~touched] - was[:, ~touched]).norm() <= (4e-3 if half and was is not out else 4e-6) * was[:, ~touched].norm()


@pytest.mark.parametrize("m,rows_left", [(1600, 0), (1608, 8)])
def test_fewer_nonzeros_where_the_tiles_have_all_rows(m, rows_left):
    """0.4 M nonzeros and more, on either side of the rule that gives them to the tiles."""
    csr, dense = _mask(m, 250, 1, 20, seed=m)
    assert csr.plan.counts[3] == m // 16 and 400_000 < csr.nnz < 1_500_000 and csr.plan.counts[2] == 0 and m % 16 == rows_left
    gen = torch.Generator(device="cuda").manual_seed(m)
    q, k, v, g = (torch.randn(r, 64, device="cuda", generator=gen) for r in (m, csr.n, csr.n, m))
    ins = [t.double().requires_grad_() for t in (q, k, v)]
    want = _reference(dense, *ins, 0.125)
    want = (want,) + torch.autograd.grad(want, ins, g.double())
    ins = [t.clone().requires_grad_() for t in (q, k, v)]
    out = sparse_attention(csr, *ins, scale=0.125)
    for a, b in zip((out,) + torch.autograd.grad(out, ins, g), want):
        assert (a.double() - b).norm() <= 2e-6 * b.norm()


@pytest.mark.parametrize("m,window,extra,d,half", [
    (1024, 360, 40, 64, False), (1024, 720, 40, 64, False), (1040, 360, 40, 64, False),  # up to 64 tiles, and more
    (1024, 360, 40, 128, True), (1024, 720, 40, 128, True), (1040, 360, 40, 128, True),
    (512, 660, 40, 128, False), (512, 740, 40, 128, False),  # below and above 700 nonzeros a row, and 0.4 M
    (1600, 240, 20, 32, True), (2400, 240, 20, 32, True),    # below and above 0.6 M
])
def test_few_tiles_that_have_all_rows(m, window, extra, d, half):
    """Either side of the lines between a wave per row and the tiles, where these have all rows."""
    csr, dense = _mask(m, window, 1, extra, seed=m + window)
    assert csr.plan.counts[3] == m // 16 and csr.plan.counts[2] == 0 and csr.nnz < 1_500_000
    dt = torch.float16 if half else torch.float32
    gen = torch.Generator(device="cuda").manual_seed(m)
    q, k, v, g = (torch.randn(r, d, device="cuda", generator=gen) for r in (m, csr.n, csr.n, m))
    q, k, v = (t.to(dt) for t in (q, k, v))
    ins = [t.double().requires_grad_() for t in (q, k, v)]
    want = _reference(dense, *ins, d ** -0.5)
    want = (want,) + torch.autograd.grad(want, ins, g.double())
    ins = [t.clone().requires_grad_() for t in (q, k, v)]
    out = sparse_attention(csr, *ins, scale=d ** -0.5)
    for a, b in zip((out,) + torch.autograd.grad(out, ins, g), want):
        assert (a.double() - b).norm() <= (2e-3 if half and b is not want[0] else 2e-6) * b.norm()


FOURS = [  # m, window, columns the window moves per row, random columns, width, scale; rows of three columns
    (16, 64, 0, 0, 64, 0.3, ()),              # one tile of four
    (75, 69, 1, 5, 64, 0.3, ()),              # four tiles and rows after the last
    (160, 260, 3, 70, 64, -0.3, (40,)),       # two and a half times four, one tile missing; more than 64 nonzeros outside a run
    (144, 97, 2, 20, 128, 0.2, (3, 70)),      # the first of four missing, the second
    (128, 130, 1, 16, 32, 0.4, tuple(range(0, 64, 16))),  # none of the first four
    (80, 400, 2, 130, 32, 0.2, ()),           # three times 64 outside a run
]


@pytest.mark.parametrize("m,window,shift,extra,d,scale,short", FOURS)
def test_four_tiles_a_workgroup_against_fp64(m, window, shift, extra, d, scale, short):
    """Halves; four tiles whatever their number (the figure that the call goes by is knowledge and changes no result)."""
    csr, dense = _mask(m, window, shift, extra, seed=m + window, short_rows=short)
    assert csr.plan.counts[3] == m // 16 - len(short)
    csr.call_plans().tile_fours = 1 << 20
    heads = _heads(csr)
    gen = torch.Generator(device="cuda").manual_seed(d)
    q, k, v = (torch.randn(heads, r, d, device="cuda", generator=gen).half() for r in (m, csr.n, csr.n))
    outs, scores, stats = _attention_call(csr, csr.values, q, k, v, scale, "scores")
    assert torch.equal(outs, sparse_attention(csr, q, k, v, scale=scale))
    outs_p, probs, _ = _attention_call(csr, csr.values, q, k, v, scale, "probs")
    assert torch.equal(outs, outs_p)
    rows = torch.repeat_interleave(torch.arange(m, device="cuda"), (csr.row_offsets[1:] - csr.row_offsets[:-1]).long())
    assert (probs - torch.exp(scores - stats[:, rows, 0]) * stats[:, rows, 1]).abs().max() <= 2e-6
    for h in (0, heads // 3, heads - 1):
        want = _reference(dense, q[h], k[h], v[h], scale)
        assert (outs[h].double() - want).abs().max() <= 2e-5 * want.abs().max()
        s = ((q[h].double() @ k[h].double().t()) * dense * scale)[rows, csr.column_indices.long()]
        assert (scores[h].double() - s).abs().max() <= 2e-5 * s.abs().max()


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("window,extra", [(96, 0), (160, 20), (330, 0), (520, 30)])
def test_four_tiles_a_workgroup_are_as_exact_as_one(window, extra, d):
    """2-norms of the errors against fp64 of at least 520 000 elements, each known to 0.1 %: 0.95 to 1.00 times those of a tile a workgroup. (Parts
    of four steps, put together with the nonzeros outside by a rescaling of both, had up to 1.05 times.)"""
    m, heads = 2048, 512 // d
    errors = []
    for fours in (0, 1 << 20):
        csr, dense = _mask(m, window, 1, extra, seed=window)
        assert csr.plan.counts[3] == m // 16
        csr.call_plans().tile_fours = fours
        gen = torch.Generator(device="cuda").manual_seed(d)
        q, k, v = (torch.randn(max(heads, _heads(csr)), r, d, device="cuda", generator=gen).half() for r in (m, csr.n, csr.n))
        out = sparse_attention(csr, q, k, v)
        want = torch.stack([_reference(dense, q[h], k[h], v[h], d ** -0.5) for h in range(heads)])
        errors.append((out[:heads].double() - want).norm().item())
    assert errors[0] != errors[1] and errors[1] <= 1.01 * errors[0]


def test_four_tiles_a_workgroup_without_range():
    """Infinite scores and rows of v that are not finite, in a run, at its ends and outside it: as with a tile a workgroup."""
    m, d, inf = 192, 64, float("inf")
    csr, dense = _mask(m, 100, 2, 30, seed=5)
    values = csr.values.clone()
    rows = torch.repeat_interleave(torch.arange(m, device="cuda"), (csr.row_offsets[1:] - csr.row_offsets[:-1]).long())
    for row, at, value in ((3, slice(None), -inf), (5, slice(0, 40), -inf), (50, slice(129, 130), -inf), (70, slice(50, 51), inf)):
        values[(rows == row).nonzero().flatten()[at]] = value
    one, four = (RoDeCSR(csr.row_offsets_cpu, csr.column_indices, values, "cuda", m, csr.n, 64, locality=True) for _ in range(2))
    one.call_plans().tile_fours, four.call_plans().tile_fours = 0, 1 << 20
    gen = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.rand(_heads(csr), r, d, device="cuda", generator=gen).half() for r in (m, csr.n, csr.n))
    v[:, [1, 130, 2 * 80 + 99, csr.n - 1]] = inf
    for x, y in zip(*(_attention_call(c, c.values, q, k, v, 0.125, "scores") for c in (four, one))):
        assert torch.equal(x.isnan(), y.isnan()) and torch.equal(x.isinf(), y.isinf())
        ok = y.isfinite()
        assert ok.any() and not ok.all()
        torch.testing.assert_close(x[ok], y[ok], rtol=2e-5, atol=2e-5)


def test_how_many_fours_a_plan_is_worth_and_runs_that_lie_apart():
    """A sliding window: the columns of all fours over those of one; runs that lie apart: none."""
    csr, _ = _mask(1040, 200, 1, 4, seed=1)  # 65 tiles: 16 fours of 263 columns (and what random columns add to a run), a last one of 215
    assert csr.plan.counts[3] == 65 and csr.plan.tile_fours == csr.call_plans().tile_fours == 16
    csr, _ = _mask(256, 100, 0, 0, seed=1)
    assert csr.plan.counts[3] == 16 and csr.plan.tile_fours == 4
    n = 16 * 200
    first = np.repeat(200 * np.random.default_rng(0).permutation(16), 16)
    col = (first[:, None] + np.arange(100)).astype(np.int32).ravel()
    apart = RoDeCSR(torch.arange(0, 25601, 100, dtype=torch.int32), torch.from_numpy(col), torch.ones(25600), "cuda", 256, n, 64, locality=True)
    assert apart.plan.counts[3] == 16 and apart.plan.tile_fours == 0
    gen = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(_heads(apart), r, 64, device="cuda", generator=gen).half() for r in (256, n, n))
    one = sparse_attention(apart, q, k, v)
    apart.call_plans().tile_fours = 1 << 20  # (said all the same: steps that one tile alone wants)
    torch.testing.assert_close(sparse_attention(apart, q, k, v), one, rtol=2e-5, atol=2e-6)


def test_a_few_fours_that_lie_apart():
    """Documents of 528 rows in a batch, a window of 160: at their ends, between tiles and inside of 64 rows, four tiles lie apart, three fours in
    thirty-two; with one end one."""
    m, d = 2048, 64
    gen = torch.Generator(device="cuda").manual_seed(1)
    row, column = np.arange(m)[:, None], np.arange(m)[None]
    for ends, worth in ((np.arange(528, m, 528), False), (np.array([528]), True)):
        which = np.searchsorted(ends, np.arange(m), side="right")
        allowed = (np.abs(row - column) <= 80) & (which[:, None] == which[None])
        col = np.nonzero(allowed)[1].astype(np.int32)
        rp = np.concatenate(([0], np.cumsum(allowed.sum(1)))).astype(np.int32)
        csr = RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col), torch.ones(len(col)), "cuda", m, m, d, locality=True)
        assert csr.plan.tile_fours > 20 if worth else csr.plan.tile_fours == 0
        csr.call_plans().tile_fours = 1 << 20
        q, k, v = (torch.randn(_heads(csr), m, d, device="cuda", generator=gen).half() for _ in range(3))
        out = sparse_attention(csr, q, k, v, scale=0.2)
        want = _reference(torch.from_numpy(allowed.astype(np.float64)).cuda(), q[0], k[0], v[0], 0.2)
        assert (out[0].double() - want).abs().max() <= 2e-5 * want.abs().max()


@pytest.mark.parametrize("keep", [None, "scores", "probs"])
@pytest.mark.parametrize("bad", [False, True])
def test_nonzeros_outside_the_runs_first(bad, keep):
    """fp32 with k and v of a head above 7 MB; a row of v that is not finite sends its tiles row by row after that."""
    m, d, scale = 1712, 64, 0.2
    csr, dense = _mask(m, 400, 8, 70, seed=3)
    assert csr.plan.counts[3] == m // 16 and 2 * csr.n * d * 4 >= 7_000_000
    gen = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn(3, r, d, device="cuda", generator=gen) for r in (m, csr.n, csr.n))
    clean = _reference(dense, q[1], k[1], v[1], scale)
    touched = torch.zeros(m, dtype=torch.bool, device="cuda")
    if bad:
        v[:, 2400] = float("inf")
        touched = dense[:, 2400] != 0
        assert touched.any() and not touched.all()
    out, scores, stats = _attention_call(csr, csr.values, q, k, v, scale, keep)
    assert not torch.isfinite(out[1][touched]).all(dim=1).any()
    assert (out[1].double() - clean)[~touched].abs().max() <= 2e-5 * clean.abs().max()
    if keep is not None:
        rows = torch.repeat_interleave(torch.arange(m, device="cuda"), (csr.row_offsets[1:] - csr.row_offsets[:-1]).long())
        s = (q[1].double() @ k[1].double().t()) * dense * scale
        if keep == "probs":
            s = torch.softmax(s.masked_fill(dense == 0, float("-inf")), dim=1)
        s = s[rows, csr.column_indices.long()]
        assert (scores[1].double() - s).abs().max() <= 2e-5 * s.abs().max()


@pytest.mark.parametrize("m,window,extra,d,heads,taken", [(8352, 578, 96, 128, 4, False), (8192, 320, 0, 128, 4, True), (6016, 320, 0, 128, 8, True), (17024, 440, 64, 64, 4, False),
                                                          (16384, 440, 0, 64, 4, True), (5248, 440, 64, 32, 16, False), (16384, 128, 0, 32, 4, True)])
def test_four_tiles_where_the_last_round_is_not_a_few(m, window, extra, d, heads, taken):
    """512, 1024 and 1280 workgroups of four tiles run at a time; with a few more than that the others wait for a second round of those (8352 rows x
    128, 524 workgroups: 152 us with a tile a workgroup, 181).  The bits of a tile a workgroup, or others."""
    gen, n = torch.Generator(device="cuda").manual_seed(d), m + window
    row = torch.arange(m, device="cuda")[:, None]
    col = torch.cat((row + torch.arange(window, device="cuda"), torch.randint(0, n, (m, extra), device="cuda", generator=gen)), 1)
    keys = torch.unique(row * n + col)
    ro = torch.searchsorted(keys, torch.arange(m + 1, device="cuda") * n).int().cpu()
    csr = RoDeCSR(ro, (keys % n).int(), torch.ones(len(keys), device="cuda"), "cuda", m, n, d, config="auto")
    assert csr.plan.counts[3] == m // 16
    q, k, v = (torch.randn(heads, r, d, device="cuda", generator=gen).half() for r in (m, csr.n, csr.n))
    out = sparse_attention(csr, q, k, v)
    csr.call_plans().tile_fours = 0
    assert torch.equal(out, sparse_attention(csr, q, k, v)) != taken
