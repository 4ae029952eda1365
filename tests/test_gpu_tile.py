"""Attention on the tiles of 16 rows (matrix cores) against fp64 on dense matrices."""
import numpy as np
import pytest
import torch

from rode_amd import RoDeCSR, sparse_attention
from rode_amd.autograd import _attention_call

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


CASES = [  # m, window, columns the window moves per row, random columns, width, half, scale
    (16, 64, 0, 0, 64, False, 0.3),      # one tile, nothing outside the run, whole steps only
    (75, 69, 1, 5, 64, True, 0.3),       # rows after the last tile, a cut-short last step
    (160, 260, 3, 70, 64, False, -0.3),  # more than 64 nonzeros outside a run, a negative scale
    (160, 260, 3, 70, 64, True, -0.3),
    (48, 97, 2, 20, 128, True, 0.2),
    (48, 97, 2, 20, 128, False, 0.2),
    (48, 130, 1, 16, 32, True, 0.4),
    (48, 130, 1, 16, 32, False, 0.4),
]


@pytest.mark.parametrize("m,window,shift,extra,d,half,scale", CASES)
def test_tiles_against_fp64(m, window, shift, extra, d, half, scale):
    csr, dense = _mask(m, window, shift, extra, seed=m + window, short_rows=(40,) if m == 160 else ())
    assert csr.plan.counts[3] == m // 16 - (1 if m == 160 else 0)
    dt = torch.float16 if half else torch.float32
    g = torch.Generator(device="cuda").manual_seed(d)
    heads = 256  # (fewer tiles than CUs may take other kernels)
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
    out = sparse_attention(csr, *(t.expand(64, *t.shape).contiguous() for t in (q, k, v)), scale=0.2)[63]
    touched = (dense[:, bad] != 0).any(dim=1)
    assert touched.any() and not touched.all()
    assert not torch.isfinite(out[touched]).all(dim=1).any()
    assert (out[~touched].double() - clean[~touched]).abs().max() <= 2e-5 * clean.abs().max()
