"""The window kernels (banded matrices) against fp64 on the CPU."""
import numpy as np
import pytest
import scipy.sparse
import torch

from rode_amd import RoDeCSR, rode_sddmm, rode_sddmm_hip, rode_spmm

pytestmark = pytest.mark.gpu


def _banded(m, degree, band, far, k, seed):
    """Rows of 0 .. degree nonzeros in a band, rows % 7 == 3 with `far` columns anywhere; some rows of 128 have their
    columns anywhere (a chunk without a window)."""
    rng = np.random.default_rng(seed)
    rows = []
    for r in range(m):
        lo = min(max(0, r - band // 2), m - band)
        c = lo + rng.choice(band, rng.integers(0, degree + 1), replace=False)
        if m > 1000 and r // 128 % 5 == 2:
            c = rng.choice(m, 8, replace=False)
        if far and r % 7 == 3:
            c = np.concatenate([c, rng.choice(m, far, replace=False)])
        rows.append(np.unique(c))
    rp = np.concatenate([[0], np.cumsum([len(c) for c in rows])]).astype(np.int32)
    col = np.concatenate(rows).astype(np.int32)
    val = rng.uniform(0.5, 1.5, len(col)).astype(np.float32)
    csr = RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col), torch.from_numpy(val), "cuda", m, m, k, locality=True)
    assert csr.plan is not None and csr.plan.counts[1] > 0
    return csr, scipy.sparse.csr_matrix((val.astype(np.float64), col, rp), shape=(m, m))


CASES = [  # rows, nonzeros of a row at most, band, columns outside it: one chunk cut short; several per workgroup, with misses; none missing
    (101, 25, 60, 0), (128 * 261 + 5, 21, 200, 3), (128 * 520, 31, 90, 0)]


@pytest.mark.parametrize("m,degree,band,far", CASES)
@pytest.mark.parametrize("dtype,k", [(torch.float32, 36), (torch.float32, 128), (torch.float16, 72), (torch.float16, 128),
                                     (torch.float64, 18), (torch.float64, 48)])
def test_window_kernels_against_fp64(m, degree, band, far, dtype, k):
    csr, ref = _banded(m, degree, band, far, 64 if dtype == torch.float64 else k, seed=m + far)
    g = torch.Generator().manual_seed(k)
    dense = torch.randn(m, k, generator=g, dtype=torch.float64).to(dtype)
    want = ref @ dense.double().numpy()
    if dtype == torch.float64:
        got = rode_sddmm_hip.spmm_forward(csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2, csr.row_offsets,
                                          csr.column_indices, csr.values.double(), m, m, dense.cuda(), plan=csr.plan)
        assert np.abs(got.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()
        return
    got = rode_spmm(csr, dense.cuda())
    assert np.abs(got.cpu().double().numpy() - want).max() <= 1e-5 * np.abs(want).max()
    lhs = torch.randn(m, k, generator=g).to(dtype)
    got = rode_sddmm(csr, lhs.cuda(), dense.cuda()).cpu().double().numpy()
    rows = np.repeat(np.arange(m), np.diff(ref.indptr))
    want = ref.data * np.einsum("ij,ij->i", lhs.double().numpy()[rows], dense.double().numpy()[ref.indices])
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
