"""SpMM whose column tiles are dealt out to the XCDs, against fp64."""
import numpy as np
import pytest
import torch

from rode_amd import RoDeCSR, rode_spmm

pytestmark = pytest.mark.gpu


def _matrix(lengths, n, width, seed):
    rng = np.random.default_rng(seed)
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, l, replace=False)) for l in lengths]).astype(np.int32)
    val = torch.from_numpy(rng.uniform(-1, 1, len(col)).astype(np.float32))
    return RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col), val, "cuda", len(lengths), n, width, locality=False)


def _lengths(kind, rng):
    if kind == "one":
        return np.array([40])
    if kind == "short":  # no block list; empty rows
        return rng.choice([0, 1, 3, 31], 700)
    if kind == "long":  # no residue list: multiples of 32, some of several segments
        return rng.choice([32, 512, 1024, 1056, 2080], 61)
    return rng.choice([0, 2, 31, 32, 33, 700, 1500], 333)


@pytest.mark.parametrize("half,width", [(False, 64), (False, 128), (False, 256), (True, 128), (True, 512)])
@pytest.mark.parametrize("kind", ["one", "short", "long", "mixed"])
@pytest.mark.parametrize("megabytes", [4, 8, 16, 48])  # (of B: just over an L2, and over the lines that rows with block segments have)
def test_sharded_against_fp64(kind, half, width, megabytes):
    n = megabytes * 2**20 // (width * (2 if half else 4)) + 3
    lengths = np.minimum(_lengths(kind, np.random.default_rng(width)), n // 2)
    csr = _matrix(lengths, n, width, seed=width)
    g = torch.Generator(device="cuda").manual_seed(width)
    B = torch.randn(n, width, device="cuda", generator=g).to(torch.float16 if half else torch.float32)
    dense = torch.sparse_csr_tensor(csr.row_offsets.long(), csr.column_indices.long(), csr.values.double(), (csr.m, n)).to_dense()
    want = dense @ B.double()
    torch.full((csr.m, width), float("nan"), device="cuda")  # (what the result's memory may hold before)
    into = torch.zeros(csr.m, width, device="cuda")
    for got in (rode_spmm(csr, B), rode_spmm(csr, B, values=csr.values.clone()), rode_spmm(csr, B, out=into)):
        assert (got.double() - want).abs().max() <= 1e-5 * want.abs().max()
