"""SpMM parity on the GPU, through the Python op and the C ABI.  The reference has
no SpMM test or CPU SpMM; the oracle is the textbook CSR product in fp64
(oracle.spmm_f64, pinned by scipy.sparse), judged with the row-L1-normalised
bound: 1e-4 for fp32 B, 2e-3 for fp16 B with fp32 accumulation."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(csr, rp, col, val, B, half=False):
    import oracle
    from gpu_common import TOL_F16, TOL_F32, check_csr_decomposition, round_half, run_spmm
    from helpers import spmm_row_l1_error
    check_csr_decomposition(csr, rp)
    C = run_spmm(csr, B, half)
    assert C.shape == (csr.m, B.shape[1]) and C.dtype == np.float32
    if half:
        B = round_half(B)
    ref64, scale = oracle.spmm_f64(rp, col, val, B, with_abs=True)
    err = spmm_row_l1_error(C, ref64)
    assert err <= (TOL_F16 if half else TOL_F32), f"row-L1 error {err}"
    if not half:
        strict = np.abs(C - ref64) / np.maximum(scale, 1e-30)
        assert strict.max(initial=0.0) <= 2e-6, f"per-element error {strict.max()}"
    return err


@pytest.mark.parametrize("n", [32, 64, 128, 96, 256])
@pytest.mark.parametrize("seg", [32, 512])
def test_unpadded_rows(n, seg):
    from gpu_common import make_csr
    from helpers import random_csr
    rng = np.random.default_rng(100 * n + seg)
    m, k = 1500, 1333
    rp, col, val = random_csr(rng, m, k, 37, long_rows=6, long_len=1300, empty_frac=0.15)
    B = rng.standard_normal((k, n)).astype(np.float32)
    _check(make_csr(rp, col, val, m, k, 32, seg), rp, col, val, B)


@pytest.mark.parametrize("n", [4, 8, 20, 36, 72, 100, 160, 200, 264])
def test_any_width(n):
    """Widths beyond the reference's multiples of 32: any multiple of 4 (the partial last
    tile is guarded; the columns next to it must stay untouched)."""
    import oracle
    from gpu_common import DEV, make_csr
    from helpers import random_csr, spmm_row_l1_error
    from rode_amd import rode_spmm
    rng = np.random.default_rng(n)
    m, k = 600, 650
    rp, col, val = random_csr(rng, m, k, 35, long_rows=4, long_len=600, empty_frac=0.1)
    B = rng.standard_normal((k, n)).astype(np.float32)
    csr = make_csr(rp, col, val, m, k, 32)
    _check(csr, rp, col, val, B)
    if n % 8 == 0:
        _check(csr, rp, col, val, B, half=True)
    assert rode_spmm(csr, torch.from_numpy(B).to(DEV)).shape == (m, n)
    # an fp64 run of the same width (vector of 2)
    from rode_amd import rode_sddmm_hip
    C64 = rode_sddmm_hip.spmm_forward(csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2,
                                      csr.row_offsets, csr.column_indices, csr.values.double(), m, k,
                                      torch.from_numpy(B).to(DEV).double()).cpu().numpy()
    ref = oracle.spmm_f64(rp, col, val, B)
    assert spmm_row_l1_error(C64, ref) <= 1e-12


def test_edge_tile_does_not_write_past_the_row():
    """C is (m, n) with n = 36: the second 32-wide tile has 4 live columns.  A canary row
    appended after C and the next row's first columns must be unchanged / correct."""
    import oracle
    from gpu_common import DEV, make_csr
    from helpers import random_csr
    from rode_amd import rode_sddmm_hip
    rng = np.random.default_rng(77)
    m, k, n = 300, 320, 36
    rp, col, val = random_csr(rng, m, k, 40, long_rows=3, long_len=300)
    B = rng.standard_normal((k, n)).astype(np.float32)
    csr = make_csr(rp, col, val, m, k, 32)
    buf = torch.zeros((m + 1) * n, device=DEV)
    buf[m * n:] = 123.0
    out = buf[: m * n].view(m, n)
    rode_sddmm_hip.spmm_forward(csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2,
                                csr.row_offsets, csr.column_indices, csr.values, m, k, torch.from_numpy(B).to(DEV),
                                out=out)
    assert (buf[m * n:] == 123.0).all()
    ref = oracle.spmm_f64(rp, col, val, B)
    assert np.abs(out.cpu().numpy() - ref).max() <= 1e-4 * np.abs(ref).sum(axis=1).max()


def test_padded_reference_matrices():
    """The reference generators' matrices (rows padded to 4 with explicit zeros)."""
    from gpu_common import make_csr
    from rode_amd import workloads
    for m, k, per_row, n in [(63, 67, 10, 32), (1023, 1031, 65, 128), (31, 4097, 200, 64), (1000, 1, 1, 32),
                             (1, 1000, 100, 128), (2048, 2048, 128, 64), (1024, 1024, 512, 32)]:
        rp, col, val = workloads.reference_csr(m, k, per_row, poisson=True)
        B = workloads.reference_dense(k, n, 456)
        _check(make_csr(rp, col, val, m, k, 32, 512), rp, col, val, B)


@pytest.mark.parametrize("n", [32, 64, 128])
def test_fp16_dense(n):
    from gpu_common import make_csr
    from helpers import random_csr
    rng = np.random.default_rng(n)
    m, k = 900, 1200
    rp, col, val = random_csr(rng, m, k, 50, long_rows=4, long_len=1100)
    B = rng.standard_normal((k, n)).astype(np.float32)
    for seg in (32, 512):
        _check(make_csr(rp, col, val, m, k, 32, seg), rp, col, val, B, half=True)


@pytest.mark.parametrize("n", [32, 64, 128, 96])
def test_fp64(n):
    """The double overloads (RoDeSpmm.h:10-14): fp64 values, B and C; bound 1e-12 of the row's L1 norm."""
    import oracle
    from gpu_common import DEV, make_csr
    from helpers import random_csr
    from rode_amd import rode_sddmm_hip
    rng = np.random.default_rng(n)
    m, k = 1100, 900
    rp, col, val = random_csr(rng, m, k, 41, long_rows=5, long_len=850, empty_frac=0.1)
    val64 = rng.uniform(-1, 1, len(val))
    B = rng.standard_normal((k, n))
    for seg in (32, 512):
        csr = make_csr(rp, col, val, m, k, 32, seg)
        C = rode_sddmm_hip.spmm_forward(csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2,
                                        csr.row_offsets, csr.column_indices, torch.from_numpy(val64).to(DEV), m, k,
                                        torch.from_numpy(B).to(DEV)).cpu().numpy()
        assert C.dtype == np.float64
        ref = oracle.spmm_d(rp, col, val64, B)
        l1 = np.abs(ref).sum(axis=1)
        assert (np.abs(C - ref).max(axis=1) <= 1e-12 * np.maximum(l1, 1e-300) + 1e-300).all()
        assert not C[np.diff(rp) == 0].any()
    with pytest.raises(RuntimeError, match="float64"):
        rode_sddmm_hip.spmm_forward(csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2,
                                    csr.row_offsets, csr.column_indices, csr.values, m, k, torch.from_numpy(B).to(DEV))


def test_fp64_cxx_overloads():
    """RoDeSpmm_n32(double) / RoDeSpmm_n128(double) through their mangled names."""
    import oracle
    from gpu_common import DEV, make_csr
    from helpers import random_csr
    from rode_amd import _lib
    lib = ctypes.CDLL(_lib.LIB_PATH)
    rng = np.random.default_rng(21)
    m, k = 700, 640
    rp, col, val = random_csr(rng, m, k, 45, long_rows=3, long_len=600)
    val64 = rng.uniform(-1, 1, len(val))
    csr = make_csr(rp, col, val, m, k, 32, 512)
    dv = torch.from_numpy(val64).to(DEV)
    for mangled, width in [("_Z12RoDeSpmm_n32iiiiPKdPKiS2_S2_S2_S2_S0_PdP12ihipStream_tS5_", 32),
                           ("_Z13RoDeSpmm_n128iiiiPKdPKiS2_S2_S2_S2_S0_PdP12ihipStream_tS5_", 64)]:
        fn = getattr(lib, mangled)
        fn.restype = None
        fn.argtypes = [ctypes.c_int] * 4 + [ctypes.c_void_p] * 10
        B = rng.standard_normal((k, width))
        dB = torch.from_numpy(B).to(DEV)
        C = torch.zeros(m, width, dtype=torch.float64, device=DEV)
        torch.cuda.synchronize()
        fn(csr.m1, csr.m2, k, width, dv.data_ptr(), csr.column_indices.data_ptr(), csr.row_offsets.data_ptr(),
           csr.block_indices.data_ptr(), csr.residue_indices.data_ptr(), csr.st_offsets.data_ptr(), dB.data_ptr(),
           C.data_ptr(), None, None)
        torch.cuda.synchronize()
        np.testing.assert_allclose(C.cpu().numpy(), oracle.spmm_d(rp, col, val64, B), rtol=1e-11, atol=1e-11)


def test_special_cases_and_edges():
    from gpu_common import DEV, make_csr, run_spmm
    from helpers import random_csr
    from rode_amd import rode_spmm
    rng = np.random.default_rng(4)
    m, k, n = 800, 700, 64
    rp, col, val = random_csr(rng, m, k, 45, long_rows=3, long_len=650, empty_frac=0.2)
    csr = make_csr(rp, col, val, m, k, 32, 512)
    # B = 1 -> every column holds the row sums
    C = run_spmm(csr, np.ones((k, n), np.float32))
    sums = np.array([val[rp[r]:rp[r + 1]].astype(np.float64).sum() for r in range(m)])
    assert np.abs(C - sums[:, None]).max() < 1e-4 and (C == C[:, :1]).all()
    assert not C[np.diff(rp) == 0].any()
    # permutation pattern with unit values moves rows of B exactly
    perm = rng.permutation(k).astype(np.int32)
    B = rng.standard_normal((k, n)).astype(np.float32)
    pcsr = make_csr(np.arange(k + 1, dtype=np.int32), perm, np.ones(k, np.float32), k, k, 32, 512)
    np.testing.assert_array_equal(run_spmm(pcsr, B), B[perm])
    # a non-finite B row must only reach the rows that reference it (the head slots
    # of an unaligned segment belong to the previous row and are skipped, not multiplied by 0)
    B[0, :] = np.inf
    bad = int(col[rp[17]])
    B[bad, 5] = np.nan
    C = run_spmm(csr, B)
    touches = np.array([np.isin([0, bad], col[rp[r]:rp[r + 1]]).any() for r in range(m)])
    assert np.isfinite(C[~touches]).all() and (~np.isfinite(C[touches])).any(axis=1).all()
    # accumulate-in-place semantics of the reference kernels: rows with >= 32 aligned
    # slots add to C, shorter rows overwrite, empty rows are left alone
    B = rng.standard_normal((k, n)).astype(np.float32)
    base = run_spmm(csr, B)
    pre = torch.full((m, n), 2.0, device=DEV)
    got = rode_spmm(csr, torch.from_numpy(B).to(DEV), out=pre).cpu().numpy()
    aligned = np.diff(rp) + rp[:-1] % 4
    adds = aligned >= 32
    # an empty row whose offset is a multiple of 4 is in no list; one at another offset is a zero-slot residue
    keeps = (np.diff(rp) == 0) & (rp[:-1] % 4 == 0)
    np.testing.assert_allclose(got[adds], base[adds] + 2.0, rtol=1e-5, atol=1e-5)
    np.testing.assert_array_equal(got[~adds & ~keeps], base[~adds & ~keeps])
    assert (got[keeps] == 2.0).all()
    # empty matrix
    empty = make_csr(np.zeros(6, np.int32), np.zeros(0, np.int32), np.zeros(0, np.float32), 5, 7, 32)
    assert not rode_spmm(empty, torch.ones(7, 32, device=DEV)).any()
    # width not a multiple of 32
    with pytest.raises(ValueError):
        rode_spmm(csr, torch.zeros(k, 42, device=DEV))
    with pytest.raises(ValueError):
        rode_spmm(csr, torch.zeros(k + 1, 32, device=DEV))


def test_cxx_reference_signature_entry_points():
    """RoDeSpmm_n32 / RoDeSpmm_n128 / RoDeSDDMM_n32 / RoDeSDDMM_n128 with the reference's
    signatures (RoDeSpmm.h:4-8, RoDeSddmm.h:4-9), called through their mangled names
    on two side streams, as a C++ caller would."""
    import oracle
    from gpu_common import DEV, make_csr
    from helpers import random_csr, sddmm_row_l1_error, spmm_row_l1_error
    from rode_amd import _lib
    lib = ctypes.CDLL(_lib.LIB_PATH)
    rng = np.random.default_rng(11)
    m, ncols = 1200, 1100
    rp, col, val = random_csr(rng, m, ncols, 40, long_rows=5, long_len=1000)
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    for name, mangled, width in [("spmm", "_Z12RoDeSpmm_n32iiiiPKfPKiS2_S2_S2_S2_S0_PfP12ihipStream_tS5_", 32),
                                 ("spmm", "_Z13RoDeSpmm_n128iiiiPKfPKiS2_S2_S2_S2_S0_PfP12ihipStream_tS5_", 128),
                                 ("sddmm", "_Z13RoDeSDDMM_n32iiiiPKiS0_S0_S0_S0_PKfS2_S2_PfP12ihipStream_tS5_", 32),
                                 ("sddmm", "_Z14RoDeSDDMM_n128iiiiPKiS0_S0_S0_S0_PKfS2_S2_PfP12ihipStream_tS5_", 128)]:
        fn = getattr(lib, mangled)
        fn.restype = None
        fn.argtypes = [ctypes.c_int] * 4 + [ctypes.c_void_p] * 11 if name == "sddmm" else \
            [ctypes.c_int] * 4 + [ctypes.c_void_p] * 10
        seg = 32 if (name == "sddmm" and width == 128) else 512  # the reference's parameter sets
        csr = make_csr(rp, col, val, m, ncols, 32, seg)
        if name == "spmm":
            B = rng.standard_normal((ncols, width)).astype(np.float32)
            dB = torch.from_numpy(B).to(DEV)
            C = torch.zeros(m, width, device=DEV)
            torch.cuda.synchronize()
            fn(csr.m1, csr.m2, ncols, width, csr.values.data_ptr(), csr.column_indices.data_ptr(),
               csr.row_offsets.data_ptr(), csr.block_indices.data_ptr(), csr.residue_indices.data_ptr(),
               csr.st_offsets.data_ptr(), dB.data_ptr(), C.data_ptr(), s1.cuda_stream, s2.cuda_stream)
            torch.cuda.synchronize()
            assert spmm_row_l1_error(C.cpu().numpy(), oracle.spmm_f64(rp, col, val, B)) <= 1e-4
        else:
            lhs = rng.standard_normal((m, width)).astype(np.float32)
            rhs = rng.standard_normal((ncols, width)).astype(np.float32)
            dl, dr = torch.from_numpy(lhs).to(DEV), torch.from_numpy(rhs).to(DEV)
            out = torch.full((len(val),), float("nan"), device=DEV)
            torch.cuda.synchronize()
            fn(csr.m1, csr.m2, ncols, width, csr.block_indices.data_ptr(), csr.residue_indices.data_ptr(),
               csr.st_offsets.data_ptr(), csr.row_offsets.data_ptr(), csr.column_indices.data_ptr(),
               csr.values.data_ptr(), dl.data_ptr(), dr.data_ptr(), out.data_ptr(), s1.cuda_stream, s2.cuda_stream)
            torch.cuda.synchronize()
            assert sddmm_row_l1_error(out.cpu().numpy(), oracle.sddmm_f64(rp, col, val, lhs, rhs), rp) <= 1e-4


@pytest.mark.parametrize("name,n", [("c1_uniform", 32), ("c2_lognormal", 32), ("c2_lognormal", 128)])
def test_benchmark_configs_against_oracle(name, n):
    from gpu_common import make_csr
    from rode_amd import workloads
    m, k, rp, col, val = workloads.config(name)
    B = np.random.default_rng(5000 + n).standard_normal((k, n)).astype(np.float32)
    for seg in (512, 32):
        _check(make_csr(rp, col, val, m, k, 32, seg), rp, col, val, B)


@pytest.mark.parametrize("name,n,half", [("c3_banded", 128, False), ("c4_powerlaw", 64, False),
                                         ("c5_attention", 64, False), ("c5_attention", 64, True)])
def test_large_configs_scaled_against_oracle(name, n, half):
    from gpu_common import make_csr
    from rode_amd import workloads
    scale = {"c3_banded": 1 / 16, "c4_powerlaw": 1 / 16, "c5_attention": 1 / 4}[name]
    m, k, rp, col, val = workloads.config(name, scale)
    B = np.random.default_rng(6000 + n).standard_normal((k, n)).astype(np.float32)
    _check(make_csr(rp, col, val, m, k, 32, 512), rp, col, val, B, half=half)


@pytest.mark.parametrize("name,n", [("c3_banded", 128), ("c4_powerlaw", 128), ("c4_powerlaw", 64), ("c5_attention", 64)])
def test_full_size_properties(name, n):
    """Full benchmark sizes through size-independent facts: B = 1 gives the row sums
    (checked against a segmented fp64 sum), the result is linear in B, and a checksum
    of C equals the checksum computed from column sums of the pattern."""
    from gpu_common import DEV, make_csr
    from rode_amd import rode_spmm, workloads
    m, k, rp, col, val = workloads.config(name)
    csr = make_csr(rp, col, val, m, k, 32, 512)
    C = rode_spmm(csr, torch.ones(k, n, device=DEV))
    nonempty = np.nonzero(np.diff(rp) > 0)[0]
    sums = np.zeros(m)
    sums[nonempty] = np.add.reduceat(val.astype(np.float64), rp[nonempty].astype(np.int64))
    abs_sums = np.zeros(m)
    abs_sums[nonempty] = np.add.reduceat(np.abs(val.astype(np.float64)), rp[nonempty].astype(np.int64))
    # every column holds the same sum (atomic accumulation order may differ per column)
    dsums = torch.from_numpy(sums).to(DEV)[:, None]
    dabs = torch.from_numpy(np.maximum(abs_sums, 1e-30)).to(DEV)[:, None]
    assert ((C.double() - dsums).abs() / dabs).max().item() <= 1e-5
    del C
    # checksum of checksums: sum_r C[r, j] = sum_c w[c] * B[c, j] with w = column sums of A
    g = torch.Generator(device=DEV).manual_seed(n)
    B = torch.randn(k, n, device=DEV, generator=g)
    C = rode_spmm(csr, B)
    w = np.bincount(col, weights=val.astype(np.float64), minlength=k)
    want = torch.from_numpy(w).to(DEV) @ B.double()
    wabs = torch.from_numpy(np.bincount(col, weights=np.abs(val.astype(np.float64)), minlength=k)).to(DEV) @ B.double().abs()
    assert ((C.double().sum(0) - want).abs() / wabs).max().item() < 1e-5
    # linearity
    B2 = torch.randn(k, n, device=DEV, generator=g)
    C2 = rode_spmm(csr, B2)
    C12 = rode_spmm(csr, B + B2)
    denom = torch.from_numpy(abs_sums).to(DEV).float()[:, None] * 8 + 1e-20
    assert ((C12 - (C + C2)).abs() / denom).max().item() < 1e-4


def test_dense_operand_beyond_2_gib():
    """B and rhs of 2.4 GB: byte offsets col * n * 4 exceed 2^31, where the reference's
    32-bit offset arithmetic (RoDeSpmm.cu:153,287) overflows.  Checked on the rows'
    exact expected values: B[c, j] = (c % 1000) + j / 256 is exactly representable."""
    from gpu_common import DEV, make_csr
    from rode_amd import rode_sddmm, rode_spmm
    rng = np.random.default_rng(31)
    m, n, k = 2000, 4_700_000, 128
    lens = rng.integers(0, 90, m)
    lens[7] = 3000
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, size=l, replace=False)) for l in lens]).astype(np.int32)
    col[rp[7 + 1] - 1] = n - 1  # the very last dense row
    val = np.ones(len(col), np.float32)
    csr = make_csr(rp, col, val, m, n, k)
    B = (torch.arange(n, device=DEV) % 1000).float()[:, None] + torch.arange(k, device=DEV).float()[None, :] / 256
    assert B.numel() * 4 > 2**31
    C = rode_spmm(csr, B).cpu().numpy().astype(np.float64)
    colsum = np.zeros(m)
    nonempty = np.nonzero(lens > 0)[0]
    colsum[nonempty] = np.add.reduceat((col % 1000).astype(np.float64), rp[nonempty].astype(np.int64))
    want = colsum[:, None] + lens[:, None] * (np.arange(k) / 256.0)[None, :]
    # fp32 accumulation of up to 3000 terms per row
    assert (np.abs(C - want).max(axis=1) <= 1e-4 * np.abs(want).max(axis=1) + 1e-30).all()
    # SDDMM with lhs = e_0: out[idx] = rhs[col, 0] = col % 1000
    lhs = torch.zeros(m, k, device=DEV)
    lhs[:, 0] = 1
    out = rode_sddmm(csr, lhs, B).cpu().numpy()
    np.testing.assert_array_equal(out, (col % 1000).astype(np.float32))


def test_clear_rows_prepares_exactly_what_spmm_does_not_overwrite():
    from gpu_common import DEV, make_csr
    from helpers import random_csr
    from rode_amd import _lib, rode_sddmm_hip
    lib = _lib.load()
    rng = np.random.default_rng(13)
    m, k, n = 900, 800, 96
    rp, col, val = random_csr(rng, m, k, 30, long_rows=4, long_len=700, empty_frac=0.2)
    csr = make_csr(rp, col, val, m, k, 32)
    C = torch.full((m, n), float("nan"), device=DEV)
    assert lib.rode_hip_spmm_clear_rows(m, n, 4, csr.row_offsets.data_ptr(), C.data_ptr(), None) == 0
    torch.cuda.synchronize()
    aligned = np.diff(rp) + rp[:-1] % 4
    cleared = (aligned >= 32) | (aligned == 0)
    got = C.cpu().numpy()
    assert (got[cleared] == 0).all() and np.isnan(got[~cleared]).all()
    # SpMM on the prepared buffer == SpMM on a fully zeroed one
    B = torch.from_numpy(rng.standard_normal((k, n)).astype(np.float32)).to(DEV)
    args = (csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2, csr.row_offsets,
            csr.column_indices, csr.values, m, k, B)
    a = rode_sddmm_hip.spmm_forward(*args, out=C)
    b = rode_sddmm_hip.spmm_forward(*args, out=torch.zeros(m, n, device=DEV))
    assert torch.isfinite(a).all() and (a - b).abs().max().item() <= 1e-5 * b.abs().max().item()
    # fp64 element size, bad arguments
    C64 = torch.full((m, 6), float("nan"), dtype=torch.float64, device=DEV)
    assert lib.rode_hip_spmm_clear_rows(m, 6, 8, csr.row_offsets.data_ptr(), C64.data_ptr(), None) == 0
    torch.cuda.synchronize()
    assert (C64[torch.from_numpy(cleared).to(DEV)] == 0).all()
    assert lib.rode_hip_spmm_clear_rows(m, 6, 4, csr.row_offsets.data_ptr(), C64.data_ptr(), None) != 0  # 24-byte rows
    assert lib.rode_hip_spmm_clear_rows(m, 8, 2, csr.row_offsets.data_ptr(), C64.data_ptr(), None) != 0


@pytest.mark.parametrize("seg,half", [(32, False), (96, False), (512, False), (512, True), (160, True)])
def test_whole_row_mode_and_split_calls(seg, half):
    """With >= 16384 block segments and the whole-lists promise (what the Python op
    passes), rows of 32..1024 slots are summed by one wave, tail included; rows just
    outside that range, unaligned starts and empty rows sit next to them here.  The
    typed entry points make no such promise: a caller who feeds the two lists in
    separate calls, or the block list in two halves, must get the same matrix (with
    >= 16384 segments per call the block kernel still merges short segments of a row,
    within the slice it was given: seg 32 and 96 here)."""
    import oracle
    from gpu_common import DEV, TOL_F16, TOL_F32, make_csr, round_half, run_spmm
    from helpers import spmm_row_l1_error
    from rode_amd import _lib
    lib = _lib.load()
    rng = np.random.default_rng(seg)
    m, k, n = 24000, 3000, 64
    lens = rng.choice([0, 1, 5, 31, 32, 33, 63, 64, 100, 500, 1000, 1020, 1021, 1024, 1025, 1056, 1500], size=m,
                      p=[.05, .05, .1, .05, .05, .05, .05, .05, .2, .1, .05, .03, .03, .03, .03, .03, .05])
    lens[::4000] = [2999, 2500, 2048, 1999, 2990, 1600]  # several merge windows per row (k = 3000 columns)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(k, size=l, replace=False)) for l in lens]).astype(np.int32)
    val = rng.uniform(-1, 1, rp[-1]).astype(np.float32)
    B = rng.standard_normal((k, n)).astype(np.float32)
    csr = make_csr(rp, col, val, m, k, 32, seg)
    assert csr.m1 >= 16384
    ref = oracle.spmm_f64(rp, col, val, round_half(B) if half else B)
    tol = TOL_F16 if half else TOL_F32
    assert spmm_row_l1_error(run_spmm(csr, B, half), ref) <= tol
    if half:
        return
    dB = torch.from_numpy(B).to(DEV)
    if seg == 96:  # the fp64 instantiation through the same promise
        from rode_amd import rode_sddmm_hip
        C64 = rode_sddmm_hip.spmm_forward(csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2,
                                          csr.row_offsets, csr.column_indices, csr.values.double(), m, k,
                                          dB.double()).cpu().numpy()
        assert spmm_row_l1_error(C64, ref) <= 1e-12

    def typed(m1, m2, blk_ptr, st_ptr, C):
        _lib.check(lib.rode_hip_spmm_f32(m1, m2, k, n, csr.values.data_ptr(), csr.column_indices.data_ptr(),
                                         csr.row_offsets.data_ptr(), blk_ptr, csr.residue_indices.data_ptr(), st_ptr,
                                         dB.data_ptr(), C.data_ptr(), None, None), "spmm")

    C = torch.zeros(m, n, device=DEV)
    half_m1 = csr.m1 // 2  # very likely inside a row
    typed(half_m1, 0, csr.block_indices.data_ptr(), csr.st_offsets.data_ptr(), C)
    typed(csr.m1 - half_m1, 0, csr.block_indices.data_ptr() + 4 * half_m1, csr.st_offsets.data_ptr() + 4 * half_m1, C)
    typed(0, csr.m2, csr.block_indices.data_ptr(), csr.st_offsets.data_ptr(), C)
    torch.cuda.synchronize()
    assert spmm_row_l1_error(C.cpu().numpy(), ref) <= tol


def test_headline_configuration_full_size_against_oracle():
    """Power law, full size, width 128, through rode_spmm (whole-lists promise with >= 16384
    block segments: rows of 32..1024 slots are summed by one wave, longer rows by merged
    leaders plus atomics) against the fp64 oracle on a fixed sample of rows that holds the
    longest row and rows of every kind."""
    import oracle
    from gpu_common import DEV, TOL_F32, make_csr
    from helpers import spmm_row_l1_error
    from rode_amd import rode_spmm, workloads
    from test_gpu_sddmm import sample_rows, sub_csr
    m, k, rp, col, val = workloads.config("c4_powerlaw")
    n = 128
    csr = make_csr(rp, col, val, m, k, n)
    assert csr.m1 >= 16384
    g = torch.Generator(device=DEV).manual_seed(78)
    B = torch.randn(k, n, device=DEV, generator=g)
    C = rode_spmm(csr, B)
    rows = sample_rows(rp, np.random.default_rng(5))
    sub_rp, idx = sub_csr(rp, rows)
    ref, scale = oracle.spmm_f64(sub_rp, col[idx], val[idx], B.cpu().numpy(), with_abs=True)
    got = C[torch.from_numpy(rows).to(DEV)].cpu().numpy()
    err = spmm_row_l1_error(got, ref)
    assert err <= TOL_F32, f"row-L1 error {err}"
    assert (np.abs(got - ref) / np.maximum(scale, 1e-30)).max() <= 2e-6
    print(f"c4 width 128 full size: {len(rows)} rows, {len(idx)} nnz, row-L1 error {err:.2e}")


def test_measurement_flags_launch_one_kernel_of_the_pair():
    """RODE_SPMM_ONLY_BLOCK + RODE_SPMM_ONLY_RESIDUE in two calls give the result of one
    normal call, also under the whole-lists promise (each kernel still skips what the
    other one sums)."""
    from gpu_common import DEV, make_csr
    from rode_amd import _lib
    lib = _lib.load()
    rng = np.random.default_rng(9)
    m, k, n = 20000, 2500, 64
    lens = rng.choice([0, 3, 31, 40, 100, 700, 1100, 2400], size=m, p=[.1, .2, .1, .2, .2, .1, .05, .05])
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(k, size=l, replace=False)) for l in lens]).astype(np.int32)
    val = rng.uniform(-1, 1, rp[-1]).astype(np.float32)
    csr = make_csr(rp, col, val, m, k, n, 32)
    assert csr.m1 >= 16384
    B = torch.from_numpy(rng.standard_normal((k, n)).astype(np.float32)).to(DEV)

    def call(flags, C):
        _lib.check(lib.rode_hip_spmm_ex(0, flags, csr.m1, csr.m2, k, n, csr.values.data_ptr(),
                                        csr.column_indices.data_ptr(), csr.row_offsets.data_ptr(),
                                        csr.block_indices.data_ptr(), csr.residue_indices.data_ptr(),
                                        csr.st_offsets.data_ptr(), B.data_ptr(), C.data_ptr(), None, None), "spmm")

    for base in (0, _lib.SPMM_WHOLE_LISTS):
        both, split = torch.zeros(m, n, device=DEV), torch.zeros(m, n, device=DEV)
        call(base, both)
        call(base | _lib.SPMM_ONLY_BLOCK, split)
        call(base | _lib.SPMM_ONLY_RESIDUE, split)
        torch.cuda.synchronize()
        assert (both - split).abs().max().item() <= 1e-4 * both.abs().max().item()
    assert lib.rode_hip_spmm_ex(0, 6, csr.m1, csr.m2, k, n, csr.values.data_ptr(), csr.column_indices.data_ptr(),
                                csr.row_offsets.data_ptr(), csr.block_indices.data_ptr(),
                                csr.residue_indices.data_ptr(), csr.st_offsets.data_ptr(), B.data_ptr(),
                                both.data_ptr(), None, None) != 0


def _spmm_overwrite(csr, B, C, flags):
    import ctypes
    from rode_amd import _lib, rode_sddmm_hip
    lib = _lib.load()
    plans = rode_sddmm_hip.plans_struct(csr.plan, B.shape[1], 4, True, seg_length=csr.config["seg_length"])
    s = torch.cuda.current_stream().cuda_stream
    code = lib.rode_hip_spmm_planned(_lib.DENSE_CODE["f16" if B.dtype == torch.float16 else "f32"], flags, csr.m1, csr.m2, csr.n,
                                     B.shape[1], csr.values.data_ptr(), csr.column_indices.data_ptr(), csr.row_offsets.data_ptr(),
                                     csr.block_indices.data_ptr(), csr.residue_indices.data_ptr(), csr.st_offsets.data_ptr(),
                                     B.data_ptr(), C.data_ptr(), ctypes.byref(plans), s, s)
    torch.cuda.synchronize()
    return code


@pytest.mark.parametrize("case", ["one_segment_rows", "short_rows_only", "segments_of_32", "every_row_in_a_group", "half"])
def test_overwrite_stores_rows_that_have_one_owner(case):
    """RODE_SPMM_OVERWRITE: C = A B into a C full of NaN, on matrices whose every row has slots
    and a single work item (rows summed whole by one wave, rows of fewer than 32 slots, rows of
    kept groups); ``RoDeCSR.spmm_stores_every_row`` says so and ``rode_spmm`` then clears nothing."""
    import oracle
    from gpu_common import DEV, TOL_F16, TOL_F32, make_csr, round_half
    from helpers import spmm_row_l1_error
    from rode_amd import _lib, rode_sddmm_hip, rode_spmm
    rng = np.random.default_rng(len(case))
    width, half, seg, locality = 64, case == "half", None, False
    if case in ("one_segment_rows", "half"):
        m, n = 6000, 3000
        lens = rng.integers(1, 900, m)     # aligned lengths up to 903 slots: whole rows (m1 >= 1024 segments)
    elif case == "short_rows_only":
        m, n = 5000, 3000
        lens = rng.integers(1, 28, m)      # residue rows only
    elif case == "segments_of_32":
        m, n, seg = 3000, 3000, 32
        lens = rng.integers(200, 1000, m)  # >= 16384 segments of 32 slots: a wave walks a chunk of them
    else:
        m, n, locality = 2000, 2400, True
        lens = None
    if lens is not None:
        rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        col = np.concatenate([np.sort(rng.choice(n, size=l, replace=False)) for l in lens]).astype(np.int32)
    else:
        rows = [np.arange(r, r + 300, dtype=np.int32) for r in range(m)]  # a window that moves one column per row
        rp = np.concatenate([[0], np.cumsum([len(c) for c in rows])]).astype(np.int32)
        col = np.concatenate(rows)
    val = rng.uniform(-1, 1, rp[-1]).astype(np.float32)
    csr = make_csr(rp, col, val, m, n, width, seg, locality=locality)
    if case == "every_row_in_a_group":
        assert isinstance(csr.plan, rode_sddmm_hip.GroupPlan) and csr.plan.counts[2] == 0
    if case == "segments_of_32":
        assert csr.m1 >= 16384
    assert csr.spmm_stores_every_row()
    B = rng.standard_normal((n, width)).astype(np.float32)
    dB = torch.from_numpy(B).to(DEV, torch.float16 if half else torch.float32)
    C = torch.full((m, width), float("nan"), device=DEV)
    assert _spmm_overwrite(csr, dB, C, _lib.SPMM_WHOLE_LISTS | _lib.SPMM_OVERWRITE) == 0
    ref = oracle.spmm_f64(rp, col, val, round_half(B) if half else B)
    got = C.cpu().numpy()
    assert np.isfinite(got).all(), "a row was added to, or left alone"
    assert spmm_row_l1_error(got, ref) <= (TOL_F16 if half else TOL_F32)
    again = rode_spmm(csr, dB).cpu().numpy()  # the op: an uninitialised C and no clearing
    assert spmm_row_l1_error(again, ref) <= (TOL_F16 if half else TOL_F32)


def test_overwrite_leaves_other_rows_to_the_callers_clearing():
    """Rows of several work items are still added to and rows without slots still untouched under
    RODE_SPMM_OVERWRITE (C holds 7 on entry); the limit function says which rows are which, and
    the flag needs the whole-lists promise."""
    import oracle
    from gpu_common import DEV, make_csr
    from rode_amd import _lib
    lib = _lib.load()
    rng = np.random.default_rng(77)
    m, n, width = 4000, 5000, 32
    lens = rng.integers(1, 600, m)
    lens[10], lens[11], lens[12] = 3000, 0, 1025   # several work items; no slots; one slot too many
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, size=l, replace=False)) for l in lens]).astype(np.int32)
    val = rng.uniform(-1, 1, rp[-1]).astype(np.float32)
    csr = make_csr(rp, col, val, m, n, width, locality=False)
    assert not csr.spmm_stores_every_row()
    limit = lib.rode_hip_spmm_overwrite_limit(csr.m1, None)
    assert limit == 1024 and lib.rode_hip_spmm_overwrite_limit(1023, None) == 0
    B = rng.standard_normal((n, width)).astype(np.float32)
    dB = torch.from_numpy(B).to(DEV)
    C = torch.full((m, width), 7.0, device=DEV)
    assert _spmm_overwrite(csr, dB, C, _lib.SPMM_WHOLE_LISTS | _lib.SPMM_OVERWRITE) == 0
    aligned = lens + rp[:-1] % 4
    added = (aligned > limit) | (aligned == 0)
    want = oracle.spmm_f64(rp, col, val, B) + np.where(added[:, None], 7.0, 0.0)
    assert np.abs(C.cpu().numpy() - want).max() <= 1e-4 * max(1.0, np.abs(want).max())
    assert _spmm_overwrite(csr, dB, C, _lib.SPMM_OVERWRITE) != 0   # not without the whole-lists promise


@pytest.mark.parametrize("dtype", ["f32", "f16", "f64"])
@pytest.mark.parametrize("rows,lengths,longest,k", [
    (300, (0, 5), 0, 32),           # residue rows only, and empty ones
    (5000, (0, 9), 0, 64),
    (40000, (0, 4), 0, 128),        # ... too many workgroups for one launch (fp32)
    (700, (0, 60), 0, 128),         # fewer than 1024 segments, every row short: owned by a wave each
    (700, (0, 60), 384, 40),        # (the longest such row; a width that ends inside a tile)
    (700, (0, 60), 385, 64),        # one row past it: cleared beforehand
    (3000, (0, 80), 1024, 64),      # the longest row with one owner
    (3000, (0, 80), 1025, 64),      # more than that: cleared beforehand
    (6000, (0, 70), 500, 256),      # several column tiles
    (64, (32, 33), 0, 32),          # (aligned lists: most rows have no tail)
])
def test_product_into_memory_that_holds_anything(rows, lengths, longest, k, dtype):
    """rode_hip_spmm_new: every row of C stored or cleared, whatever C holds before (NaN here), against 64 bits.  A
    sum of n products is off by at most (n + 2) roundings of the sum of their magnitudes (twice that where the reference is
    no wider).  ``longest``: the longest row, in aligned slots (0: as drawn)."""
    import oracle
    from gpu_common import DEV, round_half
    from rode_amd import RoDeCSR, _lib, rode_spmm
    rng = np.random.default_rng(rows + k)
    lens = rng.integers(*lengths, rows)
    lens[rng.integers(0, rows, rows // 8)] = 0
    if longest:
        lens[rows // 2] = longest - sum(lens[:rows // 2]) % 4
    cols = 6000
    row_ptr = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(cols, n, replace=False)) for n in lens]).astype(np.int32)
    val, B = rng.uniform(-1, 1, len(col)).astype(np.float32), rng.standard_normal((cols, k)).astype(np.float32)
    B = round_half(B) if dtype == "f16" else B
    want, scale = oracle.spmm_f64(row_ptr, col, val, B, with_abs=True)
    bound = torch.from_numpy(scale * (lens[:, None] + 2) * (2.0 ** -52 if dtype == "f64" else 2.0 ** -24)).to(DEV)
    want, val = torch.from_numpy(want).to(DEV), torch.from_numpy(val).to(DEV, torch.float64 if dtype == "f64" else torch.float32)
    B = torch.from_numpy(B).to(DEV, torch.float16 if dtype == "f16" else val.dtype)
    csr = RoDeCSR(torch.from_numpy(row_ptr), torch.from_numpy(col), val.float(), DEV, rows, cols, k, config="auto").with_values(val)
    assert not longest or csr.longest_row == longest
    lib = _lib.load()
    for longest_row in (csr.longest_row, 0):
        out = torch.full((rows, k), float("nan"), dtype=val.dtype, device=DEV)
        code = lib.rode_hip_spmm_new({"f32": 0, "f16": 1, "f64": 2}[dtype], rows, longest_row, csr.m1, csr.m2, cols, k, val.data_ptr(),
                                     csr.column_indices.data_ptr(), csr.row_offsets.data_ptr(), csr.block_indices.data_ptr(),
                                     csr.residue_indices.data_ptr(), csr.st_offsets.data_ptr(), B.data_ptr(), out.data_ptr(),
                                     ctypes.addressof(csr.call_plans(k, val.element_size())), torch.cuda.current_stream().cuda_stream)
        assert code == 0
        assert bool(((out.double() - want).abs() <= bound).all())
    if dtype != "f64":
        assert bool(((rode_spmm(csr, B).double() - want).abs() <= bound).all())


@pytest.mark.parametrize("dtype", ["f32", "f16", "f64"])
@pytest.mark.parametrize("rows,filled,length,k", [
    (1, [], 5, 32), (1, [0], 5, 32), (63, [62], 5, 64), (64, [0], 40, 128), (65, [64], 5, 128), (257, [3, 256], 40, 40),
    (1000, [0, 63, 64, 127, 128, 999], 200, 96), (70000, [5, 69999], 8, 32), (70000, [5, 69999], 40, 200),
])
def test_product_of_mostly_empty_rows(rows, filled, length, k, dtype):
    """A C of which nearly every row is one that no work item has: exactly zero there, the products in the others."""
    from gpu_common import DEV
    from rode_amd import RoDeCSR, _lib
    rng = np.random.default_rng(rows + k)
    lens = np.zeros(rows, dtype=np.int64)
    lens[filled] = length
    lens[filled[-1:]] += -lens.sum() % 4  # (a row without nonzeros after a ragged end has slots: here none does)
    lens[filled] += -lens[filled] % 4
    cols = 300
    row_ptr = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(cols, n, replace=False)) for n in lens[filled]] or [np.zeros(0)]).astype(np.int32)
    val = torch.from_numpy(rng.uniform(-1, 1, len(col))).to(torch.float64 if dtype == "f64" else torch.float32)
    dense = torch.from_numpy(rng.standard_normal((cols, k))).to(torch.float16 if dtype == "f16" else val.dtype)
    csr = RoDeCSR(torch.from_numpy(row_ptr), torch.from_numpy(col), val.float(), DEV, rows, cols, 32, config="auto")
    val, B = val.to(DEV), dense.to(DEV)
    code, lib = {"f32": 0, "f16": 1, "f64": 2}[dtype], _lib.load()
    for longest in (csr.longest_row, 0):
        out = torch.full((rows, k), float("nan"), dtype=val.dtype, device=DEV)
        assert lib.rode_hip_spmm_new(code, rows, longest, csr.m1, csr.m2, cols, k, val.data_ptr(), csr.column_indices.data_ptr(),
                                     csr.row_offsets.data_ptr(), csr.block_indices.data_ptr(), csr.residue_indices.data_ptr(),
                                     csr.st_offsets.data_ptr(), B.data_ptr(), out.data_ptr(), ctypes.addressof(csr.call_plans()),
                                     torch.cuda.current_stream().cuda_stream) == 0
        want = torch.zeros(rows, k, dtype=torch.float64)
        for r in filled:
            want[r] = val.cpu().double()[row_ptr[r]:row_ptr[r + 1]] @ dense.double()[col[row_ptr[r]:row_ptr[r + 1]].astype(np.int64)]
        got = out.cpu().double()
        # (a sum of up to 204 products of at most 5: (n + 2) roundings of the sum of their magnitudes)
        assert (got - want).abs().max() <= 206 * 204 * 5 * (2.0 ** -52 if dtype == "f64" else 2.0 ** -24)
        empty = torch.ones(rows, dtype=torch.bool)
        empty[filled] = False
        assert bool((got[empty] == 0).all())


def _sum_in_segments(val, dense, groups, segment=128):
    """Rows summed as segments of 128 slots and a tail that meet in C: in a segment 64 slots at a time, lane group g takes quads g,
    g + groups, ..., one fused multiply-add after the other in 32 bits.  val (rows, n), dense (rows, n, k)."""
    def chain(acc, at):
        return (acc.astype(np.float64) + val[:, at, None].astype(np.float64) * dense[:, at].astype(np.float64)).astype(np.float32)
    rows, n, k = dense.shape
    total = np.zeros((rows, k), dtype=np.float32)
    for s in range(0, n // 32 * 32, segment):
        accs = [np.zeros((rows, k), dtype=np.float32) for _ in range(groups)]
        for at in range(s, min(s + segment, n // 32 * 32)):
            g = at // 4 % 16 % groups
            accs[g] = chain(accs[g], at)
        while len(accs) > 1:
            accs = [accs[i] + accs[i + len(accs) // 2] for i in range(len(accs) // 2)]
        total = total + accs[0]
    tail = np.zeros((rows, k), dtype=np.float32)
    for at in range(n // 32 * 32, n):
        tail = chain(tail, at)
    return total + tail


@pytest.mark.parametrize("k,half,groups", [(128, False, 2), (64, False, 4), (32, False, 8), (128, True, 4)])
@pytest.mark.parametrize("length", [168, 252, 380])
def test_whole_rows_in_small_matrices_are_no_less_exact(length, k, half, groups):
    """Fewer than 1024 segments, every row summed by one wave: the error against 64 bits is no larger than that of segments of
    128 slots that meet in C.  (Root mean squares over 25 600 sums and more, known to a percent or two: a margin of a twentieth.)"""
    from gpu_common import DEV, round_half
    from rode_amd import RoDeCSR, rode_spmm
    rng = np.random.default_rng(length + k)
    rows, cols = 200, 3000
    col = np.stack([np.sort(rng.choice(cols, length, replace=False)) for _ in range(rows)]).astype(np.int32)
    val, B = rng.uniform(-1, 1, (rows, length)).astype(np.float32), rng.standard_normal((cols, 4 * k)).astype(np.float32)
    B = round_half(B) if half else B
    csr = RoDeCSR(torch.arange(0, rows * length + 1, length, dtype=torch.int32), torch.from_numpy(col.ravel()), torch.from_numpy(val.ravel()),
                  DEV, rows, cols, 32, config="auto")
    assert csr.m1 < 1024 and csr.config["seg_length"] == 128
    mine, segments = 0.0, 0.0
    for part in range(4):
        dense = np.ascontiguousarray(B[:, part * k:(part + 1) * k])
        got = rode_spmm(csr, torch.from_numpy(dense).to(DEV, torch.float16 if half else torch.float32)).cpu().numpy()
        want = np.einsum("rn,rnk->rk", val.astype(np.float64), dense[col].astype(np.float64))
        mine += ((got - want) ** 2).sum()
        segments += ((_sum_in_segments(val, dense[col], groups) - want) ** 2).sum()
    assert mine ** 0.5 <= 1.05 * segments ** 0.5


def _into_nan(csr, B, longest, plans):
    """rode_hip_spmm_new into a C full of NaN."""
    from rode_amd import _lib
    code = {torch.float32: 0, torch.float16: 1, torch.float64: 2}[B.dtype]
    out = torch.full((csr.m, B.shape[1]), float("nan"), dtype=csr.values.dtype, device=B.device)
    assert _lib.load().rode_hip_spmm_new(code, csr.m, longest, csr.m1, csr.m2, csr.n, B.shape[1], csr.values.data_ptr(), csr.column_indices.data_ptr(),
                                         csr.row_offsets.data_ptr(), csr.block_indices.data_ptr(), csr.residue_indices.data_ptr(),
                                         csr.st_offsets.data_ptr(), B.data_ptr(), out.data_ptr(), ctypes.addressof(plans),
                                         torch.cuda.current_stream().cuda_stream) == 0
    return out.double().cpu().numpy()


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("long_rows,longest", [(60, 380), (400, 1000)])  # fewer than 1024 segments, summed in parts; more
def test_new_product_with_column_tiles_dealt_out(long_rows, longest, half):
    """Tiles of C dealt out to the XCDs and rows without slots zeroed in the same launch: block segments, tails and empty rows."""
    import oracle
    from gpu_common import DEV, round_half
    from rode_amd import RoDeCSR
    rng = np.random.default_rng(long_rows)
    m, n, k = 20000, 20000, 128
    lens = rng.integers(4, 20, m)
    lens[rng.choice(m, long_rows, replace=False)] = rng.integers(100, longest - 3, long_rows)
    lens[rng.choice(m, m // 10, replace=False)] = 0
    rp = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    row = np.repeat(np.arange(m), lens)
    col = ((np.arange(len(row)) - rp[row]) * n // np.maximum(lens[row], 1) + rng.integers(0, 20, len(row))).astype(np.int32)  # (ascending, distinct)
    val, dense = rng.uniform(-1, 1, len(col)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
    dense = round_half(dense) if half else dense
    csr = RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col), torch.from_numpy(val), DEV, m, n, k, config="auto")
    assert csr.plan is None and not csr.columns_local and csr.longest_row <= longest and (csr.m1 >= 1024) == (long_rows == 400)
    # where tiles are dealt out: 2, 4 or 8 lines of 128 bytes a row, more than 4 MB, up to 9 MB a tile, few segments, 6 nonzeros a dense row
    size = n * k * (2 if half else 4)
    assert size > 4 << 20 and n * 128 <= 9 << 20 and 3 * csr.m1 <= csr.m2 and csr.nnz >= 6 * n
    want, scale = oracle.spmm_f64(rp, col, val, dense, with_abs=True)
    got = _into_nan(csr, torch.from_numpy(dense).to(DEV, torch.float16 if half else torch.float32), csr.longest_row, csr.call_plans())
    assert (np.abs(got - want) <= scale * (lens[:, None] + 2) * 2.0 ** -24).all()  # (n + 2 roundings)


@pytest.mark.parametrize("kind,k,dtype", [(kind, k, dtype) for kind in ("group", "hub", "hub without scratch", "window")
                                          for k, dtype in ((64, "f32"), (128, "f16"), (200, "f32"), (32, "f64"), (64, "f64"))])
def test_new_product_with_plans(kind, k, dtype):
    """rode_hip_spmm_new into NaN with each kind of plan, in matrices with empty rows: C is what it should be in every row, known
    longest row or not."""
    import oracle
    from gpu_common import DEV, round_half
    from rode_amd import RoDeCSR, rode_sddmm_hip
    rng = np.random.default_rng(k)
    if kind == "group":  # runs of 100 columns, with other columns beside them
        m, n = 1000, 1300
        rows = [np.union1d(np.arange(r, r + 100), rng.choice(n, 12, replace=False)) for r in range(m)]
    elif kind == "window":
        m, n = 3000, 3000
        rows = [np.unique(np.clip(r + rng.integers(-100, 100, 20), 0, n - 1)) for r in range(m)]
    else:
        m, n = 2500, 70000
        rows = [np.unique(rng.integers(0, n, L)) for L in np.where(rng.random(m) < 0.3, rng.integers(540, 600, m), rng.integers(0, 70, m))]
        for r in (5, 77, 900):
            rows[r] = np.unique(rng.integers(0, n, 6000))
    for r in (0, 1, 2, 3, 50, 51, 64, 999, m - 1):  # (among them all rows of a group)
        rows[r] = rows[r][:0]
    lens = np.array([len(r) for r in rows])
    rp, col = np.concatenate(([0], np.cumsum(lens))).astype(np.int32), np.concatenate(rows).astype(np.int32)
    val, dense = rng.uniform(-1, 1, len(col)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
    dense = round_half(dense) if dtype == "f16" else dense
    old = RoDeCSR.HUB_MIN_SLABS
    RoDeCSR.HUB_MIN_SLABS = 1 if "hub" in kind else 10 ** 6
    try:
        csr = RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col), torch.from_numpy(val), DEV, m, n, k, locality=True)
    finally:
        RoDeCSR.HUB_MIN_SLABS = old
    assert isinstance(csr.plan, {"group": rode_sddmm_hip.GroupPlan, "window": rode_sddmm_hip.WindowPlan}.get(kind, rode_sddmm_hip.HubPlan))
    if dtype == "f64":
        csr = csr.with_values(csr.values.double())
    B = torch.from_numpy(dense).to(DEV, {"f32": torch.float32, "f16": torch.float16, "f64": torch.float64}[dtype])
    plans, scratch = csr.call_plans(), None
    if kind == "hub":
        plans, scratch = rode_sddmm_hip._with_scratch(plans, k, csr.values.element_size(), csr.device)
        assert scratch.numel() > 0
    want, scale = oracle.spmm_f64(rp, col, val, dense, with_abs=True)
    for longest in (csr.longest_row, 0):
        got = _into_nan(csr, B, longest, plans)
        assert (np.abs(got - want) <= scale * (lens[:, None] + 2) * (2.0 ** -52 if dtype == "f64" else 2.0 ** -24)).all()


@pytest.mark.parametrize("k,dtype", [(32, "f32"), (64, "f32"), (96, "f32"), (128, "f32"), (200, "f32"), (32, "f16"), (64, "f16"), (128, "f16"), (64, "f64")])
@pytest.mark.parametrize("seg,said", [(128, 128), (32, 32), (512, 128)])
def test_long_rows_by_a_workgroup_each(seg, said, k, dtype):
    """Rows of 1000 to 4096 aligned slots (3072, 2048 where tiles are wider), which the waves of a workgroup share, into NaN: at the bounds of
    what one wave sums (1024), of a part (512 of a quarter) and of the row, at every place in a workgroup, first and last in the lists, next to each other and beside
    empty rows; and, where the segments are longer than said, rows that have no workgroup.  NaN and Inf in dense rows that no long row uses."""
    import oracle
    from gpu_common import DEV, round_half
    from rode_amd import RoDeCSR, rode_sddmm_hip
    rng = np.random.default_rng(seg + k)
    long_ones = [4090, 1024, 1025, 1026, 1023, 1027, 1030, 2047, 2048, 2049, 2052, 3000, 4093, 1100, 1300, 1537, 1800, 2560, 4089]
    dealt = (k, dtype, seg) == (128, "f32", 128)  # (column tiles dealt out to the XCDs: 4 MB of dense rows, few segments beside the tails)
    m, n = (8000, 9000) if dealt else (3000, 6000)
    lens = rng.integers(0, 36 if dealt else 70, m)
    lens[rng.choice(m, m // 8, replace=False)] = 0
    lens[0], lens[-1] = 4080, 2200
    at = np.arange(40, 40 + 97 * len(long_ones), 97)
    lens[at] = long_ones
    lens[at[5] + 1: at[5] + 3] = 1200, 1500
    lens[at[7] - 1] = lens[at[7] + 1] = 0
    most = {(64, "f32"): 3072, (128, "f16"): 3072, (128, "f32"): 4096 if dealt else 2048, (64, "f64"): 2048}.get((k, dtype), 4096)
    lens = np.minimum(lens, most - 3)
    rp = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n - 1, L, replace=False)) for L in lens]).astype(np.int32)
    short = np.flatnonzero((lens > 0) & (lens < 1000))[17]
    col[rp[short + 1] - 1] = n - 1  # the one nonzero of the last column
    val, dense = rng.uniform(-1, 1, len(col)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
    dense = round_half(dense) if dtype == "f16" else dense
    dense[n - 1] = np.inf
    csr = RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col), torch.from_numpy(val), DEV, m, n, k, config={"seg_length": seg, "k_block": 32, "vec_len": 4},
                  locality=False)
    csr = csr.with_values(csr.values.double()) if dtype == "f64" else csr
    assert csr.m1 >= 1024 and (not dealt or 3 * csr.m1 <= csr.m2)  # (as many segments as the rule for whole rows wants)
    assert most - 3 <= csr.longest_row <= most
    B = torch.from_numpy(dense).to(DEV, {"f32": torch.float32, "f16": torch.float16, "f64": torch.float64}[dtype])
    got = _into_nan(csr, B, csr.longest_row, rode_sddmm_hip.plans_struct(None, whole_lists=True, seg_length=said))
    assert not np.isfinite(got[short]).any()
    dense[n - 1] = 0
    want, scale = oracle.spmm_f64(rp, col, val, dense, with_abs=True)
    got[short] = want[short]
    # roundings of a sum: 512 slots over two lane groups, seven more parts, the groups (5), the waves (3) and the product
    assert (np.abs(got - want) <= scale * (256 + 7 + 5 + 3 + 1) * (2.0 ** -53 if dtype == "f64" else 2.0 ** -24)).all()


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("m,n,mean,k", [(300, 500, 20, 96), (300, 500, 20, 224), (2000, 16500, 30, 96), (20000, 20000, 8, 96), (17000, 17000, 6, 160), (500, 215000, 20, 96)])
def test_tiles_that_are_not_the_least_padded(m, n, mean, k, half):
    """Widths of 32 (2 i + 1) columns, where the tile follows from the sizes of the call: 32, 64 or 128 columns, the last tile part of one; into NaN."""
    import oracle
    from gpu_common import DEV, round_half
    from rode_amd import RoDeCSR
    rng = np.random.default_rng(m + k)
    lens = rng.integers(0, 2 * mean, m)
    lens[m // 2], lens[m // 3] = 400, 1500 if n > 1500 else 450
    rp = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    row = np.repeat(np.arange(m), lens)
    col = ((np.arange(len(row)) - rp[row]) * n // np.maximum(lens[row], 1)).astype(np.int32)  # (ascending, distinct, far apart)
    val, dense = rng.uniform(-1, 1, len(col)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
    dense = round_half(dense) if half else dense
    csr = RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col), torch.from_numpy(val), DEV, m, n, k, config="auto", locality=False)
    want, scale = oracle.spmm_f64(rp, col, val, dense, with_abs=True)
    got = _into_nan(csr, torch.from_numpy(dense).to(DEV, torch.float16 if half else torch.float32), csr.longest_row, csr.call_plans())
    assert (np.abs(got - want) <= scale * (lens[:, None] + 2) * 2.0 ** -24).all()  # (n + 2 roundings)


@pytest.mark.parametrize("half,width,rows,degree", [(True, 96, 8000, 40), (True, 160, 16000, 110), (True, 224, 12000, 40), (True, 96, 30000, 14), (True, 96, 16000, 300),
                                                    (False, 96, 4000, 40), (False, 224, 2000, 60)])
def test_wider_tiles_are_as_exact_as_those_of_32_columns(half, width, rows, degree):
    """2-norms of the errors against fp64, of the product and of the same columns 32 at a time. Of 448 000 and more elements each is known to
    0.1 %, and with sums of eight slots the wider tiles' are smaller (0.97 to 1.004); one chain over a lane group's slots had 1.09 to 1.38 times the error."""
    from gpu_common import DEV
    from rode_amd import RoDeCSR, rode_spmm
    gen = torch.Generator(device=DEV).manual_seed(width + degree)
    lens = torch.poisson(torch.full((rows,), float(degree), device=DEV), generator=gen).long()
    ro = torch.cat((torch.zeros(1, dtype=torch.int64, device=DEV), lens.cumsum(0)))
    row, nnz = torch.arange(rows, device=DEV).repeat_interleave(lens), int(ro[-1])
    col = torch.sort(torch.randint(0, rows, (nnz,), device=DEV, generator=gen) + row * rows)[0] % rows
    csr = RoDeCSR(ro.int().cpu(), col.int(), torch.rand(nnz, device=DEV, generator=gen) * 2 - 1, DEV, rows, rows, width, config="auto")
    B = torch.randn(rows, width, device=DEV, generator=gen).to(torch.float16 if half else torch.float32)
    want = torch.zeros(rows, width, dtype=torch.float64, device=DEV)
    for at in range(0, nnz, 1 << 19):
        part = slice(at, at + (1 << 19))
        want.index_add_(0, row[part], csr.values[part, None].double() * B[col[part]].double())
    narrow = torch.cat([rode_spmm(csr, B[:, at:at + 32].contiguous()) for at in range(0, width, 32)], 1)
    assert (rode_spmm(csr, B).double() - want).norm() <= 1.01 * (narrow.double() - want).norm()


@pytest.mark.parametrize("half,width,rows,degree,longest", [(True, 96, 12000, 14, 900), (True, 160, 4000, 32, 1020), (False, 96, 4000, 32, 1020), (False, 224, 2000, 56, 1000)])
def test_a_long_row_in_a_small_matrix_keeps_the_narrow_tiles(half, width, rows, degree, longest):
    """One wave has all of a row of up to 1024 slots, and twice to four times as long for it with wider tiles: the same bits as 32 columns at a time.
    (12 K rows of 14 halves x 96, longest 899: 11.4 us, and 16.3 with tiles of 128 columns.)"""
    from gpu_common import DEV
    from rode_amd import RoDeCSR, rode_spmm
    gen = torch.Generator(device=DEV).manual_seed(rows)
    lens = torch.randint(degree // 2, degree + degree // 2, (rows,), device=DEV, generator=gen)
    lens[::8], lens[rows // 2] = 100, longest
    ro = torch.cat((torch.zeros(1, dtype=torch.int64, device=DEV), lens.cumsum(0)))
    col = torch.randint(0, rows, (int(ro[-1]),), device=DEV, generator=gen).int()
    csr = RoDeCSR(ro.int().cpu(), col, torch.rand(col.numel(), device=DEV, generator=gen), DEV, rows, rows, width, config="auto")
    assert csr.m1 >= 1024  # (rows with one work item each: no sum depends on the order of several)
    B = torch.randn(rows, width, device=DEV, generator=gen).to(torch.float16 if half else torch.float32)
    narrow = torch.cat([rode_spmm(csr, B[:, at:at + 32].contiguous()) for at in range(0, width, 32)], 1)
    assert torch.equal(rode_spmm(csr, B), narrow)


@pytest.mark.parametrize("k,dtype", [(32, "f32"), (64, "f32"), (128, "f32"), (64, "f16"), (128, "f16"), (64, "f64")])
def test_rows_of_thousands_of_slots_by_a_workgroup_each(k, dtype):
    """Rows of 5 000 to 20 000 aligned slots in segments of 512, which the rule leaves to workgroups in matrices with 2 GB to gather (said of a smaller one): quarters
    of two to ten parts.  Not the bits of adding their segments up, and none left of what C held."""
    import oracle
    from gpu_common import DEV, round_half
    from rode_amd import RoDeCSR, rode_sddmm_hip
    rng = np.random.default_rng(k)
    m, n = 3000, 24000
    lens = rng.integers(0, 70, m)
    long_ones = np.arange(100, 900, 100)
    lens[long_ones] = 5000, 6656, 19990, 8191, 8193, 12001, 4097, 16001
    rp = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, L, replace=False)) for L in lens]).astype(np.int32)
    val, dense = rng.uniform(-1, 1, len(col)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
    dense = round_half(dense) if dtype == "f16" else dense
    csr = RoDeCSR(torch.from_numpy(rp), torch.from_numpy(col), torch.from_numpy(val), DEV, m, n, k, config={"seg_length": 512, "k_block": 32, "vec_len": 4},
                  locality=False)
    csr = csr.with_values(csr.values.double()) if dtype == "f64" else csr
    assert csr.m1 >= 1024 and 19990 <= csr.longest_row <= 20000
    B = torch.from_numpy(dense).to(DEV, {"f32": torch.float32, "f16": torch.float16, "f64": torch.float64}[dtype])
    plans = rode_sddmm_hip.plans_struct(None, whole_lists=True, seg_length=512, nonzeros=2_000_000_000 // (k * B.element_size()))
    got, added = (_into_nan(csr, B, longest, plans) for longest in (csr.longest_row, 0))
    assert not np.array_equal(got[long_ones], added[long_ones])
    want, scale = oracle.spmm_f64(rp, col, val, dense, with_abs=True)
    # roundings of a sum: 512 slots over two lane groups, nine more parts, the groups (5), the waves (3) and the product
    assert (np.abs(got - want) <= scale * (256 + 9 + 5 + 3 + 1) * (2.0 ** -53 if dtype == "f64" else 2.0 ** -24)).all()


@pytest.mark.parametrize("half,width,tiles", [(False, 48, 64), (False, 100, 128), (False, 40, 64), (True, 48, 64), (True, 104, 128)])
def test_widths_that_are_no_multiple_of_32_are_summed_as_those_that_are(half, width, tiles):
    """Tiles of that many columns are theirs anyway: the bits of the same columns of a whole tile, not sums of eight slots (rows of 30 on average, lognormal,
    100 K x 48: 93.3 us, and 100.2 with those)."""
    from gpu_common import DEV
    from rode_amd import RoDeCSR, rode_spmm
    gen = torch.Generator(device=DEV).manual_seed(width)
    rows = 3000
    lens = torch.randint(33, 120, (rows,), device=DEV, generator=gen)
    ro = torch.cat((torch.zeros(1, dtype=torch.int64, device=DEV), lens.cumsum(0)))
    col = torch.randint(0, rows, (int(ro[-1]),), device=DEV, generator=gen).int()
    csr = RoDeCSR(ro.int().cpu(), col, torch.rand(col.numel(), device=DEV, generator=gen), DEV, rows, rows, width, config="auto")
    assert csr.m1 >= 1024  # (rows with one work item each)
    B = torch.randn(rows, tiles, device=DEV, generator=gen).to(torch.float16 if half else torch.float32)
    assert torch.equal(rode_spmm(csr, B[:, :width].contiguous()), rode_spmm(csr, B)[:, :width])


@pytest.mark.parametrize("rows,degree,width,wide", [(4000, 60, 96, True), (12000, 30, 224, True), (30000, 22, 96, True), (4000, 14, 96, False)])
def test_rows_of_equal_length_take_the_wider_tiles(rows, degree, width, wide):
    """No long row is waited for there, in calls too whose rows are all stored, which do not say their longest (4000 rows of 60 halves x 96: 6.4 us, 8.9 in
    tiles of 32 columns): not the bits of the same columns 32 at a time, but where rows are tails of a small matrix."""
    from gpu_common import DEV
    from rode_amd import RoDeCSR, rode_spmm
    gen = torch.Generator(device=DEV).manual_seed(rows + degree)
    lens = torch.poisson(torch.full((rows,), float(degree), device=DEV), generator=gen).long().clamp(min=4, max=2 * degree - 6)
    ro = torch.cat((torch.zeros(1, dtype=torch.int64, device=DEV), lens.cumsum(0)))
    col = torch.randint(0, rows, (int(ro[-1]),), device=DEV, generator=gen).int()
    csr = RoDeCSR(ro.int().cpu(), col, torch.rand(col.numel(), device=DEV, generator=gen), DEV, rows, rows, width, config="auto")
    assert csr.equal_rows == col.numel() // rows
    B = torch.randn(rows, width, device=DEV, generator=gen).half()
    narrow = torch.cat([rode_spmm(csr, B[:, at:at + 32].contiguous()) for at in range(0, width, 32)], 1)
    got = rode_spmm(csr, B)
    assert torch.equal(got, narrow) != wide
    assert (got - narrow).abs().max() <= 1e-5 * narrow.abs().max()


def test_longest_rows_with_partial_tiles_are_added_to():
    """Rows of 12 000 slots in a matrix with 1.3 GB to gather, width 100: not by a workgroup each (30 K rows of 110: 154 us added to, 166 stored), of 6000 they are.
    Said of a smaller matrix; what is by a workgroup is summed in quarters."""
    from gpu_common import DEV
    from rode_amd import RoDeCSR, rode_sddmm_hip
    gen = torch.Generator(device=DEV).manual_seed(0)
    rows, width = 3000, 100
    lens = torch.randint(33, 60, (rows,), device=DEV, generator=gen)
    lens[5] = 5996
    ro = torch.cat((torch.zeros(1, dtype=torch.int64, device=DEV), lens.cumsum(0))).int().cpu()
    col = torch.randint(0, 20000, (int(ro[-1]),), device=DEV, generator=gen).int()
    csr = RoDeCSR(ro, col, torch.rand(col.numel(), device=DEV, generator=gen), DEV, rows, 20000, width, locality=False, config="auto")
    B = torch.randn(20000, width, device=DEV, generator=gen)
    plans = rode_sddmm_hip.plans_struct(None, whole_lists=True, seg_length=csr.config["seg_length"], nonzeros=1_300_000_000 // (width * 4))
    short, long_one, added = (torch.from_numpy(_into_nan(csr, B, longest, plans)) for longest in (6000, 12000, 0))
    others = torch.arange(rows) != 5
    assert torch.equal(short[others], added[others]) and torch.equal(long_one[others], added[others])
    assert not torch.equal(short[5], long_one[5]) and not torch.equal(short[5], added[5])  # (adding its segments up has another order)
    part = csr.values[ro[5]:ro[6]].double(), B[col[ro[5]:ro[6]].long()].double()
    # roundings of a sum: 512 slots over two lane groups, up to 47 segments, the groups (5), the waves (3) and the product
    bound = (part[0] @ part[1].abs()).cpu() * (256 + 47 + 5 + 3 + 1) * 2.0 ** -24
    assert all(((C[5] - (part[0] @ part[1]).cpu()).abs() <= bound).all() for C in (short, long_one, added))
