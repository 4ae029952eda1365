"""Hub plan: rows with thousands of nonzeros are processed column slab by column slab by
kernels of their own (rode_hub.hip, spmm_hub_kernel, sddmm_hub_kernel).  The plan changes
where dense rows are found, never a result: everything here is checked against the fp64
oracle with the tolerances of the unplanned kernels."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _matrix(rng, m, n, hub_lens, sort_hubs=True, mean_len=20):
    """Short rows plus a few very long ones (sorted columns unless asked otherwise)."""
    lens = rng.poisson(mean_len, m)
    where = rng.choice(m, len(hub_lens), replace=False)
    lens[where] = hub_lens
    rp = np.zeros(m + 1, dtype=np.int32)
    rp[1:] = np.cumsum(lens)
    col = np.empty(rp[-1], dtype=np.int32)
    for r in range(m):
        c = rng.choice(n, lens[r], replace=False)
        col[rp[r]:rp[r + 1]] = np.sort(c) if (sort_hubs or lens[r] < 1000) else c
    val = rng.uniform(-1, 1, rp[-1]).astype(np.float32)
    return rp, col, val, np.sort(where)


def test_plan_contents():
    from rode_amd import rode_sddmm_hip
    rng = np.random.default_rng(0)
    m, n = 3000, 50000
    rp, col, val, where = _matrix(rng, m, n, [5000, 9000, 4096, 4095, 20000])
    dev = torch.device("cuda:0")
    plan = rode_sddmm_hip.hub_plan(torch.from_numpy(rp).to(dev), torch.from_numpy(col).to(dev), m, n, 4096)
    lens = np.diff(rp) + rp[:-1] % 4
    hubs = np.nonzero(lens >= 4096)[0]
    assert plan.usable and plan.counts[0] == len(hubs) and plan.counts[1] == (n + 2047) // 2048 and plan.counts[2] == 4096
    assert np.array_equal(plan.hub_rows(), hubs)
    pieces = plan.pieces()
    for h, r in enumerate(hubs):
        c = col[rp[r]:rp[r + 1]]
        want = rp[r] + np.searchsorted(c, np.arange(plan.counts[1] + 1) * 2048, side="left")
        want[-1] = rp[r + 1]
        assert np.array_equal(pieces[h], want)
    # a hub row whose columns do not ascend makes the plan unusable
    rp2, col2, _, _ = _matrix(rng, 500, 40000, [6000], sort_hubs=False)
    bad = rode_sddmm_hip.hub_plan(torch.from_numpy(rp2).to(dev), torch.from_numpy(col2).to(dev), 500, 40000, 4096)
    assert bad.counts[0] == 1 and not bad.usable
    # no hub rows at all
    none = rode_sddmm_hip.hub_plan(torch.from_numpy(rp2).to(dev), torch.from_numpy(col2).to(dev), 500, 40000, 100000)
    assert none.counts[0] == 0 and not none.usable


@pytest.mark.parametrize("k,half", [(128, False), (64, False), (32, False), (128, True), (200, False)])
def test_hub_rows_against_oracle(k, half):
    """A matrix whose long rows the hub kernels take (min_len lowered so that pieces of one
    nonzero, empty pieces and pieces of hundreds occur), every width class and fp16."""
    import oracle
    from gpu_common import TOL_F16, TOL_F32, make_csr, round_half, run_sddmm, run_spmm
    from helpers import spmm_row_l1_error, sddmm_row_l1_errors
    from rode_amd import RoDeCSR, rode_sddmm_hip
    rng = np.random.default_rng(k)
    m, n = 2000, 70000
    rp, col, val, where = _matrix(rng, m, n, [5000, 300, 64, 12000, 700, 65, 33000])
    old = RoDeCSR.HUB_MIN_LEN, RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE
    RoDeCSR.HUB_MIN_LEN, RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = 64, 1, 0.0
    try:
        csr = make_csr(rp, col, val, m, n, k)
    finally:
        RoDeCSR.HUB_MIN_LEN, RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = old
    assert isinstance(csr.plan, rode_sddmm_hip.HubPlan) and csr.plan.usable
    assert csr.plan.counts[2] == max(64, 8 * ((n + 4095) // 4096)) and csr.plan.counts[0] >= 5
    B = rng.standard_normal((n, k)).astype(np.float32)
    L = rng.standard_normal((m, k)).astype(np.float32)
    Bq, Lq = (round_half(B), round_half(L)) if half else (B, L)
    tol = TOL_F16 if half else TOL_F32
    assert spmm_row_l1_error(run_spmm(csr, B, half), oracle.spmm_f64(rp, col, val, Bq)) <= tol
    if k == 64:  # fp64 through the same plan, and accumulation into a C that is not zero
        from rode_amd import rode_sddmm_hip
        dev = csr.device
        C0 = torch.from_numpy(rng.standard_normal((m, k))).to(dev)
        C = C0.clone()
        rode_sddmm_hip.spmm_forward(csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2,
                                    csr.row_offsets, csr.column_indices, csr.values.double(), m, n,
                                    torch.from_numpy(B).to(dev).double(), out=C, plan=csr.plan)
        ref = oracle.spmm_f64(rp, col, val, B)
        added = (np.diff(rp) + rp[:-1] % 4) >= 32  # long rows are added to, short rows overwritten
        want = ref + np.where(added[:, None], C0.cpu().numpy(), 0.0)
        assert spmm_row_l1_error(C.cpu().numpy(), want) <= 1e-12
    ref64, scale = oracle.sddmm_f64(rp, col, val, Lq, Bq, with_abs=True)
    out = run_sddmm(csr, L, B, half)
    err, cond = sddmm_row_l1_errors(out, ref64, scale, rp)
    assert float(err[cond <= 100].max(initial=0.0)) <= tol
    if not half:
        assert (np.abs(out - ref64) / np.maximum(scale, 1e-30)).max() <= 2e-6


@pytest.mark.parametrize("k", [64, 32])
def test_hub_plan_through_the_c_abi(k):
    """The planned entry points with a hub plan against the same calls without one; the
    atomic fallback of SpMM (no workspace); what is refused.  (k = 32: rows of one 128-byte
    tile, for which a locality plan is ignored - a hub plan and the flags are not.)"""
    import ctypes
    from gpu_common import DEV, make_csr
    from rode_amd import RoDeCSR, _lib, rode_sddmm_hip
    lib = _lib.load()
    rng = np.random.default_rng(3)
    m, n = 1500, 40000
    rp, col, val, _ = _matrix(rng, m, n, [4500, 8000, 2000])
    csr = make_csr(rp, col, val, m, n, k, locality=False)
    assert csr.plan is None
    plan = rode_sddmm_hip.hub_plan(csr.row_offsets, csr.column_indices, m, n, 2000)
    assert plan.usable and plan.counts[0] == 3
    B = torch.from_numpy(rng.standard_normal((n, k)).astype(np.float32)).to(DEV)
    L = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(DEV)

    def plans(hub, ws=None, window=None):
        p = _lib.Plans()
        if hub:
            p.hub, p.hub_counts = plan.data.data_ptr(), ctypes.addressof(plan._header)
        if ws is not None:
            p.hub_workspace, p.hub_workspace_bytes = ws.data_ptr(), ws.numel()
        if window is not None:
            p.window, p.window_rows = window.data_ptr(), window.data_ptr()
        return p

    def spmm(flags, hub, ws):
        C = torch.zeros(m, k, device=DEV)
        code = lib.rode_hip_spmm_planned(0, flags, csr.m1, csr.m2, n, k, csr.values.data_ptr(), csr.column_indices.data_ptr(),
                                         csr.row_offsets.data_ptr(), csr.block_indices.data_ptr(),
                                         csr.residue_indices.data_ptr(), csr.st_offsets.data_ptr(), B.data_ptr(),
                                         C.data_ptr(), ctypes.byref(plans(hub, ws)), None, None)
        torch.cuda.synchronize()
        return code, C

    code, plain = spmm(_lib.SPMM_WHOLE_LISTS, False, None)
    assert code == 0
    ws = plan.workspace(k, 4)
    assert ws.numel() == lib.rode_hip_hub_workspace_bytes(ctypes.addressof(plan._header), k, 4) > 0
    scale = plain.abs().max().item()
    for workspace in (ws, None, ws[: ws.numel() // 2]):  # partial rows; atomics; too small a workspace -> atomics
        code, got = spmm(_lib.SPMM_WHOLE_LISTS, True, workspace)
        assert code == 0 and (got - plain).abs().max().item() <= 2e-5 * scale
    # the three kernel families one by one add up to the whole
    parts = [spmm(_lib.SPMM_WHOLE_LISTS | f, True, ws) for f in (_lib.SPMM_ONLY_BLOCK, _lib.SPMM_ONLY_RESIDUE, _lib.SPMM_ONLY_HUB)]
    assert all(c == 0 for c, _ in parts)
    assert (sum(p for _, p in parts) - plain).abs().max().item() <= 2e-5 * scale
    # refused: a hub plan without the whole-lists promise, two ONLY bits, a hub plan next to a locality plan
    assert spmm(0, True, ws)[0] != 0
    assert spmm(_lib.SPMM_WHOLE_LISTS | _lib.SPMM_ONLY_BLOCK | _lib.SPMM_ONLY_HUB, True, ws)[0] != 0

    def sddmm(flags, hub, window=None):
        out = torch.full((len(val),), float("nan"), device=DEV)
        code = lib.rode_hip_sddmm_planned(0, flags, csr.m1, csr.m2, n, k, csr.block_indices.data_ptr(),
                                          csr.residue_indices.data_ptr(), csr.st_offsets.data_ptr(),
                                          csr.row_offsets.data_ptr(), csr.column_indices.data_ptr(), csr.values.data_ptr(),
                                          L.data_ptr(), B.data_ptr(), out.data_ptr(), ctypes.byref(plans(hub, None, window)),
                                          None, None)
        torch.cuda.synchronize()
        return code, out

    code, plain_out = sddmm(0, False)
    code2, hub_out = sddmm(0, True)
    assert code == 0 and code2 == 0 and not torch.isnan(hub_out).any()
    assert (hub_out - plain_out).abs().max().item() <= 2e-5 * plain_out.abs().max().item()
    # every output is written by exactly one of the three kernel families
    written = [~torch.isnan(sddmm(f, True)[1]) for f in (_lib.SPMM_ONLY_BLOCK, _lib.SPMM_ONLY_RESIDUE, _lib.SPMM_ONLY_HUB)]
    assert (written[0].int() + written[1].int() + written[2].int() == 1).all()
    fake = torch.zeros(64, dtype=torch.int32, device=DEV)
    assert sddmm(0, True, fake)[0] != 0


@pytest.mark.parametrize("hubs,k,half", [(2, 64, False), (40, 128, False), (300, 128, False), (1200, 128, True), (2300, 64, False), (4600, 128, False)])
def test_pieces_shared_by_waves(hubs, k, half):
    """Pieces shared by the waves of a workgroup, with pieces of one nonzero, empty ones and some that several waves have a part
    of.  (How many waves and pieces: test_pieces_per_workgroup.)"""
    import oracle
    from gpu_common import TOL_F16, TOL_F32, make_csr, round_half, run_sddmm, run_spmm
    from helpers import spmm_row_l1_error, sddmm_row_l1_errors
    from rode_amd import RoDeCSR
    rng = np.random.default_rng(hubs)
    m, n = 5000, 70000
    lens = rng.integers(150, 400, hubs)
    lens[:2] = 30000, 7000
    rp, col, val, where = _matrix(rng, m, n, lens)
    old = RoDeCSR.HUB_MIN_LEN, RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE
    RoDeCSR.HUB_MIN_LEN, RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = 64, 1, 0.0
    try:
        csr = make_csr(rp, col, val, m, n, k)
    finally:
        RoDeCSR.HUB_MIN_LEN, RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = old
    assert csr.plan.counts[0] >= hubs
    B = rng.standard_normal((n, k)).astype(np.float32)
    L = rng.standard_normal((m, k)).astype(np.float32)
    Bq, Lq = (round_half(B), round_half(L)) if half else (B, L)
    tol = TOL_F16 if half else TOL_F32
    got = run_spmm(csr, B, half)
    assert spmm_row_l1_error(got, oracle.spmm_f64(rp, col, val, Bq)) <= tol
    assert np.array_equal(got[where], run_spmm(csr, B, half)[where])  # (a piece's parts are added in one order)
    ref, scale = oracle.sddmm_f64(rp, col, val, Lq, Bq, with_abs=True)
    err, cond = sddmm_row_l1_errors(run_sddmm(csr, L, B, half), ref, scale, rp)
    assert float(err[cond <= 100].max(initial=0.0)) <= tol


@pytest.mark.parametrize("way", ["streams", "threads", "graph"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.float64])
def test_calls_on_one_matrix_from_two_streams(dtype, way):
    """Overlapping products of one matrix have partial rows of their own - on two streams, from two threads on one, and in the replays of
    a captured graph: every result is the one that the call gives alone.
    (Rows of the plan are summed in one order whatever else runs, so the bits are equal.)"""
    import threading
    from gpu_common import DEV, make_csr
    from rode_amd import RoDeCSR, rode_sddmm_hip, rode_spmm
    rng = np.random.default_rng(17)
    m, n, k = 3000, 70000, 128
    lens = rng.integers(600, 900, 700)
    lens[:2] = 30000, 7000
    rp, col, val, where = _matrix(rng, m, n, lens)
    old = RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE
    RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = 1, 0.0
    try:
        csr = make_csr(rp, col, val, m, n, k)
    finally:
        RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = old
    assert csr.plan.usable and csr.plan.counts[0] == len(where)
    where = torch.from_numpy(where).to(DEV)
    operands = [torch.from_numpy(rng.standard_normal((n, k))).to(DEV, dtype) for _ in range(2)]

    def product(B):
        if dtype == torch.float64:
            return rode_sddmm_hip.spmm_forward(csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2, csr.row_offsets,
                                               csr.column_indices, csr.values.double(), m, n, B, plan=csr.plan)
        return rode_spmm(csr, B)

    alone = [product(B)[where] for B in operands]
    torch.cuda.synchronize()
    got = [[], []]
    if way == "streams":
        streams = [torch.cuda.Stream() for _ in operands]
        for _ in range(8):
            for i, (s, B) in enumerate(zip(streams, operands)):
                with torch.cuda.stream(s):
                    got[i].append(product(B)[where])
    elif way == "threads":
        def calls(i):
            got[i].extend(product(operands[i])[where] for _ in range(8))
        threads = [threading.Thread(target=calls, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert len(got[0]) == len(got[1]) == 8
    else:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = [product(B)[where] for B in operands]
        for _ in range(4):
            graph.replay()
            got[0].append(product(operands[0])[where])  # (the program's own work between the replays)
            for g, c in zip(got, captured):
                g.append(c.clone())
            torch.cuda.synchronize()
    torch.cuda.synchronize()
    assert not torch.equal(*alone)
    assert all(torch.equal(a, alone[i]) for i in range(2) for a in got[i])
    assert csr.plan._workspaces == {}  # nothing that two calls could share is kept


@pytest.mark.parametrize("rows,k,dtype,spmm_all,sddmm_all", [
    (700, 64, "f32", True, True),      # 500 to 600 nonzeros in 5 pieces each
    (700, 128, "f16", True, True),
    (700, 512, "f32", True, False),    # SDDMM: 35 pieces; SpMM works on 128 columns at a time: 9
    (700, 512, "f16", True, True),
    (700, 200, "f32", True, True),     # no multiple of 128: 18 pieces, SDDMM wants 28 nonzeros in each, has 32
    (700, 260, "f32", True, False),    # (35)
    (700, 320, "f32", True, False),
    (300, 128, "f32", False, True),    # SpMM: too few rows share a slab
    (300, 36, "f32", False, True),
    (700, 64, "f64", True, None),
    (700, 130, "f64", True, None),
    (300, 32, "f64", False, None),
])
def test_rows_of_the_plan_that_a_call_takes(rows, k, dtype, spmm_all, sddmm_all):
    """All hub rows or the long ones (4096 slots and more), by the width of the call: which ones the hub kernels write, and the whole
    result against 64 bits, where the other rows are the list kernels'."""
    import ctypes
    import oracle
    from gpu_common import DEV, TOL_F16, TOL_F32, make_csr, round_half
    from helpers import spmm_row_l1_error
    from rode_amd import RoDeCSR, _lib, rode_sddmm_hip
    rng = np.random.default_rng(rows + k)
    m, n = 3000, 70000
    lens = rng.integers(516, 600, rows)
    lens[:5] = 4100, 4200, 5000, 6000, 4097
    rp, col, val, where = _matrix(rng, m, n, lens, mean_len=8)
    long_rows = where[np.diff(rp)[where] >= 4097]
    old = RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE
    RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = 1, 0.0
    try:
        csr = make_csr(rp, col, val, m, n, 32)
    finally:
        RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = old
    assert csr.plan.counts[0] == rows and csr.plan.counts[5] == 5
    assert csr.plan.counts[6] == np.diff(rp)[where].sum() and csr.plan.counts[7] == np.diff(rp)[long_rows].sum()
    assert np.array_equal(csr.plan.hub_rows(), where)
    half, lib, plans = dtype == "f16", _lib.load(), csr.call_plans()
    B, L = rng.standard_normal((n, k)).astype(np.float32), rng.standard_normal((m, k)).astype(np.float32)
    B, L = (round_half(B), round_half(L)) if half else (B, L)
    kind = {"f32": torch.float32, "f16": torch.float16, "f64": torch.float64}[dtype]
    values = csr.values.double() if dtype == "f64" else csr.values
    dB, dL = torch.from_numpy(B).to(DEV, kind), torch.from_numpy(L).to(DEV, kind)
    own, scratch = rode_sddmm_hip._with_scratch(plans, k, values.element_size(), csr.device)
    assert (own.hub_workspace_bytes > rows * 2 * k * values.element_size()) == spmm_all

    def spmm(flags, plans, C):
        assert lib.rode_hip_spmm_planned(_lib.DENSE_CODE[dtype], _lib.SPMM_WHOLE_LISTS | flags, csr.m1, csr.m2, n, k, values.data_ptr(),
                                         csr.column_indices.data_ptr(), csr.row_offsets.data_ptr(), csr.block_indices.data_ptr(),
                                         csr.residue_indices.data_ptr(), csr.st_offsets.data_ptr(), dB.data_ptr(), C.data_ptr(),
                                         ctypes.byref(plans), None, None) == 0
        return C.cpu().numpy()

    want, tol = oracle.spmm_f64(rp, col, val, B), 1e-12 if dtype == "f64" else TOL_F16 if half else TOL_F32
    for p in (own, plans):  # (partial rows; atomics)
        written = np.nonzero(np.abs(spmm(_lib.SPMM_ONLY_HUB, p, torch.zeros(m, k, device=DEV, dtype=values.dtype))).max(axis=1))[0]
        assert np.array_equal(written, where if spmm_all else long_rows)
        assert spmm_row_l1_error(spmm(0, p, torch.zeros(m, k, device=DEV, dtype=values.dtype)), want) <= tol
    if sddmm_all is None:
        return
    ref, scale = oracle.sddmm_f64(rp, col, val, L, B, with_abs=True)
    row = np.repeat(np.arange(m), np.diff(rp))
    stale = _lib.Plans.from_buffer_copy(plans)  # (a header made before its last three counts were: whatever rows it leads to, the result holds)
    header = (ctypes.c_int * 8)(*csr.plan.counts[:5], 0, 0, 0)
    stale.hub_counts = ctypes.addressof(header)
    for p in (plans, stale):
        for flags in (_lib.SPMM_ONLY_HUB, 0):
            out = torch.full((len(val),), float("nan"), device=DEV)
            assert lib.rode_hip_sddmm_planned(_lib.DENSE_CODE[dtype], flags, csr.m1, csr.m2, n, k, csr.block_indices.data_ptr(),
                                              csr.residue_indices.data_ptr(), csr.st_offsets.data_ptr(), csr.row_offsets.data_ptr(),
                                              csr.column_indices.data_ptr(), csr.values.data_ptr(), dL.data_ptr(), dB.data_ptr(),
                                              out.data_ptr(), ctypes.byref(p), None, None) == 0
            got = out.cpu().numpy()
            if flags and p is plans:
                assert np.array_equal(~np.isnan(got), np.isin(row, where if sddmm_all else long_rows))
            elif not flags:
                # (products and a sum of k terms: k + 2 roundings of the sum of their magnitudes at most)
                assert (np.abs(got - ref) <= (k + 2) * 2.0 ** -24 * scale).all()


@pytest.mark.parametrize("bad", ["none", "shorter", "long", "shorter, no long"])
def test_hub_rows_without_ascending_columns(bad):
    """One row of 512 to 4095 nonzeros in another order leaves a plan of the rows of 4096 and more; one of those leaves none."""
    import oracle
    from gpu_common import TOL_F32, make_csr, run_sddmm, run_spmm
    from helpers import spmm_row_l1_error
    from rode_amd import RoDeCSR
    rng = np.random.default_rng(5)
    m, n, k = 3000, 70000, 64
    lens = rng.integers(520, 600, 700)
    if bad != "shorter, no long":
        lens[:3] = 4500, 6000, 9000
    rp, col, val, where = _matrix(rng, m, n, lens, mean_len=8)
    length = np.diff(rp)
    if bad != "none":
        row = where[(length[where] > 4096) == (bad == "long")][1]
        col[rp[row]:rp[row + 1]] = rng.permutation(col[rp[row]:rp[row + 1]])
    old = RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE
    RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = 1, 0.0
    try:
        csr = make_csr(rp, col, val, m, n, k)
        if bad == "shorter, no long":  # (_may_hub asks for one; a caller of the C ABI may still want the plan)
            from rode_amd import rode_sddmm_hip
            assert not rode_sddmm_hip.hub_plan(csr.row_offsets, csr.column_indices, m, n, 512).usable
    finally:
        RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = old
    if bad in ("none", "shorter"):
        assert csr.plan.usable and csr.plan.counts[3] == (1 if bad == "none" else 2) and csr.plan.counts[5] == 3
    else:
        assert csr.plan is None or not hasattr(csr.plan, "hub_rows")
    B, L = rng.standard_normal((n, k)).astype(np.float32), rng.standard_normal((m, k)).astype(np.float32)
    assert spmm_row_l1_error(run_spmm(csr, B), oracle.spmm_f64(rp, col, val, B)) <= TOL_F32
    ref, scale = oracle.sddmm_f64(rp, col, val, L, B, with_abs=True)
    assert (np.abs(run_sddmm(csr, L, B) - ref) <= (k + 2) * 2.0 ** -24 * scale).all()


def test_plan_that_a_product_takes_no_rows_of():
    """A plan of 300 rows without a long one: SpMM leaves them to the list kernels, which add to them as
    ``rode_hip_spmm_overwrite_limit`` says (0 with a hub plan)."""
    import ctypes
    import oracle
    from gpu_common import DEV, TOL_F32, make_csr
    from helpers import spmm_row_l1_error
    from rode_amd import _lib, rode_sddmm_hip
    lib, rng = _lib.load(), np.random.default_rng(8)
    m, n, k = 3000, 70000, 64
    rp, col, val, _ = _matrix(rng, m, n, rng.integers(516, 600, 1100), mean_len=8)
    csr = make_csr(rp, col, val, m, n, k, locality=False)
    lens = np.diff(rp) + rp[:-1] % 4
    plan = rode_sddmm_hip.hub_plan(csr.row_offsets, csr.column_indices, m, n, int(np.sort(lens)[-300]))
    assert plan.usable and 300 <= plan.counts[0] < 400 and plan.counts[5] == 0 and csr.m1 >= 1024
    plans, B = rode_sddmm_hip.plans_struct(plan), rng.standard_normal((n, k)).astype(np.float32)
    assert lib.rode_hip_spmm_overwrite_limit(csr.m1, ctypes.byref(plans)) == 0
    dB, C = torch.from_numpy(B).to(DEV), torch.full((m, k), 7.0, device=DEV)
    assert lib.rode_hip_spmm_planned(0, _lib.SPMM_WHOLE_LISTS | _lib.SPMM_OVERWRITE, csr.m1, csr.m2, n, k, csr.values.data_ptr(),
                                     csr.column_indices.data_ptr(), csr.row_offsets.data_ptr(), csr.block_indices.data_ptr(),
                                     csr.residue_indices.data_ptr(), csr.st_offsets.data_ptr(), dB.data_ptr(), C.data_ptr(),
                                     ctypes.byref(plans), None, None) == 0
    C = C.cpu().numpy()
    touched = lens > 0
    want = oracle.spmm_f64(rp, col, val, B) + np.where(lens >= 32, 7.0, 0.0)[:, None]
    assert spmm_row_l1_error(C[touched], want[touched]) <= TOL_F32


@pytest.mark.parametrize("rows,n,k,dtype,waves,pieces", [
    (300, 70000, 128, "f32", 8, 1),      # the three long rows alone: 9 groups of slabs
    (1200, 70000, 128, "f32", 8, 2),
    (1200, 70000, 64, "f64", 8, 2),
    (2300, 70000, 128, "f32", 4, 2),
    (2300, 70000, 64, "f64", 4, 2),
    (4600, 70000, 128, "f32", 4, 4),
    (4600, 70000, 64, "f64", 4, 4),
    (4600, 140000, 128, "f32", 4, 8),    # 18 groups
    (4600, 140000, 64, "f64", 4, 8),
])
def test_pieces_per_workgroup(rows, n, k, dtype, waves, pieces):
    """Every number of waves and pieces that a workgroup of the hub kernels can have (by the pieces there are in all, which the
    workspace has a row each for)."""
    import oracle
    from gpu_common import DEV, make_csr
    from rode_amd import RoDeCSR, rode_sddmm_hip
    rng = np.random.default_rng(rows + n)
    m = 5000
    lens = rng.integers(0, 40, m)
    where = rng.choice(m, rows, replace=False)
    lens[where] = rng.integers(350, 420, rows) if n > 100000 else rng.integers(200, 400, rows)
    lens[where[:3]] = 30000, 7000, 4200
    rp = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    row = np.repeat(np.arange(m), lens)
    step = n // lens[row]  # (one column in every n / length: ascending, distinct)
    col = ((np.arange(len(row)) - rp[row]) * step + rng.integers(0, step)).astype(np.int32)
    val = rng.uniform(-1, 1, len(col)).astype(np.float32)
    old = RoDeCSR.HUB_MIN_LEN, RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE
    RoDeCSR.HUB_MIN_LEN, RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = 64, 1, 0.0
    try:
        csr = make_csr(rp, col, val, m, n, k)
    finally:
        RoDeCSR.HUB_MIN_LEN, RoDeCSR.HUB_MIN_SLABS, RoDeCSR.HUB_MIN_SHARE = old
    assert csr.plan.usable
    values = csr.values.double() if dtype == "f64" else csr.values
    plans, scratch = rode_sddmm_hip._with_scratch(csr.call_plans(), k, values.element_size(), csr.device)
    items = plans.hub_workspace_bytes // (k * values.element_size())
    assert waves == (4 if items >= 20000 else 8)
    assert pieces == (8 if items >= 80000 else 4 if items >= 40000 else 2 if items >= 5000 else 1)
    B = rng.standard_normal((n, k)).astype(np.float32)
    got = rode_sddmm_hip.spmm_forward(csr.block_indices, csr.residue_indices, csr.st_offsets, csr.m1, csr.m2, csr.row_offsets, csr.column_indices,
                                      values, m, n, torch.from_numpy(B).to(DEV, values.dtype), plans=plans)
    want, scale = oracle.spmm_f64(rp, col, val, B, with_abs=True)
    # (a sum of n products: n + 2 roundings of the sum of their magnitudes at most)
    assert (np.abs(got.cpu().numpy() - want) <= scale * (lens[:, None] + 2) * (2.0 ** -52 if dtype == "f64" else 2.0 ** -24)).all()
