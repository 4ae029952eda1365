"""The native pass over the row offsets, against numpy."""
import numpy as np
import pytest
import torch

from rode_amd import _lib


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
