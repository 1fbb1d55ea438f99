"""GPU tests of what runs in place of a named walk that cannot be taken: the lean
path, with the row splitting that was asked for and the limits of the call.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import lower_from_rows
from sptrsv_amd import _lib as L
from sptrsv_amd import interface as I

pytestmark = pytest.mark.gpu


def long_rows(n, length):
    """Rows without off-diagonals but for the last eight, which have `length`."""
    rng = np.random.default_rng(3)
    rows = [[] for _ in range(n)]
    for i in range(n - 8, n):
        rows[i] = sorted(rng.choice(n - 8, size=length, replace=False).tolist())
    return rows


@pytest.mark.parametrize("variant", [5, 6, 7])
@pytest.mark.parametrize("split", [-1, 0])
def test_row_splitting_is_kept(variant, split):
    ia, ja, a = lower_from_rows(long_rows(5000, 1500))
    b = np.random.default_rng(1).uniform(-1.0, 1.0, len(ia) - 1)
    mat = I.allocate_memory(ia, ja, a)
    info = I.multirow_analysis_base_GPU(mat, I.ALL)
    assert I.analysis_segments(info)[0] == 8
    if variant != 5:
        I.trace(mat, True)                          # taken by the walks row by row
    db, out = I.DeviceArray.from_numpy(b), {}
    for v in (1, variant):
        dx = I.DeviceArray(mat.nr, np.float64)
        I.solve(mat, info, I.PREC_F64, db, dx, cfg=I._cfg(kernel=I.KERNEL_MULTIROW, lanes=4, wg=256, variant=v,
                                                          split_rows=split))
        assert I.check_watchdog(mat) == 0
        out[v] = dx.numpy()
    assert np.array_equal(out[variant], out[1])
    I.free_device_analysis(mat, info)


def test_allocation_free_solve_counts_the_partials_of_what_runs():
    """The block walk does not take rows of 600 entries; the lean MULTIROW walk
    that runs instead splits them, and finds no room for the partial sums."""
    n = L.NOALLOC_MAX_WORDS
    ia = np.arange(n + 1, dtype=np.int32)
    ia[n] += 600
    ja = np.concatenate([np.arange(n - 1), np.arange(600) * 2, [n - 1]]).astype(np.int32)
    a = np.ones(len(ja))
    mat = I.allocate_memory(ia, ja, a)
    info = I.multirow_analysis_base_GPU(mat, I.ALL)
    assert I.analysis_segments(info)[0] == 1
    db, dx = I.DeviceArray.from_numpy(np.ones(n)), I.DeviceArray(n, np.float64)
    for variant in (1, 5):
        cfg = I._cfg(kernel=I.KERNEL_MULTIROW, lanes=4, wg=256, variant=variant)
        with pytest.raises(L.SptrsvError) as e:
            I.solve_mixed_noalloc(mat, info, db, dx, cfg=cfg)
        assert e.value.status == L.E_CAPACITY
        cfg.split_rows = -1
        I.solve_mixed_noalloc(mat, info, db, dx, cfg=cfg)
        assert I.check_watchdog(mat) == 0
        x = dx.numpy()
        assert np.all(x[:-1] == 1.0) and x[-1] == -599.0
    I.free_device_analysis(mat, info)
