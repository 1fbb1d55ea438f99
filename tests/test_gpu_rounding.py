"""GPU tests of the rounding error of the walks that give a row fewer lanes than
a row per wave (variant 1 with the default lanes) has: in the 2-norm, against
extended precision, on a strictly dominant matrix, it is no larger than that
walk's.
"""
from __future__ import annotations

import numpy as np
import pytest

from sptrsv_amd import interface as I

pytestmark = pytest.mark.gpu

N = 4000


def matrix(entries, reach, near, seed=1):
    """`entries` off-diagonals a row among the last `reach`, the row before
    among them where near."""
    rng = np.random.default_rng([entries, reach, seed])
    ia, ja, a = [0], [], []
    for i in range(N):
        lo = max(0, i - reach)
        cols = set(rng.choice(i - lo, size=min(entries, i - lo), replace=False) + lo) if i else set()
        if near and i and i - 1 not in cols:
            cols = set(sorted(cols)[1:]) | {i - 1}
        v = rng.uniform(-1.0, 1.0, len(cols))
        ja += sorted(int(c) for c in cols) + [i]
        a += v.tolist() + [1.0 + float(np.abs(v).sum())]
        ia.append(len(ja))
    return np.array(ia, np.int32), np.array(ja, np.int32), np.array(a)


def default_lanes(ia):
    return min(64, max(4, 1 << int(ia[-1] // N - 1).bit_length()))


def errors(ia, ja, a, k, cfgs, mode):
    b = np.random.default_rng(5).uniform(-1.0, 1.0, (N, k))
    wide, ref = a.astype(np.longdouble), np.zeros((N, k), np.longdouble)
    for i in range(N):
        s, d = ia[i], ia[i + 1] - 1
        ref[i] = (b[i] - wide[s:d] @ ref[ja[s:d]]) / wide[d]
    mat = I.allocate_memory(ia, ja, a)
    info = I.multirow_analysis_base_GPU(mat, mode)
    db, dx = I.DeviceArray.from_numpy(b.ravel()), I.DeviceArray(N * k, np.float64)
    out = []
    for cfg in cfgs:
        I.solve(mat, info, I.PREC_F64, db, dx, k=k, cfg=I._cfg(wg=256, **cfg))
        assert I.check_watchdog(mat) == 0
        e = dx.numpy().reshape(N, k) - ref
        out.append(float(np.sqrt((e * e).sum() / (ref * ref).sum())))
    I.free_device_analysis(mat, info)
    return out


@pytest.mark.parametrize("entries", [1, 2, 4, 5, 8])
def test_block_walk_of_short_rows(entries):
    ia, ja, a = matrix(entries, 200, True)
    got, bar = errors(ia, ja, a, 1, [dict(kernel=I.KERNEL_SIMPLE, lanes=4, variant=5),
                                     dict(kernel=I.KERNEL_SIMPLE, lanes=default_lanes(ia), variant=1)], I.ORDER)
    assert got <= bar


@pytest.mark.parametrize("entries", [1, 4, 8, 16, 32, 64])
def test_level_walk(entries):
    ia, ja, a = matrix(entries, 1500, False)
    got, bar = errors(ia, ja, a, 1, [dict(kernel=I.KERNEL_ORDER, lanes=4, variant=4),
                                     dict(kernel=I.KERNEL_ORDER, lanes=default_lanes(ia), variant=1)], I.ORDER)
    assert got <= bar


@pytest.mark.parametrize("entries", [1, 8, 20, 40, 64])
def test_group_walk(entries):
    ia, ja, a = matrix(entries, 1500, False)
    got, bar = errors(ia, ja, a, 1, [dict(kernel=I.KERNEL_SIMPLE, lanes=8, variant=7),
                                     dict(kernel=I.KERNEL_SIMPLE, lanes=default_lanes(ia), variant=1)], I.ORDER)
    assert got <= bar


@pytest.mark.parametrize("entries", [1, 3, 8, 20])
def test_several_right_hand_sides(entries):
    """One entry lane in level order against the general engine's default."""
    ia, ja, a = matrix(entries, 3900, False)
    got, bar = errors(ia, ja, a, 16, [dict(kernel=I.KERNEL_ORDER, lanes=1, variant=2, cu_waves=16),
                                      dict(kernel=I.KERNEL_SIMPLE, lanes=4, variant=0)], I.ORDER)
    assert got <= bar


def test_group_walk_with_more_lanes_than_entries():
    ia, ja, a = matrix(10, 1500, False)
    got, bar = errors(ia, ja, a, 1, [dict(kernel=I.KERNEL_SIMPLE, lanes=32, variant=7),
                                     dict(kernel=I.KERNEL_SIMPLE, lanes=default_lanes(ia), variant=1)], I.ORDER)
    assert got <= bar
