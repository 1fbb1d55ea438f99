"""GPU tests of the persistent level-order walk with several right-hand sides:
the rows of one level are solved together by the lean turn, an item that
reaches over level ends level by level, on one XCD or on the whole device.

Bars (the repository's): FP64 within 1e-12 relative (max-norm) of the oracle's
serial substitution, fused mixed within 1e-10, FP32 within 1e-5; repeated
solves bit-identical.

The shapes have levels of one row (an item then holds one level per row), of
less and of more rows than an item, and levels on both sides of the line
between one XCD and the whole device; the widths include one that is no power
of two and the widest.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle_py as O
from conftest import lower_from_rows
from sptrsv_amd import _lib as L
from sptrsv_amd import interface as I

pytestmark = pytest.mark.gpu

BARS = {I.PREC_F64: 1e-12, I.PREC_MIXED: 1e-10, I.PREC_F32: 1e-5}


def relerr(x, ref):
    return float(np.max(np.abs(x - ref)) / max(np.max(np.abs(ref)), 1e-300))


def layered(levels, width, length, seed):
    rng = np.random.default_rng(seed)
    rows = []
    for lev in range(levels):
        start = lev * width
        for _ in range(width):
            if lev == 0:
                rows.append([])
                continue
            cols = {int(rng.integers(start - width, start))}
            cols |= set(rng.choice(start, size=min(length - 1, start), replace=False).tolist())
            rows.append(sorted(cols))
    ia, ja, a = lower_from_rows(rows, rng)
    return ia, ja, a


@pytest.mark.parametrize("k", [2, 5, 16, 64])
@pytest.mark.parametrize("levels,width,length", [(60, 1, 1), (20, 7, 3), (12, 33, 9), (5, 700, 4), (3, 6000, 2)])
def test_level_order_rhs_matches_oracle(levels, width, length, k):
    print(f"level order, {levels} levels of {width} rows, k={k}", flush=True)
    ia, ja, a = layered(levels, width, length, seed=k)
    n = len(ia) - 1
    b = np.random.default_rng(1).uniform(-1.0, 1.0, (n, k))
    ref = O.fwd_f64(ia, ja, a, b.ravel(), k)
    mat = I.allocate_memory(ia, ja, a)
    for mode in (I.ORDER, I.MULTIROW):
        info = I.multirow_analysis_base_GPU(mat, mode)
        shapes = [dict()]  # the default shape of the analysis
        if mode == I.ORDER:
            shapes += [dict(kernel=I.KERNEL_ORDER, variant=2, lanes=lanes, wg=wg, cu_waves=cw)
                       for lanes, wg, cw in ((1, 256, 4), (1, 1024, 16), (4, 1024, 16))]
        for prec, bar in BARS.items():
            dt = np.float32 if prec == I.PREC_F32 else np.float64
            db, dx = I.DeviceArray.from_numpy(b.astype(dt).ravel()), I.DeviceArray(n * k, dt)
            for shape in shapes:
                got = []
                for _ in range(2):
                    I.solve(mat, info, prec, db, dx, k=k, cfg=I._cfg(**shape))
                    assert I.check_watchdog(mat) == 0, L.last_error()
                    got.append(dx.numpy())
                assert relerr(got[0].astype(np.float64), ref.ravel()) <= bar, (mode, prec, shape)
                assert np.array_equal(got[0], got[1])
            db.free()
            dx.free()
        I.free_device_analysis(None, info)
    I.free_device_analysis(mat, None)
