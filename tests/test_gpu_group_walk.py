"""GPU tests of the group walk (variant 7): rows in natural order, a group of
lanes each, walked by the workgroups of one XCD; every row publishes on its own.

Bars (the repository's): FP64 within 1e-12 relative (max-norm) of the oracle's
serial substitution, fused mixed within 1e-10, FP32 within 1e-5; levels equal
the oracle's; repeated solves bit-identical.

The shapes have rows that depend on others of their wave (a chain), rows of
none, of as many entries as lanes and of one more, rows of several turns, and
sizes around a wave's rows, a workgroup's rows and one row.
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


def windowed(n, lengths, reach, seed):
    rng = np.random.default_rng(seed)
    rows = []
    for i in range(n):
        lo = max(0, i - reach)
        rows.append(sorted(rng.choice(np.arange(lo, i), size=min(lengths[i % len(lengths)], i - lo), replace=False).tolist()))
    return lower_from_rows(rows, rng)


def solve(mat, info, b, prec, **cfg):
    dt = np.float32 if prec == I.PREC_F32 else np.float64
    db, dx = I.DeviceArray.from_numpy(b.astype(dt)), I.DeviceArray(mat.nr, dt)
    I.solve(mat, info, prec, db, dx, cfg=I._cfg(**cfg))
    assert I.check_watchdog(mat) == 0, L.last_error()
    x = dx.numpy()
    db.free()
    dx.free()
    return x


CASES = {
    "one row": (1, [0], 1),
    "chain": (300, [1], 1),
    "no entries": (1000, [0], 1),
    "lanes": (1500, [0, 1, 7, 8, 9, 16, 17, 31, 33], 400),
    "wave end": (129, [5], 60),
    "workgroup end": (16 * 16 * 2 + 1, [3, 4], 90),
    "wide": (20000, [8], 900),
    "long rows": (1200, [1, 2, 64, 65, 400], 1000),
}


@pytest.mark.parametrize("lanes", [1, 8, 32, 64])
@pytest.mark.parametrize("name", CASES)
def test_group_walk_matches_oracle(name, lanes):
    print(f"group walk {name}, {lanes} lanes", flush=True)
    ia, ja, a = windowed(*CASES[name], seed=4)
    b = np.random.default_rng(2).uniform(-1.0, 1.0, len(ia) - 1)
    ref = O.fwd_f64(ia, ja, a, b)
    mat = I.allocate_memory(ia, ja, a)
    for prec, bar in BARS.items():
        x = solve(mat, None, b, prec, kernel=I.KERNEL_SIMPLE, variant=7, lanes=lanes)
        assert relerr(x.astype(np.float64), ref) <= bar, prec
        assert np.array_equal(x, solve(mat, None, b, prec, kernel=I.KERNEL_SIMPLE, variant=7, lanes=lanes))
        # the default shape and the general path
        assert relerr(solve(mat, None, b, prec, kernel=I.KERNEL_SIMPLE).astype(np.float64), ref) <= bar
        assert relerr(solve(mat, None, b, prec, kernel=I.KERNEL_SIMPLE, variant=0, lanes=4).astype(np.float64), ref) <= bar
    for mode in (I.ORDER, I.ALL):
        info = I.multirow_analysis_base_GPU(mat, mode)
        lev, nlevs = O.levels(ia, ja)
        assert info.nlevs == nlevs and np.array_equal(I.analysis_arrays(info)["level"], lev)
        for kernel in (I.KERNEL_ORDER, I.KERNEL_AUTO):
            assert relerr(solve(mat, info, b, I.PREC_F64, kernel=kernel), ref) <= 1e-12
        assert relerr(solve(mat, info, b, I.PREC_F64, kernel=I.KERNEL_ORDER, variant=7, lanes=lanes), ref) <= 1e-12
        I.free_device_analysis(None, info)
    I.free_device_analysis(mat, None)


def test_refusals():
    ia, ja, a = windowed(100, [2], 50, 1)
    mat = I.allocate_memory(ia, ja, a)
    info = I.multirow_analysis_base_GPU(mat, I.ALL)
    db, dx = I.DeviceArray.from_numpy(np.ones(200)), I.DeviceArray(200, np.float64)
    for bad in (dict(kernel=I.KERNEL_SIMPLE, k=2), dict(kernel=I.KERNEL_ORDER, reorder=1), dict(kernel=I.KERNEL_SIMPLE, variant=8)):
        k = bad.pop("k", 1)
        with pytest.raises(L.SptrsvError):
            I.solve(mat, info, I.PREC_F64, db, dx, k=k, cfg=I._cfg(**{"lanes": 4, "variant": 7, **bad}))
    db.free()
    dx.free()
    I.free_device_analysis(mat, info)
