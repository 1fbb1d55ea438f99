"""GPU tests of the packed walk (variant 6 of ORDER / MULTIROW): the wave64
layout of an analysis walked by one XCD or by the whole device.

Bars (the repository's): FP64 within 1e-12 relative (max-norm) of the oracle's
serial substitution, fused mixed within 1e-10, FP32 within 1e-5; repeated
solves bit-identical.

The shapes sit on both sides of the walk's own lines (20, 100 and 400 waves per
level), on the row-length classes of the layout (1, 2, 4, 8, 16, 32 lanes and
beyond, rows split from 257 off-diagonals on), and on last workgroups with one
wave.
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


def solve(mat, info, b, prec, kernel, variant=6, split_rows=0):
    dt = np.float32 if prec == I.PREC_F32 else np.float64
    db, dx = I.DeviceArray.from_numpy(b.astype(dt)), I.DeviceArray(mat.nr, dt)
    cfg = I._cfg(kernel=kernel, lanes=4, wg=256, variant=variant, split_rows=split_rows)
    I.solve(mat, info, prec, db, dx, cfg=cfg)
    assert I.check_watchdog(mat) == 0, L.last_error()
    x = dx.numpy()
    db.free()
    dx.free()
    return x


def layered(levels, width, lengths, seed):
    """`levels` levels of `width` rows; row i of a level depends on a row of the
    level before and on lengths[i % len] - 1 more earlier rows."""
    rng = np.random.default_rng(seed)
    rows = []
    for lev in range(levels):
        start = lev * width
        for i in range(width):
            if lev == 0:
                rows.append([])
                continue
            want = lengths[i % len(lengths)]
            cols = {int(rng.integers(start - width, start))} if want else set()
            if want > 1:
                cols |= set(rng.choice(start, size=min(want - 1, start), replace=False).tolist())
            rows.append(sorted(cols))
    ia, ja, a = lower_from_rows(rows, rng)
    return ia, ja, a, rng.uniform(-1.0, 1.0, len(rows))


SHAPES = {
    "one row per level": (70, 1, [1]),
    "few waves": (12, 65, [1, 2, 3, 5]),
    "classes": (9, 300, [1, 2, 3, 4, 5, 8, 9, 16, 17, 32, 33, 64]),
    "19 waves": (6, 19 * 4, [16]),
    "21 waves": (6, 21 * 4, [16]),
    "99 waves": (4, 99 * 4, [16]),
    "101 waves": (4, 101 * 4, [16]),
    "401 waves": (3, 401 * 2, [32]),
    "wide": (3, 40000, [1, 2]),
    "diagonal": (1, 5000, [0]),
    "long rows": (5, 130, [1, 3, 256, 257, 300]),
}


@pytest.mark.parametrize("name", SHAPES)
def test_packed_walk_matches_oracle(name):
    print(f"packed walk {name}", flush=True)
    ia, ja, a, b = layered(*SHAPES[name], seed=3)
    mat = I.allocate_memory(ia, ja, a)
    ref = O.fwd_f64(ia, ja, a, b)
    for mode, kernel in ((I.ORDER, I.KERNEL_ORDER), (I.MULTIROW, I.KERNEL_MULTIROW), (I.ALL, I.KERNEL_ORDER)):
        info = I.multirow_analysis_base_GPU(mat, mode)
        for prec, bar in BARS.items():
            x = solve(mat, info, b, prec, kernel)
            assert relerr(x.astype(np.float64), ref) <= bar, (mode, prec)
            assert np.array_equal(x, solve(mat, info, b, prec, kernel)), (mode, prec)
            assert relerr(solve(mat, info, b, prec, kernel, split_rows=-1).astype(np.float64), ref) <= bar
            # and through the lean path
            assert relerr(solve(mat, info, b, prec, kernel, variant=1).astype(np.float64), ref) <= bar
        # default shapes, named and automatic, eager, captured and allocation-free
        db, dx = I.DeviceArray.from_numpy(b), I.DeviceArray(len(b), np.float64)
        for k in (kernel, I.KERNEL_AUTO):
            for _ in range(3):
                I.solve_graph(mat, info, I.PREC_F64, db, dx, I._cfg(kernel=k))
                I.synchronize()
                assert relerr(dx.numpy(), ref) <= BARS[I.PREC_F64]
            I.solve_mixed_noalloc(mat, info, db, dx, cfg=I._cfg(kernel=k))
            I.synchronize()
            assert I.check_watchdog(mat) == 0 and relerr(dx.numpy(), ref) <= BARS[I.PREC_MIXED]
        db.free()
        dx.free()
        I.free_device_analysis(None, info)
    I.free_device_analysis(mat, None)


def test_loaded_and_copied_analyses(tmp_path):
    """An ORDER analysis from a file or copied from another handle has the
    layout too, and none in its public arrays."""
    ia, ja, a, b = layered(6, 200, [1, 4, 20, 300], seed=8)
    mat, twin = I.allocate_memory(ia, ja, a), I.allocate_memory(ia, ja, a)
    ref = O.fwd_f64(ia, ja, a, b)
    info = I.multirow_analysis_base_GPU(mat, I.ORDER)
    I.save_analysis(str(tmp_path / "order.bin"), mat, info)
    loaded = I.load_analysis(str(tmp_path / "order.bin"), mat)
    copied = I.copy_analysis(mat, info, twin)
    x = solve(mat, info, b, I.PREC_F64, I.KERNEL_ORDER)
    assert relerr(x, ref) <= 1e-12
    for m, i in ((mat, loaded), (twin, copied)):
        assert i.n_waves == 0 and I.analysis_segments(i) == (0, 0)
        assert np.array_equal(x, solve(m, i, b, I.PREC_F64, I.KERNEL_ORDER))
        I.free_device_analysis(None, i)
    I.free_device_analysis(mat, info)
    I.free_device_analysis(twin, None)


def test_refusals():
    ia, ja, a, b = layered(4, 50, [2], seed=1)
    mat = I.allocate_memory(ia, ja, a)
    info = I.multirow_analysis_base_GPU(mat, I.ALL)
    db, dx = I.DeviceArray.from_numpy(np.repeat(b, 2)), I.DeviceArray(2 * len(b), np.float64)
    for bad in (dict(kernel=I.KERNEL_SIMPLE), dict(kernel=I.KERNEL_ORDER, k=2), dict(kernel=I.KERNEL_MULTIROW, reorder=1)):
        k = bad.pop("k", 1)
        with pytest.raises(L.SptrsvError):
            I.solve(mat, info, I.PREC_F64, db, dx, k=k, cfg=I._cfg(lanes=4, variant=6, **bad))
    db.free()
    dx.free()
    I.free_device_analysis(mat, info)
