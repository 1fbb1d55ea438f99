"""GPU tests of the level walk (variant 4 of ORDER / MULTIROW): one workgroup
solves level by level, exchanging results through LDS.

Bars (the repository's): FP64 within 1e-12 relative (max-norm) of the oracle's
serial substitution, fused mixed within 1e-10, FP32 within 1e-5; repeated
solves bit-identical; exact x == 1 on the known-answer input.

The shapes sit on the edges of the walk's layout: row lengths around 4 entries
per lane for 1, 2, 4, ..., 64 lanes and beyond 256 entries (overflow lists),
level sizes around 64 rows and around a step of 1, 4 and 8 slices, more than
16384 rows (right-hand side and result pass through position order), and
dependencies further back than the 8192 to 12288 words kept in LDS.
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


def walk(mat, info, b, prec, kernel=I.KERNEL_ORDER, variant=4):
    dt = np.float32 if prec == I.PREC_F32 else np.float64
    db, dx = I.DeviceArray.from_numpy(b.astype(dt)), I.DeviceArray(mat.nr, dt)
    I.solve(mat, info, prec, db, dx, kernel=kernel, lanes=4, wg=256, variant=variant)
    assert I.check_watchdog(mat) == 0, L.last_error()
    x = dx.numpy()
    db.free()
    dx.free()
    return x


def layered(sizes, lengths, reach, seed):
    """Levels of the given sizes; row i of a level has a dependency in the
    level before and lengths[i % len] - 1 more among the last `reach` rows."""
    rng = np.random.default_rng(seed)
    rows, prev = [], None
    for size in sizes:
        start = len(rows)
        for i in range(size):
            if prev is None:
                rows.append([])
                continue
            want = lengths[i % len(lengths)]
            cols = {int(rng.integers(prev, start))} if want else set()
            lo = max(0, start - reach)
            cols |= set(rng.choice(np.arange(lo, start), size=min(max(want - 1, 0), start - lo), replace=False).tolist())
            rows.append(sorted(cols))
        prev = start
    return rows


def check_system(ia, ja, a, seed=0):
    n = len(ia) - 1
    b = np.random.default_rng(seed).uniform(-1, 1, n)
    ref = O.fwd_f64(ia, ja, a, b)
    mat = I.allocate_memory(ia, ja, a)
    info = I.multirow_analysis_base_GPU(mat, I.ALL)
    for prec, bar in BARS.items():
        want = O.fwd_f32(ia, ja, a.astype(np.float32), b.astype(np.float32)) if prec == I.PREC_F32 else ref
        x = walk(mat, info, b, prec)
        assert relerr(x.astype(np.float64), want.astype(np.float64)) <= bar, prec
        assert np.array_equal(x, walk(mat, info, b, prec)), prec
    I.free_device_analysis(mat, info)


SHAPES = {
    "one row": ([1], [0], 1),
    "level of 63, 64, 65 rows": ([63, 64, 65, 1, 64], [1, 3, 4], 200),
    "lengths around 4, 8, 16": ([40, 50, 40, 50, 40], [1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17], 90),
    "lengths around 32 to 256": ([300, 20, 20, 20], [31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256], 290),
    "overflow lists": ([700, 12, 9], [257, 300, 512, 513, 5, 640], 650),
    "steps of 4 slices": ([250, 256, 257, 130, 200], [2, 3], 500),
    "steps of 8 slices": ([500, 512, 513, 1030, 640], [2, 4], 900),
    "one row per level": ([1] * 300, [1, 9, 2], 40),
}


@pytest.mark.parametrize("name", list(SHAPES))
def test_shapes(name):
    sizes, lengths, reach = SHAPES[name]
    check_system(*lower_from_rows(layered(sizes, lengths, reach, 3)))


@pytest.mark.parametrize("gen,param", [(1, 130), (2, 20000), (3, 3000), (4, 27)])
def test_generated(gen, param):
    s = I.generate(gen, param)
    check_system(s.ia, s.ja, s.a)


def test_far_dependencies():
    # 100 rows per level, every 50th row with up to three dependencies 13000 to
    # 20000 rows back: beyond the words in LDS, some in one lane's overflow
    n, per = 40000, 100
    rng = np.random.default_rng(5)
    rows = []
    for i in range(n):
        lev = i // per
        if lev == 0:
            rows.append([])
            continue
        cols = {int(rng.integers((lev - 1) * per, lev * per))}
        if i > 21000 and i % 50 == 0:
            cols |= {i - int(v) for v in rng.integers(13000, 20000, 1 + (i // 50) % 3)}
        rows.append(sorted(cols))
    check_system(*lower_from_rows(rows))


def test_known_answer_default_shape_values_and_replays():
    s = I.generate(1)
    mat = I.allocate_memory(s.ia, s.ja, s.a)
    info = I.multirow_analysis_base_GPU(mat, I.ALL)
    cfg = I._cfg(kernel=I.KERNEL_MULTIROW)      # the shape left open
    for prec in (I.PREC_F64, I.PREC_MIXED):
        assert O.validate_x(walk(mat, info, s.b, prec)) == 0
    # new values reach the plan, eager and in a captured solve made before
    db, dx = I.DeviceArray.from_numpy(s.b), I.DeviceArray(s.n, np.float64)
    for scale in (1.0, 2.0, 0.5):
        I.update_values(mat, s.a * scale)
        for _ in range(3):
            I.solve_graph(mat, info, I.PREC_F64, db, dx, cfg)
            assert np.array_equal(dx.numpy(), np.full(s.n, 1.0 / scale))
            I.csr_L_solve_multirow(mat, info, db, dx)
            assert np.array_equal(dx.numpy(), np.full(s.n, 1.0 / scale))
    # two analyses of one matrix, each with its own plan; the first one's goes
    # with it
    info2 = I.multirow_analysis_base_GPU(mat, I.ORDER)
    I.csr_L_solve_order(mat, info2, db, dx)
    I.free_device_analysis(None, info)
    I.csr_L_solve_order(mat, info2, db, dx)
    assert np.array_equal(dx.numpy(), np.full(s.n, 2.0))
    I.free_device_analysis(mat, info2)


def test_refusals_and_fallbacks():
    s = I.generate(2, 5000)
    mat = I.allocate_memory(s.ia, s.ja, s.a)
    info = I.multirow_analysis_base_GPU(mat, I.ALL)
    ref = O.fwd_f64(s.ia, s.ja, s.a, s.b)
    db, dx = I.DeviceArray.from_numpy(s.b), I.DeviceArray(s.n * 2, np.float64)
    for bad in (dict(kernel=I.KERNEL_SIMPLE), dict(kernel=I.KERNEL_ORDER, k=2)):
        with pytest.raises(L.SptrsvError):
            I.solve(mat, info, I.PREC_F64, db, dx, lanes=4, variant=4, **bad)
    # a trace is taken by the walks through memory
    I.trace(mat, True)
    assert relerr(walk(mat, info, s.b, I.PREC_F64), ref) <= 1e-12
    assert I.trace_read(mat)[0][:, 2].all()
    I.trace(mat, False)
    # an upper handle (b and x reversed around the walk)
    up = I.transpose(mat)
    upi = I.multirow_analysis_base_GPU(up, I.ALL)
    x = walk(up, upi, s.b, I.PREC_F64)
    r = s.b - np.bincount(s.ja, weights=s.a * np.repeat(x, np.diff(s.ia)), minlength=s.n)
    assert np.max(np.abs(r)) <= 1e-12 * np.max(np.abs(s.b))
    I.free_device_analysis(up, upi)
    I.free_device_analysis(mat, info)
