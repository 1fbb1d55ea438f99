"""GPU tests of the block walk (variant 5): 64 consecutive rows per wave, one
row per lane, results of the block's own rows exchanged in registers.

Bars (the repository's): FP64 within 1e-12 relative (max-norm) of the oracle's
serial substitution, fused mixed within 1e-10, FP32 within 1e-5; levels equal
the oracle's; repeated solves bit-identical.

The shapes sit on the edges of the walk: sizes around one and two blocks,
columns 1, 63 and 64 rows back (the last one leaves the banded kernel), rows of
4, 5, 8 and 9 off-diagonals (the last one leaves the walk), unsorted and
repeated columns, blocks whose rows form no, one or many chains.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle_py as O
from sptrsv_amd import _lib as L
from sptrsv_amd import interface as I

pytestmark = pytest.mark.gpu

BARS = {I.PREC_F64: 1e-12, I.PREC_MIXED: 1e-10, I.PREC_F32: 1e-5}


def relerr(x, ref):
    return float(np.max(np.abs(x - ref)) / max(np.max(np.abs(ref)), 1e-300))


def matrix(n, offsets, share=1.0, seed=0, shuffle=False, twice=False):
    """Lower CSR, diagonal last: row i depends on i - o for o in offsets, each
    with probability share."""
    rng = np.random.default_rng(seed)
    ia, ja, a = [0], [], []
    for i in range(n):
        c = [i - o for o in offsets if o <= i and (share >= 1.0 or rng.random() < share)]
        c = sorted(c)
        if twice and c:
            c = c + [c[0]]
        if shuffle:
            rng.shuffle(c)
        v = rng.uniform(-1.0, 1.0, len(c)) / max(1, len(c))
        ja += c + [i]
        a += v.tolist() + [1.0 + float(np.abs(v).sum())]
        ia.append(len(ja))
    return np.array(ia, np.int32), np.array(ja, np.int32), np.array(a), rng.uniform(-1.0, 1.0, n)


def solve(mat, b, prec, info=None, kernel=I.KERNEL_SIMPLE, variant=5):
    dt = np.float32 if prec == I.PREC_F32 else np.float64
    db, dx = I.DeviceArray.from_numpy(b.astype(dt)), I.DeviceArray(mat.nr, dt)
    I.solve(mat, info, prec, db, dx, kernel=kernel, lanes=4, wg=256, variant=variant)
    assert I.check_watchdog(mat) == 0, L.last_error()
    x = dx.numpy()
    db.free()
    dx.free()
    return x


CASES = {
    "chain": dict(offsets=[1]),
    "band17": dict(offsets=range(1, 18)),
    "band63": dict(offsets=range(1, 64)),
    "only63": dict(offsets=[63]),
    "only64": dict(offsets=[1, 64]),
    "sparse band": dict(offsets=range(1, 64), share=0.1),
    "diagonal": dict(offsets=[]),
    "grid": dict(offsets=[1, 100]),
    "row4": dict(offsets=[1, 2, 70, 99]),
    "row5": dict(offsets=[1, 2, 70, 99, 130]),
    "row8": dict(offsets=[1, 2, 3, 5, 70, 99, 130, 300]),
    "row9": dict(offsets=[1, 2, 3, 5, 7, 70, 99, 130, 300]),
    "unsorted band": dict(offsets=[1, 3, 20, 40], shuffle=True),
    "unsorted": dict(offsets=[1, 3, 90, 200], shuffle=True),
    "repeated band": dict(offsets=[1, 3], twice=True),
    "repeated": dict(offsets=[1, 3, 80], twice=True),
}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("n", [1, 63, 64, 65, 129, 1500])
def test_block_walk_matches_oracle(name, n):
    print(f"block walk {name} n={n}", flush=True)
    ia, ja, a, b = matrix(n, seed=n, **CASES[name])
    mat = I.allocate_memory(ia, ja, a)
    ref = O.fwd_f64(ia, ja, a, b)
    for prec, bar in BARS.items():
        x = solve(mat, b, prec)
        assert relerr(x.astype(np.float64), ref) <= bar, prec
        assert np.array_equal(x, solve(mat, b, prec)), prec
        # and through the general path
        assert relerr(solve(mat, b, prec, variant=1).astype(np.float64), ref) <= bar, prec
    # the default shape, the level pass and the walks of an analysis
    info = I.multirow_analysis_base_GPU(mat, I.ALL)
    lev, nlevs = O.levels(ia, ja)
    assert info.nlevs == nlevs and np.array_equal(I.analysis_arrays(info)["level"], lev)
    for kernel in (I.KERNEL_SIMPLE, I.KERNEL_ORDER, I.KERNEL_MULTIROW):
        db, dx = I.DeviceArray.from_numpy(b), I.DeviceArray(n, np.float64)
        I.solve(mat, info, I.PREC_F64, db, dx, kernel=kernel)
        assert I.check_watchdog(mat) == 0
        assert relerr(dx.numpy(), ref) <= BARS[I.PREC_F64]
        db.free()
        dx.free()
    I.free_device_analysis(mat, info)


@pytest.mark.parametrize("offsets", [[1, 2, 17], [3, 100]])
def test_other_handles_values_and_replays(offsets):
    """Upper, transposed and device-built handles, new values, replays."""
    print(f"block walk handles {offsets}", flush=True)
    n = 700
    ia, ja, a, b = matrix(n, offsets, seed=5)
    ref = O.fwd_f64(ia, ja, a, b)
    mat = I.allocate_memory(ia, ja, a)
    T = I.transpose(mat)
    dense = np.zeros((n, n))
    dense[np.repeat(np.arange(n), np.diff(ia)), ja] = a
    xt = np.linalg.solve(dense.T, b)
    db, dx = I.DeviceArray.from_numpy(b), I.DeviceArray(n, np.float64)
    I.csr_L_solve_simple(T, db, dx)
    assert I.check_watchdog(T) == 0 and relerr(dx.numpy(), xt) <= 1e-12
    # L^T given as an upper triangle
    up = [(ja[p], i, a[p]) for i in range(n) for p in range(ia[i], ia[i + 1])]
    up.sort()
    ui = np.zeros(n + 1, np.int32)
    ui[1:] = np.cumsum(np.bincount([r for r, _, _ in up], minlength=n))
    U = I.allocate_memory_upper(ui, np.array([c for _, c, _ in up], np.int32), np.array([v for _, _, v in up]))
    I.csr_L_solve_simple(U, db, dx)
    assert I.check_watchdog(U) == 0 and relerr(dx.numpy(), xt) <= 1e-12
    rows = np.repeat(np.arange(n), np.diff(ia)).astype(np.int32)
    C = I.coo_to_lower(rows, ja, a, n, False, unit=False)
    I.csr_L_solve_simple(C, db, dx)
    assert I.check_watchdog(C) == 0 and relerr(dx.numpy(), ref) <= 1e-12
    a2 = a.copy()
    a2[ia[1:] - 1] *= 3.0
    I.update_values(mat, a2)
    ref2 = O.fwd_f64(ia, ja, a2, b)
    cfg = I._cfg(kernel=I.KERNEL_SIMPLE)
    for _ in range(3):
        I.solve_graph(mat, None, I.PREC_F64, db, dx, cfg)
        I.synchronize()
        assert relerr(dx.numpy(), ref2) <= 1e-12
    for m in (mat, T, U, C):
        I.free_device_analysis(m, None)
    db.free()
    dx.free()


@pytest.mark.parametrize("offsets", [[1, 2], [1, 100]])
def test_infinite_row_stays_its_own(offsets):
    """A row that overflows reaches the rows that depend on it and no other."""
    n = 300
    ia, ja, a, b = matrix(n, offsets, share=0.6, seed=9)
    b[40] = np.inf
    ref = O.fwd_f64(ia, ja, a, b)
    mat = I.allocate_memory(ia, ja, a)
    x = solve(mat, b, I.PREC_F64)
    ok = np.isfinite(ref)
    assert 0 < ok.sum() < n and np.array_equal(np.isfinite(x), ok)
    assert relerr(x[ok], ref[ok]) <= 1e-12
    I.free_device_analysis(mat, None)


def test_refusals():
    ia, ja, a, b = matrix(100, [1], seed=1)
    mat = I.allocate_memory(ia, ja, a)
    db, dx = I.DeviceArray.from_numpy(np.tile(b[:, None], (1, 2)).ravel()), I.DeviceArray(200, np.float64)
    with pytest.raises(L.SptrsvError):
        I.solve(mat, None, I.PREC_F64, db, dx, k=2, kernel=I.KERNEL_SIMPLE, lanes=4, variant=5)
    with pytest.raises(L.SptrsvError):
        I.solve(mat, None, I.PREC_F64, db, dx, kernel=I.KERNEL_SIMPLE, lanes=4, variant=6)
    I.free_device_analysis(mat, None)
    db.free()
    dx.free()


@pytest.mark.parametrize("prec", [I.PREC_F64, I.PREC_MIXED])
def test_batch_members_in_blocks(prec):
    """Banded members of a batch go through the block walk beside the others,
    eager and replayed."""
    from sptrsv_amd.interface import System

    shapes = [(1, [1]), (63, [1, 2]), (64, range(1, 64)), (65, [1]), (200, [1, 17]), (700, [1, 64]), (500, [2, 90, 300]),
              (1500, range(1, 18)), (300, [])]
    systems, refs = [], []
    for q, (n, offsets) in enumerate(shapes):
        ia, ja, a, b = matrix(n, offsets, seed=q)
        systems.append(System(n, ia, ja, a, b))
        refs.append(O.fwd_f64(ia, ja, a, b))
    ref = np.concatenate(refs)
    bt = I.Batch(systems)
    bt.tune(prec, tune=False)
    db = I.DeviceArray.from_numpy(np.concatenate([s.b for s in systems]))
    dx = I.DeviceArray(len(ref), np.float64)
    for graph in (False, True, True, True):
        bt.solve(prec, db, dx, graph=graph)
        I.synchronize()
        assert bt.check() == 0, L.last_error()
        assert relerr(dx.numpy(), ref) <= BARS[prec]
    bt.close()
    db.free()
    dx.free()


@pytest.mark.parametrize("band", [1, 4, 17, 32, 63])
@pytest.mark.parametrize("prec", [I.PREC_F64, I.PREC_F32])
def test_banded_rounding_error(band, prec):
    """The banded kernel's rounding error (2-norm, against extended precision) is
    no larger than that of a row per wave, whose lanes' sums meet in a tree."""
    ia, ja, a, b = matrix(4000, range(1, band + 1), seed=band)
    if prec == I.PREC_F32:
        a, b = a.astype(np.float32), b.astype(np.float32)
    wide, ref = a.astype(np.longdouble), np.zeros(len(b), np.longdouble)
    for i in range(len(b)):
        s, d = ia[i], ia[i + 1] - 1
        ref[i] = (b[i] - wide[s:d] @ ref[ja[s:d]]) / wide[d]
    mat = (I.allocate_memory_f32 if prec == I.PREC_F32 else I.allocate_memory)(ia, ja, a)

    def error(variant, lanes):
        db, dx = I.DeviceArray.from_numpy(b), I.DeviceArray(len(b), a.dtype)
        I.solve(mat, None, prec, db, dx, kernel=I.KERNEL_SIMPLE, lanes=lanes, wg=256, variant=variant)
        e = dx.numpy() - ref
        return float(np.sqrt((e @ e) / (ref @ ref)))

    lanes = min(64, max(4, 1 << int(len(ja) // len(b) - 1).bit_length()))     # of a row per wave by default
    assert error(5, 4) <= error(1, lanes)
    I.free_device_analysis(mat, None)


@pytest.mark.parametrize("prec,big", [(I.PREC_F64, 1.5e308), (I.PREC_F32, 3.0e38)])
def test_a_column_twice_keeps_both_products(prec, big):
    """The entries of a column that a row holds twice are multiplied each by the
    solution, whose product fits where the entries' sum does not; eager on
    every kind of handle, and as a batch member."""
    n = 200
    ia = np.zeros(n + 1, np.int32)
    ja, a = [], []
    for i in range(n):
        if i % 2:
            ja += [i - 1, i - 1, i]
            a += [big, big, 1.0]
        else:
            ja += [i - 1, i] if i else [i]          # (a chain, whose rows are taken in order)
            a += [0.0, 1.0] if i else [1.0]
        ia[i + 1] = len(ja)
    ja, a = np.array(ja, np.int32), np.array(a)
    b = np.where(np.arange(n) % 2 == 0, 1.0 / big, 3.0)
    if prec == I.PREC_F32:
        a, b = a.astype(np.float32), b.astype(np.float32)
    want = np.where(np.arange(n) % 2 == 0, b, 1.0)
    mats = [(I.allocate_memory_f32 if prec == I.PREC_F32 else I.allocate_memory)(ia, ja, a)]
    spsv = None
    if prec == I.PREC_F64:
        spsv = I.Spsv(n, *(I.DeviceArray.from_numpy(v) for v in (ia, ja, a)))
        mats.append(spsv.matrix())
    db, dx = I.DeviceArray.from_numpy(b), I.DeviceArray(n, a.dtype)
    for mat in mats:
        for variant, lanes in ((0, 0), (5, 4)):
            I.solve(mat, None, prec, db, dx, kernel=I.KERNEL_SIMPLE, lanes=lanes, wg=256, variant=variant)
            assert relerr(dx.numpy(), want) <= 1e-6
    I.free_device_analysis(mats[0], None)
    if prec == I.PREC_F64:
        spsv.close()
        bt = I.Batch([I.System(n, ia, ja, a, b), I.System(n, ia, ja, a, b)])
        bt.tune(prec, tune=False)
        db, dx = I.DeviceArray.from_numpy(np.tile(b, 2)), I.DeviceArray(2 * n, np.float64)
        bt.solve(prec, db, dx)
        I.synchronize()
        assert relerr(dx.numpy(), np.tile(want, 2)) <= 1e-12
        bt.close()


@pytest.mark.parametrize("offsets", [[1, 40], range(1, 10), [7, 300], [600, 900], []])
def test_separate_matrix_of_a_tuned_batch(offsets):
    """The members that stay sync-free, as a matrix of their own, whatever their
    rows look like (grids, bands, far and no dependencies)."""
    systems = []
    for q in range(6):
        ia, ja, a, b = matrix(1000 + 37 * q, offsets, seed=q)
        a[ia[1:] - 1] = 0.6 if len(ja) > len(b) else 1.0     # not dominant: no Jacobi
        systems.append(I.System(len(b), ia, ja, a, b))
    ref = np.concatenate([O.fwd_f64(s.ia, s.ja, s.a, s.b) for s in systems])
    bt = I.Batch(systems)
    bt.tune(I.PREC_MIXED)
    db, dx = I.DeviceArray.from_numpy(np.concatenate([s.b for s in systems])), I.DeviceArray(len(ref), np.float64)
    for separate in (0, 1):
        L.check(L.lib().sptrsv_batch_set_schedule(bt.h, 0, separate))
        bt.solve(I.PREC_MIXED, db, dx)
        I.synchronize()
        assert bt.check() == 0 and relerr(dx.numpy(), ref) <= BARS[I.PREC_MIXED]
    bt.close()


@pytest.mark.parametrize("prec", [I.PREC_F64, I.PREC_MIXED])
def test_batch_tuner_times_the_walk_it_will_use(prec):
    """A banded member takes some 40 ns a row in blocks and 800 as tasks, and is
    never solved as tasks: no launch of the FP64 tuner's is as long as those (the
    mixed one also tries the sync-free members as a matrix of their own, row by
    row among others)."""
    n = 20000
    systems = []
    for q, offsets in enumerate(([1, 2, 3], [1], [3, 400])):
        ia, ja, a, b = matrix(n if q < 2 else 500, offsets, seed=q)
        a[ia[1:] - 1] = 0.9                                  # not dominant: no Jacobi
        systems.append(I.System(len(b), ia, ja, a, b))
    ref = np.concatenate([O.fwd_f64(s.ia, s.ja, s.a, s.b) for s in systems])
    bt = I.Batch(systems)
    I.kernel_timer(2)
    bt.tune(prec)
    ms, launches = I.kernel_timer_read()
    I.kernel_timer(0)
    assert launches > 0 and (prec == I.PREC_MIXED or ms / launches < n * 0.2e-3)
    db, dx = I.DeviceArray.from_numpy(np.concatenate([s.b for s in systems])), I.DeviceArray(len(ref), np.float64)
    bt.solve(prec, db, dx)
    I.synchronize()
    assert bt.check() == 0 and relerr(dx.numpy(), ref) <= BARS[prec]
    bt.close()
