"""GPU tests of what a handle finds out about its rows: the same matrix gets the
same default walk whichever entry point it came through and in whatever order
its columns were given.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle_py as O
from sptrsv_amd import interface as I

pytestmark = pytest.mark.gpu


def relerr(x, ref):
    return float(np.max(np.abs(x - ref)) / max(np.max(np.abs(ref)), 1e-300))


def grid(side):
    s = I.generate(1, side)
    return s.ia, s.ja, s.a


def windowed(n, entries, reach, seed=3):
    """`entries` off-diagonals a row among the last `reach`."""
    rng = np.random.default_rng(seed)
    ia, ja = [0], []
    for i in range(n):
        c = set(rng.integers(max(0, i - reach), i, entries).tolist()) if i else set()
        ja += sorted(c) + [i]
        ia.append(len(ja))
    ia, ja = np.array(ia, np.int32), np.array(ja, np.int32)
    a = np.full(len(ja), -0.05)
    a[ia[1:] - 1] = 1.0
    return ia, ja, a


def upper(ia, ja, a):
    """The matrix with rows and columns in reversed order: an upper triangle,
    columns ascending."""
    n = len(ia) - 1
    r = n - 1 - np.repeat(np.arange(n), np.diff(ia))
    c = n - 1 - ja
    o = np.lexsort((c, r))
    ui = np.zeros(n + 1, np.int32)
    ui[1:] = np.cumsum(np.bincount(r, minlength=n))
    return ui, c[o].astype(np.int32), a[o]


def reordered(ia, ja, a, seed=1):
    """Off-diagonals of every row in random order, the diagonal last."""
    n = len(ia) - 1
    key = np.random.default_rng(seed).random(len(ja))
    key[ia[1:] - 1] = 2.0
    o = np.lexsort((key, np.repeat(np.arange(n), np.diff(ia))))
    return ia, ja[o], a[o]


def device(*arrays):
    return [I.DeviceArray.from_numpy(v) for v in arrays]


def shapes(handle, info=None):
    c = I.default_config(handle, info, I.PREC_F64, 1)
    return c.kernel, c.variant, c.lanes, c.wg, c.cu_waves


MATRICES = {"grid 100^2": lambda: grid(100), "windowed 400": lambda: windowed(6000, 4, 400),
            "windowed 12000": lambda: windowed(30000, 3, 12000)}


@pytest.mark.parametrize("name", MATRICES)
def test_upper_triangles_take_the_lower_one_s_walk(name):
    ia, ja, a = MATRICES[name]()
    n = len(ia) - 1
    ui, uj, ua = upper(ia, ja, a)
    low, up = I.allocate_memory(ia, ja, a), I.allocate_memory_upper(ui, uj, ua)
    h = I.Spsv(n, *device(ui, uj, ua), fill=I.FILL_UPPER)
    assert shapes(up) == shapes(low)
    assert shapes(h.matrix()) == shapes(low)
    h.analysis(I.PREC_F64)
    b = np.random.default_rng(2).uniform(-1.0, 1.0, n)
    db, dx = device(b, b)
    h.solve(db, dx)
    assert relerr(dx.numpy()[::-1], O.fwd_f64(ia, ja, a, b[::-1].copy())) <= 1e-12
    h.close()
    I.free_device_analysis(low, None)
    I.free_device_analysis(up, None)


@pytest.mark.parametrize("name", MATRICES)
def test_order_of_columns_does_not_matter(name):
    ia, ja, a = MATRICES[name]()
    n = len(ia) - 1
    _, sj, sa = reordered(ia, ja, a)
    low, mixed = I.allocate_memory(ia, ja, a), I.allocate_memory(ia, sj, sa)
    assert shapes(mixed) == shapes(low)
    h = I.Spsv(n, *device(ia, sj, sa))
    assert shapes(h.matrix()) == shapes(low)
    rows = np.repeat(np.arange(n), np.diff(ia)).astype(np.int32)
    coo = [I.coo_to_lower(rows, c, v, n, False, unit=False) for c, v in ((ja, a), (sj, sa))]
    assert [shapes(m) for m in coo] == [shapes(low)] * 2
    b = np.random.default_rng(2).uniform(-1.0, 1.0, n)
    db, dx = device(b, b)
    for m in [mixed, h.matrix()] + coo:
        I.csr_L_solve_simple(m, db, dx)
        assert relerr(dx.numpy(), O.fwd_f64(ia, ja, a, b)) <= 1e-12
    h.close()
    for m in [low, mixed] + coo:
        I.free_device_analysis(m, None)


def test_rows_without_dependencies_have_no_distance():
    """Rows that wait for nothing do not bring the others' dependencies nearer:
    one of five waiting rows and all of them get the same walk."""
    n, reach = 60000, 20000
    rng = np.random.default_rng(7)

    def some(share):
        ia, ja = [0], []
        for i in range(n):
            ja += [max(0, i - int(rng.integers(100, reach))), i] if i and rng.random() < share else [i]
            ia.append(len(ja))
        ia, ja = np.array(ia, np.int32), np.array(ja, np.int32)
        return ia, ja, np.where(np.arange(len(ja)) == np.repeat(ia[1:] - 1, np.diff(ia)), 1.0, -0.5)

    dense, sparse = some(1.0), some(0.2)
    mats = [I.allocate_memory(*dense), I.allocate_memory(*sparse)]
    h = I.Spsv(n, *device(*sparse))
    rows = np.repeat(np.arange(n), np.diff(sparse[0])).astype(np.int32)
    mats.append(I.coo_to_lower(rows, sparse[1], sparse[2], n, False, unit=False))
    variants = [shapes(m)[1] for m in mats] + [shapes(h.matrix())[1]]
    assert variants == variants[:1] * 4
    h.close()
    for m in mats:
        I.free_device_analysis(m, None)


def band(n, offsets):
    ia, ja = [0], []
    for i in range(n):
        ja += [i - o for o in sorted(offsets, reverse=True) if o <= i] + [i]
        ia.append(len(ja))
    ia, ja = np.array(ia, np.int32), np.array(ja, np.int32)
    return ia, ja, np.where(np.arange(len(ja)) == np.repeat(ia[1:] - 1, np.diff(ia)), 1.0, -0.1)


@pytest.mark.parametrize("offsets", [[32], [17, 40, 63], [10], [1, 2, 17], [], [40]])
@pytest.mark.parametrize("n", [900, 4000])
def test_banded_handles_made_on_the_device(offsets, n):
    """A banded matrix gets the walk that the host's count of its levels gives it
    when it is made on the device, where they are not counted (only the row 32
    before, n = 4000: 178 us with the block walk, 112 without)."""
    ia, ja, a = band(n, offsets)
    low = I.allocate_memory(ia, ja, a)
    h = I.Spsv(n, *device(ia, ja, a))
    rows = np.repeat(np.arange(n), np.diff(ia)).astype(np.int32)
    coo = I.coo_to_lower(rows, ja, a, n, False, unit=False)
    assert shapes(h.matrix()) == shapes(low) and shapes(coo) == shapes(low)
    b = np.random.default_rng(2).uniform(-1.0, 1.0, n)
    db, dx = device(b, b)
    for m in (low, coo, h.matrix()):
        I.csr_L_solve_simple(m, db, dx)
        assert relerr(dx.numpy(), O.fwd_f64(ia, ja, a, b)) <= 1e-12
    h.close()
    I.free_device_analysis(low, None)
    I.free_device_analysis(coo, None)
