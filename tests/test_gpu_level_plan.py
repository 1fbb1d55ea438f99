"""GPU tests of what the level walk keeps between solves.

Bars (the repository's): FP64 within 1e-12 relative (max-norm) of the oracle's
serial substitution, FP32 within 1e-5.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle_py as O
from sptrsv_amd import _lib as L
from sptrsv_amd import interface as I

pytestmark = pytest.mark.gpu

BARS = {I.PREC_F64: 1e-12, I.PREC_MIXED: 1e-10, I.PREC_F32: 1e-5}


def relerr(x, ref):
    return float(np.max(np.abs(x - ref)) / max(np.max(np.abs(ref)), 1e-300))


def write_device(ptr, array):
    L.check(L.lib().sptrsv_memcpy_htod(ctypes.c_void_p(ptr), ctypes.c_void_p(array.ctypes.data), array.nbytes))


@pytest.mark.parametrize("n", [3000, 20000])
def test_values_written_in_place(n):
    """sp_mat_t::a and a32 are the caller's to write: a solve reads them as they
    are, whether the walk has run before or not, eager and replayed."""
    print(f"values in place n={n}", flush=True)
    s = I.generate(2, n)
    mat = I.allocate_memory(s.ia, s.ja, s.a)
    info = I.multirow_analysis_base_GPU(mat, I.ALL)
    cfg = I._cfg(kernel=I.KERNEL_ORDER, lanes=4, variant=4)
    for scale in (1.0, 1.0 + 2.0 ** -8, 0.75):
        a = s.a * scale
        write_device(mat.a, a)
        write_device(mat.a32, a.astype(np.float32))
        for prec, bar in BARS.items():
            dt = np.float32 if prec == I.PREC_F32 else np.float64
            ref = O.fwd_f64(s.ia, s.ja, a, s.b)
            db, dx = I.DeviceArray.from_numpy(s.b.astype(dt)), I.DeviceArray(s.n, dt)
            I.solve(mat, info, prec, db, dx, cfg=cfg)
            assert relerr(dx.numpy().astype(np.float64), ref) <= bar, (prec, scale)
            for again in (1.0, 0.5):
                write_device(mat.a, a * again)
                write_device(mat.a32, (a * again).astype(np.float32))
                I.solve_graph(mat, info, prec, db, dx, cfg)
                I.synchronize()
                assert relerr(dx.numpy().astype(np.float64), ref / again) <= bar, (prec, scale, again)
            write_device(mat.a, a)
            write_device(mat.a32, a.astype(np.float32))
            db.free()
            dx.free()
    I.free_device_analysis(mat, info)


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert L.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_one_plan_serves_every_precision():
    """Once the walk has run, a solve of another precision needs no memory (so
    none can fail for want of it, and take with it what a captured solve holds)."""
    s = I.generate(1, 500)
    mat = I.allocate_memory(s.ia, s.ja, s.a)
    info = I.multirow_analysis_base_GPU(mat, I.ALL)
    I.reserve(mat, 1)
    cfg = I._cfg(kernel=I.KERNEL_MULTIROW, lanes=4, variant=4)
    bufs = {p: (I.DeviceArray.from_numpy(s.b.astype(t)), I.DeviceArray(s.n, t))
            for p, t in ((I.PREC_F64, np.float64), (I.PREC_MIXED, np.float64), (I.PREC_F32, np.float32))}
    I.solve_graph(mat, info, I.PREC_F64, *bufs[I.PREC_F64], cfg)
    I.synchronize()
    before = free_bytes()
    for prec in (I.PREC_F32, I.PREC_MIXED):
        I.solve(mat, info, prec, *bufs[prec], cfg=cfg)
        I.synchronize()
        assert free_bytes() == before, prec
    for prec in (I.PREC_F64, I.PREC_F32, I.PREC_MIXED, I.PREC_F64):
        bufs[prec][1].fill_bytes(0)
        I.solve_graph(mat, info, prec, *bufs[prec], cfg)
        I.synchronize()
        assert O.validate_x(bufs[prec][1].numpy().astype(np.float64)) == 0, prec
    I.free_device_analysis(mat, info)


def test_analyses_freed_while_values_change():
    """One thread updates a matrix's values and solves while another releases
    other analyses of it, whose plans go with them."""
    import threading

    s = I.generate(1, 40)
    mat = I.allocate_memory(s.ia, s.ja, s.a)
    cfg = I._cfg(kernel=I.KERNEL_ORDER, lanes=4, variant=4)
    db, dx = I.DeviceArray.from_numpy(s.b), I.DeviceArray(s.n, np.float64)
    keep, others = I.multirow_analysis_base_GPU(mat, I.ORDER), []
    for _ in range(40):
        others.append(I.multirow_analysis_base_GPU(mat, I.ORDER))
        I.solve(mat, others[-1], I.PREC_F64, db, dx, cfg=cfg)
    I.synchronize()

    def release():
        for info in others:
            I.free_device_analysis(None, info)

    t = threading.Thread(target=release)
    t.start()
    for i in range(60):
        scale = 2.0 ** (i % 3 - 1)
        I.update_values(mat, s.a * scale)
        I.solve(mat, keep, I.PREC_F64, db, dx, cfg=cfg)
        assert np.array_equal(dx.numpy(), np.full(s.n, 1.0 / scale))
    t.join()
    I.free_device_analysis(mat, keep)


@pytest.mark.parametrize("mode", [I.ORDER, I.MULTIROW, I.ALL])
def test_first_solve_beside_a_capture(mode):
    """The first solve with an analysis allocates nothing and waits for nothing:
    it runs while another stream is captured in the mode that forbids both."""
    hip = L.lib()
    s = I.generate(1, 200)
    mat = I.allocate_memory(s.ia, s.ja, s.a)
    info = I.multirow_analysis_base_GPU(mat, mode)
    db, dx = I.DeviceArray.from_numpy(s.b), I.DeviceArray(s.n, np.float64)
    b32, x32 = I.DeviceArray.from_numpy(s.b.astype(np.float32)), I.DeviceArray(s.n, np.float32)
    dx.fill_bytes(0)
    x32.fill_bytes(0)
    I.synchronize()
    streams = [ctypes.c_void_p() for _ in range(2)]
    for st in streams:
        assert hip.hipStreamCreateWithFlags(ctypes.byref(st), 1) == 0      # not tied to the null stream
    graph, errors = ctypes.c_void_p(), []
    assert hip.hipStreamBeginCapture(streams[0], 0) == 0                   # global mode
    try:
        if mode == I.MULTIROW:
            I.csr_L_solve_multirow(mat, info, db, dx, stream=streams[1])
            I.csr_L_solve_multirow_f32(mat, info, b32, x32, stream=streams[1])
        else:
            I.csr_L_solve_order(mat, info, db, dx, stream=streams[1])
            I.csr_L_solve_order_f32(mat, info, b32, x32, stream=streams[1])
    except L.SptrsvError as e:
        errors.append(str(e))
    ended = hip.hipStreamEndCapture(streams[0], ctypes.byref(graph))
    assert not errors and ended == 0
    assert hip.hipGraphDestroy(graph) == 0
    assert hip.hipStreamSynchronize(streams[1]) == 0
    assert O.validate_x(dx.numpy()) == 0 and np.all(x32.numpy() == 1.0)
    for st in streams:
        assert hip.hipStreamDestroy(st) == 0
    I.free_device_analysis(mat, info)


@pytest.mark.parametrize("gen,param,walk", [(1, 64, True), (1, 250, True), (1, 600, False), (2, 2000, True),
                                            (2, 8000, False), (3, 2000, False)])
def test_walk_is_the_default_where_it_wins(gen, param, walk):
    """The default shape of an ORDER solve on both sides of each line: levels
    of the matrix of at most 16 KB with rows of up to 4 off-diagonals (2D grids
    of 64^2 and 250^2, not of 600^2), 6 KB with longer ones (random), and no rows
    of more than 64 (power law)."""
    s = I.generate(gen, param)
    mat = I.allocate_memory(s.ia, s.ja, s.a)
    info = I.multirow_analysis_base_GPU(mat, I.ORDER)
    assert (I.default_config(mat, info, I.PREC_F64, 1).variant == 4) == walk
    I.free_device_analysis(mat, info)
