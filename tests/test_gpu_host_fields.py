"""Fields to and from host buffers: spectral and physical round trips against numpy over the edges of the
transfer (one slot, several slots, a last chunk of a few rows, kx-ky planes larger than a slot, rows of
every padding), from several host threads with a context each, and at odd offsets of a caller's array.

The values only change type on the way, so they come back bit for bit."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(16, 16, 16), (24, 48, 16), (96, 64, 192), (1024, 16, 1024), (16, 1024, 24), (128, 192, 96)]


def _case(g, engine, n, prec, seed):
    s = g.Solver(g.Config(n=n, sc=(), precision=prec), engine)
    s.init_wavenumbers()
    rng = np.random.default_rng(seed)
    real = np.float32 if prec else np.float64
    x = rng.standard_normal(n).astype(real).astype(np.float64)
    h = (n[1], n[0], n[2] // 2 + 1)
    q = (rng.standard_normal(h).astype(real) + 1j * rng.standard_normal(h).astype(real)).astype(np.complex128)
    s.set_physical(1, x)
    s.set_spectral(2, q)
    assert np.array_equal(s.get_physical(1), x)
    assert np.array_equal(s.get_spectral(2), q)
    # the spectral order: a forward transform against numpy's, read in [ky][kx][kz]
    s.set_physical(0, x)
    s.forward(0)
    ref = np.fft.rfftn(x).transpose(1, 0, 2)
    assert np.linalg.norm(s.get_spectral(0) - ref) <= (2e-6 if prec else 1e-13) * np.linalg.norm(ref)
    # the kz padding holds zeros: the inverse of what was set is numpy's
    s.set_spectral(0, ref)
    s.inverse(0)
    assert np.linalg.norm(s.get_physical(0) - x) <= (2e-6 if prec else 1e-13) * np.linalg.norm(x)
    s.close()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", GRIDS, ids=lambda n: "x".join(map(str, n)))
def test_fields_come_back_bit_for_bit(g, engine, n, prec):
    _case(g, engine, n, prec, 1)


def test_fields_from_several_threads(g, engine):
    bad = []

    def one(seed):
        try:
            for _ in range(3):
                _case(g, engine, (96, 64, 128), seed % 2, seed)
        except BaseException as e:  # noqa: B902
            bad.append(e)

    th = [threading.Thread(target=one, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad


def test_fields_into_part_of_an_array(g, engine):
    import ctypes
    n = (48, 32, 96)
    s = g.Solver(g.Config(n=n, sc=()), engine)
    x = np.random.default_rng(6).standard_normal(n)
    s.set_physical(0, x)
    buf = np.full(x.size + 6, -7.0)
    part = buf[3:3 + x.size]
    rc = engine.gnss_get_field(s.ctx, 0, g.PHYSICAL, part.ctypes.data_as(ctypes.POINTER(ctypes.c_double)))
    assert rc == 0 and np.array_equal(part.reshape(n), x)
    assert (buf[:3] == -7.0).all() and (buf[-3:] == -7.0).all()
