"""Whole transforms of arrays beyond the last-level cache, whose x passes load a tile ahead, against numpy and back.
FP64 1e-14 and FP32 1e-6 of the norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec", [((256, 512, 512), 0), ((1024, 256, 512), 1)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else ("f32" if v else "f64"))
def test_large_whole_transforms(g, engine, n, prec):
    tol = 1e-6 if prec else 1e-14
    s = g.Solver(g.Config(n=n, precision=prec), engine)
    s.init_wavenumbers()
    p = np.random.default_rng(2).standard_normal(n)
    s.set_physical(0, p)
    s.forward(0)
    got = s.get_spectral(0)
    for ky in (0, 1, n[1] // 2, n[1] - 1):  # numpy along y for these rows only, then x and z
        w = np.exp(-2j * np.pi * (ky * np.arange(n[1]) % n[1]) / n[1])
        ref = np.fft.fft(np.fft.rfft(np.einsum("xyz,y->xz", p, w.real), axis=1)
                         + 1j * np.fft.rfft(np.einsum("xyz,y->xz", p, w.imag), axis=1), axis=0)
        assert np.linalg.norm(got[ky] - ref) <= tol * np.linalg.norm(ref), ky
    s.inverse(0)
    assert np.linalg.norm(s.get_physical(0) - p) <= tol * np.linalg.norm(p)
    s.close()
