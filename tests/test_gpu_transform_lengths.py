"""Every transform length with a factor of three, along each axis, against numpy's 64-bit transform.

The tolerances are the rounding of the transforms: eps * (a few) * log2(points) relative to the
norm, 1e-13 in FP64 and 2e-6 in FP32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [(24, 48, 96), (48, 96, 192), (96, 192, 24), (192, 24, 384), (384, 16, 48)],
                         ids=lambda n: "x".join(map(str, n)))
def test_lengths_with_a_factor_of_three(g, engine, n, prec):
    tol = 2e-6 if prec else 1e-13
    s = g.Solver(g.Config(n=n, sc=(), precision=prec), engine)
    x = np.random.default_rng(5).standard_normal(n)
    s.set_physical(0, x)
    s.forward(0)
    ref = np.fft.rfftn(x).transpose(1, 0, 2)
    assert np.linalg.norm(s.get_spectral(0) - ref) <= tol * np.linalg.norm(ref)
    s.inverse(0)
    assert np.linalg.norm(s.get_physical(0) - x) <= tol * np.linalg.norm(x)
