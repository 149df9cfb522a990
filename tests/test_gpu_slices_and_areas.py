"""Slices (summed over their axis in the spectrum, then transformed as a plane) against the planes of the
inverse transform, and iso-surface areas against numpy, over every axis, first, middle and last planes,
grids longest along each axis, states with the removed modes and without, both precisions.

A slice is the same sum in another order: 1e-13 (FP64) and 2e-6 (FP32) of the field's rms per value.
The area is the sum of numpy's terms on the same physical values: 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(16, 24, 32), (1024, 16, 24), (24, 1024, 16), (16, 24, 1024), (96, 48, 128), (32, 512, 16)]


def _state(g, engine, n, prec, clean):
    s = g.Solver(g.Config(n=n, L=(3.0, 2 * np.pi, 4.0), re=300.0, sc=(0.7,), theta=0.2, noise_kmax=4.0, noise_amp=0.2,
                          dt=1e-4, precision=prec), engine).setup()
    if clean:
        s.step(1)
    else:
        rng = np.random.default_rng(5)
        for f in range(4):
            s.set_physical(f, rng.standard_normal(n))
            s.forward(f)
    return s


@pytest.mark.parametrize("clean", [True, False])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", GRIDS, ids=lambda n: "x".join(map(str, n)))
def test_slices_are_the_planes_of_the_field(g, engine, n, prec, clean):
    s = _state(g, engine, n, prec, clean)
    tol = 2e-6 if prec else 1e-13
    for f in (0, 3):
        before = s.get_spectral(f)
        s.inverse(f)
        p = s.get_physical(f)
        rms = np.sqrt((p ** 2).mean())
        for axis in range(3):
            for index in (0, n[axis] // 2, n[axis] - 1):
                got = s.slice(f, axis, index)
                ref = np.take(p, index, axis)
                assert got.shape == ref.shape
                assert np.abs(got - ref).max() <= 20 * tol * rms, (f, axis, index)
                assert np.sqrt(((got - ref) ** 2).mean()) <= tol * rms, (f, axis, index)
        assert np.array_equal(s.get_spectral(f), before)
    s.close()


@pytest.mark.parametrize("clean", [True, False])
@pytest.mark.parametrize("n", GRIDS, ids=lambda n: "x".join(map(str, n)))
def test_areas_match_numpy(g, engine, n, clean):
    s = _state(g, engine, n, 0, clean)
    L = (3.0, 2 * np.pi, 4.0)
    s.inverse(3)
    F = s.get_physical(3)
    iso = float(F.mean()) + 1e-3
    d = [a / b for a, b in zip(L, n)]
    chi = (F <= iso).astype(float)
    grad = lambda a: [(np.roll(a, -1, i) - np.roll(a, 1, i)) / (2 * d[i]) for i in range(3)]
    gF, gC = grad(F), grad(chi)
    size = np.sqrt(sum(v * v for v in gF))
    dot = -sum(a * b for a, b in zip(gF, gC))
    ref = np.where(size > 0, dot / np.where(size > 0, size, 1), 0).sum() * d[0] * d[1] * d[2]
    assert abs(s.surface_area(3, iso) - ref) <= 1e-12 * abs(ref)
    s.close()
