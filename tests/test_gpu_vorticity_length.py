"""The vorticity magnitude, whose length is taken in the z pass of its three components, against the oracle on the
same spectra: every row length, both precisions, states with the removed modes and without.  FP64: 1e-12 of the
field's largest value; FP32: 5e-6 (three transforms and a square root)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("clean", [True, False])
@pytest.mark.parametrize("prec", [0, 1], ids=["f64", "f32"])
@pytest.mark.parametrize("nz", [16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512, 1024])
def test_vorticity_length_matches_the_oracle(g, engine, oracle, nz, prec, clean):
    n = (24, 16, nz)
    cfg = dict(n=n, L=(3.0, 2 * np.pi, 4.0), re=300.0, theta=0.2, noise_kmax=4.0, noise_amp=0.2, dt=1e-4)
    s = g.Solver(g.Config(precision=prec, **cfg), engine).setup()
    if clean:
        s.step(1)
    else:
        rng = np.random.default_rng(5)
        for f in range(3):
            s.set_physical(f, rng.standard_normal(n))
            s.forward(f)
    ref = g.Solver(g.Config(**cfg), oracle)
    ref.init_wavenumbers()
    for f in range(3):
        ref.set_spectral(f, s.get_spectral(f))
    planes = [(axis, i, s.slice(g.FIELD_VORTICITY, axis, i), ref.slice(g.FIELD_VORTICITY, axis, i))
              for axis in range(3) for i in (0, n[axis] - 1)]
    size = max(np.abs(p[3]).max() for p in planes)
    for axis, i, got, want in planes:
        assert np.abs(got - want).max() <= (5e-6 if prec else 1e-12) * size, (axis, i)
    s.close()
    ref.close()
