"""Inverse transforms of a state the engine knows to be dealiased (only kept columns and rows are read)
against the same state written from outside (every mode is read), and the bookkeeping behind it: any
write from outside is dealiased again by the next step and seen whole by inverse, statistics and slices.

Both sides transform the same numbers in another pass order: rounding of the transforms, 1e-13 (FP64)
and 2e-6 (FP32) of the norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(16, 24, 32), (96, 64, 48), (32, 16, 1024), (512, 16, 16), (16, 512, 24)]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", GRIDS, ids=lambda n: "x".join(map(str, n)))
def test_clean_state_transforms_alike(g, engine, n, prec):
    tol = 2e-6 if prec else 1e-13
    cfg = g.Config(n=n, re=300.0, sc=(0.7, 1.0), theta=0.2, noise_kmax=4.0, noise_amp=0.2, dt=1e-3, precision=prec)
    a = g.Solver(cfg, engine).setup()
    a.step(1)
    b = g.Solver(cfg, engine)
    b.init_wavenumbers()
    for f in range(5):
        b.set_spectral(f, a.get_spectral(f))
    for cp in (0, 1):
        for s in (a, b):
            s.set_tuning(f"cp={cp} zp={cp}")
        for f in range(5):
            for s in (a, b):
                s.inverse(f)
            x, y = a.get_physical(f), b.get_physical(f)
            assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y)
            assert np.linalg.norm(a.slice(f) - y[:, :, n[2] // 2]) <= tol * np.linalg.norm(y)
        w = [s.slice(g.FIELD_VORTICITY, 1) for s in (a, b)]
        assert np.linalg.norm(w[0] - w[1]) <= 20 * tol * np.linalg.norm(w[1])  # k amplifies the rounding
        (sa, pa, ea), (sb, pb, eb) = a.stats(), b.stats()
        assert np.array_equal(ea, eb)  # spectral sums read the same numbers
        assert np.abs(pa - pb).max() <= tol * np.abs(pb).max()


def test_writes_from_outside_are_seen_whole_and_dealiased(g, engine, oracle):
    n = (24, 32, 48)
    cfg = g.Config(n=n, re=300.0, sc=(0.7,), theta=0.2, noise_kmax=4.0, noise_amp=0.2, dt=1e-3)
    rng = np.random.default_rng(2)
    x = [0.3 * rng.standard_normal(n) for _ in range(4)]
    out = []
    for lib in (engine, oracle):
        s = g.Solver(cfg, lib).setup()
        s.step(1)
        got = []
        for f in range(4):  # physical fields with every mode, over a clean state
            s.set_physical(f, x[f])
            s.forward(f)
        s.inverse(0)
        got.append(s.get_physical(0))
        got.append(s.slice(3))
        s.step(1)
        got += [s.get_spectral(f) for f in range(4)]
        q = s.get_spectral(1)
        q[n[1] // 2 - 1, n[0] // 2 - 1, 3] = 5.0  # a removed mode, then again a step
        s.set_spectral(1, q)
        s.step(1)
        got += [s.get_spectral(f) for f in range(4)]
        out.append(got)
        s.close()
    assert np.abs(out[0][0] - x[0]).max() < 1e-12
    for a, b in zip(*out):
        assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(b)
