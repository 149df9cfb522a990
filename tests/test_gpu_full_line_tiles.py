"""Passes of 1024 rows take tiles of whole memory lines where they are given half ones: whole transforms against numpy,
two steps against the oracle (FP64) and FP64 (FP32), with the long side along x, along y and along both, and a kept
kz range that ends inside a tile, at its end and in its first half.  FP64: 1e-14 for a transform, 1e-12 for the
steps; FP32: 1e-6 and 5e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1024, 24, 16), (24, 1024, 96), (1024, 32, 64), (32, 1024, 24), (1024, 1024, 16)],
                         ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("colloid", [False, True], ids=["plain", "colloid"])
def test_long_passes(g, engine, oracle, n, colloid):
    cfg = g.Config(n=n, re=400.0, sc=(0.7,), theta=0.2, noise_kmax=4.0, noise_amp=0.2, dt=5e-4)
    if colloid:
        cfg = g.with_colloid(cfg, alpha=0.02)
    F = 3 + len(cfg.sc)
    p = np.random.default_rng(4).standard_normal(n)
    want = np.fft.rfftn(p).transpose(1, 0, 2)
    out = []
    for lib, prec in ((oracle, 0), (engine, 0), (engine, 1)):
        s = g.Solver(g.Config(**{**cfg.__dict__, "precision": prec}), lib).setup()
        s.step(2)
        out.append([s.get_spectral(f) for f in range(F)])
        s.set_physical(0, p)
        s.forward(0)
        tol = 1e-6 if prec else 1e-14
        assert np.linalg.norm(s.get_spectral(0) - want) <= tol * np.linalg.norm(want), prec
        s.inverse(0)
        assert np.linalg.norm(s.get_physical(0) - p) <= tol * np.linalg.norm(p), prec
        s.close()
    for f in range(F):
        size = np.linalg.norm(out[0][f])
        assert np.linalg.norm(out[1][f] - out[0][f]) <= 1e-12 * size, f
        assert np.linalg.norm(out[2][f] - out[0][f]) <= 5e-6 * size, f
