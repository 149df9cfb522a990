"""Fused z variant 10 (pairs of rows with a colloid) against variant 7 over every row length it is built
for, two to four scalars (the carrier alone, and with plain scalars before it), and refused elsewhere.
The same products in another transform: FP64 1e-13, FP32 2e-6 of the norm after two steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("nz", [16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512])
def test_pairs_with_a_colloid_match(g, engine, prec, nz):
    for sc in ((0.7,), (0.7, 2.0), (0.7, 2.0, 0.5)):
        cfg = g.with_colloid(g.Config(n=(32, 16, nz), re=400.0, sc=sc, theta=0.08, noise_kmax=6.0, noise_amp=0.2,
                                      dt=1e-3, precision=prec), alpha=0.02)
        out = []
        for zf in (7, 10):
            s = g.Solver(cfg, engine).setup()
            s.set_tuning(f"zf={zf}")
            s.step(2)
            out.append([s.get_spectral(f) for f in range(4 + len(sc))])
            s.close()
        for a, b in zip(*out):
            assert np.linalg.norm(a - b) <= (2e-6 if prec else 1e-13) * np.linalg.norm(b), sc


def test_variant_needs_a_colloid_and_short_rows(g, engine):
    plain = g.Config(n=(32, 16, 64), sc=(0.7, 2.0))
    for cfg in (plain, g.with_colloid(g.Config(n=(16, 16, 1024), sc=(0.7,)))):
        s = g.Solver(cfg, engine)
        with pytest.raises(g.GnssError):
            s.set_tuning("zf=10")
        s.close()
