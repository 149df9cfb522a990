"""Grids without an entry in the tuning table get their pass variants from a rule on sizes, precision and
the colloid; the step must give the oracle's numbers on every side of its lines (FP64: 1e-12 of the norm),
and the FP32 form FP64's to its usual error."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [((16, 1024, 24), 0, False), ((1024, 24, 16), 1, False), ((256, 128, 128), 1, False), ((512, 96, 96), 2, False),
         ((384, 48, 192), 1, False), ((24, 16, 1024), 1, False), ((48, 32, 512), 4, False), ((32, 48, 256), 1, False),
         ((96, 128, 96), 1, False), ((64, 48, 128), 3, False), ((256, 128, 128), 2, True), ((96, 64, 192), 3, True),
         ((32, 24, 1024), 2, True)]


@pytest.mark.parametrize("n,S,colloid", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_rule_matches_the_oracle(g, engine, oracle, n, S, colloid):
    cfg = g.Config(n=n, re=400.0, sc=(0.7, 1.0, 2.0, 0.5)[:S - colloid], theta=0.2, noise_kmax=4.0, noise_amp=0.2, dt=5e-4)
    if colloid:
        cfg = g.with_colloid(cfg, alpha=0.02)
    out = []
    for lib, prec in ((engine, 0), (engine, 1), (oracle, 0)):
        c = g.Config(**{**cfg.__dict__, "precision": prec})
        s = g.Solver(c, lib).setup()
        s.step(2)
        out.append([s.get_spectral(f) for f in range(3 + S)])
        s.close()
    for f in range(3 + S):
        norm = np.linalg.norm(out[2][f])
        assert np.linalg.norm(out[0][f] - out[2][f]) <= 1e-12 * norm, f
        assert np.linalg.norm(out[1][f] - out[2][f]) <= 5e-6 * norm, f
