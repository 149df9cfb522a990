"""FP64 fused z variant 7, whose exchanges are lane swaps for rows of 128, 256 and 512, against variant 6
(every exchange through LDS) and the oracle: zero to four scalars, work-field and late-derivative modes,
with a colloid.  The same radix stages on the same numbers: 1e-13 of the norm against variant 6 (which
also scales elsewhere), 1e-12 against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(g, lib, cfg, spec=None):
    s = g.Solver(cfg, lib).setup()
    if spec:
        s.set_tuning(spec)
    s.step(2)
    out = [s.get_spectral(f) for f in range(3 + len(cfg.sc))]
    s.close()
    return out


def _near(a, b, tol):
    for x, y in zip(a, b):
        assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y)


@pytest.mark.parametrize("nz", [128, 256, 512])
@pytest.mark.parametrize("S", [0, 1, 4])
def test_lane_swaps_match(g, engine, oracle, nz, S):
    cfg = g.Config(n=(24, 16, nz), re=400.0, sc=(0.7, 2.0, 1.0, 0.5)[:S], theta=0.08, noise_kmax=6.0, noise_amp=0.2,
                   dt=1e-3)
    ref = _run(g, oracle, cfg)
    for xf in (2, 4):
        old, new = (_run(g, engine, cfg, f"zf={zf} xf={xf}") for zf in (6, 7))
        _near(new, old, 1e-13)
        _near(new, ref, 1e-12)


@pytest.mark.parametrize("nz", [128, 256, 512])
def test_lane_swaps_match_with_a_colloid(g, engine, nz):
    cfg = g.with_colloid(g.Config(n=(16, 24, nz), re=400.0, sc=(0.7, 2.0), theta=0.08, noise_kmax=6.0, noise_amp=0.2,
                                  dt=1e-3), alpha=0.02)
    _near(_run(g, engine, cfg, "zf=7"), _run(g, engine, cfg, "zf=6"), 1e-13)
