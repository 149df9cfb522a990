"""A colloid's substage with every derivative taken in the inverse pass of its own axis, lap Z among them
(x modes 2 and 3), against the oracle and against the group-fused mode 1, over every fused z variant, with two
to four scalars and on grids small enough for single-output x entries and too large for them.  FP64: 1e-12 of the
norm, the bar of the other step tests; FP32 forms of one step agree to 2e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(16, 24, 48), (96, 128, 96), (256, 192, 128), (24, 16, 384), (32, 16, 1024)]


@pytest.mark.parametrize("n", GRIDS, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("sc", [(0.7,), (0.7, 2.0, 0.5)], ids=["2 scalars", "4 scalars"])
def test_colloid_derivatives_per_axis(g, engine, oracle, n, sc):
    cfg = g.with_colloid(g.Config(n=n, re=400.0, sc=sc, theta=0.2, noise_kmax=6.0, noise_amp=0.2, dt=5e-4), alpha=0.02)
    F = 4 + len(sc)

    def run(lib, prec, tuning=None):
        s = g.Solver(g.Config(**{**cfg.__dict__, "precision": prec}), lib).setup()
        if tuning:
            s.set_tuning(tuning)
        s.step(2)
        out = [s.get_spectral(f) for f in range(F)]
        s.close()
        return out

    def check(got, ref, tol, what):
        for f in range(F):
            assert np.linalg.norm(got[f] - ref[f]) <= tol * np.linalg.norm(ref[f]), (what, f)

    ref = run(oracle, 0)
    ref32 = run(engine, 1, "xf=1 zf=3 xc=8")
    for xf in (2, 3):
        for zf in (0, 3, 6, 7, 8, 10)[:5 + (n[2] <= 512)]:
            check(run(engine, 0, f"xf={xf} zf={zf} xc=4"), ref, 1e-12, (xf, zf))
        for zf in (0, 1, 2, 3, 4, 5, 6, 7, 10)[:8 + (n[2] <= 512)]:
            check(run(engine, 1, f"xf={xf} zf={zf} xc=8"), ref32, 2e-6, (xf, zf))
