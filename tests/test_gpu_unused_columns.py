"""The last column tile of a substage's passes reaches past the kept modes; what lies there is neither read
nor of any consequence.  The work arrays of one solver hold NaN from an earlier state, another's are
fresh: their steps have to agree bit by bit, in every x mode, where the kept modes end inside a tile,
at its end and where they fill less than half of one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [16, 24, 64, 96, 192])
@pytest.mark.parametrize("prec", [0, 1], ids=["f64", "f32"])
@pytest.mark.parametrize("colloid", [False, True], ids=["plain", "colloid"])
def test_steps_do_not_see_the_columns_without_modes(g, engine, nz, prec, colloid):
    n = (32, 24, nz)
    cfg = g.Config(n=n, re=200.0, sc=(0.7, 1.3), precision=prec, dt=2e-4)
    if colloid:
        cfg = g.with_colloid(cfg, sc_c=2.0, alpha=0.3)
    F = 3 + len(cfg.sc)
    rng = np.random.default_rng(3)
    fields = [0.3 * rng.standard_normal(n) for _ in range(F)]

    def start(tuning, before):
        s = g.Solver(cfg, engine)
        s.init_wavenumbers()
        s.set_tuning(tuning)
        for values in (before, fields) if before else (fields,):
            for f, a in enumerate(values):
                s.set_physical(f, a)
                s.forward(f)
            if values is before:
                for f in range(F):
                    s.inverse(f)
        s.dealias()
        return s

    for xf in range(4 if colloid else 6):
        for tuning in (f"cb=1 cp=0 xf={xf}", f"cb=0 cp=1 xf={xf}"):
            out = []
            for before in (None, [np.full(n, np.nan)] * F):
                s = start(tuning, before)
                s.step(2)
                out.append([s.get_spectral(f) for f in range(F)])
                s.close()
            for f in range(F):
                assert np.isfinite(out[0][f]).all(), (tuning, f)
                assert np.array_equal(out[0][f], out[1][f]), (tuning, f)
