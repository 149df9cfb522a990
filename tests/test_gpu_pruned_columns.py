"""The substage's strided passes under the 2/3 rule's ellipsoid (columns of removed modes passed over,
rows outside neither loaded nor stored) against the oracle: every x mode and tile width, grids whose
ellipsoid is stretched along each axis, lengths with one and several transform groups per block.

The start is white noise, so that the modes on the ellipsoid's border carry as much as the others, and
the second step meets the work buffers of the first.  FP64: 1e-12 of the norm, the bar of the other
step tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(16, 1024, 24), (1024, 16, 48), (16, 24, 512), (96, 128, 64), (24, 16, 1024)],
                         ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("batch", ["cb=0 cp=0", "cb=1 cp=0", "cb=1 cp=1"])
def test_pruned_passes_match_the_oracle(g, engine, oracle, n, batch):
    cfg = g.Config(n=n, re=200.0, sc=(0.7,), dt=2e-4)
    rng = np.random.default_rng(8)
    fields = [0.3 * rng.standard_normal(n) for _ in range(4)]

    def run(lib, tuning=None):
        s = g.Solver(cfg, lib)
        s.init_wavenumbers()
        if tuning:
            s.set_tuning(tuning)
        for f, a in enumerate(fields):
            s.set_physical(f, a)
            s.forward(f)
        s.dealias()
        s.step(2)
        out = [s.get_spectral(f) for f in range(4)]
        s.close()
        return out

    ref = run(oracle)
    removed = g.Solver(cfg, oracle)
    removed.init_wavenumbers()
    mask = removed.mask() == 0
    for xf in range(6):
        wide = 4 if max(n[0], n[1]) > 512 else 8
        for c in sorted({4, wide}):
            got = run(engine, f"{batch} xf={xf} xc={c} cx={c} cy={c}")
            for f in range(4):
                assert np.linalg.norm(got[f] - ref[f]) <= 1e-12 * np.linalg.norm(ref[f]), (xf, c, f)
                assert not got[f][mask].any(), (xf, c, f)  # removed modes stay zero
