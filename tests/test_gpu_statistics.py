"""The statistics kernels against the oracle on states that are not dealiased, over the edges of their
dispatch: rows shorter and longer than a wave, no scalar to four, one wave per row of bins up to
sixteen, bins that fit the LDS of fewer waves, and shells too many for the LDS.

FP64, both sides on the same physical fields.  The engine and the oracle add the same up to 1e6 terms in
different orders and transform with different FFTs: 1e-12 of the largest value covers both."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TWO_PI = 2 * np.pi


@pytest.mark.parametrize("n,L,S", [((16, 16, 16), (TWO_PI,) * 3, 4), ((24, 48, 192), (TWO_PI, 2.5, 3.1), 0),
                                   ((32, 16, 1024), (TWO_PI,) * 3, 1), ((16, 384, 64), (TWO_PI, 5.1, 2.9), 2),
                                   ((256, 16, 16), (0.5, TWO_PI, TWO_PI), 1),
                                   ((256, 16, 16), (0.1, TWO_PI, TWO_PI), 1)],
                         ids=lambda v: "x".join(str(x)[:4] for x in v) if isinstance(v, tuple) else str(v))
def test_statistics_match_the_oracle(g, engine, oracle, n, L, S):
    rng = np.random.default_rng(3)
    y = np.arange(n[1])[None, :, None] / n[1]
    fields = [rng.standard_normal(n) * 0.1 + (np.tanh(8 * (0.3 - abs(y - 0.5))) if f in (0, 3) else 0.02 * f)
              for f in range(3 + S)]
    out = []
    for lib in (engine, oracle):
        s = g.Solver(g.Config(n=n, L=L, re=300.0, sc=(0.7, 1.0, 2.0, 0.5)[:S], dt=1e-3), lib)
        s.init_wavenumbers()
        for f, a in enumerate(fields):
            s.set_physical(f, a)
            s.forward(f)
        out.append((s.stats(), s.stats(False, False)))
        s.close()
    (a, a0), (b, _) = out
    for k in b[0]:
        x, r = np.asarray(a[0][k], float), np.asarray(b[0][k], float)
        assert np.abs(x - r).max(initial=0.0) <= 1e-12 * max(np.abs(r).max(initial=0.0), 1e-3), k
        assert np.array_equal(x, np.asarray(a0[0][k], float)), k  # the same without profiles and spectrum
    for x, r in zip(a[1:], b[1:]):
        assert np.abs(x - r).max() <= 1e-12 * np.abs(r).max()


def test_profile_moments_keep_small_fluctuations(g, engine):
    """Second moments of fluctuations a million times smaller than the mean: their error stays at the
    rounding of the mean (1e-16 of mean squared would be 1e-4 of them)."""
    n = (32, 16, 48)
    x = 1.0 + 1e-6 * np.random.default_rng(4).standard_normal(n)
    s = g.Solver(g.Config(n=n, sc=()), engine)
    s.init_wavenumbers()
    for f in range(3):
        s.set_physical(f, x)
        s.forward(f)
    _, prof, _ = s.stats()
    s.inverse(0)
    p = s.get_physical(0)
    ref = p.var(axis=(0, 2))
    assert np.abs(prof[3] - ref).max() <= 1e-9 * ref.max()
