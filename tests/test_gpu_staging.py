"""Transfers through the engine's pinned slots where their shapes change: calls whose arrays share a
slot, fill several and pass through all of them more than once (more than 8 MiB up and down), after
calls of other sizes, and after a call that failed. Every variant's results are those of a call of
its own size class: equal bits."""

import numpy as np
import pytest

from mikroptim_amd import abi, systems
from mikroptim_amd.batch import ResidualSettings

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variants", [1, 3, 180, 1700])
def test_downloads(engine, variants):
    b, _ = systems.singlet_multistart(variants, seed=3)
    s = systems.singlet_settings(abi.FAILURE_SOFT)
    res, opd, status = engine.residuals(b, s)  # 1700 variants: 26 MB
    for at in sorted({0, variants // 2, variants - 1}):
        r1, o1, s1 = engine.residuals(b.take([at]), s)
        assert np.array_equal(res[at], r1[0], equal_nan=True)
        assert np.array_equal(opd[at], o1[0], equal_nan=True)
        assert np.array_equal(status[at], s1[0])


@pytest.mark.parametrize("variants", [1, 40, 5000])
def test_uploads(engine, variants):
    b, _ = systems.objective(variants=variants, seed=6)  # 5000 variants: 11 MB
    s = ResidualSettings(rings=2, spokes=3, failure=abi.FAILURE_HARD)
    m, f, h = engine.merit(b, s)
    ids = np.unique(np.linspace(0, variants - 1, 30).astype(int))
    m1, f1, h1 = engine.merit(b.take(ids), s)
    assert np.array_equal(m[ids], m1) and np.array_equal(f[ids], f1) and np.array_equal(h[ids], h1)


def test_points_after_a_refused_call(engine):
    b, v = systems.objective(variants=5, seed=6)
    s = ResidualSettings(rings=3, spokes=5, failure=abi.FAILURE_HARD)
    x = v.extract(b)
    a, g = engine.normal_equations(b.take([0]), s, v, x, method="fd")
    bad = x.copy()
    bad[2, 1] = np.nan
    for method in ("fd", "adjoint"):
        with pytest.raises(Exception):
            engine.normal_equations(b.take([0]), s, v, bad, method=method)
    a1, g1 = engine.normal_equations(b.take([0]), s, v, x, method="fd")
    assert np.array_equal(a, a1) and np.array_equal(g, g1)
    for i in range(5):
        ai, gi = engine.normal_equations(b.take([0]), s, v, x[i:i + 1], method="fd")
        assert np.array_equal(ai[0], a[i]) and np.array_equal(gi[0], g[i])


def test_points_of_more_than_two_slots(engine):
    b, v = systems.singlet(2)
    runs = (5 << 19) // (8 * v.size) + 1  # 2.5 MiB of points and of each array of the pattern
    x = v.extract(b)[1] * (1.0 + 1e-3 * np.random.default_rng(8).standard_normal((runs, v.size)))
    s = ResidualSettings(rings=1, spokes=2, failure=abi.FAILURE_HARD)
    a, g = engine.normal_equations(b.take([0]), s, v, x, method="fd")
    ids = np.unique(np.linspace(0, runs - 1, 40).astype(int))
    a1, g1 = engine.normal_equations(b.take([0]), s, v, x[ids], method="fd")
    assert np.array_equal(a[ids], a1) and np.array_equal(g[ids], g1)
