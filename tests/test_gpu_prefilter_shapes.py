"""The prefilter kernel where its shapes change: tuples of 1 ... 2048 rays (8, 16, 32 and 64 lanes per
tuple and whole workgroups; full, ragged and mostly idle last rays; one ring, one spoke), batches
that are traced with more lanes than they are summed with, a last workgroup of few variants. Ray
classes are the oracle's; a variant's values do not depend on the batch it is in, bit for bit. The
merits: sqrt(F) is the 2-norm of residuals whose weights add up to 1, so it moves by at most the
error of an optical length over the wavelength; in float, over 3 surfaces, that error is some 12 u
of the length on either path (a rounding of the sum per surface, 4 of the steps, as many from the
positions), u = 2^-24: 24 u between the two. (Relative to F the difference has no bound: a tuple of
one ring or of near-perfect focus has residuals in the rounding of its lengths.)"""

import numpy as np
import pytest

from mikroptim_amd import abi, systems
from mikroptim_amd.batch import ResidualSettings
from oracle_lib import oracle
from test_prefilter import stats

pytestmark = pytest.mark.gpu

U_F = 2.0 ** -24
NAMES = ("merit", "optical_length", "failed", "uncertain_ok", "uncertain_failed")


@pytest.mark.parametrize("rings,spokes", [(1, 1), (1, 7), (1, 8), (3, 3), (3, 5), (2, 16), (3, 11),
                                          (6, 12), (4, 16), (5, 13), (3, 43), (8, 16), (16, 16),
                                          (1, 257), (16, 17), (16, 128)])
def test_tuple_sizes(engine, rings, spokes):
    b, _ = systems.singlet_multistart(2001, seed=17)
    s = ResidualSettings(rings=rings, spokes=spokes, failure=abi.FAILURE_HARD)
    g = engine.prefilter(b, s)
    for count in (1, 3, 130):
        part = engine.prefilter(b.take(np.arange(count)), s)
        for name in NAMES:
            assert np.array_equal(getattr(part, name), getattr(g, name)[:count]), (name, count)
    count = 130
    o = stats(oracle(), b.take(np.arange(count)), s)
    for name in NAMES[2:]:
        assert np.array_equal(getattr(g, name)[:count], getattr(o, name)), name
    d = np.abs(np.sqrt(g.merit[:count]) - np.sqrt(o.merit))
    assert np.all(d <= 24 * U_F * o.optical_length / (b.reference_wavelength_nm * 1e-6))
    assert np.max(np.abs(g.optical_length[:count] - o.optical_length) /
                  np.maximum(o.optical_length, 1e-30)) <= 1e-5


@pytest.mark.parametrize("rings,spokes", [(3, 5), (6, 12), (16, 16), (16, 32)])
def test_many_surfaces(engine, rings, spokes):
    b, _ = systems.objective(variants=70, seed=4)
    s = ResidualSettings(rings=rings, spokes=spokes, failure=abi.FAILURE_HARD)
    g = engine.prefilter(b, s)
    one = engine.prefilter(b.take([69]), s)
    for name in NAMES:
        assert np.array_equal(getattr(one, name), getattr(g, name)[69:]), name
    m, f, _ = engine.merit(b, s)
    assert np.all(g.failed == 0) and np.all(f == 0)
    assert np.all(g.merit_lower <= m) and np.all(m <= g.merit_upper)


def test_axis_fields_take_any_number_of_spokes(engine):
    """An axis field has one spoke, whatever the settings say."""
    b, _ = systems.singlet_multistart(40, seed=5)
    b.pupil_mode = np.full(b.fields, abi.PUPIL_AXIS, dtype=np.uint8)
    g = [engine.prefilter(b, ResidualSettings(rings=6, spokes=n, failure=abi.FAILURE_HARD))
         for n in (1, 50000)]
    for name in NAMES:
        assert np.array_equal(getattr(g[0], name), getattr(g[1], name)), name
