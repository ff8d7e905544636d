"""The fused mixed-precision normal equations where the kernel's shapes change: variable counts at
the edges of its 8-, 16- and 32-row blocks, of one and two variables per lane and of the two tile
grids; tuples of 1 ... 600 rays (1, 2 and 4 waves, one to three chunks, ragged ends); rays, waves and
whole first chunks that fail. Against the FP64 stored-Jacobian path in the bounds of its arithmetic:
with u_bf = 2^-8, u_f = 2^-24, ||dA||_F <= (3 u_bf^2 + 514 u_f) ||J||_F^2 (the dropped lo lo product,
the float rounding of the staged gradients, the float accumulation of up to 512 rays) and
||dg|| <= 4 u_f ||J||_F ||r|| (the gradients' float rounding; J^T r accumulates in FP64)."""

import numpy as np
import pytest

from mikroptim_amd import abi, systems
from mikroptim_amd.batch import ResidualSettings

pytestmark = pytest.mark.gpu

U_BF, U_F = 2.0 ** -8, 2.0 ** -24


def _check(engine, base, s, v, x):
    J, r0, ad, gd = engine.jacobian(base, s, v, x, method="adjoint", precision="fp64")
    a, g = engine.normal_equations(base, s, v, x, method="adjoint", precision="mixed")
    nJ = np.linalg.norm(J.reshape(len(x), -1), axis=1)
    nr = np.linalg.norm(r0, axis=1)
    assert np.isfinite(a).all() and np.isfinite(g).all()
    assert np.all(np.linalg.norm(a - ad, axis=(1, 2)) <= (3 * U_BF ** 2 + 514 * U_F) * nJ ** 2)
    assert np.all(np.linalg.norm(g - gd, axis=1) <= 4 * U_F * nJ * nr)
    assert np.array_equal(a, np.swapaxes(a, 1, 2))
    return J


@pytest.mark.parametrize("P", [1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 79, 80,
                               81, 95, 96])
@pytest.mark.parametrize("rings,spokes", [(6, 8), (5, 25), (9, 30)])
def test_variable_counts(engine, P, rings, spokes):
    b, v = systems.uneven_topology(0, variants=3, surfaces=32, variables=P)
    s = ResidualSettings(rings=rings, spokes=spokes, failure=abi.FAILURE_HARD)
    _check(engine, b.take([0]), s, v, v.extract(b)[:2])


@pytest.mark.parametrize("rings,spokes", [(1, 1), (1, 63), (4, 16), (5, 13), (8, 16), (3, 43),
                                          (16, 16), (1, 257), (8, 64), (3, 200)])
def test_tuple_sizes(engine, rings, spokes):
    b, v = systems.objective(variants=3, seed=2, fields=2, wavelengths=2)
    s = ResidualSettings(rings=rings, spokes=spokes, failure=abi.FAILURE_HARD)
    _check(engine, b.take([0]), s, v, v.extract(b)[1:])


@pytest.mark.parametrize("radius", [5.5, 8.0, 60.0])
@pytest.mark.parametrize("rings,spokes", [(6, 12), (4, 32), (16, 32)])
def test_failing_rays(engine, rings, spokes, radius):
    """The front radius at 5 mm: outer rings miss (from single rays to whole waves, to every ray of
    some tuples)."""
    b, v = systems.singlet(2)
    b.curvature[:, 1] = 0.2
    b.pupil_radius[:] = radius
    s = ResidualSettings(rings=rings, spokes=spokes, failure=abi.FAILURE_HARD)
    base = b.take([0])
    _, _, st = engine.residuals(base, s)
    assert (st != 0).any()
    v.upper[:2] = 0.3
    _check(engine, base, s, v, v.extract(b)[:1])


def test_outer_rays_first(engine):
    """Ring-major order starts at the axis; a point source far off the axis makes the first chunk of
    some waves fail while later ones reach the image."""
    b, v = systems.point_singlet(point=(0.0, 40.0, -300.0), na=0.12)
    s = ResidualSettings(rings=16, spokes=40, failure=abi.FAILURE_HARD)
    _check(engine, b.take([0]), s, v, v.extract(b)[:2])
