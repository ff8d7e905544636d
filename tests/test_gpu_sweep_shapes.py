"""The reverse sweep's kernels (stored Jacobian, vector-Jacobian product) where their launch shapes
change: tuples of 1 ... 2048 rays around the edges of a wave, of a workgroup of 1 ... 4 waves and of
1, 2, 4 and 8 rays per lane; hard and soft failure with failing rays; glass variables; the three
reference spheres; a point source; a curvature variable on a plane, which no ray's sweep reaches.
Columns against the oracle's adjoint Jacobian: relative 1e-10 (kAdjointCpuGpu), or 4e-16 * n_rays^(1/2)
of the unprojected gradients' size where the oracle's own columns hold no more digits (a thickness
gradient is n plus its variation over the pupil: the oracle's rounding, 2^-53 of n per operation over
a few operations per surface, stays when the common part is projected out)."""

import numpy as np
import pytest

from mikroptim_amd import abi, systems
from mikroptim_amd.batch import ResidualSettings, rays_per_variant
from oracle_lib import oracle

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (3, 21), (4, 16), (5, 13), (8, 16), (16, 16), (1, 257), (9, 57), (16, 65),
          (16, 128)]


def _scales(base, s):
    """Largest residual scale of a tuple, for the rounding floor of a column."""
    w = np.outer(base.field_weight / base.field_weight.sum(),
                 base.wavelength_weight / base.wavelength_weight.sum())
    return float(np.sqrt(w.max()) / (base.reference_wavelength_nm * 1e-6))


def _check(engine, base, s, v, x, seed=0):
    J, r0, a, g = engine.jacobian(base, s, v, x, method="adjoint", precision="fp64")
    Jo, r0o, _ = oracle().adjoint_jacobian(base, s, v, x)
    rays = rays_per_variant(base, s)
    floor = 4e-16 * _scales(base, s) * np.sqrt(base.fields * base.wavelengths)
    err = np.linalg.norm((J - Jo)[:, :, :rays], axis=2)
    ref = np.linalg.norm(Jo[:, :, :rays], axis=2)
    assert np.all(err <= 1e-10 * ref + floor), (err / (ref + floor)).max()
    if s.failure == abi.FAILURE_SOFT:
        perr = np.linalg.norm((J - Jo)[:, :, rays:], axis=2)
        assert np.all(perr <= 1e-9 * np.linalg.norm(Jo[:, :, rays:], axis=2))
    if not v.has_glass:
        import torch
        from mikroptim_amd.autograd import trace_residuals

        xt = torch.tensor(x, dtype=torch.float64, device="cuda", requires_grad=True)
        r = trace_residuals(xt, engine, base, s, v)
        grad = np.random.default_rng(seed).standard_normal(J.shape[::2])
        r.backward(torch.tensor(grad, device="cuda"))
        gx = xt.grad.cpu().numpy()
        want = np.einsum("npr,nr->np", J, grad)
        size = np.linalg.norm(J, axis=2) * np.linalg.norm(grad, axis=1)[:, None]
        assert np.all(np.abs(gx - want) <= 1e-13 * size + 4 * floor * np.sqrt(rays))
    return J


@pytest.mark.parametrize("failure", [abi.FAILURE_HARD, abi.FAILURE_SOFT])
@pytest.mark.parametrize("rings,spokes", SHAPES)
def test_tuple_shapes(engine, rings, spokes, failure):
    b, v = systems.singlet(4)
    x = v.extract(b)[:3].copy()
    x[1:, 0] = (0.19, 0.23)  # front radius near the pupil radius: rays fail
    s = ResidualSettings(rings=rings, spokes=spokes, failure=failure)
    base = b.take([0])
    if failure == abi.FAILURE_HARD:
        base.pupil_radius[:] = 4.9
    _check(engine, base, s, v, x)


@pytest.mark.parametrize("failure", [abi.FAILURE_HARD, abi.FAILURE_SOFT])
def test_glass_columns(engine, failure):
    b, v = systems.glass_singlet(4)
    s = ResidualSettings(rings=5, spokes=13, failure=failure)
    _check(engine, b.take([0]), s, v, v.extract(b)[:2])


@pytest.mark.parametrize("kind", [abi.REF_IMAGE_EXIT_PUPIL, abi.REF_IMAGE_INFINITE])
def test_image_references(engine, kind):
    b, v = systems.singlet(3)
    b.reference_sphere = kind
    b.reference_curvature = np.full((3, b.fields), 0.0 if kind == abi.REF_IMAGE_INFINITE else 0.009)
    s = ResidualSettings(rings=6, spokes=11, failure=abi.FAILURE_HARD)
    _check(engine, b.take([0]), s, v, v.extract(b)[:2])


def test_point_source(engine):
    b, v = systems.point_singlet()
    s = ResidualSettings(rings=7, spokes=9, failure=abi.FAILURE_HARD)
    _check(engine, b.take([0]), s, v, v.extract(b)[:2])


def test_unswept_column_is_zero(engine):
    b, v = systems.singlet(3)
    b.type = b.type.copy()
    b.type[2] = abi.SURFACE_PLANE
    b.curvature[:, 2] = 0.0
    s = ResidualSettings(rings=4, spokes=17, failure=abi.FAILURE_HARD)
    x = v.extract(b)[:2].copy()
    J = _check(engine, b.take([0]), s, v, x)
    assert np.all(J[:, 1] == 0.0) and np.all(np.any(J[:, [0, 2, 3]] != 0.0, axis=2))


def test_grazing_rays_leave_finite_gradients(engine):
    """The outer ring meets the first sphere within rounding of grazing (its radius is the ring's, to a
    few units in the last place): whatever rounding makes of the sweep's cosine there, the columns,
    the products with them and the fused normal equations stay finite wherever the trace accepts
    the rays with a cosine above zero."""
    import torch
    from mikroptim_amd.autograd import trace_residuals

    b, v = systems.singlet(2)
    base = b.take([0])
    base.index[:, 2] = base.index[:, 1]  # the second sphere refracts nothing
    base.field_angle[:] = base.field_target[:] = 0.0
    base.pupil_mode[:] = abi.PUPIL_FULL
    base.thickness[:, 2] = 400.0
    s = ResidualSettings(rings=2, spokes=6, failure=abi.FAILURE_HARD)
    u = np.polynomial.legendre.leggauss(2)[0][1]
    edge = 1.0 / (base.pupil_radius[0] * np.sqrt(0.5 * (u + 1.0)))
    x = np.tile(v.extract(base), (40, 1))
    # the last variable is the working distance; curvature 0 towards the edge, 1 to 40 units below
    x[:, 0] = edge * (1.0 - np.arange(1, 41) * 2.0 ** -52)
    v.upper[0] = 1.0
    J, _, a, g = engine.jacobian(base, s, v, x, method="adjoint", precision="fp64")
    assert np.isfinite(J).all() and np.isfinite(a).all() and np.isfinite(g).all()
    Jo = oracle().adjoint_jacobian(base, s, v, x)[0]
    grazing = np.abs(Jo[:, 0]).max(axis=1)
    assert np.sum(grazing > 1e5) > 10  # the rays are accepted and graze
    am, gm = engine.normal_equations(base, s, v, x, method="adjoint", precision="mixed")
    assert np.isfinite(am).all() and np.isfinite(gm).all()
    xt = torch.tensor(x, dtype=torch.float64, device="cuda", requires_grad=True)
    trace_residuals(xt, engine, base, s, v).sum().backward()
    assert torch.isfinite(xt.grad).all()
