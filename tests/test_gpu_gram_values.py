"""mko_gram_device and mko_gram_mfma_device bit for bit with normal_equations_host where a sum of
products leaves the normal numbers: products and sums that are subnormal or underflow to zero of
either sign, that overflow, infinities and NaN (of any payload) in single columns. On the tile kernel
(up to 127 variables, 1 ... 4 rows in its last matrix instruction) and the wide one."""

import ctypes as C

import numpy as np
import pytest

from mikroptim_amd.engine import library
from oracle_lib import oracle

pytestmark = pytest.mark.gpu


def _gram(name, J, r0):
    import torch

    runs, P, rows = J.shape
    Jd, rd = torch.tensor(J, device="cuda"), torch.tensor(r0, device="cuda")
    a = torch.full((runs, P, P), 3.0, dtype=torch.float64, device="cuda")
    g = torch.full((runs, P), 3.0, dtype=torch.float64, device="cuda")
    ptr = [C.cast(C.c_void_p(t.data_ptr()), C.POINTER(C.c_double)) for t in (rd, a, g)]
    rc = getattr(library(), name)(C.c_void_p(Jd.data_ptr()), ptr[0], runs, P, rows, ptr[1], ptr[2],
                                  None)
    assert rc == 0, library().mko_last_error()
    torch.cuda.synchronize()
    return a.cpu().numpy(), g.cpu().numpy()


def _check(J, r0):
    ao, go = oracle().normal_equations(np.ascontiguousarray(J), np.ascontiguousarray(r0))
    for name in ["mko_gram_device"] + (["mko_gram_mfma_device"] if J.shape[1] <= 127 else []):
        a, g = _gram(name, J, r0)
        for x, xo in ((a, ao), (g, go)):
            assert np.array_equal(x, xo, equal_nan=True), name
            assert np.array_equal(np.signbit(x) & ~np.isnan(x), np.signbit(xo) & ~np.isnan(xo)), name
    return ao, go


SHAPES = [(2, 8, 1), (2, 9, 2), (2, 20, 3), (2, 20, 4), (1, 60, 5), (1, 48, 130), (2, 100, 67), (1, 130, 33)]


@pytest.mark.parametrize("runs,P,rows", SHAPES)
def test_subnormal_products(runs, P, rows):
    g = np.random.default_rng([1, runs, P, rows])
    J = g.standard_normal((runs, P, rows)) * 10.0 ** g.uniform(-163, -155, (runs, P, rows))
    r0 = g.standard_normal((runs, rows)) * 10.0 ** g.uniform(-163, -155, (runs, rows))
    J[:, -3:] *= 1e-8  # columns whose every product is zero
    a, _ = _check(J, r0)
    assert np.any((a != 0.0) & (np.abs(a) < 2.0 ** -1022))


@pytest.mark.parametrize("runs,P,rows", SHAPES)
def test_subnormal_values(runs, P, rows):
    g = np.random.default_rng([2, runs, P, rows])
    J = g.standard_normal((runs, P, rows)) * 10.0 ** g.uniform(-320, 8, (runs, P, rows))
    r0 = g.standard_normal((runs, rows)) * 10.0 ** g.uniform(-320, 8, (runs, rows))
    _check(J, r0)


@pytest.mark.parametrize("runs,P,rows", SHAPES)
def test_overflow_infinities_and_nan(runs, P, rows):
    g = np.random.default_rng([3, runs, P, rows])
    J = g.standard_normal((runs, P, rows)) * 10.0 ** g.uniform(-20, 152, (runs, P, rows))
    r0 = g.standard_normal((runs, rows)) * 10.0 ** g.uniform(-20, 152, (runs, rows))
    # entries below 6e152, sums of 130 products below 5e307: only what follows leaves the range
    J[0, 0] *= 1e100  # overflows
    J[0, 1, rows // 2] = np.inf
    J[0, 2, rows - 1] = -np.inf
    J[0, 3, 0] = np.nan
    J[-1, 4] = 0.0
    a, _ = _check(J, r0)
    assert np.isinf(a[0, 0, 0]) and np.isnan(a[0, 3]).all()
    assert np.isfinite(np.delete(np.delete(a[0], [0, 1, 2, 3], 0), [0, 1, 2, 3], 1)).all()
