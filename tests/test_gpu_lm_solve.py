"""The step solve of the device LM control where its shapes change: one and two rows per lane (63,
64 and 65 variables: the right-hand side is a row of its own), remainders of its batches of eight,
variables that their bounds fix at the start or during the solve, and matrices whose factorisation
fails. The host control performs the same operations in the same order: equal bits."""

import numpy as np
import pytest

from mikroptim_amd import abi, systems
from mikroptim_amd.batch import ResidualSettings
from test_gpu_parity import _same_lm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 2, 7, 8, 9, 16, 31, 62, 63, 64, 65, 72, 96, 127])
@pytest.mark.parametrize("bounds", ["free", "tight", "singular"])
def test_device_solve_equals_host(engine, P, bounds):
    b, v = systems.uneven_topology(1, variants=4, surfaces=40, variables=P)
    assert len(v.lower) == P
    s = ResidualSettings(rings=3, spokes=8, failure=abi.FAILURE_SOFT)
    x0 = v.extract(b)[:3]
    damping = 1e-3
    if bounds == "tight":  # every third variable fixed, the others leave their range soon
        width = np.abs(x0).max(axis=0) * 10.0 ** -(2 + np.arange(P) % 4)
        v.lower[:], v.upper[:] = x0.min(axis=0) - width, x0.max(axis=0) + width
        v.lower[::3] = v.upper[::3] = x0[0, ::3]
        x0 = v.clamp(x0)
    elif bounds == "singular":
        damping = 1e-300
    kw = dict(max_iterations=5, threads=4, jacobian_method=abi.JACOBIAN_ADJOINT,
              initial_damping=damping)
    rd = engine.optimize(b.take([0]), s, v, x0, abi.lm_options(**kw))
    rh = engine.optimize(b.take([0]), s, v, x0, abi.lm_options(host_control=True, **kw))
    _same_lm(rd, rh)
