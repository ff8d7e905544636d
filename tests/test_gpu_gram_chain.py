"""mko_gram_device and mko_gram_mfma_device bit for bit with normal_equations_host (one FMA chain
per element, ascending rows) where the kernel's shapes change: edges of 16-column tiles and of
64-column g units, the column counts with another stage (55 / 56, 64 / 65), the most variables of
the tile kernel (127) and the wide kernel above them, rows around the staged 64 / 128, and run
counts with one or several workgroups per run, also where they do not divide its tiles. Values of
mixed signs over 24 decades, so that another order of any sum shows."""

import ctypes as C

import numpy as np
import pytest

from mikroptim_amd.engine import library
from oracle_lib import oracle

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 1, 5), (3, 15, 3), (1, 16, 127), (5, 17, 128), (2, 47, 129),
          (1, 48, 1000), (600, 48, 131), (3, 55, 257), (2, 56, 64), (3, 64, 300), (2, 65, 63),
          (7, 96, 193), (520, 96, 65), (2, 127, 130), (600, 127, 33), (2, 128, 70), (1, 200, 40),
          (70, 100, 70), (54, 120, 65)]


@pytest.mark.parametrize("runs,P,rows", SHAPES)
def test_gram_equals_host_chain(runs, P, rows):
    import torch

    g = np.random.default_rng([runs, P, rows])
    J = g.standard_normal((runs, P, rows)) * 10.0 ** g.uniform(-12, 12, (runs, P, rows))
    r0 = g.standard_normal((runs, rows)) * 10.0 ** g.uniform(-12, 12, (runs, rows))
    Jd, rd = torch.tensor(J, device="cuda"), torch.tensor(r0, device="cuda")
    few = slice(0, 8) if runs > 8 else slice(None)
    ao, go = oracle().normal_equations(np.ascontiguousarray(J[few]), np.ascontiguousarray(r0[few]))
    names = ["mko_gram_device"] + (["mko_gram_mfma_device"] if P <= 127 else [])
    for name in names:
        a = torch.full((runs, P, P), float("nan"), dtype=torch.float64, device="cuda")
        gg = torch.full((runs, P), float("nan"), dtype=torch.float64, device="cuda")
        ptr = [C.cast(C.c_void_p(t.data_ptr()), C.POINTER(C.c_double)) for t in (rd, a, gg)]
        rc = getattr(library(), name)(C.c_void_p(Jd.data_ptr()), ptr[0], runs, P, rows, ptr[1],
                                      ptr[2], None)
        assert rc == 0, library().mko_last_error()
        torch.cuda.synchronize()
        an, gn = a.cpu().numpy(), gg.cpu().numpy()
        assert np.array_equal(an[few], ao) and np.array_equal(gn[few], go), name
        assert np.array_equal(an, np.swapaxes(an, 1, 2)) and np.isfinite(gn).all()
