"""Kernels of the pressure and momentum solves at the sizes where they can go
wrong: remainders, the ends of their ranges, forms that take another route."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    m = np.isfinite(a) & np.isfinite(b)
    return float(np.linalg.norm(a[m] - b[m]) / max(np.linalg.norm(b[m]), 1e-300))


@pytest.mark.parametrize("shape", [(45, 16, 16), (46, 15, 13), (17, 12, 10)])
def test_pressure_cycle_of_odd_rows_converges_as_of_even_rows(new_gpu, cases, shape):
    """The FP64 cycle starts from zero on every cell of a row, the last one of
    an odd row among them: the pressure solve takes no more iterations on an
    odd row than on the next even one (within two)."""
    its = []
    for nx in (shape[0], shape[0] + 1):
        s = new_gpu()
        cases.setup_cavity(s, shape=(nx, *shape[1:]), Re=400.0, tol=1e-12)
        s.iterate(4)
        its.append(int(s.last_iters()[3]))
    assert abs(its[0] - its[1]) <= 2, its
