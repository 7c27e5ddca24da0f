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


@pytest.mark.parametrize("shape", [(33, 31, 35), (64, 5, 7), (6, 40, 66), (128, 32, 33)])
def test_fields_cross_the_host_boundary_unchanged(new_gpu, I, cases, shape):
    """set / get of a cell field move every padded cell to its place (tile
    remainders on both transposed axes, small and large fields), and a face
    field is the interpolation of the cells it lies between."""
    s = new_gpu()
    cases.setup_cavity(s, shape=shape, tol=1e-10)
    rng = np.random.default_rng(3)
    a = {n: rng.standard_normal(s.shape) for n in ("U1", "U2", "U3", "P")}
    for n, v in a.items():
        s.set(n, v)
    for n, v in a.items():
        np.testing.assert_array_equal(s.get(n), v)
    s.iterate(0)  # outer layers and face velocities from the cell fields
    for ax, n in enumerate(("U1", "U2", "U3")):
        u = s.get(n)
        sl = [slice(2, -2)] * 3
        lo, hi = list(sl), list(sl)
        lo[ax], hi[ax] = slice(1, -2), slice(2, -1)
        f = s.get("FACE_" + n)
        inner = list(sl)
        inner[ax] = slice(None)
        np.testing.assert_allclose(f[tuple(inner)], 0.5 * (u[tuple(lo)] + u[tuple(hi)]), rtol=1e-13, atol=1e-13)


MOMENTUM_CASES = [
    # (set-up, grid, further arguments): remainders of the launch shapes, with
    # and without a body, sweep rates from 0.002 to just below the largest one
    ("cavity", (17, 13, 11), dict(Re=100.0)),
    ("cavity", (130, 9, 10), dict(Re=100.0, dt=0.001)),
    ("cavity", (40, 40, 40), dict(Re=20.0, dt=0.008)),
    ("sphere", (66, 33, 35), dict()),
    ("sphere", (131, 24, 25), dict()),
]


@pytest.mark.parametrize("precision", [0, 2], ids=["fp64", "mixed"])
@pytest.mark.parametrize("kind,grid,kw", MOMENTUM_CASES)
def test_batched_momentum_sweeps_match_bicgstab(new_gpu, cases, kind, grid, kw, precision):
    """Two steps with the momentum sweeps of the three components in one
    launch against BiCGSTAB at tol 1e-12: both solve the same systems, so the
    fields agree to the tolerance times the conditioning of a strongly
    diagonally dominant system (a few), 1e-10 with room for the projection."""
    out = []
    for mode in (0, 1):
        s = new_gpu()
        s.set_momentum_solver(mode)
        if kind == "cavity":
            cases.setup_cavity(s, shape=grid, tol=1e-12, precision=precision, **kw)
        else:
            cases.setup_sphere(s, *grid, tol=1e-12, precision=precision, **kw)
        s.iterate(2)
        assert (s.last_norms()[:3] <= 1e-12).all()
        out.append([s.get(n) for n in ("U1_STAR", "U2_STAR", "U3_STAR", "U1", "U2", "U3")])
    scale = max(np.nanmax(np.abs(a[2:-2, 2:-2, 2:-2])) for a in out[1])
    for a, b in zip(*out):
        a, b = a[2:-2, 2:-2, 2:-2], b[2:-2, 2:-2, 2:-2]
        m = np.isfinite(b)
        assert np.array_equal(np.isfinite(a), m)
        assert np.abs(a[m] - b[m]).max() <= 1e-10 * scale
