"""The iterative solves by themselves: multigrid settings and
IBMSolver_set_momentum_solver select them on systems that the default route
solves directly or by sweeps. Each test looks at the iteration counts, so that
a change of the routes cannot empty it."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

INNER = (slice(2, -2),) * 3
BOTH = pytest.mark.parametrize("precision", [0, 2], ids=["fp64", "mixed"])


def velocity(s):
    return np.stack([s.get(n)[INNER] for n in ("U1", "U2", "U3")])


def rel(a, b):
    m = np.isfinite(a) & np.isfinite(b)
    return float(np.linalg.norm(a[m] - b[m]) / np.linalg.norm(b[m]))


@pytest.mark.parametrize("shape", [(45, 16, 16), (46, 15, 13), (17, 12, 10)])
def test_cycles_on_odd_rows_converge_as_on_even_rows(new_gpu, cases, shape):
    """The FP64 cycle starts from zero on every cell of a row, the last one of
    an odd row among them: the iterations of an odd row length are those of the
    next one within two (a row's stale last cell: twice as many and more)."""
    its = []
    for nx in (shape[0], shape[0] + 1):
        s = new_gpu()
        s.set_mg_relaxation(1.3)
        cases.setup_cavity(s, shape=(nx, *shape[1:]), Re=400.0, tol=1e-12)
        s.iterate(4)
        assert s.last_norms()[3] <= 1e-12
        its.append(int(s.last_iters()[3]))
    assert abs(its[0] - its[1]) <= 2 and min(its) > 2, its


@pytest.mark.parametrize("kind,shape", [("sphere", (67, 33, 35)), ("sphere", (51, 32, 30)), ("cavity", (45, 37, 29)),
                                        ("cavity", (31, 17, 64))])
def test_odd_rows_in_fp64_directly_and_by_cycles(new_gpu, cases, kind, shape):
    """Rows of odd length in FP64, the direct solve against the cycles: both
    residuals are below tol, so the fields differ by at most 2 tol times the
    span of the operator's eigenvalues, bounded by sum_a 4 / h_a^2 over the
    lowest one, min_a (pi / (2 L_a))^2."""
    tol = 1e-12
    out, its = [], []
    for direct in (True, False):
        s = new_gpu()
        if not direct:
            s.set_mg_relaxation(1.3)
        if kind == "sphere":
            cases.setup_sphere(s, *shape, tol=tol)
        else:
            cases.setup_cavity(s, shape=shape, tol=tol)
        s.iterate(3)
        assert s.last_norms()[3] <= tol
        its.append(int(s.last_iters()[3]))
        out.append((velocity(s), s.get("P")[INNER]))
    assert its[0] <= 2 < its[1], its
    f = [s.xf, s.yf, s.zf]
    span = sum(4 / np.diff(x).min() ** 2 for x in f) / min((np.pi / (2 * (x[-1] - x[0]))) ** 2 for x in f)
    for a, b in zip(*out):
        assert rel(a, b) <= 2 * tol * span


@BOTH
def test_lanes_and_graphs_match_serial_eager_solves(new_gpu, cases, precision):
    """BiCGSTAB for the momentum, three lanes at once, with replayed multigrid
    graphs, against the three one after the other and cycles launched kernel by
    kernel (the per-kernel timers select that): the same kernels and
    decisions, hence the same bits."""
    runs = []
    for timed in (False, True):
        s = new_gpu()
        s.set_mg_relaxation(1.3)
        s.set_momentum_solver(1)
        cases.setup_sphere(s, 96, 48, 48, tol=1e-10, precision=precision)
        if timed:
            s.enable_timing(1)
        s.iterate(3)
        names = {k["name"] for k in s.kernel_stats()}
        assert ("rbgs_L0" in names and "spmv_u64" in names) == timed, names
        runs.append((s.last_iters().tolist(), s.last_norms().tolist(), velocity(s), s.get("P")))
    assert runs[0][0] == runs[1][0] and min(runs[0][0]) > 2
    assert runs[0][1] == runs[1][1]
    for a, b in zip(runs[0][2:], runs[1][2:]):
        assert np.array_equal(a, b, equal_nan=True)


@BOTH
def test_iterative_solves_are_bitwise_reproducible(new_gpu, cases, precision):
    """Two solvers with the iterative solves on a grid where waves overlap."""
    runs = []
    for _ in range(2):
        s = new_gpu()
        s.set_mg_relaxation(1.3)
        s.set_momentum_solver(1)
        cases.setup_sphere(s, 128, 64, 64, tol=1e-10, precision=precision)
        s.iterate(2)
        runs.append((s.last_iters().tolist(), velocity(s), s.get("P")))
    assert runs[0][0] == runs[1][0] and min(runs[0][0]) > 2
    for a, b in zip(runs[0][1:], runs[1][1:]):
        assert np.array_equal(a, b, equal_nan=True)


def test_stalling_fp32_cycles_switch_to_fp64(new_gpu, cases, I):
    """The pinned pressure system of the channel 192 x 96 x 128 at tol 1e-11
    makes BiCGSTAB with FP32 cycles stall: the mixed mode starts with them,
    switches to the FP64 cycle (in the first step that stalls twice: rounding
    in the momentum decides between the first and the second) and then needs
    the iterations of the FP64 mode (within two)."""
    its, out = [], []
    for prec in (I.PREC_FP64, I.PREC_MIXED_KRYLOV):
        s = new_gpu()
        s.set_mg_relaxation(1.3)
        cases.setup_channel(s, tol=1e-11, precision=prec, turb=(I.TURBMODEL_SMAGORINSKY_VD, 0.1))
        assert s.pressure_mg_bits() == (64 if prec == I.PREC_FP64 else 32)
        s.iterate(3)
        assert s.pressure_mg_bits() == 64
        s.iterate(1)
        its.append(int(s.last_iters()[3]))
        out.append((velocity(s), s.get("P")[INNER]))
        s.close()
    assert 2 < its[1] <= its[0] + 2, its
    assert rel(out[1][0], out[0][0]) <= 1e-5 and rel(out[1][1], out[0][1]) <= 1e-5


def test_fp32_cycles_hold_on_the_sphere(new_gpu, cases, I):
    """The sphere 256 x 128 x 128 with its convective outflow, 100 steps at
    tol 1e-9: the FP32 cycles do not stall twice in a solve, and velocity and
    pressure stay within 1e-5 of the FP64 mode."""
    out = []
    for prec in (I.PREC_FP64, I.PREC_MIXED_KRYLOV):
        s = new_gpu()
        s.set_mg_relaxation(1.3)
        cases.setup_sphere(s, 256, 128, 128, tol=1e-9, precision=prec, outflow="convective")
        s.iterate(100)
        assert int(s.last_iters()[3]) > 2
        out.append((velocity(s), s.get("P")[INNER], s.max_div(), s.pressure_mg_bits()))
        s.close()
    assert out[0][3] == 64 and out[1][3] == 32
    assert rel(out[1][0], out[0][0]) <= 1e-5 and rel(out[1][1], out[0][1]) <= 1e-5
    assert max(out[0][2], out[1][2]) <= 1e-8
