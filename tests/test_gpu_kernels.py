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


def tanh_faces(n, lo, hi, a):
    t = np.linspace(-1.0, 1.0, n + 1)
    return lo + (hi - lo) * 0.5 * (1.0 + np.tanh(a * t) / np.tanh(a))


def setup_duct(s, I, shape, outlet, tol):
    """Channel between stretched walls with an inflow of 1 and an outlet of
    fixed pressure or convective outflow: a pressure system that is not pinned."""
    nx, ny, nz = shape
    f = [np.linspace(0.0, 2.0, nx + 1), tanh_faces(ny, -0.5, 0.5, 1.5), np.linspace(0.0, 1.0, nz + 1)]
    s.set_grid(*f)
    s.set_params(100.0, 0.002)
    s.set_bc(I.DIR_WEST, I.BC_VELOCITY_COMPONENT, I.VAL_CONST, 1.0, 0.0, 0.0)
    if outlet == "pressure":
        s.set_bc(I.DIR_EAST, I.BC_PRESSURE, I.VAL_CONST, 0.0)
    else:
        s.set_bc(I.DIR_EAST, I.BC_CONVECTIVE_OUTFLOW, 1.0)
    s.set_bc(I.DIR_NORTH | I.DIR_SOUTH, I.BC_STATIONARY_WALL)
    s.set_bc(I.DIR_DOWN | I.DIR_UP, I.BC_FREE_SLIP_WALL)
    s.set_obstacle(None)
    s.set_linear_solver(I.SOLVER_BiCGSTAB, I.PRECOND_AMG, tol)
    s.assemble()
    s.init_flow_const(1.0, 0.0, 0.0, 0.0)
    return f


SEPARABLE_CASES = [
    # remainders of the 16-wide tiles, one to several tiles per workgroup, the
    # smallest boxes, the longest axis whose tile fits the LDS and the next
    ("cavity", (4, 3, 2)), ("cavity", (8, 8, 8)), ("cavity", (17, 16, 15)), ("cavity", (33, 47, 20)),
    ("cavity", (9, 10, 512)), ("cavity", (528, 8, 8)), ("cavity", (64, 48, 33)), ("cavity", (130, 36, 65)), ("cavity", (20, 272, 18)), ("cavity", (10, 9, 400)),
    ("cavity", (416, 10, 9)), ("channel", (16, 12, 8)), ("channel", (34, 18, 22)), ("channel", (64, 70, 80)),
    ("pressure", (32, 20, 12)), ("pressure", (49, 33, 18)), ("outflow", (49, 33, 18)),
]


@pytest.mark.parametrize("kind,shape", SEPARABLE_CASES)
def test_direct_pressure_solve_matches_multigrid(new_gpu, I, cases, kind, shape):
    """Boxes without a body: the direct solve meets the tolerance of the FP64
    residual (formed by the operator kernel) in at most two rounds, and the
    fields agree with those of the multigrid solve, which an explicit
    multigrid setting selects. Both residuals are below tol, so the solutions
    differ by at most 2 tol times the span of the operator's eigenvalues, here
    bounded by sum_a 4 / h_a^2 over the lowest one, min_a (pi / (2 L_a))^2."""
    tol = 1e-12
    out, its = [], []
    for direct in (True, False):
        s = new_gpu()
        if not direct:
            s.set_mg_relaxation(1.3)
        if kind == "cavity":
            cases.setup_cavity(s, shape=shape, Re=100.0, dt=0.002, tol=tol)
            f = [np.linspace(0.0, 1.0, n + 1) for n in shape]
        elif kind == "channel":
            cases.setup_channel(s, *shape, tol=tol)
            f = cases.channel_faces(*shape)
        else:
            f = setup_duct(s, I, shape, kind, tol)
        s.iterate(3)
        its.append(int(s.last_iters()[3]))
        assert s.last_norms()[3] <= tol
        out.append({n: s.get(n)[2:-2, 2:-2, 2:-2] for n in ("U1", "U2", "U3", "P")})
    if max(shape) <= 400:
        assert its[0] <= 2, its
    span = sum(4 / np.diff(x).min() ** 2 for x in f) / min((np.pi / (2 * (x[-1] - x[0]))) ** 2 for x in f)
    scale = {"P": np.linalg.norm(out[1]["P"])}
    speed = np.sqrt(sum(np.linalg.norm(out[1][n]) ** 2 for n in ("U1", "U2", "U3")))
    for n, a in out[0].items():
        assert np.linalg.norm(a - out[1][n]) <= 2 * tol * span * scale.get(n, speed), n


@pytest.mark.parametrize("shape", [(18, 18, 18), (26, 22, 18), (30, 30, 26)])
def test_coarsest_level_inverse_at_block_remainders(new_gpu, cases, shape):
    """Two levels, the coarser one solved through its dense inverse, whose size
    (729, 1287, 2925 rows) leaves a remainder of the inversion's blocks of 64: the iteration counts of an exact coarse solve, at most 10
    (6 or 7 on the cavities of even sizes; with an inexact one the cycle
    contracts like its smoother alone and takes several times as many)."""
    s = new_gpu()
    s.set_mg_relaxation(1.3)
    cases.setup_cavity(s, shape=shape, Re=400.0, tol=1e-12)
    assert np.prod(s.mg_levels()[-1]) % 16 != 0 and len(s.mg_levels()) == 2
    s.iterate(2)
    assert s.last_norms()[3] <= 1e-12
    assert int(s.last_iters()[3]) <= 10


def setup_blocks(s, I, cases, shape, tol, precision):
    """Six blocks of the canopy on its grid, uniform inflow."""
    s.set_grid(*cases.urban_faces(*shape))
    s.set_params(2.0e4, 0.001)
    s.set_bc(I.DIR_WEST, I.BC_VELOCITY_COMPONENT, I.VAL_CONST, 1.0, 0.0, 0.0)
    s.set_bc(I.DIR_EAST, I.BC_PRESSURE, I.VAL_CONST, 0.0)
    s.set_bc(I.DIR_NORTH | I.DIR_SOUTH | I.DIR_UP, I.BC_FREE_SLIP_WALL)
    s.set_bc(I.DIR_DOWN, I.BC_STATIONARY_WALL)
    s.set_obstacle_stl_bytes(cases.blocks_stl(cases.urban_blocks(n=6)))
    s.set_linear_solver(I.SOLVER_BiCGSTAB, I.PRECOND_AMG, tol)
    s.set_precision(precision)
    s.assemble()
    s.init_flow_const(1.0, 0.0, 0.0, 0.0)


BODY_CASES = [
    # (set-up, grid, precision, most rounds of the direct solve, further
    # arguments): tile remainders, both outlets, the inverse of the ghost rows
    # in FP64 and (blocks 160 x 80 x 48, mixed mode) in FP32. None: too many
    # ghost cells for the grid, both solves are the iterative one.
    ("sphere", (66, 33, 35), 0, 2, dict()), ("sphere", (131, 48, 50), 2, 2, dict()),
    ("sphere", (70, 65, 34), 0, 2, dict(outflow="convective")),
    ("sphere", (48, 32, 32), 2, 2, dict(outflow="convective")),
    ("urban", (80, 40, 24), 0, 2, dict()), ("urban", (80, 40, 24), 2, 2, dict()),
    ("urban", (120, 60, 36), 2, None, dict()), ("blocks", (160, 80, 48), 2, 4, dict()),
]


@pytest.mark.parametrize("kind,shape,precision,rounds,kw", BODY_CASES)
def test_direct_pressure_solve_with_a_body_matches_multigrid(new_gpu, I, cases, kind, shape, precision, rounds, kw):
    """As without a body, at most four rounds where the ghost rows' inverse is
    kept in FP32 (each round gains four decades or more of the twelve). The
    ghost rows are normalised interpolations: their lowest eigenvalues are not
    below those of the fluid rows, so the same span bounds the difference."""
    tol = 1e-12
    out, its = [], []
    for direct in (True, False):
        s = new_gpu()
        if not direct:
            s.set_mg_relaxation(1.3)
        if kind == "blocks":
            setup_blocks(s, I, cases, shape, tol, precision)
        else:
            setup = cases.setup_sphere if kind == "sphere" else cases.setup_urban
            setup(s, *shape, tol=tol, precision=precision, **kw)
        s.iterate(3)
        its.append(int(s.last_iters()[3]))
        assert s.last_norms()[3] <= tol
        out.append({n: s.get(n)[2:-2, 2:-2, 2:-2] for n in ("U1", "U2", "U3", "P")})
    if rounds is None:
        assert its[0] == its[1]
    else:
        assert its[0] <= rounds and its[0] < its[1], its
    f = cases.sphere_faces(*shape, cases.SPHERE_DMIN * 128.0 / shape[1]) if kind == "sphere" \
        else cases.urban_faces(*shape)
    span = sum(4 / np.diff(x).min() ** 2 for x in f) / min((np.pi / (2 * (x[-1] - x[0]))) ** 2 for x in f)
    m = {n: np.isfinite(a) for n, a in out[1].items()}
    speed = np.sqrt(sum(np.linalg.norm(out[1][n][m[n]]) ** 2 for n in ("U1", "U2", "U3")))
    for n, a in out[0].items():
        assert np.array_equal(np.isfinite(a), m[n])
        ref = out[1][n][m[n]]
        assert np.linalg.norm(a[m[n]] - ref) <= 2 * tol * span * (speed if n != "P" else np.linalg.norm(ref)), n


OUTER_CASES = [
    # boundary types per face (west, east, south, north, down, up)
    ("velocity", "pressure", "slip", "slip", "wall", "wall"),
    ("func", "pressure", "pressure", "func", "pressure", "slip"),
    ("periodic", "periodic", "wall", "pressure", "pressure", "pressure"),
    ("slip", "velocity", "uperiodic", "uperiodic", "periodic", "periodic"),
]


@pytest.mark.parametrize("shape", [(6, 4, 8), (34, 18, 20)])
@pytest.mark.parametrize("faces", OUTER_CASES)
def test_outer_layers_match_the_oracle(new_gpu, new_oracle, I, faces, shape):
    """Both outer layers, edges and corners of the four fields from random
    interior ones, on stretched axes where they may be: an outer value is a
    short sum of products, so the two agree to a few roundings (1e-12 of the
    largest value, which extrapolation at edges and corners can raise)."""
    periodic = [faces[2 * a] == "periodic" or faces[2 * a] == "uperiodic" for a in range(3)]
    out = []
    for new in (new_gpu, new_oracle):
        s = new()
        f = [np.linspace(0.0, 1.0, n + 1) if p else tanh_faces(n, 0.0, 1.0 + a, 1.2)
             for a, (n, p) in enumerate(zip(shape, periodic))]
        s.set_grid(*f)
        s.set_params(100.0, 0.002)
        for d, t in zip((I.DIR_WEST, I.DIR_EAST, I.DIR_SOUTH, I.DIR_NORTH, I.DIR_DOWN, I.DIR_UP), faces):
            if t == "velocity":
                s.set_bc(d, I.BC_VELOCITY_COMPONENT, I.VAL_CONST, 1.0, 0.25, -0.5)
            elif t == "func":
                s.set_bc(d, I.BC_VELOCITY_COMPONENT, I.VAL_FUNC, *[
                    (lambda c: lambda t, x, y, z: c + x + 2 * y * z)(c) for c in (1.0, 2.0, 3.0)])
            elif t == "pressure":
                s.set_bc(d, I.BC_PRESSURE, I.VAL_CONST, 0.75)
            elif t == "uperiodic":
                s.set_bc(d, I.BC_VELOCITY_PERIODIC, I.VAL_CONST, 0.5)
            else:
                s.set_bc(d, {"slip": I.BC_FREE_SLIP_WALL, "wall": I.BC_STATIONARY_WALL,
                             "periodic": I.BC_ALL_PERIODIC}[t])
        s.set_obstacle(None)
        s.set_linear_solver(I.SOLVER_BiCGSTAB, I.PRECOND_AMG, 1e-10)
        s.assemble()
        s.init_flow_const(0, 0, 0, 0)
        rng = np.random.default_rng(5)
        for n in ("U1", "U2", "U3", "P"):
            s.set(n, rng.standard_normal(s.shape))
        s.iterate(0)
        out.append({n: s.get(n) for n in ("U1", "U2", "U3", "P")})
    for n, a in out[0].items():
        b = out[1][n]
        assert np.array_equal(np.isfinite(a), np.isfinite(b)), n
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max(), n


@pytest.mark.parametrize("precision", [0, 2], ids=["fp64", "mixed"])
@pytest.mark.parametrize("kind,shape", [("channel", (34, 18, 22)), ("channel", (64, 48, 32)),
                                        ("pressure", (49, 33, 18)), ("outflow", (49, 33, 18))])
def test_momentum_of_boxes_matches_bicgstab(new_gpu, I, cases, kind, shape, precision):
    """Periodic axes, walls, free slip and outlets (the axis of a pressure
    outlet extrapolates the velocity and may leave the direct solve to the
    sweeps) against BiCGSTAB at tol 1e-12, as for the sweeps: 1e-10 with room
    for the projection."""
    out = []
    for mode in (0, 1):
        s = new_gpu()
        s.set_momentum_solver(mode)
        s.set_precision(precision)
        if kind == "channel":
            cases.setup_channel(s, *shape, tol=1e-12, precision=precision)
        else:
            setup_duct(s, I, shape, kind, 1e-12)
        s.iterate(2)
        assert (s.last_norms()[:3] <= 1e-12).all()
        if mode == 0 and kind == "channel":
            assert list(s.last_iters()[:3]) == [1, 1, 1]
        out.append([s.get(n)[2:-2, 2:-2, 2:-2] for n in ("U1_STAR", "U2_STAR", "U3_STAR", "U1", "U2", "U3")])
    scale = max(np.abs(a).max() for a in out[1])
    for a, b in zip(*out):
        assert np.abs(a - b).max() <= 1e-10 * scale


@pytest.mark.parametrize("shape", [(124, 92, 86), (128, 92, 92), (150, 110, 97)])
def test_large_fields_reach_the_host_unchanged(new_gpu, cases, shape):
    """Cell and face fields of just below, at and above the size that crosses
    through the ring of pinned chunks (8 MiB; the ring's 8 chunks of 1 MiB used
    once, and again with a part of a chunk left): as set, bit for bit, twice."""
    s = new_gpu()
    cases.setup_cavity(s, shape=shape, tol=1e-8)
    rng = np.random.default_rng(11)
    a = {n: rng.standard_normal(s.shape) for n in ("U1", "P")}
    for n, v in a.items():
        s.set(n, v)
    for _ in range(2):
        for n, v in a.items():
            np.testing.assert_array_equal(s.get(n), v)
    s.iterate(0)
    u, f = s.get("U1"), s.get("FACE_U1")
    np.testing.assert_allclose(f[:, 2:-2, 2:-2], 0.5 * (u[1:-2, 2:-2, 2:-2] + u[2:-1, 2:-2, 2:-2]),
                               rtol=1e-13, atol=1e-13)
