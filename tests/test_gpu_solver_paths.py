"""Pressure and direct solves: the routes a solve takes when its first step is
not enough, and the buffers it shares with the caller."""
import contextlib
import ctypes as C

import numpy as np
import pytest

from oracle import orc
from tests.case_util import gpu_from_case, make_case

pytestmark = pytest.mark.gpu

I = (slice(1, -1),) * 3
GRID = (70, 12, 21)


@pytest.fixture(scope="module")
def tbl():
    from turbulentbl_amd import tbl as t
    t.load()
    return t


def _rhs(g, seed=22):
    b = g.zeros()
    b[I] = np.random.default_rng(seed).standard_normal([n - 2 for n in (g.nX, g.nY, g.nZ)])
    return b


def _solve(tbl, sv, g, b, **kw):
    sv.set_field(tbl.F_PCORR, g.zeros())
    sv.set_field(tbl.F_PRHS, b)
    out = sv.ppe_solve(**kw)
    return out, sv.get_field(tbl.F_PCORR)


def test_true_residual_solve_leaves_the_work_field(tbl):
    g, s = make_case(GRID, seed=4)
    b = _rhs(g)
    w = np.asfortranarray(np.random.default_rng(1).standard_normal(b.shape))
    with gpu_from_case(g, s, tol_mode=tbl.TBL_TOL_TRUE, errtol=1e-10, inner_tol=1e-12, precond=tbl.TBL_PC_FAST) as sv:
        sv.set_field(tbl.F_WORK, w)
        _solve(tbl, sv, g, b, errtol=1e-10)
        assert np.array_equal(sv.get_field(tbl.F_WORK)[I], w[I])


class _hip:
    """the runtime that the library is linked to"""

    def __init__(self):
        self.lib = C.CDLL("libamdhip64.so.7")
        self.lib.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.lib.hipFree.argtypes = [C.c_void_p]

    def free(self):
        a, b = C.c_size_t(), C.c_size_t()
        assert self.lib.hipDeviceSynchronize() == 0 and self.lib.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    @contextlib.contextmanager
    def left(self, nbytes):
        """no more than nbytes of the device's memory are to be had: they are taken,
        then all the rest down to 16 MB (what the runtime keeps of freed memory
        too), then given back"""
        def take(size):
            p = C.c_void_p()
            return p if self.lib.hipMalloc(C.byref(p), int(size)) == 0 else None

        spare, held, size = take(nbytes), [], self.free()
        assert spare
        while size >= 16e6:
            p = take(size)
            if p:
                held.append(p)
            else:
                size /= 2
        self.lib.hipFree(spare)
        self.lib.hipGetLastError()               # of the allocations that failed
        try:
            yield
        finally:
            for p in held:
                self.lib.hipFree(p)


def _solver(tbl, grid, **kw):
    nX = grid[0]
    return tbl.Solver(*grid, i_rec=int(0.8 * (nX - 1)), planes=(2, 3, 4, 5, 6), **kw)


# fields beyond the size up to which three components go through one solve
# (6 N values above 256 MB), and below it
@pytest.mark.parametrize("precision,grid", [("fp64", (900, 96, 64)), ("mixed", (1100, 100, 98)), ("fp64", GRID), ("mixed", GRID)])
def test_direct_diffusion_solve(tbl, precision, grid):
    """(I - hA) u = Q + boundary terms, three different components; memory beyond
    the solver's own is taken for three components at once only"""
    rng = np.random.default_rng(2)
    h = 1e-4 / 150.92
    N, es = int(np.prod(grid)), 4 if precision == "mixed" else 8
    one = 6 * N * es > 256e6
    with _solver(tbl, grid, precision=precision, helm_mode=tbl.TBL_HELM_DIRECT, precond=tbl.TBL_PC_FAST, kmax=1) as sv:
        U, Q = sv.zeros(3), sv.zeros(3)
        for a in (U, Q):
            a[...] = rng.standard_normal(a.shape, dtype=np.float32)
        sv.upload(U)
        sv.set_field(tbl.F_Q, Q)
        held = sv.device_bytes
        sv.diffusion_solve()
        assert sv.device_bytes - held == (0 if one else (3 + 4) * N * es)
        u, m = sv.get_field(tbl.F_UT), sv.mesh()
    dx, dy = m["x1"][1] - m["x1"][0], m["x2"][1] - m["x2"][0]
    At, Ab, Ap = (m[q][1:-1] for q in ("At", "Ab", "Ap"))
    c = u[I]
    rows = np.arange(1, grid[1] - 1)
    up, dn = np.where(rows == rows[-1], 1, rows + 1), np.where(rows == 1, rows[-1], rows - 1)
    x = u[1:-1, :, 1:-1]
    A = ((u[2:, 1:-1, 1:-1] + u[:-2, 1:-1, 1:-1]) / dx ** 2 + (x[:, up] + x[:, dn]) / dy ** 2
         + At[:, None] * u[1:-1, 1:-1, 2:] + Ab[:, None] * u[1:-1, 1:-1, :-2] + Ap[:, None] * c)
    r = Q[I] - (c - h * A)
    # a solution rounded to the storage type: its rounding times the row sum of
    # I - hA, at most 1 + 2 h max |Ap|; the FP64 solve refines once
    eps = 1.2e-7 if precision == "mixed" else 2.3e-16
    assert np.abs(r).max() <= 64 * eps * np.abs(u).max() * (1 + 2 * h * np.abs(Ap).max())


def test_device_bytes_are_those_held(tbl):
    """what a context takes from the device, first solves included"""
    free = _hip().free
    for grid, kw in (((900, 96, 64), dict(helm_mode=tbl.TBL_HELM_DIRECT)), ((256, 96, 64), dict(helm_mode=tbl.TBL_HELM_DIRECT)),
                     ((1024, 8, 130), dict(helm_mode=tbl.TBL_HELM_LEX_SLAB, precond=tbl.TBL_PC_SSOR_BLOCK, slabs=64))):
        before = free()
        with _solver(tbl, grid, kmax=4, **kw) as sv:
            sv.upload(sv.zeros(3))
            sv.diffusion_solve(1e-6, 1)
            sv.ppe_solve(1e-5, 4, 1)
            taken = before - free()
            # each of some 45 allocations takes whole 2 MB pages
            assert 0.98 * sv.device_bytes <= taken <= sv.device_bytes + 100e6


# long lines whose diagonal is close to twice the streamwise coupling.  The
# residual that the FP64 solve leaves with every quotient of the cyclic reduction
# rounded once (divided), measured, and three times that: products with a rounded
# reciprocal leave 5 to 22 times as much on these three
@pytest.mark.parametrize("nX,Lx,divided", [(100, 6.0, 7.2e-13), (2000, 3.0, 2.6e-9), (2050, 1.0, 1.4e-8)])
def test_line_solve_rounding(tbl, nX, Lx, divided):
    grid = (nX, 10, 20)
    x = [np.sin(np.pi * np.arange(n) / (n - 1)) for n in grid]
    with _solver(tbl, grid, precond=tbl.TBL_PC_FAST, kmax=1, Lx=Lx, Ly=4.0, Lz=3.4) as sv:
        b = sv.zeros()
        b[...] = x[0][:, None, None] * (1 + 0.3 * np.cos(2 * np.pi * np.arange(10) / 8))[None, :, None] * x[2][None, None, :]
        b[I] *= 1 + 0.1 * np.random.default_rng(nX).standard_normal((nX - 2, 8, 18))
        for q in range(3):
            f = np.moveaxis(b, q, 0)
            f[0] = f[-1] = 0.0
        r = b - sv.apply_operator(0, sv.apply_operator(1, b))
    assert np.linalg.norm(r[I]) <= 3 * divided * np.linalg.norm(b)


def test_solve_without_memory_for_unit_steps(tbl):
    """a solve by the reference's rule did without the second pressure
    correction's 8 N bytes before unit steps, and does when they are not there"""
    grid = (600, 250, 200)
    N = int(np.prod(grid))
    with _solver(tbl, grid, precond=tbl.TBL_PC_FAST, kmax=1, errtol=1e-6) as sv:
        b = sv.zeros()
        b[I] = np.random.default_rng(3).standard_normal([n - 2 for n in grid], dtype=np.float32)
        sv.set_field(tbl.F_PRHS, b)
        held = sv.device_bytes
        with _hip().left(5 * N):
            out = sv.ppe_solve(1e-6, 1, 20)
        assert sv.device_bytes == held
        x = sv.get_field(tbl.F_PCORR)
        r = b - sv.apply_operator(0, x)
        for q in range(3):
            f = np.moveaxis(r, q, 0)
            f[0] = f[-1] = 0.0
        assert np.linalg.norm(sv.apply_operator(1, r)) <= 1e-6 * np.linalg.norm(sv.apply_operator(1, b))
        assert abs(out["true_res"] - np.linalg.norm(r)) <= 1e-6 * np.linalg.norm(r) + 1e-13 * np.linalg.norm(b)
        sv.set_field(tbl.F_PCORR, np.zeros_like(x, order="F"))
        sv.ppe_solve(1e-6, 1, 20)
        assert sv.device_bytes == held + 8 * N


@pytest.mark.parametrize("rule", ["ref", "true"])
def test_timers_see_an_accepted_unit_step(tbl, rule):
    """two residual passes and two applications by the reference's rule (of M^-1 b
    and of what the step left), one application where the true residual is asked for"""
    g, s = make_case(GRID, seed=4)
    with gpu_from_case(g, s, precond=tbl.TBL_PC_FAST, tol_mode=int(rule == "true"), inner_tol=1e-6) as sv:
        sv.timer_enable(["resid", "precond"])
        out, _ = _solve(tbl, sv, g, _rhs(g), errtol=1e-5)
        n = {q: v["count"] for q, v in sv.timer_read().items()}
    assert out["iters"] == 1
    assert n == dict(resid=2, precond=2 if rule == "ref" else 1)


# the usual tolerance, and one that no solve's accuracy meets
@pytest.mark.parametrize("errtol", [1e-5, 1e-16])
def test_no_step_is_tried_that_cannot_be_accepted(tbl, errtol):
    """reference's rule: one application at each cycle's start and one for each
    step, an accepted unit step among them"""
    g, s = make_case((64, 32, 48), seed=4)
    with gpu_from_case(g, s, precond=tbl.TBL_PC_FAST) as sv:
        sv.timer_enable(["precond"])
        out, _ = _solve(tbl, sv, g, _rhs(g), errtol=errtol, kmax=5, mmax=3)
        n = sv.timer_read()["precond"]["count"]
    assert n == out["cycles"] + out["iters"]


# FP32 fields on both sides of the sizes from which a transfer goes through the
# pinned ring (393216 values from the device, 1310720 to it)
@pytest.mark.parametrize("grid", [(64, 64, 94), (64, 64, 96), (128, 128, 78), (128, 128, 80)])
def test_converted_transfers(tbl, grid):
    with _solver(tbl, grid, precision="mixed", kmax=1) as sv:
        x = np.asfortranarray(np.random.default_rng(7).standard_normal(grid))
        sv.set_field(tbl.F_PRESS, x)
        assert np.array_equal(sv.get_field(tbl.F_PRESS), x.astype(np.float32))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_transfers_of_page_locked_arrays(tbl, precision):
    """a size that goes through the ring from pageable memory"""
    grid = (128, 128, 66)
    n, hip = 3 * int(np.prod(grid)), _hip()
    p = C.c_void_p()
    hip.lib.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    hip.lib.hipHostFree.argtypes = [C.c_void_p]
    with _solver(tbl, grid, precision=precision, kmax=1) as sv:
        assert hip.lib.hipHostMalloc(C.byref(p), 8 * n, 0) == 0
        a = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (n,))
        x = np.random.default_rng(8).standard_normal(n)
        a[:] = x
        sv._chk(sv.lib.tbl_field_set(sv.h, tbl.F_UT, p))
        a[:] = 0.0
        sv._chk(sv.lib.tbl_field_get(sv.h, tbl.F_UT, p))
        assert np.array_equal(a, x if precision == "fp64" else x.astype(np.float32))
        hip.lib.hipHostFree(p)
        assert np.array_equal(sv.get_field(tbl.F_UT).ravel(order="F"), x if precision == "fp64" else x.astype(np.float32))


def test_window_without_memory_for_the_adjoint_fields(tbl):
    """the forward sweep needs the snapshots only: J is there when the call fails"""
    grid = (900, 96, 64)
    N = int(np.prod(grid))
    rng = np.random.default_rng(9)
    with _solver(tbl, grid, kmax=1) as sv:
        U = sv.zeros(3)
        U[..., 0] = 19.8 * np.tanh(4.0 * sv.mesh()["x3"])
        U[I] += 0.02 * rng.standard_normal(U[I].shape, dtype=np.float32)

        def window(forward_only):
            sv.upload(U, sv.zeros(), sv.zeros())
            sv.set_state()
            o, J = tbl.AdjointOpts(2, 1, 500, 800, forward_only, 0), C.c_double(-1.0)
            grad = np.zeros(grid[:2], order="F")
            rc = sv.lib.tbl_adjoint_window(sv.h, C.byref(o), None, C.byref(J), None if forward_only else grad.ctypes.data,
                                           None, None)
            return rc, J.value

        rc, J = window(1)
        assert rc == 0 and J > 0.0
        # three snapshots of 40 bytes a cell; the adjoint fields take 72
        with _hip().left((3 * 40 + 36) * N):
            rc, Jg = window(0)
        assert rc != 0 and Jg == J
        assert window(0) == (0, J)               # and the next call is not taken for failed
        with _hip().left((3 * 40 + 72) * N + 200e6):
            assert window(0) == (0, J)


# thin slabs, whose sweeps' copy is larger than the rest of the context: with that
# much memory gone the context is made all the same and sweeps in place
@pytest.mark.parametrize("grid,P,precision,leave", [((1024, 8, 130), 43, "fp64", 0.6), ((1024, 8, 130), 43, "mixed", 0.6),
                                                    ((512, 130, 60), 20, "fp64", 0.87)])
def test_slab_sweeps_without_memory_for_their_copy(tbl, grid, P, precision, leave):
    g, s = make_case(grid, seed=2, P=P)
    _, Q = g.momentum_rhs(s.Ut, s.Press)
    x = g.zeros()
    x[I] = np.random.default_rng(5).standard_normal([n - 2 for n in grid])
    kw = dict(precision=precision, helm_mode=tbl.TBL_HELM_LEX_SLAB, precond=tbl.TBL_PC_SSOR_BLOCK, slabs=P, kmax=2)
    got, held = [], []

    def sweeps(sv):
        sv.set_field(tbl.F_Q, Q)
        y = sv.apply_operator(1, x)
        sw, _ = sv.diffusion_solve(1e-30, 2)
        got.append((sv.get_field(tbl.F_UT), y, list(sw)))
        held.append(sv.device_bytes)

    with gpu_from_case(g, s, **kw) as sv:
        sweeps(sv)
    with _hip().left(leave * held[0]), gpu_from_case(g, s, **kw) as sv:
        sweeps(sv)
    assert held[1] < 0.9 * held[0]
    assert got[1][2] == got[0][2] and np.array_equal(got[1][0], got[0][0]) and np.array_equal(got[1][1], got[0][1])
    if precision == "fp64":
        Uo = s.Ut.copy(order="F")
        g.diffusion_solve(Q, Uo, order=orc.GS_LEX_BLOCK, errorstop=1e-30, mmax=2)
        assert np.array_equal(got[1][0], Uo) and np.array_equal(got[1][1][I], g.precond_apply(x, orc.PC_SSOR_BLOCK)[I])


# a tolerance between what a solve is expected to reach on this grid and what it
# reaches: the unit step is tried, refused, and the Arnoldi steps start from V_0
def test_refused_unit_step_by_the_reference_rule(tbl):
    grid, errtol = (33, 128, 40), 3e-11
    with _solver(tbl, grid, precond=tbl.TBL_PC_FAST, kmax=8) as sv:
        b, got = sv.zeros(), []
        b[I] = np.random.default_rng(1).standard_normal([n - 2 for n in grid])
        sv.set_field(tbl.F_PRHS, b)
        sv.timer_enable(["precond"])
        out = sv.ppe_solve(errtol, 8, 50)
        n = sv.timer_read()["precond"]["count"]
        x = sv.get_field(tbl.F_PCORR)
        r = b - sv.apply_operator(0, x)
        for q in range(3):
            f = np.moveaxis(r, q, 0)
            f[0] = f[-1] = 0.0
        rel = np.linalg.norm(sv.apply_operator(1, r)) / np.linalg.norm(sv.apply_operator(1, b))
    assert n == out["cycles"] + out["iters"] + 1 and out["iters"] > 1
    # the rule's last test is the Arnoldi estimate; it and the residual of the
    # solution differ by the rounding of the solves
    assert rel <= 2 * errtol


# true residual: a tolerance that rounding does not let be met, so that no step of
# the cycle is accepted in the end; refused at once (V_0 in the first vector), or
# after an accepted step (V_0 in the other one)
@pytest.mark.parametrize("inner_tol,accepted", [(1e-16, 0), (1e-6, 1)])
def test_refused_unit_step_by_the_true_residual(tbl, inner_tol, accepted):
    g, s = make_case(GRID, seed=4)
    b, got = _rhs(g), []
    bn = np.linalg.norm(b[I])
    for errtol, timed in ((1e-9, False), (1e-17, False), (1e-17, True)):
        with gpu_from_case(g, s, precond=tbl.TBL_PC_FAST, tol_mode=tbl.TBL_TOL_TRUE, inner_tol=inner_tol, kmax=6) as sv:
            # timed, the next step's first transform is not queued ahead
            sv.timer_enable(["precond", "poisson"] if timed else [])
            out, x = _solve(tbl, sv, g, b, errtol=errtol, kmax=6, mmax=3)
            n = sv.timer_read()
        rn = np.linalg.norm(b[I] - g.poisson_apply(x)[I])
        assert abs(out["true_res"] - rn) <= 1e-6 * rn + 1e-15 * bn
        got.append((out, x, rn))
    assert got[0][0]["iters"] == 1
    assert got[1][0] == got[2][0] and np.array_equal(got[1][1], got[2][1])
    # the steps that follow work at rounding level and leave no more than it
    assert got[1][0]["cycles"] == 3 and n["poisson"]["count"] == got[1][0]["iters"] - accepted
    assert got[1][2] <= 2 * got[0][2]


def test_window_whose_solves_go_one_by_one(tbl):
    """a gradient on a grid beyond the size of batched solves, FP64 (central
    differences, the switches replayed: 1e-5 as on small grids) and mixed (against
    FP64: J 1e-6, gradient 1e-4, as on small grids)"""
    grid, i0, i1 = (1100, 100, 98), 600, 900
    rng = np.random.default_rng(9)
    w = 1e-2 * rng.standard_normal(grid[:2])
    d = rng.standard_normal(grid[:2])
    noise = 0.02 * rng.standard_normal([n - 2 for n in grid] + [3], dtype=np.float32)
    got = []
    for precision in ("fp64", "mixed"):
        with _solver(tbl, grid, precision=precision, precond=tbl.TBL_PC_FAST, kmax=1) as sv:
            U = sv.zeros(3)
            U[..., 0] = 19.8 * np.tanh(4.0 * sv.mesh()["x3"])
            U[I] += noise

            def window(wall, **kw):
                sv.upload(U, sv.zeros(), sv.zeros())
                sv.set_state()
                return sv.adjoint_window(2, i0, i1, wall_w=wall, nsnap=1, **kw)

            got.append(window(w, branch_mode=1)[:2])
            if precision == "fp64":
                eps, ad = 1e-5, float((got[0][1] * d).sum())
                Jp, Jm = (window(w + q * eps * d, forward_only=True, branch_mode=2)[0] for q in (1, -1))
                assert abs((Jp - Jm) / (2 * eps) - ad) <= 1e-5 * abs(ad)
    (J, grad), (Jx, gx) = got
    assert abs(Jx - J) <= 1e-6 * abs(J) and np.abs(gx - grad).max() <= 1e-4 * np.abs(grad).max()
