"""Launch shapes: kernels whose split of the domain depends on the grid, at
grids on both sides of each rule and with remainders, against the oracle."""
import numpy as np
import pytest

from oracle import orc
from tests.case_util import gpu_from_case, make_case, ulps

pytestmark = pytest.mark.gpu

I = (slice(1, -1),) * 3
# chunks of the wall-normal march: one plane, a few planes with a shorter last
# chunk, and the longest (momentum 32, Poisson 16 planes)
CHUNKS = [(8, 8, 8), (66, 20, 13), (700, 64, 27), (520, 130, 97)]


@pytest.fixture(scope="module")
def tbl():
    from turbulentbl_amd import tbl as t
    t.load()
    return t


@pytest.mark.parametrize("grid", CHUNKS)
def test_momentum_and_poisson_chunks_bitwise(tbl, grid):
    g, s = make_case(grid, seed=3)
    rng = np.random.default_rng(0)
    s.Press[...] = rng.standard_normal(s.Press.shape)
    x = g.zeros()
    x[I] = rng.standard_normal([n - 2 for n in grid])
    with gpu_from_case(g, s) as sv:
        sv.momentum_rhs()
        Q = sv.get_field(tbl.F_Q)
        y = sv.apply_operator(0, x)
    assert ulps(Q[I], g.momentum_rhs(s.Ut, s.Press)[1][I]) == 0
    assert ulps(y[I], g.poisson_apply(x)[I]) == 0


@pytest.mark.parametrize("precision,rule,errtol,steps", [
    ("fp64", "true", 1e-9, "one"), ("mixed", "true", 1e-9, "one"),      # unit steps accepted
    ("fp64", "ref", 1e-9, "one"), ("mixed", "ref", 1e-4, "one"),
    ("mixed", "ref", 1e-9, "more"),                                     # refused: Arnoldi steps follow
    ("fp64", "true", 1e-9, "last")])                                    # one cycle allowed: not tried
def test_unit_steps_of_the_fast_preconditioner(tbl, precision, rule, errtol, steps):
    """a cycle tries the step of coefficient 1 first; accepted or refused, the
    solve meets its own stopping rule (residual by the oracle's operator) and
    counts its cycles as one-step cycles do"""
    g, s = make_case((70, 12, 21), seed=4)
    b = g.zeros()
    b[I] = np.random.default_rng(22).standard_normal([n - 2 for n in (70, 12, 21)])
    mode = tbl.TBL_TOL_TRUE if rule == "true" else tbl.TBL_TOL_REF
    with gpu_from_case(g, s, precision=precision, tol_mode=mode, errtol=errtol, kmax=8) as sv:
        sv.set_field(tbl.F_PCORR, g.zeros())
        sv.set_field(tbl.F_PRHS, b)
        out = sv.ppe_solve(errtol=errtol, kmax=8, mmax=1 if steps == "last" else 50)
        x = sv.get_field(tbl.F_PCORR)
    rn, bn = np.linalg.norm(b[I] - g.poisson_apply(x)[I]), np.linalg.norm(b[I])
    assert abs(out["true_res"] - rn) <= 1e-6 * rn + 1e-15 * bn
    # the preconditioned residual falls by errtol; A and its inverse are
    # within a factor 1e3 of each other's scaling on this grid.  After refused
    # FP32 steps the rule tests the Arnoldi estimate in FP32, not this residual
    if steps != "more":
        assert rn <= errtol * bn * (1 if rule == "true" else 1e3)
    if steps == "one":
        assert out["iters"] == out["cycles"] - (rule == "true")
    elif steps == "more":
        assert out["iters"] > 1
    else:
        assert out == dict(cycles=1, iters=1, true_res=out["true_res"])


# partial 64-column tiles, partial row tiles, one and several k chunks with a
# shorter last one
@pytest.mark.parametrize("grid", [(66, 20, 13), (130, 10, 70), (101, 34, 45)])
def test_adjoint_momentum_tiles(tbl, grid):
    """the gradient along seeded directions against central differences (the
    switches replayed); eps 1e-6 of a quadratic map: 1e-5 relative, as over the
    longer windows"""
    import torch
    from turbulentbl_amd.autograd import wall_shear_objective
    from tests.case_util import load_case
    g, s = make_case(grid, seed=6)
    i0, i1 = int(0.6 * (g.nX - 1)) + 1, int(0.9 * (g.nX - 1)) + 1
    rng = np.random.default_rng(8)
    base = torch.from_numpy(1e-3 * g.Ue * rng.standard_normal((g.nX, g.nY)))

    def reset(solver):
        load_case(solver, s)

    with gpu_from_case(g, s) as sv:
        w = base.clone().requires_grad_(True)
        wall_shear_objective(w, sv, reset, 3, i0, i1, nsnap=2, freeze=True).backward()
        for _ in range(2):
            d = torch.from_numpy(rng.standard_normal((g.nX, g.nY)) * g.Ue)
            ad, eps = float((w.grad * d).sum()), 1e-6
            with torch.no_grad():
                Jp = wall_shear_objective(base + eps * d, sv, reset, 3, i0, i1, freeze=True)
                Jm = wall_shear_objective(base - eps * d, sv, reset, 3, i0, i1, freeze=True)
            assert abs(float((Jp - Jm) / (2 * eps)) - ad) <= 1e-5 * abs(ad)


# below one chunk of the pinned ring, exactly one, one and a little, more chunks
# than slots; on both sides of the sizes that take a plain copy
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("grid", [(8, 8, 8), (64, 64, 64), (67, 64, 62), (131, 130, 129)])
def test_field_transfers(tbl, grid, precision):
    """what goes to the device comes back, FP32 fields rounded once"""
    rng = np.random.default_rng(3)
    held = np.float32 if precision == "mixed" else np.float64
    with tbl.Solver(*grid, precision=precision, kmax=2, i_rec=4, planes=(2, 3, 4, 5, 6)) as sv:
        U, P, PC = sv.zeros(3), sv.zeros(), sv.zeros()
        for a in (U, P, PC):
            a[...] = rng.standard_normal(a.shape)
        for _ in range(2):
            sv.upload(U, P, PC)
            got = sv.download()
        assert np.array_equal(got[0], U.astype(held)) and np.array_equal(got[1], P.astype(held))
        assert np.array_equal(got[2], PC)


# slab sweeps: one, two and partly filled row blocks; 1, 1, 2, 5, 6, 8 and 32 lines
# a thread; slabs of unequal thickness, partly filled chunks.  FP32 against the
# FP64 oracle: a chain of at most 260 points, four roundings each, 6e-8 relative
# to the largest value
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("grid,P", [((9, 8, 13), 4), ((70, 66, 13), 2), ((12, 68, 39), 3), ((20, 130, 57), 3),
                                    ((67, 66, 44), 1), ((9, 130, 66), 1), ((8, 130, 130), 1)])
def test_slab_sweeps(tbl, grid, P, precision):
    g, s = make_case(grid, seed=2, P=P)
    _, Q = g.momentum_rhs(s.Ut, s.Press)
    x = g.zeros()
    x[1:-1, 1:-1, 1:-1] = np.random.default_rng(5).standard_normal((g.nX - 2, g.nY - 2, g.nZ - 2))
    with gpu_from_case(g, s, precision=precision, helm_mode=tbl.TBL_HELM_LEX_SLAB, precond=tbl.TBL_PC_SSOR_BLOCK,
                       slabs=P) as sv:
        sv.set_field(tbl.F_Q, Q)
        y = sv.apply_operator(1, x)
        sw, _ = sv.diffusion_solve(1e-30, 2)
        Ut = sv.get_field(tbl.F_UT)
    Uo = s.Ut.copy(order="F")
    swo, _ = g.diffusion_solve(Q, Uo, order=orc.GS_LEX_BLOCK, errorstop=1e-30, mmax=2)
    yo = g.precond_apply(x, orc.PC_SSOR_BLOCK)
    assert list(sw) == list(swo)
    if precision == "fp64":
        assert np.array_equal(Ut, Uo) and np.array_equal(y[I], yo[I])
    else:
        assert np.abs(Ut - Uo).max() <= 1e-4 * np.abs(Uo).max()
        assert np.abs(y[I] - yo[I]).max() <= 1e-4 * np.abs(yo[I]).max()


# chunks of the FP64 reductions: one plane, a few with a shorter last chunk, the
# 12-plane limit, and few planes on many tiles.  A sum of n terms in another order
# moves by at most n eps sum |terms|
@pytest.mark.parametrize("grid", [(8, 8, 8), (66, 130, 131), (520, 130, 97), (700, 200, 150), (1500, 400, 8)])
def test_reduction_chunks(tbl, grid):
    g, s = make_case(grid, seed=5)
    _, Q = g.momentum_rhs(s.Ut, s.Press)
    n = (grid[0] - 2) * (grid[1] - 2) * (grid[2] - 2)
    with gpu_from_case(g, s) as sv:
        _, sdiv = sv.div_check()
        sv.set_field(tbl.F_Q, Q)
        _, res = sv.diffusion_solve(1e-30, 1)
    _, sdivo = g.div_check(s.Ut)
    mag = np.abs(g.ppe_rhs(s.Ut)).sum() * g.dt * 10 + 1.0
    assert abs(sdiv - sdivo) <= n * 2.2e-16 * mag
    _, reso = g.diffusion_solve(Q, s.Ut.copy(order="F"), order=orc.GS_LEX_BLOCK, errorstop=1e-30, mmax=1)
    assert np.all(np.abs(res - reso) <= n * 2.2e-16 * reso)


# k groups of the FP64 transforms: one (8 rows are less than a group), two, three,
# four, five and eight, odd counts and partly filled last groups.  The inverse of A
# applied to A x gives x up to rounding times the operator's condition (1e3 to 1e6
# on these grids)
@pytest.mark.parametrize("grid", [(16, 8, 10), (20, 34, 18), (24, 50, 45), (20, 66, 66), (16, 82, 50), (12, 130, 130)])
def test_transform_groups(tbl, grid):
    g, s = make_case(grid, seed=7)
    x = g.zeros()
    x[I] = np.random.default_rng(4).standard_normal([n - 2 for n in grid])
    with gpu_from_case(g, s, precond=tbl.TBL_PC_FAST) as sv:
        y = sv.apply_operator(1, g.poisson_apply(x))
    assert np.abs(y[I] - x[I]).max() <= 1e-9 * np.abs(x).max()
