"""Pressure and direct solves: the routes a solve takes when its first step is
not enough, and the buffers it shares with the caller."""
import numpy as np
import pytest

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
