"""Launch shapes: kernels whose split of the domain depends on the grid, at
grids on both sides of each rule and with remainders, against the oracle."""
import numpy as np
import pytest

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
