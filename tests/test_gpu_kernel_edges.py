"""HIP kernels at the sizes where their tilings and dispatch rules have edges
(gfx950 only)."""
import numpy as np
import pytest

from invdft_amd import abi
from tests.helpers import bare_pair

pytestmark = pytest.mark.gpu


def _say(*a):
    print("CASE", *a, flush=True)


def _boundary(n1):
    i = np.arange(n1)
    e = (i == 0) | (i == n1 - 1)
    return (e[:, None, None] | e[None, :, None] | e[None, None, :]).reshape(-1)


@pytest.mark.parametrize("n_cells,degree,b", [(2, 2, 1), (3, 4, 3), (5, 5, 12), (4, 3, 80)])
def test_vmult_clears_exactly_the_boundary_rows(glib, olib, n_cells, degree, b):
    """vmult zeroes the boundary rows of its input and leaves the others."""
    _say("boundary", n_cells, degree, b)
    g, _, s = bare_pair(glib, olib, n_cells, degree, 4)
    rng = np.random.default_rng(b)
    x = rng.uniform(1.0, 2.0, (s.n_nodes, b))
    psi, xv, out = g.mv(b, x), g.mv(b, x), g.mv(b)
    g.adj_update_input_psi(psi, np.ones(b), np.zeros(s.n_cells * s.quad_per_cell), [], 0.0,
                           np.zeros(b))
    g.adj_vmult(out, xv)
    want = np.where(_boundary(n_cells * degree + 1)[:, None], 0.0, x)
    assert np.array_equal(xv.get(), want)
    assert np.array_equal(psi.get(), want)
