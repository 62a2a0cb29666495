"""MINRES iterates that a step limit stops, against fixed values (gfx950 only).

Once a Ritz value has converged, rounding decides such an iterate: two orders of the
same sums give solutions 6e-9 to 1e-5 apart here, so no other arithmetic can be the
reference.  The FP64 steps and their right-hand side keep one order of sums instead,
and tests/golden/stopped_iterates.npz holds its values (golden/make_stopped_iterates.py).
"""
import os

import numpy as np
import pytest

from invdft_amd import abi

pytestmark = pytest.mark.gpu

FIX = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "stopped_iterates.npz")
STEPS = 96
# cells, degree, columns, fused steps, columns per work-group of the cell product
CASES = [(6, 2, 3, 1, 4), (4, 3, 4, 1, 4), (3, 4, 5, 1, 2), (3, 5, 2, 1, 4), (4, 3, 9, 1, 8),
         (3, 5, 9, 0, 4)]


def name(case):
    return "x_" + "_".join(str(v) for v in case)


def _dyadic(n, salt):
    """n numbers k / 1024 in [0, 1) from integer arithmetic alone."""
    h = (np.arange(n, dtype=np.uint64) + np.uint64(1000003 * salt)) * np.uint64(0x9E3779B97F4A7C15)
    h = (h ^ (h >> np.uint64(29))) * np.uint64(0xBF58476D1CE4E5B9)
    return ((h ^ (h >> np.uint64(32))) >> np.uint64(54)).astype(np.float64) / 1024.0


def iterate(lib, n_cells, degree, b, fused, columns):
    """Every fifth row of x after STEPS steps of one adjoint block."""
    d = abi.default_desc(lib, n_cells=n_cells, degree=degree, half_width=4.0, n_eig=b,
                         n_electrons=2.0, minres_fused=fused)
    s = abi.geometry(lib, d)
    nq = s.n_cells * s.quad_per_cell
    ctx = abi.Context(lib, d, np.zeros(nq), np.zeros(nq), np.ones(nq), np.ones(s.n_nodes))
    ctx.set_apply_shape(abi.FP64, 1, columns, kernel=abi.KERNEL_SUM_FACTOR)
    ctx.set_veff_quad(-2.0 * _dyadic(nq, 1))
    psi = _dyadic(s.n_nodes * b, 2).reshape(-1, b) - 0.5
    mp, mx = ctx.mv(b, psi), ctx.mv(b)
    pairs = [(i, i) for i in range(b)] + [(0, 1), (1, 0)]
    ctx.adj_update_input_psi(mp, np.full(b, 0.5), _dyadic(nq, 3) - 0.5, pairs, 0.0,
                             -0.5 + 0.25 * np.arange(b))
    ctx.minres_solve(mx, None, 1e-30, STEPS, distribute=False)
    return mx.get()[::5]


@pytest.mark.parametrize("case", CASES, ids=name)
def test_stopped_iterates_keep_their_values(glib, case):
    print("CASE stopped_iterates", case, flush=True)
    want = np.load(FIX)[name(case)]
    x = iterate(glib, *case)
    # equal roundings give equal bits; the bound is that of a result known to 64 bits
    assert np.linalg.norm(x - want) < 1e-9 * np.linalg.norm(want)
