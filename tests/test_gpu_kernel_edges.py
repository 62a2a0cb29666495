"""HIP kernels at the sizes where their tilings and dispatch rules have edges
(gfx950 only)."""
import numpy as np
import pytest

from invdft_amd import abi
from tests.helpers import bare_pair, random_veff, rel
from tests.setup_abi import poisson

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


def _adjoint_pair(glib, olib, n_cells, degree, b, pairs, seed=3):
    """computeRhs and distributeX of both backends on the same block."""
    g, o, s = bare_pair(glib, olib, n_cells, degree, 4)
    rng = np.random.default_rng(seed)
    psi = np.linalg.qr(rng.standard_normal((s.n_nodes, b)))[0]
    x = rng.standard_normal((s.n_nodes, b))
    u = rng.standard_normal(s.n_cells * s.quad_per_cell)
    eig = np.sort(rng.uniform(-2.0, -0.5, b))
    occ = rng.uniform(0.1, 1.0, b)
    out = []
    for c in (g, o):
        mp, mx, rhs = c.mv(b, psi), c.mv(b, x), c.mv(b)
        c.adj_update_input_psi(mp, occ, u, pairs, -0.5, eig.copy())
        c.adj_compute_rhs(None, mx, rhs)
        dots = c.adj_dot_quad_wise(mx, mp, len(pairs))
        c.adj_distribute_x()
        out.append((rhs.get(), mx.get(), dots))
    return out


# one column, odd and even widths, more pairs than columns (the dense product),
# and more than one run of 256 pairs
@pytest.mark.parametrize("n_cells,degree,b,extra", [(2, 2, 1, 0), (3, 5, 3, 2), (2, 4, 24, 6),
                                                    (2, 3, 11, 90), (2, 2, 20, 300)])
def test_adjoint_ends_match_oracle(glib, olib, n_cells, degree, b, extra):
    _say("ends", n_cells, degree, b, extra)
    rng = np.random.default_rng(b + extra)
    pairs = {(i, i) for i in range(b)}
    while len(pairs) < min(b + extra, b * b):
        pairs.add(tuple(int(v) for v in rng.integers(0, b, 2)))
    (rg, xg, dg), (ro, xo, do) = _adjoint_pair(glib, olib, n_cells, degree, b, sorted(pairs))
    # sums of some 10^4 products in another order: 1e-15 sqrt(1e4) relative
    assert rel(rg, ro) < 1e-12 and rel(xg, xo) < 1e-12
    assert np.max(np.abs(np.asarray(dg) - do)) < 1e-12 * np.max(np.abs(do))


# interior sizes n = N1 - 2 of the axis transforms: 3, 8, 15, 32 (whole tiles), 65
@pytest.mark.parametrize("n_cells,degree,with_bc", [(2, 2, True), (3, 3, False), (8, 2, True),
                                                    (11, 3, False), (22, 3, True)])
def test_poisson_tile_edges_match_oracle(glib, olib, n_cells, degree, with_bc):
    _say("poisson", n_cells, degree, with_bc)
    d = abi.default_desc(olib, n_cells=n_cells, degree=degree, half_width=3.0)
    xyz = abi.quad_points(olib, d)
    c = np.exp(-np.sum((xyz - [0.4, -0.3, 0.2]) ** 2, axis=1)) * (1.0 + 0.3 * xyz[:, 1])
    bc = None
    if with_bc:
        nx = abi.node_points(olib, d)
        bc = 0.5 + 0.1 * nx[:, 0] - 0.2 * nx[:, 1] * nx[:, 2]
    pg, ng, sg = poisson(glib, d, c, bc=bc, tol=1e-12)
    po, no, so = poisson(olib, d, c, bc=bc, tol=1e-12)
    # both stop at a relative residual of 1e-12; the operator's condition number
    # in the residual's norm is below 1e3 here
    assert rel(pg, po) < 1e-9 and rel(ng, no) < 1e-9
    assert sg.rel_residual <= 1e-12 and abs(sg.charge - so.charge) < 1e-12 * abs(so.charge)


# slots (cell, column) against the slots of a wave, 12, 10, 9 and 8 at p = 2 to 5: a
# wave not filled, exactly filled (8, 40, 72 slots), and one slot more
@pytest.mark.parametrize("p", [2, 3, 4, 5])
@pytest.mark.parametrize("n_cells,ncols", [(2, 1), (2, 5), (2, 9), (3, 3)])
def test_cell_product_wave_edges_match_oracle(glib, olib, p, n_cells, ncols):
    _say("cell_product", n_cells, p, ncols)
    g, o, s = bare_pair(glib, olib, n_cells, p, 4, precision=abi.MIXED)
    x = np.random.default_rng(p + ncols).standard_normal((s.n_nodes, ncols))
    want = o.apply_hamiltonian(x)
    # sums of some 10^2 products per entry and axis: well below 1e3 roundings
    assert rel(g.apply_hamiltonian(x, precision=abi.FP64), want) < 1e-13
    assert rel(g.apply_hamiltonian(x, precision=abi.MIXED), want) < 2e-6


# runs of 1, 2, 3, 8 and 9 steps (batches of 1, 2, 3, 8, and 5 + 4; with the checkpoint
# option at most 3), the last run of a solve cut short by its step limit
@pytest.mark.parametrize("check_every,steps,ckpt", [(1, 3, 0), (2, 5, 0), (3, 7, 1), (8, 8, 1),
                                                    (8, 19, 0), (9, 20, 0)])
def test_batched_minres_updates_match_separate_steps(glib, olib, check_every, steps, ckpt):
    _say("minres_batch", check_every, steps, ckpt)
    b, rng = 3, np.random.default_rng(steps)
    out = []
    for fused in (1, 0):
        d = abi.default_desc(olib, n_cells=3, degree=3, half_width=4.0, n_eig=b, n_electrons=2.0,
                             check_every=check_every, minres_fused=fused, psi_checkpoint=ckpt)
        s = abi.geometry(olib, d)
        zq = np.zeros(s.n_cells * s.quad_per_cell)
        g = abi.Context(glib, d, zq, zq, np.ones(zq.size), np.ones(s.n_nodes))
        g.set_veff_quad(random_veff(olib, d, 0))
        if not out:
            psi = np.linalg.qr(rng.standard_normal((s.n_nodes, b)))[0]
            u = rng.standard_normal(s.n_cells * s.quad_per_cell)
        mp, x = g.mv(b, psi), g.mv(b)
        g.adj_update_input_psi(mp, np.full(b, 0.5), u, [(i, i) for i in range(b)], -0.5,
                               np.array([-1.5, -1.2, -0.7]))
        g.minres_solve(x, None, 1e-30, steps, distribute=False)
        out.append(x.get())
    # at most 20 steps from the same start: rounding grows by the condition number, < 1e4
    assert rel(out[0], out[1]) < 1e-10
