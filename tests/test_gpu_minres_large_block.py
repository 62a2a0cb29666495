"""MINRES on blocks of 4 Mi entries and more, whose batches exchange the newest Lanczos
vector's buffer with the spare one instead of copying it back, and whose graphs depend
on which of the two holds it (gfx950 only)."""
import numpy as np
import pytest

from invdft_amd import abi
from tests.helpers import random_veff, rel

pytestmark = pytest.mark.gpu

N_CELLS, DEGREE = 20, 5  # 101^3 nodes: 5 columns are 5.2 M entries


@pytest.fixture(scope="module")
def inputs(olib):
    d = abi.default_desc(olib, n_cells=N_CELLS, degree=DEGREE, half_width=4.0, n_eig=6,
                         n_electrons=2.0)
    s = abi.geometry(olib, d)
    rng = np.random.default_rng(5)
    return (s, random_veff(olib, d, 0), rng.standard_normal((s.n_nodes, 6)),
            rng.standard_normal(s.n_cells * s.quad_per_cell))


def _solve(glib, inputs, b, steps, **kw):
    s, veff, psi, u = inputs
    d = abi.default_desc(glib, n_cells=N_CELLS, degree=DEGREE, half_width=4.0, n_eig=b,
                         n_electrons=2.0, **kw)
    z = np.zeros(veff.size)
    g = abi.Context(glib, d, z, z, np.ones(veff.size), np.ones(s.n_nodes))
    g.set_veff_quad(veff)
    mp, x = g.mv(b, np.ascontiguousarray(psi[:, :b])), g.mv(b)
    g.adj_update_input_psi(mp, np.full(b, 0.5), u, [(i, i) for i in range(b)], -0.5,
                           np.linspace(-1.5, -0.7, b))
    g.minres_solve(x, None, 1e-30, steps, distribute=False)
    return x.get()


# runs of check_every steps, more than six of them so that both graphs are captured
# and replayed, then a shorter run: one batch of 2, 6 and 7 + 7 steps; with at most 3 steps a batch (psi_checkpoint) 3 + 3 + 2 and 2 + 2, an odd and
# an even number of exchanges; the last run of the first case is one step long
@pytest.mark.parametrize("b,check_every,steps,ckpt", [(5, 2, 17, 0), (6, 6, 50, 0), (5, 14, 114, 0),
                                                      (6, 8, 67, 1), (5, 4, 33, 1)])
def test_graph_replays_equal_launches(glib, inputs, b, check_every, steps, ckpt):
    print("CASE large_block", b, check_every, steps, ckpt, flush=True)
    kw = dict(check_every=check_every, psi_checkpoint=ckpt)
    x = _solve(glib, inputs, b, steps, minres_graph=1, **kw)
    assert np.array_equal(x, _solve(glib, inputs, b, steps, minres_graph=0, **kw))
    if steps <= 20:
        # the separate steps' sums in another order: rounding grows by the condition
        # number, below 1e4 in so few steps
        assert rel(x, _solve(glib, inputs, b, steps, minres_fused=0, **kw)) < 1e-10


@pytest.mark.parametrize("steps", [12, 14, 20])
def test_batches_equal_separate_steps(glib, inputs, steps):
    """Batches of 6, 7 and 7, 7, 6 steps in one run, at an even width."""
    print("CASE large_block batches", steps, flush=True)
    x = _solve(glib, inputs, 6, steps, check_every=steps)
    assert rel(x, _solve(glib, inputs, 6, steps, check_every=steps, minres_fused=0)) < 1e-10
