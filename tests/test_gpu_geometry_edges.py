"""GPU tests of elem_jacobian at the edges of its split: element counts that
leave a partial step and a partial workgroup, and tables of derivatives that
are no tensor product (more than porder+1 entries in a row), against the C
oracle.  Bar as in the geometry tests (the same terms in the same order, FMA
contraction apart); for the dense tables the sums have porder+1 squared times
as many terms of mixed signs, so theirs is 1e-11."""
import numpy as np
import pytest

import minisod2d_amd as m
from oracle_lib import Oracle, rel_l2

pytestmark = pytest.mark.gpu


def both(p, n, dNgp):
    prob = m.box_problem(n[0], p, ny=n[1], nz=n[2], jitter=0.05)
    t = prob.tables
    He, gp = np.zeros_like(prob.He), np.zeros_like(prob.gpvol)
    D = np.asfortranarray(t.dNgp if dNgp is None else dNgp(t))
    print(f"[gpu] geometry p={p} nelem={prob.nelem}", flush=True)
    m.copyin(prob.connec, prob.coord)
    m.create(He, gp)
    try:
        m.elem_jacobian(p, prob.nelem, prob.npoin, prob.connec, prob.coord, D, t.wgp, gp, He)
        m.update_host(He, gp)
    finally:
        m.delete(prob.connec, prob.coord, He, gp)
    return He, gp, Oracle().jacobian(p, prob.nelem, prob.npoin, prob.connec, prob.coord, D, t.wgp)


@pytest.mark.parametrize("p,n", [(1, (31, 1, 1)), (1, (11, 3, 1)), (2, (17, 1, 1)), (2, (7, 5, 1)), (3, (6, 3, 1)),
                                 (4, (33, 1, 1)), (5, (29, 1, 1)), (6, (9, 1, 1)), (7, (13, 1, 1)), (8, (5, 1, 1))])
def test_ragged_counts(gpu, p, n):
    He, gp, (Ho, go) = both(p, n, None)
    assert rel_l2(He, Ho) < 1e-13 and rel_l2(gp, go) < 1e-13


@pytest.mark.parametrize("p", [1, 4, 7])
def test_dense_tables(gpu, p):
    def dense(t):
        # a small full perturbation: det stays away from zero
        return t.dNgp + 1e-3 / t.nnode * np.random.default_rng(p).normal(size=t.dNgp.shape)

    He, gp, (Ho, go) = both(p, (3, 3, 2), dense)
    assert rel_l2(He, Ho) < 1e-11 and rel_l2(gp, go) < 1e-11
