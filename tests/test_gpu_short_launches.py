"""GPU tests of both sides of the lines that send short launches of the default
assembly to the kernels with one node per thread (nodes_for_atomics in
csrc/msod_runtime.hip), in every storage form: a batch below the line and at
it, with a last batch of one element, of all but one and full.  The FP64 oracle
on the form's rounded inputs; bars: 1e-12 relative L2 (the parity tests'), 1e-6
with FP32 outputs.  And the two forms of the network's diffusion against the
same call with the viscosity predicted beforehand (1e-10, the closure tests')."""
import numpy as np
import pytest

import minisod2d_amd as m
from forms_lib import FORMS, Arrays, network, rounded
from oracle_lib import Oracle, rel_l2

pytestmark = pytest.mark.gpu

EPB = {3: 16, 4: 10, 5: 7, 6: 5, 8: 3}  # ColShape<P>::EPB in csrc/msod_columns.h
# column batches from which on a launch takes columns: convection, diffusion
LINES = [(3, 48), (4, 88), (5, 80), (6, 24), (6, 128), (8, 80)]


def mesh(p, nelem):
    """The first nelem elements of a box one to six elements deep."""
    nz = 1 if nelem < 100 else 6
    nx = 11
    ny = -(-nelem // (nx * nz))
    prob = m.box_problem(nx, p, ny=ny, nz=nz, jitter=0.05)
    for k in ("connec", "mu_e", "mu_sgs"):
        setattr(prob, k, np.asfortranarray(getattr(prob, k)[:nelem]))
    prob.He = np.asfortranarray(prob.He[:, :, :, :nelem])
    prob.gpvol = np.asfortranarray(prob.gpvol[:, :, :nelem])
    prob.nelem = nelem
    return prob


@pytest.mark.parametrize("p,line", LINES)
def test_both_sides_of_the_line(gpu, p, line):
    for nelem in ((line - 2) * EPB[p] + 1, (line - 1) * EPB[p], (line - 1) * EPB[p] + 1, line * EPB[p] - 1, line * EPB[p]):
        prob = mesh(p, nelem)
        forms = FORMS if nelem == (line - 1) * EPB[p] + 1 else ("f64",)
        for form in forms:
            print(f"[gpu] short launches p={p} nelem={nelem} {form}", flush=True)
            with Arrays(prob, form) as a:
                a.convec()
                a.diffu()
                got = a.results()
                q = rounded(prob, a)
            want = Oracle().convec(q) + Oracle().diffu(q)
            for g, w in zip(got, want):
                assert rel_l2(g, w) <= (1e-6 if form == "r4" else 1e-12), (form, nelem)


@pytest.mark.parametrize("p,nelem", [(2, 100), (3, 700), (3, 800), (4, 900), (5, 1000), (6, 1000), (6, 1100), (7, 20),
                                     (7, 600), (8, 250)])
def test_network(gpu, p, nelem):
    prob = mesh(p, nelem)
    t, P = prob.tables, network(prob)
    F = np.zeros((nelem * t.nnode, m.CLOSURE_NFEAT), np.float32)
    mu = np.zeros((nelem, t.nnode), order="F")
    print(f"[gpu] network p={p} nelem={nelem}", flush=True)
    with Arrays(prob, "f64") as a:
        m.create(F, mu)
        try:
            m.closure_features(nelem, prob.npoin, prob.connec, prob.He, prob.gpvol, t.dlxigp_ip, t.invAtoIJK, t.AtoI,
                               t.AtoJ, t.AtoK, prob.rho, prob.u, F)
            m.closure_predict(nelem, t.invAtoIJK, P, F, mu)
            a.diffu(mu_sgs=mu)
            want = a.results(slice(3, 6))
            assert a.closure(P)
            got = a.results(slice(3, 6))
        finally:
            m.delete(F, mu)
    for g, w in zip(got, want):
        assert rel_l2(g, w) <= 1e-10
