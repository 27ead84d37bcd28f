"""GPU test of the order in which a launch takes its batches (xcd_runs in
csrc/msod_columns.h): every batch once, at launches around one and two whole
rounds of 8 XCDs times 32 batches, and at one batch and a part of a round.
Against the CPU oracle, 1e-12 relative L2 as in the parity tests."""
import numpy as np
import pytest

import minisod2d_amd as m
from forms_lib import Arrays
from oracle_lib import Oracle, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 31, 255, 256, 257, 300, 511, 512, 513, 777])
def test_every_batch_once(gpu, nb):
    """Order 1: 64 elements a batch."""
    prob = m.box_problem(16, 1, ny=4, nz=nb, jitter=0.05)
    assert prob.nelem == 64 * nb
    print(f"[gpu] batch order nb={nb}", flush=True)
    with Arrays(prob, "f64") as a:
        a.convec()
        a.diffu()
        got = a.results()
    for g, w in zip(got, Oracle().convec(prob) + Oracle().diffu(prob)):
        assert rel_l2(g, w) <= 1e-12


@pytest.mark.parametrize("along", ["y", "z"])
def test_elements_across_the_rows(gpu, along):
    """Consecutive elements along y or z, several rounds of batches."""
    n = 24
    prob = m.box_problem(n, 2, jitter=0.05)
    e = np.arange(n ** 3).reshape(n, n, n)
    perm = (e.transpose(0, 2, 1) if along == "y" else e.transpose(1, 2, 0)).ravel()
    for k in ("connec", "mu_e", "mu_sgs"):
        setattr(prob, k, np.asfortranarray(getattr(prob, k)[perm]))
    prob.He = np.asfortranarray(prob.He[:, :, :, perm])
    prob.gpvol = np.asfortranarray(prob.gpvol[:, :, perm])
    print(f"[gpu] elements along {along}", flush=True)
    with Arrays(prob, "f64") as a:
        a.convec()
        a.diffu()
        got = a.results()
    for g, w in zip(got, Oracle().convec(prob) + Oracle().diffu(prob)):
        assert rel_l2(g, w) <= 1e-12
