"""GPU tests of the order in which a launch takes its batches (xcd_runs in
csrc/msod_columns.h): every batch once, at launches around one and two whole
rounds of 8 XCDs times 32 batches, and at one batch and a part of a round; and
of the rule that goes by the order of the elements (nodes_for_order in
csrc/msod_runtime.hip).  Against the CPU oracle on the form's inputs, 1e-12
relative L2 as in the parity tests, 1e-6 with FP32 outputs."""
import numpy as np
import pytest

import minisod2d_amd as m
from forms_lib import FORMS, Arrays, rounded, shuffle
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
    prob = shuffle(prob, perm)
    print(f"[gpu] elements along {along}", flush=True)
    with Arrays(prob, "f64") as a:
        a.convec()
        a.diffu()
        got = a.results()
    for g, w in zip(got, Oracle().convec(prob) + Oracle().diffu(prob)):
        assert rel_l2(g, w) <= 1e-12


@pytest.mark.parametrize("order", ["rows", "z", "random", "rows but for one batch"])
@pytest.mark.parametrize("p,n", [(4, 11), (5, 11)])
def test_orders_of_the_elements(gpu, p, n, order):
    """Launches long enough for columns: the diffusion takes one node per thread
    but for rows, and at order 4 also where one batch is scattered."""
    prob = m.box_problem(n, p, jitter=0.05)
    perm = np.arange(n ** 3)
    if order == "z":
        perm = perm.reshape(n, n, n).transpose(1, 2, 0).ravel()
    elif order == "random":
        perm = np.random.default_rng(5).permutation(perm)
    elif order != "rows":
        far = 133 * np.arange(10)
        perm = np.concatenate([far, np.setdiff1d(perm, far)])
    prob = shuffle(prob, perm)
    for form in FORMS if order == "random" else ("f64", "r4"):
        print(f"[gpu] order of elements p={p} {order} {form}", flush=True)
        with Arrays(prob, form) as a:
            a.convec()
            a.diffu()
            got = a.results()
            q = rounded(prob, a)
        for g, w in zip(got, Oracle().convec(q) + Oracle().diffu(q)):
            assert rel_l2(g, w) <= (1e-6 if form == "r4" else 1e-12), form
