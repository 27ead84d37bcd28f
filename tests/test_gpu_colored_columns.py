"""GPU tests of the column kernels' coloured form at the smallest meshes that
take it (nodes_for_colors in csrc/msod_runtime.hip): every storage form and
the closure, a partial last batch, the elements of each batch in random order
(their colours within the batch then differ from a row's) and nodes that no
element references, which have to come out as zero.  Against the atomic
assembly and, bit for bit, against a second run.  Bars: 1e-12 relative L2 (the
parity tests'), 1e-6 with FP32 outputs, 1e-4 with the network (bf16 inputs of
sums in another order, the closure tests' bar)."""
import numpy as np
import pytest

import minisod2d_amd as m
from forms_lib import FORMS, Arrays, network, shuffle
from oracle_lib import Oracle, rel_l2

pytestmark = pytest.mark.gpu

EPB = {1: 64, 2: 28, 3: 16, 4: 10, 6: 5}  # ColShape<P>::EPB in csrc/msod_columns.h


def mesh(p, n):
    """n^3 elements but the last four, scrambled within their batches."""
    prob = m.box_problem(n, p, jitter=0.05)
    rng = np.random.default_rng(p)
    keep = prob.nelem - 4
    order = np.concatenate([b + rng.permutation(min(EPB[p], keep - b)) for b in range(0, keep, EPB[p])])
    prob = shuffle(prob, order)
    prob.nelem = keep
    return prob


def run(a, mode, calls):
    m.set_assembly(mode)
    try:
        for o in a.out:
            o.fill(np.nan)
        m.update_device(*a.out)
        for f in calls:
            f()
        return a.results()
    finally:
        m.set_assembly(m.ASSEMBLY_DEFAULT)


# the convection alone takes columns at orders 4 and 6
@pytest.mark.parametrize("p,n,kernels", [(1, 5, "cd"), (1, 13, "cd"), (2, 13, "cd"), (3, 13, "cd"), (4, 30, "c"),
                                         (6, 18, "c")])
def test_forms(gpu, p, n, kernels):
    prob = mesh(p, n)
    referenced = np.zeros(prob.npoin, bool)
    referenced[prob.connec.ravel() - 1] = True
    assert not referenced.all()
    for form in FORMS if p < 4 else ("f64", "r4"):
        print(f"[gpu] coloured columns p={p} n={n} {form}", flush=True)
        with Arrays(prob, form) as a:
            calls = [a.convec] + ([a.diffu] if kernels == "cd" else [])
            want = run(a, m.ASSEMBLY_ATOMIC, calls)
            got = run(a, m.ASSEMBLY_COLORED, calls)
            again = run(a, m.ASSEMBLY_COLORED, calls)
            back = run(a, m.ASSEMBLY_ATOMIC, calls)
        k = 6 if kernels == "cd" else 3
        for x, y, w, v in zip(got[:k], again[:k], want[:k], back[:k]):
            assert np.array_equal(x, y), form
            assert np.all(x[~referenced] == 0), form
            bar = 1e-6 if form == "r4" else 1e-12
            assert rel_l2(x, w) <= bar and rel_l2(v, w) <= bar, form
        if form == "f64" and p < 4:
            for x, w in zip(got, Oracle().convec(prob) + Oracle().diffu(prob)):
                assert rel_l2(x, w) <= 1e-12


@pytest.mark.parametrize("p,n", [(1, 13), (2, 13), (3, 13)])
def test_closure(gpu, p, n):
    prob = mesh(p, n)
    P = network(prob)
    print(f"[gpu] coloured closure columns p={p} n={n}", flush=True)
    with Arrays(prob, "f64") as a:
        call = [lambda: a.closure(P)]
        want, got, again = (run(a, mode, call) for mode in (m.ASSEMBLY_ATOMIC, m.ASSEMBLY_COLORED, m.ASSEMBLY_COLORED))
    for x, y, w in zip(got[3:], again[3:], want[3:]):
        assert np.array_equal(x, y)
        assert rel_l2(x, w) <= 1e-4
