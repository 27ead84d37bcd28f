"""GPU tests of the coloured assembly on meshes whose elements are in no
spatial order, in every storage form and with the closure's network.  The
batches of the column kernels need more than 32 colours there, smaller batches
do not: the call runs on those, equals the atomic assembly and repeats bit for
bit.  Bars: 1e-12 relative L2 against the atomic assembly (the parity tests'),
1e-6 with FP32 outputs (a float's rounding per batch), 1e-4 with the network
(its inputs are rounded to bf16 after sums of another order; the closure tests'
bar)."""
import numpy as np
import pytest

import minisod2d_amd as m
from forms_lib import FORMS, Arrays, network, shuffle
from oracle_lib import rel_l2

pytestmark = pytest.mark.gpu

# random element order: more than 32 colours at ColShape<P>::EPB elements a
# batch, fewer at Shape<P>::BATCH and CShape<P>::BATCH
MESHES = [(4, 10), (5, 8), (6, 18)]


def scattered(p, n):
    prob = m.box_problem(n, p, jitter=0.05)
    return shuffle(prob, np.random.default_rng(3).permutation(prob.nelem))


@pytest.mark.parametrize("p,n", MESHES)
def test_scattered_elements(gpu, p, n):
    prob = scattered(p, n)
    for form in FORMS:
        print(f"[gpu] coloured, scattered elements p={p} n={n} {form}", flush=True)
        got = {}
        with Arrays(prob, form) as a:
            try:
                for mode in (m.ASSEMBLY_ATOMIC, m.ASSEMBLY_COLORED):
                    m.set_assembly(mode)
                    for _ in range(2):
                        a.convec()
                        a.diffu()
                        got.setdefault(mode, []).append(a.results())
            finally:
                m.set_assembly(m.ASSEMBLY_DEFAULT)
        first, again = got[m.ASSEMBLY_COLORED]
        for x, y, w in zip(first, again, got[m.ASSEMBLY_ATOMIC][0]):
            assert np.array_equal(x, y), form
            assert rel_l2(x, w) <= (1e-6 if form == "r4" else 1e-12), form


@pytest.mark.parametrize("p,n", MESHES)
def test_scattered_elements_with_the_network(gpu, p, n):
    prob = scattered(p, n)
    P = network(prob)
    print(f"[gpu] coloured closure, scattered elements p={p} n={n}", flush=True)
    got = []
    with Arrays(prob, "f64") as a:
        try:
            for mode in (m.ASSEMBLY_ATOMIC, m.ASSEMBLY_COLORED, m.ASSEMBLY_COLORED):
                m.set_assembly(mode)
                assert a.closure(P)
                got.append(a.results(slice(3, 6)))
        finally:
            m.set_assembly(m.ASSEMBLY_DEFAULT)
    for w, x, y in zip(*got):
        assert np.array_equal(x, y)
        assert rel_l2(x, w) <= 1e-4
