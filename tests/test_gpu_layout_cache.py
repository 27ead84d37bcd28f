"""GPU tests of the cache of derived layouts: four meshes keep all the layouts
that their calls take (both assemblies, FP64 and FP32 outputs, both kernels),
and a fifth takes the oldest one's place.  A layout that is kept is seen by
writing over the connectivity's device copy behind the library's back: calls on
kept layouts do not notice, rebuilt ones do."""
import ctypes

import numpy as np
import pytest

import minisod2d_amd as m
from forms_lib import Arrays
from oracle_lib import Oracle, rel_l2

pytestmark = pytest.mark.gpu


def overwrite(host, values):
    """values into the device copy of a present array, unknown to the library."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    dev = m.hip_lib().msod_data_deviceptr(host.ctypes.data)
    assert hip.hipMemcpy(ctypes.c_void_p(dev), ctypes.c_void_p(values.ctypes.data), ctypes.c_size_t(values.nbytes), 1) == 0


def evaluate(a64, a4):
    """Every layout of a mesh: columns and one node per thread, plans of both kernels, with and without colours."""
    out = []
    for mode in (m.ASSEMBLY_ATOMIC, m.ASSEMBLY_COLORED):
        m.set_assembly(mode)
        try:
            for a in (a64, a4):
                a.convec()
                a.diffu()
                out += a.results()
        finally:
            m.set_assembly(m.ASSEMBLY_DEFAULT)
    return out


def close(x, y):
    return rel_l2(x, y) <= (1e-6 if x.dtype == np.float32 else 1e-12)


def enter(count):
    cases = []
    for i in range(count):
        # order 6, 40 column batches: the convection takes columns, the diffusion and the coloured mode do not
        prob = m.box_problem(5 + i, 6, ny=5, nz=8, jitter=0.05)
        a64, a4 = Arrays(prob, "f64").__enter__(), Arrays(prob, "r4")
        a4.ins = [x for x in a4.ins if x is not prob.connec]
        cases.append((prob, a64, a4.__enter__()))
    return cases


def leave(cases):
    for _, a64, a4 in cases:
        a4.__exit__()
        a64.__exit__()


def test_four_meshes_keep_their_layouts(gpu):
    print("[gpu] layout cache, four meshes", flush=True)
    cases = enter(4)
    try:
        first = [evaluate(a64, a4) for _, a64, a4 in cases]
        for (prob, _, _), got in zip(cases, first):
            for g, w in zip(got, Oracle().convec(prob) + Oracle().diffu(prob)):
                assert rel_l2(g, w) <= 1e-12
        for prob, _, _ in cases:
            overwrite(prob.connec, np.asfortranarray(prob.connec[::-1]))
        for (_, a64, a4), want in zip(cases, first):
            assert all(close(x, y) for x, y in zip(evaluate(a64, a4), want))
    finally:
        leave(cases)


def test_a_fifth_mesh_takes_the_oldest_ones_place(gpu):
    print("[gpu] layout cache, five meshes", flush=True)
    cases = enter(5)
    try:
        first = [evaluate(a64, a4) for _, a64, a4 in cases]
        for prob, _, _ in cases:
            overwrite(prob.connec, np.asfortranarray(prob.connec[::-1]))
        for (_, a64, a4), want in zip(cases[1:], first[1:]):
            assert all(close(x, y) for x, y in zip(evaluate(a64, a4), want))
        prob, a64, a4 = cases[0]
        assert not close(evaluate(a64, a4)[0], first[0][0])  # rebuilt, from the other elements
        # told of new contents, the library rebuilds, and the old layouts go
        m.update_device(prob.connec)
        assert all(close(x, y) for x, y in zip(evaluate(a64, a4), first[0]))
    finally:
        leave(cases)
