"""GPU tests of the plan that the atomic assembly builds on the device, against
the CPU oracle and the host's plan (the coloured assembly's) on the same
arrays: node numbers in no order, elements in no order, nodes that repeat
within an element and a batch (atomic assembly alone: the coloured sums take an
element's nodes to be distinct), a partial last batch, and the refusal of node
numbers out of range.  Bar: 1e-12 relative L2 as in the parity tests."""
import numpy as np
import pytest

import minisod2d_amd as m
from oracle_lib import Oracle, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("repeat", [False, True])
@pytest.mark.parametrize("p,n", [(1, (13, 5, 1)), (2, (5, 3, 2)), (3, (17, 1, 1)), (4, (7, 3, 1)), (5, (5, 1, 1)),
                                 (6, (3, 1, 1)), (7, (3, 1, 1)), (8, (1, 1, 1))])
def test_device_plan_matches_host_plan(gpu, p, n, repeat):
    prob = m.box_problem(n[0], p, ny=n[1], nz=n[2], jitter=0.05)
    rng = np.random.default_rng(p)
    connec = (rng.permutation(prob.npoin) + 1).astype(np.int32)[prob.connec - 1][rng.permutation(prob.nelem)]
    if repeat:
        connec[0, 1] = connec[0, 0]  # a node twice in an element,
        connec[-1, 2] = connec[0, 0]  # and far from its place
    prob.connec = np.asfortranarray(connec)
    print(f"[gpu] plan p={p} nelem={prob.nelem}", flush=True)
    want = Oracle().convec(prob) + Oracle().diffu(prob)
    R, D = prob.outputs(), prob.outputs()
    ins = prob.device_inputs()
    m.copyin(*ins)
    m.create(*R, *D)
    try:
        for mode in (m.ASSEMBLY_ATOMIC,) if repeat else (m.ASSEMBLY_ATOMIC, m.ASSEMBLY_COLORED, m.ASSEMBLY_ATOMIC):
            m.set_assembly(mode)
            m.full_convec_ijk(*prob.convec_args(*R))
            m.full_diffusion_ijk(*prob.diffu_args(*D))
            m.update_host(*R, *D)
            for g, w in zip(R + D, want):
                assert rel_l2(g, w) <= 1e-12, mode
    finally:
        m.set_assembly(m.ASSEMBLY_DEFAULT)
        m.delete(*ins, *R, *D)


@pytest.mark.parametrize("p", [2, 4, 7])
def test_bad_entries_are_counted(gpu, p):
    prob = m.box_problem(5, p, ny=3, nz=1)
    bad = np.asfortranarray(prob.connec.copy())
    bad[0, 0], bad[7, 3], bad[14, 5] = 0, prob.npoin + 1, -2  # the last: in the padded last batch
    prob.connec = bad
    R = prob.outputs()
    ins = prob.device_inputs()
    print(f"[gpu] bad connec p={p}", flush=True)
    m.copyin(*ins)
    m.create(*R)
    try:
        with pytest.raises(m.MsodError, match="connec holds 3 node numbers outside") as e:
            m.full_convec_ijk(*prob.convec_args(*R))
    finally:
        m.delete(*ins, *R)
    assert e.value.status == m.MSOD_ERR_MESH
