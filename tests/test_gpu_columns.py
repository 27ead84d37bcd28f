"""GPU tests of the column kernels (porder 1..8) at the edges of their batches,
through the C ABI against the CPU oracle: element counts of one, one less
than a batch, a batch, one more and two batches and one, in both assembly
modes, FP64 and the FP32 storage forms (the FP64 oracle on the rounded
inputs).  Bars as in the parity tests: 1e-12 relative L2 per residual (FP64
arithmetic and sums), 5e-5 for FP32 arithmetic."""
import numpy as np
import pytest

import minisod2d_amd as m
from oracle_lib import Oracle, rel_l2

pytestmark = pytest.mark.gpu

# elements per batch of each order (ColShape<P>::EPB in csrc/msod_columns.h)
EPB = {1: 64, 2: 28, 3: 16, 4: 10, 5: 7, 6: 5, 7: 4, 8: 3}


def on_gpu(prob, convec, diffu, ins):
    R, D = prob.outputs(), prob.outputs()
    m.copyin(*ins)
    m.create(*R, *D)
    try:
        convec(R)
        diffu(D)
        m.update_host(*R, *D)
    finally:
        m.delete(*ins, *R, *D)
    return R + D


@pytest.mark.parametrize("mode", [m.ASSEMBLY_ATOMIC, m.ASSEMBLY_COLORED])
@pytest.mark.parametrize("p", range(1, 9))
def test_batch_edges(gpu, p, mode):
    for n in (1, EPB[p] - 1, EPB[p], EPB[p] + 1, 2 * EPB[p] + 1):
        prob = m.box_problem(n, p, ny=1, nz=1, jitter=0.05)
        print(f"[gpu] p={p} mode={mode} nelem={n}", flush=True)
        m.set_assembly(mode)
        try:
            got = on_gpu(prob, lambda R: m.full_convec_ijk(*prob.convec_args(*R)),
                         lambda D: m.full_diffusion_ijk(*prob.diffu_args(*D)), prob.device_inputs())
        finally:
            m.set_assembly(m.ASSEMBLY_DEFAULT)
        o = Oracle()
        for g, w in zip(got, o.convec(prob) + o.diffu(prob)):
            assert rel_l2(g, w) <= 1e-12


@pytest.mark.parametrize("p", [2, 4, 5, 7, 8])
def test_fp32_storage_at_a_batch_edge(gpu, p):
    prob = m.box_problem(EPB[p] + 1, p, ny=2, nz=1, jitter=0.05)
    f, t = prob.fp32(), prob.tables
    idx = (t.dlxigp_ip, t.invAtoIJK, t.AtoI, t.AtoJ, t.AtoK)
    head = (prob.nelem, prob.npoin, prob.connec, f["He"], f["gpvol"])
    ins = [prob.connec, *f.values(), prob.u, prob.pr]
    for k, v in f.items():
        if k != "u":
            setattr(prob, k, v.astype(np.float64, order="F"))
    o = Oracle()
    got = on_gpu(prob, lambda R: m.full_convec_ijk_f32split(*head, *idx, prob.u, f["q"], f["rho"], prob.pr, f["E"], *R),
                 lambda D: m.full_diffusion_ijk_f32split(*head, *idx, prob.Cp, prob.Pr, f["rho"], prob.u, f["Tem"],
                                                         f["mu_fluid"], f["mu_e"], f["mu_sgs"], *D), ins)
    for g, w in zip(got, o.convec(prob) + o.diffu(prob)):
        assert rel_l2(g, w) <= 1e-12
    prob.u = f["u"].astype(np.float64, order="F")
    prob.pr = (prob.gamma - 1.0) * (prob.E - prob.rho * 0.5 * (prob.u**2).sum(axis=1))
    want = o.convec(prob) + o.diffu(prob)
    for fn, bar in (("mixed", 1e-12), ("fp32", 5e-5)):
        got = on_gpu(prob, lambda R: getattr(m, f"full_convec_ijk_{fn}")(*head, *idx, f["u"], f["q"], f["rho"], f["E"],
                                                                          prob.gamma, *R),
                     lambda D: getattr(m, f"full_diffusion_ijk_{fn}")(*head, *idx, prob.Cp, prob.Pr, f["rho"], f["u"],
                                                                      f["Tem"], f["mu_fluid"], f["mu_e"], f["mu_sgs"],
                                                                      *D), ins)
        for g, w in zip(got, want):
            assert rel_l2(g, w) <= bar


@pytest.mark.parametrize("p,n", [(2, 39), (3, 33), (4, 28), (6, 22)])
def test_colored_batches_of_a_large_mesh(gpu, p, n):
    """Enough batches a colour for the column kernels' coloured form (smaller
    meshes run one node per thread there), against the atomic assembly."""
    prob = m.box_problem(n, p, jitter=0.05)
    print(f"[gpu] coloured columns p={p} nelem={prob.nelem}", flush=True)
    R, D = prob.outputs(), prob.outputs()
    ins = prob.device_inputs()
    got = {}
    m.copyin(*ins)
    m.create(*R, *D)
    try:
        for mode in (m.ASSEMBLY_ATOMIC, m.ASSEMBLY_COLORED):
            m.set_assembly(mode)
            m.full_convec_ijk(*prob.convec_args(*R))
            m.full_diffusion_ijk(*prob.diffu_args(*D))
            m.update_host(*R, *D)
            got[mode] = [x.copy() for x in R + D]
    finally:
        m.set_assembly(m.ASSEMBLY_DEFAULT)
        m.delete(*ins, *R, *D)
    for g, w in zip(got[m.ASSEMBLY_COLORED], got[m.ASSEMBLY_ATOMIC]):
        assert rel_l2(g, w) <= 1e-12
