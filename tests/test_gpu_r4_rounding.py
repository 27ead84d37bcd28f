"""GPU test of the rounding that the rp = 4 entry points state: the
contributions that a workgroup's elements make to a node are summed in FP64
and rounded once to float.  On a mesh of one workgroup every output is then
the FP64 residual rounded once, also where consecutive elements meet along J
or K, at an edge, or with their axes turned against each other.  Bar, per
value: half a unit in the last place of the float nearest the FP64 oracle's
value, plus 1e-12 of the array's largest value for the FP64 sums (the parity
tests' bar).  Two roundings, one per element, miss it at the nodes where the
elements' contributions cancel."""
import numpy as np
import pytest

import minisod2d_amd as m
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

# elements of a workgroup: ColShape<P>::EPB in csrc/msod_columns.h; the
# diffusion at order 7 takes half a batch
EPB = {1: 64, 2: 28, 3: 16, 4: 10, 5: 7, 6: 5, 7: 4, 8: 3}
SHAPES = {"i": lambda n: (n, 1, 1), "j": lambda n: (1, n, 1), "k": lambda n: (1, 1, n),
          "block": lambda n: (2, n // 2, 1) if n > 3 else (1, n, 1)}


def turn_every_other(prob):
    """Every other element's local axes turned by a quarter about K: I -> J, J -> -I."""
    t = prob.tables
    q = t.porder + 1
    line = [0] + list(range(2, q)) + [1]                 # 1-D order by ascending xi
    pos = {s: i for i, s in enumerate(line)}
    perm = np.empty(t.nnode, np.int64)
    for k in range(q):
        for j in range(q):
            for i in range(q):
                i2, j2 = line[q - 1 - pos[j]], i
                inv = lambda a, b, c: t.invAtoIJK[a, b, c] - 1
                perm[inv(i, j, k)] = inv(i2, j2, k)
    connec = prob.connec.copy(order="F")
    connec[1::2] = connec[1::2][:, perm]
    return connec, perm


@pytest.mark.parametrize("shape", ["i", "j", "k", "block", "turned"])
@pytest.mark.parametrize("p", [2, 4, 5, 6, 7, 8])
def test_one_rounding_per_workgroup(gpu, p, shape):
    for kernel in ("convec", "diffu"):
        n = 2 if kernel == "diffu" and p == 7 else EPB[p]
        nx, ny, nz = SHAPES["j" if shape == "turned" else shape](n)
        prob = m.box_problem(nx, p, ny=ny, nz=nz, jitter=0.05)
        if shape == "turned":
            prob.connec, perm = turn_every_other(prob)
            H = m.host_lib()
            bad = H.msodh_elem_jacobian(prob.nelem, prob.npoin, prob.tables.nnode, prob.connec.ctypes.data,
                                        prob.coord.ctypes.data, prob.tables.dNgp.ctypes.data,
                                        prob.tables.wgp.ctypes.data, prob.gpvol.ctypes.data, prob.He.ctypes.data)
            assert bad == 0
        f = {k: np.asfortranarray(getattr(prob, k), dtype=np.float32)
             for k in ("He", "gpvol", "u", "q", "rho", "pr", "E", "Tem", "mu_fluid", "mu_e", "mu_sgs")}
        t = prob.tables
        dlx = np.asfortranarray(t.dlxigp_ip, dtype=np.float32)
        Cp, Pr = np.float32(prob.Cp), np.float32(prob.Pr)
        prob.Cp, prob.Pr = float(Cp), float(Pr)
        for k, v in f.items():
            setattr(prob, k, v.astype(np.float64, order="F"))
        keep, t.dlxigp_ip = t.dlxigp_ip, dlx.astype(np.float64, order="F")
        want = (Oracle().convec if kernel == "convec" else Oracle().diffu)(prob)
        t.dlxigp_ip = keep
        out = [np.zeros(w.shape, np.float32, order="F") for w in want]
        idx = (None, None, f["He"], f["gpvol"], dlx, None, t.invAtoIJK, t.AtoI, t.AtoJ, t.AtoK)
        print(f"[gpu] one rounding {kernel} p={p} {shape} nelem={prob.nelem}", flush=True)
        ins = [prob.connec, *f.values()]
        m.copyin(*ins)
        m.create(*out)
        try:
            if kernel == "convec":
                m.full_convec_ijk_r4(prob.nelem, prob.npoin, prob.connec, *idx, f["u"], f["q"], f["rho"], f["pr"], f["E"],
                                     *out)
            else:
                m.full_diffusion_ijk_r4(prob.nelem, prob.npoin, prob.connec, *idx, Cp, Pr, f["rho"], f["u"], f["Tem"],
                                        f["mu_fluid"], f["mu_e"], f["mu_sgs"], *out)
            m.update_host(*out)
        finally:
            m.delete(*ins, *out)
        for got, w in zip(out, want):
            err = np.abs(got.astype(np.float64) - w)
            bar = 0.5 * np.spacing(np.abs(w).astype(np.float32)).astype(np.float64) + 1e-12 * np.abs(w).max()
            assert (err <= bar).all(), (kernel, float((err / bar).max()), int((err > bar).sum()))
