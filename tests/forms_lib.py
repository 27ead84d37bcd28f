"""Both residuals of a problem through each storage form's entry points, for
the GPU tests that run several of them."""
import numpy as np

import minisod2d_amd as m
from minisod2d_amd import closure as C

FORMS = ("f64", "geo32", "f32split", "mixed", "r4")
F32 = {"f64": (), "geo32": ("He", "gpvol", "mu_e", "mu_sgs"),
       "f32split": ("He", "gpvol", "q", "rho", "E", "Tem", "mu_fluid", "mu_e", "mu_sgs")}
F32["mixed"] = F32["r4"] = ("He", "gpvol", "u", "q", "rho", "pr", "E", "Tem", "mu_fluid", "mu_e", "mu_sgs")
ARRAYS = ("He", "gpvol", "u", "q", "rho", "pr", "E", "Tem", "mu_fluid", "mu_e", "mu_sgs")


def shuffle(prob, perm):
    """The problem with its elements in another order."""
    for k in ("connec", "mu_e", "mu_sgs"):
        setattr(prob, k, np.asfortranarray(getattr(prob, k)[perm]))
    prob.He = np.asfortranarray(prob.He[:, :, :, perm])
    prob.gpvol = np.asfortranarray(prob.gpvol[:, :, perm])
    return prob


def rounded(prob, a):
    """The problem on the form's inputs, widened."""
    q = m.box_problem(1, prob.porder)
    for k in ("nelem", "npoin", "connec"):
        setattr(q, k, getattr(prob, k))
    for k in ("He", "gpvol", "u", "q", "rho", "pr", "E", "Tem", "mu_fluid", "mu_e", "mu_sgs"):
        setattr(q, k, np.asfortranarray(getattr(a, k), dtype=np.float64))
    if a.form == "mixed":
        q.pr = (q.gamma - 1.0) * (q.E - q.rho * 0.5 * (q.u ** 2).sum(axis=1))
    if a.form == "r4":
        q.tables.dlxigp_ip = np.asfortranarray(a.dlx, dtype=np.float64)
        q.Cp, q.Pr = float(np.float32(q.Cp)), float(np.float32(q.Pr))
    return q


def network(prob, seed=7):
    """Weights near a constant viscosity, standardised by rough scales of the fields."""
    rng = np.random.default_rng(seed)
    P = np.zeros(m.CLOSURE_NPARAM, np.float32)
    for a, b, sd in ((C.OW1, C.OB1, 0.3), (C.OB1, C.OW2, 0.1), (C.OW2, C.OB2, 0.2), (C.OB2, C.OW3, 0.1),
                     (C.OW3, C.OB3, 0.1)):
        P[a:b] = rng.normal(0.0, sd, b - a)
    P[C.OB3] = 0.5
    P[C.OISTD:C.OSCALE] = 0.2
    P[C.OSCALE] = 5e-4
    return P


class Arrays:
    """The problem's arrays in the storage of a form, in the data region."""

    def __init__(self, prob, form):
        self.prob, self.form = prob, form
        for k in ARRAYS:
            a = getattr(prob, k)
            setattr(self, k, np.asfortranarray(a, dtype=np.float32) if k in F32[form] else a)
        out = np.float32 if form == "r4" else np.float64
        n = prob.npoin
        self.out = [np.zeros(s, out, order="F") for s in (n, (n, 3), n, n, (n, 3), n)]
        self.ins = [prob.connec] + [getattr(self, k) for k in ARRAYS]
        self.dlx = prob.tables.dlxigp_ip
        if form == "r4":
            self.dlx = np.asfortranarray(self.dlx, dtype=np.float32)

    def __enter__(self):
        m.copyin(*self.ins)
        m.create(*self.out)
        return self

    def __exit__(self, *a):
        m.delete(*self.ins, *self.out)

    def _head(self):
        p, t = self.prob, self.prob.tables
        idx = (t.invAtoIJK, t.AtoI, t.AtoJ, t.AtoK)
        a = (p.nelem, p.npoin, p.connec)
        if self.form in ("f64", "r4"):
            return (*a, t.Ngp, t.dNgp, self.He, self.gpvol, self.dlx, t.xgp, *idx) if self.form == "f64" else \
                   (*a, None, None, self.He, self.gpvol, self.dlx, None, *idx)
        return (*a, self.He, self.gpvol, self.dlx, *idx)

    def convec(self):
        fn = getattr(m, "full_convec_ijk" + ("" if self.form == "f64" else "_" + self.form))
        if self.form == "mixed":
            fn(*self._head(), self.u, self.q, self.rho, self.E, self.prob.gamma, *self.out[:3])
        else:
            fn(*self._head(), self.u, self.q, self.rho, self.pr, self.E, *self.out[:3])

    def diffu(self, mu_sgs=None):
        fn = getattr(m, "full_diffusion_ijk" + ("" if self.form == "f64" else "_" + self.form))
        fn(*self._head(), self.prob.Cp, self.prob.Pr, self.rho, self.u, self.Tem, self.mu_fluid, self.mu_e,
           self.mu_sgs if mu_sgs is None else mu_sgs, *self.out[3:])

    def closure(self, params):
        return m.full_diffusion_ijk_closure(*self._head(), self.prob.Cp, self.prob.Pr, self.rho, self.u, self.Tem,
                                            self.mu_fluid, self.mu_e, params, *self.out[3:])

    def results(self, k=slice(None)):
        m.update_host(*self.out)
        return [o.copy() for o in self.out[k]]
