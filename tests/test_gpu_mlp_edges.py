"""GPU tests of the closure's network kernels at the edges of their tiles,
through the C ABI against the CPU oracle: element counts around the 16 of a
prediction workgroup and node counts below and above its 64, sample counts
around the 64 of a gradient chunk and past one round of workgroups, and
features that start off a 16-byte boundary.  Bars as in the closure tests:
bf16 operands on both sides, FP32 sums (1e-3 and 2e-2 per value for the
prediction; the gradient also rounds the back-propagated deltas: 2e-2)."""
import numpy as np
import pytest

import minisod2d_amd as m
from minisod2d_amd import closure as C
from oracle_lib import Oracle, rel_l2

pytestmark = pytest.mark.gpu


def inputs(n, seed, pad):
    rng = np.random.default_rng(seed)
    base = np.zeros(n * 12 + pad, np.float32)
    base[pad:] = rng.normal(0.0, 1.0, n * 12)
    P = np.zeros(m.CLOSURE_NPARAM, np.float32)
    for a, b, sd in ((C.OW1, C.OB1, 0.5), (C.OB1, C.OW2, 0.2), (C.OW2, C.OB2, 0.3), (C.OB2, C.OW3, 0.2),
                     (C.OW3, C.OB3, 0.5)):
        P[a:b] = rng.normal(0.0, sd, b - a)
    P[C.OB3] = -0.3
    P[C.OMEAN:C.OISTD] = 0.1
    P[C.OISTD:C.OSCALE] = 1.1
    P[C.OSCALE] = 1e-4
    return base, base[pad:], P


@pytest.mark.parametrize("nelem,p,pad", [(1, 1, 0), (15, 2, 0), (17, 2, 1), (16, 3, 0), (33, 4, 0), (5, 7, 3)])
def test_predict(gpu, nelem, p, pad):
    t = m.hex_tables(p)
    base, F, P = inputs(nelem * t.nnode, 10 * p + nelem, pad)
    mu = np.zeros((nelem, t.nnode), order="F")
    print(f"[gpu] predict nelem={nelem} p={p} pad={pad}", flush=True)
    m.copyin(base)
    m.create(mu)
    try:
        m.closure_predict(nelem, t.invAtoIJK, P, F, mu)
        m.update_host(mu)
    finally:
        m.delete(base, mu)
    _, ref = Oracle().mlp_forward(P, F.reshape(-1, 12), quant=1)
    got = mu[:, t.invAtoIJK.ravel(order="F") - 1].ravel()
    assert rel_l2(got, ref) <= 1e-3
    assert np.max(np.abs(got - ref) / np.abs(ref)) <= 2e-2


@pytest.mark.parametrize("n,pad", [(1, 0), (63, 0), (64, 2), (65, 0), (1024 * 64 + 17, 0), (3 * 1024 * 64 - 1, 0)])
def test_gradient(gpu, n, pad):
    base, F, P = inputs(n, n, pad)
    gnu = np.random.default_rng(3).uniform(0.5, 1.5, n).astype(np.float32)
    grad = np.full(m.CLOSURE_NTRAIN, np.nan, np.float32)
    print(f"[gpu] gradient n={n} pad={pad}", flush=True)
    m.copyin(base, gnu)
    m.create(grad)
    try:
        m.closure_gradient(n, P, F, gnu, grad)
        m.update_host(grad)
    finally:
        m.delete(base, gnu, grad)
    ref = Oracle().mlp_gradient(P, F.reshape(-1, 12), gnu.astype(np.float64), quant=1)
    assert rel_l2(grad, ref) <= 2e-2
