"""GPU test of the closure's network on a feature that has overflowed: with
weights of one sign the infinity goes through the layers, and the prediction is
infinite (0 where the output weights are negative), not a NaN; the samples
beside it do not notice.  Expected values by the network's definition in NumPy."""
import numpy as np
import pytest

import minisod2d_amd as m
from minisod2d_amd import closure as C
from oracle_lib import Oracle, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("feature", [0, 3, 4, 11])
def test_predict_with_an_infinite_feature(gpu, feature, sign):
    nelem, t = 20, m.hex_tables(2)
    rng = np.random.default_rng(feature)
    P = np.zeros(m.CLOSURE_NPARAM, np.float32)
    P[:C.OW3] = rng.uniform(0.05, 0.3, C.OW3)
    P[C.OW3:C.OB3] = sign * rng.uniform(0.05, 0.3, C.OB3 - C.OW3)
    P[C.OISTD:C.OSCALE] = 1.0
    P[C.OSCALE] = 1e-4
    F = rng.uniform(0.0, 1.0, (nelem * t.nnode, m.CLOSURE_NFEAT)).astype(np.float32)
    hit = np.zeros(len(F), bool)
    hit[[5, 64, 200, 539]] = True
    F[hit, feature] = np.inf
    mu = np.zeros((nelem, t.nnode), order="F")
    print(f"[gpu] infinite feature {feature}, output weights {sign:+.0f}", flush=True)
    m.copyin(F)
    m.create(mu)
    try:
        m.closure_predict(nelem, t.invAtoIJK, P, F, mu)
        m.update_host(mu)
    finally:
        m.delete(F, mu)
    got = mu[:, t.invAtoIJK.ravel(order="F") - 1].ravel()
    assert np.all(got[hit] == (np.inf if sign > 0 else 0.0)), got[hit]
    _, ref = Oracle().mlp_forward(P, F[~hit], quant=1)
    assert rel_l2(got[~hit], ref) <= 1e-3
