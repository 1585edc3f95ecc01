"""GPU tests of the training loss at the edges of its tiles (64 positives, 128 anchors per
work-group, chunks of the positives) against the oracle, and of the first index among equal
hardest positives.

The hardest positive's score must be within 1e-5 of the best in FP64 from the same codes: two
unit vectors normalised in FP32 (each component within 20 roundings of 2^-24: the sum of
squares, the root, the reciprocal and the product) and a 32-term FP32 dot product err by less
than 2 * 20 * 2^-24 + 32 * 2^-24 = 4.3e-6, twice for the two scores compared.
"""
import numpy as np
import pytest

import v3dmatch
from oracle import learned as OL
from v3dmatch import learned, synth

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


@pytest.fixture(scope="module")
def network():
    m = v3dmatch.SIFT_Matching(0)
    net = learned.Network(m)
    params = learned.init_params(11)
    params["b1"] = (0.05 * np.random.default_rng(2).standard_normal(256)).astype(np.float32)
    net.set_params(params)
    yield net, params
    m.close()


@pytest.mark.parametrize("B", [2, 3, 63, 64, 65, 127, 128, 129, 513, 2050])
def test_hardest_and_gradients(network, B):
    net, params = network
    qA, qP, _ = synth.make_pair(B, B, 1.0, config=7, pair=B)
    pool = np.concatenate([synth.dequantise(qA), synth.dequantise(qP), synth.dequantise(synth.fresh(B, B))])
    i = np.arange(B, dtype=np.int32)
    tri = np.stack([i, B + i, 2 * B + i], 1)
    if B > 8:  # the same positive in two triplets, far apart: equal scores for every other anchor
        tri[B - 2, 1] = tri[1, 1]
    net.set_training(pool, tri)
    loss, g, hard = net.gradients(i)
    z = net.embed(pool[tri.T.reshape(-1)]).astype(np.float64)
    c = z / np.linalg.norm(z, axis=1, keepdims=True)
    S = c[:B] @ c[B:2 * B].T
    np.fill_diagonal(S, -np.inf)
    assert ((hard >= 0) & (hard < B) & (hard != i)).all()
    assert (S.max(1) - S[i, hard] <= 1e-5).all()
    if B > 8:
        assert not ((hard == B - 2) & (i != 1)).any()  # index 1 has the same score and comes first
    Lo, go, _ = OL.loss_and_grads(params, pool, tri, bf16=True, hard=hard)
    assert abs(loss - Lo) <= 1e-3 * abs(Lo) + 1e-5
    for k in g:
        assert _rel(g[k], go[k]) < 1e-2, k
