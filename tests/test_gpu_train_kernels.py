"""Weight gradients of the training pass at the edges of its tiles: one 64-row tile pair, widths and
descriptor sizes that leave remainders of the padding, batches that are no multiple of 256, and the
widest rows that the loss keeps in LDS (10,240 components) and the narrowest that it does not."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO
from turbogap_amd import surrogate as SG

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from turbogap_amd import Context
    with Context(0) as c:
        yield c


@pytest.mark.parametrize("D,Hd,B", [(40, 128, 128), (130, 256, 1152), (324, 128, 384), (1224, 384, 256),
                                    (10240, 128, 128), (10241, 128, 128)])
def test_weight_gradients(ctx, D, Hd, B):
    rng = np.random.default_rng(D + B)
    net = SG.MLP(ctx, D, Hd, B + 128, seed=3)
    w = {"W1": rng.normal(size=(Hd, D)), "b1": 0.1 * rng.normal(size=Hd), "W2": rng.normal(size=(Hd, Hd)) / np.sqrt(Hd),
         "b2": 0.1 * rng.normal(size=Hd), "w3": rng.normal(size=Hd) / np.sqrt(Hd), "b3": np.array([0.02])}
    w = {k: v.astype(np.float32) for k, v in w.items()}
    net.set_weights(w)
    q = rng.normal(size=(B, D))
    q = (q / np.linalg.norm(q, axis=1)[:, None]).astype(np.float32)
    e_ref = rng.normal(size=B).astype(np.float32)
    g_ref = (0.3 * rng.normal(size=(B, D))).astype(np.float32)
    grads, le, lg = net.gradients(q, e_ref, g_ref, 0.7, 1.3)
    le_o, lg_o, go = MO.loss_and_grads(w, q.astype(np.float64), e_ref.astype(np.float64), g_ref.astype(np.float64),
                                       0.7, 1.3, emulate_bf16=True)
    # the oracle rounds the same operands to BF16; an activation whose FP32 and FP64 values straddle a
    # rounding boundary differs by one BF16 ulp (2^-8), a few per cent of them at most
    assert abs(le - le_o) <= 1e-2 * le_o and abs(lg - lg_o) <= 1e-2 * lg_o
    for k, v in go.items():
        err = np.linalg.norm(grads[k] - v) / np.linalg.norm(v)
        assert err < 1e-2, (k, err)
    net.close()
