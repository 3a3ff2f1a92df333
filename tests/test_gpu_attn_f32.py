"""GPU: fp32 attention, whose kernel rounds its operands itself, against
float64 at the edges of its key tiles and of the route that reads keys and
values in fp32 (eight tiles), both layouts, query counts off the 64-row blocks,
and outputs over an input's buffer.

Bound: operands in fp16 (2^-11 each on q, k, v and on the probabilities, whose
own error is the score's: |score error| <= 2^-9.5 * |q||k| scale, observed rms
5e-4), asserted as rel-L2 2e-3 and max 2e-2 of the rms."""
import math

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _ref(q, k, v):  # [B, H, S, 64]
    s = np.einsum("bhqd,bhkd->bhqk", q.astype(np.float64), k.astype(np.float64)) / 8.0
    p = np.exp(s - s.max(-1, keepdims=True))
    return np.einsum("bhqk,bhkd->bhqd", p / p.sum(-1, keepdims=True), v.astype(np.float64))


@pytest.mark.parametrize("bhsd", [0, 1])
@pytest.mark.parametrize("over", ["none", "q", "k", "v"])
@pytest.mark.parametrize("B,H,Sq,Skv", [(1, 1, 1, 1), (2, 3, 65, 63), (1, 2, 64, 64), (1, 5, 130, 65),
                                        (2, 2, 100, 512), (1, 3, 70, 513), (1, 2, 576, 576),
                                        (1, 2, 2112, 2112)])
def test_attention_fp32(dev, rng, B, H, Sq, Skv, bhsd, over):
    import drawinstant
    if over in ("k", "v") and Sq != Skv:
        pytest.skip("an output over k or v needs their shape")
    q, k, v = (rng.standard_normal((B, H, s, 64)).astype(np.float32) for s in (Sq, Skv, Skv))
    lay = (lambda a: a) if bhsd else (lambda a: np.ascontiguousarray(a.transpose(0, 2, 1, 3)))
    bufs = {n: dev.storage(lay(a)) for n, a in (("q", q), ("k", k), ("v", v))}
    o = bufs[over] if over != "none" else dev.create_buffer(q.nbytes)
    drawinstant.call("di_attn_cross", dev.ctx, bufs["q"].handle, bufs["k"].handle,
                     bufs["v"].handle, o.handle, B, H, Sq, Skv, 64, bhsd, 0.0, 0)
    got = dev.download(o, np.float32, lay(q).shape)
    ref = lay(_ref(q, k, v))
    assert np.isfinite(got).all()
    assert rel_l2(got, ref) <= 2e-3
    assert np.abs(got - ref).max() <= 2e-2 * math.sqrt(np.mean(ref ** 2))
