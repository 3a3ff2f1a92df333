"""Flash attention with two 16-query groups per wave against one: the same sums
in the same order, so bit-identical, at query counts on and off the 128-query
blocks, masked last key tiles, key ranges over workgroups, scores that raise
the running max in one group only, and fp16 and fp32 tensors; and the rule's
own choice at a grid that takes two, against float64."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

BHSD = 1


def attend(dev, q, k, v, B, H, Sq, Skv, dt):
    import drawinstant
    es = 2 if dt else 4
    o = dev.create_buffer(B * H * Sq * 64 * es)
    dev.fill_normal(o, B * H * Sq * 64, 5, dtype=dt)  # stale output must be overwritten
    drawinstant.call("di_attn_cross", dev.ctx, q.handle, k.handle, v.handle, o.handle, B, H, Sq, Skv,
                     64, BHSD, 0.0, dt)
    return dev.download(o, np.float16 if dt else np.float32, (B, H, Sq, 64))


@pytest.mark.parametrize("dt", [1, 0])
@pytest.mark.parametrize("B,H,Sq,Skv", [(1, 1, 1, 1), (1, 2, 17, 64), (2, 1, 64, 65), (1, 3, 127, 300),
                                        (2, 2, 129, 77), (1, 1, 300, 449), (1, 5, 2049, 4100)])
def test_two_groups_bit_identical(dev, rng, monkeypatch, B, H, Sq, Skv, dt):
    t = np.float16 if dt else np.float32
    q, k, v = (rng.standard_normal((B, H, s, 64)).astype(t) for s in (Sq, Skv, Skv))
    q[:, :, 16 % Sq::32] *= 30  # one group's max rises past the first key tile's
    q, k, v = dev.storage(q), dev.storage(k), dev.storage(v)
    out = []
    for n in ("1", "2"):
        monkeypatch.setenv("DI_ATTN_QGROUPS", n)
        monkeypatch.setenv("DI_ATTN_KGROUPS", "1")
        out.append(attend(dev, q, k, v, B, H, Sq, Skv, dt))
    assert np.isfinite(out[0]).all()
    np.testing.assert_array_equal(out[0], out[1])


def test_large_grid(dev, rng):
    B, H, S = 2, 10, 3001
    q, k, v = (rng.standard_normal((B, H, S, 64)).astype(np.float16) for _ in range(3))
    got = attend(dev, dev.storage(q), dev.storage(k), dev.storage(v), B, H, S, S, 1)
    q, k, v = (a[1, 7].astype(np.float64) for a in (q, k, v))
    p = np.exp(q @ k.T / 8 - (q @ k.T / 8).max(axis=1, keepdims=True))
    # fp16 queries, probabilities and output: 2^-11 each, relative to the result's norm
    assert rel_l2(got[1, 7], p @ v / p.sum(axis=1, keepdims=True)) <= 3 * 2.0 ** -11
