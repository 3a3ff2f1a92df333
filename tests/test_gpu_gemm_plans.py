"""fp16 plans of shapes without a tuned plan: a ResNet shortcut that does not
split hands its sums to a split conv2 as one fp32 slot, with and without the
next GroupNorm in conv2's reducer; and linears whose plans lie at the edges of
the planner's ranges, against float64."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

ACT_GEGLU = 2


@pytest.fixture(scope="module")
def unet(dev):
    from drawinstant.unet import UNet
    u = UNet(dev, seed=501)
    yield u
    u.destroy()


@pytest.mark.parametrize("B,H,W", [(1, 24, 88), (1, 32, 32), (2, 16, 32), (1, 64, 32)])
def test_lone_shortcut_slot(unet, rng, monkeypatch, B, H, W):
    """Against the shortcut as a tensor of its own, and with every GroupNorm as
    its own launch: they differ by fp16 roundings of intermediates (a slot in
    the wrong layout is an error of order one)."""
    x = rng.standard_normal((B, 4, H, W)).astype(np.float32)
    ctx = rng.standard_normal((B, 77, 1024)).astype(np.float32)
    got = unet(x, 999.0, ctx)
    assert np.isfinite(got).all()
    for name in ("DI_SK_PARTIALS", "DI_GN_REDUCE_FUSE"):
        monkeypatch.setenv(name, "0")
        assert rel_l2(unet(x, 999.0, ctx), got) <= 5e-3  # as at 64 x 64: 1.4e-3 measured
        monkeypatch.delenv(name)


@pytest.mark.parametrize("M,N,K,act", [
    (1, 32, 64, ACT_GEGLU), (1, 8, 128, 0), (3, 64, 64, ACT_GEGLU), (65, 104, 4096, 0),
    (17, 4, 640, 0), (2049, 72, 1280, 0), (129, 10240, 64, ACT_GEGLU), (4097, 320, 2048, 0)])
def test_linear(dev, rng, M, N, K, act):
    import drawinstant
    from scipy.special import erf
    geglu = act == ACT_GEGLU
    x = rng.standard_normal((M, K)).astype(np.float16)
    w = (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float16)
    b = rng.standard_normal(N).astype(np.float32)
    nout = N // 2 if geglu else N
    y = dev.create_buffer(M * nout * 2)
    drawinstant.call("di_linear", dev.ctx, dev.storage(x).handle, dev.storage(w).handle,
                     dev.storage(b).handle, 0, y.handle, M, N, K, act, drawinstant.F16)
    got = dev.download(y, np.float16).reshape(M, nout).astype(np.float64)
    x, w = x.astype(np.float64), w.astype(np.float64)
    # fp32 sums: K + 16 roundings of 2^-24 of sum |x w|, then one to fp16
    err = (K + 16) * 2.0 ** -24 * (np.linalg.norm(x, axis=1)[:, None] *
                                   np.linalg.norm(w, axis=1)[None, :] + np.abs(b))
    z = x @ w.T + b
    if geglu:  # 32-column groups [16 hidden | 16 gate]; |gelu'| <= 1.13, erf to 2^-20
        h, g = z.reshape(M, -1, 2, 16)[:, :, 0].reshape(M, nout), z.reshape(M, -1, 2, 16)[:, :, 1].reshape(M, nout)
        eh, eg = err.reshape(M, -1, 2, 16)[:, :, 0].reshape(M, nout), err.reshape(M, -1, 2, 16)[:, :, 1].reshape(M, nout)
        gelu = 0.5 * g * (1 + erf(g / np.sqrt(2)))
        z, err = h * gelu, np.abs(gelu) * eh + np.abs(h) * (1.13 * eg + 2.0 ** -20 * np.abs(g))
    assert (np.abs(got - z) <= err + 2.0 ** -11 * np.abs(z) + 2.0 ** -24).all()
