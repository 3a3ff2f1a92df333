"""GPU: the large-image 3x3 convolution kernel (16 x 16 pixel blocks x 128
channels) against a float64 convolution of the fp16-rounded operands: image
sizes on and off the block edges, channel counts off the 128-channel tile, one
to nine channel chunks, several tiles per workgroup, 2x upsampling, batch,
residual and SiLU; and its GroupNorm statistics through the ResNet block.  The
launches' trace shows that the kernel ran (tile 15).

Bound per element: one fp16 rounding of the result and of the residual's sum
(2^-11 each), and (K / 4 + 16) fp32 roundings of sum |x w|."""
import numpy as np
import pytest
import torch
import torch.nn.functional as TF

from conftest import rel_l2

pytestmark = pytest.mark.gpu

F16, NHWC, UP2X, SILU = 1, 1, 2, 4


def conv_tiles(capfd):
    """Tiles of the 3x3 convolutions launched since the last look."""
    lines = [ln.split() for ln in capfd.readouterr().err.splitlines() if ln.startswith("[di_gemm]")]
    return [w[5:] for f in lines if "ks=3" in f for w in f if w.startswith("tile=")]


@pytest.mark.parametrize("N,ci,co,H,W,flags,res", [
    (1, 64, 128, 16, 16, 0, False), (1, 128, 64, 17, 33, 0, True), (2, 192, 192, 24, 40, SILU, True),
    (1, 64, 320, 50, 18, 0, False), (3, 128, 128, 16, 48, UP2X, True), (1, 576, 64, 30, 31, 0, True),
    (1, 64, 128, 264, 272, SILU, True), (1, 128, 128, 136, 150, UP2X, False)])
def test_conv(dev, rng, monkeypatch, capfd, N, ci, co, H, W, flags, res):
    import drawinstant
    x = rng.standard_normal((N, H, W, ci)).astype(np.float16)
    w = (rng.standard_normal((co, 3, 3, ci)) / np.sqrt(9 * ci)).astype(np.float16)
    b = rng.standard_normal(co).astype(np.float32)
    up = 2 if flags & UP2X else 1
    shape = (N, H * up, W * up, co)
    r = rng.standard_normal(shape).astype(np.float16)
    y = dev.create_buffer(int(np.prod(shape)) * 2)
    monkeypatch.setenv("DI_GEMM_TILE", "15")
    monkeypatch.setenv("DI_TRACE_GEMM", "1")
    drawinstant.call("di_conv2d", dev.ctx, dev.storage(x).handle, dev.storage(w).handle,
                     dev.storage(b).handle, dev.storage(r).handle if res else 0, y.handle, N, ci,
                     co, H, W, 3, 1, 1, flags, F16, NHWC)
    assert conv_tiles(capfd) == ["15"]
    got = dev.download(y, np.float16, shape).astype(np.float64)

    def conv(x_, w_, b_):
        t = torch.from_numpy(x_.astype(np.float64)).permute(0, 3, 1, 2)
        t = TF.interpolate(t, scale_factor=2, mode="nearest") if up == 2 else t
        o = TF.conv2d(t, torch.from_numpy(w_.astype(np.float64)).permute(0, 3, 1, 2),
                      torch.from_numpy(b_.astype(np.float64)), padding=1)
        return o.permute(0, 2, 3, 1).numpy()
    z, mag = conv(x, w, b), conv(np.abs(x), np.abs(w), np.abs(b))
    ref = z / (1 + np.exp(-z)) if flags & SILU else z
    ref = ref + r if res else ref
    bound = 2.0 ** -11 * np.abs(ref) + 2.0 ** -24 + \
        1.1 * (9 * ci / 4 + 16) * 2.0 ** -24 * mag + (2.0 ** -20 * np.abs(z) if flags & SILU else 0)
    assert np.isfinite(got).all()
    assert (np.abs(got - ref) <= bound).all(), (np.abs(got - ref) / bound).max()


@pytest.mark.parametrize("B,ci,co,H,W", [(1, 128, 128, 240, 256), (2, 128, 64, 168, 168),
                                         (1, 64, 128, 248, 248), (3, 64, 192, 24, 40)])
def test_resnet_statistics(dev, rng, monkeypatch, capfd, B, ci, co, H, W):
    """The block's second GroupNorm takes conv1's statistics: whole blocks, and
    ragged images whose blocks share slots, against the same block on the other
    conv kernels (equal up to fp16 rounding of the intermediates)."""
    from drawinstant import blocks
    sd = {}
    for i, (o, c) in ((1, (co, ci)), (2, (co, co))):
        sd[f"p.norm{i}.weight"] = (1 + 0.1 * rng.standard_normal(c)).astype(np.float32)
        sd[f"p.norm{i}.bias"] = (0.1 * rng.standard_normal(c)).astype(np.float32)
        sd[f"p.conv{i}.weight"] = (rng.standard_normal((o, c, 3, 3)) / np.sqrt(9 * c)).astype(np.float32)
        sd[f"p.conv{i}.bias"] = rng.standard_normal(o).astype(np.float32)
    if ci != co:
        sd["p.conv_shortcut.weight"] = (rng.standard_normal((co, ci, 1, 1)) / np.sqrt(ci)).astype(np.float32)
        sd["p.conv_shortcut.bias"] = rng.standard_normal(co).astype(np.float32)
    w = blocks.upload_resnet(dev, sd, "p")
    x = dev.storage(rng.standard_normal((B, H, W, ci)).astype(np.float16))
    out = []
    monkeypatch.setenv("DI_TRACE_GEMM", "1")
    for big in (True, False):
        if big:
            monkeypatch.setenv("DI_GEMM_TILE", "15")
        else:
            monkeypatch.delenv("DI_GEMM_TILE")
            monkeypatch.setenv("DI_CONV_BIG", "0")
        y = dev.create_buffer(B * H * W * co * 2)
        blocks.resnet_block(dev, w, x, None, y, B, ci, co, H, W, groups=32)
        out.append(dev.download(y, np.float16, (B, H, W, co)).astype(np.float64))
        tiles = conv_tiles(capfd)
        assert len(tiles) == 2 and all((t == "15") == big for t in tiles), tiles
    assert np.isfinite(out[0]).all() and rel_l2(out[0], out[1]) <= 1e-3
    w.destroy()
