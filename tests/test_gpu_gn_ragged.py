"""GroupNorm from its producer's statistics on single images whose pixels are
no multiple of the 64-row chunks: the ResNet block of one image against the
same image in a batch of two, where the statistics come from a pass of their
own.  The two differ by the order of fp32 sums and by fp16 roundings of
intermediates that it moves (2^-11 of a few stages)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ci,co,H,W", [
    (64, 64, 1, 1), (64, 320, 3, 11), (128, 64, 9, 7), (320, 640, 5, 13), (1280, 1280, 6, 22),
    (960, 320, 13, 17), (64, 128, 48, 43), (128, 128, 150, 141), (64, 64, 131, 129)])
def test_single_ragged_image(dev, rng, ci, co, H, W):
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
    x = (1 + rng.standard_normal((1, H, W, ci))).astype(np.float16)
    out = []
    for B in (1, 2):
        y = dev.create_buffer(B * H * W * co * 2)
        xb = dev.storage(np.concatenate([x, 0.5 * x][:B]).astype(np.float16))
        blocks.resnet_block(dev, w, xb, None, y, B, ci, co, H, W, groups=32)
        out.append(dev.download(y, np.float16, (B, H, W, co))[0].astype(np.float64))
    assert np.isfinite(out[0]).all() and rel_l2(out[0], out[1]) <= 1e-3
    w.destroy()
