"""Split-K partials where the workspace cannot grow: without memory the problem
runs in one piece, any other failure is passed on.  On the host the decision
itself; on a GPU the calls that fall back, against float64 or the same call with
its partials."""
import os
import subprocess

import numpy as np
import pytest

from conftest import rel_l2
from test_gemm_plans import CSRC, HIPCC, LIB, REPO

LIMIT = str(1 << 20)  # the smallest workspace: the GroupNorms' fits, partials do not


def test_decision(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("needs hipcc")
    exe = tmp_path / "workspace_check"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-x", "hip", "-std=c++17", "-O1", "-I", CSRC,
                    os.path.join(REPO, "tests", "workspace_check.cpp"), "-o", str(exe), "-L", LIB,
                    "-l:libdrawinstant_hip.so", "-Wl,-rpath," + LIB], check=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr


@pytest.fixture
def fresh(monkeypatch, capfd):
    """A device of its own (a workspace never shrinks) and the split counts that
    its contractions ran with since the last look."""
    import drawinstant
    d = drawinstant.Device(0)
    monkeypatch.setenv("DI_TRACE_GEMM", "1")

    def splits():
        return [int(w[7:]) for ln in capfd.readouterr().err.splitlines()
                if ln.startswith("[di_gemm]") for w in ln.split() if w.startswith("splits=")]
    yield d, splits
    d.sync()
    d.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [0, 1])
def test_product(fresh, rng, monkeypatch, dt):
    import drawinstant
    dev, splits = fresh
    M, N, K = 256, 1280, 5120
    t = np.float16 if dt else np.float32
    x = rng.standard_normal((M, K)).astype(t)
    w = (rng.standard_normal((N, K)) / np.sqrt(K)).astype(t)
    bx, bw, y = dev.storage(x), dev.storage(w), dev.create_buffer(M * N * x.itemsize)
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    for limit in (True, False):
        dev.fill_normal(y, M * N, 3, dtype=dt)
        if limit:
            monkeypatch.setenv("DI_WORKSPACE_LIMIT", LIMIT)
        else:
            monkeypatch.delenv("DI_WORKSPACE_LIMIT")
        drawinstant.call("di_linear", dev.ctx, bx.handle, bw.handle, 0, 0, y.handle, M, N, K, 0, dt)
        got = dev.download(y, t, (M, N))
        n = splits()
        assert len(n) == 1 and (n[0] == 1) == limit, n
        # fp32 sums in either case, then one fp16 rounding: 2^-11 / sqrt(3) rms at most
        assert rel_l2(got, ref) <= (2.0 ** -11 if dt else 2e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("ci,co,H,W", [(320, 640, 32, 32), (1280, 1280, 16, 16), (640, 320, 24, 88)])
def test_resnet(fresh, rng, monkeypatch, ci, co, H, W):
    """Shared shortcut slots, GroupNorm in a reducer and statistics in the epilogue
    give way to their unsplit forms: equal up to fp16 roundings of intermediates."""
    from drawinstant import blocks
    dev, splits = fresh
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
    x = dev.storage(rng.standard_normal((1, H, W, ci)).astype(np.float16))
    out = []
    for limit in (True, False):
        if limit:
            monkeypatch.setenv("DI_WORKSPACE_LIMIT", LIMIT)
        else:
            monkeypatch.delenv("DI_WORKSPACE_LIMIT")
        y = dev.create_buffer(H * W * co * 2)
        blocks.resnet_block(dev, w, x, None, y, 1, ci, co, H, W, groups=32)
        out.append(dev.download(y, np.float16, (H, W, co)).astype(np.float64))
        n = splits()
        assert (max(n) == 1) == limit, n
    assert np.isfinite(out[0]).all() and rel_l2(out[0], out[1]) <= 1e-3
    w.destroy()


@pytest.mark.gpu
def test_vae_decode(fresh, rng, monkeypatch):
    """The whole decode, the mid block's attention products among it."""
    from drawinstant.vae import VAE
    dev, splits = fresh
    v = VAE(dev, seed=9)
    z = rng.standard_normal((1, 4, 24, 20)).astype(np.float32)
    out = []
    for limit in (True, False):
        if limit:
            monkeypatch.setenv("DI_WORKSPACE_LIMIT", LIMIT)
        else:
            monkeypatch.delenv("DI_WORKSPACE_LIMIT")
        out.append(np.asarray(v(z), np.float64))
        n = splits()
        assert (max(n) == 1) == limit, n
    assert np.isfinite(out[0]).all() and rel_l2(out[0], out[1]) <= 5e-3
    v.destroy()


@pytest.mark.gpu
def test_unet_step(fresh, rng, monkeypatch):
    """A whole step, GroupNorms of the next block in a reducer among it."""
    from drawinstant.unet import UNet
    dev, splits = fresh
    u = UNet(dev, seed=501)
    x = rng.standard_normal((1, 4, 32, 32)).astype(np.float32)
    ctx = rng.standard_normal((1, 77, 1024)).astype(np.float32)
    out, split = [], []
    for limit in (True, False):
        if limit:
            monkeypatch.setenv("DI_WORKSPACE_LIMIT", LIMIT)
        else:
            monkeypatch.delenv("DI_WORKSPACE_LIMIT")
        out.append(np.asarray(u(x, 999.0, ctx), np.float64))
        split.append(sum(n > 1 for n in splits()))
    assert split[0] < split[1]  # (partials of the 4 x 4 level fit a MiB)
    # fp16 roundings of intermediates through the whole model: 1.4e-3 measured
    assert np.isfinite(out[0]).all() and rel_l2(out[0], out[1]) <= 5e-3
    u.destroy()
