"""Plans of the contractions (gemm_plan), computed on the host: every plan's
launch stays within what a grid may span, at the sizes where it could pass it."""
import os
import shutil
import subprocess

import numpy as np
import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "draw-instant_amd", "csrc")
LIB = os.path.join(REPO, "draw-instant_amd", "drawinstant")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# rows, columns and threads of the built tiles (TileCfg)
TILES = {0: (64, 64, 256), 1: (128, 64, 256), 2: (64, 128, 256), 3: (128, 128, 256),
         5: (64, 160, 256), 6: (64, 64, 512), 7: (128, 64, 512), 8: (64, 128, 512),
         9: (64, 128, 1024), 10: (128, 64, 1024), 11: (128, 128, 1024), 12: (64, 64, 1024),
         14: (64, 32, 512)}
F32_TILES = (0, 1, 3)  # k_gemm_f32


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("needs hipcc")
    exe = tmp_path_factory.mktemp("plans") / "gemm_plan_check"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-x", "hip", "-std=c++17", "-O1", "-I", CSRC,
                    os.path.join(REPO, "tests", "gemm_plan_check.cpp"), "-o", str(exe), "-L", LIB,
                    "-l:libdrawinstant_hip.so", "-Wl,-rpath," + LIB], check=True, timeout=300)

    def plan(problems, **env):
        """(tile, splits) of each problem: dicts of gemm_plan_check's fields."""
        rows = []
        for p in problems:
            q = dict(elem=0, b_mode=0, cus=256, batch=1, act=0, cin=0, h=0, w=0, ks=1, stride=1, up=1,
                     rstats=0)
            q.update(p)
            rows.append(" ".join(str(int(q[k])) for k in (
                "elem", "b_mode", "cus", "batch", "M", "N", "K", "act", "cin", "h", "w", "ks",
                "stride", "up", "rstats")))
        r = subprocess.run([str(exe)], input="\n".join(rows) + "\n", capture_output=True, text=True,
                           timeout=120, env={**os.environ, **env}, check=True)
        out = [tuple(int(v) for v in ln.split()) for ln in r.stdout.splitlines()]
        assert len(out) == len(rows)
        return out
    return plan


def _check(p, tile, splits):
    bm, bn, threads = TILES[tile]
    tiles = -(-p["M"] // bm) * -(-p["N"] // bn)
    assert tiles * threads < 2 ** 32, (p, tile)
    assert splits >= 1 and (splits == 1 or p.get("batch", 1) * splits <= 65535), (p, splits)


def test_grids(planner):
    r = np.random.default_rng(3)
    probs = []
    for elem in (0, 1):
        for b_mode in (0, 1):
            for batch in (1, 3, 1000, 5000, 10000, 20000, 32768, 65535):
                for m, n in ((1, 1), (1, 64), (3, 500), (128, 128)):
                    probs += [dict(elem=elem, b_mode=b_mode, batch=batch, M=m, N=n, K=k)
                              for k in (1, 64, 512, 1024, 4096, 65536, int(r.integers(1, 9000)))]
    # more than 2^32 / 1024 tiles of some shapes
    probs += [dict(elem=1, M=2 ** 24, N=4096, K=64), dict(elem=1, M=2 ** 24, N=8192, K=64),
              dict(elem=0, M=2 ** 18, N=2 ** 18, K=32), dict(elem=0, M=2 ** 24, N=4096, K=64),
              dict(elem=0, M=1, N=2 ** 30, K=4, b_mode=1)]
    for env in ({}, {"DI_GEMM_SPLITS": "64"}):
        for p, (tile, splits) in zip(probs, planner(probs, **env)):
            _check(p, tile, splits)


def test_tile_override_of_fp32(planner):
    """An override names a tile that the fp32 kernel has, or is ignored."""
    probs = [dict(M=m, N=n, K=k, b_mode=b) for m, n, k in ((200, 70, 40), (2048, 1280, 640), (1, 9, 5000))
             for b in (0, 1)] + [dict(M=256, N=64, K=576, cin=64, h=16, w=16, ks=3)]
    own = planner(probs)
    for t in range(-1, 17):
        got = planner(probs, DI_GEMM_TILE=str(t))
        assert got == ([(t, s) for _, s in own] if t in F32_TILES else own), t


def test_large_conv_override_does_not_split(planner):
    """The large-image conv kernel has no split-K: an override that names it runs
    it, in one piece, whatever the plan it replaces or the splits asked for."""
    probs = [dict(elem=1, M=h * w, N=co, K=9 * ci, cin=ci, h=h, w=w, ks=3)
             for ci, co, h, w in ((576, 64, 30, 31), (64, 128, 16, 16), (1280, 1280, 8, 8))]
    for env in ({}, {"DI_GEMM_SPLITS": "3"}):
        assert planner(probs, DI_GEMM_TILE="15", **env) == [(15, 1)] * len(probs)


def test_large_conv_by_the_device_s_cus(planner):
    """60 tiles are less than a third of 256 CUs, and fill 64."""
    p = dict(elem=1, M=45 * 66, N=512, K=9 * 512, cin=512, h=45, w=66, ks=3)
    (whole, _), (part, splits) = planner([p, dict(p, cus=64)])
    assert whole != 15 and (part, splits) == (15, 1)


def test_columns_of_160(planner):
    """Sizes where the 64 x 160 tile is the fastest by 4 to 15 % (N of whole 160s,
    deep K, more than a round of the chip), unless its rows' statistics are wanted,
    which it cannot write; and none of it for GEGLU."""
    probs = [dict(elem=1, M=m, N=n, K=k) for m, n, k in ((3270, 1280, 2560), (3713, 1280, 2560),
                                                         (8016, 640, 2560), (14456, 320, 2560))]
    assert [t for t, _ in planner(probs)] == [5] * 4
    assert 5 not in [t for t, _ in planner([dict(p, rstats=1) for p in probs])]
    assert 5 not in [t for t, _ in planner([dict(p, act=2) for p in probs])]


def test_deep_1x1_convolutions_split(planner):
    """1x1 convolutions of small images over many channels: a split saves 10 to 25 %."""
    probs = [dict(elem=1, M=h * w, N=co, K=1920, cin=1920, h=h, w=w)
             for co, h, w in ((320, 17, 17), (640, 26, 7), (152, 12, 29))]
    assert all(s > 1 for _, s in planner(probs))
