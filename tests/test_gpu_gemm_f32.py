"""GPU: the fp32 contractions on the bf16 matrix cores (k_gemm_f32.hip) against
float64, at the edges of their tiles (64 / 128 rows and columns, 32-deep
stages), over both operand orders, fp16-resident weights, every convolution
form and non-finite inputs.

Bound per element: an fp32 sum of K products in any order of at least four
products per rounding step errs by at most (K / 4 + 16) roundings of 2^-24 of
sum |a b| (the 16 covers the split's remainder and the last additions)."""
import numpy as np
import pytest
import torch
import torch.nn.functional as TF

pytestmark = pytest.mark.gpu

F32, F32W16, NCHW = 0, 2, 0
UP2X, SILU, GEGLU = 2, 4, 2


def _call(dev, fn, *a):
    import drawinstant
    drawinstant.call(fn, dev.ctx, *a)


def _check(got, ref, mag, K, extra=0.0):
    err = np.abs(got.astype(np.float64) - ref)
    bound = (K / 4 + 16) * 2.0 ** -24 * mag + 2.0 ** -23 * np.abs(ref) + extra
    assert got.shape == ref.shape and np.isfinite(got).all()
    assert (err <= bound).all(), f"{(err / bound).max():.2f} x the bound"


def _mats(rng, ash, bsh, scale=1.0, w16=False):
    a = (rng.standard_normal(ash) * scale).astype(np.float32)
    b = rng.standard_normal(bsh).astype(np.float32)
    return a, b.astype(np.float16) if w16 else b


@pytest.mark.parametrize("w16", [False, True])
@pytest.mark.parametrize("trans_b", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (63, 65, 31), (64, 64, 32), (65, 130, 33),
                                   (129, 127, 100), (3, 1281, 2049), (300, 64, 4100)])
def test_gemm(dev, rng, M, N, K, trans_b, w16):
    a, b = _mats(rng, (M, K), (N, K) if trans_b else (K, N), w16=w16)
    c = rng.standard_normal(N).astype(np.float32)
    y = dev.create_buffer(M * N * 4)
    _call(dev, "di_gemm", dev.storage(a).handle, dev.storage(b).handle, dev.storage(c).handle,
          y.handle, M, N, K, trans_b, F32W16 if w16 else F32)
    b64 = b.astype(np.float64).T if trans_b else b.astype(np.float64)
    a64 = a.astype(np.float64)
    _check(dev.download(y).reshape(M, N), a64 @ b64 + c, np.abs(a64) @ np.abs(b64) + np.abs(c), K)


@pytest.mark.parametrize("batched", [0, 1])
@pytest.mark.parametrize("M,N,K,bt,scale", [(77, 66, 64, 3, 1.0), (40, 77, 130, 5, 2.0 ** -60),
                                            (128, 64, 257, 2, 2.0 ** 60)])
def test_matmul(dev, rng, M, N, K, bt, scale, batched):
    a, b = _mats(rng, (bt, M, K), (bt, K, N) if batched else (K, N), scale)
    y = dev.create_buffer(bt * M * N * 4)
    _call(dev, "di_matmul", dev.storage(a).handle, dev.storage(b).handle, y.handle, M, N, K, bt,
          batched, F32)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    _check(dev.download(y).reshape(bt, M, N), a64 @ b64, np.abs(a64) @ np.abs(b64), K)


@pytest.mark.parametrize("M,N,K", [(70, 96, 40), (33, 32, 1500)])
def test_linear_geglu_residual(dev, rng, M, N, K):
    x, w = _mats(rng, (M, K), (N, K))
    w /= np.float32(np.sqrt(K))
    b = rng.standard_normal(N).astype(np.float32)
    r = rng.standard_normal((M, N // 2)).astype(np.float32)
    y = dev.create_buffer(M * N * 2)
    _call(dev, "di_linear", dev.storage(x).handle, dev.storage(w).handle, dev.storage(b).handle,
          dev.storage(r).handle, y.handle, M, N, K, GEGLU, F32)
    h = x.astype(np.float64) @ w.astype(np.float64).T + b
    g = h.reshape(M, N // 32, 2, 16)
    ref = (g[:, :, 0] * TF.gelu(torch.from_numpy(g[:, :, 1])).numpy()).reshape(M, N // 2) + r
    got = dev.download(y).reshape(M, N // 2)
    # the GELU's erf polynomial (1.5e-7) times |hidden * gate| dominates
    assert np.abs(got - ref).max() <= 4e-6 * (1 + np.abs(ref).max())


@pytest.mark.parametrize("w16", [False, True])
@pytest.mark.parametrize("N,ci,co,H,W,k,s,flags", [
    (1, 3, 5, 9, 11, 3, 1, 0), (2, 64, 70, 8, 8, 3, 2, 0), (1, 67, 65, 13, 10, 1, 1, 0),
    (3, 33, 64, 5, 7, 3, 1, SILU), (1, 20, 130, 12, 12, 5, 1, 0), (2, 40, 64, 6, 9, 3, 1, UP2X),
    (1, 300, 64, 16, 8, 3, 1, 0), (1, 7, 3, 20, 20, 7, 3, SILU), (2, 96, 128, 8, 16, 1, 2, 0)])
def test_conv(dev, rng, N, ci, co, H, W, k, s, flags, w16):
    x, w = _mats(rng, (N, ci, H, W), (co, ci, k, k), w16=w16)
    b = rng.standard_normal(co).astype(np.float32)

    def conv(x_, w_, b_):
        x_ = torch.from_numpy(x_.astype(np.float64))
        x_ = TF.interpolate(x_, scale_factor=2, mode="nearest") if flags & UP2X else x_
        return TF.conv2d(x_, torch.from_numpy(w_.astype(np.float64)),
                         torch.from_numpy(b_.astype(np.float64)), s, k // 2).numpy()
    z, mag = conv(x, w, b), conv(np.abs(x), np.abs(w), np.abs(b))
    r = rng.standard_normal(z.shape).astype(np.float32)
    y = dev.create_buffer(z.size * 4)
    _call(dev, "di_conv2d", dev.storage(x).handle, dev.storage(w).handle, dev.storage(b).handle,
          dev.storage(r).handle, y.handle, N, ci, co, H, W, k, s, k // 2, flags,
          F32W16 if w16 else F32, NCHW)
    ref = (z / (1 + np.exp(-z)) if flags & SILU else z) + r
    # SiLU: slope at most 1.1, and a 2-ulp exponential and reciprocal
    _check(dev.download(y).reshape(z.shape), ref, 1.1 * mag + np.abs(r), ci * k * k,
           2.0 ** -20 * np.abs(z) if flags & SILU else 0.0)


@pytest.mark.parametrize("M,N,K", [(70, 66, 40), (130, 128, 1100)])
def test_non_finite(dev, rng, M, N, K):
    """Infinities, NaNs and a value that rounds past bf16's largest follow the
    fp32 rules (inf * 0 is NaN); rows without them keep the bound."""
    a, b = _mats(rng, (M, K), (N, K))
    b[1] = 1.0  # exact in one part: its other parts are zeros
    a[0, 3], a[2, K - 1], a[5, 7] = np.inf, -np.inf, np.nan
    a[66, 0] = 3.4e38
    b[:, 0] *= 1e-3
    b[4, 3] = 0.0
    y = dev.create_buffer(M * N * 4)
    _call(dev, "di_gemm", dev.storage(a).handle, dev.storage(b).handle, 0, y.handle, M, N, K, 1, F32)
    got = dev.download(y).reshape(M, N)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref, mag = a64 @ b64.T, np.abs(a64) @ np.abs(b64).T
    bad = ~np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[bad & ~np.isnan(ref)], ref[bad & ~np.isnan(ref)])
    rows = [i for i in range(M) if i not in (0, 2, 5)]
    _check(got[rows], ref[rows], mag[rows], K)


# Operands down to fp32's smallest subnormals (2^-149) and up to the overflow of
# the scaled split (2^112, sums of 2^96): every bit of either counts against a
# partner that brings the product back to an ordinary size.
SCALES = [(-102, 100), (-111, 100), (-118, 100), (-126, 100), (-140, 100), (-60, -50), (100, -126),
          (111, -40), (120, -20), (48, 47), (60, 60)]


@pytest.mark.parametrize("trans_b", [0, 1])
@pytest.mark.parametrize("ea,eb", SCALES)
@pytest.mark.parametrize("M,N,K", [(65, 66, 40), (130, 64, 1100)])
def test_operand_scales(dev, rng, M, N, K, ea, eb, trans_b):
    a = (rng.standard_normal((M, K)) * 2.0 ** ea).astype(np.float32)
    b = (rng.standard_normal((N, K) if trans_b else (K, N)) * 2.0 ** eb).astype(np.float32)
    y = dev.create_buffer(M * N * 4)
    _call(dev, "di_gemm", dev.storage(a).handle, dev.storage(b).handle, 0, y.handle, M, N, K,
          trans_b, F32)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    b64 = b64.T if trans_b else b64
    _check(dev.download(y).reshape(M, N), a64 @ b64, np.abs(a64) @ np.abs(b64), K, 2.0 ** -149)


@pytest.mark.parametrize("w16", [False, True])
@pytest.mark.parametrize("ea", [-118, -130, 114])
def test_conv_operand_scales(dev, rng, ea, w16):
    x = (rng.standard_normal((1, 40, 9, 8)) * 2.0 ** ea).astype(np.float32)
    w = (rng.standard_normal((66, 40, 3, 3)) * (1.0 if w16 or ea > 0 else 2.0 ** 90)) \
        .astype(np.float16 if w16 else np.float32)
    y = dev.create_buffer(66 * 9 * 8 * 4)
    _call(dev, "di_conv2d", dev.storage(x).handle, dev.storage(w).handle, 0, 0, y.handle, 1, 40, 66,
          9, 8, 3, 1, 1, 0, F32W16 if w16 else F32, NCHW)
    x64, w64 = (torch.from_numpy(v.astype(np.float64)) for v in (x, w))
    z, mag = (TF.conv2d(u, v, padding=1).numpy() for u, v in ((x64, w64), (x64.abs(), w64.abs())))
    _check(dev.download(y).reshape(z.shape), z, mag, 360, 2.0 ** -149)


@pytest.mark.parametrize("batch,K", [(10000, 512), (5000, 1024), (20000, 1024), (65535, 40)])
def test_long_batches(dev, rng, batch, K):
    """Batches whose splits would pass the grid's 65535 along z."""
    a, b = _mats(rng, (batch, 1, K), (batch, K, 1))
    y = dev.create_buffer(batch * 4)
    _call(dev, "di_matmul", dev.storage(a).handle, dev.storage(b).handle, y.handle, 1, 1, K, batch,
          1, F32)
    a64, b64 = a.astype(np.float64)[:, 0], b.astype(np.float64)[..., 0]
    _check(dev.download(y).reshape(batch), (a64 * b64).sum(1), np.abs(a64 * b64).sum(1), K)


# ---- operands past 31-bit offsets: the bounds-checked fp32 MFMA kernel ----
@pytest.mark.parametrize("w16", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 1, 4200007), (3, 2, 4300000)])
def test_long_rows(dev, rng, M, N, K, w16):
    a, b = _mats(rng, (M, K), (N, K), w16=w16)
    y = dev.create_buffer(M * N * 4)
    _call(dev, "di_gemm", dev.storage(a).handle, dev.storage(b).handle, 0, y.handle, M, N, K, 1,
          F32W16 if w16 else F32)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    _check(dev.download(y).reshape(M, N), a64 @ b64.T, np.abs(a64) @ np.abs(b64).T, K)


@pytest.mark.parametrize("M,N,K", [(2, 16800003, 3), (1, 2 ** 30, 2)])
def test_wide_columns(dev, rng, M, N, K):
    """B [K][N] with rows past 31-bit offsets, the second also past 2^32 threads
    of 64 x 64 tiles: columns from the start, the middle and the end."""
    a = rng.standard_normal((M, K)).astype(np.float32)
    b, y = dev.create_buffer(K * N * 4), dev.create_buffer(M * N * 4)
    dev.fill_normal(b, K * N, 11)
    _call(dev, "di_matmul", dev.storage(a).handle, b.handle, y.handle, M, N, K, 1, 0, F32)
    n, a64 = 3000, a.astype(np.float64)
    for c in (0, N // 2 - 5, N - n):
        cols = np.stack([dev.download(b, np.float32, (n,), (k * N + c) * 4) for k in range(K)])
        got = np.stack([dev.download(y, np.float32, (n,), (m * N + c) * 4) for m in range(M)])
        c64 = cols.astype(np.float64)
        _check(got, a64 @ c64, np.abs(a64) @ np.abs(c64), K)
    b.destroy()
    y.destroy()


def test_large_image_conv(dev, rng):
    """An NCHW image of more than 2^31 bytes: rows of the output at both ends."""
    ci, co, H, W = 70, 3, 2901, 2700
    x, y = dev.create_buffer(ci * H * W * 4), dev.create_buffer(co * H * W * 4)
    dev.fill_normal(x, ci * H * W, 12)
    w = rng.standard_normal((co, ci, 3, 3)).astype(np.float32)
    _call(dev, "di_conv2d", x.handle, dev.storage(w).handle, 0, 0, y.handle, 1, ci, co, H, W, 3, 1, 1,
          0, F32, NCHW)
    w64 = torch.from_numpy(w.astype(np.float64))
    for r0 in (0, H - 4):  # four input rows, of which the outer ones have a padded neighbour
        rows = np.stack([dev.download(x, np.float32, (4, W), ((c * H) + r0) * W * 4)
                         for c in range(ci)]).astype(np.float64)
        t = torch.from_numpy(rows)[None]
        z, mag = (TF.conv2d(u, v, padding=1)[0].numpy() for u, v in ((t, w64), (t.abs(), w64.abs())))
        sl = slice(0, 3) if r0 == 0 else slice(1, 4)
        got = np.stack([dev.download(y, np.float32, (4, W), ((o * H) + r0) * W * 4) for o in range(co)])
        _check(got[:, sl], z[:, sl], mag[:, sl], ci * 9)
    x.destroy()
    y.destroy()


@pytest.mark.parametrize("tile", range(16))
def test_tile_override(dev, rng, monkeypatch, tile):
    """Every row is written whatever tile an override names."""
    M, N, K = 200, 70, 300
    a, b = _mats(rng, (M, K), (N, K))
    y = dev.create_buffer(M * N * 4)
    dev.fill_normal(y, M * N, 3)  # stale output must be overwritten
    monkeypatch.setenv("DI_GEMM_TILE", str(tile))
    for splits in ("1", "3"):
        monkeypatch.setenv("DI_GEMM_SPLITS", splits)
        _call(dev, "di_gemm", dev.storage(a).handle, dev.storage(b).handle, 0, y.handle, M, N, K, 1, F32)
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        _check(dev.download(y).reshape(M, N), a64 @ b64.T, np.abs(a64) @ np.abs(b64).T, K)


@pytest.mark.parametrize("trans_b", [0, 1])
@pytest.mark.parametrize("M,N,K", [(240, 5, 2), (65, 15, 31), (65, 15, 32), (130, 13, 64), (130, 13, 65),
                                   (64, 16, 20), (3, 1, 8)])
def test_narrow(dev, rng, M, N, K, trans_b):
    """Both sides of the line up to which the fp32 MFMA takes narrow products."""
    a, b = _mats(rng, (M, K), (N, K) if trans_b else (K, N))
    c = rng.standard_normal(N).astype(np.float32)
    y = dev.create_buffer(M * N * 4)
    _call(dev, "di_gemm", dev.storage(a).handle, dev.storage(b).handle, dev.storage(c).handle,
          y.handle, M, N, K, trans_b, F32)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    b64 = b64.T if trans_b else b64
    _check(dev.download(y).reshape(M, N), a64 @ b64 + c, np.abs(a64) @ np.abs(b64) + np.abs(c), K)


@pytest.mark.parametrize("N,co,H,W,silu", [(3, 66, 1, 1, 0), (2, 70, 1, 3, SILU), (5, 5, 3, 3, 0),
                                           (2, 130, 5, 5, SILU)])
def test_ragged_images(dev, rng, N, co, H, W, silu):
    """Images of no multiple of four pixels: a stored vector spans one to four."""
    ci = 40
    x = rng.standard_normal((N, ci, H, W)).astype(np.float32)
    w = rng.standard_normal((co, ci, 3, 3)).astype(np.float32)
    b = rng.standard_normal(co).astype(np.float32)
    r = rng.standard_normal((N, co, H, W)).astype(np.float32)
    y = dev.create_buffer(r.size * 4)
    _call(dev, "di_conv2d", dev.storage(x).handle, dev.storage(w).handle, dev.storage(b).handle,
          dev.storage(r).handle, y.handle, N, ci, co, H, W, 3, 1, 1, silu, F32, NCHW)
    t = [torch.from_numpy(v.astype(np.float64)) for v in (x, w, b)]
    z = TF.conv2d(*t, padding=1).numpy()
    mag = TF.conv2d(*(v.abs() for v in t), padding=1).numpy()
    ref = (z / (1 + np.exp(-z)) if silu else z) + r
    _check(dev.download(y).reshape(r.shape), ref, 1.1 * mag + np.abs(r), ci * 9,
           2.0 ** -20 * np.abs(z) if silu else 0.0)
