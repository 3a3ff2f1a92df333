"""GPU: the strided executor ops (transpose, slice, broadcasts) over axis
orders, ragged and vector-sized axes and both types, against numpy bit for bit
(one rounded operation per element); row softmax at the edges of its register
forms against float64."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = {np.float32: 0, np.float16: 1}


def _call(dev, fn, *a):
    import drawinstant
    drawinstant.call(fn, dev.ctx, *a)


def _u32(v):
    import ctypes
    return (ctypes.c_uint32 * 4)(*(list(v) + [0] * (4 - len(v))))


def _strides(shape):
    s = [1] * len(shape)
    for i in range(len(shape) - 2, -1, -1):
        s[i] = s[i + 1] * shape[i + 1]
    return s


@pytest.mark.parametrize("dt", [np.float32, np.float16])
@pytest.mark.parametrize("shape", [(1,), (260,), (5, 7), (64, 132), (65, 63), (1, 70, 4, 64),
                                   (2, 33, 5, 12), (3, 1, 66, 20), (2, 3, 17, 65), (4, 16, 16, 8)])
def test_transpose(dev, rng, shape, dt):
    x = rng.standard_normal(shape).astype(dt)
    bx, y = dev.storage(x), dev.create_buffer(max(x.nbytes, 4))
    r = len(shape)
    for perm in itertools.permutations(range(r)):
        _call(dev, "di_transpose", bx.handle, y.handle, r, _u32([shape[p] for p in perm]),
              _u32(_strides(shape)), _u32(perm), x.size, DT[dt])
        ref = np.ascontiguousarray(x.transpose(perm))
        assert np.array_equal(dev.download(y, dt, ref.shape), ref), perm


@pytest.mark.parametrize("dt", [np.float32, np.float16])
@pytest.mark.parametrize("shape,start,out", [((20,), (4,), (16,)), ((20,), (3,), (16,)),
                                             ((6, 40), (1, 8), (4, 32)), ((6, 41), (1, 8), (4, 32)),
                                             ((2, 9, 5, 64), (0, 2, 1, 0), (2, 7, 3, 64)),
                                             ((3, 4, 5, 6), (1, 1, 1, 1), (2, 3, 4, 5))])
def test_slice(dev, rng, shape, start, out, dt):
    x = rng.standard_normal(shape).astype(dt)
    y = dev.create_buffer(x.nbytes)
    n = int(np.prod(out))
    _call(dev, "di_slice", dev.storage(x).handle, y.handle, len(shape), _u32(out),
          _u32(_strides(shape)), _u32(start), n, DT[dt])
    ref = x[tuple(slice(s, s + o) for s, o in zip(start, out))]
    assert np.array_equal(dev.download(y, dt, (y.size // x.itemsize,))[:n].reshape(out), ref)


def _bstr(shape, dims):
    st = _strides(shape)
    return [0 if s == 1 and d != 1 else t for s, d, t in zip(shape, dims, st)]


@pytest.mark.parametrize("dt", [np.float32, np.float16])
@pytest.mark.parametrize("a,b", [((3, 64, 64), (1, 1, 1)), ((2, 8, 5, 12), (1, 8, 1, 1)),
                                 ((2, 8, 5, 7), (1, 8, 1, 1)), ((6, 1, 20), (1, 9, 20)),
                                 ((4, 1), (4, 128)), ((1, 130, 64), (1, 1, 64)), ((5,), (5,))])
def test_broadcasts(dev, rng, a, b, dt):
    dims = np.broadcast_shapes(a, b)
    x, w, z = (rng.standard_normal(s).astype(dt) for s in (a, b, b))
    bx, bw, bz = dev.storage(x), dev.storage(w), dev.storage(z)
    n = int(np.prod(dims))
    y = dev.create_buffer(n * 4)
    args = (len(dims), _u32(dims), _u32(_bstr(a, dims)), _u32(_bstr(b, dims)), n, DT[dt])
    f = [v.astype(np.float32) for v in (x, w, z)]
    for op, ref in ((0, f[0] + f[1]), (1, f[0] - f[1]), (2, f[0] * f[1])):
        _call(dev, "di_binary_bcast", op, bx.handle, bw.handle, y.handle, *args)
        got = dev.download(y, dt, (y.size // x.itemsize,))[:n].reshape(dims)
        assert np.array_equal(got, ref.astype(dt)), op
    _call(dev, "di_affine_bcast", bx.handle, bw.handle, bz.handle, y.handle, *args)
    got = dev.download(y, dt, (y.size // x.itemsize,))[:n].reshape(dims).astype(np.float64)
    ref = f[0].astype(np.float64) * f[1] + f[2]
    eps = 2.0 ** -10 if dt == np.float16 else 2.0 ** -23
    mag = np.abs(f[0].astype(np.float64) * f[1]) + np.abs(f[2])
    assert (np.abs(got - ref) <= eps * mag + 1e-7).all()  # at most two roundings


@pytest.mark.parametrize("dt", [np.float32, np.float16])
@pytest.mark.parametrize("inner", [1, 3, 64, 77, 128, 256, 260, 1000, 1023, 2048, 2304, 3072, 3076,
                                   4096, 4100, 4104, 5120, 5128, 8192, 8196, 9216, 16384, 16392])
def test_softmax(dev, rng, inner, dt):
    rows = 7
    x = (rng.standard_normal((rows, inner)) * 4).astype(dt)
    if inner > 2:
        x[1, inner // 2] = -np.inf
        x[2, 0] = np.inf
        x[3, 1] = np.nan
    x[4] = -np.inf
    b = dev.storage(x)
    _call(dev, "di_softmax", b.handle, b.handle, inner, rows, DT[dt])  # in place
    got = dev.download(b, dt, x.shape).astype(np.float64)
    x64 = x.astype(np.float64)
    with np.errstate(invalid="ignore"):
        e = np.exp(x64 - x64.max(1, keepdims=True))
        ref = e / e.sum(1, keepdims=True)
    whole = [0, 1, 5, 6]
    # exp(d) as exp2(d log2 e): d, log2 e and their product are each rounded,
    # 3 |d| 2^-24 relative in all; 16 more roundings for the exponential, the
    # sum, its reciprocal and the product
    with np.errstate(invalid="ignore"):
        d = np.abs(x64 - x64.max(1, keepdims=True))[whole]
    eps = (3 * np.minimum(d, 110.0) + 16) * 2.0 ** -24 + (2.0 ** -11 if dt == np.float16 else 0.0)
    err = np.abs(got[whole] - ref[whole])
    assert (err <= eps * ref[whole] + (2.0 ** -25 if dt == np.float16 else 1e-37)).all()
    assert np.isnan(got[4]).all()
    if inner > 2:
        assert np.isnan(got[2, 0]) and np.isnan(got[3]).all()


@pytest.fixture
def large():
    """A device of its own: buffers of tens of GiB go back with it."""
    import drawinstant
    d = drawinstant.Device(0)
    yield d
    d.sync()
    d.destroy()


def test_softmax_more_rows_than_workgroups(large):
    """Rows that a workgroup each would take past 2^32 threads (69 GB)."""
    rows, inner = (1 << 24) + 3, 2049
    x = large.create_buffer(rows * inner * 2)
    large.fill_normal(x, rows * inner, 5, dtype=1)
    at = [0, 77, rows // 2, (1 << 24) - 1, 1 << 24, rows - 1]
    src = [large.download(x, np.float16, (inner,), r * inner * 2).astype(np.float64) for r in at]
    _call(large, "di_softmax", x.handle, x.handle, inner, rows, 1)
    for r, v in zip(at, src):
        got = large.download(x, np.float16, (inner,), r * inner * 2).astype(np.float64)
        e = np.exp(v - v.max())
        # fp32 arithmetic, one rounding to fp16 (2^-11 relative, 2^-25 below the normals)
        assert (np.abs(got - e / e.sum()) <= 1.1 * 2.0 ** -11 * e / e.sum() + 2.0 ** -25).all(), r


def test_transpose_longer_than_grid(large):
    """An axis of 2^30 values: its 64 x 64 tiles would take 2^32 threads (34 GB)."""
    n, r = 1 << 30, 16
    x, y = large.create_buffer(n * r * 2), large.create_buffer(n * r * 2)
    large.fill_normal(x, n * r, 6, dtype=1)
    _call(large, "di_transpose", x.handle, y.handle, 2, _u32([n, r]), _u32([n, 1]), _u32([1, 0]),
          n * r, 1)
    w = 5000
    for c in (0, n // 2 - 7, n - w):
        ref = np.stack([large.download(x, np.float16, (w,), (i * n + c) * 2) for i in range(r)], 1)
        assert np.array_equal(large.download(y, np.float16, (w, r), c * r * 2), ref)
