"""fp16 contractions whose B operand is past the L2: the tiles run down blocks
of 8 tile rows, and every output element is written once for whole blocks,
ragged last blocks and a single row, against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 8 * 128, 8 * 128 + 1, 11 * 64 + 5])
@pytest.mark.parametrize("tile,splits", [(0, 1), (3, 1), (8, 1), (11, 1), (14, 1), (6, 2)])
def test_linear_blocked_tile_order(dev, rng, monkeypatch, M, tile, splits):
    import drawinstant
    N, K = 2 * 2184, 512 * splits  # B past 4 MiB per split, N off every tile
    x = rng.standard_normal((M, K)).astype(np.float16)
    w = (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float16)
    y = dev.create_buffer(M * N * 2)
    dev.fill_normal(y, M * N, 3, dtype=drawinstant.F16)  # stale output must be overwritten
    monkeypatch.setenv("DI_GEMM_TILE", str(tile))
    monkeypatch.setenv("DI_GEMM_SPLITS", str(splits))
    drawinstant.call("di_linear", dev.ctx, dev.storage(x).handle, dev.storage(w).handle, 0, 0,
                     y.handle, M, N, K, 0, drawinstant.F16)
    got = dev.download(y, np.float16).reshape(M, N).astype(np.float64)
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    # fp32 sums of K products: K roundings of 2^-24 of sum |x w| <= |x| |w|,
    # then one rounding to fp16 (2^-11 relative, 2^-25 below the normal range)
    mag = np.linalg.norm(x.astype(np.float64), axis=1)[:, None] * \
        np.linalg.norm(w.astype(np.float64), axis=1)[None, :]
    bound = K * 2.0 ** -24 * mag + np.abs(ref) * 2.0 ** -11 + 2.0 ** -24
    assert (np.abs(got - ref) <= bound).all(), np.abs(got - ref).max()
