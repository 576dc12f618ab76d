"""The tiles whose two wave groups alternate (gemm_pingpong_kernel), forced, where the phase tables, the ring and
the out-of-range loads can go wrong: fewer stages than ring slots, odd and even stage counts, K tails, partial tiles,
K splits whose last part is short, batches."""
import numpy as np
import pytest

import mvlm_amd as m
from mvlm_amd import BF16, F16, F32
from test_gpu_parity import check_packed, within

pytestmark = pytest.mark.gpu

TILES = ["256x256s2w8", "256x128s3w8", "192x128s4w8", "128x128s4w8"]


@pytest.fixture(scope="module")
def dev():
    d = m.Device(0)
    yield d
    d.close()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K,splits", [
    (1, 1, 136, 1),          # one row, one column; 3 stages, the last of 8 columns
    (129, 131, 192, 1),      # 3 full stages; rows off the vector grid
    (256, 384, 320, 1),      # 5 stages
    (257, 130, 1032, 1),     # 17 stages, a tail of 8 columns
    (200, 260, 1992, 3),     # 32 stages in 3 splits of 11, 11 and 10
    (70, 129, 520, 2),       # 9 stages: 5 and 4
])
def test_forced(dev, orc, monkeypatch, tile, M, N, K, splits):
    monkeypatch.setenv("MVLM_GEMM_TILE", tile)
    monkeypatch.setenv("MVLM_GEMM_SPLITS", str(splits))
    check_packed(dev, orc, M, N, K, F16, F32, seed=400)
    check_packed(dev, orc, M, N, K, BF16, BF16, seed=401)


@pytest.mark.parametrize("tile", TILES)
def test_batches(dev, orc, monkeypatch, tile):
    """strided batches: each one's product, and nothing outside it (the oracle's own sums bound the error)"""
    monkeypatch.setenv("MVLM_GEMM_TILE", tile)
    H, S, D = 3, 150, 200
    q, k = orc.normal_f16(S * H * D, 0x420), orc.normal_f16(S * H * D, 0x421)
    pad = 64
    C = dev.upload(np.full(H * (S * S + pad), 7.0, np.float32))
    dev.gemm_batched(dev.upload(q), dev.upload(k), C, H, S, S, D, H * D, H * D, S, D, D, S * S + pad)
    got = C.download(np.float32).reshape(H, S * S + pad)
    assert (got[:, S * S:] == 7.0).all()
    for h in range(H):
        a, b = (v.reshape(S, H, D)[:, h, :].copy() for v in (q, k))
        ref = orc.gemm_nk("f16", a, b, S, S, D)
        _, bound = orc.gemm_f64(orc.f16_to_f32(a).astype(np.float64), orc.f16_to_f32(b).astype(np.float64), S, S, D)
        ok, worst = within(got[h, :S * S].reshape(S, S), ref, bound, 1e-3)
        assert ok, (h, worst)
