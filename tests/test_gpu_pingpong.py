"""The GEMM tiles whose two wave groups alternate (gemm_pingpong_kernel), forced, where the phase tables, the ring and
the out-of-range loads can go wrong: fewer stages than ring slots, odd and even stage counts, K tails, partial tiles,
K splits whose last part is short, batches; and the store pass with its epilogue."""
import numpy as np
import pytest

import mvlm_amd as m
from mvlm_amd import BF16, F16, F32, native
from test_gpu_epilogue import check, from_storage, make_operands, to_storage
from test_gpu_parity import check_packed, gen, widen, within

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


@pytest.mark.parametrize("tile", TILES + ["64x64s4w4", "64x64s2w4k128"])
@pytest.mark.parametrize("dt,offset,splits,act,names", [
    (F32, 0, 1, native.ACT_GELU_TANH, ("bias", "mul", "residual")),
    (F16, 0, 1, native.ACT_SILU, ("bias", "residual")),
    (BF16, 0, 1, native.ACT_NONE, ("bias", "mul")),
    (F16, 1, 1, native.ACT_GELU_TANH, ("bias", "residual")),     # operands off the 8-byte grid: read one by one
    (F16, 0, 2, native.ACT_GELU_TANH, ("bias", "mul", "residual")),   # applied by the split-K reduction
])
def test_epilogue(dev, orc, monkeypatch, tile, dt, offset, splits, act, names):
    """operands read four columns at a time for groups of tiles: rows and columns that end inside a tile"""
    monkeypatch.setenv("MVLM_GEMM_TILE", tile)
    monkeypatch.setenv("MVLM_GEMM_SPLITS", str(splits))
    M, N, K, ab = 201, 332, 520, BF16 if dt == BF16 else F16
    A, Wt = gen(orc, ab, M * K, 0x430), gen(orc, ab, N * K, 0x431, 0.05)
    _, vals = make_operands(dev, orc, M, N, dt, 0x432, *(n in names for n in ("bias", "mul", "residual")))
    es = 4 if dt == F32 else 2
    ops = {}
    for n in names:
        raw = to_storage(orc, vals[n].astype(np.float32), dt)[0]
        buf = dev.upload(np.concatenate([np.zeros(offset, raw.dtype), raw]))
        ops[n] = buf.view(offset * es, raw.size * es) if offset else buf
    C = dev.alloc(M * N * es)
    dev.gemm_packed_ex(dev.upload(A), ab, dev.pack(Wt, ab, N, K), C, dt, M, N, K, act=act, **ops)
    got = from_storage(orc, C.download(np.float32 if dt == F32 else np.uint16, M * N), dt).reshape(M, N)
    Y64, S = orc.gemm_f64(widen(orc, A, ab).reshape(M, K), widen(orc, Wt, ab).reshape(N, K), M, N, K)
    check(orc, got, Y64, S, vals, act, dt, 1e-4)


@pytest.mark.parametrize("tile", ["64x64s4w4", "64x64s2w4k128"])
@pytest.mark.parametrize("K", [2112, 2239, 4096])
def test_one_accumulator_tiles_sum_in_four_chains(dev, orc, monkeypatch, tile, K):
    """K without a split, error against 64 bits.  Normal factors: the roundings of a chain of K / 16 sums add up as a
    random walk, so relative to the result they grow with the square root of its length.  K = 2112: 2.75e-7 with one
    chain, half of that (1.34e-7 measured) with four a quarter as long.  The limit is sqrt(2) from both."""
    monkeypatch.setenv("MVLM_GEMM_TILE", tile)
    monkeypatch.setenv("MVLM_GEMM_SPLITS", "1")
    M, N = 121, 200
    A, Wt = gen(orc, BF16, M * K, 0x440), gen(orc, BF16, N * K, 0x441)
    C = dev.alloc(M * N * 4)
    dev.gemm_packed(dev.upload(A), BF16, dev.pack(Wt, BF16, N, K), C, F32, M, N, K)
    exact, _ = orc.gemm_f64(widen(orc, A, BF16).reshape(M, K), widen(orc, Wt, BF16).reshape(N, K), M, N, K)
    got = C.download(np.float32).reshape(M, N)
    err = np.linalg.norm(got - exact) / np.linalg.norm(exact)
    assert err < 1.94e-7 * (K / 2112) ** 0.5, err


def test_gelu_extremes(dev, orc):
    """the values that the tanh form gives: inf and large x pass, large -x is zero, -inf (0 times inf) is NaN"""
    x = np.array([np.inf, 65504.0, 12.0, 0.0, -12.0, -65504.0, -np.inf, np.nan], np.float16)
    A = np.zeros((x.size, 8), np.float16)
    A[:, 0] = x
    Wt = np.zeros((4, 8), np.float16)
    Wt[:, 0] = 1.0
    C = dev.alloc(x.size * 4 * 4)
    dev.gemm_packed_ex(dev.upload(A.view(np.uint16)), F16, dev.pack(Wt.view(np.uint16), F16, 4, 8), C, F32, x.size, 4, 8,
                       act=native.ACT_GELU_TANH)
    got = C.download(np.float32).reshape(x.size, 4)[:, 0]
    assert np.array_equal(got[:6], np.float32([np.inf, 65504.0, 12.0, 0.0, 0.0, 0.0])), got
    assert np.isnan(got[6:]).all(), got
