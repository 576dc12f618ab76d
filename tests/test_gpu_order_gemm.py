"""mvlm_gemm_naive / mvlm_gemm_tiled at the edges of the matrix-core kernel's
tiles (32, 64 and 128 outputs on a side; slices of 128, 64 and 32 k) and on
operands that do not start, or whose rows do not start, 16-byte aligned:
bit-exact against the oracle's fp32 fma chain."""
import numpy as np
import pytest

import mvlm_amd as m

pytestmark = pytest.mark.gpu

# 32-wide tiles: up to a few hundred outputs on a side; 64: about 16 x 16
# tiles; 128: more than 256 tiles of 64 that round up to 256 of 128
SHAPES = [(1500, 1500, 8), (2045, 2043, 1), (128, 33000, 17), (31, 33, 127), (32, 64, 128), (33, 40, 129), (16, 256, 256), (1000, 1001, 65), (1024, 960, 64),
          (1985, 2047, 33), (2048, 1992, 40), (1921, 2048, 31)]


def expect(orc, A, B, M, N, K):
    return orc.f32_to_f16(orc.gemm_nk("f16", A, B.reshape(K, N).T.copy(), M, N, K)).ravel()


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_tile_edges(dev, orc, M, N, K):
    A, B = orc.normal_f16(M * K, 301), orc.normal_f16(K * N, 302, 0.02)
    dC = dev.alloc(M * N * 2)
    dev.gemm_tiled(dev.upload(A), dev.upload(B), dC, M, N, K)
    got = dC.download(np.uint16)
    assert np.array_equal(got, expect(orc, A, B, M, N, K))


@pytest.mark.parametrize("oa,ob,oc", [(2, 0, 0), (0, 2, 2), (8, 6, 4)])
@pytest.mark.parametrize("M,N,K", [(40, 72, 136), (1000, 1000, 64)])
def test_views_off_the_vector_grid(dev, orc, M, N, K, oa, ob, oc):
    """Rows that are whole 16-byte vectors in buffers that start off the grid."""
    A, B = orc.normal_f16(M * K, 303), orc.normal_f16(K * N, 304, 0.02)
    a, b, c = dev.alloc(M * K * 2 + oa), dev.alloc(K * N * 2 + ob), dev.alloc(M * N * 2 + oc + 16).zero()
    a.upload(A, oa)
    b.upload(B, ob)
    dev.gemm_naive(a.view(oa, M * K * 2), b.view(ob, K * N * 2), c.view(oc, M * N * 2), M, N, K)
    got = c.download(np.uint16)
    assert np.array_equal(got[oc // 2:oc // 2 + M * N], expect(orc, A, B, M, N, K))
    assert not got[:oc // 2].any() and not got[oc // 2 + M * N:].any()


def test_every_fp16_class(dev, orc):
    """Random fp16 bit patterns (subnormals, infinities and NaN among them): the
    same class everywhere, and the same bits wherever the result is a number."""
    M, N, K = 70, 90, 50
    rng = np.random.default_rng(5)
    A = rng.integers(0, 1 << 16, M * K).astype(np.uint16)
    B = rng.integers(0, 1 << 16, K * N).astype(np.uint16)
    # special values in a few rows and columns only, so that most outputs are numbers
    keep = np.ones((M, K), bool)
    keep[::7] = False
    A = np.where(keep & ((A & 0x7C00).reshape(M, K) >= 0x5000), A.reshape(M, K) & 0x8FFF, A.reshape(M, K)).ravel().astype(np.uint16)
    B = np.where((B & 0x7C00) >= 0x5000, B & 0x8FFF, B).astype(np.uint16)
    want = expect(orc, A, B, M, N, K)
    dC = dev.alloc(M * N * 2)
    dev.gemm_tiled(dev.upload(A), dev.upload(B), dC, M, N, K)
    got = dC.download(np.uint16)
    nan = lambda v: (v & 0x7FFF) > 0x7C00
    assert np.array_equal(nan(got), nan(want)) and nan(want).any() and not nan(want).all()
    assert np.array_equal(got[~nan(want)], want[~nan(want)])
