"""The skinny GEMM over quantized weights (5 to 16 rows of x) where its work is
cut: K of one chunk, of a full one (64 blocks), of two and more chunks that
start at even and odd blocks, with fewer blocks than waves; row counts that are
no multiple of 16; one row group per workgroup, more than a batch of four, and
more than one round of workgroups; each epilogue operand; and without
workspace.  Each on the kernel that keeps X, on the one that walks K, and on the
one that the launch's size picks."""
import numpy as np
import pytest

import mvlm_amd as m
from tests.test_gpu_parity import make_quant, within

pytestmark = pytest.mark.gpu

F32, Q8, Q4 = m.F32, m.Q8_0, m.Q4_0


@pytest.fixture(autouse=True, params=["x", "k", None])
def form(request, monkeypatch):
    if request.param:
        monkeypatch.setenv("MVLM_SKINNY_FORM", request.param)
    return request.param


def reference(orc, qt, X, blocks, M, N, K):
    kind, deq = ("q8_0", orc.dequant_q8_0) if qt == Q8 else ("q4_0", orc.dequant_q4_0)
    ref = orc.gemm_nk(kind, X, blocks, M, N, K).reshape(M, N)
    _, S = orc.gemm_f64(X.astype(np.float64).reshape(M, K), deq(blocks).astype(np.float64).reshape(N, K), M, N, K)
    return ref, S.reshape(M, N)


def run(dev, orc, qt, M, N, K, seed=611):
    X, blocks = orc.normal_f32(M * K, seed), make_quant(orc, qt, N, K, seed + 1)
    dY = dev.upload(np.full(M * N, np.nan, np.float32))
    dev.gemm_quant(dev.upload(X), dev.pack(blocks, qt, N, K), dY, M, N, K)
    got = dY.download(np.float32).reshape(M, N)
    ref, S = reference(orc, qt, X, blocks, M, N, K)
    ok, worst = within(got, ref, S, 1e-5)
    assert ok, worst
    return got


@pytest.mark.parametrize("qt", [Q8, Q4])
@pytest.mark.parametrize("M,N,K", [(5, 1, 32), (16, 16, 7 * 32), (9, 47, 33 * 32), (8, 100, 2048), (16, 33, 65 * 32),
                                   (7, 50, 130 * 32), (13, 64, 8192), (16, 21, 191 * 32), (6, 20485, 96),
                                   (16, 57400, 64), (10, 57361, 32)])
def test_cuts(dev, orc, qt, M, N, K):
    run(dev, orc, qt, M, N, K)


@pytest.mark.parametrize("qt", [Q8, Q4])
@pytest.mark.parametrize("M,N,K", [(16, 37, 65 * 32), (5, 4200, 130 * 32), (12, 300, 8192)])
def test_without_workspace(dev, orc, monkeypatch, qt, M, N, K):
    """on the kernel that needs none"""
    with_ws = run(dev, orc, qt, M, N, K)
    monkeypatch.setenv("MVLM_SKINNY_WORKSPACE", "0")
    # one kernel's chunk sums against the other's fma chains
    assert np.allclose(run(dev, orc, qt, M, N, K), with_ws, rtol=0, atol=1e-5 * np.abs(with_ws).max())


@pytest.mark.parametrize("qt", [Q8, Q4])
@pytest.mark.parametrize("M", [5, 9, 16])
@pytest.mark.parametrize("ep", ["bias", "mul", "residual", "all"])
def test_epilogue_operands(dev, orc, qt, M, ep):
    """three problems in one launch: seven row groups per workgroup, a short
    one, and one of two chunks (its epilogue is the second launch's)"""
    shapes = [(16 * 1600 + 5, 64), (40, 96), (50, 70 * 32)]
    descs, eps, want = [], [], []
    for i, (N, K) in enumerate(shapes):
        X, blocks = orc.normal_f32(M * K, 631 + i), make_quant(orc, qt, N, K, 641 + i)
        ref, S = reference(orc, qt, X, blocks, M, N, K)
        bias, mul, res = orc.normal_f32(N, 651), orc.normal_f32(M * N, 652), orc.normal_f32(M * N, 653)
        out, size, e = ref.astype(np.float64), S, {}
        if ep in ("bias", "all"):
            e["bias"], out, size = dev.upload(bias), out + bias, size + np.abs(bias)
        if ep in ("mul", "all"):
            mm = mul.reshape(M, N)
            e["mul"], out, size = dev.upload(mul), out * mm, size * np.abs(mm)
        if ep in ("residual", "all"):
            rr = res.reshape(M, N)
            e["residual"], out, size = dev.upload(res), out + rr, size + np.abs(rr)
        y = dev.upload(np.full(M * N, np.nan, np.float32))
        descs.append((dev.upload(X), F32, dev.pack(blocks, qt, N, K), y, F32))
        eps.append(e)
        want.append((y, out, size))
    dev.gemm_quant_grouped(M, descs, epilogues=eps)
    for (y, out, size), (N, K) in zip(want, shapes):
        ok, worst = within(y.download(np.float32).reshape(M, N), out, size, 1e-5)
        assert ok, (N, K, worst)


# blocks of K that leave the last or most of the eight waves of a workgroup
# without work, and enough row groups per workgroup (10 and more for Q8_0, 12
# for Q4_0) that epilogue operands are requested again while codes still follow
@pytest.mark.parametrize("qt,N,K", [(Q8, 40005, 28 * 32), (Q8, 40005, 9 * 32), (Q8, 57301, 2 * 32),
                                    (Q4, 50005, 28 * 32), (Q4, 50005, 18 * 32), (Q4, 57301, 2 * 32)])
@pytest.mark.parametrize("M", [5, 9, 16])
def test_epilogue_of_waves_without_blocks(dev, orc, qt, N, K, M):
    X, blocks = orc.normal_f32(M * K, 671), make_quant(orc, qt, N, K, 672)
    ref, S = reference(orc, qt, X, blocks, M, N, K)
    bias, mul, res = orc.normal_f32(N, 673), orc.normal_f32(M * N, 674).reshape(M, N), orc.normal_f32(M * N, 675).reshape(M, N)
    y = dev.upload(np.full(M * N, np.nan, np.float32))
    dev.gemm_quant_grouped(M, [(dev.upload(X), F32, dev.pack(blocks, qt, N, K), y, F32)],
                           epilogues=[{"bias": dev.upload(bias), "mul": dev.upload(mul), "residual": dev.upload(res)}])
    want = (ref.astype(np.float64) + bias) * mul + res
    ok, worst = within(y.download(np.float32).reshape(M, N), want, (S + np.abs(bias)) * np.abs(mul) + np.abs(res), 1e-5)
    assert ok, worst


@pytest.mark.parametrize("qt", [Q8, Q4])
def test_not_a_number_stays_in_its_row(dev, orc, qt):
    M, N, K = 9, 70, 300 * 32
    X, blocks = orc.normal_f32(M * K, 661).reshape(M, K), make_quant(orc, qt, N, K, 662)
    X[3, 17], X[6, 9000], X[8, 40] = np.nan, np.inf, -np.inf
    dY = dev.alloc(M * N * 4)
    dev.gemm_quant(dev.upload(X), dev.pack(blocks, qt, N, K), dY, M, N, K)
    bad = ~np.isfinite(dY.download(np.float32).reshape(M, N))
    assert bad[[3, 6, 8]].all() and not bad[[0, 1, 2, 4, 5, 7]].any()


@pytest.mark.parametrize("form", [None], indirect=True)
@pytest.mark.parametrize("qt", [Q8, Q4])
@pytest.mark.parametrize("N,K", [(2048, 768), (2048, 2048), (512, 8192)])
def test_walking_k_is_no_less_exact(dev, orc, monkeypatch, form, qt, N, K):
    """2-norm of the error against 64 bits: the kernel that walks K within 1.05
    of the one that keeps X (with one chain per wave and -8 x applied to a
    block's sum it was 1.1 to 1.4 of it)"""
    M = 16
    X, blocks = orc.normal_f32(M * K, 681), make_quant(orc, qt, N, K, 682)
    deq = orc.dequant_q8_0 if qt == Q8 else orc.dequant_q4_0
    want = X.astype(np.float64).reshape(M, K) @ deq(blocks).astype(np.float64).reshape(N, K).T
    dX, W, err = dev.upload(X), dev.pack(blocks, qt, N, K), {}
    for kernel in "xk":
        monkeypatch.setenv("MVLM_SKINNY_FORM", kernel)
        dY = dev.alloc(M * N * 4)
        dev.gemm_quant(dX, W, dY, M, N, K)
        err[kernel] = np.linalg.norm(dY.download(np.float32).reshape(M, N) - want) / np.linalg.norm(want)
    assert err["k"] <= 1.05 * err["x"], err
