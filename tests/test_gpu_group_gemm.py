"""The prefill GEMMs, of the formats whose group scales fold into int8 weights (mmg.hip) and of those scaled
per 32 weights (mmb.hip), at the edges of their tiles, against the products in float64 from the oracle's decoders and quantizer."""
from __future__ import annotations

import numpy as np
import pytest

from hk_amd import formats as F
from hk_amd import synth
from hk_amd.engine import ACCUMULATE, SILU_MUL, STORE
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch

    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    return torch


@pytest.fixture(scope="module")
def eng(torch_cuda):
    from hk_amd import Engine

    e = Engine(0)
    e.set_stream(torch_cuda.cuda.current_stream().cuda_stream)
    yield e
    e.close()


def products64(t, raw, m, k, x):
    """(y, a bound on the f32 summation's error) of W times the quantized x, in float64: the exact
    integers' scaled sums add k / 32 (k / 256) terms and scale each with at most 3 roundings, so they are
    within (terms + 4) * 2^-23 of the sum of the terms' magnitudes."""
    w = np.stack([O.dequantize(t, raw[r], k) for r in range(m)]).astype(np.float64)
    kind = F.ACT_KIND[t]
    el = 32 if kind == F.ACT_A8 else 256
    a = np.empty(x.shape, np.float64)
    for i, row in enumerate(x):
        blk = (O.quantize_a8 if kind == F.ACT_A8 else O.quantize_q8k)(row).view(np.uint8).reshape(k // el, -1)
        d = blk[:, :4].copy().view(np.float32).astype(np.float64)
        qs = blk[:, 8:8 + el] if kind == F.ACT_A8 else blk[:, 4:4 + el]
        a[i] = (d * qs.copy().view(np.int8)).reshape(-1)
    return a @ w.T, (k // el + 4) * 2.0 ** -23 * (np.abs(a) @ np.abs(w).T)


# (rows, K, tokens): each tile of the dispatch (by the rounds its grid takes), with whole and ragged
# last rows and tokens, K of one super-block, and K slices that end at different super-blocks.
SHAPES = [(32, 256, 9), (33, 256, 41), (70, 1280, 33), (96, 2304, 64), (1000, 768, 130), (4100, 1024, 65),
          (8200, 512, 257), (14340, 256, 511), (8200, 512, 700), (8200, 768, 900)]


def check_gemm(eng, torch, t, m, k, n, mode, raw):
    m -= m % 2 if mode == SILU_MUL else 0
    x = synth.activations_np(n, k, seed=9101 + n, outliers=0.01)
    want, bound = products64(t, raw, m, k, x)
    bias = None if mode == SILU_MUL else np.linspace(-1, 1, m).astype(np.float32)
    w = eng.upload(raw, t, m, k)
    xq = torch.empty(eng.act_bytes(n, k), dtype=torch.uint8, device="cuda")
    eng.qact(torch.from_numpy(x).cuda(), n, k, F.ACT_KIND[t], xq)
    y0 = synth.activations_np(n, m // 2 if mode == SILU_MUL else m, seed=9102)
    y = torch.from_numpy(y0.copy()).cuda()
    eng.gemm(w, xq, y, n, bias=None if bias is None else torch.from_numpy(bias).cuda(), mode=mode)
    got = y.cpu().numpy().astype(np.float64)
    eng.free(w)
    if mode == SILU_MUL:
        g, u = want[:, 0::2], want[:, 1::2]
        sig = 1.0 / (1.0 + np.exp(-g))
        # d silu(g) u = (sig + g sig (1 - sig)) u dg + silu(g) du, and the f32 silu itself.
        slope = np.abs(sig * (1.0 + g * (1.0 - sig)))
        bound = slope * np.abs(u) * bound[:, 0::2] + np.abs(g * sig) * bound[:, 1::2] + 2.0 ** -20 * np.abs(g * sig * u)
        want = g * sig * u
    else:
        want = want + bias
        if mode == ACCUMULATE:
            want = want + y0
        bound = bound + 2.0 ** -22 * (np.abs(want) + np.abs(y0) + 1.0)
    assert np.all(np.abs(got - want) <= bound + 1e-30)


@pytest.mark.parametrize("t", [F.Q6_K, F.Q5_K, F.Q4_K, F.Q3_K, F.Q2_K])
@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("mode", [STORE, ACCUMULATE, SILU_MUL])
def test_group_gemm(eng, torch_cuda, t, m, k, n, mode):
    m -= m % 2 if mode == SILU_MUL else 0
    check_gemm(eng, torch_cuda, t, m, k, n, mode, synth.weights_np(t, m, k, seed=9100 + t + m))


@pytest.mark.parametrize("t", [F.Q8_0, F.IQ4_NL, F.MXFP4, F.Q4_0, F.Q4_1, F.Q5_0, F.Q5_1, F.IQ4_XS])
@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("mode", [STORE, ACCUMULATE, SILU_MUL])
def test_block_gemm(eng, torch_cuda, t, m, k, n, mode):
    """The GEMM of the formats scaled per 32 weights."""
    m -= m % 2 if mode == SILU_MUL else 0
    check_gemm(eng, torch_cuda, t, m, k, n, mode, synth.weights_np(t, m, k, seed=9300 + t + m))


@pytest.mark.parametrize("t", [F.Q8_0, F.IQ4_NL, F.Q4_0])
@pytest.mark.parametrize("m,k,n", [(1, 32, 9), (45, 96, 40), (33, 288, 12), (1000, 1824, 33), (4100, 544, 130),
                                   (8200, 288, 257), (8200, 800, 700), (5000, 480, 430)])
@pytest.mark.parametrize("mode", [STORE, ACCUMULATE])
def test_block_gemm_k_tails(eng, torch_cuda, t, m, k, n, mode):
    """K that is not a multiple of 256: a last step of one to seven blocks, alone or after whole steps,
    in one K slice or several."""
    check_gemm(eng, torch_cuda, t, m, k, n, mode, synth.weights_np(t, m, k, seed=9400 + t + m))


@pytest.mark.parametrize("m,k,n", [(70, 512, 40), (8200, 256, 300)])
def test_block_gemm_large_scales(eng, torch_cuda, m, k, n):
    """Scales of 2^100 and more: MXFP4 exponents up to 2^120, and infinite Q8_0 scales, whose products are
    infinite with the sign of the block's integer sum."""
    torch = torch_cuda
    raw = synth.weights_np(F.MXFP4, m, k, seed=9500 + m)
    blocks = raw.reshape(-1, 17)
    blocks[::29, 0] = 248
    blocks[3::31, 0] = 228
    x = synth.activations_np(n, k, seed=9501 + n) * np.float32(2.0 ** -20)
    xq = torch.empty(eng.act_bytes(n, k), dtype=torch.uint8, device="cuda")
    y = torch.empty((n, m), device="cuda")
    eng.qact(torch.from_numpy(x).cuda(), n, k, F.ACT_A8, xq)
    want, bound = products64(F.MXFP4, raw, m, k, x)
    w = eng.upload(raw, F.MXFP4, m, k)
    eng.gemm(w, xq, y, n)
    got = y.cpu().numpy().astype(np.float64)
    eng.free(w)
    assert np.all(np.abs(got - want) <= bound + 1e-30)

    raw = synth.weights_np(F.Q8_0, m, k, seed=9502 + m)
    rows = np.arange(3, m, 37)
    want, bound = products64(F.Q8_0, raw, m, k, x)
    a8 = np.stack([O.quantize_a8(row).view(np.uint8).reshape(k // 32, -1)[1, 8:40].copy().view(np.int8) for row in x])
    q = raw.reshape(m, k // 32, 34)[rows, 1, 2:].copy().view(np.int8)
    sums = a8.astype(np.int64) @ q.astype(np.int64).T
    want[:, rows] = np.where(sums == 0, np.nan, np.copysign(np.inf, sums))
    raw.reshape(m, k // 32, 34)[rows, 1, :2] = np.array([0x00, 0x7C], np.uint8)
    w = eng.upload(raw, F.Q8_0, m, k)
    eng.gemm(w, xq, y, n)
    got = y.cpu().numpy().astype(np.float64)
    eng.free(w)
    hit = np.zeros(m, bool)
    hit[rows] = True
    assert np.array_equal(got[:, hit], want[:, hit], equal_nan=True)
    assert np.all(np.abs(got[:, ~hit] - want[:, ~hit]) <= bound[:, ~hit] + 1e-30)


@pytest.mark.parametrize("n", [33, 70, 300])
@pytest.mark.parametrize("m,k", [(40, 256), (300, 2048), (8200, 256)])
def test_mxfp4_gemm(eng, torch_cuda, m, k, n):
    """MXFP4's products from 9 tokens: the 32-weight GEMM on a power-of-two scale plane, the smallest
    and largest exponents among them."""
    torch = torch_cuda
    raw = synth.weights_np(F.MXFP4, m, k, seed=9200 + m)
    raw.reshape(-1, 17)[::37, 0] = 0
    raw.reshape(-1, 17)[5::41, 0] = 1
    raw.reshape(-1, 17)[7::43, 0] = 140
    x = synth.activations_np(n, k, seed=9201 + n)
    want, bound = products64(F.MXFP4, raw, m, k, x)
    w = eng.upload(raw, F.MXFP4, m, k)
    xq = torch.empty(eng.act_bytes(n, k), dtype=torch.uint8, device="cuda")
    eng.qact(torch.from_numpy(x).cuda(), n, k, F.ACT_A8, xq)
    y = torch.full((n, m), float("nan"), device="cuda")
    eng.mm(w, xq, y, n)
    assert np.all(np.abs(y.cpu().numpy() - want) <= bound + 1e-30)
    eng.free(w)
