"""skv_linear over more than 64 rows (csrc/gemm.hip) at the edges of its tiles
and of its split products, against float64."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import banner

pytestmark = pytest.mark.gpu


def _linear(x, w, bias=None, res=None, ln=None, ws=True, act=0, split=0):
    from simple_llm_amd import _lib

    M, K = x.shape
    N = w.shape[0]
    L = _lib.lib()
    y = torch.full((M, N), float("nan"), device="cuda")
    n = L.skv_linear_workspace_bytes(M, N, K) if ws else 0
    buf = torch.zeros(max(n, 4), dtype=torch.uint8, device="cuda")
    dev = [None if t is None else torch.from_numpy(np.ascontiguousarray(t)).cuda()
           for t in (x, w, bias, res, *(ln or (None, None)))]
    p = [None if t is None else t.data_ptr() for t in dev]
    _lib.check(L.skv_linear(y.data_ptr(), p[0], p[1], p[2], p[3], p[4], p[5], 1e-5, M, N, K, act,
                            split, buf.data_ptr() if ws else None, n, _lib.stream_handle()),
               "skv_linear")
    return y.cpu().numpy()


def _bound(x, w, extra):
    """Rounding of one output: 6 accumulations per 16 k and the omitted partial
    products (below 2^-24 of a product), each against sum |x w|."""
    K = x.shape[1]
    return (6 * -(-K // 16) + 2 + extra) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T) + 1e-30


# 64 x 64 tiles, 128 x 64 (from 128 of them), 256 x 128 (past 512), each with
# rows, columns and k past a tile's edge
@pytest.mark.parametrize("M,N,K", [(65, 1, 4), (65, 64, 28), (127, 65, 36), (129, 130, 100),
                                   (257, 63, 768), (300, 3000, 64), (1030, 1090, 132),
                                   (2050, 8500, 36), (4097, 4160, 20)])
def test_gemm_edges(gpu_ctx, M, N, K):
    banner(f"gemm M={M} N={N} K={K}")
    rng = np.random.default_rng(M + N + K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    w = rng.standard_normal((N, K)).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    r = rng.standard_normal((M, N)).astype(np.float32)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    want = x64 @ w64.T + b + r
    # bias and residual: two more roundings of the result
    tol = _bound(x64, w64, 0) + 2.0 ** -23 * (np.abs(want) + np.abs(b) + np.abs(r) + 1e-6)
    got = _linear(x, w, b, r)
    assert (np.abs(got - want) <= tol).all()


@pytest.mark.parametrize("ws", [True, False])
@pytest.mark.parametrize("M,N,K", [(70, 66, 36), (130, 192, 260), (700, 1536, 128)])
def test_gemm_layernorm(gpu_ctx, M, N, K, ws):
    banner(f"gemm LN M={M} N={N} K={K} ws={ws}")
    rng = np.random.default_rng(K)
    x = (rng.standard_normal((M, K)) * 3 + 5).astype(np.float32)
    w = rng.standard_normal((N, K)).astype(np.float32)
    g = rng.standard_normal(K).astype(np.float32)
    b = rng.standard_normal(K).astype(np.float32)
    x64 = x.astype(np.float64)
    d = x64 - x64.mean(1, keepdims=True)
    y64 = d / np.sqrt((d * d).mean(1, keepdims=True) + 1e-5) * g + b
    want = y64 @ w.astype(np.float64).T
    # each normalised value: a few roundings of x - mean (|x| <= ~20 times its spread)
    tol = _bound(np.abs(y64) + 20, w.astype(np.float64), 32)
    seg = N // 2  # two output segments
    got = _linear(x, w, ln=(g, b), ws=ws, split=seg).reshape(2, M, seg)
    assert (np.abs(np.concatenate([got[0], got[1]], 1) - want) <= tol).all()


@pytest.mark.parametrize("M,N", [(70, 70), (1100, 1090), (4097, 4160)])
def test_gemm_nonfinite_and_large(gpu_ctx, M, N):
    """Infinities, NaN and values next to the largest float give what fp32
    products give; other rows and columns keep their values."""
    banner(f"gemm non-finite M={M} N={N}")
    K = 40
    rng = np.random.default_rng(5)
    x = rng.standard_normal((M, K)).astype(np.float32)
    w = rng.standard_normal((N, K)).astype(np.float32)
    x[3, 7] = np.inf
    x[M - 1, 39] = -np.inf
    x[5, 0] = np.nan
    x[6] = 0.0
    x[6, 2] = np.finfo(np.float32).min  # rounds to -inf in bf16
    w[:, 2] *= 0.25
    w[9, 11] = np.inf
    w[10, 7] = 0.0                      # times x[3, 7]: NaN
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    with np.errstate(all="ignore"):
        want = x64 @ w64.T
        big = np.abs(want) > np.finfo(np.float32).max
        want[big] = np.sign(want[big]) * np.inf
        tol = _bound(x64, w64, 0) * 2
    got = _linear(x, w).astype(np.float64)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    np.testing.assert_array_equal(got[inf], want[inf])
    fin = np.isfinite(want)
    assert (np.abs(got[fin] - want[fin]) <= tol[fin]).all()


@pytest.mark.parametrize("M,N", [(70, 70), (1100, 1090), (4097, 4160)])
@pytest.mark.parametrize("e", [-111, -113, -119, -126, -134, -149])
def test_gemm_small_operands(gpu_ctx, M, N, e):
    """Operands down to the smallest fp32 value keep every bit (three bf16 parts
    of the value itself would lose them below 2^-111), on either side."""
    banner(f"gemm small operands 2^{e} M={M} N={N}")
    K = 36
    rng = np.random.default_rng(-e)
    with np.errstate(under="ignore"):
        small = (rng.standard_normal((M, K)) * 2.0 ** e).astype(np.float32)
    big = (rng.standard_normal((N, K)) * 2.0 ** 100).astype(np.float32)
    want = small.astype(np.float64) @ big.astype(np.float64).T
    tol = _bound(small.astype(np.float64), big.astype(np.float64), 0)
    tol += 2.0 ** -149 - 1e-30  # (outputs as small as 2^-60: no room of _bound's own)
    assert (np.abs(_linear(small, big) - want) <= tol).all()
    assert (np.abs(_linear(big, small) - want.T) <= tol.T).all()


@pytest.mark.parametrize("ln", [False, True])
@pytest.mark.parametrize("M,N", [(70, 70), (1100, 1090), (4097, 4160)])
def test_gemm_rows_beside_non_finite_ones_keep_their_bits(gpu_ctx, M, N, ln):
    """An infinite or NaN operand changes its own row (or column) alone."""
    banner(f"gemm rows beside non-finite ones M={M} N={N} ln={ln}")
    K = 44
    rng = np.random.default_rng(11)
    x = rng.standard_normal((M, K)).astype(np.float32)
    w = rng.standard_normal((N, K)).astype(np.float32)
    g = (rng.standard_normal(K).astype(np.float32), rng.standard_normal(K).astype(np.float32))
    for ws in (True, False) if ln else (False,):
        clean = _linear(x, w, ln=g if ln else None, ws=ws)
        xb, wb = x.copy(), w.copy()
        xb[[2, 40], 5] = np.inf, np.nan
        wb[[1, N - 1], 7] = -np.inf, np.float32(3e38)
        got = _linear(xb, wb, ln=g if ln else None, ws=ws)
        rows, cols = np.ones(M, bool), np.ones(N, bool)
        rows[[2, 40]] = cols[[1, N - 1]] = False
        np.testing.assert_array_equal(got[np.ix_(rows, cols)], clean[np.ix_(rows, cols)])
        assert not np.isfinite(got[~rows]).any() and np.isinf(got[rows][:, 1]).all()


@pytest.mark.parametrize("K", [(1 << 22) - 4, 1 << 22, (1 << 22) + 36])
def test_gemm_long_rows(gpu_ctx, K):
    """Rows on both sides of a tile's 32-bit byte range. Values of -1, 0 and 1:
    every sum is exact. With LayerNorm: 1e-3, above a random walk of the 1.6 M
    roundings of a sum (4e-5)."""
    banner(f"gemm long rows K={K}")
    from simple_llm_amd import _lib
    L = _lib.lib()
    M, N = 67, 5
    gen = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randint(-1, 2, (M, K), device="cuda", generator=gen).float()
    w = torch.randint(-1, 2, (N, K), device="cuda", generator=gen).float()
    g = torch.rand(K, device="cuda", generator=gen) + 0.5
    b = torch.rand(K, device="cuda", generator=gen)
    x64 = x.double()
    norm = (x64 - x64.mean(1, keepdim=True)) / torch.sqrt(x64.var(1, unbiased=False, keepdim=True)
                                                         + 1e-5) * g + b
    ws = torch.zeros(L.skv_linear_workspace_bytes(M, N, K), dtype=torch.uint8, device="cuda")
    for ln, buf in ((False, None), (True, None), (True, ws)):
        y = torch.full((M, N), float("nan"), device="cuda")
        _lib.check(L.skv_linear(y.data_ptr(), x.data_ptr(), w.data_ptr(), None, None,
                                g.data_ptr() if ln else None, b.data_ptr() if ln else None, 1e-5,
                                M, N, K, 0, 0, buf.data_ptr() if buf is not None else None,
                                buf.numel() if buf is not None else 0, _lib.stream_handle()),
                   "skv_linear")
        want = (norm if ln else x64) @ w.double().T.contiguous()
        if ln:
            assert float((y - want).norm() / want.norm()) < 1e-3
        else:
            assert torch.equal(y.double(), want)
