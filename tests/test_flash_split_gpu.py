"""The fp32 flash kernels' split products (csrc/flash_split.hip): head dims at
the edges of the 16- and 32-wide padding with lengths at the edges of a piece
and a workgroup, and operands that have no finite bf16 parts."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import banner
from oracle import kv_oracle as ko
from test_flash_bwd_gpu import flash_bwd
from test_flash_fwd_gpu import flash_fwd
from test_flash_split_oracle import BAR, flash_reference

pytestmark = pytest.mark.gpu

TOL = 1e-4  # the bar of the fp32 flash tests


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def flash_fwd_into(out, q, k, v, N, H, D):
    from simple_llm_amd import _lib
    st = torch.empty(2 * N * H, device=q.device)
    _lib.check(_lib.lib().skv_flash_fwd(out.data_ptr(), st.data_ptr(), st[N * H:].data_ptr(),
                                        q.data_ptr(), k.data_ptr(), v.data_ptr(), 1, N, H, D,
                                        float(1 / np.sqrt(D)), _lib.stream_handle(q.device)),
               "skv_flash_fwd")


def _dev(x):
    return torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda()


@pytest.mark.parametrize("N", [31, 33, 128, 161])
@pytest.mark.parametrize("D", [15, 16, 17, 33, 50, 64, 65, 84, 97, 112, 128])
def test_edges_match_oracle(gpu_ctx, N, D):
    banner(f"flash split N={N} D={D}")
    B, H = 2, 2
    rng = np.random.default_rng(N + D)
    Q, K, V, dO = (rng.standard_normal((B * N, H * D)).astype(np.float32) for _ in range(4))
    O, L, M = ko.flash_attention(Q, K, V, B, N, H, D)
    o, Ls, Ms = flash_fwd(_dev(Q), _dev(K), _dev(V), B, N, H, D)
    for got, want in ((o, O), (Ls, L), (Ms, M)):
        assert _rel(got.cpu().numpy().reshape(-1), np.asarray(want).reshape(-1)) < TOL
    want = ko.flash_attention_backward(Q, K, V, O, L, M, dO, B, N, H, D)
    for fast in (False, True):
        got = flash_bwd(_dev(Q), _dev(K), _dev(V), _dev(O), _dev(L), _dev(M), _dev(dO), B, N, H,
                        D, fast=fast)
        for g, w in zip(got, want):
            assert _rel(g.cpu().numpy(), w) < TOL


# every padded head dim, in one of its load modes
@pytest.mark.parametrize("D", [15, 16, 32, 34, 48, 52, 64, 80, 84, 96, 112, 128])
def test_accuracy_against_float64(gpu_ctx, D):
    """Forward and both forms of the backward within the bar that tells all six
    partial products from any five (test_flash_split_oracle.py)."""
    banner(f"flash split accuracy D={D}")
    N, H = 161, 2
    rng = np.random.default_rng(D)
    t = [rng.standard_normal((N, H, D)).astype(np.float32) for _ in range(4)]
    q, k, v, go = (_dev(x.reshape(N, H * D)) for x in t)
    o, L, M = flash_fwd(q, k, v, 1, N, H, D)
    want = [np.stack(x, 1) for x in zip(*(flash_reference(*(x[:, h] for x in t))
                                          for h in range(H)))]
    for fast in (False, True):
        got = (o, *flash_bwd(q, k, v, o, L, M, go, 1, N, H, D, fast=fast))
        for g, w, name in zip(got, want, ("o", "dq", "dk", "dv")):
            err = _rel(g.cpu().numpy().reshape(N, H, D).astype(np.float64), w)
            print(f"{name} rel_err={err:.2e}")
            assert err < BAR, (name, fast)


@pytest.mark.parametrize("D", [24, 64, 96, 128])
def test_prefill_accuracy_against_float64(gpu_ctx, D):
    """An fp32 cache's chunk, grouped queries after a prefix, within the same bar."""
    from simple_llm_amd.gpu import gpu
    banner(f"fp32 prefill accuracy D={D}")
    B, Hq, Hkv, C, start = 2, 4, 2, 70, np.array([0, 90], np.int64)
    T = int(start.max()) + C
    rng = np.random.default_rng(D)
    k, v = (rng.standard_normal((B, T, Hkv, D)).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((B, C, Hq, D)).astype(np.float32)
    cache = gpu.kv_cache_create(gpu_ctx, gpu.KVCacheConfig(B, T, 1, Hq, D, n_kv_heads=Hkv))
    layer = cache.layers[0]
    layer.k_cache.buffer.copy_(_dev(k.reshape(B * T, Hkv * D)))
    layer.v_cache.buffer.copy_(_dev(v.reshape(B * T, Hkv * D)))
    layer.lens.copy_(torch.from_numpy(start))
    layer.host_lens = start.copy()
    new = [_dev(np.stack([x[b, start[b]:start[b] + C] for b in range(B)])) for x in (k, v)]
    out = torch.empty(B, C, Hq, D, device="cuda")
    gpu.kv_cache_prefill(gpu_ctx, cache, 0, *new, _dev(q), out)
    got = out.cpu().numpy().astype(np.float64)
    for b in range(B):
        n = int(start[b]) + C
        for h in range(Hq):
            s = (q[b, :, h].astype(np.float64) @ k[b, :n, h // 2].astype(np.float64).T) / D ** 0.5
            s[np.arange(n)[None] > start[b] + np.arange(C)[:, None]] = -np.inf
            e = np.exp(s - s.max(1, keepdims=True))
            want = (e / e.sum(1, keepdims=True)) @ v[b, :n, h // 2].astype(np.float64)
            assert _rel(got[b, :, h], want) < BAR, (b, h)


def _reference(q, k, v, go):
    """float64 O, dQ, dK, dV of one causal head [N, D], each query over the
    keys it sees alone."""
    q, k, v, go = (t.astype(np.float64) for t in (q, k, v, go))
    o, dq, dk, dv = (np.zeros_like(q) for _ in range(4))
    sc = 1.0 / np.sqrt(q.shape[1])
    for i in range(len(q)):
        s = (k[:i + 1] @ q[i]) * sc
        e = np.exp(s - s.max())
        pr = e / e.sum()
        o[i] = pr @ v[:i + 1]
        ds = pr * (v[:i + 1] @ go[i] - (go[i] * o[i]).sum())
        dq[i] = (ds @ k[:i + 1]) * sc
        dk[:i + 1] += np.outer(ds, q[i]) * sc
        dv[:i + 1] += np.outer(pr, go[i])
    return o, dq, dk, dv


@pytest.mark.parametrize("D", [48, 64, 128])
@pytest.mark.parametrize("what,value", [(w, v) for w in ("q", "k", "v", "go")
                                        for v in (np.inf, -np.inf)]
                         + [("q", 3.4e38), ("k", -3.4e38)])
def test_values_without_bf16_parts(gpu_ctx, D, what, value):
    """One infinite element, or one that rounds to infinity in bf16, at row 40
    of head 0: values, infinities and NaN as in the plain computation. (Rows 32
    to 63 share a piece with it, where a masked key weighs 0 times infinity.)"""
    banner(f"flash split {what}={value} D={D}")
    N, H = 200, 2
    rng = np.random.default_rng(D)
    t = {n: rng.standard_normal((N, H, D)).astype(np.float32) for n in ("q", "k", "v", "go")}
    if np.isfinite(value):  # what it meets is small, so the scores stay ordinary
        t["k" if what == "q" else "q"] *= np.float32(1e-38)
    t[what][40, 0, 5] = value
    flat = {n: _dev(x.reshape(N, H * D)) for n, x in t.items()}
    o, L, M = flash_fwd(flat["q"], flat["k"], flat["v"], 1, N, H, D)
    grads = flash_bwd(flat["q"], flat["k"], flat["v"], o, L, M, flat["go"], 1, N, H, D,
                      fast=D <= 64)
    got = [x.cpu().numpy().reshape(N, H, D).astype(np.float64) for x in (o, *grads)]
    with np.errstate(all="ignore"):
        want = [_reference(*(t[n][:, h] for n in ("q", "k", "v", "go"))) for h in range(H)]
    rows = np.r_[0:32, 64:N]
    for i, name in enumerate(("o", "dq", "dk", "dv")):
        a, b = got[i][rows, 0], want[0][i][rows]
        # sums of 3.4e38 values; and rows whose Dl is not finite, where every
        # masked key of a piece weighs 0 times infinity
        if name == {"q": "dk", "k": "dq"}.get(what) and np.isfinite(value):
            continue
        if name in ("dq", "dk") and np.isinf(value) and what in ("k", "v"):
            continue
        assert _rel(got[i][:, 1], want[1][i]) < TOL, name  # the other head
        np.testing.assert_array_equal(np.isnan(a), np.isnan(b), err_msg=name)
        np.testing.assert_array_equal(np.where(np.isinf(a), a, 0), np.where(np.isinf(b), b, 0),
                                      err_msg=name)
        fin = np.isfinite(b)
        assert _rel(np.where(fin, a, 0), np.where(fin, b, 0)) < TOL, name


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("D", [48, 64, 128])
@pytest.mark.parametrize("scale", [{"go": -120}, {"v": -120}, {"k": -120, "q": 20},
                                   {"q": -120, "k": 20}, {"go": -145, "v": 60},
                                   {"q": -145, "k": 30}, {"k": -145, "q": 30},
                                   {"go": 50}])
def test_small_operands(gpu_ctx, D, scale, fast):
    """Operands of 2^-120 (three bf16 parts of the values themselves would keep
    14 of their bits) and 2^-145 (fp32 subnormals) give outputs, row maxima and
    gradients as accurate as ordinary ones: within 5e-6, ten times the error of
    ordinary operands at this size. (Results that are subnormal themselves: within
    the spacing of those, 2^-149, of each.) The last: gradients too large for what
    the chain of products carries."""
    banner(f"flash small operands {scale} D={D} fast={fast}")
    N, H = 200, 2
    rng = np.random.default_rng(D)
    t = {n: (rng.standard_normal((N, H, D)) * 2.0 ** scale.get(n, 0)).astype(np.float32)
         for n in ("q", "k", "v", "go")}
    flat = {n: _dev(x.reshape(N, H * D)) for n, x in t.items()}
    o, L, M = flash_fwd(flat["q"], flat["k"], flat["v"], 1, N, H, D)
    grads = flash_bwd(flat["q"], flat["k"], flat["v"], o, L, M, flat["go"], 1, N, H, D, fast=fast)
    got = [x.cpu().numpy().reshape(N, H, D).astype(np.float64) for x in (o, *grads)]
    want = [_reference(*(t[n][:, h] for n in ("q", "k", "v", "go"))) for h in range(H)]
    for i, name in enumerate(("o", "dq", "dk", "dv")):
        ref = np.stack([w[i] for w in want], 1)
        err = _rel(got[i], ref)
        print(f"{name} rel_err={err:.2e}")
        few = 5e-6 * np.linalg.norm(ref) < 2.0 ** -149 * ref.size ** 0.5
        assert (np.abs(got[i] - ref).max() < 2.0 ** -149 if few else err < 5e-6), name
    s = np.einsum("qhd,khd->hqk", t["q"].astype(np.float64), t["k"].astype(np.float64))
    s = np.where(np.tril(np.ones((N, N), bool)), s / np.sqrt(D), -np.inf).max(-1).T
    assert _rel(M.cpu().numpy().reshape(N, H).astype(np.float64), s) < 5e-6


@pytest.mark.parametrize("D", [20, 50, 64, 96, 128])
@pytest.mark.parametrize("what", ["q", "k", "v", "go"])
def test_rows_beside_non_finite_ones_keep_their_bits(gpu_ctx, D, what):
    """An infinite element at row 40 leaves the bits of every row that does not
    see it: queries before it (queries other than 40 where it is a query's),
    keys after it, and the other head. (Rows 32 to 63 share a piece with it, where
    a masked pair weighs 0 times infinity.)"""
    banner(f"flash rows beside a non-finite {what} D={D}")
    N, H, at = 150, 2, 40
    rng = np.random.default_rng(D)
    t = {n: rng.standard_normal((N, H, D)).astype(np.float32) for n in ("q", "k", "v", "go")}
    runs = []
    for bad in (False, True):
        if bad:
            t[what][at, 0, 5] = np.inf
        f = {n: _dev(x.reshape(N, H * D)) for n, x in t.items()}
        o, L, M = flash_fwd(f["q"], f["k"], f["v"], 1, N, H, D)
        row = f["q"].clone()  # the output in place of the queries
        flash_fwd_into(row, row, f["k"], f["v"], N, H, D)
        assert torch.equal(row.view(torch.int32), o.view(torch.int32))
        for fast in (False, True):
            grads = flash_bwd(f["q"], f["k"], f["v"], o, L, M, f["go"], 1, N, H, D, fast=fast)
            runs.append([x.cpu().numpy().reshape(N, H, -1) for x in (o, L, M, *grads)])
    own = what in ("q", "go")  # a query's operand
    queries = np.delete(np.arange(N), at) if own else np.arange(32)
    keys = np.arange(64, N) if own else np.arange(0)  # (queries from 40 on see every key)
    for a, b in zip(runs[:2], runs[2:]):
        for i, rows in enumerate((queries,) * 4 + (keys,) * 2):
            np.testing.assert_array_equal(a[i][rows, 0], b[i][rows, 0])
            np.testing.assert_array_equal(a[i][:, 1], b[i][:, 1])
    assert what == "go" or not np.isfinite(runs[2][0][at:, 0]).all()
