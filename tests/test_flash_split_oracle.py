"""How far a flash attention is from float64 when its products are taken from
operands split into three bf16 parts (csrc/split_bf16.h), emulated on the CPU
with every other step exact: the bar of the kernels' accuracy test must lie
above what all six partial products give and below what any lost part gives."""
from __future__ import annotations

import numpy as np
import pytest
import torch

#: Relative 2-norm error of O, dQ, dK and dV that the GPU test allows. The
#: kernels measure 1e-7 to 4e-7 at its sizes (fp32 sums, and the rounding of
#: exponents of up to ~8: 2^-22); without the third parts the products alone
#: give 2e-6 and more.
BAR = 1e-6

SIX = ((2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0))  # planes of the two factors


def flash_reference(q, k, v, go, prod=None):
    """O, dQ, dK, dV of one causal head [N, D] in float64; prod(a, b) gives a . b^T
    of the four products (default: exact)."""
    prod = prod or (lambda a, b: a @ b.T)
    q, k, v, go = (t.astype(np.float64) for t in (q, k, v, go))
    sc = 1.0 / np.sqrt(q.shape[1])
    mask = np.tril(np.ones((len(q), len(q)), bool))
    s = np.where(mask, prod(q * sc, k), -np.inf)
    e = np.exp(s - s.max(1, keepdims=True))
    p = e / e.sum(1, keepdims=True)
    o = prod(e, v.T) / e.sum(1, keepdims=True)
    ds = p * (prod(go, v) - (go * o).sum(1, keepdims=True))
    return o, prod(ds, k.T) * sc, prod(ds.T, q.T) * sc, prod(p.T, go.T)


def _parts(x):
    """The three bf16 parts of 2^24 x, as float64."""
    r = torch.from_numpy(np.ascontiguousarray(x * 2.0 ** 24)).float()
    out = []
    for _ in range(3):
        h = r.to(torch.bfloat16).float()
        out.append(h.double().numpy())
        r = r - h
    return out


def _split_prod(terms):
    def prod(a, b):
        pa, pb = _parts(a.astype(np.float32)), _parts(b.astype(np.float32))
        return sum(pa[i] @ pb[j].T for i, j in terms) * 2.0 ** -48
    return prod


def _errors(N, D, terms):
    rng = np.random.default_rng(N + D)
    x = [rng.standard_normal((N, D)).astype(np.float32) for _ in range(4)]
    return [float(np.linalg.norm(a - b) / np.linalg.norm(b))
            for a, b in zip(flash_reference(*x, prod=_split_prod(terms)), flash_reference(*x))]


@pytest.mark.parametrize("N,D", [(33, 15), (161, 16), (161, 64), (161, 128)])
def test_bar_tells_six_partial_products_from_fewer(N, D):
    assert max(_errors(N, D, SIX)) < BAR / 8
    lost = {"x third part": (2, 0), "w third part": (0, 2), "second parts": (1, 1)}
    for name, term in lost.items():
        errs = _errors(N, D, [t for t in SIX if t != term])
        print(name, ["%.1e" % e for e in errs])
        assert min(errs) > BAR, name
    assert min(_errors(N, D, SIX[3:])) > BAR  # neither third parts nor m m
