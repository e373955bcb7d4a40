"""The 2-norm bar that the GPU tests hold the fp32 mode to (tests/_util.py) tells
three bf16 pieces and six products from two pieces, on a model of the forward and
of dV with exact sums (CPU)."""
import math

import numpy as np
import pytest

from tests._util import bf16_round, fp32_bar, randn


def _pieces(x, n):
    out = []
    for _ in range(n):
        out.append(bf16_round(x))
        x = x - out[-1]
    return [p.astype(np.float64) for p in out]


def _product(a, b, n):
    """a @ b of fp32 matrices by the piece products of order 2^-8(n-1) and above."""
    pa, pb = _pieces(a, n), _pieces(b, n)
    return sum(pa[i] @ pb[j] for i in range(n) for j in range(n) if i + j < n)


def _model(q, k, v, dO, n):
    """O and dV; n pieces, or 0 for 64 bits."""
    mm = (lambda a, b: _product(a.astype(np.float32), b.astype(np.float32), n)) if n else np.matmul
    s = mm(q, k.T) / math.sqrt(q.shape[1])
    e = np.exp(s - s.max(-1, keepdims=True))
    l = e.sum(-1, keepdims=True)
    return mm(e, v) / l, mm((e / l).T, dO)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Sk", [(1, 1), (33, 31), (129, 64), (257, 300)])
def test_bar_tells_three_pieces_from_two(Sq, Sk, D):
    q, k, v, dO = (randn((n, D), i).astype(np.float64) for i, n in enumerate((Sq, Sk, Sk, Sq)))
    exact = _model(q, k, v, dO, 0)
    for n, ok in ((3, True), (2, False)):
        for i, (a, r) in enumerate(zip(_model(q, k, v, dO, n), exact)):
            bar = fp32_bar(D + Sk if i == 0 else 2 * D + Sq)
            rel = np.linalg.norm(a - r) / np.linalg.norm(r)
            assert (rel <= 0.5 * bar) if ok else (rel >= 2 * bar), (n, i, rel, bar)
