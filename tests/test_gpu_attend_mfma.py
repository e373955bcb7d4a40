"""The matrix-core causal attend over the cache: both rows-per-workgroup
variants and the VALU kernel on either side of their bounds, query counts and
cache lengths at the edges of the tiles and splits, and infinite operands,
against fp64 torch over each query's positions."""
import math

import pytest
import torch

from gonn_amd import hip
from tests._util import fp32_bar

pytestmark = pytest.mark.gpu

# K and V are exact; a score (below 6) takes D/16 + 2 roundings of its size and
# O one per 32 keys and merge, so O (below 5) stays within 1e-5.
TOL = 1e-5


def _fill(B, H, Lmax, D, lens, seed):
    g = torch.Generator().manual_seed(seed)
    k, v = (torch.randn(B, H, Lmax, D, generator=g).cuda().bfloat16() for _ in range(2))
    cache = hip.KVCache(B, H, Lmax, D)
    cache.append(k, v, counts=lens)
    return k, v, cache


def _check(o, ref, n):
    assert float((o.double() - ref).abs().max()) <= TOL
    # At most D roundings of a score and n of O's sum (n cached positions).
    rel = float((o.double() - ref).norm() / ref.norm())
    print("rel %.2e of %.2e" % (rel, fp32_bar(o.shape[-1] + n)))
    assert rel <= fp32_bar(o.shape[-1] + n)


def _ref(q, k, v, lens, scale):
    B, H, T, D = q.shape
    out = torch.empty(B, H, T, D, dtype=torch.float64, device="cuda")
    for b in range(B):
        n = int(lens[b])
        s = scale * (q[b].double() @ k[b, :, :n].double().transpose(-1, -2))
        lim = torch.arange(n - T + 1, n + 1, device="cuda")[:, None]
        s = s.masked_fill(torch.arange(n, device="cuda")[None, None, :] >= lim, -math.inf)
        out[b] = torch.softmax(s, -1) @ v[b, :, :n].double()
    return out


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [1, 2, 4, 5, 31, 32, 33, 63, 64, 65, 130])
@pytest.mark.parametrize("B,H", [(3, 2), (3, 100)])  # fewer and more slices than CUs
def test_query_counts(B, H, T, D):
    lens = [T, T + 1, max(T, 257)]
    k, v, cache = _fill(B, H, 300, D, lens, T + D)
    q = torch.randn(B, H, T, D, generator=torch.Generator().manual_seed(T)).cuda()
    for scale in (1.0 / math.sqrt(D), -0.05, 0.0):
        o = cache.attend_causal(q, scale=scale)
        torch.cuda.synchronize()
        _check(o, _ref(q, k, v, lens, scale), min(lens))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [7, 65, 130])
def test_dealt_slices(D, T):
    # 16 slices, times the splits: whole slices for each of the 8 XCDs.
    lens = [T, 700]
    k, v, cache = _fill(2, 8, 700, D, lens, T + D)
    q = torch.randn(2, 8, T, D, generator=torch.Generator().manual_seed(T)).cuda()
    o = cache.attend_causal(q)
    torch.cuda.synchronize()
    _check(o, _ref(q, k, v, lens, 1 / math.sqrt(D)), min(lens))


@pytest.mark.parametrize("D,T", [(64, 40), (128, 40), (128, 7)])
def test_long_caches_split(D, T):
    lens = [9000, 4097, T]
    k, v, cache = _fill(3, 2, 9000, D, lens, D)
    q = torch.randn(3, 2, T, D, generator=torch.Generator().manual_seed(D)).cuda()
    o = cache.attend_causal(q)
    torch.cuda.synchronize()
    _check(o, _ref(q, k, v, lens, 1 / math.sqrt(D)), min(lens))


@pytest.mark.parametrize("T", [8, 48])
def test_infinite_operands(T):
    D, lens = 64, [200, 150]
    g = torch.Generator().manual_seed(T)
    k, v = (torch.randn(2, 2, 200, D, generator=g) for _ in range(2))
    q = torch.randn(2, 2, T, D, generator=g)
    k[0, 0, 20] = 0.0
    k[0, 0, 20, 3] = -math.inf
    q[0, 0, :, 3] = q[0, 0, :, 3].abs() + 0.1  # score -inf, weight 0
    v[1, 1, 30, 5] = math.inf
    q[0, 1, 2, 9] = math.nan
    q, k, v = q.cuda(), k.cuda().bfloat16(), v.cuda().bfloat16()
    cache = hip.KVCache(2, 2, 200, D)
    cache.append(k, v, counts=lens)
    o = cache.attend_causal(q)
    ref = _ref(q, k, v, lens, 1 / math.sqrt(D))
    torch.cuda.synchronize()
    assert torch.equal(torch.isnan(o), torch.isnan(ref))
    assert torch.equal(torch.isinf(o), torch.isinf(ref))
    ok = torch.isfinite(ref)
    assert float((o.double() - ref).abs()[ok].max()) <= TOL


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [5, 8, 31, 32, 48, 130])
@pytest.mark.parametrize("Lmax", [300, 9000])  # one split and several
def test_later_positions_stay_unseen(D, T, Lmax):
    # An infinite or NaN row counts only for the queries that see it, whatever
    # it shares a tile with.
    n = 290
    g = torch.Generator().manual_seed(T + D)
    k, v = (torch.randn(2, 2, n, D, generator=g) for _ in range(2))
    q = torch.randn(2, 2, T, D, generator=g).cuda()
    clean = k.cuda().bfloat16(), v.cuda().bfloat16()
    at = {0: n - 1, 1: n - 3, 2: n - T + 1}  # slice -> position
    for i, pos in at.items():
        v[i // 2, i % 2, pos, 5] = (math.inf, -math.inf, math.nan)[i]
    k[1, 1, n - 2, 4] = math.nan
    at[3] = n - 2
    cache = hip.KVCache(2, 2, Lmax, D)
    cache.append(k.cuda().bfloat16(), v.cuda().bfloat16(), counts=[n, n])
    o = cache.attend_causal(q)
    ref = _ref(q, *clean, [n, n], 1 / math.sqrt(D))
    torch.cuda.synchronize()
    for i, pos in at.items():
        got, want = o[i // 2, i % 2], ref[i // 2, i % 2].clone()
        sees = torch.arange(n - T, n, device="cuda") >= pos
        want[sees] = math.nan
        if i < 3:  # one column of V only
            want[sees] = ref[i // 2, i % 2][sees]
            want[sees, 5] = (math.inf, -math.inf, math.nan)[i]
        assert torch.equal(torch.isnan(got), torch.isnan(want)), i
        assert torch.equal(got[torch.isinf(want)].double(), want[torch.isinf(want)]), i
        ok = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got), ok), i
        assert float((got.double() - want).abs()[ok].max()) <= TOL, i


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [3, 40])
@pytest.mark.parametrize("Lmax", [70, 10000])  # one split and several
def test_all_scores_minus_infinite(D, T, Lmax):
    # No key has a weight: O = 0, however many splits the cache has.
    k = torch.zeros(1, 2, 70, D)
    k[..., 0] = -math.inf
    v = torch.randn(1, 2, 70, D, generator=torch.Generator().manual_seed(D))
    cache = hip.KVCache(1, 2, Lmax, D)
    cache.append(k.cuda().bfloat16(), v.cuda().bfloat16(), counts=[70])
    o = cache.attend_causal(torch.ones(1, 2, T, D, device="cuda"))
    torch.cuda.synchronize()
    assert torch.equal(o, torch.zeros_like(o))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [4, 40])
@pytest.mark.parametrize("Lmax", [80, 10000])  # O written by the attend, by the combine
def test_any_float_alignment(D, T, Lmax):
    k, v, _ = _fill(2, 2, 80, D, [80, 77], D)
    cache = hip.KVCache(2, 2, Lmax, D)
    cache.append(k, v, counts=[80, 77])
    q = torch.randn(2, 2, T, D, generator=torch.Generator().manual_seed(T)).cuda()
    want = cache.attend_causal(q)
    for off in (1, 2, 3):
        q2 = torch.empty(q.numel() + off, device="cuda")[off:].view_as(q).copy_(q)
        guard = torch.full((q.numel() + off + 1,), 7.0, device="cuda")
        o2 = guard[off:-1].view_as(q)
        got = cache.attend_causal(q2, out=o2)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and bool((guard[:off] == 7.0).all()) and float(guard[-1]) == 7.0
