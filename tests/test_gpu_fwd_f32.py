"""The fp32 forward's split products: every rows-per-workgroup variant at the
edges of its tiles, and inputs the three-piece split cannot hold (infinite,
NaN, near the largest float), against the oracle or fp64 torch."""
import math

import numpy as np
import pytest
import torch

from gonn_amd import hip
from tests._util import fp32_bar, median_us

pytestmark = pytest.mark.gpu

# Scores of N(0,1) data at scale 1/sqrt(D) stay below about 6. Each is formed
# in at most 6 D/16 = 48 roundings of 2^-24 of its size, so P and with it O
# (|O| <= 5) move by at most 48 * 2^-24 * 6 = 1.7e-5, plus the same again for
# the PV sums' roundings.
TOL = 4e-5


def _run(B, H, Sq, Sk, D, causal, seed, pad=False, mask=False):
    rng = np.random.default_rng(seed)
    q = rng.standard_normal((B * H, Sq, D)).astype(np.float32)
    k, v = (rng.standard_normal((B * H, Sk, D)).astype(np.float32) for _ in range(2))
    lens = rng.integers(1, Sk + 1, B).astype(np.int32) if pad else None
    am = rng.standard_normal((B, Sq, Sk)).astype(np.float32) if mask else None
    dev = lambda x: torch.from_numpy(x).cuda()  # noqa: E731
    o, l = hip.attn_fwd(dev(q).view(B, H, Sq, D), dev(k).view(B, H, Sk, D), dev(v).view(B, H, Sk, D),
                        causal=causal, kv_len=dev(lens) if pad else None,
                        attn_mask=dev(am) if mask else None)
    torch.cuda.synchronize()
    s = np.einsum("bqd,bkd->bqk", q.astype(np.float64), k.astype(np.float64)) / math.sqrt(D)
    if mask:
        s += np.repeat(am.astype(np.float64), H, axis=0)
    if causal:
        s = np.where(np.arange(Sk)[None, None, :] > np.arange(Sq)[None, :, None], -np.inf, s)
    if pad:
        s = np.where(np.arange(Sk)[None, None, :] >= np.repeat(lens, H)[:, None, None], -np.inf, s)
    mx = s.max(-1, keepdims=True)
    p = np.exp(s - mx)
    ref = (p / p.sum(-1, keepdims=True)) @ v.astype(np.float64)
    rl = (mx + np.log(p.sum(-1, keepdims=True)))[..., 0]
    err = o.cpu().numpy().reshape(ref.shape) - ref
    assert np.abs(err).max() <= TOL
    # At most D roundings of a score and Sk of O's sum.
    rel = np.linalg.norm(err) / np.linalg.norm(ref)
    print("rel %.2e of %.2e" % (rel, fp32_bar(D + Sk)))
    assert rel <= fp32_bar(D + Sk)
    assert np.abs(l.cpu().numpy() - rl).max() <= TOL


# Grids on both sides of every bound of the waves-and-rows rule on 256 CUs: over
# 128 keys D = 64 takes 64 rows and 8 waves up to 256 such blocks (causal from
# 1024 keys: 512), then 128 rows and 8 waves up to as many blocks of 128; 64
# rows and 4 waves up to 512 blocks where keys are few, to 1024 where a causal
# chain is shorter than 1024; D = 128 64 rows (4 waves) over 32 keys, then 128
# rows and 8 waves over 128; 128 rows and 4 waves beyond.
@pytest.mark.parametrize("BH,D", [(3, 64), (33, 64), (130, 64), (200, 64), (260, 64), (520, 64),
                                  (3, 128), (65, 128), (140, 128), (260, 128), (520, 128)])
@pytest.mark.parametrize("Sq,Sk", [(1, 1), (31, 33), (33, 31), (127, 129), (129, 64), (257, 97), (257, 300)])
@pytest.mark.parametrize("causal", [False, True])
def test_tile_edges(BH, D, Sq, Sk, causal):
    _run(BH, 1, Sq, Sk, D, causal, BH + Sq + Sk)


@pytest.mark.parametrize("BH", [60, 160])
def test_long_causal_chains(BH):
    _run(BH, 1, 257, 1025, 64, True, BH)


@pytest.mark.parametrize("B,D", [(2, 64), (30, 64), (90, 64), (2, 128), (50, 128)])
@pytest.mark.parametrize("causal", [False, True])
def test_pad_and_mask(B, D, causal):
    _run(B, 3, 131, 97, D, causal, B, pad=True)
    _run(B, 3, 70, 161, D, causal, B, mask=True)


def _ref32(q, k, v, causal):
    s = (q.double() @ k.double().transpose(-1, -2)) / math.sqrt(q.shape[-1])
    if causal:
        i = torch.arange(s.shape[-2], device=s.device)[:, None]
        s = s.masked_fill(torch.arange(s.shape[-1], device=s.device)[None, :] > i, -math.inf)
    return torch.softmax(s, -1) @ v.double()


@pytest.mark.parametrize("BH,D", [(2, 64), (48, 64), (200, 64), (2, 128), (200, 128)])
def test_nonfinite_and_extreme_inputs(BH, D):
    g = torch.Generator().manual_seed(BH + D)
    q, k, v = (torch.randn(BH, 160, D, generator=g) for _ in range(3))
    k[0, 40] = 0.0
    k[0, 40, 3] = -math.inf   # -inf or +inf scores, by the sign of q
    q[0, :, 3] = q[0, :, 3].abs() + 0.1  # here: -inf, weight 0
    v[1, 17, 5] = math.inf
    v[1, 90, 7] = 3.4e38      # rounds to an infinite bf16
    q[-1, 33, 0] = math.nan
    o, _ = hip.attn_fwd(q.cuda(), k.cuda(), v.cuda())
    ref = _ref32(q.cuda(), k.cuda(), v.cuda(), False)
    torch.cuda.synchronize()
    assert torch.equal(torch.isnan(o), torch.isnan(ref))
    assert torch.equal(torch.isinf(o), torch.isinf(ref))
    ok = torch.isfinite(ref)
    err = (o.double() - ref).abs()[ok]
    assert bool((err <= TOL + 1e-5 * ref.abs()[ok]).all())


@pytest.mark.parametrize("D", [64, 128])
def test_wide_magnitudes(D):
    # Operands over 40 binary orders: each product keeps its own relative
    # accuracy, as in plain fp32.
    g = torch.Generator().manual_seed(D)
    e = torch.randint(-20, 21, (2, 1, D), generator=g).float()
    q, k = torch.randn(2, 200, D, generator=g), torch.randn(2, 200, D, generator=g)
    v = torch.randn(2, 200, D, generator=g) * torch.exp2(e)
    q, k = q * torch.exp2(e), k * torch.exp2(-e)
    o, _ = hip.attn_fwd(q.cuda(), k.cuda(), v.cuda(), causal=True)
    ref = _ref32(q.cuda(), k.cuda(), v.cuda(), True)
    torch.cuda.synchronize()
    scale = torch.exp2(e).cuda()
    assert float(((o.double() - ref).abs() / scale).max()) <= TOL


@pytest.mark.parametrize("BH,D", [(2, 64), (300, 64), (2, 128), (300, 128)])
def test_exact_large_scores(BH, D):
    # Integer scores that fp32 holds exactly, rising by 6 from tile to tile, so
    # that each tile but the last keeps a weight under a moved offset.
    S = 1100
    q, k = torch.zeros(BH, S, D), torch.zeros(BH, S, D)
    q[..., :2] = 1.0
    k[..., 0] = 1.0e6
    k[..., 1] = 6.0 * (torch.arange(S) // 32)
    v = torch.randn(BH, S, D, generator=torch.Generator().manual_seed(D))
    q, k, v = q.cuda(), k.cuda(), v.cuda()
    o, l = hip.attn_fwd(q, k, v, scale=1.0)
    s = q.double() @ k.double().transpose(-1, -2)
    torch.cuda.synchronize()
    assert float((o.double() - torch.softmax(s, -1) @ v.double()).abs().max()) <= TOL
    assert float((l.double() / torch.logsumexp(s, -1) - 1).abs().max()) <= 2.0 ** -23


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("mag", [10, 14, 16, 20, 30])
def test_huge_scores_of_single_rows(D, mag):
    # Scores of 2^(2 mag) and more, one query per slice: the largest takes all
    # the weight where it leads by more than the scores' rounding.
    g = torch.Generator().manual_seed(D + mag)
    q, k = (torch.randn(300, n, D, generator=g).bfloat16().float() * 2.0 ** mag for n in (1, 40))
    v = torch.randn(300, 40, D, generator=g)
    o, l = hip.attn_fwd(q.cuda(), k.cuda(), v.cuda())
    s = (q.double() @ k.double().transpose(-1, -2))[:, 0] / math.sqrt(D)
    top = s.topk(2, -1).values
    clear = top[:, 0] - top[:, 1] > 100 + 1e-5 * s.abs().amax(-1)
    assert int(clear.sum()) > 200
    best = torch.gather(v, 1, s.argmax(-1)[:, None, None].expand(-1, 1, D))[:, 0]
    torch.cuda.synchronize()
    assert bool(torch.isfinite(o).all())
    assert float((o.cpu()[:, 0] - best)[clear].abs().max()) <= TOL
    assert float((l.cpu()[:, 0] / top[:, 0] - 1).abs()[clear].max()) <= 1e-5


@pytest.mark.parametrize("D", [64, 128])
def test_blocked_rows_take_no_longer(D):
    # A query whose mask is -inf on every key has no result (O NaN, LSE -inf);
    # it is not one to repeat with the plain products (about five times slower).
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(8, 12, 700, D, generator=g).cuda() for _ in range(3))
    clear = torch.zeros(8, 700, 700, device="cuda")
    blocked = clear.clone()
    blocked[:, ::37] = -math.inf
    o, l = hip.attn_fwd(q, k, v, attn_mask=blocked)
    want, wl = hip.attn_fwd(q, k, v, attn_mask=clear)
    rows = torch.arange(700, device="cuda") % 37 != 0
    torch.cuda.synchronize()
    assert torch.equal(o[:, :, rows], want[:, :, rows])
    assert bool(torch.isnan(o[:, :, ~rows]).all())
    l, wl = l.view(8, 12, 700), wl.view(8, 12, 700)
    assert torch.equal(l[..., rows], wl[..., rows]) and bool((l[..., ~rows] == -math.inf).all())
    a, b = (median_us(lambda m=m: hip.attn_fwd(q, k, v, attn_mask=m)) for m in (clear, blocked))
    assert b <= 2 * a, (a, b)


@pytest.mark.parametrize("D", [64, 128])
def test_fallback_cost(D):
    # Every wave repeats its rows: a few times the ordinary call, not ten.
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(8, 12, 700, D, generator=g).cuda() for _ in range(3))
    nan = torch.full_like(q, math.nan)
    a, b = (median_us(lambda x=x: hip.attn_fwd(x, k, v)) for x in (q, nan))
    assert b <= 5 * a, (a, b)


@pytest.mark.parametrize("BH,D", [(2, 64), (300, 64), (2, 128), (300, 128)])
@pytest.mark.parametrize("e", [-90, -100, -106, -112, -116, -120])
def test_small_magnitudes(BH, D, e):
    # Pieces of values below 2^-110 have fewer than 24 bits; results that small
    # come from the plain products. (At 2^-124 fp32 itself loses bits of P V.)
    g = torch.Generator().manual_seed(D - e)
    q, k, v = (torch.randn(BH, 300, D, generator=g).cuda() for _ in range(3))
    v = (v.double() * 2.0 ** e).float()
    o, _ = hip.attn_fwd(q, k, v, causal=True)
    ref = _ref32(q, k, v, True)
    torch.cuda.synchronize()
    assert float((o.double() - ref).norm() / ref.norm()) <= fp32_bar(D + 300)
