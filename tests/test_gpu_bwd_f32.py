"""The fp32 backward's split products: every keys- and rows-per-workgroup
variant at the edges of its tiles, and inputs the three-piece split cannot
hold, against fp64 torch."""
import math

import pytest
import torch

from gonn_amd import hip
from tests._util import fp32_bar, median_us

pytestmark = pytest.mark.gpu


def _inputs(BH, Sq, Sk, D, seed):
    g = torch.Generator().manual_seed(seed)
    q, dO = (torch.randn(BH, Sq, D, generator=g).cuda() for _ in range(2))
    k, v = (torch.randn(BH, Sk, D, generator=g).cuda() for _ in range(2))
    return q, k, v, dO


def _ref(q, k, v, dO, causal, lens=None, mask=None):
    q, k, v, dO = (x.double() for x in (q, k, v, dO))
    scale = 1.0 / math.sqrt(q.shape[-1])
    s = (q @ k.transpose(-1, -2)) * scale
    if mask is not None:
        s = s + mask.double()
    j = torch.arange(s.shape[-1], device=s.device)
    if causal:
        s = s.masked_fill(j[None, :] > torch.arange(s.shape[-2], device=s.device)[:, None], -math.inf)
    if lens is not None:
        s = s.masked_fill(j[None, None, :] >= lens[:, None, None], -math.inf)
    p = torch.softmax(s, -1)
    o = p @ v
    ds = p * (dO @ v.transpose(-1, -2) - (dO * o).sum(-1, keepdim=True)) * scale
    return ds @ k, ds.transpose(-1, -2) @ q, p.transpose(-1, -2) @ dO


def _check(q, k, v, dO, causal, lens=None, mask=None):
    opt = dict(causal=causal, kv_len=lens.int() if lens is not None else None, attn_mask=mask)
    o, l = hip.attn_fwd(q, k, v, **opt)
    got = hip.attn_bwd(q, k, v, o, l, dO, **opt)
    torch.cuda.synchronize()
    for name, a, r in zip(("dQ", "dK", "dV"), got, _ref(q, k, v, dO, causal, lens, mask)):
        # P and dS carry the score's error, at most 48 roundings of 2^-24 of a
        # score below 6 (1.7e-5 of each entry); a row's entries are held to
        # that of the row's largest, or of 1 where the row cancels.
        row = r.abs().amax(-1, keepdim=True).clamp_min(1.0)
        assert float(((a.double() - r).abs() / row).max()) <= 4e-5, name
        # At most D roundings of the score, D of dP and S or Sk of the sum. (With
        # one key dS is zero, and dQ and dK are the noise of its two terms.)
        if k.shape[-2] > 1 or name == "dV":
            n = 2 * q.shape[-1] + (k.shape[-2] if name == "dQ" else q.shape[-2])
            rel = float((a.double() - r).norm() / r.norm())
            print("rel %s %.2e of %.2e" % (name, rel, fp32_bar(n)))
            assert rel <= fp32_bar(n), name


# Both sides of every bound of the two rules on 256 CUs (D = 64: 32-row blocks
# up to 256 or, uneven causal, 512; 64-row blocks up to 256 / 512; 128-row
# blocks beyond, changing at 512 and 1536 of them when causal). The first shapes
# stay within two blocks of 128; the last two are uneven when causal, with query
# blocks that start past key 0 and diagonals inside later blocks.
@pytest.mark.parametrize("BH,D,Sq,Sk", [
    (BH, D, Sq, Sk)
    for BH, D in [(2, 64), (100, 64), (200, 64), (300, 64), (900, 64), (2, 128), (70, 128), (300, 128)]
    for Sq, Sk in [(1, 1), (33, 31), (31, 33), (129, 127), (64, 193), (193, 64)]
] + [
    (BH, D, Sq, Sk)
    for BH, D in [(40, 64), (60, 64), (120, 64), (300, 64), (600, 64), (40, 128), (70, 128), (300, 128)]
    for Sq, Sk in [(257, 300), (300, 257)]
])
@pytest.mark.parametrize("causal", [False, True])
def test_tile_edges(BH, D, Sq, Sk, causal):
    _check(*_inputs(BH, Sq, Sk, D, BH + Sq + Sk), causal)


@pytest.mark.parametrize("BH,D", [(3, 64), (120, 64), (300, 64), (3, 128), (300, 128)])
@pytest.mark.parametrize("causal", [False, True])
def test_pad_and_mask(BH, D, causal):
    q, k, v, dO = _inputs(BH, 131, 97, D, BH)
    g = torch.Generator().manual_seed(BH)
    lens = torch.randint(1, 98, (BH,), generator=g).cuda()
    # Padded rows are never used, whatever they hold.
    k2, v2 = k.clone(), v.clone()
    for b in range(BH):
        k2[b, int(lens[b]):] = math.nan
        v2[b, int(lens[b]):] = math.nan
    opt = dict(causal=causal, kv_len=lens.int())
    o, l = hip.attn_fwd(q, k, v, **opt)
    a = hip.attn_bwd(q, k, v, o, l, dO, **opt)
    o2, l2 = hip.attn_fwd(q, k2, v2, **opt)
    a2 = hip.attn_bwd(q, k2, v2, o2, l2, dO, **opt)
    torch.cuda.synchronize()
    for x, y in zip((o, l) + a, (o2, l2) + a2):
        assert torch.equal(x, y)
    _check(q, k, v, dO, causal, lens=lens)
    _check(q, k, v, dO, causal, mask=torch.randn(BH, 131, 97, generator=g).cuda())


@pytest.mark.parametrize("BH,D", [(40, 64), (60, 64), (120, 64), (300, 64), (600, 64), (40, 128), (120, 128)])
def test_uneven_causal_mask(BH, D):
    g = torch.Generator().manual_seed(BH)
    _check(*_inputs(BH, 257, 300, D, BH), True, mask=torch.randn(BH, 257, 300, generator=g).cuda())


@pytest.mark.parametrize("BH,D", [(3, 64), (300, 64), (3, 128), (300, 128)])
def test_nonfinite_inputs(BH, D):
    q, k, v, dO = _inputs(BH, 70, 60, D, D)
    o, l = hip.attn_fwd(q, k, v)
    clean = hip.attn_bwd(q, k, v, o, l, dO)
    q2, k2, dO2 = q.clone(), k.clone(), dO.clone()
    k2[0, 40] = 0.0
    k2[0, 40, 3] = -math.inf
    q2[0, :, 3] = q2[0, :, 3].abs() + 0.1  # score -inf, weight 0
    dO2[1, 5, 7] = math.inf
    dO2[1, 9, 2] = 3.4e38
    o2, l2 = hip.attn_fwd(q2, k2, v)
    got = hip.attn_bwd(q2, k2, v, o2, l2, dO2)
    ref = _ref(q2, k2, v, dO2, False)
    torch.cuda.synchronize()

    def close(a, r):
        assert torch.equal(torch.isfinite(a), torch.isfinite(r.float()))
        ok = torch.isfinite(r.float())
        row = torch.where(ok, r, 0.0).abs().amax(-1, keepdim=True).clamp_min(1.0)
        assert float(((a.double() - r).abs() / row)[ok].max()) <= 4e-5

    # Slice 0: key 40 has weight 0, so only dQ's column 3 (0 x -inf) is not
    # finite, and the key's rows of dK and dV are 0.
    for a, r in zip(got, ref):
        close(a[0], r[0])
    assert int((~torch.isfinite(got[0][0])).sum()) == 70 and float(got[1][0, 40].abs().max()) == 0.0
    # Slice 1: row 5 leaves nothing finite in its own row of dQ and in dK, and
    # its column of dV; row 9 nearly overflows, the others are ordinary.
    rows = [i for i in range(70) if i not in (5, 9)]
    close(got[0][1, rows], ref[0][1, rows])
    assert torch.equal(torch.isfinite(got[0][1, 5]), torch.isfinite(ref[0][1, 5].float()))
    assert torch.equal(torch.isfinite(got[1][1]), torch.isfinite(ref[1][1].float()))
    close(got[2][1], ref[2][1])
    # The others are what they were.
    for a, b in zip(got, clean):
        assert torch.equal(a[2:], b[2:])


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_fallback_cost(D, causal):
    # Every block is repeated: a few times the ordinary call, not ten.
    q, k, v, dO = _inputs(96, 1000, 1000, D, D)
    o, l = hip.attn_fwd(q, k, v, causal=causal)
    nan = torch.full_like(dO, math.nan)
    a, b = (median_us(lambda x=x: hip.attn_bwd(q, k, v, o, l, x, causal=causal)) for x in (dO, nan))
    assert b <= 6 * a, (a, b)


@pytest.mark.parametrize("BH,D", [(2, 64), (300, 64), (2, 128), (300, 128)])
@pytest.mark.parametrize("e", [-90, -100, -106, -112, -116, -120])
def test_small_magnitudes(BH, D, e):
    # Pieces of values below 2^-110 have fewer than 24 bits; gradients that small
    # come from the plain products.
    S = 300
    q, k, v, dO = _inputs(BH, S, S, D, D - e)
    o, l = hip.attn_fwd(q, k, v, causal=True)
    dO = (dO.double() * 2.0 ** e).float()
    got = hip.attn_bwd(q, k, v, o, l, dO, causal=True)
    torch.cuda.synchronize()
    for name, a, r in zip(("dQ", "dK", "dV"), got, _ref(q, k, v, dO, True)):
        assert float((a.double() - r).norm() / r.norm()) <= fp32_bar(2 * D + S), name


@pytest.mark.parametrize("BH,D", [(2, 64), (300, 64), (300, 128)])
def test_key_of_small_weight(BH, D):
    # A key 76 nats below the others has weights near 2^-110, and so have its
    # rows of dV and dK.
    S, drop = 300, 76.0
    q, k, v, dO = _inputs(BH, S, S, D, D)
    mask = torch.zeros(BH, S, S, device="cuda")
    mask[:, :, 7] = -drop
    o, l = hip.attn_fwd(q, k, v, attn_mask=mask)
    got = hip.attn_bwd(q, k, v, o, l, dO, attn_mask=mask)
    torch.cuda.synchronize()
    for a, r in list(zip(got, _ref(q, k, v, dO, False, mask=mask)))[1:]:
        a, r = a[:, 7].double(), r[:, 7]
        # exp2's argument is rounded at its size: drop * 2^-24 of each weight.
        assert float((a - r).norm() / r.norm()) <= drop * 2.0 ** -24
