"""Padded calls deal their slices over the XCDs, unpadded ones do not: with
every length at its full value the two must agree bit for bit, since the same
blocks do the same sums."""
import pytest
import torch

from gonn_amd import hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fp32", "bf16"])
@pytest.mark.parametrize("B,H", [(2, 4), (8, 3), (16, 2), (3, 5)])  # (3, 5): no whole slices per XCD
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal,mask", [(False, False), (True, False), (False, True)])
def test_full_lengths_match_unpadded(mode, B, H, D, causal, mask):
    Sq, Sk = (300, 300) if causal else (257, 323)
    g = torch.Generator().manual_seed(B * D)
    q, dO = (torch.randn(B, H, Sq, D, generator=g).cuda() for _ in range(2))
    k, v = (torch.randn(B, H, Sk, D, generator=g).cuda() for _ in range(2))
    am = torch.randn(B, Sq, Sk, generator=g).cuda() if mask else None
    out = []
    for kl in (None, torch.full((B,), Sk, dtype=torch.int32, device="cuda")):
        opt = dict(causal=causal, mode=mode, kv_len=kl, attn_mask=am)
        o, l = hip.attn_fwd(q, k, v, **opt)
        out.append((o, l, *hip.attn_bwd(q, k, v, o, l, dO, **opt)))
    torch.cuda.synchronize()
    for a, b in zip(*out):
        assert torch.equal(a, b)
