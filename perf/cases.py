"""The attention work this library is asked to do, as timed cases.

Each case is one call (or one forward and backward) through the public entry
points of gonn_amd.hip, at sizes of this repository's benchmark and tests or
of common transformer shapes. The kinds:

  fwd     hip.attn_fwd on device tensors, O and LSE
  train   hip.attn_fwd and hip.attn_bwd: O, LSE, dQ, dK, dV
  decode  hip.attn_decode: one query per (b, h) over a bf16 KV cache
  attend  KVCache.attend_causal: the last T cached positions of every sequence
          attend the cache (a chunk of a prompt, or a few tokens of one step)
  mha     DeviceMHA.forward_dev: projections, core and output projection with
          the weights in HBM, fp64 in and out
  seam    FlashAttnF64Fwd and FlashAttnF64Bwd on host fp64 arrays, the calls
          GoNN's autograd node makes

listed() names the cases, draw(rng) gives another one of the same ranges.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from gonn_amd import hip


def _fwd(name, mode, B, H, Sq, Sk, D, causal, pad=False, mask=False, kind="fwd"):
    return {"name": name, "kind": kind, "mode": mode, "B": B, "H": H, "Sq": Sq, "Sk": Sk, "D": D,
            "causal": causal, "pad": pad, "mask": mask}


def listed():
    return [
        # A prompt of 4096 tokens through one layer of a 32-head model: the
        # headline workload, fp32 tensors on the bf16 matrix cores.
        _fwd("prefill_bf16", "bf16", 4, 32, 4096, 4096, 128, True),
        # A BERT-base layer over a full batch, in the default fp32 mode.
        _fwd("encoder_fp32", "fp32", 8, 12, 1024, 1024, 64, False),
        # The smallest layer the repository's configurations name (2 x 128
        # tokens, 4 heads): launches and host time count here.
        _fwd("small_fp32", "fp32", 2, 4, 128, 128, 64, True),
        # One training step of a long-context layer.
        _fwd("train_long_bf16", "bf16", 2, 16, 8192, 8192, 128, True, kind="train"),
        # A decoder-only training step in the default fp32 mode.
        _fwd("train_causal_fp32", "fp32", 4, 12, 1024, 1024, 64, True, kind="train"),
        # Training with an additive (B, S, S) mask (packed documents).
        _fwd("train_masked_bf16", "bf16", 8, 12, 1024, 1024, 64, False, mask=True, kind="train"),
        # A decoder's cross-attention over padded memories, odd lengths, in
        # the default fp32 mode.
        _fwd("train_cross_fp32", "fp32", 4, 16, 500, 2001, 128, False, pad=True, kind="train"),
        # Serving: 64 ragged sequences, one new token each.
        {"name": "decode_batch", "kind": "decode", "B": 64, "H": 32, "Lmax": 8192, "lo": 512, "D": 128},
        # Serving one user: one new token, latency counts.
        {"name": "decode_single", "kind": "decode", "B": 1, "H": 32, "Lmax": 4096, "lo": 3001, "D": 128},
        # Chunked prefill: 256 prompt tokens per sequence over a filled cache.
        {"name": "attend_chunk", "kind": "attend", "B": 4, "H": 32, "Lmax": 4096, "lo": 2048,
         "T": 256, "D": 128},
        # A resident layer at BERT-large width.
        {"name": "mha_layer", "kind": "mha", "B": 4, "T": 512, "E": 1024, "H": 16, "causal": True},
        # GoNN's published fused shape (BH 32, S 1024, d 64): its training
        # calls on host fp64 data.
        {"name": "seam_f64_host", "kind": "seam", "BH": 32, "S": 1024, "d": 64, "causal": True,
         "mode": "fp32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fwd", "fwd", "train", "train", "decode", "attend", "mha", "seam"])
    if kind in ("fwd", "train"):
        mode = rng.choice(["fp32", "bf16"])
        D = rng.choice([64, 128])
        cross = rng.random() < 0.25
        Sq = _log_int(rng, 16, 4096 if mode == "fp32" else 8192)
        Sk = _log_int(rng, 16, 4096 if mode == "fp32" else 8192) if cross else Sq
        # Heads over the batch: as many as keep the work below the largest
        # listed case's.
        top = (0.1 if mode == "fp32" else 1.0) * 2.0e11 / (float(Sq) * Sk * D)
        BH = max(1, min(_log_int(rng, 1, 256), int(top)))
        H = max(1, min(rng.choice([4, 8, 12, 16, 32]), BH))
        opt = rng.random()
        big_mask = (BH // H) * Sq * Sk > 1 << 27
        return _fwd(None, mode, max(1, BH // H), H, Sq, Sk, D, rng.random() < 0.5,
                    pad=opt < 0.25, mask=opt > 0.85 and not big_mask, kind=kind) | {"name": ""}
    if kind == "decode":
        Lmax = _log_int(rng, 128, 8192)
        return {"name": "", "kind": kind, "B": _log_int(rng, 1, 64), "H": rng.choice([8, 16, 32]),
                "Lmax": Lmax, "lo": rng.randint(max(1, Lmax // 8), Lmax), "D": rng.choice([64, 128])}
    if kind == "attend":
        Lmax = _log_int(rng, 512, 8192)
        T = _log_int(rng, 1, 512)
        B = _log_int(rng, 1, 16 if T <= 16 else 4)
        return {"name": "", "kind": kind, "B": B, "H": rng.choice([8, 16, 32]), "Lmax": Lmax,
                "lo": rng.randint(min(T, Lmax), Lmax), "T": min(T, Lmax), "D": rng.choice([64, 128])}
    if kind == "mha":
        H = rng.choice([4, 8, 12, 16])
        return {"name": "", "kind": kind, "B": rng.randint(1, 8), "T": _log_int(rng, 16, 512),
                "E": H * rng.choice([32, 64]), "H": H, "causal": rng.random() < 0.5}
    S = _log_int(rng, 64, 2048)
    return {"name": "", "kind": "seam", "BH": max(1, min(64, 32768 // S)), "S": S,
            "d": rng.choice([32, 64, 128]), "causal": rng.random() < 0.5,
            "mode": rng.choice(["fp32", "bf16", "f64"])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _lens(case, seed, lo, hi, n):
    return np.random.default_rng(seed + 7).integers(lo, hi + 1, n).astype(np.int32)


def _attn_inputs(case, seed):
    g = _gen(seed)
    B, H, Sq, Sk, D = (case[x] for x in ("B", "H", "Sq", "Sk", "D"))

    def t(*s):
        return torch.randn(*s, generator=g, device="cuda")
    q, k, v = t(B, H, Sq, D), t(B, H, Sk, D), t(B, H, Sk, D)
    dO = t(B, H, Sq, D) if case["kind"] == "train" else None
    kv_len = None
    if case["pad"]:
        kv_len = torch.from_numpy(_lens(case, seed, max(1, Sk // 2), Sk, B)).cuda()
    mask = None
    if case["mask"]:
        # Packed documents: a token sees the tokens of its own document, plus
        # a small additive bias.
        doc = torch.sort(torch.randint(0, 4, (B, max(Sq, Sk)), generator=g, device="cuda"), dim=1)[0]
        doc[:, 0] = 0
        same = doc[:, :Sq, None] == doc[:, None, :Sk]
        same[:, :, 0] = True
        mask = torch.where(same, 0.25 * t(B, Sq, Sk), torch.tensor(-1e30, device="cuda"))
    return q, k, v, dO, kv_len, mask


def _mha_inputs(case, seed):
    rng = np.random.default_rng(seed)
    E, B, T = case["E"], case["B"], case["T"]
    W = [rng.standard_normal((E, E)) / math.sqrt(E) for _ in range(4)]
    b = [0.1 * rng.standard_normal(E) for _ in range(4)]
    return W, b, rng.standard_normal((B, T, E))


def _seam_inputs(case, seed):
    rng = np.random.default_rng(seed)
    n = case["BH"] * case["S"] * case["d"]
    return [rng.standard_normal(n) for _ in range(4)]


def _cache_inputs(case, seed):
    g = _gen(seed)
    B, H, L, D = (case[x] for x in ("B", "H", "Lmax", "D"))

    def t(*s):
        return torch.randn(*s, generator=g, device="cuda", dtype=torch.bfloat16)
    k, v = t(B, H, L, D), t(B, H, L, D)
    lens = _lens(case, seed, case["lo"], L, B)
    nq = case.get("T", 1)
    q = torch.randn(B, H, nq, D, generator=g, device="cuda")
    return q, k, v, lens


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("fwd", "train"):
        q, k, v, dO, kv_len, mask = _attn_inputs(case, seed)
        return {"case": case, "q": q, "k": k, "v": v, "dO": dO, "kv_len": kv_len, "mask": mask}
    if kind == "decode":
        q, k, v, lens = _cache_inputs(case, seed)
        return {"case": case, "q": q[:, :, 0].bfloat16().contiguous(), "k": k, "v": v,
                "lens": torch.from_numpy(lens).cuda()}
    if kind == "attend":
        q, k, v, lens = _cache_inputs(case, seed)
        cache = hip.KVCache(case["B"], case["H"], case["Lmax"], case["D"])
        cache.append(k, v, counts=lens)
        return {"case": case, "q": q, "cache": cache}
    if kind == "mha":
        W, b, x = _mha_inputs(case, seed)
        layer = hip.DeviceMHA(case["E"], case["H"], W[0], b[0], W[1], b[1], W[2], b[2], W[3], b[3])
        ws = torch.empty(layer.workspace_bytes(case["B"], case["T"], case["T"]), dtype=torch.uint8,
                         device="cuda")
        return {"case": case, "layer": layer, "x": torch.from_numpy(x).cuda(), "ws": ws}
    return {"case": case, "host": _seam_inputs(case, seed)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("fwd", "train"):
        opt = dict(causal=case["causal"], mode=case["mode"], kv_len=state["kv_len"],
                   attn_mask=state["mask"])
        q, k, v = state["q"], state["k"], state["v"]
        o, lse = hip.attn_fwd(q, k, v, **opt)
        if kind == "fwd":
            return o, lse
        return (o, lse) + tuple(hip.attn_bwd(q, k, v, o, lse, state["dO"], **opt))
    if kind == "decode":
        return hip.attn_decode(state["q"], state["k"], state["v"], state["lens"])
    if kind == "attend":
        return state["cache"].attend_causal(state["q"])
    if kind == "mha":
        x = state["x"]
        hip.SetAttnMode("fp32")
        return state["layer"].forward_dev(x, x, x, causal=case["causal"], ws=state["ws"])
    hip.SetAttnMode(case["mode"])
    Q, K, V, dO = state["host"]
    BH, S, d = case["BH"], case["S"], case["d"]
    scale = 1.0 / math.sqrt(d)
    O, L = hip.FlashAttnF64Fwd(Q, K, V, BH, S, d, scale, case["causal"])
    return (O, L) + tuple(hip.FlashAttnF64Bwd(Q, K, V, O, L, dO, BH, S, d, scale, case["causal"]))


# ---------------------------------------------------------------------------
# work and tolerances
# ---------------------------------------------------------------------------
def _pairs(Sq, Sk, causal):
    if not causal:
        return float(Sq) * Sk
    n = min(Sq, Sk)
    return n * (n + 1) / 2.0 + float(max(0, Sq - Sk)) * Sk


def work(case):
    kind = case["kind"]
    if kind in ("fwd", "train"):
        B, H, Sq, Sk, D = (case[x] for x in ("B", "H", "Sq", "Sk", "D"))
        BH = B * H
        keys = 0.75 * Sk if case["pad"] else Sk  # mean of the drawn lengths
        fl = 4.0 * BH * D * _pairs(Sq, int(keys), case["causal"])
        by = 4.0 * BH * (2 * Sq * D + 2 * keys * D + Sq)
        if case["mask"]:
            by += 4.0 * B * Sq * Sk
        if kind == "train":  # + dO in, dQ, dK, dV out
            fl *= 3.5
            by += 4.0 * BH * (2 * Sq * D + 2 * Sk * D)
        return {"bytes": by, "flops": fl}
    if kind in ("decode", "attend"):
        B, H, D, T = case["B"], case["H"], case["D"], case.get("T", 1)
        mean = (case["lo"] + case["Lmax"]) / 2.0
        rows = B * H * mean
        return {"bytes": rows * D * 4 + B * H * T * D * (8 if kind == "attend" else 6),
                "flops": 4.0 * D * B * H * T * max(1.0, mean - (T - 1) / 2.0)}
    if kind == "mha":
        B, T, E = case["B"], case["T"], case["E"]
        return {"bytes": 8.0 * (2 * B * T * E + 4 * E * E),
                "flops": 8.0 * B * T * E * E + 4.0 * B * E * _pairs(T, T, case["causal"])}
    BH, S, d = case["BH"], case["S"], case["d"]
    return {"bytes": 8.0 * BH * (12.0 * S * d + 2 * S),
            "flops": 14.0 * BH * d * _pairs(S, S, case["causal"])}


def tolerance(case):
    # About four times the error against 64 bits measured over these ranges.
    kind = case["kind"]
    if kind == "seam" and case["mode"] == "f64":
        return {"rel": 4e-15}
    if kind in ("fwd", "train", "seam"):
        return {"rel": 2e-2 if case["mode"] == "bf16" else 5e-6}
    return {"rel": 2e-6}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _attn64(q, k, v, scale, allow, bias, dO=None):
    """One (b, h) slice: allow (Sq, Sk) bool or None, bias (Sq, Sk) or None."""
    s = (q @ k.T) * scale
    if bias is not None:
        s = s + bias
    if allow is not None:
        s = s.masked_fill(~allow, -math.inf)
    lse = torch.logsumexp(s, dim=-1)
    p = torch.exp(s - lse[:, None])
    o = p @ v
    if dO is None:
        return o, lse
    ds = p * (dO @ v.T - (dO * o).sum(-1, keepdim=True)) * scale
    return o, lse, ds @ k, ds.T @ q, p.T @ dO


def _allow(Sq, Sk, causal, n=None):
    if not causal and (n is None or n == Sk):
        return None
    j = torch.arange(Sk, device="cuda")[None, :]
    a = torch.ones(Sq, Sk, dtype=torch.bool, device="cuda")
    if causal:
        a &= j <= torch.arange(Sq, device="cuda")[:, None]
    if n is not None:
        a &= j < n
    return a


def exact(case, seed):
    kind = case["kind"]
    if kind in ("fwd", "train"):
        q, k, v, dO, kv_len, mask = _attn_inputs(case, seed)
        B, H, Sq, Sk, D = (case[x] for x in ("B", "H", "Sq", "Sk", "D"))
        out = [torch.empty(q.shape, dtype=torch.float64, device="cuda"),
               torch.empty((B * H, Sq), dtype=torch.float64, device="cuda")]
        if dO is not None:
            out += [torch.empty(x.shape, dtype=torch.float64, device="cuda") for x in (q, k, v)]
        lens = kv_len.cpu().tolist() if kv_len is not None else [None] * B
        for b in range(B):
            allow = _allow(Sq, Sk, case["causal"], lens[b])
            bias = mask[b].double() if mask is not None else None
            for h in range(H):
                r = _attn64(q[b, h].double(), k[b, h].double(), v[b, h].double(),
                            1.0 / math.sqrt(D), allow, bias,
                            dO[b, h].double() if dO is not None else None)
                out[0][b, h] = r[0]
                out[1][b * H + h] = r[1]
                for o, x in zip(out[2:], r[2:]):
                    o[b, h] = x
        return tuple(out)
    if kind in ("decode", "attend"):
        q, k, v, lens = _cache_inputs(case, seed)
        if kind == "decode":
            q = q.bfloat16()
        B, H, D = case["B"], case["H"], case["D"]
        T = q.shape[2]
        out = torch.empty(B, H, T, D, dtype=torch.float64, device="cuda")
        for b in range(B):
            n = int(lens[b])
            allow = torch.arange(n, device="cuda")[None, :] <= \
                torch.arange(n - T, n, device="cuda")[:, None]
            for h in range(H):
                out[b, h] = _attn64(q[b, h].double(), k[b, h, :n].double(), v[b, h, :n].double(),
                                    1.0 / math.sqrt(D), allow, None)[0]
        return out[:, :, 0].contiguous() if kind == "decode" else out
    if kind == "mha":
        W, bias, x = _mha_inputs(case, seed)
        W = [torch.from_numpy(w).cuda() for w in W]
        bias = [torch.from_numpy(w).cuda() for w in bias]
        x = torch.from_numpy(x).cuda()
        B, T, E, H = case["B"], case["T"], case["E"], case["H"]
        D = E // H
        q, k, v = ((x @ W[i].T + bias[i]).reshape(B, T, H, D).transpose(1, 2) for i in range(3))
        ctx = torch.empty(B, T, H, D, dtype=torch.float64, device="cuda")
        allow = _allow(T, T, case["causal"])
        for b in range(B):
            for h in range(H):
                ctx[b, :, h] = _attn64(q[b, h], k[b, h], v[b, h], 1.0 / math.sqrt(D), allow, None)[0]
        return ctx.reshape(B, T, E) @ W[3].T + bias[3]
    BH, S, d = case["BH"], case["S"], case["d"]
    x = [torch.from_numpy(a).cuda().reshape(BH, S, d) for a in _seam_inputs(case, seed)]
    allow = _allow(S, S, case["causal"])
    parts = [_attn64(x[0][i], x[1][i], x[2][i], 1.0 / math.sqrt(d), allow, None, x[3][i])
             for i in range(BH)]
    return tuple(torch.stack([p[j] for p in parts]).reshape(-1).cpu().numpy() for j in range(5))
