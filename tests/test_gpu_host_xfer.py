"""The host entry points' transfers: chunk edges, padded head dims and more
callers at once than there are pinned lanes give exactly what the device entry
gives on the same values."""
import math
import threading

import numpy as np
import pytest
import torch

from gonn_amd import hip

pytestmark = pytest.mark.gpu


def _case(BH, S, d, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(BH * S * d) for _ in range(3)]


def _device(x, BH, S, d):
    dp = 64 if d <= 64 else 128
    t = [torch.nn.functional.pad(torch.from_numpy(a).float().reshape(BH, S, d), (0, dp - d)).cuda()
         for a in x]
    o, l = hip.attn_fwd(*t, causal=True, scale=1 / math.sqrt(d))
    torch.cuda.synchronize()
    return o[..., :d].double().cpu().numpy().reshape(-1), l.double().cpu().numpy().reshape(-1)


# A chunk is 1 MiB: 4096 rows of 64 floats, 2048 of 128, 262144 of the LSE.
@pytest.mark.parametrize("BH,S,d", [(1, 1, 1), (2, 2047, 64), (2, 2048, 64), (3, 1366, 64),
                                    (1, 4097, 128), (5, 1999, 40), (3, 2050, 100)])
def test_chunk_edges(BH, S, d):
    x = _case(BH, S, d, S)
    O, L = hip.FlashAttnF64Fwd(*x, BH, S, d, 1 / math.sqrt(d), True)
    o, l = _device(x, BH, S, d)
    assert np.array_equal(O, o) and np.array_equal(L, l)


def test_many_callers():
    BH, S, d, n = 4, 3000, 64, 10  # more than there are pinned lanes for
    xs = [_case(BH, S, d, i) for i in range(n)]
    want = [_device(x, BH, S, d) for x in xs]
    got = [None] * n
    start = threading.Barrier(n)

    def call(i):
        start.wait()
        for _ in range(3):
            got[i] = hip.FlashAttnF64Fwd(*xs[i], BH, S, d, 1 / math.sqrt(d), True)

    ts = [threading.Thread(target=call, args=(i,)) for i in range(n)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for (O, L), (o, l) in zip(got, want):
        assert np.array_equal(O, o) and np.array_equal(L, l)


def test_lanes_come_and_go():
    # Large calls take eight pinned lanes, small ones one; lanes that no call
    # needed for a while are freed, and made again when one does.
    big, small = (4, 3000, 64), (1, 20, 64)
    x, y = _case(*big, 1), _case(*small, 2)
    want, wanty = _device(x, *big), _device(y, *small)

    def check(c, shape, w):
        O, L = hip.FlashAttnF64Fwd(*c, *shape, 1 / math.sqrt(shape[2]), True)
        assert np.array_equal(O, w[0]) and np.array_equal(L, w[1])

    for _ in range(2):
        check(x, big, want)
        for _ in range(150):
            check(y, small, wanty)
        ts = [threading.Thread(target=check, args=(x, big, want)) for _ in range(3)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    check(x, big, want)
