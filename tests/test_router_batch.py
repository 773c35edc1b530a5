"""The batched prefill router: its rounding bound, and its tiles.

The bound is restated here from the text of k_router_batch (eight ranges of K,
runs of 16 products, |prefix| at both ends of a run and two norms) and checked
against the CPU's serial float32 sum; the kernel's sums are checked through
pk_hip_moe_prefill, whose ids and route weights must be the decode path's.
"""
import math

import numpy as np
import pytest

from pokitlms_amd import synth as S

OMEGA = np.array([8, 7, 6, 5, 4, 3, 2, 1, 0, 1, 2, 3, 4, 5, 6, 7], np.float64) + 1.001


def batch_bound(w, x):
    n = w.size
    p = (w * x).astype(np.float32).astype(np.float64)  # the CPU's rounded products
    q, off = 0.0, 0.0
    for r in range(8):
        pre = np.cumsum(p[r * n // 8:(r + 1) * n // 8])[15::16]
        q += 16.0 * np.abs(pre).sum() - 8.0 * abs(pre[-1]) + n / 8 * abs(off)
        off += pre[-1]
    om = np.tile(OMEGA, n // 16)
    norms = math.sqrt(float((x.astype(np.float64) ** 2).sum()) *
                      float(((om * w.astype(np.float64)) ** 2).sum()))
    return (q + norms) * (2.0 ** -24 * (1.0 + 2.0 ** -10) + 2.0 ** -39)


def serial_error(w, x):
    p = w * x
    return abs(float(np.cumsum(p, dtype=np.float32)[-1]) - math.fsum(p.astype(np.float64)))


@pytest.mark.parametrize("n", (512, 2048, 3072))
def test_bound_holds(n):
    g = np.random.default_rng(n)
    for trial in range(120):
        w = (g.standard_normal(n) * 0.02).astype(np.float32)
        x = g.standard_normal(n).astype(np.float32)
        if trial % 4 == 1:
            x *= np.exp(2.0 * g.standard_normal(n)).astype(np.float32)  # heavy tails
        elif trial % 4 == 2:
            x = np.sign(w) * np.abs(x)  # one sign: the prefixes only grow
        elif trial % 4 == 3:
            w[n // 2:], x[n // 2:] = -w[:n // 2], x[:n // 2]  # cancels to zero
        assert serial_error(w.astype(np.float32), x.astype(np.float32)) <= batch_bound(w, x), trial


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,experts,tokens", ((512, 128, 2049), (512, 16, 7), (512, 33, 17),
                                                   (1024, 31, 9), (3072, 64, 40), (4096, 20, 10)))
def test_routes_equal_decode(hip, hidden, experts, tokens):
    """2049 tokens x 128 rows take the 16 x 32 tile, the others 8 x 16; partly
    filled tiles both ways; near-equal rows make rankings the coarse bound leaves
    open."""
    layer = S.moe_layer(seed=hidden + experts, hidden=hidden, experts=experts, ffn=256, top_k=4)
    layer.router[1::3] = layer.router[0::3][:layer.router[1::3].shape[0]] * np.float32(1 + 2e-6)
    h = hip.upload_moe_layer(layer)
    x = S.normal_f32(S.rng(tokens), tokens * hidden).reshape(tokens, hidden)
    _, ids, probs = hip.moe_prefill(h, x)
    for t in range(0, tokens, 1 if tokens < 100 else 41):
        _, di, dp = hip.moe_decode(h, x[t])
        assert np.array_equal(ids[t], di) and np.array_equal(probs[t].view(np.uint32), dp.view(np.uint32)), t
    h.release()
