"""The prefill's expert GEMMs at the edges of their tiles and number formats.

Expert groups of exactly 1 to 130 rows (tiles hold 64 assignments, or 32 where
an expert has no more left; only 32 while that makes few workgroups, so once
with eight experts and once with sixty-four), every weight format, blocks whose scales are zero
(Q4_K keeps its accumulator in units of the block's d), and activations over a
wide range (each row is split into fp16 pairs under its own scale), through
pk_hip_moe_prefill against the CPU oracle.

Tolerance: both sides sum at most 1024 FP32 products twice; a random walk of
roundings is 1024**0.5 * 2**-24 = 1.9e-6 per sum and side, times about four where
quants and mins are summed apart: 1e-5 normwise.
"""
import numpy as np
import pytest

from pokitlms_amd import synth as S
from tests.conftest import normwise_rel

pytestmark = pytest.mark.gpu

TOL = 1e-5
GROUPS = (1, 31, 32, 33, 63, 64, 65, 130)
QUANT = (S.Q4_0, S.Q4_1, S.Q8_0, S.Q4_K, S.Q5_K, S.Q6_K)


def grouped_layer(gate_type, down_type, seed, repeat=1, hidden=512, ffn=256):
    """A top-1 layer whose expert e takes the tokens with x[e] large, and its
    tokens: GROUPS[e % 8] of them, shuffled."""
    groups = GROUPS * repeat
    E = len(groups)
    layer = S.moe_layer(seed=seed, hidden=hidden, experts=E, ffn=ffn, top_k=1,
                        gate_type=gate_type, up_type=gate_type, down_type=down_type)
    layer.router = np.zeros((E, hidden), np.float32)
    layer.router[np.arange(E), np.arange(E)] = 1.0
    g = S.rng(seed + 1)
    who = g.permutation(np.repeat(np.arange(E), groups))
    x = S.normal_f32(g, who.size * hidden).reshape(who.size, hidden)
    x[np.arange(who.size), who] = 30.0
    return layer, x, who


def check(hip, port, layer, x, who, tokens):
    h = hip.upload_moe_layer(layer)
    y, ids, _ = hip.moe_prefill(h, x)
    h.release()
    assert np.array_equal(ids[:, 0], who)
    blk = port.moe(layer)
    for t in tokens:
        cy = blk.forward(x[t])[0]
        assert np.all(np.isfinite(y[t])) and normwise_rel(y[t], cy) <= TOL, (t, who[t])


@pytest.mark.parametrize("gtype", QUANT, ids=lambda t: S.TYPE_NAMES[t])
def test_group_sizes(hip, port, gtype):
    layer, x, who = grouped_layer(gtype, gtype, 900 + gtype)
    check(hip, port, layer, x, who, range(0, who.size, 3))


@pytest.mark.parametrize("gtype", QUANT, ids=lambda t: S.TYPE_NAMES[t])
def test_group_sizes_many_experts(hip, port, gtype):
    """136 tiles of 32 rows times four workgroups each are more than 512, so tiles
    hold 64 rows."""
    layer, x, who = grouped_layer(gtype, gtype, 910 + gtype, repeat=8, hidden=1024, ffn=512)
    check(hip, port, layer, x, who, range(0, who.size, 23))


@pytest.mark.parametrize("gtype", (S.Q4_K, S.Q5_K), ids=lambda t: S.TYPE_NAMES[t])
def test_zero_and_spread_block_scales(hip, port, gtype):
    """d zero in the first, the last, or both blocks of a row, dmin zero or not,
    and d five decades apart between neighbouring blocks."""
    layer, x, who = grouped_layer(gtype, gtype, 950 + gtype, repeat=8, hidden=1024, ffn=512)
    for name in ("gate", "up", "down"):
        w = getattr(layer, name)
        b = w.reshape(-1, S.BLOCK_BYTES[gtype])
        n = np.arange(b.shape[0])
        b[n % 7 == 0, 0:2] = 0
        b[n % 5 == 1, 0:2] = 0
        b[n % 11 == 3, 2:4] = 0
        tiny = np.float16(1e-6).reshape(1).view(np.uint8)
        b[n % 6 == 2, 0:2] = tiny
    check(hip, port, layer, x, who, range(0, who.size, 29))


def centred_matrix(gtype, rows, cols, gen):
    """Q4_K or Q5_K rows whose weights lie around zero, as trained ones do: uniform
    quants, 6-bit scales 20 to 63, the mins the same numbers, dmin the mid quant times d."""
    b = gen.integers(0, 256, (rows * cols // 256, S.BLOCK_BYTES[gtype]), dtype=np.uint8)
    q, mid = (4.6, 7.5) if gtype == S.Q4_K else (9.2, 15.5)
    d = (0.02 / (q * 42.0) * gen.uniform(0.75, 1.25, len(b))).astype(np.float16)
    b[:, 0:2] = d.view(np.uint8).reshape(-1, 2)
    b[:, 2:4] = (d.astype(np.float32) * mid).astype(np.float16).view(np.uint8).reshape(-1, 2)
    sc = gen.integers(20, 64, (len(b), 8), dtype=np.uint8)
    b[:, 4:8] = b[:, 8:12] = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
    b[:, 12:16] = (sc[:, 4:] & 15) | ((sc[:, 4:] & 15) << 4)
    return b.reshape(-1)


def float64_error(hip, port, gtype, hidden, ffn, tokens, experts=4):
    """2-norm of the prefill's difference from float64 over the result's."""
    g = S.rng(980 + hidden + tokens)
    layer = S.moe_layer(seed=981, hidden=hidden, experts=experts, ffn=ffn, top_k=1, gate_type=gtype,
                        up_type=gtype, down_type=gtype)
    layer.gate, layer.up = (centred_matrix(gtype, experts * ffn, hidden, g) for _ in range(2))
    layer.down = centred_matrix(gtype, experts * hidden, ffn, g)
    x = S.normal_f32(g, tokens * hidden).reshape(tokens, hidden)
    h = hip.upload_moe_layer(layer)
    y, ids, _ = hip.moe_prefill(h, x)
    h.release()

    def w(data, e, rows, cols):
        n = len(data) // experts
        f = port.dequantize_row(gtype, data[e * n:(e + 1) * n], rows * cols)
        return f.astype(np.float64).reshape(rows, cols)

    want = np.zeros((tokens, hidden))
    for e in range(experts):
        t = ids[:, 0] == e
        xe = x[t].astype(np.float64)
        gate, up = xe @ w(layer.gate, e, ffn, hidden).T, xe @ w(layer.up, e, ffn, hidden).T
        want[t] = (gate / (1.0 + np.exp(-gate)) * up) @ w(layer.down, e, hidden, ffn).T
    return float(np.linalg.norm(y - want) / np.linalg.norm(want))


@pytest.mark.parametrize("tokens", (20, 300))  # 32-row tiles, 64-row tiles
@pytest.mark.parametrize("hidden,bound", ((512, 2.87e-7), (1024, 3.35e-7), (2048, 4.1e-7)))
def test_q5_k_error_against_float64(hip, port, hidden, bound, tokens):
    """The bounds are what GEMMs on three exact bf16 parts of x, with one FP32 sum per
    32 values, have on these inputs; two fp16 halves must not be further off (2.7e-7,
    3.1e-7 and 3.5e-7; one sum of both halves over 256 values: 3.2e-7, 3.4e-7, 3.8e-7)."""
    err = float64_error(hip, port, S.Q5_K, hidden, 512, tokens)
    print(f"Q5_K hidden {hidden} tokens {tokens}: {err:.3g}")
    assert err <= bound


def test_activation_range(hip, port):
    """Rows scaled by 1e-12 to 1e12, and values down to 2^-27 of their row's maximum; a
    zero row, and one so small that its scale is the smallest there is."""
    layer, x, who = grouped_layer(S.Q4_K, S.Q6_K, 970)
    x[:, 64:] *= np.float32(2.0) ** -np.arange(0, 28).repeat(16).astype(np.float32)
    x *= (np.float32(10.0) ** (np.arange(who.size) % 25 - 12).astype(np.float32))[:, None]
    x[0] = 0.0  # every logit equal: the first expert
    who[0] = 0
    x[2] = x[2] / np.abs(x[2]).max() * np.float32(1e-35)
    layer.router *= np.float32(1e-3)
    check(hip, port, layer, x, who, range(0, who.size, 2))


@pytest.mark.parametrize("down_type", QUANT, ids=lambda t: S.TYPE_NAMES[t])
@pytest.mark.parametrize("ratio", (22, 24, 25, 26, 28))
def test_chunks_far_below_their_row(hip, port, down_type, ratio):
    """Activations whose first 32 values are 2^ratio times the others (from Q8_0 up rows
    of such scales) and whose down weights there are zero: what is left comes from the
    small chunks alone.  Each of a value's two halves is rounded to 2^-39 of the row's
    maximum, together 2^(ratio - 38) of the small chunks' maximum; a value is about half
    of that, and quants and mins summed apart take both: 2^(ratio - 36).  One expert has
    20 rows, one 50."""
    hidden, ffn = 512, 256
    layer = S.moe_layer(seed=990, hidden=hidden, experts=2, ffn=ffn, top_k=1, gate_type=S.Q8_0,
                        up_type=S.Q8_0, down_type=down_type)
    layer.router = np.zeros((2, hidden), np.float32)
    layer.router[:, 2:4] = np.eye(2, dtype=np.float32)
    gate = np.zeros((2 * ffn, hidden // 32, 34), np.uint8)
    gate[:, 0, 0:2] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)
    gate[:, 0, 2] = 1  # g = x[0]
    layer.gate = gate.reshape(-1)
    up = layer.up.reshape(2, ffn, hidden // 32, 34)
    for rows, d in ((up[:, :32], 2.0 ** 9), (up[:, 32:], 2.0 ** (9 - ratio))):
        rows[..., 0:2] = np.frombuffer(np.float16(d).tobytes(), np.uint8)
    down = layer.down.reshape(2 * hidden, -1, S.BLOCK_BYTES[down_type])[:, 0]  # each row's first block
    if down_type in (S.Q4_K, S.Q5_K):
        down[:, 4] &= 0xC0  # scale and min of the first group
        down[:, 8] &= 0xC0
    elif down_type == S.Q6_K:
        down[:, 192:194] = 0
    else:
        down[:, 0:4 if down_type == S.Q4_1 else 2] = 0
    who = np.repeat((0, 1), (20, 50))
    x = S.normal_f32(S.rng(991), who.size * hidden).reshape(who.size, hidden)
    x[:, 0] = 6.0
    x[:, 2:4] = 0.0
    x[np.arange(who.size), 2 + who] = 30.0
    h = hip.upload_moe_layer(layer)
    y, ids, _ = hip.moe_prefill(h, x)
    h.release()
    assert np.array_equal(ids[:, 0], who)
    blk = port.moe(layer)
    for t in range(0, who.size, 3):
        assert normwise_rel(y[t], blk.forward(x[t])[0]) <= max(TOL, 2.0 ** (ratio - 36)), (t, who[t])
