"""The fast mode's batched prompt (prompt.hip) against the reference-order kernels.

The reference-order model is the CPU's bits (tests/test_gpu_model.py); the fast
mode is within FP32 reassociation of it, which two layers carry to about 5e-5
normwise in the logits, and to 1e-3 where a rounding decides a router near-tie
(the bound tests/test_gpu_model.py holds every depth to).  Prompt lengths on both
sides of the shortest batch (5 positions, then the last token as a step), of a
32-row tile's end, of one chunk, and of the KV window; a model wide enough for the
projections' 64-row tiles; every attention format the batch takes.
"""
import numpy as np
import pytest

from pokitlms_amd import synth as S
from pokitlms_amd import synth_model as SM
from pokitlms_amd.backend import HipError
from tests.conftest import normwise_rel

pytestmark = pytest.mark.gpu


def shape(head_dim=64, heads=8, kv_heads=4, attn=S.Q4_K, gate=S.Q4_K, down=S.Q6_K, **kw):
    return SM.Qwen3MoeShape(layers=2, hidden=512, heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                            experts=16, top_k=4, ffn=256, vocab=2048, attn_type=attn, gate_type=gate,
                            down_type=down, **kw)


def generate(hip, m, prompt, n_new, reference_order):
    from pokitlms_amd.model import Qwen3MoeModel
    with Qwen3MoeModel.synthetic(hip, m, seed=31, reference_order=reference_order) as model:
        return model.generate(prompt, n_new, want_logits=True)


def compare(hip, m, n, n_new=4):
    prompt = SM.prompt_tokens(n, n, m.vocab)
    want, wl, _ = generate(hip, m, prompt, n_new, True)
    got, gl, st = generate(hip, m, prompt, n_new, False)
    assert st["prompt_tokens"] == n
    assert normwise_rel(gl, wl) <= 1e-3, n
    assert np.array_equal(got, want), n


@pytest.mark.parametrize("n", (1, 5, 6, 7, 33, 34, 65, 66, 130, 513, 530, 1100))
def test_prompt_lengths(hip, n):
    """513 positions fill the window (512 in one chunk and a step); beyond it the
    ring wraps under token steps."""
    compare(hip, shape(), n)


@pytest.mark.parametrize("kw", (dict(head_dim=128, heads=4, kv_heads=2, attn=S.Q6_K, gate=S.Q6_K, down=S.Q4_K),
                                dict(head_dim=256, heads=2, kv_heads=1, attn=S.Q5_K, gate=S.Q5_K, down=S.Q5_K),
                                dict(head_dim=128, heads=16, kv_heads=4)),
                         ids=("planar", "q5k", "wide"))
def test_prompt_formats(hip, kw):
    """q, k and v as three GEMMs (a planar format) and as one; 64- to 256-wide heads;
    q wider than the hidden state."""
    for n in (40, 200):
        compare(hip, shape(**kw), n)


@pytest.mark.parametrize("n", (449, 450, 498, 513))
def test_prompt_wide_projections(hip, n):
    """q, k and v of 9216 rows: 449 positions and more make too many 32-row tiles for the
    chip, so the projections take 64-row ones (the last one short, or whole at 512)."""
    compare(hip, SM.Qwen3MoeShape(layers=1, hidden=512, heads=64, kv_heads=4, head_dim=128, experts=16,
                                  top_k=4, ffn=256, vocab=2048), n)


@pytest.mark.parametrize("gtype", (S.Q4_0, S.Q4_1, S.Q8_0), ids=lambda t: S.TYPE_NAMES[t])
def test_prompt_attention_formats(hip, gtype):
    """The projections in the formats the synthetic model has no recipe for."""
    from pokitlms_amd.model import Qwen3MoeModel
    m = shape()
    out = []
    for reference_order in (True, False):
        weights = Qwen3MoeModel.synthetic_weights(hip, m, 31)
        gen = S.rng(70 + gtype)
        for layer in range(m.layers):
            for name, inn, rows in (("attn_q", 512, 512), ("attn_k", 512, 256), ("attn_v", 512, 256),
                                    ("attn_output", 512, 512)):
                data = S.quant_matrix(gtype, rows, inn, gen)
                blocks = data.reshape(-1, S.BLOCK_BYTES[gtype])
                flip = gen.integers(0, 2, len(blocks), dtype=np.uint8) << 7
                for off in S.SCALE_OFFSETS[gtype]:  # half the blocks negated: weights around zero
                    blocks[:, off + 1] ^= flip
                key = f"blk.{layer}.{name}.weight"
                weights[key].release()
                weights[key] = hip.upload(gtype, inn, rows, data)
        with Qwen3MoeModel(hip, m, weights, reference_order) as model:
            out.append([model.generate(SM.prompt_tokens(n, n, m.vocab), 4, want_logits=True)
                        for n in (8, 40, 200)])
    for (want, wl, _), (got, gl, _) in zip(*out):
        assert normwise_rel(gl, wl) <= 1e-3
        assert np.array_equal(got, want)


def test_prompt_narrow_kv_takes_steps(hip):
    """kv_heads * head_dim below one 256-row block of the GEMM: token steps."""
    compare(hip, shape(head_dim=64, heads=8, kv_heads=2), 40)


def test_repeat_and_second_prompt(hip):
    """The kept scratch and the ring carry nothing over between calls."""
    from pokitlms_amd.model import Qwen3MoeModel
    m = shape()
    a, b = SM.prompt_tokens(1, 100, m.vocab), SM.prompt_tokens(2, 300, m.vocab)
    with Qwen3MoeModel.synthetic(hip, m, seed=31, reference_order=False) as model:
        first = model.generate(a, 4, want_logits=True)
        model.generate(b, 4)
        again = model.generate(a, 4, want_logits=True)
    assert np.array_equal(first[0], again[0])
    assert np.array_equal(first[1].view(np.uint32), again[1].view(np.uint32))


def test_non_finite_prompt_is_an_error(hip):
    from pokitlms_amd.model import Qwen3MoeModel
    m = shape()
    weights = Qwen3MoeModel.synthetic_weights(hip, m, 31)
    bad = np.ones(m.hidden, np.float32)
    bad[7] = np.inf
    weights["blk.0.ffn_norm.weight"].release()
    weights["blk.0.ffn_norm.weight"] = hip.upload(S.F32, m.hidden, 1, bad)
    with Qwen3MoeModel(hip, m, weights, False) as model:
        with pytest.raises(HipError, match="non-finite"):
            model.generate(SM.prompt_tokens(3, 40, m.vocab), 2)
