"""The reference order's batched prompt (exact.hip) against its own token steps.

A chunk computes each position with the token step's operations in the token
step's order, so the greedy tokens after a prompt have to be the ones that the
steps gave: a sequence is generated token by token from a one-token prompt (which
has no batch), and every prefix of it used as a prompt must continue it.  The
logits of a prompt must not depend on the scratch it finds, bit for bit;
tests/test_gpu_model.py compares them with the CPU's.
"""
import numpy as np
import pytest

from pokitlms_amd import synth as S
from pokitlms_amd import synth_model as SM

pytestmark = pytest.mark.gpu


def shape(head_dim=64, heads=8, kv_heads=4, attn=S.Q4_K, gate=S.Q4_K, down=S.Q6_K, **kw):
    return SM.Qwen3MoeShape(layers=2, hidden=512, heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                            experts=16, top_k=4, ffn=256, vocab=2048, attn_type=attn, gate_type=gate,
                            down_type=down, **kw)


@pytest.mark.parametrize("kw,lengths", (
    (dict(), (2, 3, 4, 5, 32, 33, 34, 35, 128, 129, 130, 131, 257, 511, 512, 513, 514, 600)),
    (dict(head_dim=128, heads=4, kv_heads=2, attn=S.Q6_K, gate=S.Q6_K, down=S.Q4_K), (3, 33, 130)),
    (dict(head_dim=256, heads=2, kv_heads=1, attn=S.Q5_K, gate=S.Q5_K, down=S.Q5_K), (3, 33, 130)),
), ids=("q4k", "q6k", "q5k"))
def test_prefixes_continue_the_steps(hip, kw, lengths):
    """Both sides of the chunk sizes (32 and 128), and of the KV window (512), past
    which the prompt goes on in steps."""
    from pokitlms_amd.model import Qwen3MoeModel
    m = shape(**kw)
    n_new = 4
    with Qwen3MoeModel.synthetic(hip, m, seed=31) as model:
        first = SM.prompt_tokens(7, 1, m.vocab)
        steps, _, _ = model.generate(first, max(lengths) + n_new)
        seq = np.concatenate((first, steps))
        for n in lengths:
            got, _, st = model.generate(seq[:n], n_new)
            assert st["prompt_tokens"] == n
            assert np.array_equal(got, seq[n:n + n_new]), n


def test_scratch_leaves_the_bits(hip):
    """The same prompts on the small scratch, on a grown one and on a used one."""
    from pokitlms_amd.model import Qwen3MoeModel
    m = shape()
    p = SM.prompt_tokens(3, 100, m.vocab)
    out = []
    with Qwen3MoeModel.synthetic(hip, m, seed=31) as model:
        out.append(model.generate(p[:20], 3, want_logits=True))
        out.append(model.generate(p, 3, want_logits=True))
        out.append(model.generate(p[:20], 3, want_logits=True))
        out.append(model.generate(p, 3, want_logits=True))
    for i in (0, 1):
        assert np.array_equal(out[i][0], out[i + 2][0])
        assert np.array_equal(out[i][1].view(np.uint32), out[i + 2][1].view(np.uint32))


@pytest.mark.parametrize("gtype", (S.Q4_0, S.Q4_1, S.Q5_0, S.Q5_1, S.Q8_0, S.Q2_K, S.Q3_K, S.Q4_K,
                                   S.Q5_K, S.Q6_K))
def test_formats(hip, gtype):
    """Every format of the chunk's matrices (experts: those the MoE block takes): 3 positions take their
    routes one by one (12 routes, 16 experts), 4 and more share the experts' rows, an
    odd number of inputs to a matrix ends in a single one."""
    from pokitlms_amd.model import Qwen3MoeModel
    m = shape()
    weights = Qwen3MoeModel.synthetic_weights(hip, m, 31)
    gen = S.rng(80 + gtype)
    names = {"attn_q": (512, 512, 0), "attn_k": (512, 256, 0), "attn_v": (512, 256, 0),
             "attn_output": (512, 512, 0), "ffn_gate_exps": (512, 256, 16),
             "ffn_up_exps": (512, 256, 16), "ffn_down_exps": (256, 512, 16)}
    if gtype in (S.Q5_0, S.Q5_1, S.Q2_K, S.Q3_K):
        names = {k: v for k, v in names.items() if v[2] == 0}
    for layer in range(m.layers):
        for name, (inn, out, ne) in names.items():
            key = f"blk.{layer}.{name}.weight"
            weights[key].release()
            rows = S.quant_matrix(gtype, out * max(ne, 1), inn, gen)
            blocks = rows.reshape(-1, S.BLOCK_BYTES[gtype])
            flip = gen.integers(0, 2, len(blocks), dtype=np.uint8) << 7
            for off in S.SCALE_OFFSETS[gtype]:  # half the blocks negated: weights around zero
                blocks[:, off + 1] ^= flip
            weights[key] = hip.upload(gtype, inn, out, rows, ne)
    with Qwen3MoeModel(hip, m, weights) as model:
        seen = set()
        for start in (9, 10, 11):
            first = SM.prompt_tokens(start, 1, m.vocab)
            steps, _, _ = model.generate(first, 48)
            seen.update(steps.tolist())
            seq = np.concatenate((first, steps))
            for n in (3, 4, 5, 6, 18, 41):
                got, _, _ = model.generate(seq[:n], 4)
                assert np.array_equal(got, seq[n:n + 4]), (start, n)
    assert len(seen) >= 3  # sequences worth comparing


@pytest.mark.parametrize("n", (1, 4, 40))
def test_non_finite_prompt_is_an_error(hip, n):
    """Non-finite router logits in a token step, in a chunk that takes its routes one by
    one (3 positions, 12 routes) and in one that groups them: every route falls to
    expert 0 and the call reports the error."""
    from pokitlms_amd.backend import HipError
    from pokitlms_amd.model import Qwen3MoeModel
    m = shape()
    weights = Qwen3MoeModel.synthetic_weights(hip, m, 31)
    bad = np.ones(m.hidden, np.float32)
    bad[7] = np.inf
    weights["blk.0.ffn_norm.weight"].release()
    weights["blk.0.ffn_norm.weight"] = hip.upload(S.F32, m.hidden, 1, bad)
    with Qwen3MoeModel(hip, m, weights) as model:
        for _ in range(2):
            with pytest.raises(HipError, match="non-finite"):
                model.generate(SM.prompt_tokens(3, n, m.vocab), 3)
