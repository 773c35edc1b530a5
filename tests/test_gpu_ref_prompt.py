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
