"""The calls whose speed this repository is judged by, and how each is made.

Every case goes through the Python surface of the library (``HipBackend``,
``Qwen3MoeModel``) as a user's program does: weights uploaded once and kept,
one call per pass.  Kinds:

* ``linear``: y = W . x for a run of ``count`` matrices of one type and shape
  (a model's projections, one after the other), 1 to 8 vectors; through host
  buffers (the plugin's ``try_linear`` use), device buffers, or a captured HIP
  graph (a serving loop);
* ``moe``: one token through ``layers`` routed-MoE layers (decode), plain or
  with a shared expert, through host buffers, device buffers or a graph;
* ``prefill``: a batch of tokens through one routed-MoE layer;
* ``generate``: a whole small-depth model: prompt, then greedy tokens, with
  the logits after the prompt.

Weights are random in every quant field, with scales that centre them on zero
and give them a trained layer's spread (standard deviation 0.02); activations
are normalised hidden states, N(0, 1) with a few wide channels.
"""
import math

import numpy as np
import torch

from pokitlms_amd import synth as S
from pokitlms_amd import synth_model as SM
from pokitlms_amd.backend import HipBackend, Moe35LayerHandles, MoeLayerHandles
from pokitlms_amd.model import Qwen3MoeModel

STD = 0.02
TYPES = {name: gtype for gtype, name in S.TYPE_NAMES.items()}
F64 = torch.float64


# ---- the cases ------------------------------------------------------------------------

def listed():
    return [
        # the smallest call a plugin makes: a 37-row projection on host buffers
        {"name": "linear_small_host", "kind": "linear", "type": "Q8_0", "out": 37, "in": 512,
         "batch": 1, "count": 1, "via": "host"},
        # single-token decode of a square projection, layer after layer, in a graph
        {"name": "linear_q4k_4096", "kind": "linear", "type": "Q4_K", "out": 4096, "in": 4096,
         "batch": 1, "count": 16, "via": "graph"},
        # eight sequences decoding together through a wide projection, in a graph
        {"name": "linear_q6k_batch8", "kind": "linear", "type": "Q6_K", "out": 2048, "in": 6144,
         "batch": 8, "count": 16, "via": "graph"},
        # three vectors, ragged row count, plain device calls
        {"name": "linear_q8_ragged", "kind": "linear", "type": "Q8_0", "out": 1027, "in": 2560,
         "batch": 3, "count": 4, "via": "device"},
        # the output head of a 151,936-token vocabulary, one vector
        {"name": "head_q6k", "kind": "linear", "type": "Q6_K", "out": 151936, "in": 2048,
         "batch": 1, "count": 1, "via": "device"},
        # one token through eight MoE layers of the 128-expert shape, in a graph
        {"name": "moe_token", "kind": "moe", "gate": "Q4_K", "down": "Q6_K", "hidden": 2048,
         "ffn": 768, "experts": 128, "top_k": 8, "shared": False, "layers": 8, "skew": 0.0,
         "via": "graph"},
        # a plugin's MoE block with a shared expert on host buffers
        {"name": "moe_shared_host", "kind": "moe", "gate": "Q5_K", "down": "Q8_0", "hidden": 2048,
         "ffn": 512, "experts": 64, "top_k": 6, "shared": True, "layers": 1, "skew": 0.0,
         "via": "host"},
        # a short prompt of odd length through a smaller layer with a shared expert
        {"name": "prefill_77_shared", "kind": "prefill", "gate": "Q5_K", "down": "Q8_0",
         "hidden": 1024, "ffn": 512, "experts": 64, "top_k": 6, "shared": True, "tokens": 77,
         "skew": 0.0},
        # an ordinary prompt, expert load skewed as trained routers skew it
        {"name": "prefill_512", "kind": "prefill", "gate": "Q4_K", "down": "Q6_K", "hidden": 2048,
         "ffn": 768, "experts": 128, "top_k": 8, "shared": False, "tokens": 512, "skew": 1.0},
        # the longest batch the entry takes
        {"name": "prefill_4096", "kind": "prefill", "gate": "Q4_K", "down": "Q6_K", "hidden": 2048,
         "ffn": 768, "experts": 128, "top_k": 8, "shared": False, "tokens": 4096, "skew": 0.5},
        # whole model in the reference's operation order (the default mode)
        {"name": "generate_reference", "kind": "generate", "layers": 2, "prompt": 32, "new": 16,
         "vocab": 151936, "reference": True},
        # whole model on the fast kernels: a question's prompt and a few tokens
        {"name": "generate_fast", "kind": "generate", "layers": 4, "prompt": 128, "new": 8,
         "vocab": 151936, "reference": False},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "moe", "moe", "prefill", "prefill", "prefill",
                       "generate"])
    if kind == "linear":
        gtype = rng.choice(["Q4_0", "Q4_1", "Q5_0", "Q5_1", "Q8_0", "Q4_K", "Q5_K", "Q6_K", "Q4_K",
                            "Q6_K", "F16", "BF16"])
        mm = gtype in ("Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K")  # in use for batches
        return {"kind": kind, "type": gtype, "out": _log_int(rng, 16, 16384),
                "in": 256 * _log_int(rng, 1, 24 if mm else 16),
                "batch": rng.choice([1, 1, 2, 3, 4, 5, 7, 8]) if mm else rng.choice([1, 1, 2, 4]),
                "count": rng.choice([1, 4, 8]), "via": rng.choice(["host", "device", "graph"])}
    if kind == "generate":
        return {"kind": kind, "layers": rng.randint(1, 3), "prompt": _log_int(rng, 3, 128),
                "new": rng.randint(1, 8), "vocab": rng.choice([4096, 32000, 151936]),
                "reference": rng.random() < 0.5}
    gate = rng.choice(["Q4_K", "Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0"])
    down = rng.choice(["Q6_K", "Q6_K", "Q4_K", "Q5_K", "Q8_0", "Q4_0"])
    experts = rng.choice([16, 32, 64, 128])
    case = {"kind": kind, "gate": gate, "down": down, "hidden": rng.choice([512, 1024, 2048, 2048]),
            "ffn": rng.choice([512, 768, 768, 1024]), "experts": experts,
            "top_k": rng.randint(2, 8), "shared": rng.random() < 0.3}
    if kind == "moe":
        case.update(layers=rng.choice([1, 4, 8]), skew=0.0,
                    via=rng.choice(["host", "device", "graph", "graph"]))
    else:
        case.update(tokens=_log_int(rng, 2, 3000), skew=rng.choice([0.0, 0.5, 1.0]))
    return case


# ---- inputs: GGUF bytes and activations from the seed ---------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rand(gen, shape, lo, hi):
    return torch.randint(lo, hi, shape, dtype=torch.uint8, device="cuda", generator=gen)


def _half(gen, n, mean):
    """n fp16 scales within a quarter of `mean`, as byte pairs [n, 2]."""
    h = mean * (0.75 + 0.5 * torch.rand(n, device="cuda", generator=gen))
    return h.to(torch.float16).view(torch.uint8).view(n, 2)


def _scaled(h, factor):
    """The scales `h` (byte pairs) times `factor`, as byte pairs."""
    v = h.contiguous().view(torch.float16).float() * factor
    return v.to(torch.float16).view(torch.uint8).view(-1, 2)


def _quant(gen, gtype, rows, cols):
    """Encoded rows of `cols` weights (uint8, 1-D): uniform quants, scales that
    centre them on zero with standard deviation about STD."""
    if gtype in (S.F32, S.F16, S.BF16):
        w = STD * torch.randn(rows * cols, device="cuda", generator=gen)
        dt = {S.F32: torch.float32, S.F16: torch.float16, S.BF16: torch.bfloat16}[gtype]
        return w.to(dt).view(torch.uint8)
    n = rows * cols // S.BLOCK_ELEMENTS[gtype]
    b = _rand(gen, (n, S.BLOCK_BYTES[gtype]), 0, 256)
    if gtype in (S.Q4_0, S.Q5_0, S.Q8_0):
        b[:, 0:2] = _half(gen, n, STD / {S.Q4_0: 4.6, S.Q5_0: 9.2, S.Q8_0: 74.0}[gtype])
    elif gtype in (S.Q4_1, S.Q5_1):
        q = 4.6 if gtype == S.Q4_1 else 9.2
        b[:, 0:2] = _half(gen, n, STD / q)
        b[:, 2:4] = _scaled(b[:, 0:2], -7.5 if gtype == S.Q4_1 else -15.5)
    elif gtype in (S.Q4_K, S.Q5_K):
        q, mid = (4.6, 7.5) if gtype == S.Q4_K else (9.2, 15.5)
        b[:, 0:2] = _half(gen, n, STD / (q * 42.0))
        b[:, 2:4] = _scaled(b[:, 0:2], mid)
        sc = _rand(gen, (n, 8), 20, 64)  # the 6-bit scales; the mins are the same numbers
        b[:, 4:8] = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
        b[:, 8:12] = b[:, 4:8]
        b[:, 12:16] = (sc[:, 4:] & 15) | ((sc[:, 4:] & 15) << 4)
    else:  # Q6_K
        b[:, 208:210] = _half(gen, n, STD / (74.0 * 18.5))
    return b.view(-1)


def _hidden_states(gen, tokens, hidden):
    x = torch.randn(tokens, hidden, device="cuda", generator=gen)
    x[:, 5::max(1, hidden // 4)] *= 8.0  # the few wide channels of a trained model
    return x


def _upload(hip, gtype, rows, cols, data, experts=0):
    return hip.upload_device(gtype, cols, rows, data.data_ptr(), data.numel(), experts)


def _linear_inputs(case, seed):
    gen = _gen(seed)
    gtype = TYPES[case["type"]]
    w = _quant(gen, gtype, case["count"] * case["out"], case["in"])
    return gtype, w, _hidden_states(gen, case["batch"], case["in"])


def _layer_inputs(case, gen):
    """One MoE layer's tensors: (router, gate, up, down, shared tensors)."""
    H, F, E = case["hidden"], case["ffn"], case["experts"]
    gt, dt = TYPES[case["gate"]], TYPES[case["down"]]
    router = STD * torch.randn(E, H, device="cuda", generator=gen)
    # column 0 of x is 1: its router weights are the experts' popularity
    router[:, 0] = case["skew"] * torch.randn(E, device="cuda", generator=gen)
    experts = [_quant(gen, gt, E * F, H), _quant(gen, gt, E * F, H), _quant(gen, dt, E * H, F)]
    shared = None
    if case["shared"]:
        shared = [STD * torch.randn(1, H, device="cuda", generator=gen), _quant(gen, gt, F, H),
                  _quant(gen, gt, F, H), _quant(gen, dt, H, F)]
    return router, experts, shared


def _moe_inputs(case, seed):
    gen = _gen(seed)
    layers = [_layer_inputs(case, gen) for _ in range(case.get("layers", 1))]
    n = case["tokens"] if case["kind"] == "prefill" else case["layers"]
    x = _hidden_states(gen, n, case["hidden"])
    x[:, 0] = 1.0
    return layers, x


def _model_shape(case):
    return SM.Qwen3MoeShape(layers=case["layers"], vocab=case["vocab"])


def _model_inputs(case, seed):
    """Every tensor of the model by GGUF name: (type, in, out, experts, bytes), and the prompt."""
    gen, shape, tensors = _gen(seed), _model_shape(case), {}
    for name, dims, gtype, kind in SM.tensor_list(shape):
        cols, rows, experts = dims[0], dims[1] if len(dims) > 1 else 1, dims[2] if len(dims) > 2 else 0
        if kind == SM.KIND_NORM:
            w = 1.0 + 0.1 * torch.rand(cols, device="cuda", generator=gen)
            data = w.view(torch.uint8)
        else:
            data = _quant(gen, gtype, rows * max(experts, 1), cols)
        tensors[name] = (gtype, cols, rows, experts, data)
    prompt = np.random.RandomState(seed % (1 << 31)).randint(0, case["vocab"], case["prompt"])
    return shape, tensors, prompt.astype(np.uint32)


# ---- prepare and run --------------------------------------------------------------------

_backend = None


def _hip():
    global _backend
    if _backend is None:
        _backend = HipBackend(0)
    return _backend


class _State:
    """What the program keeps between calls; its weights go when it goes."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        self.graph = None
        for held in self.held:
            (held.close if hasattr(held, "close") else held.release)()


def _captured(enqueue):
    """`enqueue(stream)` captured into a HIP graph after one plain call."""
    stream = torch.cuda.Stream()
    enqueue(stream.cuda_stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        enqueue(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return graph


def _prepare_linear(case, seed):
    hip = _hip()
    gtype, data, x = _linear_inputs(case, seed)
    n = case["count"]
    w = _upload(hip, gtype, case["out"], case["in"], data, n if n > 1 else 0)
    experts = list(range(n)) if n > 1 else [None]
    y = torch.empty(n, case["batch"], case["out"], device="cuda")
    s = _State(case=case, held=[w], w=w, experts=experts, x=x, y=y, graph=None)
    if case["via"] == "host":
        s.host_x = x.cpu().numpy()
    elif case["via"] == "graph":
        s.graph = _captured(lambda st: _enqueue_linear(s, st))
    return s


def _enqueue_linear(s, stream):
    hip = _hip()
    for i, e in enumerate(s.experts):
        hip.matvec_async(s.w, s.x.data_ptr(), s.case["batch"], s.y[i].data_ptr(), stream, e)


def _upload_layer(hip, case, tensors):
    H, F, E = case["hidden"], case["ffn"], case["experts"]
    gt, dt = TYPES[case["gate"]], TYPES[case["down"]]
    router, experts, shared = tensors
    scale = 2.5 if shared else 1.0
    routed = MoeLayerHandles(_upload(hip, S.F32, E, H, router.view(torch.uint8).view(-1)),
                             _upload(hip, gt, F, H, experts[0], E),
                             _upload(hip, gt, F, H, experts[1], E),
                             _upload(hip, dt, H, F, experts[2], E), case["top_k"], True, scale)
    if shared is None:
        return routed
    return Moe35LayerHandles(routed, _upload(hip, S.F32, 1, H, shared[0].view(torch.uint8).view(-1)),
                             _upload(hip, gt, F, H, shared[1]), _upload(hip, gt, F, H, shared[2]),
                             _upload(hip, dt, H, F, shared[3]))


def _prepare_moe(case, seed):
    hip = _hip()
    layers, x = _moe_inputs(case, seed)
    handles = [_upload_layer(hip, case, t) for t in layers]
    n, K = x.shape[0], case["top_k"]
    s = _State(case=case, held=handles, layers=handles, x=x, y=torch.empty_like(x),
               ids=torch.zeros(n, K, dtype=torch.int32, device="cuda"),
               probs=torch.zeros(n, K, device="cuda"), graph=None)
    if case.get("via") == "host":
        s.host_x = x.cpu().numpy()
    elif case.get("via") == "graph":
        s.graph = _captured(lambda st: _enqueue_moe(s, st))
    return s


def _enqueue_moe(s, stream):
    hip = _hip()
    decode = hip.moe35_decode_async if s.case["shared"] else hip.moe_decode_async
    for i, layer in enumerate(s.layers):
        decode(layer, s.x[i].data_ptr(), s.y[i].data_ptr(), s.ids[i].data_ptr(),
               s.probs[i].data_ptr(), stream)


def _prepare_model(case, seed):
    hip = _hip()
    shape, tensors, prompt = _model_inputs(case, seed)
    weights = {name: _upload(hip, t, rows, cols, data, experts)
               for name, (t, cols, rows, experts, data) in tensors.items()}
    model = Qwen3MoeModel(hip, shape, weights, case["reference"])
    return _State(case=case, held=[model], model=model, prompt=prompt)


def prepare(case, seed):
    if case["kind"] == "linear":
        return _prepare_linear(case, seed)
    if case["kind"] == "generate":
        return _prepare_model(case, seed)
    return _prepare_moe(case, seed)


def run(s):
    case, hip = s.case, _hip()
    kind, via = case["kind"], case.get("via")
    if kind == "generate":
        tokens, logits, _ = s.model.generate(s.prompt, case["new"], want_logits=True)
        return {"tokens": tokens.astype(np.int64), "logits": logits}
    if s.graph is not None:
        s.graph.replay()
    elif kind == "linear" and via == "host":
        return {"y": [hip.matvec(s.w, s.host_x, e) for e in s.experts]}
    elif kind == "linear":
        _enqueue_linear(s, 0)
    elif kind == "moe" and via == "host":
        decode = hip.moe35_decode if case["shared"] else hip.moe_decode
        out = [decode(layer, s.host_x[i]) for i, layer in enumerate(s.layers)]
        return {"y": np.stack([o[0] for o in out]),
                "ids": np.stack([o[1] for o in out]).astype(np.int32),
                "probs": np.stack([o[2] for o in out])}
    elif kind == "moe":
        _enqueue_moe(s, 0)
    else:
        prefill = hip.moe35_prefill_async if case["shared"] else hip.moe_prefill_async
        prefill(s.layers[0], s.x.data_ptr(), case["tokens"], s.y.data_ptr(), s.ids.data_ptr(),
                s.probs.data_ptr())
    if kind == "linear":
        return {"y": [s.y[i] for i in range(case["count"])]}
    return {"y": s.y, "ids": s.ids, "probs": s.probs}


# ---- what a pass cannot do without ------------------------------------------------------

def _expert_bytes(case):
    H, F = case["hidden"], case["ffn"]
    return (2 * S.matrix_bytes(TYPES[case["gate"]], H, F) +
            S.matrix_bytes(TYPES[case["down"]], F, H))


def work(case):
    if case["kind"] == "linear":
        n, B, o, i = case["count"], case["batch"], case["out"], case["in"]
        return {"bytes": n * (S.matrix_bytes(TYPES[case["type"]], i, o) + 4 * B * o) + 4 * B * i,
                "flops": 2.0 * n * B * o * i}
    if case["kind"] == "generate":
        m = _model_shape(case)
        qd, kd = m.heads * m.head_dim, m.kv_heads * m.head_dim
        attn = S.matrix_bytes(m.attn_type, m.hidden, qd + 2 * kd) + S.matrix_bytes(m.attn_type, qd,
                                                                                 m.hidden)
        expert = (2 * S.matrix_bytes(m.gate_type, m.hidden, m.ffn) +
                  S.matrix_bytes(m.down_type, m.ffn, m.hidden))
        router, head = 4 * m.experts * m.hidden, S.matrix_bytes(m.out_type, m.hidden, m.vocab)
        touched = min(m.experts, case["prompt"] * m.top_k)  # the prompt in one batch
        steps = case["new"] - 1
        bytes_ = (m.layers * (attn + router + touched * expert) + head +
                  steps * (m.layers * (attn + router + m.top_k * expert) + head))
        per_token = 2.0 * m.layers * (m.hidden * (2 * qd + 2 * kd) + m.experts * m.hidden +
                                      3 * m.top_k * m.hidden * m.ffn)
        return {"bytes": bytes_, "flops": per_token * (case["prompt"] + steps) +
                2.0 * case["new"] * m.hidden * m.vocab}
    H, F, E, K = case["hidden"], case["ffn"], case["experts"], case["top_k"]
    extra = 1 if case["shared"] else 0
    prefill = case["kind"] == "prefill"
    layers, tokens = (1, case["tokens"]) if prefill else (case["layers"], 1)
    touched = min(E, tokens * K) + extra
    return {"bytes": layers * (4 * (E + extra) * H + touched * _expert_bytes(case) +
                               tokens * (8 * H + 8 * K)),
            "flops": 2.0 * layers * tokens * ((E + extra) * H + 3 * (K + extra) * H * F)}


def tolerance(case):
    """About four times what a path shows against float64 (FP32 sums in another
    order, whose rounding differs); routes, counted exactly, do not differ."""
    if case["kind"] == "generate":
        if case["reference"]:
            return "exact"  # the reference's bits
        # logits of a few layers: 3e-5 to 6e-5, plus now and then a router near-tie that
        # rounding in an earlier layer decides the other way for one prompt token
        return {"rel": 1e-3, "max": 2e-2}
    if case["kind"] == "linear":
        return {"rel": 4e-6, "max": 2e-4}
    return {"rel": 1.5e-5, "max": 6e-4}


# ---- the same in 64 bits, in plain torch -------------------------------------------------

def _f16(b):
    return b.contiguous().view(torch.float16).to(F64)


def _dequant(gtype, data, rows, cols):
    """float64 [rows, cols] of GGUF rows (uint8, 1-D)."""
    if gtype in (S.F32, S.F16, S.BF16):
        dt = {S.F32: torch.float32, S.F16: torch.float16, S.BF16: torch.bfloat16}[gtype]
        return data.view(dt).view(rows, cols).to(F64)
    b = data.view(-1, S.BLOCK_BYTES[gtype])
    n = b.shape[0]
    if gtype == S.Q8_0:
        w = _f16(b[:, 0:2]) * b[:, 2:34].contiguous().view(torch.int8).to(F64)
    elif gtype in (S.Q4_0, S.Q4_1, S.Q5_0, S.Q5_1):
        has_min, five = gtype in (S.Q4_1, S.Q5_1), gtype in (S.Q5_0, S.Q5_1)
        at = 4 if has_min else 2
        qs = b[:, at + (4 if five else 0):]
        q = torch.cat([qs & 15, qs >> 4], 1).to(torch.int32)
        if five:
            i = torch.arange(32, device=b.device)
            q |= ((b[:, at:at + 4][:, i // 8] >> (i % 8).to(torch.uint8)) & 1).to(torch.int32) << 4
        d = _f16(b[:, 0:2])
        w = d * q + _f16(b[:, 2:4]) if has_min else d * (q - (16 if five else 8))
    elif gtype in (S.Q4_K, S.Q5_K):
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = b[:, 16 if gtype == S.Q4_K else 48:].view(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(n, 8, 32)
        if gtype == S.Q5_K:
            j = torch.arange(8, dtype=torch.uint8, device=b.device).view(1, 8, 1)
            q = q | (((b[:, 16:48].view(n, 1, 32) >> j) & 1) << 4)
        w = (_f16(b[:, 0:2]) * sc).unsqueeze(2) * q - (_f16(b[:, 2:4]) * mn).unsqueeze(2)
    else:  # Q6_K
        ql, qh = b[:, 0:128].view(n, 2, 2, 32), b[:, 128:192].view(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # [n, half, run g, 32]
        g = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=b.device).view(1, 1, 4, 1)
        q = (lo | (((qh >> g) & 3) << 4)).to(torch.int32) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).to(F64)
        w = (_f16(b[:, 208:210]) * sc).unsqueeze(2) * q.view(n, 16, 16)
    return w.reshape(rows, cols)


def _matmul(gtype, data, rows, cols, x):
    """x [n, cols] . W^T in float64, a few thousand rows of W at a time."""
    per, out = len(data) // rows, []
    for r in range(0, rows, 8192):
        m = min(8192, rows - r)
        out.append(x @ _dequant(gtype, data[r * per:(r + m) * per], m, cols).t().contiguous())
    return torch.cat(out, 1)


def _route(router, x, x32, top_k):
    """The experts of each token, by the FP32 logits as one serial sum makes them
    (which is what orders them), and the float64 logits."""
    logits = torch.zeros(x32.shape[0], router.shape[0], device="cuda")
    for i in range(router.shape[1]):
        logits += x32[:, i:i + 1] * router[:, i]
    order = torch.sort(logits, dim=1, descending=True, stable=True)[1]
    return order[:, :top_k], x @ router.to(F64).t().contiguous()


def _moe_block(case, tensors, x, x32):
    """(y, ids, probs) of x [n, hidden] through one layer in float64."""
    H, F, E, K = case["hidden"], case["ffn"], case["experts"], case["top_k"]
    gt, dt = TYPES[case["gate"]], TYPES[case["down"]]
    router, (gate, up, down), shared = tensors
    ids, logits = _route(router, x, x32, K)
    probs = torch.softmax(logits, 1).gather(1, ids)
    probs = probs / probs.sum(1, keepdim=True)
    if shared is not None:
        probs = probs * 2.5

    def mlp(xe, g, u, d):
        a = torch.nn.functional.silu(_matmul(gt, g, F, H, xe)) * _matmul(gt, u, F, H, xe)
        return _matmul(dt, d, H, F, a)

    y = torch.zeros_like(x)
    for e in ids.unique().tolist():
        t, r = (ids == e).nonzero(as_tuple=True)
        part = [w.view(E, -1)[e] for w in (gate, up, down)]
        y.index_add_(0, t, mlp(x[t], *part) * probs[t, r].unsqueeze(1))
    if shared is not None:
        y += torch.sigmoid(x @ shared[0].to(F64).t().contiguous()) * mlp(x, *shared[1:])
    return y, ids.to(torch.int32), probs


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope(x, pos, theta):
    half = x.shape[-1] // 2
    f = theta ** (-torch.arange(half, dtype=F64, device="cuda") / half)
    a = (pos.to(F64).unsqueeze(1) * f).unsqueeze(1)
    x0, x1 = x[..., :half], x[..., half:]
    return torch.cat([x0 * a.cos() - x1 * a.sin(), x0 * a.sin() + x1 * a.cos()], -1)


def _prompt_logits(case, seed):
    shape, tensors, prompt = _model_inputs(case, seed)
    n, hd = len(prompt), shape.head_dim
    moe = {"hidden": shape.hidden, "ffn": shape.ffn, "experts": shape.experts,
           "top_k": shape.top_k, "gate": S.TYPE_NAMES[shape.gate_type],
           "down": S.TYPE_NAMES[shape.down_type]}
    pos = torch.arange(n, device="cuda")

    def mul(name, x):
        t, cols, rows, _, data = tensors[name]
        return _matmul(t, data, rows, cols, x)

    def norm(name, x):
        return _rms(x, tensors[name][4].view(torch.float32).to(F64), shape.rms_eps)

    t, cols, rows, _, data = tensors["token_embd.weight"]
    at = torch.from_numpy(prompt.astype(np.int64)).cuda()
    h = _dequant(t, data.view(rows, -1)[at].reshape(-1), n, cols)
    for l in range(shape.layers):
        p = f"blk.{l}."
        x = norm(p + "attn_norm.weight", h)
        q = norm(p + "attn_q_norm.weight", mul(p + "attn_q.weight", x).view(n, shape.heads, hd))
        k = norm(p + "attn_k_norm.weight", mul(p + "attn_k.weight", x).view(n, shape.kv_heads, hd))
        v = mul(p + "attn_v.weight", x).view(n, shape.kv_heads, hd)
        q, k = _rope(q, pos, shape.rope_theta), _rope(k, pos, shape.rope_theta)
        rep = shape.heads // shape.kv_heads
        k = k.to(torch.float16).to(F64).repeat_interleave(rep, 1).permute(1, 2, 0).contiguous()
        v = v.to(torch.float16).to(F64).repeat_interleave(rep, 1).permute(1, 0, 2).contiguous()
        s = torch.bmm(q.permute(1, 0, 2).contiguous(), k) / math.sqrt(hd)
        s = s.masked_fill(pos.view(1, -1, 1) < pos.view(1, 1, -1), -math.inf)
        att = torch.bmm(torch.softmax(s, 2), v).permute(1, 0, 2).reshape(n, -1)
        h = h + mul(p + "attn_output.weight", att)
        x = norm(p + "ffn_norm.weight", h)
        router = tensors[p + "ffn_gate_inp.weight"][4].view(torch.float32).view(shape.experts, -1)
        experts = [tensors[p + f"ffn_{m}_exps.weight"][4] for m in ("gate", "up", "down")]
        h = h + _moe_block(moe, (router, experts, None), x, x.float())[0]
    return mul("output.weight", norm("output_norm.weight", h[-1:]))[0]


def exact(case, seed):
    if case["kind"] == "generate":
        return {"tokens": None, "logits": _prompt_logits(case, seed)}
    if case["kind"] == "linear":
        gtype, data, x = _linear_inputs(case, seed)
        y = [_matmul(gtype, d, case["out"], case["in"], x.to(F64))
             for d in data.view(case["count"], -1)]
        return {"y": y}
    layers, x = _moe_inputs(case, seed)
    if case["kind"] == "prefill":
        y, ids, probs = _moe_block(case, layers[0], x.to(F64), x)
    else:
        rows = [_moe_block(case, t, x[i:i + 1].to(F64), x[i:i + 1]) for i, t in enumerate(layers)]
        y, ids, probs = (torch.cat(v) for v in zip(*rows))
    return {"y": y, "ids": ids, "probs": probs}
