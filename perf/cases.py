"""The work a program built on this package has it do, as cases that can be timed and compared.

Every case goes through the runtime's own calls on device buffers, the way the model backends and
the benchmark use them: launches queued in one command and kept as a prepared plan, activations
and weights resident. The inputs are drawn on the GPU from the case's seed.

Kinds of cases:
  attention   `layers` calls of the fused q/k RMSNorm + RoPE + causal GQA attention on fp16
              activations (16 query heads, 8 key/value heads of 128), fp32 or fp16 output
  block       the uint4 q/k/v projection of fp16 activations feeding that attention
  qwen_layer  token ids -> embedding -> `layers` Qwen3-0.6B decoder layers (uint4 weights, fp32
              activations), the hidden states returned
  bge_layer   token ids -> embedding + LayerNorm -> `layers` BGE-small encoder layers (fp32)
  qwen_model, bge_model   a whole embedding forward, from host ids to pooled host vectors
"""

from __future__ import annotations

import ctypes
import math
import random

import numpy as np
import torch

from tessery_amd import HipRuntime
from tessery_amd import backends
from tessery_amd.packs import BertDims, DeviceWeights, Qwen3Dims

EPS, THETA = 1e-6, 1e6
HEADS, KV_HEADS, DIM = 16, 8, 128          # Qwen3-0.6B attention
HIDDEN, INTER = 1024, 3072                 # Qwen3-0.6B widths
QWEN_LAYERS, BGE_LAYERS = 28, 12
BGE_HIDDEN, BGE_INTER, BGE_HEADS = 384, 1536, 12
BGE_EPS = 1e-12
# rows of the embedding tables (a table's size does not change the work of a call)
QWEN_VOCAB, BGE_VOCAB, POSITIONS, TYPES = 4096, 4096, 512, 2


def listed():
    return [
        # the headline: prefill attention of a full batch of documents of mixed lengths (most
        # short, a few long), at the execution width of the longest
        dict(name="attention_mixed_32x464", kind="attention", batch=32, seq=464, lengths="log",
             lengths_seed=4, layers=4, out="f32"),
        # the same batch with every document cut at the maximum length, fp16 output
        dict(name="attention_full_32x512", kind="attention", batch=32, seq=512, lengths="full",
             lengths_seed=0, layers=2, out="f16"),
        # attention of one short search query: launches and latency
        dict(name="attention_query_1x24", kind="attention", batch=1, seq=24, lengths="full",
             lengths_seed=0, layers=4, out="f32"),
        # projection and attention of a medium batch of passages on fp16 activations
        dict(name="block_16x256", kind="block", batch=16, seq=256, lengths="uniform",
             lengths_seed=5, layers=2, out="f32"),
        # one decoder layer: a search query, a few passages of odd width, the largest batch the
        # backend takes (4096 padded tokens)
        dict(name="qwen_layer_1x24", kind="qwen_layer", batch=1, seq=24, lengths="full",
             lengths_seed=0, layers=1),
        dict(name="qwen_layer_4x77", kind="qwen_layer", batch=4, seq=77, lengths="half",
             lengths_seed=1, layers=1),
        dict(name="qwen_layer_8x512", kind="qwen_layer", batch=8, seq=512, lengths="half",
             lengths_seed=2, layers=1),
        # one encoder layer: a batch of short queries, a few passages of odd width, the full
        # 32 x 512 batch
        dict(name="bge_layer_16x41", kind="bge_layer", batch=16, seq=41, lengths="half",
             lengths_seed=3, layers=1),
        dict(name="bge_layer_3x181", kind="bge_layer", batch=3, seq=181, lengths="half",
             lengths_seed=4, layers=1),
        dict(name="bge_layer_32x512", kind="bge_layer", batch=32, seq=512, lengths="uniform",
             lengths_seed=2, layers=1),
        # whole forwards: one query through Qwen3-0.6B, a batch of documents through BGE-small
        dict(name="qwen_model_1x24", kind="qwen_model", batch=1, seq=24, lengths="full",
             lengths_seed=0, layers=QWEN_LAYERS),
        dict(name="bge_model_8x512", kind="bge_model", batch=8, seq=512, lengths="half",
             lengths_seed=6, layers=BGE_LAYERS),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    kind = rng.choice(("attention", "attention", "block", "qwen_layer", "qwen_layer", "bge_layer",
                       "bge_layer", "qwen_model", "bge_model"))
    tokens = {"attention": 16384, "block": 4096, "qwen_layer": 4096, "bge_layer": 16384,
              "qwen_model": 128, "bge_model": 4096}[kind]
    seq = _log_int(rng, 2, min(512, tokens))
    case = dict(kind=kind, batch=_log_int(rng, 1, min(32, tokens // seq)), seq=seq,
                lengths="half" if kind.endswith("model") or "layer" in kind
                else rng.choice(("log", "uniform", "full")),
                lengths_seed=rng.randrange(1 << 20),
                layers={"qwen_model": QWEN_LAYERS, "bge_model": BGE_LAYERS, "attention": 2,
                        "block": 2}.get(kind, 1))
    if kind in ("attention", "block"):
        case["out"] = rng.choice(("f32", "f16"))
    return case


def _lengths(case):
    """Valid tokens of each row; the longest row is the batch's width. "half": at least half the
    width (what a length bucket of the batching plan holds); "log" and "uniform" from 1."""
    rng, seq = random.Random(case["lengths_seed"]), case["seq"]
    low = 2 if case["kind"].startswith("bge") else 1
    pick = {"full": lambda: seq, "uniform": lambda: rng.randint(low, seq),
            "log": lambda: _log_int(rng, low, seq),
            "half": lambda: rng.randint(max(low, (seq + 1) // 2), seq)}[case["lengths"]]
    got = [pick() for _ in range(case["batch"])]
    got[rng.randrange(len(got))] = seq
    return got


# ---- inputs, drawn by torch from the seed alone ----------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _uniform(g, low, high, *shape):
    return torch.rand(*shape, generator=g, device="cuda") * (high - low) + low


def _uint4(g, prefix, outputs, inputs, scale):
    """Packed codes U{0..15} with near zero-mean affine groups of 64, bf16 scales and biases."""
    words = torch.randint(-2**31, 2**31, (outputs, inputs // 8), generator=g, device="cuda",
                          dtype=torch.int32)
    s = _uniform(g, 0.5, 1.5, outputs, inputs // 64) * scale
    b = -(7.5 + _uniform(g, -0.5, 0.5, outputs, inputs // 64)) * s
    return {prefix + ".weight": words, prefix + ".scales": s.bfloat16(),
            prefix + ".biases": b.bfloat16()}


def _qwen_weights(g, layers):
    w = _uint4(g, "model.embed_tokens", QWEN_VOCAB, HIDDEN, 0.2)
    w["model.norm.weight"] = _uniform(g, 0.5, 1.5, HIDDEN).bfloat16()
    for i in range(layers):
        p = f"model.layers.{i}."
        for name, n in (("input_layernorm", HIDDEN), ("post_attention_layernorm", HIDDEN),
                        ("self_attn.q_norm", DIM), ("self_attn.k_norm", DIM)):
            w[p + name + ".weight"] = _uniform(g, 0.5, 1.5, n).bfloat16()
        for name, n, k in (("self_attn.q_proj", HEADS * DIM, HIDDEN),
                           ("self_attn.k_proj", KV_HEADS * DIM, HIDDEN),
                           ("self_attn.v_proj", KV_HEADS * DIM, HIDDEN),
                           ("self_attn.o_proj", HIDDEN, HEADS * DIM),
                           ("mlp.gate_proj", INTER, HIDDEN), ("mlp.up_proj", INTER, HIDDEN),
                           ("mlp.down_proj", HIDDEN, INTER)):
            w.update(_uint4(g, p + name, n, k, 0.2 / math.sqrt(k)))
    return w


def _bge_weights(g, layers):
    h, w = BGE_HIDDEN, {}
    for name, rows in (("word", BGE_VOCAB), ("position", POSITIONS), ("token_type", TYPES)):
        w[f"embeddings.{name}_embeddings.weight"] = _normal(g, rows, h, std=0.5)

    def norm(prefix):
        w[prefix + ".weight"] = _uniform(g, 0.5, 1.5, h)
        w[prefix + ".bias"] = _normal(g, h, std=0.1)

    norm("embeddings.LayerNorm")
    for i in range(layers):
        p = f"encoder.layer.{i}."
        for name, n, k in (("attention.self.query", h, h), ("attention.self.key", h, h),
                           ("attention.self.value", h, h), ("attention.output.dense", h, h),
                           ("intermediate.dense", BGE_INTER, h), ("output.dense", h, BGE_INTER)):
            w[p + name + ".weight"] = _normal(g, n, k, std=k**-0.5)
            w[p + name + ".bias"] = _normal(g, n, std=0.1)
        norm(p + "attention.output.LayerNorm")
        norm(p + "output.LayerNorm")
    return w


def _inputs(case, seed):
    g = _generator(seed)
    b, s, kind = case["batch"], case["seq"], case["kind"]
    t = {"lengths": torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")}
    if kind in ("attention", "block"):
        for i in range(case["layers"]):
            if kind == "attention":
                t[f"q{i}"] = _normal(g, b, s, HEADS, DIM).half()
                t[f"k{i}"] = _normal(g, b, s, KV_HEADS, DIM).half()
                t[f"v{i}"] = _normal(g, b, s, KV_HEADS, DIM).half()
            else:
                t[f"x{i}"] = _normal(g, b * s, HIDDEN).half()
                w = _uint4(g, "w", (HEADS + 2 * KV_HEADS) * DIM, HIDDEN, 0.02)
                for part in ("weight", "scales", "biases"):
                    t[f"{part}{i}"] = w["w." + part]
            t[f"q_norm{i}"] = _uniform(g, 0.5, 1.5, DIM).bfloat16()
            t[f"k_norm{i}"] = _uniform(g, 0.5, 1.5, DIM).bfloat16()
        return t
    qwen = kind.startswith("qwen")
    t["ids"] = torch.randint(0, QWEN_VOCAB if qwen else BGE_VOCAB, (b, s), generator=g,
                             device="cuda", dtype=torch.int32)
    t["weights"] = (_qwen_weights if qwen else _bge_weights)(g, case["layers"])
    return t


# ---- device state ----------------------------------------------------------------------------

_runtime = None


def _rt():
    """The one runtime a process keeps (the benchmark's workspace budget)."""
    global _runtime
    if _runtime is None:
        _runtime = HipRuntime(workspace_limit_bytes=1 << 30)
    return _runtime


class _Memory:
    """A runtime buffer's device memory for torch: what the buffer's handle points at begins with
    the device address. A tensor over it holds this object, and so the buffer."""

    def __init__(self, buffer):
        self.buffer = buffer
        address = ctypes.c_void_p.from_address(buffer.pointer).value
        self.__cuda_array_interface__ = {"shape": (buffer.size,), "typestr": "|u1",
                                         "data": (address, False), "version": 2}


def _view(buffer, shape, dtype):
    """A torch tensor over a runtime buffer's device memory."""
    return torch.as_tensor(_Memory(buffer), device="cuda").view(dtype).view(shape)


def _upload(tensor):
    buffer = _rt().buffer(tensor.numel() * tensor.element_size())
    _view(buffer, tensor.shape, tensor.dtype).copy_(tensor)
    return buffer


def _dims(case):
    if case["kind"].startswith("qwen"):
        return Qwen3Dims(hidden=HIDDEN, intermediate=INTER, layers=case["layers"], heads=HEADS,
                         kv_heads=KV_HEADS, head_dim=DIM, vocab=QWEN_VOCAB, eps=EPS, theta=THETA)
    return BertDims(hidden=BGE_HIDDEN, intermediate=BGE_INTER, layers=case["layers"],
                    heads=BGE_HEADS, vocab=BGE_VOCAB, positions=POSITIONS, types=TYPES,
                    eps=BGE_EPS)


def prepare(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    b, s = case["batch"], case["seq"]
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "lengths_seed")))
    state = {"case": case, "key": ("case",) + key}
    if kind in ("attention", "block"):
        bufs = {name: _upload(x) for name, x in t.items()}
        size = {"f32": 4, "f16": 2}[case["out"]]
        dtype = {"f32": torch.float32, "f16": torch.float16}[case["out"]]
        outs = {}
        for i in range(case["layers"]):
            bufs[f"out{i}"] = _rt().buffer(b * s * HEADS * DIM * size)
            outs[f"out{i}"] = _view(bufs[f"out{i}"], (b, s, HEADS, DIM), dtype)
            if kind == "block":
                for name, heads in (("q", HEADS), ("k", KV_HEADS), ("v", KV_HEADS)):
                    bufs[f"{name}{i}"] = _rt().buffer(b * s * heads * DIM * 2)
                    outs[f"{name}{i}"] = _view(bufs[f"{name}{i}"], (b, s, heads, DIM),
                                               torch.float16)
        # the normalized keys of one layer are scratch of its attention: two layers' worth, so
        # that a layer's keys can be made while the layer before it runs
        for i in range(2):
            bufs[f"work{i}"] = _rt().buffer(2 * b * s * KV_HEADS * DIM * 2)
        torch.cuda.synchronize()
        return dict(state, bufs=bufs, outs=outs)
    weights = DeviceWeights(_rt())
    for name, x in t["weights"].items():
        weights.buffers[name] = _upload(x)
    dims = _dims(case)
    if kind.startswith("qwen"):
        program = backends.qwen3_program(dims, b, s, HIDDEN)
    else:
        program = backends.bert_program(dims, b, s)
    state.update(weights=weights, program=program)
    if kind.endswith("model"):
        ids = t["ids"].cpu().numpy().astype(np.uint32)
        lengths = t["lengths"].cpu().numpy().astype(np.uint32)
        torch.cuda.synchronize()
        return dict(state, ids=ids, lengths=lengths)
    # the layers alone: the program without its model end (final norm and pooling), on
    # activations that stay resident
    ops = tuple(o for o in program.ops[:-1] if kind == "bge_layer" or o is not program.ops[-2])
    bound = {"%ids": _upload(t["ids"]), "%lengths": _upload(t["lengths"])}
    for slot, nbytes in program.activations:
        bound[slot] = _rt().buffer(nbytes)
    hidden = HIDDEN if kind == "qwen_layer" else BGE_HIDDEN
    torch.cuda.synchronize()
    return dict(state, ops=ops, bound=bound,
                outs={"x": _view(bound["%x"], (b, s, hidden), torch.float32)})


# ---- one pass --------------------------------------------------------------------------------


def _attention_layers(state):
    """What bench.py queues for its attention layers: layer after layer, each with its own inputs."""
    rt, case, bufs = _rt(), state["case"], state["bufs"]
    tokens = case["batch"] * case["seq"]
    for i in range(case["layers"]):
        if case["kind"] == "block":
            rt._qkv4([bufs[n] for n in (f"x{i}", f"weight{i}", f"scales{i}", f"biases{i}",
                                        f"q{i}", f"k{i}", f"v{i}")],
                     rows=tokens, k=HIDDEN, q_cols=HEADS * DIM, kv_cols=KV_HEADS * DIM)
        rt._attention_norm_rope([bufs[n] for n in (f"q{i}", f"k{i}", f"v{i}", "lengths",
                                                   f"out{i}", f"q_norm{i}", f"k_norm{i}",
                                                   f"work{i % 2}")],
                                tokens=tokens, seq=case["seq"], heads=HEADS, kv_heads=KV_HEADS,
                                dim=DIM, eps=EPS, theta=THETA, out_dtype=case["out"])


def _model_layers(state):
    weights, bound = state["weights"], state["bound"]

    def resolve(slot):
        if isinstance(slot, tuple):
            return weights.group(*slot)
        return [bound[slot] if slot.startswith("%") else weights[slot]]

    for o in state["ops"]:
        buffers = [b for slot in o.slots for b in resolve(slot)]
        backends.EMITTERS[o.kind](_rt(), buffers, **dict(o.params))


def run(state):
    rt, kind = _rt(), state["case"]["kind"]
    if kind.endswith("model"):
        return backends.execute(rt, state["program"], state["weights"], state["ids"],
                                state["lengths"])
    if kind in ("attention", "block"):
        bindings, emit = list(state["bufs"].values()), _attention_layers
    else:
        bindings = [*state["weights"].buffers.values(), *state["bound"].values()]
        emit = _model_layers
    with rt._workspace(), rt.command(), rt._execution_plan(state["key"], bindings) as replayed:
        if not replayed:
            emit(state)
    return state["outs"]


# ---- what a pass cannot do without -----------------------------------------------------------


def _pairs(case, causal):
    """Attended (query, key) pairs: padded query rows are outputs too."""
    s, total = case["seq"], 0
    for n in _lengths(case):
        total += n * (n + 1) // 2 + (s - n) * n if causal else s * n
    return total


def work(case):
    kind, layers = case["kind"], case["layers"]
    b, s = case["batch"], case["seq"]
    tokens, valid = b * s, sum(_lengths(case))
    if kind in ("attention", "block"):
        out = tokens * HEADS * DIM * (4 if case["out"] == "f32" else 2)
        flops = 4 * DIM * HEADS * _pairs(case, True)
        if kind == "attention":
            nbytes = tokens * HEADS * DIM * 2 + 2 * valid * KV_HEADS * DIM * 2 + out
        else:
            n = (HEADS + 2 * KV_HEADS) * DIM
            nbytes = tokens * HIDDEN * 2 + n * HIDDEN // 2 + n * HIDDEN // 16 + tokens * n * 2 + out
            flops += 2 * tokens * HIDDEN * n
        return {"bytes": layers * nbytes, "flops": layers * flops}
    if kind.startswith("qwen"):
        params = HIDDEN * ((HEADS + 2 * KV_HEADS) * DIM + HEADS * DIM + 3 * INTER)
        weights, hidden = params // 2 + params // 16, HIDDEN  # codes, then scales and biases
        attention = 4 * DIM * HEADS * _pairs(case, True)
    else:
        params = 4 * BGE_HIDDEN**2 + 2 * BGE_HIDDEN * BGE_INTER
        weights, hidden = 4 * params, BGE_HIDDEN
        attention = 4 * BGE_HIDDEN * _pairs(case, False)
    out = (b if kind.endswith("model") else tokens) * hidden * 4
    return {"bytes": layers * weights + tokens * 4 + out,
            "flops": layers * (2 * tokens * params + attention)}


def tolerance(case):
    """About four times the distance from the 64-bit results measured for each kind."""
    kind = case["kind"]
    if kind == "block" or case.get("out") == "f16":  # fp16 results: 2.1e-4
        return {"rel": 8e-4, "max": 8e-3}
    if kind.endswith("model"):  # 6.2e-7 and 4.8e-7
        return {"rel": 2.5e-6}
    return {"rel": 1.2e-6}  # 1.2e-7 to 2.8e-7


# ---- the same in 64 bits ---------------------------------------------------------------------


def _dequantize(words, scales, biases):
    shifts = torch.arange(0, 32, 4, device=words.device, dtype=torch.int32)
    codes = ((words[:, :, None] >> shifts) & 15).reshape(words.shape[0], -1, 64).double()
    return (codes * scales.double()[:, :, None] + biases.double()[:, :, None]).reshape(
        words.shape[0], -1)


def _rms(x, weight, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * weight.double()


def _rope(x):
    """x [b, s, heads, d]: split-half pairs rotated by the token's position in its row."""
    s, d = x.shape[1], x.shape[3]
    inv = THETA ** (-2.0 * torch.arange(d // 2, dtype=torch.float64, device=x.device) / d)
    angle = torch.arange(s, dtype=torch.float64, device=x.device)[:, None, None] * inv
    cos, sin = torch.cos(angle), torch.sin(angle)
    a, c = x[..., :d // 2], x[..., d // 2:]
    return torch.cat((a * cos - c * sin, a * sin + c * cos), -1)


def _attend(q, k, v, lengths, causal):
    """q [b, s, h, d], k and v [b, s, kv, d] in float64; every query row attends valid keys."""
    b, s, h, d = q.shape
    group = h // k.shape[2]
    out = torch.empty_like(q)
    at = torch.arange(s, device=q.device)
    for i, n in enumerate(lengths):
        kk = k[i, :n].repeat_interleave(group, 1).permute(1, 2, 0).contiguous()
        vv = v[i, :n].repeat_interleave(group, 1).permute(1, 0, 2).contiguous()
        scores = torch.matmul(q[i].permute(1, 0, 2).contiguous(), kk) * d**-0.5
        if causal:
            scores = scores.masked_fill(at[None, None, :n] > at[None, :, None], -math.inf)
        out[i] = torch.matmul(torch.softmax(scores, -1), vv).permute(1, 0, 2)
    return out


def _exact_qwen(case, t):
    w, b, s = t["weights"], case["batch"], case["seq"]

    def matrix(name):
        return _dequantize(w[name + ".weight"], w[name + ".scales"], w[name + ".biases"])

    x = matrix("model.embed_tokens")[t["ids"].long().reshape(-1)]
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        a = p + "self_attn."
        h = _rms(x, w[p + "input_layernorm.weight"], EPS)
        q, k, v = ((h @ matrix(a + n + "_proj").T).view(b, s, -1, DIM) for n in "qkv")
        q = _rope(_rms(q, w[a + "q_norm.weight"], EPS))
        k = _rope(_rms(k, w[a + "k_norm.weight"], EPS))
        x = x + _attend(q, k, v, _lengths(case), True).view(b * s, -1) @ matrix(a + "o_proj").T
        h = _rms(x, w[p + "post_attention_layernorm.weight"], EPS)
        gate = torch.nn.functional.silu(h @ matrix(p + "mlp.gate_proj").T)
        x = x + (gate * (h @ matrix(p + "mlp.up_proj").T)) @ matrix(p + "mlp.down_proj").T
    return x, lambda: _rms(x, w["model.norm.weight"], EPS)


def _exact_bge(case, t):
    w = {name: x.double() for name, x in t["weights"].items()}
    b, s = case["batch"], case["seq"]

    def norm(x, p):
        return torch.nn.functional.layer_norm(x, (BGE_HIDDEN,), w[p + ".weight"], w[p + ".bias"],
                                              BGE_EPS)

    def dense(x, p):
        return x @ w[p + ".weight"].T + w[p + ".bias"]

    x = (w["embeddings.word_embeddings.weight"][t["ids"].long()]
         + w["embeddings.token_type_embeddings.weight"][0]
         + w["embeddings.position_embeddings.weight"][:s]).view(b * s, -1)
    x = norm(x, "embeddings.LayerNorm")
    for i in range(case["layers"]):
        p = f"encoder.layer.{i}."
        q, k, v = (dense(x, p + "attention.self." + n).view(b, s, BGE_HEADS, -1)
                   for n in ("query", "key", "value"))
        att = _attend(q, k, v, _lengths(case), False).view(b * s, -1)
        x = norm(x + dense(att, p + "attention.output.dense"), p + "attention.output.LayerNorm")
        act = torch.nn.functional.gelu(dense(x, p + "intermediate.dense"))
        x = norm(x + dense(act, p + "output.dense"), p + "output.LayerNorm")
    return x


def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    b, s = case["batch"], case["seq"]
    if kind in ("attention", "block"):
        outs = {}
        for i in range(case["layers"]):
            if kind == "block":
                w = _dequantize(t[f"weight{i}"], t[f"scales{i}"], t[f"biases{i}"])
                y = t[f"x{i}"].double() @ w.T
                q, k, v = (p.reshape(b, s, -1, DIM) for p in
                           y.split([HEADS * DIM, KV_HEADS * DIM, KV_HEADS * DIM], 1))
                outs.update({f"q{i}": q, f"k{i}": k, f"v{i}": v})
                q, k, v = q.half().double(), k.half().double(), v.half().double()
            else:
                q, k, v = (t[f"{n}{i}"].double() for n in "qkv")
            outs[f"out{i}"] = _attend(_rope(_rms(q, t[f"q_norm{i}"], EPS)),
                                      _rope(_rms(k, t[f"k_norm{i}"], EPS)), v, _lengths(case),
                                      True)
        return outs
    if kind.startswith("qwen"):
        x, final = _exact_qwen(case, t)
        if kind == "qwen_layer":
            return {"x": x.view(b, s, -1)}
        x = final()
        rows = [i * s + n - 1 for i, n in enumerate(_lengths(case))]  # the last valid token
    else:
        x = _exact_bge(case, t)
        if kind == "bge_layer":
            return {"x": x.view(b, s, -1)}
        rows = [i * s for i in range(b)]  # the first token
    return torch.nn.functional.normalize(x[rows], dim=1)
