"""Timed workloads of the FP32 batch-1 SmolLM2-135M token loop.

Each case is one thing that a program using this framework has it do, through the entry points that such a program
calls: the native prefill and greedy generation (``flux_amd.runtime``), the layer blocks of the C ABI
(``include/flux_amd.h``) and the eager operators (``flux_amd.ops``).  A case is a dict of plain values:

* ``prefill`` (tokens): a prompt through ``NativeSmolLM2Prefill.prefill``: logits and the K/V cache it leaves.
* ``generate`` (tokens, new): the same, then ``generate_greedy(new)`` and one more ``replay()`` for the last logits.
* ``attention`` (tokens): causal GQA of one layer's prompt, ``flux_prefill_attention_f32``.
* ``mlp`` (tokens): one layer's feed-forward block over prompt rows: residual RMSNorm, gate/up + SwiGLU, down.
* ``projections`` (tokens): one layer's other GEMMs: RMSNorm, QKV with RoPE and cache rows, the output projection.
* ``decode_layer`` (context): one token through one layer as separate kernels, at the end of a ``context``-row cache.
* ``lm_head`` (vocab): final norm, LM head and greedy token of one row.
* ``eager_prompt`` (tokens): the operators an enabled Hugging Face layer calls for a prompt.
* ``eager_token`` (context): the operators it calls for one token over a cache.

Weights are N(0, 0.02) and norm weights 1, as the benchmark's; activations that follow an RMSNorm are N(0, 1).
"""

from __future__ import annotations

import ctypes
import math

import torch

from flux_amd import _native, ops, synthetic
from flux_amd.model import FINAL_FLUX_OPERATOR_CATEGORIES, enable_flux_ops
from flux_amd.runtime import NativeSmolLM2Prefill

LAYERS, HIDDEN, INTER = synthetic.LAYERS, synthetic.HIDDEN, synthetic.INTERMEDIATE
QH, KVH, D = synthetic.Q_HEADS, synthetic.KV_HEADS, synthetic.HEAD_DIM
QKV, GATE_UP, VOCAB = synthetic.QKV_WIDTH, synthetic.GATE_UP_WIDTH, synthetic.VOCAB
EPS, STD, SCALE = synthetic.RMS_EPS, synthetic.INIT_STD, D ** -0.5
MASKED = torch.finfo(torch.float32).min
LAYER_WEIGHTS = QKV * HIDDEN + HIDDEN * HIDDEN + GATE_UP * HIDDEN + HIDDEN * INTER


def listed():
    return [
        # The benchmark's long prompt: a document read in one call.
        {"name": "prefill_8192", "kind": "prefill", "tokens": 8192},
        # A chat turn: a short prompt and a reply of 64 tokens.
        {"name": "generate_128_64", "kind": "generate", "tokens": 128, "new": 64},
        # Attention of a long document's layer, and of a short question's (odd, so the last tile is ragged).
        {"name": "attention_8192", "kind": "attention", "tokens": 8192},
        {"name": "attention_301", "kind": "attention", "tokens": 301},
        # Feed-forward blocks of a mid-length prompt that fills no tile evenly, and of a one-line question.
        {"name": "mlp_3001", "kind": "mlp", "tokens": 3001},
        {"name": "mlp_45", "kind": "mlp", "tokens": 45},
        # The attention block's GEMMs at the benchmark's context lengths between the two.
        {"name": "projections_8192", "kind": "projections", "tokens": 8192},
        {"name": "projections_1000", "kind": "projections", "tokens": 1000},
        # One decoded token: a layer at the end of a long context, and the vocabulary projection that follows.
        {"name": "decode_layer_8192", "kind": "decode_layer", "context": 8192},
        {"name": "lm_head_49152", "kind": "lm_head", "vocab": VOCAB},
        # The op-at-a-time model: a layer's operators for a prompt, and for one token over a static cache.
        {"name": "eager_prompt_1024", "kind": "eager_prompt", "tokens": 1024},
        {"name": "eager_token_4096", "kind": "eager_token", "context": 4096},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["prefill", "generate", "attention", "attention", "mlp", "mlp", "projections", "projections",
                       "decode_layer", "lm_head", "eager_prompt", "eager_token"])
    if kind == "prefill":
        return {"kind": kind, "tokens": _log_int(rng, 1, 8192)}
    if kind == "generate":
        return {"kind": kind, "tokens": _log_int(rng, 1, 2048), "new": rng.randint(4, 48)}
    if kind == "decode_layer":
        return {"kind": kind, "context": _log_int(rng, 1, 16384)}
    if kind == "lm_head":
        return {"kind": kind, "vocab": _log_int(rng, 128, VOCAB)}
    if kind == "eager_prompt":
        return {"kind": kind, "tokens": _log_int(rng, 2, 2048)}
    if kind == "eager_token":
        return {"kind": kind, "context": _log_int(rng, 64, 16384)}
    return {"kind": kind, "tokens": _log_int(rng, 1, 16384)}


# ---------------------------------------------------------------------------------------------------------------
# Inputs

class _Draw:
    def __init__(self, seed, salt):
        self.generator = torch.Generator(device="cuda").manual_seed(1_000_003 * int(seed) + salt)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, device="cuda", generator=self.generator).mul_(std)

    def integers(self, high, *shape):
        return torch.randint(0, high, shape, device="cuda", generator=self.generator)


def _rope(length):
    """cos/sin [length, 64] with Hugging Face's float32 formula."""
    inv_freq = 1.0 / (synthetic.ROPE_THETA ** (torch.arange(0, D, 2, dtype=torch.float32) / D))
    freqs = torch.arange(length, dtype=torch.float32)[:, None] * inv_freq[None, :]
    table = torch.cat((freqs, freqs), dim=-1)
    return table.cos().cuda(), table.sin().cuda()


def _model_state(seed):
    d = _Draw(seed, 1)
    state = {"model.embed_tokens.weight": d.normal(VOCAB, HIDDEN, std=STD)}
    for layer in range(LAYERS):
        p = f"model.layers.{layer}."
        for key, shape in ((p + "self_attn.q_proj.weight", (QH * D, HIDDEN)),
                           (p + "self_attn.k_proj.weight", (KVH * D, HIDDEN)),
                           (p + "self_attn.v_proj.weight", (KVH * D, HIDDEN)),
                           (p + "self_attn.o_proj.weight", (HIDDEN, QH * D)),
                           (p + "mlp.gate_proj.weight", (INTER, HIDDEN)),
                           (p + "mlp.up_proj.weight", (INTER, HIDDEN)),
                           (p + "mlp.down_proj.weight", (HIDDEN, INTER))):
            state[key] = d.normal(*shape, std=STD)
        state[p + "input_layernorm.weight"] = torch.ones(HIDDEN, device="cuda")
        state[p + "post_attention_layernorm.weight"] = torch.ones(HIDDEN, device="cuda")
    state["model.norm.weight"] = torch.ones(HIDDEN, device="cuda")
    state["lm_head.weight"] = state["model.embed_tokens.weight"]
    return state


def _model(seed):
    from transformers import LlamaForCausalLM

    config = synthetic.llama_config()
    with torch.device("meta"):
        model = LlamaForCausalLM(config)
    model.load_state_dict(_model_state(seed), assign=True, strict=True)
    model.tie_weights()
    model.model.rotary_emb = type(model.model.rotary_emb)(config)
    model = model.float().eval().to("cuda")
    enable_flux_ops(model, operators=FINAL_FLUX_OPERATOR_CATEGORIES)
    return model


def _prompt(seed, tokens):
    return _Draw(seed, 2).integers(VOCAB, 1, tokens)


def _layer(seed):
    d = _Draw(seed, 3)
    return {"qkv": d.normal(QKV, HIDDEN, std=STD), "o": d.normal(HIDDEN, HIDDEN, std=STD),
            "gate_up": d.normal(GATE_UP, HIDDEN, std=STD), "down": d.normal(HIDDEN, INTER, std=STD),
            "norm": torch.ones(HIDDEN, device="cuda")}


def _inputs(case, seed):
    """The tensors a block is called with (not the whole-model kinds)."""
    kind, d = case["kind"], _Draw(seed, 4)
    if kind == "attention":
        s = case["tokens"]
        return {"q": d.normal(QH, s, D), "k": d.normal(KVH, s, D), "v": d.normal(KVH, s, D)}
    if kind == "mlp":
        s = case["tokens"]
        return {"hidden": d.normal(s, HIDDEN), "residual": d.normal(s, HIDDEN), **_layer(seed)}
    if kind == "projections":
        s = case["tokens"]
        cos, sin = _rope(s)
        return {"hidden": d.normal(s, HIDDEN), "rows": d.normal(s, HIDDEN), "cos": cos, "sin": sin, **_layer(seed)}
    if kind == "decode_layer":
        n = case["context"]
        cos, sin = _rope(n)
        return {"hidden": d.normal(HIDDEN), "k": d.normal(KVH, n, D), "v": d.normal(KVH, n, D), "cos": cos, "sin": sin,
                "position": torch.tensor([n - 1], device="cuda"), **_layer(seed)}
    if kind == "lm_head":
        return {"hidden": d.normal(HIDDEN), "norm": torch.ones(HIDDEN, device="cuda"),
                "lm_head": d.normal(case["vocab"], HIDDEN, std=STD)}
    if kind == "eager_prompt":
        s = case["tokens"]
        cos, sin = _rope(s)
        mask = torch.full((1, 1, s, s), MASKED, device="cuda").triu_(1)
        return {"hidden": d.normal(1, s, HIDDEN), "residual": d.normal(1, s, HIDDEN),
                "norm": torch.ones(HIDDEN, device="cuda"),
                # Views of the projections' [1, S, heads, 64] rows, as the model passes them.
                "q": d.normal(1, s, QH, D).transpose(1, 2), "k": d.normal(1, s, KVH, D).transpose(1, 2),
                "cos": cos[None], "sin": sin[None], "scores": d.normal(1, QH, s, s, std=8.0), "mask": mask,
                "packed": d.normal(1, s, GATE_UP)}
    n = case["context"]
    return {"hidden": d.normal(1, 1, HIDDEN), "q": d.normal(1, QH, 1, D), "k": d.normal(1, KVH, n, D),
            "v": d.normal(1, KVH, n, D), "length": torch.tensor(n - n // 8, device="cuda"), **_layer(seed)}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "generate"):
        ids = _prompt(seed, case["tokens"])
        runtime = NativeSmolLM2Prefill.capture(_model(seed), ids, max_decode_steps=case.get("new", 0))
        return {"kind": kind, "runtime": runtime, "ids": ids, "new": case.get("new", 0)}
    state = dict(_inputs(case, seed), kind=kind)

    def new(*shape, dtype=torch.float32):
        return torch.empty(*shape, dtype=dtype, device="cuda")

    lib = _native.load()
    need = ctypes.c_int64()
    if kind == "attention":
        s = case["tokens"]
        _native.check(lib.flux_prefill_attention_workspace_bytes(s, ctypes.byref(need)))
        state.update(tokens=s, out=new(s, HIDDEN), workspace=new(need.value // 4) if need.value else None)
    elif kind == "mlp":
        s = case["tokens"]
        state.update(tokens=s, normed=new(s, HIDDEN), sums=new(s, HIDDEN), act=new(s, INTER), out=new(s, HIDDEN))
    elif kind == "projections":
        s = case["tokens"]
        state.update(tokens=s, normed=new(s, HIDDEN), q_out=new(QH, s, D), k_out=new(KVH, s, D), v_out=new(KVH, s, D),
                     out=new(s, HIDDEN))
    elif kind == "decode_layer":
        _native.check(lib.flux_gqa_decode_workspace_bytes(case["context"], ctypes.byref(need)))
        state.update(context=case["context"], workspace=new(need.value // 4), workspace_bytes=need.value,
                     q_out=new(QH, D), attn=new(HIDDEN), sums=new(HIDDEN), act=new(INTER), out=new(HIDDEN))
    elif kind == "lm_head":
        _native.check(lib.flux_lm_head_workspace_bytes(ctypes.byref(need)))
        state.update(vocab=case["vocab"], workspace=new(need.value // 4), workspace_bytes=need.value,
                     logits=new(case["vocab"]), token=new(1, dtype=torch.int64))
    elif kind == "eager_token":
        state.update(qkv_out=new(1, 1, QKV), o_out=new(1, 1, HIDDEN), act=new(1, 1, INTER))
    return state


# ---------------------------------------------------------------------------------------------------------------
# One pass

def run(state):
    kind = state["kind"]
    if kind in ("prefill", "generate"):
        runtime = state["runtime"]
        result = {"prompt_logits": runtime.prefill(state["ids"])}
        if kind == "generate":
            result["tokens"] = runtime.generate_greedy(state["new"])
            result["logits"] = runtime.replay()
        result["key_cache"], result["value_cache"] = runtime.key_cache, runtime.value_cache
        return result
    if kind == "eager_prompt":
        with torch.inference_mode():
            normed, sums = ops.residual_rmsnorm_native(state["hidden"], state["residual"], state["norm"], EPS)
            q, k = ops.rope_native(state["q"], state["k"], state["cos"], state["sin"])
            probs = ops.attention_score_softmax_native(state["scores"], state["mask"], SCALE)
            act = ops.packed_swiglu_native(state["packed"])
        return {"normed": normed, "sums": sums, "q": q, "k": k, "probs": probs, "act": act}
    if kind == "eager_token":
        with torch.inference_mode():
            normed = ops.rms_norm_native(state["hidden"], state["norm"], EPS)
            qkv = ops.decode_projection_out(normed, state["qkv"], state["qkv_out"])
            attn = ops.gqa_decode_attention_native(state["q"], state["k"], state["v"], None, SCALE, state["length"])
            out = ops.decode_projection_out(attn.view(1, 1, HIDDEN), state["o"], state["o_out"])
            act = ops.packed_gate_up_swiglu_native_out(normed, state["gate_up"], state["act"])
        return {"normed": normed, "qkv": qkv, "attn": attn, "out": out, "act": act}

    lib, check, stream = _native.load(), _native.check, _native.current_stream()
    p = {k: v.data_ptr() for k, v in state.items() if isinstance(v, torch.Tensor)}
    if kind == "attention":
        s = state["tokens"]
        check(lib.flux_prefill_attention_f32(p["q"], p["k"], p["v"], s, s, SCALE, p.get("workspace"), p["out"], stream))
        return {"out": state["out"]}
    if kind == "mlp":
        s = state["tokens"]
        check(lib.flux_residual_rmsnorm_f32(p["hidden"], p["residual"], p["norm"], p["normed"], p["sums"], s, HIDDEN,
                                            EPS, stream))
        check(lib.flux_gate_up_swiglu_rows_f32(p["normed"], p["gate_up"], p["act"], s, stream))
        check(lib.flux_linear_f32(p["act"], p["down"], p["sums"], p["out"], s, HIDDEN, INTER, stream))
        return {k: state[k] for k in ("normed", "sums", "act", "out")}
    if kind == "projections":
        s = state["tokens"]
        check(lib.flux_rmsnorm_f32(p["hidden"], p["norm"], p["normed"], s, HIDDEN, EPS, stream))
        check(lib.flux_qkv_rope_cache_rows_f32(p["normed"], p["qkv"], p["cos"], p["sin"], s, p["q_out"], p["k_out"],
                                               p["v_out"], s, stream))
        check(lib.flux_linear_f32(p["rows"], p["o"], p["hidden"], p["out"], s, HIDDEN, HIDDEN, stream))
        return {k: state[k] for k in ("normed", "q_out", "k_out", "v_out", "out")}
    if kind == "decode_layer":
        n = state["context"]
        check(lib.flux_qkv_rope_cache_f32(p["hidden"], p["norm"], EPS, p["qkv"], p["cos"], p["sin"], p["position"], n,
                                          p["k"], p["v"], p["q_out"], stream))
        check(lib.flux_gqa_decode_attention_f32(p["q_out"], p["k"], p["v"], p["position"], n, SCALE, p["workspace"],
                                                state["workspace_bytes"], p["attn"], stream))
        check(lib.flux_linear576_f32(p["attn"], p["o"], p["hidden"], p["sums"], HIDDEN, stream))
        check(lib.flux_gate_up_swiglu_f32(p["sums"], p["norm"], EPS, p["gate_up"], p["act"], stream))
        check(lib.flux_down_residual_f32(p["act"], p["down"], p["sums"], p["out"], stream))
        return {k: state[k] for k in ("k", "v", "q_out", "attn", "sums", "act", "out")}
    check(lib.flux_lm_head_argmax_f32(p["hidden"], p["norm"], EPS, p["lm_head"], state["vocab"], p["logits"],
                                      p["token"], p["workspace"], state["workspace_bytes"], stream))
    return {"logits": state["logits"], "token": state["token"]}


# ---------------------------------------------------------------------------------------------------------------
# What a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind in ("prefill", "generate"):
        s = case["tokens"]
        steps = case.get("new", 0)  # decode steps: new - 1 of generate_greedy, one replay
        pairs = s * (s + 1) // 2
        flops = 2 * LAYERS * LAYER_WEIGHTS * s + 4 * D * QH * LAYERS * pairs + 2 * VOCAB * HIDDEN
        nbytes = 4 * (LAYERS * LAYER_WEIGHTS + VOCAB * HIDDEN + s * HIDDEN + VOCAB) + 8 * LAYERS * KVH * D * s
        for t in range(steps):
            attended = s + 1 + t
            flops += 2 * (LAYERS * LAYER_WEIGHTS + VOCAB * HIDDEN) + 4 * D * QH * LAYERS * attended
            nbytes += 4 * (LAYERS * LAYER_WEIGHTS + VOCAB * HIDDEN + VOCAB) + 8 * LAYERS * KVH * D * attended
        return {"bytes": nbytes, "flops": flops}
    if kind == "attention":
        s = case["tokens"]
        return {"bytes": 4 * s * D * (2 * QH + 2 * KVH), "flops": 4 * D * QH * (s * (s + 1) // 2)}
    if kind == "mlp":
        s = case["tokens"]
        weights = (GATE_UP + INTER) * HIDDEN
        return {"bytes": 4 * (weights + s * (5 * HIDDEN + INTER)), "flops": 2 * weights * s}
    if kind == "projections":
        s = case["tokens"]
        weights = (QKV + HIDDEN) * HIDDEN
        return {"bytes": 4 * (weights + s * (4 * HIDDEN + QKV + 2 * D)), "flops": 2 * weights * s}
    if kind == "decode_layer":
        n = case["context"]
        return {"bytes": 4 * (LAYER_WEIGHTS + 2 * KVH * D * n), "flops": 2 * LAYER_WEIGHTS + 4 * D * QH * n}
    if kind == "lm_head":
        return {"bytes": 4 * (case["vocab"] * (HIDDEN + 1) + 2 * HIDDEN), "flops": 2 * case["vocab"] * HIDDEN}
    if kind == "eager_prompt":
        s = case["tokens"]
        return {"bytes": 4 * (s * (4 * HIDDEN + 2 * (QH + KVH) * D + 2 * D + GATE_UP + INTER) + s * s * (2 * QH + 1)),
                "flops": s * (8 * HIDDEN + 3 * (QH + KVH) * D + 6 * INTER) + 6 * QH * s * s}
    n = case["context"] - case["context"] // 8
    weights = (QKV + HIDDEN + GATE_UP) * HIDDEN
    return {"bytes": 4 * (weights + 2 * KVH * D * n), "flops": 2 * weights + 4 * D * QH * n}


def tolerance(case):
    if case["kind"] in ("prefill", "generate"):
        return {"rel": 8e-6, "max": 1e-3, "differ": 0.0}
    return {"rel": 4e-6, "max": 2e-4, "differ": 0.0}


# ---------------------------------------------------------------------------------------------------------------
# The same in 64 bits

def _norm64(x, weight):
    return weight * (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS))


def _rotate64(x, cos, sin):
    half = torch.cat((-x[..., D // 2:], x[..., :D // 2]), dim=-1)
    return x * cos + half * sin


def _attention64(q, k, v, first=0):
    """q [9, S, 64] at positions first.. over k, v [3, N, 64]; rows [S, 576]."""
    s, n = q.shape[1], k.shape[1]
    out = torch.empty(s, HIDDEN, dtype=torch.float64, device=q.device)
    keys = torch.arange(n, device=q.device)
    for h in range(QH):
        g = h // (QH // KVH)
        for b in range(0, s, 2048):
            e = min(s, b + 2048)
            scores = (q[h, b:e] @ k[g].T).mul_(SCALE)
            last = torch.arange(b, e, device=q.device) + first
            scores.masked_fill_(keys[None, :] > last[:, None], -math.inf)
            out[b:e, h * D:(h + 1) * D] = torch.softmax(scores, -1) @ v[g]
    return out


def _swiglu64(packed):
    gate, up = packed.chunk(2, dim=-1)
    return gate * torch.sigmoid(gate) * up


def _model64(case, seed):
    state = {k: v.double() for k, v in _model_state(seed).items()}
    s, new = case["tokens"], case.get("new", 0)
    cos, sin = (t.double() for t in _rope(s + new))
    keys = torch.zeros(LAYERS, 1, KVH, s + new, D, dtype=torch.float64, device="cuda")
    values = torch.zeros_like(keys)

    def forward(ids, first):
        n = ids.shape[0]
        h = state["model.embed_tokens.weight"][ids]
        c, t = cos[first:first + n], sin[first:first + n]
        for i in range(LAYERS):
            p = f"model.layers.{i}."
            x = _norm64(h, state[p + "input_layernorm.weight"])
            q = (x @ state[p + "self_attn.q_proj.weight"].T).view(n, QH, D).transpose(0, 1)
            k = (x @ state[p + "self_attn.k_proj.weight"].T).view(n, KVH, D).transpose(0, 1)
            v = (x @ state[p + "self_attn.v_proj.weight"].T).view(n, KVH, D).transpose(0, 1)
            keys[i, 0, :, first:first + n] = _rotate64(k, c, t)
            values[i, 0, :, first:first + n] = v
            rows = _attention64(_rotate64(q, c, t), keys[i, 0, :, :first + n], values[i, 0, :, :first + n], first)
            h = h + rows @ state[p + "self_attn.o_proj.weight"].T
            x = _norm64(h, state[p + "post_attention_layernorm.weight"])
            gate = x @ state[p + "mlp.gate_proj.weight"].T
            up = x @ state[p + "mlp.up_proj.weight"].T
            h = h + (gate * torch.sigmoid(gate) * up) @ state[p + "mlp.down_proj.weight"].T
        return _norm64(h[-1], state["model.norm.weight"]) @ state["lm_head.weight"].T

    logits = forward(_prompt(seed, s)[0], 0)
    result = {"prompt_logits": logits.view(1, 1, VOCAB)}
    if new:
        tokens = [logits.argmax()]
        for t in range(new):
            logits = forward(tokens[-1].view(1), s + t)
            tokens.append(logits.argmax())
        result["tokens"] = torch.stack(tokens[:new]).view(1, new)
        result["logits"] = logits.view(1, 1, VOCAB)
    result["key_cache"], result["value_cache"] = keys, values
    return result


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "generate"):
        return _model64(case, seed)
    x = {k: v.double() if v.dtype == torch.float32 else v for k, v in _inputs(case, seed).items()}
    if kind == "attention":
        return {"out": _attention64(x["q"], x["k"], x["v"])}
    if kind == "mlp":
        sums = x["hidden"] + x["residual"]
        normed = _norm64(sums, x["norm"])
        act = _swiglu64(normed @ x["gate_up"].T)
        return {"normed": normed, "sums": sums, "act": act, "out": sums + act @ x["down"].T}
    if kind == "projections":
        s = case["tokens"]
        normed = _norm64(x["hidden"], x["norm"])
        heads = (normed @ x["qkv"].T).view(s, QH + 2 * KVH, D).transpose(0, 1)
        return {"normed": normed, "q_out": _rotate64(heads[:QH], x["cos"], x["sin"]),
                "k_out": _rotate64(heads[QH:QH + KVH], x["cos"], x["sin"]), "v_out": heads[QH + KVH:],
                "out": x["hidden"] + x["rows"] @ x["o"].T}
    if kind == "decode_layer":
        n = case["context"]
        heads = (_norm64(x["hidden"], x["norm"]) @ x["qkv"].T).view(QH + 2 * KVH, D)
        q = _rotate64(heads[:QH], x["cos"][n - 1], x["sin"][n - 1])
        x["k"][:, n - 1] = _rotate64(heads[QH:QH + KVH], x["cos"][n - 1], x["sin"][n - 1])
        x["v"][:, n - 1] = heads[QH + KVH:]
        attn = _attention64(q[:, None], x["k"], x["v"], n - 1)[0]
        sums = x["hidden"] + attn @ x["o"].T
        act = _swiglu64(_norm64(sums, x["norm"]) @ x["gate_up"].T)
        return {"k": x["k"], "v": x["v"], "q_out": q, "attn": attn, "sums": sums, "act": act,
                "out": sums + act @ x["down"].T}
    if kind == "lm_head":
        logits = _norm64(x["hidden"], x["norm"]) @ x["lm_head"].T
        return {"logits": logits, "token": logits.argmax().view(1)}
    if kind == "eager_prompt":
        sums = x["hidden"] + x["residual"]
        return {"normed": _norm64(sums, x["norm"]), "sums": sums, "q": _rotate64(x["q"], x["cos"], x["sin"]),
                "k": _rotate64(x["k"], x["cos"], x["sin"]), "probs": torch.softmax(x["scores"] * SCALE + x["mask"], -1),
                "act": _swiglu64(x["packed"])}
    n = case["context"] - case["context"] // 8
    normed = _norm64(x["hidden"], x["norm"])
    attn = _attention64(x["q"][0], x["k"][0, :, :n], x["v"][0, :, :n], n - 1)
    return {"normed": normed, "qkv": normed @ x["qkv"].T, "attn": attn.view(1, QH, 1, D),
            "out": (attn @ x["o"].T).view(1, 1, HIDDEN), "act": _swiglu64(normed @ x["gate_up"].T)}
