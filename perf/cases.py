"""The work a user of the KV data path has it do, as cases that can be timed and checked.

A case is a dict of plain values; ``op`` says which entry points one pass calls:

* ``prefill``  one layer of a prompt (or of a later chunk of it, ``past`` > 0): the K/V write into
  the cache and the causal attention over it (``mha._update_kv_cache`` + ``mha.FlashCrossAttention``);
* ``handoff``  the live rows of every layer's prefill cache into one packed buffer and from there
  into the decode cache (``ops.pack_live`` + ``ops.unpack_live``);
* ``step``     one decode step over ``layers`` layers called eagerly, each an append fused with its
  attention (``mha.update_and_attend``), at one offset for the batch or at per-sample lengths that
  only the device knows;
* ``replay``   the same step planned on the host's lengths and replayed as a HIP graph
  (``ops.DecodeStepGraph``), as a serving loop keeps it;
* ``ft``       one layer on FasterTransformer caches: the prompt's store, then four decode steps at
  per-sample lengths with rotary embedding;
* ``legacy``   the older scripts' batching: every request's tensor-parallel shards joined along the
  heads, then the requests zero-padded into one batch (``kv_formats``);
* ``model``    a small Llama (``llama.LlamaHost``): prompt, handoff and three decode steps, logits out.

Shapes are those of ``hexgen2_amd.workloads`` and of the reference pilot's prompts, or generic.
"""
from __future__ import annotations

import math

import torch

from hexgen2_amd import kv_formats, mha, ops
from hexgen2_amd.generation import InferenceParams
from hexgen2_amd.llama import LlamaHost, LlamaShape

_DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
_FT_STEPS, _MODEL_STEPS = 4, 3

# (q_heads, kv_heads, head_dim, dtype, layers) of the workloads
_TINY = (4, 4, 16, "float32", 2)
_TINYLLAMA = (32, 4, 64, "float16", 22)
_LLAMA2_7B = (32, 32, 128, "float16", 32)
_LLAMA2_70B_TP8 = (8, 1, 128, "bfloat16", 80)
_LLAMA3_8B = (32, 8, 128, "bfloat16", 32)
_GEOMETRIES = (_TINYLLAMA, _LLAMA2_7B, _LLAMA2_70B_TP8, _LLAMA3_8B)


def _case(op, geometry, name=None, **sizes):
    q_heads, kv_heads, head_dim, dtype, layers = geometry
    case = dict(op=op, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, dtype=dtype, layers=layers)
    case.update(sizes)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # the pilot's 82-token prompt: one layer of a short prompt, where launches count
        _case("prefill", _TINYLLAMA, "prefill-tinyllama-82", batch=1, length=82, past=0),
        # the second chunk of two prompts of odd length, one query head per KV head
        _case("prefill", _LLAMA2_7B, "prefill-llama2-7b-chunk", batch=2, length=611, past=512),
        # the longest prompt of the Llama-3-8B workload
        _case("prefill", _LLAMA3_8B, "prefill-llama3-8b-8192", batch=1, length=8192, past=0),
        # the handoff of one request of the pilot's model
        _case("handoff", _TINYLLAMA, "handoff-tinyllama-512", batch=1, lo=512, hi=512, capacity=2048),
        # the handoff of a ragged batch of the largest workload
        _case("handoff", _LLAMA3_8B, "handoff-llama3-8b", batch=8, lo=128, hi=8192, capacity=8192),
        # one request decoding eagerly, as Engine.decode does it: every layer a call of a few KB
        _case("step", _TINYLLAMA, "step-tinyllama-eager", batch=1, lo=577, hi=577, capacity=2048, ragged=False),
        # a ragged batch whose lengths only the device knows (lengths_per_sample)
        _case("step", _LLAMA2_7B, "step-llama2-7b-ragged", batch=8, lo=256, hi=2048, capacity=4096, ragged=True,
              layers=2),
        # the tensor-parallel share of a large model: little work per layer and call, replayed
        _case("replay", _LLAMA2_70B_TP8, "replay-llama2-70b-tp8", batch=32, lo=512, hi=4096, capacity=4128,
              layers=16),
        # the largest decode batch: about a gigabyte of keys and values a layer
        _case("replay", _LLAMA3_8B, "replay-llama3-8b", batch=64, lo=128, hi=8192, capacity=8448, layers=4),
        # the FasterTransformer layout: prompt store and decode steps of a ragged batch
        _case("ft", _LLAMA3_8B, "ft-llama3-8b", batch=16, lo=128, hi=2048, capacity=2304),
        # four requests prefilled on two tensor-parallel shards, batched for one decoder
        _case("legacy", _LLAMA2_7B, "legacy-llama2-7b", batch=4, lo=128, hi=2048, shards=2, layers=8),
        # a whole request: prompt, handoff, decode
        _case("model", _TINYLLAMA, "model-prompt-512", length=512, layers=4),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _most_rows(geometry, most_bytes, most, positions):
    """The largest batch, up to ``most``, whose caches of ``positions`` positions hold ``most_bytes``."""
    _, kv_heads, head_dim, dtype, _ = geometry
    return max(1, min(most, most_bytes // (positions * 2 * kv_heads * head_dim * (4 if dtype == "float32" else 2))))


def draw(rng):
    op = rng.choice(("prefill", "prefill", "prefill", "handoff", "handoff", "step", "step", "replay", "replay",
                     "ft", "legacy", "model"))
    # now and then the fp32 correctness model, the smallest geometry there is
    geometry = _TINY if op in ("prefill", "step") and rng.random() < 0.1 else rng.choice(_GEOMETRIES)
    layers = geometry[4]
    if op == "prefill":
        length = _log_int(rng, 6, 1024 if geometry is _TINY else 6144)
        batch = rng.randint(1, max(1, min(8, 6144 // length)))
        past = _log_int(rng, 16, 4096) if length <= 1024 and rng.random() < 0.4 else 0
        return _case(op, geometry, batch=batch, length=length, past=past)
    if op == "handoff":
        hi = _log_int(rng, 64, 8192)
        layers = max(2, layers // rng.randint(1, 4))
        return _case(op, geometry, batch=rng.randint(1, _most_rows(geometry, 7 << 29, 8, layers * hi)),
                     lo=max(1, hi // rng.randint(1, 32)), hi=hi, capacity=hi + rng.randint(1, 512), layers=layers)
    if op == "step":
        hi = _log_int(rng, 16, 2048)
        ragged = rng.random() < 0.5
        lo = max(1, hi // rng.randint(2, 16)) if ragged else hi
        return _case(op, geometry, batch=rng.randint(2, 16) if ragged else 1, lo=lo, hi=hi,
                     capacity=hi + rng.randint(1, 2048), ragged=ragged, layers=rng.randint(1, min(4, layers)))
    if op == "replay":
        hi = _log_int(rng, 64, 8192)
        return _case(op, geometry, batch=_log_int(rng, 1, _most_rows(geometry, 3 << 30, 64, 2 * hi)),
                     lo=max(1, hi // rng.randint(1, 32)), hi=hi, capacity=hi + rng.randint(1, 256), layers=2)
    if op == "ft":
        hi = _log_int(rng, 32, 2048)
        return _case(op, geometry, batch=rng.randint(1, 16), lo=max(1, hi // rng.randint(1, 16)), hi=hi,
                     capacity=hi + rng.randint(_FT_STEPS, 256))
    if op == "legacy":
        hi = _log_int(rng, 16, 2048)
        shards = 1 if geometry[1] == 1 else rng.choice((2, 4))
        return _case(op, geometry, batch=rng.randint(2, 6), lo=max(1, hi // rng.randint(1, 16)), hi=hi,
                     shards=shards, layers=rng.randint(2, 8))
    return _case(op, geometry, length=_log_int(rng, 6, 512), layers=rng.randint(2, 4 if geometry[0] * geometry[2] <= 2048 else 2))


# ---------------------------------------------------------------- inputs ---


def _lens(case):
    """The batch's cached lengths: part of the case, not of its inputs, so
    that every seed moves the same bytes."""
    if case["lo"] == case["hi"]:
        return [case["hi"]] * case["batch"]
    g = torch.Generator().manual_seed(case["batch"] * 100003 + case["hi"])
    return torch.randint(case["lo"], case["hi"] + 1, (case["batch"],), generator=g).tolist()


class _Inputs:
    """Keys, values and queries of a case from its seed: unit variance, the
    queries at twice that, so that the softmax is neither flat nor one-hot."""

    def __init__(self, case, seed):
        self.dtype = _DTYPES[case["dtype"]]
        self.device = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.device).manual_seed(seed)

    def normal(self, *shape, std=1.0):
        t = torch.randn(shape, generator=self.gen, device=self.device, dtype=self.dtype)
        return t if std == 1.0 else t.mul_(std)

    def ints(self, values):
        return torch.tensor(values, dtype=torch.int32, device=self.device)


def _geometry(case):
    return case["q_heads"], case["kv_heads"], case["head_dim"]


def _model_shape(case):
    hidden = case["q_heads"] * case["head_dim"]
    return LlamaShape(vocab_size=4000, hidden_size=hidden, intermediate_size=hidden * 11 // 4,
                      num_hidden_layers=case["layers"], num_attention_heads=case["q_heads"],
                      num_key_value_heads=case["kv_heads"], rms_norm_eps=1e-5)


def _model_weights(case, inputs):
    s = _model_shape(case)
    d, kv = s.head_dim, s.num_key_value_heads * s.head_dim

    def matrix(rows, cols):
        return inputs.normal(rows, cols, std=cols ** -0.5)

    def gain():
        return torch.ones(s.hidden_size, dtype=inputs.dtype, device=inputs.device)

    w = {"model.embed_tokens.weight": inputs.normal(s.vocab_size, s.hidden_size), "model.norm.weight": gain(),
         "lm_head.weight": matrix(s.vocab_size, s.hidden_size)}
    for i in range(s.num_hidden_layers):
        p = f"model.layers.{i}."
        w.update({p + "input_layernorm.weight": gain(), p + "post_attention_layernorm.weight": gain(),
                  p + "self_attn.q_proj.weight": matrix(s.num_attention_heads * d, s.hidden_size),
                  p + "self_attn.k_proj.weight": matrix(kv, s.hidden_size),
                  p + "self_attn.v_proj.weight": matrix(kv, s.hidden_size),
                  p + "self_attn.o_proj.weight": matrix(s.hidden_size, s.num_attention_heads * d),
                  p + "mlp.gate_proj.weight": matrix(s.intermediate_size, s.hidden_size),
                  p + "mlp.up_proj.weight": matrix(s.intermediate_size, s.hidden_size),
                  p + "mlp.down_proj.weight": matrix(s.hidden_size, s.intermediate_size)})
    return s, w


def _model_tokens(case, inputs):
    ids = torch.randint(0, 4000, (1, case["length"] + _MODEL_STEPS), generator=inputs.gen, device=inputs.device)
    return ids[:, :case["length"]], [ids[:, case["length"] + t:case["length"] + t + 1] for t in range(_MODEL_STEPS)]


def _tensors(case, seed):
    """The inputs of every op but ``model``, by name."""
    x = _Inputs(case, seed)
    hq, hkv, d = _geometry(case)
    op = case["op"]
    if op == "prefill":
        b, s = case["batch"], case["length"]
        return dict(cache=x.normal(b, case["past"] + s, 2, hkv, d), kv=x.normal(b, s, 2, hkv, d),
                    q=x.normal(b, s, hq, d, std=2.0))
    if op in ("step", "replay"):
        n, b = case["layers"], case["batch"]
        return dict(cache=x.normal(n, b, case["capacity"], 2, hkv, d), kv=x.normal(n, b, 1, 2, hkv, d),
                    q=x.normal(n, b, 1, hq, d, std=2.0))
    if op == "handoff":
        return dict(cache=x.normal(case["layers"], case["batch"], case["capacity"], 2, hkv, d))
    if op == "ft":
        b = case["batch"]
        return dict(prompt=x.normal(b, case["hi"], 2, hkv, d), kv=x.normal(_FT_STEPS, b, 1, 2, hkv, d),
                    q=x.normal(_FT_STEPS, b, 1, hq, d, std=2.0))
    if op == "legacy":
        return dict(shards=[[{i: x.normal(1, n, 2, hkv // case["shards"], d) for i in range(case["layers"])}
                             for _ in range(case["shards"])] for n in _lens(case)])
    raise KeyError(op)


def prepare(case, seed):
    op = case["op"]
    x = _Inputs(case, seed)
    state = dict(case=case)
    if op == "model":
        shape, weights = _model_weights(case, x)
        state["model"] = LlamaHost(shape, weights, x.device, x.dtype)
        state["prompt"], state["tokens"] = _model_tokens(case, x)
        return state
    state.update(_tensors(case, seed))
    hq, hkv, d = _geometry(case)
    if op == "prefill":
        b, s, past = case["batch"], case["length"], case["past"]
        state["params"] = InferenceParams(max_sequence_len=past + s, max_batch_size=b, sequence_len_offset=past,
                                          key_value_memory_dict={0: state["cache"]})
        state["attention"] = mha.FlashCrossAttention(causal=True, softmax_scale=d ** -0.5)
    elif op == "handoff":
        state["lens"] = _lens(case)
        state["decode"] = torch.zeros_like(state["cache"])
    elif op == "step":
        lens = _lens(case)
        state["params"] = InferenceParams(
            max_sequence_len=case["capacity"], max_batch_size=case["batch"], sequence_len_offset=max(lens),
            key_value_memory_dict=dict(enumerate(state["cache"].unbind(0))),
            lengths_per_sample=x.ints(lens) if case["ragged"] else None)
    elif op == "replay":
        lens = _lens(case)
        q, cache = state["q"], state["cache"]
        kv = state["kv"].squeeze(2)
        out = torch.zeros_like(q)
        positions = x.ints(lens)
        # one eager call first: the code objects load on the first launch
        ops.decode_attention(q[0], cache[0], max_seqlen=max(lens) + 1, seqlens=positions, kv_new=kv[0], lens=lens)
        state.update(out=out, kv=kv, positions=positions,
                     graph=ops.DecodeStepGraph(q, cache, out, kv, positions, max(lens) + 1, lens=lens))
    elif op == "ft":
        lens = _lens(case)
        caches = mha.inference_cache(case["batch"], case["capacity"], hkv, d, x.dtype, x.device, fused_ft_kernel=True)
        for t in caches:
            t.zero_()
        state["params"] = InferenceParams(max_sequence_len=case["capacity"], max_batch_size=case["batch"],
                                          key_value_memory_dict={0: caches}, fused_ft_kernel=True)
        state["positions"] = [x.ints([n + t for n in lens]) for t in range(_FT_STEPS)]
    return state


# ---------------------------------------------------------------- passes ---


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "prefill":
        view = mha._update_kv_cache(state["kv"], state["params"], 0)
        return dict(context=state["attention"](state["q"], view), cache=view)
    if op == "handoff":
        packed = ops.pack_live(state["cache"], state["lens"])
        ops.unpack_live(packed, state["decode"], state["lens"])
        return dict(packed=packed, cache=state["decode"])
    if op == "step":
        q, kv, params = state["q"], state["kv"], state["params"]
        scale = case["head_dim"] ** -0.5
        outs = [mha.update_and_attend(q[l], kv[l], params, l, scale) for l in range(case["layers"])]
        return dict(context=outs, cache=state["cache"])
    if op == "replay":
        state["graph"].restart()
        state["graph"].replay()
        return dict(context=state["out"], cache=state["cache"], positions=state["positions"])
    if op == "ft":
        params, d = state["params"], case["head_dim"]
        params.sequence_len_offset, params.lengths_per_sample = 0, None
        mha._update_kv_cache(state["prompt"], params, 0)
        outs = []
        for t in range(_FT_STEPS):
            params.sequence_len_offset, params.lengths_per_sample = case["hi"] + t, state["positions"][t]
            outs.append(mha._apply_rotary_single_query_attention(state["q"][t], params, 0, d, 10000.0,
                                                                 kv=state["kv"][t]))
        return dict(context=outs, cache=list(params.key_value_memory_dict[0]))
    if op == "legacy":
        return kv_formats.batch_key_value_memory_dicts([kv_formats.concat_dicts(s) for s in state["shards"]])
    # model: prompt, handoff of the live rows, decode steps on the decode side's cache
    model, n = state["model"], case["length"]
    with torch.inference_mode():
        params = InferenceParams(max_sequence_len=n + _MODEL_STEPS)
        logits = [model.forward(state["prompt"], params)]
        layers = [params.key_value_memory_dict[i] for i in range(case["layers"])]
        packed = ops.pack_live(layers, [n])
        full = torch.zeros((case["layers"], *layers[0].shape), dtype=model.dtype, device=model.device)
        ops.unpack_live(packed, full, [n])
        params = InferenceParams(max_sequence_len=n + _MODEL_STEPS, sequence_len_offset=n,
                                 key_value_memory_dict=dict(enumerate(full.unbind(0))))
        for token in state["tokens"]:
            logits.append(model.forward(token, params, fused_append=True))
            params.sequence_len_offset += 1
    return dict(logits=logits, cache=full)


# ------------------------------------------------------------------ work ---


def work(case):
    hq, hkv, d = _geometry(case)
    elem = 4 if case["dtype"] == "float32" else 2
    row = 2 * hkv * d * elem
    op = case["op"]
    if op == "prefill":
        b, s, past = case["batch"], case["length"], case["past"]
        keys = s * past + s * (s + 1) // 2
        # q in, out, new K/V in and into the cache, earlier K/V in
        return dict(bytes=b * (2 * s * hq * d * elem + (2 * s + past) * row), flops=4.0 * b * hq * d * keys)
    if op == "handoff":
        return dict(bytes=4 * case["layers"] * sum(_lens(case)) * row, flops=0)
    if op in ("step", "replay"):
        lens = _lens(case)
        one = (sum(lens) + 2 * len(lens)) * row + 2 * len(lens) * hq * d * elem
        return dict(bytes=case["layers"] * one, flops=4.0 * case["layers"] * hq * d * (sum(lens) + len(lens)))
    if op == "ft":
        lens = _lens(case)
        step = (sum(lens) + 2 * len(lens)) * row + 2 * len(lens) * hq * d * elem
        return dict(bytes=2 * case["batch"] * case["hi"] * row + _FT_STEPS * step,
                    flops=4.0 * _FT_STEPS * hq * d * sum(lens))
    if op == "legacy":
        lens = _lens(case)
        # shards in, joined; joined in, padded batch out (the joined caches are a result of their own)
        return dict(bytes=case["layers"] * row * (3 * sum(lens) + len(lens) * max(lens)), flops=0)
    s = _model_shape(case)
    n = case["length"]
    per_layer = s.hidden_size * (2 * hq * d + 2 * hkv * d + 3 * s.intermediate_size)
    params = case["layers"] * per_layer + s.vocab_size * s.hidden_size
    flops = 2.0 * case["layers"] * per_layer * (n + _MODEL_STEPS) + 4.0 * case["layers"] * hq * d * n * n / 2
    return dict(bytes=(1 + _MODEL_STEPS) * params * elem + 5 * case["layers"] * n * row, flops=flops)


def tolerance(case):
    if case["op"] in ("handoff", "legacy"):
        return "exact"
    if case["op"] == "model":
        # a rounding of one layer travels through those that follow
        return {"rel": {"float16": 4e-3, "bfloat16": 2.5e-2, "float32": 1e-4}[case["dtype"]]}
    # sums in fp32 rounded once to the data type: a result on the edge of two values may fall either way
    return {"rel": {"float16": 4e-4, "bfloat16": 2e-3, "float32": 1e-5}[case["dtype"]]}


# ----------------------------------------------------- the same in 64 bits ---


def _softmax_attend(q, k, v, scale, first):
    """``q [n, H, D]`` over ``k, v [S, Hkv, D]`` in 64 bits, query t seeing
    keys [0, first + t)."""
    n, hq, d = q.shape
    k = k.double().repeat_interleave(hq // k.shape[1], dim=1).permute(1, 2, 0).contiguous()
    v = v.double().repeat_interleave(hq // v.shape[1], dim=1).transpose(0, 1).contiguous()
    rows = []
    for t0 in range(0, n, 512):
        t1 = min(n, t0 + 512)
        seen = first + t1 - 1
        scores = torch.matmul(q[t0:t1].double().transpose(0, 1).contiguous(), k[:, :, :seen]) * scale
        limit = torch.arange(first + t0, first + t1, device=q.device)
        hidden = torch.arange(seen, device=q.device)[None, :] >= limit[:, None]
        scores.masked_fill_(hidden, -math.inf)
        rows.append(torch.matmul(torch.softmax(scores, -1), v[:, :seen]).transpose(0, 1))
    return torch.cat(rows)


def _turn(x, positions, base):
    """GPT-NeoX rotary of ``x [n, H, D]`` at ``positions [n]`` in 64 bits."""
    half = x.shape[-1] // 2
    j = torch.arange(half, device=x.device, dtype=torch.float64)
    angle = positions.double()[:, None] * base ** (-j / half)[None, :]
    cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]
    a, b = x.double()[..., :half], x.double()[..., half:]
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def _exact_model(case, seed):
    x = _Inputs(case, seed)
    s, w = _model_weights(case, x)
    prompt, tokens = _model_tokens(case, x)
    w = {k: v.double() for k, v in w.items()}
    ids = torch.cat([prompt, *tokens], dim=1)[0]
    n, d = ids.shape[0], s.head_dim

    def norm(h, g):
        return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + s.rms_norm_eps) * g

    h = w["model.embed_tokens.weight"][ids]
    at = torch.arange(n, device=h.device)
    for i in range(s.num_hidden_layers):
        p = f"model.layers.{i}."
        y = norm(h, w[p + "input_layernorm.weight"])
        q = (y @ w[p + "self_attn.q_proj.weight"].T).view(n, -1, d)
        k = (y @ w[p + "self_attn.k_proj.weight"].T).view(n, -1, d)
        v = (y @ w[p + "self_attn.v_proj.weight"].T).view(n, -1, d)
        c = _softmax_attend(_turn(q, at, s.rope_theta), _turn(k, at, s.rope_theta), v, d ** -0.5, 1)
        h = h + c.reshape(n, -1) @ w[p + "self_attn.o_proj.weight"].T
        y = norm(h, w[p + "post_attention_layernorm.weight"])
        gate = torch.nn.functional.silu(y @ w[p + "mlp.gate_proj.weight"].T)
        h = h + (gate * (y @ w[p + "mlp.up_proj.weight"].T)) @ w[p + "mlp.down_proj.weight"].T
    logits = norm(h, w["model.norm.weight"]) @ w["lm_head.weight"].T
    return dict(logits=[logits[case["length"] - 1 + t][None] for t in range(1 + _MODEL_STEPS)], cache=None)


def exact(case, seed):
    op = case["op"]
    if op in ("handoff", "legacy"):
        return None  # bytes moved, nothing computed
    if op == "model":
        return _exact_model(case, seed)
    x = _tensors(case, seed)
    scale = case["head_dim"] ** -0.5
    if op == "prefill":
        past = case["past"]
        context = []
        for b in range(case["batch"]):
            whole = torch.cat((x["cache"][b, :past], x["kv"][b]))
            context.append(_softmax_attend(x["q"][b], whole[:, 0], whole[:, 1], scale, past + 1))
        return dict(context=torch.stack(context), cache=None)
    if op in ("step", "replay"):
        lens = _lens(case)
        outs = []
        for l in range(case["layers"]):
            rows = []
            for b, n in enumerate(lens):
                whole = torch.cat((x["cache"][l, b, :n], x["kv"][l, b]))
                rows.append(_softmax_attend(x["q"][l, b], whole[:, 0], whole[:, 1], scale, n + 1))
            outs.append(torch.stack(rows))
        if op == "replay":
            return dict(context=torch.stack(outs), cache=None, positions=None)
        return dict(context=outs, cache=None)
    # ft: q and the new keys are rotated and held in the data type, as the layout's kernel defines it
    lens, dtype = _lens(case), _DTYPES[case["dtype"]]
    outs = [[] for _ in range(_FT_STEPS)]
    for b, n in enumerate(lens):
        whole = torch.zeros((n + _FT_STEPS, *x["prompt"].shape[2:]), dtype=dtype, device=x["prompt"].device)
        whole[:n] = x["prompt"][b, :n]
        for t in range(_FT_STEPS):
            at = torch.tensor([n + t], device=whole.device)
            new = x["kv"][t, b, 0]
            whole[n + t, 0] = _turn(new[:1], at, 10000.0)[0].to(dtype)
            whole[n + t, 1] = new[1]
            q = _turn(x["q"][t, b], at, 10000.0).to(dtype)
            outs[t].append(_softmax_attend(q, whole[:n + t + 1, 0], whole[:n + t + 1, 1], scale, n + t + 1))
    return dict(context=[torch.stack(o) for o in outs], cache=None)
