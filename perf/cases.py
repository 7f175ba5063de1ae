"""The work that users of this package have it do, as measurable cases: what a program calls, on which sizes, and how
far another correct implementation may be off.

Every case is one of six ways into the package:

  attention  an eager flash attention call on device arrays: execute_op_inplace(out, FlashAttentionOp, q, k, v[, kv_len])
  decode     an eager single-token attention call over a KV cache: execute_op_inplace(out, DecodeAttentionOp, ...)
  step       one decode step of a cached layer through a compiled graph: rotary embedding, cache append, attention
  prompt     the prompt pass of a cached layer through a compiled graph: cache append with rotated keys, causal attention
  layer      a whole attention layer (projections, heads, attention, output projection) through a compiled graph
  execute    the interpreter on host arrays: upload, attention, download

listed() fixes twelve of them over the sizes of the benchmark configurations and around them; draw() gives more of the
same ranges. A case is a dict of plain values; `seed` alone decides the inputs.
"""
import math

import numpy as np
import torch

import __graft_entry__  # the repository's root is the working folder and on the path

lm = __graft_entry__.load_package()

ELEM = {"f32": 4, "f16": 2, "bf16": 2}


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------
def _attention(dtype, B, Hq, Hkv, Sq, Sk, D, causal, ragged=False, out_f32=False, blocked=False, rope=False):
    return {"kind": "attention", "dtype": dtype, "B": B, "Hq": Hq, "Hkv": Hkv, "Sq": Sq, "Sk": Sk, "D": D, "causal": causal,
            "ragged": ragged, "out_f32": out_f32, "blocked": blocked, "rope": rope}


def _decode(dtype, B, Hq, Hkv, L, D, ragged=False, out_f32=False, blocked=False):
    return {"kind": "decode", "dtype": dtype, "B": B, "Hq": Hq, "Hkv": Hkv, "L": L, "D": D, "ragged": ragged,
            "out_f32": out_f32, "blocked": blocked}


def _step(dtype, B, Hq, Hkv, L, D, rope=True, ragged=False):
    return {"kind": "step", "dtype": dtype, "B": B, "Hq": Hq, "Hkv": Hkv, "L": L, "D": D, "rope": rope, "ragged": ragged}


def _prompt(dtype, B, Hq, Hkv, T, L, D, rope=True):
    return {"kind": "prompt", "dtype": dtype, "B": B, "Hq": Hq, "Hkv": Hkv, "T": T, "L": L, "D": D, "rope": rope}


def _layer(which, dtype, B, S, Senc, H, Hkv, D):
    return {"kind": "layer", "which": which, "dtype": dtype, "B": B, "S": S, "Senc": Senc, "H": H, "Hkv": Hkv, "D": D}


def _execute(dtype, B, Hq, Hkv, Sq, Sk, D, causal):
    return {"kind": "execute", "dtype": dtype, "B": B, "Hq": Hq, "Hkv": Hkv, "Sq": Sq, "Sk": Sk, "D": D, "causal": causal}


def listed():
    named = {
        # The reference's own example shape in its own element type: a short prompt of a small model. Latency.
        "attention f32 short": _attention("f32", 1, 8, 8, 128, 128, 64, True),
        # The headline prefill: one long prompt, multi-head attention, head dim 96.
        "attention f16 long": _attention("f16", 1, 32, 32, 4096, 4096, 96, True),
        # A batch of prompts of different lengths padded to one odd length, grouped heads, bf16.
        "attention bf16 ragged": _attention("bf16", 3, 32, 8, 1337, 1337, 128, True, ragged=True),
        # Speech decoder queries over encoder keys: no mask, 448 x 1500.
        "attention f16 cross": _attention("f16", 4, 20, 20, 448, 1500, 64, False),
        # Wide heads (256), which the package takes for prefill as it does for decode.
        "attention bf16 wide heads": _attention("bf16", 1, 16, 8, 1500, 1500, 256, True),
        # The reference's element type at a prompt's size, head dim 80, an odd number of rows, no mask.
        "attention f32 odd": _attention("f32", 2, 12, 12, 1023, 1023, 80, False),
        # Serving, long contexts of different lengths: 64 sequences up to 32k tokens.
        "decode bf16 long ragged": _decode("bf16", 64, 32, 8, 32768, 128, ragged=True, out_f32=True),
        # A decode step of a batch of 16 at 4096 tokens, and of a single short conversation (an interactive user).
        "step bf16 batch": _step("bf16", 16, 32, 8, 4096, 128),
        "step bf16 single": _step("bf16", 1, 32, 8, 512, 128),
        # Four prompts written into their caches and attended.
        "prompt f16 cached": _prompt("f16", 4, 32, 8, 777, 2048, 128),
        # A whole self attention layer on a prompt, projections in fp32, attention in bf16.
        "layer bf16": _layer("self", "bf16", 1, 700, 0, 32, 4, 64),
        # The interpreter: host arrays in, host array out, in the reference's element type.
        "execute f32": _execute("f32", 2, 8, 8, 512, 512, 64, True),
    }
    return [dict(case, name=name) for name, case in named.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# Head dims of models in use; the package takes any up to 256, the usual ones come up most.
HEAD_DIMS = [64] * 4 + [128] * 4 + [96] * 2 + [80] * 2 + [256] * 2 + [32, 40, 72, 112, 160, 192]
CACHED_HEAD_DIMS = [64] * 3 + [128] * 4 + [96, 80, 256]
DTYPES = ["f16", "bf16", "f16", "bf16", "f32"]


def _heads(rng):
    Hkv = rng.choice([1, 2, 4, 6, 8, 12, 16, 20, 32])
    return Hkv * rng.choice([g for g in (1, 1, 2, 4, 8) if Hkv * g <= 64]), Hkv


def _draw(rng):
    kind = rng.choice(["attention"] * 8 + ["decode"] * 4 + ["step"] * 2 + ["prompt"] * 2 + ["layer"] * 2 + ["execute"] * 2)
    dtype = rng.choice(DTYPES)
    Hq, Hkv = _heads(rng)
    half = dtype != "f32"
    if kind == "attention":
        D = rng.choice(HEAD_DIMS)
        mode = rng.choice(["causal", "causal", "full", "cross"])
        Sq = _log_int(rng, 16, 8192)
        Sk = _log_int(rng, 16, 8192) if mode == "cross" else Sq
        return _attention(dtype, _log_int(rng, 1, 16), Hq, Hkv, Sq, Sk, D, mode == "causal", ragged=rng.random() < 0.3,
                          out_f32=half and rng.random() < 0.3, blocked=rng.random() < 0.3,
                          rope=mode == "causal" and D in lm.FUSED_ROPE_HEAD_DIMS and rng.random() < 0.3)
    if kind == "decode":
        return _decode(dtype, _log_int(rng, 1, 128), Hq, Hkv, _log_int(rng, 64, 32768), rng.choice(CACHED_HEAD_DIMS),
                       ragged=rng.random() < 0.5, out_f32=half and rng.random() < 0.5, blocked=rng.random() < 0.3)
    if kind == "step":
        return _step(dtype, _log_int(rng, 1, 32), Hq, Hkv, _log_int(rng, 64, 8192), rng.choice(CACHED_HEAD_DIMS),
                     rope=rng.random() < 0.7, ragged=rng.random() < 0.5)
    if kind == "prompt":
        T = _log_int(rng, 16, 4096)
        return _prompt(dtype, _log_int(rng, 1, 8), Hq, Hkv, T, T + _log_int(rng, 16, 2048), rng.choice(CACHED_HEAD_DIMS),
                       rope=rng.random() < 0.7)
    if kind == "layer":
        which = rng.choice(["self", "self", "speech", "speech cross"])
        D, H = rng.choice([64, 64, 96, 128]), rng.choice([4, 6, 8, 12, 16, 20, 32])
        Hkv = H if which != "self" else H // rng.choice([g for g in (1, 2, 4, 8) if H % g == 0])
        return _layer(which, rng.choice(["f32", "f16", "bf16"]), _log_int(rng, 1, 4), _log_int(rng, 16, 1024),
                      _log_int(rng, 64, 1500) if which == "speech cross" else 0, H, Hkv, D)
    Sq = _log_int(rng, 16, 2048)
    causal = rng.random() < 0.5
    return _execute(dtype, _log_int(rng, 1, 4), Hq, Hkv, Sq, Sq if causal else _log_int(rng, 16, 2048), rng.choice([64, 80, 96, 128]), causal)


def draw(rng):
    """One more case of the same ranges."""
    top = {kind: {what: max(work(c)[what] for c in listed() if c["kind"] == kind) for what in ("bytes", "flops")} for kind in PREPARE}
    while True:  # a case of its kind's range that costs no more than a large listed one
        case = _draw(rng)
        kind, w = case["kind"], work(case)
        if kind in ("decode", "step"):  # bound by what they read
            fits = w["bytes"] <= top[kind]["bytes"]
        elif kind == "layer":
            fits = w["flops"] <= top[kind]["flops"]
        elif kind == "execute":  # host memory to the device and back
            fits = w["bytes"] <= 4 * top[kind]["bytes"] and w["flops"] <= 1e10
        else:  # attention, prompt: the matrix rate of fp32 is a part of that of the 16-bit types
            slow = (4 if case["dtype"] == "f32" else 1) * (4 if case["D"] > 128 else 1)
            fits = w["flops"] * slow <= top["attention"]["flops"] and w["bytes"] <= 1e9
        if fits:
            return case


# ---------------------------------------------------------------------------------------------
# inputs and outputs on the device
# ---------------------------------------------------------------------------------------------
TORCH_TYPES = {"f32": ("<f4", torch.float32), "f16": ("<f2", torch.float16), "bf16": ("<i2", torch.bfloat16),
               "i32": ("<i4", torch.int32)}


class _Memory:
    def __init__(self, array):
        self.array = array  # keeps the buffer alive
        self.__cuda_array_interface__ = {"shape": array.shape, "typestr": TORCH_TYPES[array.dtype][0],
                                         "data": (array.ptr, False), "version": 2}


def tensor_of(array):
    """The HipArray's own memory as a torch tensor."""
    t = torch.as_tensor(_Memory(array), device="cuda")
    return t.view(torch.bfloat16) if array.dtype == "bf16" else t


class _Inputs:
    """Normal values from one seeded generator, in the order they are asked for."""

    def __init__(self, seed):
        self.generator = torch.Generator(device="cuda").manual_seed(seed)
        self.host = torch.Generator().manual_seed(seed)

    def fill(self, array, mul=1.0):
        t = tensor_of(array)
        t.normal_(0.0, mul, generator=self.generator)
        return array

    def array(self, shape, dtype, mul=1.0):
        return self.fill(lm.HipArray(shape, dtype), mul)

    def lengths(self, n, lo, hi):
        x = torch.randint(lo, hi + 1, (n,), generator=self.host, dtype=torch.int32).numpy()
        return lm.to_device(x, lm.HIPDevice(0))

    def numpy(self, shape):
        return torch.randn(shape, generator=self.host).numpy()


# ---------------------------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------------------------
def prepare(case, seed):
    lm.get_device()
    return PREPARE[case["kind"]](case, _Inputs(seed))


def run(state):
    return state["run"](state)


def _eager(state):
    lm.execute_op_inplace(state["out"], state["op"], *state["args"])
    return state["outputs"]


def _compiled(state):
    state["graph"](state["feeds"])
    return state["outputs"]


def _prepare_attention(c, inputs):
    q = inputs.array((c["B"], c["Hq"], c["Sq"], c["D"]), c["dtype"])
    k = inputs.array((c["B"], c["Hkv"], c["Sk"], c["D"]), c["dtype"])
    v = inputs.array((c["B"], c["Hkv"], c["Sk"], c["D"]), c["dtype"])
    args = [q, k, v]
    if c["ragged"]:
        args.append(inputs.lengths(c["B"], (c["Sk"] + 1) // 2, c["Sk"]))
    op = lm.FlashAttentionOp(lm.default_scale(c["D"]), c["causal"], lm.HEADMAP_BLOCKED if c["blocked"] else lm.HEADMAP_INTERLEAVED,
                             has_kv_len=c["ragged"], q_rope_base=10000.0 if c["rope"] else None)
    out = lm.HipArray(q.shape, "f32" if c["out_f32"] else c["dtype"])
    return {"run": _eager, "out": out, "op": op, "args": args, "outputs": tensor_of(out)}


def _prepare_decode(c, inputs):
    q = inputs.array((c["B"], c["Hq"], c["D"]), c["dtype"])
    k = inputs.array((c["B"], c["Hkv"], c["L"], c["D"]), c["dtype"])
    v = inputs.array((c["B"], c["Hkv"], c["L"], c["D"]), c["dtype"])
    lens = inputs.lengths(c["B"], (c["L"] + 3) // 4 if c["ragged"] else c["L"], c["L"])
    op = lm.DecodeAttentionOp(lm.default_scale(c["D"]), lm.HEADMAP_BLOCKED if c["blocked"] else lm.HEADMAP_INTERLEAVED)
    out = lm.HipArray(q.shape, "f32" if c["out_f32"] else c["dtype"])
    return {"run": _eager, "out": out, "op": op, "args": [q, k, v, lens], "outputs": tensor_of(out)}


def _positions(c, inputs):
    """The row this step writes, per sequence: the last one of the cache, or anywhere in its upper three quarters."""
    return inputs.lengths(c["B"], (c["L"] + 3) // 4 if c["ragged"] else c["L"] - 1, c["L"] - 1)


def _prepare_step(c, inputs):
    # The caches live in the compiled graph; a step brings its projections and its positions. Running it again writes
    # the same rows again.
    g = lm.Graph()
    dt = c["dtype"]
    q = lm.tensor(g, (c["B"], c["Hq"], 1, c["D"]), dt)
    kn, vn = (lm.tensor(g, (c["B"], c["Hkv"], 1, c["D"]), dt) for _ in range(2))
    kc, vc = (lm.tensor(g, (c["B"], c["Hkv"], c["L"], c["D"]), dt) for _ in range(2))
    pos, kv_len = lm.tensor(g, (c["B"],), "i32"), lm.tensor(g, (c["B"],), "i32")
    out, k_after, v_after = lm.cached_self_attention_core(q, kn, vn, kc, vc, pos, kv_len, rope_base=10000.0 if c["rope"] else None,
                                                          fused=True)
    graph = lm.compile(g)
    for cache in (kc, vc):
        inputs.fill(graph.results[cache.id])
    p = _positions(c, inputs)
    lens = lm.to_device(p.to_host() + np.int32(1), lm.HIPDevice(0))
    feeds = {t.id: inputs.array(t.shape, dt) for t in (q, kn, vn)}
    feeds.update({pos.id: p, kv_len.id: lens})
    node = graph.results[out.id]
    return {"run": _compiled, "graph": graph, "feeds": feeds,
            "outputs": [tensor_of(node[0] if isinstance(node, tuple) else node), tensor_of(graph.results[kc.id]), tensor_of(graph.results[vc.id])]}


def _prepare_prompt(c, inputs):
    g = lm.Graph()
    dt = c["dtype"]
    q = lm.tensor(g, (c["B"], c["Hq"], c["T"], c["D"]), dt)
    kn, vn = (lm.tensor(g, (c["B"], c["Hkv"], c["T"], c["D"]), dt) for _ in range(2))
    kc, vc = (lm.tensor(g, (c["B"], c["Hkv"], c["L"], c["D"]), dt) for _ in range(2))
    pos, kv_len = lm.tensor(g, (c["B"],), "i32"), lm.tensor(g, (c["B"],), "i32")
    out, _, _ = lm.prompt_self_attention_core(q, kn, vn, kc, vc, pos, kv_len, rope_base=10000.0 if c["rope"] else None)
    graph = lm.compile(g)
    feeds = {t.id: inputs.array(t.shape, dt) for t in (q, kn, vn)}
    feeds[pos.id] = lm.to_device(np.zeros(c["B"], np.int32), lm.HIPDevice(0))
    feeds[kv_len.id] = lm.to_device(np.full(c["B"], c["T"], np.int32), lm.HIPDevice(0))
    return {"run": _compiled, "graph": graph, "feeds": feeds,
            "outputs": [tensor_of(graph.results[t.id]) for t in (out, kc, vc)]}


def _prepare_layer(c, inputs):
    # The weights are laid into the compiled graph once; a pass brings the hidden states.
    g = lm.Graph()
    hidden = c["H"] * c["D"]
    x = lm.tensor(g, (c["B"], c["S"], hidden))
    fed = [x]
    if c["which"] == "self":
        layer = lm.SelfAttention(hidden, c["H"], c["Hkv"], g, attn_dtype=c["dtype"])
        out = layer(x)
    else:
        layer = lm.WhisperAttention(hidden, c["H"], g, attn_dtype=c["dtype"])
        enc = lm.tensor(g, (c["B"], c["Senc"], hidden)) if c["which"] == "speech cross" else None
        fed += [enc] if enc is not None else []
        out = layer(x, mask=enc is None, keys_from=enc, values_from=enc)
    graph = lm.compile(g)
    for proj in (layer.q_proj, layer.k_proj, layer.v_proj, layer.o_proj):
        inputs.fill(graph.results[proj.weight.id], 1.0 / math.sqrt(hidden))
        if proj.bias is not None:
            inputs.fill(graph.results[proj.bias.id], 0.1)
    feeds = {t.id: inputs.array(t.shape, "f32") for t in fed}
    return {"run": _compiled, "graph": graph, "feeds": feeds, "outputs": tensor_of(graph.results[out.id])}


def _prepare_execute(c, inputs):
    g = lm.Graph()
    shapes = [(c["B"], c["Hq"], c["Sq"], c["D"]), (c["B"], c["Hkv"], c["Sk"], c["D"]), (c["B"], c["Hkv"], c["Sk"], c["D"])]
    q, k, v = (lm.tensor(g, s, c["dtype"]) for s in shapes)
    out = lm.flash_attention(q, k, v, causal=c["causal"])
    return {"run": _interpret, "graph": g, "out": out.id, "device": lm.HIPDevice(0),
            "values": {t.id: inputs.numpy(s) for t, s in zip((q, k, v), shapes)}}


def _interpret(state):
    return lm.execute(state["graph"], state["out"], state["values"], state["device"])


PREPARE = {"attention": _prepare_attention, "decode": _prepare_decode, "step": _prepare_step, "prompt": _prepare_prompt,
           "layer": _prepare_layer, "execute": _prepare_execute}


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------------------------
def _attention_flops(B, Hq, Sq, Sk, D, causal):
    pairs = Sq * Sk
    if causal:  # row i sees keys 0 .. i
        pairs = sum(min(i + 1, Sk) for i in range(Sq))
    return 4.0 * B * Hq * D * pairs


def _mean_length(c, top):
    return (((top + 3) // 4) + top) / 2 if c["ragged"] else top


def work(case):
    """Each input read once, each output written once; 2 flops a multiply-add, unmasked pairs only. Where the lengths
    are drawn from the seed, their expected value."""
    c, kind = case, case["kind"]
    if kind in ("attention", "execute"):
        keys = c["Sk"] if not c.get("ragged") else (c["Sk"] + (c["Sk"] + 1) // 2) / 2
        e = ELEM[c["dtype"]] if kind == "attention" else 4
        out = 4 if c.get("out_f32") or kind == "execute" else e
        b = c["B"] * c["D"] * (c["Hq"] * c["Sq"] * (e + out) + 2 * c["Hkv"] * keys * e)
        return {"bytes": b, "flops": _attention_flops(c["B"], c["Hq"], c["Sq"], int(keys), c["D"], c["causal"])}
    e = ELEM[c["dtype"]]
    if kind == "decode":
        L = _mean_length(c, c["L"])
        b = c["B"] * c["D"] * (2 * c["Hkv"] * L * e + c["Hq"] * (e + (4 if c["out_f32"] else e)))
        return {"bytes": b, "flops": 4.0 * c["B"] * c["Hq"] * c["D"] * L}
    if kind == "step":
        L = _mean_length(c, c["L"])
        b = c["B"] * c["D"] * e * (2 * c["Hkv"] * (L + 1) + 2 * c["Hq"])
        return {"bytes": b, "flops": 4.0 * c["B"] * c["Hq"] * c["D"] * L}
    if kind == "prompt":  # the new rows are read and written into the caches; attention can take them on the way
        b = c["B"] * c["D"] * e * c["T"] * (4 * c["Hkv"] + 2 * c["Hq"])
        return {"bytes": b, "flops": _attention_flops(c["B"], c["Hq"], c["T"], c["T"], c["D"], True)}
    hidden, rows, keys = c["H"] * c["D"], c["B"] * c["S"], c["B"] * (c["Senc"] or c["S"])
    weights = hidden * hidden * 2 + hidden * c["Hkv"] * c["D"] * 2
    flops = 2.0 * (rows * hidden * hidden * 2 + keys * hidden * c["Hkv"] * c["D"] * 2)
    flops += _attention_flops(c["B"], c["H"], c["S"], c["Senc"] or c["S"], c["D"], c["which"] != "speech cross")
    return {"bytes": 4 * (weights + rows * hidden * 2 + (keys * hidden if c["Senc"] else 0)), "flops": flops}


def tolerance(case):
    """fp32: sums in another order. 16-bit types: the softmax weights and the stored result carry 11 or 8 bits (fp32
    results of bf16 inputs: 11-bit weights); in a layer the projected q, k and v are rounded to the type as well."""
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    if case["dtype"] == "f16" or case.get("out_f32"):
        return {"rel": 1.5e-3}
    return {"rel": 8e-3}
