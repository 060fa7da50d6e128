"""The calls whose speed is measured: what a GPT-2-124M inference program has this library do.

Sizes are the model's own (768 wide, 12 heads of 64, 3072 feed-forward, 2304 QKV, 50257 tokens, 1024
positions): every matmul the model has, with 1 to 1024 rows, fp16 and weight-only INT8; the attention
and LayerNorm between them; and the whole calls (prefill into the K/V cache, one decode step,
greedy generation through the decode graph).  Prompt lengths and positions are ragged as prompts are.
"""
import ctypes as C
import math

import torch

import __graft_entry__

E, QKV, FFN, VOCAB, CTX, LAYERS, HEADS, HD = 768, 2304, 3072, 50257, 1024, 12, 12, 64
# weight matrices [N, K] of the model by the name of their matmul
SHAPES = {"qkv": (QKV, E), "attn_proj": (E, E), "fc": (FFN, E), "mlp_proj": (E, FFN), "head": (VOCAB, E)}
TRUNK = LAYERS * (QKV * E + E * E + 2 * FFN * E)     # elements of the 48 layer matrices
TRUNK_ROWS = LAYERS * (QKV + E + FFN + E)            # their rows (INT8 scales, biases)


def listed():
    return [
        # One token through a layer's smallest matrix: launch latency, 0.6 MB of codes.
        {"name": "gemv_int8_attn_proj", "op": "gemv", "mat": "attn_proj", "dtype": "int8"},
        # The vocabulary projection of one token: 77 MB streamed.
        {"name": "gemv_fp16_head", "op": "gemv", "mat": "head", "dtype": "fp16"},
        # A short prompt's feed-forward matmul on quantized weights.
        {"name": "matmul_int8_fc_37", "op": "matmul", "mat": "fc", "dtype": "int8", "rows": 37},
        # The benchmark's prompt length.
        {"name": "matmul_fp16_qkv_512", "op": "matmul", "mat": "qkv", "dtype": "fp16", "rows": 512},
        # A nearly full context, ragged, through the long reduction.
        {"name": "matmul_fp16_mlp_proj_1000", "op": "matmul", "mat": "mlp_proj", "dtype": "fp16", "rows": 1000},
        # Logits of every position of a full context (scoring a text): the largest matmul, odd N.
        {"name": "matmul_fp16_head_1024", "op": "matmul", "mat": "head", "dtype": "fp16", "rows": 1024},
        # Causal attention over a prompt.
        {"name": "attention_777", "op": "attention", "rows": 777},
        # One token's attention over a nearly full cache.
        {"name": "attn_decode_1000", "op": "attn_decode", "len": 1000},
        # A prompt's LayerNorm.
        {"name": "layernorm_512", "op": "layernorm", "rows": 512},
        # A whole prompt into the cache, logits of its last position, quantized trunk.
        {"name": "prefill_int8_512", "op": "prefill", "dtype": "int8", "rows": 512, "all_rows": False},
        # One token through the whole model, the caller choosing the next one (sampling).
        {"name": "decode_step_fp16_512", "op": "decode_step", "dtype": "fp16", "pos": 512},
        # Greedy generation: 32 tokens after a prompt, quantized trunk.
        {"name": "generate_int8_480_32", "op": "generate", "dtype": "int8", "pos": 480, "steps": 32},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    op = rng.choice(["gemv", "matmul", "matmul", "head", "attention", "attn_decode", "layernorm", "prefill",
                     "prefill", "decode_step", "generate"])
    dtype = rng.choice(["fp16", "int8"])
    trunk = ["qkv", "attn_proj", "fc", "mlp_proj"]
    if op == "gemv":
        return {"op": "gemv", "mat": rng.choice(trunk + ["head"]), "dtype": dtype}
    if op == "matmul":
        return {"op": "matmul", "mat": rng.choice(trunk), "dtype": dtype, "rows": _log_int(rng, 2, CTX)}
    if op == "head":
        return {"op": "matmul", "mat": "head", "dtype": dtype, "rows": _log_int(rng, 2, CTX)}
    if op in ("attention", "layernorm"):
        return {"op": op, "rows": _log_int(rng, 1, CTX)}
    if op == "attn_decode":
        return {"op": op, "len": _log_int(rng, 1, CTX)}
    if op == "prefill":
        return {"op": op, "dtype": dtype, "rows": _log_int(rng, 2, CTX), "all_rows": rng.random() < 0.25}
    if op == "decode_step":
        return {"op": op, "dtype": dtype, "pos": _log_int(rng, 1, CTX - 1)}
    steps = _log_int(rng, 1, 32)
    return {"op": "generate", "dtype": dtype, "pos": _log_int(rng, 1, CTX - 1 - steps), "steps": steps}


# ----------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(shape, std, g):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std


def _quantize(w):
    """Symmetric per-row INT8 of fp16 weights: s = absmax / 127 (1 for a zero row), q = round(w / s)."""
    w = w.float()
    peak = w.abs().amax(dim=1, keepdim=True)
    s = torch.where(peak == 0, torch.ones_like(peak), peak / 127.0)
    return torch.clamp(torch.round(w / s), -127, 127).to(torch.int8), s.squeeze(1).contiguous()


def _matmul_inputs(case, seed):
    """x [rows, K]: LayerNorm outputs, or gelu outputs ahead of mlp_proj; weights N(0, 0.02); a bias, except
    on the head."""
    g = _gen(seed)
    n, k = SHAPES[case["mat"]]
    x = _normal((case.get("rows", 1), k), 1.0, g)
    if k == FFN:
        x = torch.nn.functional.gelu(x)
    w = _normal((n, k), 0.02, g).half()
    bias = None if case["mat"] == "head" else _normal((n,), 0.01, g).half()
    q, s = _quantize(w) if case["dtype"] == "int8" else (None, None)
    return x.half(), w, q, s, bias


def _qkv_rows(rows, seed):
    """Rows of q | k | v: scores q.k / 8 of a spread of about 1.5, values of 0.6."""
    x = _normal((rows, 3, E), 1.0, _gen(seed))
    x[:, :2] *= 1.2
    x[:, 2] *= 0.6
    return x.reshape(rows, QKV).half()


def _body(seed):
    """The model's weights in file order, fp16-valued: embeddings as wide as trained ones (0.14), so that
    greedy choices have the margins that a trained model's have; the layers as GPT-2 initialises them
    (0.02, residual projections / sqrt(24)); gains about 1, small biases."""
    layout = [("wte", (VOCAB, E)), ("wpe", (CTX, E))]
    for i in range(LAYERS):
        layout += [("h%d.%s" % (i, name), shape) for name, shape in (
            ("ln1_g", (E,)), ("ln1_b", (E,)), ("qkv_w", SHAPES["qkv"]), ("qkv_b", (QKV,)),
            ("attn_proj_w", SHAPES["attn_proj"]), ("attn_proj_b", (E,)), ("ln2_g", (E,)), ("ln2_b", (E,)),
            ("fc_w", SHAPES["fc"]), ("fc_b", (FFN,)), ("proj_w", SHAPES["mlp_proj"]), ("proj_b", (E,)))]
    layout += [("lnf_g", (E,)), ("lnf_b", (E,))]
    g = _gen(seed)
    body = torch.empty(sum(math.prod(shape) for _, shape in layout), device="cuda")
    views, at = {}, 0
    for name, shape in layout:
        n = math.prod(shape)
        v = body[at:at + n].view(shape)
        std = {"g": 0.1, "b": 0.01}.get(name[-1], 0.14 if name == "wte" else 0.02)
        v.normal_(0.0, std / math.sqrt(2 * LAYERS) if name.endswith("proj_w") else std, generator=g)
        if name.endswith("_g"):
            v += 1.0
        views[name] = v
        at += n
    body.copy_(body.half().float())
    return body, views


def _ids(count, seed):
    return torch.randint(0, VOCAB, (count,), generator=_gen(seed + 7), device="cuda", dtype=torch.int32)


class _Arena:
    """A session's K/V cache as torch reads a foreign array; the tensor holds this, and this the session."""

    def __init__(self, session):
        self.session = session
        self.__cuda_array_interface__ = {"shape": (LAYERS, 2, HEADS, CTX, HD), "typestr": "<f2", "strides": None,
                                         "data": (session.kv.kv.data, False), "version": 2}


class _Session:
    """A program's model: fp16 weights on the GPU (INT8 trunk attached for "int8"), scratch, K/V cache."""

    def __init__(self, pkg, case, seed):
        self.pkg, self.lib = pkg, pkg.lib()
        body, _ = _body(seed)
        self.model = pkg.Model(body.cpu().numpy())
        self.model.body = None   # uploaded
        if case["dtype"] == "int8":
            self.model.quantize()
        self.backend = pkg.backend("int8" if case["dtype"] == "int8" else "gemv")
        self.scratch = pkg.Scratch(CTX)
        self.kv = pkg.KVCache(CTX)
        self.graph = None

    def cache(self, rows):
        """The first `rows` positions of the cache as a tensor [layer, K|V, head, rows, 64], which keeps the
        session, and with it the cache, while it is held."""
        return torch.as_tensor(_Arena(self), device="cuda")[:, :, :, :rows]

    def prefill(self, ids, caps=None):
        self.lib.gpt2_prefill_fill_cache(self.backend, C.byref(self.model.gpu), C.byref(self.kv.kv), ids.data_ptr(),
                                         ids.numel(), C.byref(self.scratch.s), C.byref(caps) if caps else None)

    def __del__(self):
        torch.cuda.synchronize()
        if self.graph:
            self.lib.gpt2_decode_graph_destroy(self.graph)
        for part in (self.kv, self.scratch, self.model):
            part.free()


def prepare(case, seed):
    pkg = __graft_entry__.load_package()
    lib, op = pkg.lib(), case["op"]
    p = lambda t: C.c_void_p(t.data_ptr() if t is not None else None)  # noqa: E731
    if op in ("gemv", "matmul"):
        x, w, q, s, bias = _matmul_inputs(case, seed)
        (n, k), m = SHAPES[case["mat"]], x.shape[0]
        out = torch.empty((m, n), dtype=torch.float16, device="cuda")
        weights = (p(w),) if q is None else (p(q), p(s))
        rows = () if op == "gemv" else (m,)
        name = {("gemv", "fp16"): "gpt2_gemv_fp16", ("gemv", "int8"): "gpt2_gemv_int8",
                ("matmul", "fp16"): "gpt2_matmul_tiled", ("matmul", "int8"): "gpt2_matmul_int8"}[op, case["dtype"]]
        return {"op": op, "call": getattr(lib, name), "args": (p(out), p(x)) + weights + (p(bias),) + rows + (n, k),
                "out": out, "hold": (x, w if q is None else q, s, bias)}
    if op == "attention":
        qkv = _qkv_rows(case["rows"], seed)
        out = torch.empty((case["rows"], E), dtype=torch.float16, device="cuda")
        return {"op": op, "call": lib.gpt2_attention_flash, "args": (p(out), p(qkv), case["rows"], E, HEADS, HD),
                "out": out, "hold": qkv}
    if op == "layernorm":
        x, gain, shift = _layernorm_inputs(case, seed)
        out = torch.empty_like(x)
        return {"op": op, "call": lib.gpt2_layernorm, "args": (p(out), p(x), p(gain), p(shift), x.shape[0], E),
                "out": out, "hold": (x, gain, shift)}
    if op == "attn_decode":
        qkv = _qkv_rows(CTX, seed)
        kv = pkg.KVCache(CTX)
        for layer in range(LAYERS):   # every layer holds the same rows: the call reads one layer's
            lib.gpt2_kv_scatter_prefill(C.byref(kv.kv), layer, p(qkv), CTX)
        out = torch.empty((E,), dtype=torch.float16, device="cuda")
        torch.cuda.synchronize()
        return {"op": op, "call": lib.gpt2_attn_decode, "out": out, "hold": (qkv, _Owner(kv)),
                "args": (p(out), p(qkv[case["len"] - 1]), C.byref(kv.kv), LAYERS // 2, case["len"])}
    s = _Session(pkg, case, seed)
    if op == "prefill":
        ids = _ids(case["rows"], seed)
        logits = torch.empty((case["rows"] if case["all_rows"] else 1, VOCAB), dtype=torch.float16, device="cuda")
        caps = pkg.GPT2CapsGPU()
        caps.logits, caps.logits_all = logits.data_ptr(), int(case["all_rows"])
        return {"op": op, "session": s, "ids": ids, "caps": caps, "logits": logits, "cache": s.cache(case["rows"])}
    ids = _ids(case["pos"] + 1, seed)
    s.prefill(ids[:-1])
    logits = torch.empty((VOCAB,), dtype=torch.float16, device="cuda")
    state = {"op": op, "session": s, "logits": logits, "token": int(ids[-1]), "pos": case["pos"]}
    if op == "decode_step":
        state["cache"] = s.cache(case["pos"] + 1)
    else:
        state["steps"] = case["steps"]
        state["tokens"] = torch.zeros((CTX,), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        s.graph = lib.gpt2_decode_graph_create(s.backend, C.byref(s.model.gpu), C.byref(s.kv.kv), C.byref(s.scratch.s),
                                               logits.data_ptr(), state["tokens"].data_ptr())
    pkg.check("prepare")
    return state


class _Owner:
    """Frees a library object with its last reference, after the GPU is done with it."""

    def __init__(self, part):
        self.part = part

    def __del__(self):
        torch.cuda.synchronize()
        self.part.free()


def _layernorm_inputs(case, seed):
    g = _gen(seed)
    x = _normal((case["rows"], E), 0.5, g) + _normal((case["rows"], 1), 0.05, g)
    return x.half(), (1.0 + _normal((E,), 0.1, g)).half(), _normal((E,), 0.01, g).half()


def run(state):
    op = state["op"]
    if "call" in state:
        state["call"](*state["args"])
        return state["out"]
    s = state["session"]
    if op == "prefill":
        s.prefill(state["ids"], state["caps"])
        return {"logits": state["logits"], "cache": state["cache"]}
    if op == "decode_step":
        s.lib.gpt2_decode_step_cuda(s.backend, C.byref(s.model.gpu), C.byref(s.kv.kv), state["token"], state["pos"],
                                    C.byref(s.scratch.s), state["logits"].data_ptr(), None)
        return {"logits": state["logits"], "cache": state["cache"]}
    # the tokens are on the host side's request: set, run, wait, as a generation loop does
    s.lib.gpt2_decode_graph_set(s.graph, state["token"], state["pos"])
    s.lib.gpt2_decode_graph_run(s.graph, state["steps"])
    if s.lib.gpt2_decode_graph_sync(s.graph, None, None):
        s.pkg.check("generate")
    return {"logits": state["logits"], "tokens": state["tokens"]}


# ----------------------------------------------------------------------------- what a pass cannot do without
def _weight_bytes(dtype):
    return (TRUNK + 4 * TRUNK_ROWS if dtype == "int8" else 2 * TRUNK) + 2 * TRUNK_ROWS + 2 * VOCAB * E


def work(case):
    op = case["op"]
    if op in ("gemv", "matmul"):
        (n, k), m = SHAPES[case["mat"]], case.get("rows", 1)
        w = n * k + 4 * n if case["dtype"] == "int8" else 2 * n * k
        return {"bytes": w + 2 * m * (n + k) + (0 if case["mat"] == "head" else 2 * n), "flops": 2 * m * n * k}
    if op == "attention":
        t = case["rows"]
        return {"bytes": 2 * t * (QKV + E), "flops": 2 * E * t * (t + 1)}
    if op == "attn_decode":
        return {"bytes": 4 * E * case["len"] + 4 * E, "flops": 4 * E * case["len"]}
    if op == "layernorm":
        return {"bytes": 4 * E * case["rows"] + 4 * E, "flops": 8 * E * case["rows"]}
    if op == "prefill":
        t = case["rows"]
        out = t if case["all_rows"] else 1
        return {"bytes": _weight_bytes(case["dtype"]) + 4 * E * t + 4 * E * LAYERS * t + 2 * VOCAB * out,
                "flops": 2 * t * TRUNK + LAYERS * 2 * E * t * (t + 1) + 2 * out * VOCAB * E}
    steps = case.get("steps", 1)
    keys = sum(case["pos"] + 1 + i for i in range(steps))
    return {"bytes": steps * (_weight_bytes(case["dtype"]) + 2 * VOCAB) + 4 * E * LAYERS * keys,
            "flops": 2 * steps * (TRUNK + VOCAB * E) + 4 * E * LAYERS * keys}


def tolerance(case):
    # Outputs are fp16 of fp32 sums: rounding puts a result 2.1e-4 off the one in 64 bits and a value up to
    # 4.9e-4.  Attention multiplies fp16 probabilities (2.3e-4; 1.9e-3); whole calls carry the roundings of
    # twelve layers (1.3e-3; 7.5e-3).  Each bound is about four times what was measured.  The choices of
    # greedy generation have wide margins here, so its tokens are the same.
    op = case["op"]
    if op in ("gemv", "matmul", "layernorm"):
        return {"rel": 8e-4, "max": 2e-3}
    if op in ("attention", "attn_decode"):
        return {"rel": 1e-3, "max": 8e-3}
    return {"rel": 5e-3, "max": 3e-2, "differ": 0.0}


# ----------------------------------------------------------------------------- the same in 64 bits
def exact(case, seed):
    op = case["op"]
    if op in ("gemv", "matmul"):
        x, w, q, s, bias = _matmul_inputs(case, seed)
        w = w.double() if q is None else q.double() * s.double()[:, None]
        y = x.double() @ w.t()
        return y if bias is None else y + bias.double()
    if op == "layernorm":
        x, gain, shift = (t.double() for t in _layernorm_inputs(case, seed))
        return _ln(x, gain, shift)
    if op == "attention":
        return _attend(_qkv_rows(case["rows"], seed).double())[0]
    if op == "attn_decode":
        return _attend(_qkv_rows(CTX, seed)[:case["len"]].double())[0][-1]
    views = {name: v.double() for name, v in _body(seed)[1].items()}
    if case["dtype"] == "int8":
        for name, v in views.items():
            if name.endswith("_w"):
                q, s = _quantize(v.half())
                views[name] = q.double() * s.double()[:, None]
    if op == "prefill":
        hidden, cache = _forward(views, _ids(case["rows"], seed), None)
        return {"logits": (hidden if case["all_rows"] else hidden[-1:]) @ views["wte"].t(), "cache": cache}
    ids = _ids(case["pos"] + 1, seed)
    _, cache = _forward(views, ids[:-1], None)
    token = ids[-1:]
    for _ in range(case.get("steps", 1)):
        hidden, cache = _forward(views, token, cache)
        logits = hidden[-1] @ views["wte"].t()
        token = logits.argmax().reshape(1)
    return {"logits": logits, "cache": cache} if op == "decode_step" else {"logits": logits, "tokens": None}


def _ln(x, gain, shift):
    d = x - x.mean(dim=-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(dim=-1, keepdim=True) + 1e-5) * gain + shift


def _attend(qkv, past=None):
    """Causal attention of the last rows of a context: [rows, 768], and the context's keys and values."""
    q, k, v = (t.reshape(-1, HEADS, HD).transpose(0, 1) for t in qkv.split(E, dim=1))
    if past is not None:
        k, v = torch.cat((past[0], k), dim=1), torch.cat((past[1], v), dim=1)
    scores = torch.matmul(q, k.transpose(1, 2).contiguous()) / 8.0
    at = torch.arange(k.shape[1] - q.shape[1], k.shape[1], device=q.device)
    scores.masked_fill_(torch.arange(k.shape[1], device=q.device)[None, :] > at[:, None], -math.inf)
    return torch.matmul(torch.softmax(scores, dim=-1), v.contiguous()).transpose(0, 1).reshape(-1, E), (k, v)


def _forward(views, ids, cache):
    """Final hidden rows of `ids` after a cached context [layer, K|V, head, rows, 64], and the longer cache."""
    start = 0 if cache is None else cache.shape[3]
    x = views["wte"][ids.long()] + views["wpe"][start:start + ids.numel()]
    kept = []
    for i in range(LAYERS):
        w = lambda name: views["h%d.%s" % (i, name)]  # noqa: E731, B023
        qkv = _ln(x, w("ln1_g"), w("ln1_b")) @ w("qkv_w").t() + w("qkv_b")
        y, kv = _attend(qkv, None if cache is None else cache[i])
        kept.append(torch.stack(kv))
        x = x + y @ w("attn_proj_w").t() + w("attn_proj_b")
        h = _ln(x, w("ln2_g"), w("ln2_b")) @ w("fc_w").t() + w("fc_b")
        h = 0.5 * h * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (h + 0.044715 * h ** 3)))
        x = x + h @ w("proj_w").t() + w("proj_b")
    return _ln(x, views["lnf_g"], views["lnf_b"]), torch.stack(kept)
