"""Workloads that the framework's speed is measured on, through its public entry points.

A case is a dict of plain values: `kind` names the call, the other keys its sizes, types and options.

  gemv    one eager matrix-vector product: a projection of a single-token step called by itself
  token   a whole single-token step replayed as one graph: per layer {QKV, fc1}, the decode attention step
          over the layer's KV cache, {dense, fc2} with bias / GELU / residual, then the LM head and the token pick
  batch   the projections of a step that decodes M sequences at once over quantized weights, as one graph
          (attention over M separate caches is not an op of this framework: its outputs come in as inputs)
  block   the forward pass of one transformer block over a whole sequence in fp16: text prefill (causal) or
          a vision tower layer; rotary embedding and norms belong to the caller, so Q, K and V are inputs
  gemm    one eager product with a packed 16-bit weight
  scores  the batched Q K^T of all heads of a layer, fp32 scores
  exact   the products that keep the reference kernels' summation order bit for bit

Inputs are made on the GPU from the seed with torch and put in place through the buffers' device addresses;
weights are packed once from GGUF blocks or row-major arrays, as a program does when it loads a model.
"""
import ctypes
import math

import torch

import mvlm_amd as m

TORCH = {m.F32: torch.float32, m.F16: torch.float16, m.BF16: torch.bfloat16}
DTYPE = {"f32": m.F32, "f16": m.F16, "bf16": m.BF16, "q8_0": m.Q8_0, "q4_0": m.Q4_0}
SIZE = {"f32": 4.0, "f16": 2.0, "bf16": 2.0, "q8_0": 34 / 32, "q4_0": 18 / 32}   # bytes per weight
HEAD_DIM = 64

_device = None


def device():
    global _device
    if _device is None:
        torch.cuda.init()
        _device = m.Device(0)
    return _device


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # the smallest call: Phi-1.5's dense projection for one token, where the launch is what counts
        {"name": "gemv_q8_0_2048x2048", "kind": "gemv", "dtype": "q8_0", "n": 2048, "k": 2048, "gelu": False},
        # an unquantized fc1 for one token
        {"name": "gemv_f32_8192x2048", "kind": "gemv", "dtype": "f32", "n": 8192, "k": 2048, "gelu": False},
        # Phi-1.5 generating a token, 512 positions into a conversation
        {"name": "token_q8_0_cache512", "kind": "token", "dtype": "q8_0", "layers": 24, "heads": 32, "inner": 8192,
         "vocab": 51200, "cache": 512},
        # the same model in 4 bits at the end of its 2048-position context
        {"name": "token_q4_0_cache2047", "kind": "token", "dtype": "q4_0", "layers": 24, "heads": 32, "inner": 8192,
         "vocab": 51200, "cache": 2047},
        # four conversations decoded together
        {"name": "batch4_q8_0", "kind": "batch", "dtype": "q8_0", "m": 4, "layers": 24, "heads": 32, "inner": 8192,
         "vocab": 51200},
        # a full batch of sixteen
        {"name": "batch16_q4_0", "kind": "batch", "dtype": "q4_0", "m": 16, "layers": 24, "heads": 32, "inner": 8192,
         "vocab": 51200},
        # Phi-1.5 reading a prompt of an image's 729 positions and some text, one of its blocks
        {"name": "prefill_block_768", "kind": "block", "seq": 768, "heads": 32, "head_dim": 64, "inner": 8192,
         "causal": True, "graph": False},
        # a SigLIP layer on one image (always 729 patches, so a program keeps its graph)
        {"name": "vision_block_729", "kind": "block", "seq": 729, "heads": 16, "head_dim": 72, "inner": 4304,
         "causal": False, "graph": True},
        # the largest product: a long batch of prompts through a square projection
        {"name": "gemm_bf16_4096", "kind": "gemm", "dtype": "bf16", "out": "f32", "m": 4096, "n": 4096, "k": 4096,
         "gelu": False},
        # a short prompt, 32 positions
        {"name": "gemm_f16_32x2048x2048", "kind": "gemm", "dtype": "f16", "out": "f16", "m": 32, "n": 2048, "k": 2048,
         "gelu": False},
        # a SigLIP layer's attention scores
        {"name": "scores_16x729x72", "kind": "scores", "heads": 16, "seq": 729, "head_dim": 72},
        # the reference's tiled GEMM at its bench's medium size, bit for bit
        {"name": "exact_tiled_2048", "kind": "exact", "op": "tiled", "m": 2048, "n": 2048, "k": 2048},
    ]


def _log(rng, lo, hi, step=1):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["gemv", "token", "batch", "block", "gemm", "scores", "exact"])
    if kind == "gemv":
        dtype = rng.choice(["f32", "f16", "bf16", "q8_0", "q4_0"])
        step = 32 if dtype[0] == "q" else rng.choice([1, 8, 64])
        return {"kind": kind, "dtype": dtype, "n": _log(rng, 64, 51200), "k": _log(rng, 256, 8192, step),
                "gelu": rng.random() < 0.3}
    if kind in ("token", "batch"):
        heads = rng.randrange(12, 33)
        case = {"kind": kind, "dtype": rng.choice(["q8_0", "q4_0"]), "layers": rng.randrange(2, 25), "heads": heads,
                "inner": 32 * rng.randrange(4 * heads, 8 * heads + 1), "vocab": _log(rng, 4000, 51200)}
        if kind == "token":
            case["cache"] = _log(rng, 16, 2047)
        else:
            case["m"] = rng.randrange(2, 17)
        return case
    if kind == "block":
        heads, head_dim = rng.randrange(8, 33), rng.choice([64, 64, 72, 80])
        hidden = heads * head_dim
        return {"kind": kind, "seq": _log(rng, 24, 1024), "heads": heads, "head_dim": head_dim,
                "inner": 8 * rng.randrange(hidden // 3, hidden // 2 + 1), "causal": rng.random() < 0.5,
                "graph": rng.random() < 0.5}
    if kind == "gemm":
        dtype = rng.choice(["f16", "bf16"])
        return {"kind": kind, "dtype": dtype, "out": rng.choice(["f32", dtype]), "m": _log(rng, 17, 4096),
                "n": _log(rng, 256, 4096), "k": _log(rng, 256, 4096, rng.choice([1, 4, 8, 64])),
                "gelu": rng.random() < 0.3}
    if kind == "scores":
        return {"kind": kind, "heads": rng.randrange(4, 33), "seq": _log(rng, 64, 1024),
                "head_dim": rng.choice([64, 72, 80])}
    op = rng.choice(["naive", "tiled", "gemv"])
    return {"kind": kind, "op": op, "m": 1 if op == "gemv" else _log(rng, 16, 2048), "n": _log(rng, 256, 2048),
            "k": _log(rng, 256, 2048)}


# ---- inputs --------------------------------------------------------------------

class _InPlace:
    """A buffer as torch sees it.  The C ABI's handles are opaque and have no
    accessor for the device address, so it is read from the handle (the second
    word of mvlm_buffer); the buffer lives as long as the tensor."""

    def __init__(self, buf, count, typestr):
        self.buf = buf
        address = ctypes.c_uint64.from_address(buf.handle.value + 8).value
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (address, False), "version": 2}


def tensor(buf, dtype, shape):
    count = math.prod(shape)
    typestr = {torch.float32: "<f4", torch.float16: "<f2", torch.bfloat16: "<i2", torch.uint8: "|u1",
               torch.int32: "<i4"}[dtype]
    t = torch.as_tensor(_InPlace(buf, count, typestr), device="cuda")
    return (t.view(torch.bfloat16) if dtype == torch.bfloat16 else t).view(shape)


def buffer(t):
    """A device buffer holding t's values (t on the GPU, contiguous)."""
    buf = device().alloc(t.numel() * t.element_size())
    tensor(buf, t.dtype, t.shape).copy_(t)
    return buf


def empty(dtype, *shape):
    return device().alloc(math.prod(shape) * torch.empty((), dtype=dtype).element_size())


class Source:
    """Seeded values on the GPU, the same for prepare() and exact()."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, std=1.0):
        t = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, std, generator=self.gen)
        return t.to(dtype)

    def blocks(self, dtype, n, k):
        """GGUF blocks of an [n][k] weight: fp16 scale, then 32 signed bytes or 16 bytes of nibbles."""
        count = n * (k // 32)
        codes = 32 if dtype == "q8_0" else 16
        raw = torch.randint(0, 256, (count, codes), dtype=torch.uint8, device="cuda", generator=self.gen)
        if dtype == "q8_0":
            raw[raw == 128] = 129   # codes are -127 .. 127
        scale = self.normal(count, std=0.02).abs_().div_(127.0 if dtype == "q8_0" else 8.0).to(torch.float16)
        return torch.cat([scale.view(torch.uint8).view(count, 2), raw], 1).contiguous()

    def weight(self, dtype, n, k):
        """What a model file holds: GGUF blocks or an [n][k] array."""
        if dtype[0] == "q":
            return self.blocks(dtype, n, k)
        return self.normal(n, k, dtype=TORCH[DTYPE[dtype]], std=0.02)


def dequant(dtype, w, n, k):
    """The weight's values in 64 bits, from the GGUF definition."""
    if dtype[0] != "q":
        return w.double()
    d = w[:, :2].contiguous().view(torch.float16).double()
    q = w[:, 2:]
    if dtype == "q8_0":
        v = q.contiguous().view(torch.int8).double()
    else:
        v = torch.cat([(q & 15), (q >> 4)], 1).double() - 8.0
    return (d * v).view(n, k)


def pack(dtype, w, n, k):
    staged = buffer(w)
    torch.cuda.synchronize()
    return device().pack_device(staged, DTYPE[dtype], n, k)


def layer_shapes(case):
    hidden = case["heads"] * HEAD_DIM
    return hidden, {"qkv": (3 * hidden, hidden), "dense": (hidden, hidden), "fc1": (case["inner"], hidden),
                    "fc2": (hidden, case["inner"])}


def gelu(v):
    return 0.5 * v * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (v + 0.044715 * v * v * v)))


class _Model:
    """The values of a token / batch case in the order both users draw them."""

    def __init__(self, case, seed):
        self.case, self.src = case, Source(seed)
        self.hidden, self.shapes = layer_shapes(case)
        self.rows = case.get("m", 1)
        self.x = self.src.normal(self.rows, self.hidden)
        self.bias = {name: self.src.normal(n, std=0.02) for name, (n, _) in self.shapes.items()}

    def layers(self):
        for _ in range(self.case["layers"]):
            w = {name: self.src.weight(self.case["dtype"], n, k) for name, (n, k) in self.shapes.items()}
            if self.case["kind"] == "token":
                kv = [self.src.normal(self.case["cache"] + 1, self.hidden, dtype=torch.float16) for _ in range(2)]
                yield w, kv
            else:
                yield w, self.src.normal(self.rows, self.hidden)

    def head(self):
        return self.src.weight(self.case["dtype"], self.case["vocab"], self.hidden)


# ---- prepare / run ---------------------------------------------------------------

def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    """One pass: the enqueued call and the tensors it writes."""
    state["call"]()
    return state["out"]


def _prepare_gemv(case, seed):
    dev, src = device(), Source(seed)
    n, k, dtype = case["n"], case["k"], case["dtype"]
    act = m.F32 if dtype[0] == "q" else DTYPE[dtype]
    x = buffer(src.normal(k, dtype=TORCH[act]))
    bias = buffer(src.normal(n, dtype=TORCH[act], std=0.02))
    W = pack(dtype, src.weight(dtype, n, k), n, k)
    y = empty(TORCH[act], n)
    if case["gelu"]:
        def call():
            dev.gemv_ex(x, act, W, y, act, n, k, bias=bias, act=m.native.ACT_GELU_TANH)
    else:
        def call():
            dev.gemv(x, act, W, y, act, n, k)
    return {"call": call, "out": [tensor(y, TORCH[act], (n,))]}


def _prepare_token(case, seed):
    dev, model = device(), _Model(case, seed)
    hidden, inner, layers, vocab = model.hidden, case["inner"], case["layers"], case["vocab"]
    x = buffer(model.x.view(-1))
    bias = {name: buffer(v) for name, v in model.bias.items()}
    # one slab per kind of output, a layer's share of it as a view
    slab = {name: empty(torch.float32, layers, n) for name, (n, _) in model.shapes.items()}
    slab["attn"] = empty(torch.float32, layers, hidden)
    rows = []
    plan = m.Plan(dev)
    for i, (w, (kc, vc)) in enumerate(model.layers()):
        W = {name: pack(case["dtype"], w[name], n, k) for name, (n, k) in model.shapes.items()}
        y = {name: slab[name].view(i * n * 4, n * 4) for name, (n, _) in model.shapes.items()}
        o = slab["attn"].view(i * hidden * 4, hidden * 4)
        kc, vc = buffer(kc), buffer(vc)
        plan.add_gemv_grouped([(x, m.F32, W["qkv"], y["qkv"], m.F32), (x, m.F32, W["fc1"], y["fc1"], m.F32)],
                              epilogues=[{"bias": bias["qkv"]}, {"bias": bias["fc1"], "act": m.native.ACT_GELU_TANH}])
        plan.add_attention_decode_step(y["qkv"], kc, vc, o, case["cache"], case["heads"], HEAD_DIM)
        plan.add_gemv_grouped([(o, m.F32, W["dense"], y["dense"], m.F32), (y["fc1"], m.F32, W["fc2"], y["fc2"], m.F32)],
                              epilogues=[{"bias": bias["dense"], "residual": x}, {"bias": bias["fc2"], "residual": x}])
        shape = (case["cache"] + 1, hidden)
        rows += [tensor(c, torch.float16, shape)[case["cache"]] for c in (kc, vc)]
        last = y["fc2"]
    W = pack(case["dtype"], model.head(), vocab, hidden)
    logits, token = empty(torch.float32, vocab), empty(torch.int32, 1)
    plan.add_gemv(last, m.F32, W, logits, m.F32, 1)
    plan.add_argmax(logits, m.F32, 1, vocab, vocab, token)
    torch.cuda.synchronize()
    plan.use_graph(True)
    out = {name: tensor(buf, torch.float32, (layers, buf.nbytes // 4 // layers)) for name, buf in slab.items()}
    return {"call": plan.run, "plan": plan,
            "out": {**out, "rows": rows, "logits": tensor(logits, torch.float32, (vocab,)),
                    "token": tensor(token, torch.int32, (1,))}}


def _prepare_batch(case, seed):
    dev, model = device(), _Model(case, seed)
    hidden, layers, vocab, M = model.hidden, case["layers"], case["vocab"], case["m"]
    x = buffer(model.x)
    bias = {name: buffer(v) for name, v in model.bias.items()}
    slab = {name: empty(torch.float32, layers, M, n) for name, (n, _) in model.shapes.items()}
    plan = m.Plan(dev)
    for i, (w, attn) in enumerate(model.layers()):
        W = {name: pack(case["dtype"], w[name], n, k) for name, (n, k) in model.shapes.items()}
        y = {name: slab[name].view(i * M * n * 4, M * n * 4) for name, (n, _) in model.shapes.items()}
        attn = buffer(attn)
        plan.add_gemm_quant_grouped(M, [(x, m.F32, W["qkv"], y["qkv"], m.F32), (x, m.F32, W["fc1"], y["fc1"], m.F32)],
                                    epilogues=[{"bias": bias["qkv"]},
                                               {"bias": bias["fc1"], "act": m.native.ACT_GELU_TANH}])
        plan.add_gemm_quant_grouped(M, [(attn, m.F32, W["dense"], y["dense"], m.F32),
                                        (y["fc1"], m.F32, W["fc2"], y["fc2"], m.F32)],
                                    epilogues=[{"bias": bias["dense"], "residual": x},
                                               {"bias": bias["fc2"], "residual": x}])
        last = y["fc2"]
    W = pack(case["dtype"], model.head(), vocab, hidden)
    logits = empty(torch.float32, M, vocab)
    plan.add_gemv(last, m.F32, W, logits, m.F32, M)
    torch.cuda.synchronize()
    plan.use_graph(True)
    out = {name: tensor(buf, torch.float32, (layers, M, buf.nbytes // 4 // layers // M)) for name, buf in slab.items()}
    return {"call": plan.run, "plan": plan, "out": {**out, "logits": tensor(logits, torch.float32, (M, vocab))}}


def _block_values(case, seed):
    src, hidden, S, inner = Source(seed), case["heads"] * case["head_dim"], case["seq"], case["inner"]
    shapes = {"qkv": (3 * hidden, hidden), "dense": (hidden, hidden), "fc1": (inner, hidden), "fc2": (hidden, inner)}
    v = {name: src.normal(S, hidden, dtype=torch.float16) for name in ("x", "Q", "K", "V")}
    w = {name: src.weight("f16", n, k) for name, (n, k) in shapes.items()}
    b = {name: src.normal(n, dtype=torch.float16, std=0.02) for name, (n, _) in shapes.items()}
    return shapes, v, w, b


def _prepare_block(case, seed):
    dev, S, F = device(), case["seq"], m.F16
    shapes, v, w, b = _block_values(case, seed)
    v = {name: buffer(t) for name, t in v.items()}
    b = {name: buffer(t) for name, t in b.items()}
    W = {name: pack("f16", w[name], n, k) for name, (n, k) in shapes.items()}
    hidden = shapes["dense"][0]
    y = {name: empty(torch.float16, S, n) for name, (n, _) in shapes.items()}
    attn = empty(torch.float16, S, hidden)
    plan = m.Plan(dev)
    plan.add_gemm_packed_ex(v["x"], F, W["qkv"], y["qkv"], F, S, bias=b["qkv"])
    plan.add_attention(v["Q"], v["K"], v["V"], attn, F, S, S, case["heads"], case["head_dim"], causal=case["causal"])
    plan.add_gemm_packed_ex(attn, F, W["dense"], y["dense"], F, S, bias=b["dense"], residual=v["x"])
    plan.add_gemm_packed_ex(v["x"], F, W["fc1"], y["fc1"], F, S, bias=b["fc1"], act=m.native.ACT_GELU_TANH)
    plan.add_gemm_packed_ex(y["fc1"], F, W["fc2"], y["fc2"], F, S, bias=b["fc2"], residual=y["dense"])
    torch.cuda.synchronize()
    if case["graph"]:
        plan.use_graph(True)
    out = {name: tensor(y[name], torch.float16, (S, n)) for name, (n, _) in shapes.items()}
    return {"call": plan.run, "plan": plan, "out": {**out, "attn": tensor(attn, torch.float16, (S, hidden))}}


def _gemm_values(case, seed):
    src, t = Source(seed), TORCH[DTYPE[case["dtype"]]]
    return (src.normal(case["m"], case["k"], dtype=t), src.weight(case["dtype"], case["n"], case["k"]),
            src.normal(case["n"], dtype=TORCH[DTYPE[case["out"]]], std=0.02))


def _prepare_gemm(case, seed):
    dev, M, N, K = device(), case["m"], case["n"], case["k"]
    a, w, b = _gemm_values(case, seed)
    A, bias, W = buffer(a), buffer(b), pack(case["dtype"], w, N, K)
    ad, cd = DTYPE[case["dtype"]], DTYPE[case["out"]]
    C = empty(TORCH[cd], M, N)
    if case["gelu"]:
        def call():
            dev.gemm_packed_ex(A, ad, W, C, cd, M, N, K, bias=bias, act=m.native.ACT_GELU_TANH)
    else:
        def call():
            dev.gemm_packed(A, ad, W, C, cd, M, N, K)
    return {"call": call, "out": [tensor(C, TORCH[cd], (M, N))]}


def _scores_values(case, seed):
    src, shape = Source(seed), (case["heads"], case["seq"], case["head_dim"])
    return src.normal(*shape, dtype=torch.float16), src.normal(*shape, dtype=torch.float16)


def _prepare_scores(case, seed):
    dev, H, S, D = device(), case["heads"], case["seq"], case["head_dim"]
    q, k = _scores_values(case, seed)
    Q, K, C = buffer(q), buffer(k), empty(torch.float32, H, S, S)

    def call():
        dev.gemm_batched(Q, K, C, H, S, S, D, D, D, S, S * D, S * D, S * S)
    return {"call": call, "out": [tensor(C, torch.float32, (H, S, S))]}


def _exact_values(case, seed):
    src = Source(seed)
    return (src.normal(case["m"], case["k"], dtype=torch.float16),
            src.normal(case["k"], case["n"], dtype=torch.float16, std=0.02))


def _prepare_exact(case, seed):
    dev, M, N, K = device(), case["m"], case["n"], case["k"]
    a, b = _exact_values(case, seed)
    A, B, C = buffer(a), buffer(b), empty(torch.float16, M, N)
    if case["op"] == "gemv":
        torch.cuda.synchronize()
        W = dev.pack_device(B, m.F16, N, K, layout=m.LAYOUT_KN)

        def call():
            dev.gemv_exact(A, W, C, N, K)
    elif case["op"] == "tiled":
        def call():
            dev.gemm_tiled(A, B, C, M, N, K)
    else:
        def call():
            dev.gemm_naive(A, B, C, M, N, K)
    return {"call": call, "out": [tensor(C, torch.float16, (M, N))]}


# ---- 64-bit results --------------------------------------------------------------

def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)


def _exact_gemv(case, seed):
    src, n, k, dtype = Source(seed), case["n"], case["k"], case["dtype"]
    act = torch.float32 if dtype[0] == "q" else TORCH[DTYPE[dtype]]
    x, bias = src.normal(k, dtype=act).double(), src.normal(n, dtype=act, std=0.02).double()
    y = dequant(dtype, src.weight(dtype, n, k), n, k) @ x
    return [gelu(y + bias) if case["gelu"] else y]


def _exact_token(case, seed):
    model, heads = _Model(case, seed), case["heads"]
    x, bias = model.x.double().view(-1), {name: v.double() for name, v in model.bias.items()}
    out = {name: [] for name in (*model.shapes, "attn")}
    rows = []
    for w, (kc, vc) in model.layers():
        w = {name: dequant(case["dtype"], w[name], n, k) for name, (n, k) in model.shapes.items()}
        qkv = w["qkv"] @ x + bias["qkv"]
        fc1 = gelu(w["fc1"] @ x + bias["fc1"])
        # the step keeps q and the new key and value in fp16, as the cache does
        q, new_k, new_v = qkv.float().to(torch.float16).double().view(3, -1)
        kk, vv = kc.double(), vc.double()
        kk[-1], vv[-1] = new_k, new_v
        s = torch.einsum("hd,chd->hc", q.view(heads, -1), kk.view(-1, heads, HEAD_DIM)) / math.sqrt(HEAD_DIM)
        o = torch.einsum("hc,chd->hd", torch.softmax(s, 1), vv.view(-1, heads, HEAD_DIM)).reshape(-1)
        y = {"qkv": qkv, "fc1": fc1, "attn": o, "dense": w["dense"] @ o + bias["dense"] + x,
             "fc2": w["fc2"] @ fc1 + bias["fc2"] + x}
        for name, v in y.items():
            out[name].append(v)
        rows += [new_k, new_v]
    logits = dequant(case["dtype"], model.head(), case["vocab"], model.hidden) @ out["fc2"][-1]
    return {**{name: torch.stack(v) for name, v in out.items()}, "rows": rows, "logits": logits, "token": None}


def _exact_batch(case, seed):
    model = _Model(case, seed)
    x, bias = model.x.double(), {name: v.double() for name, v in model.bias.items()}
    out = {name: [] for name in model.shapes}
    for w, attn in model.layers():
        w = {name: dequant(case["dtype"], w[name], n, k) for name, (n, k) in model.shapes.items()}
        fc1 = gelu(x @ w["fc1"].T + bias["fc1"])
        y = {"qkv": x @ w["qkv"].T + bias["qkv"], "fc1": fc1, "dense": attn.double() @ w["dense"].T + bias["dense"] + x,
             "fc2": fc1 @ w["fc2"].T + bias["fc2"] + x}
        for name, v in y.items():
            out[name].append(v)
    logits = out["fc2"][-1] @ dequant(case["dtype"], model.head(), case["vocab"], model.hidden).T
    return {**{name: torch.stack(v) for name, v in out.items()}, "logits": logits}


def _exact_block(case, seed):
    shapes, v, w, b = _block_values(case, seed)
    S, heads, D = case["seq"], case["heads"], case["head_dim"]
    v, w, b = ({name: t.double() for name, t in d.items()} for d in (v, w, b))
    q, k, vv = (v[name].view(S, heads, D).transpose(0, 1).contiguous() for name in "QKV")
    o = torch.empty_like(q)
    hidden_from = torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1)
    for h in range(heads):
        s = q[h] @ k[h].T.contiguous() / math.sqrt(D)
        if case["causal"]:
            s = s.masked_fill(hidden_from, -math.inf)
        o[h] = torch.softmax(s, 1) @ vv[h]
    attn = o.transpose(0, 1).reshape(S, heads * D)
    fc1 = gelu(v["x"] @ w["fc1"].T + b["fc1"])
    dense = attn @ w["dense"].T + b["dense"] + v["x"]
    return {"qkv": v["x"] @ w["qkv"].T + b["qkv"], "attn": attn, "dense": dense, "fc1": fc1,
            "fc2": fc1 @ w["fc2"].T + b["fc2"] + dense}


def _exact_gemm(case, seed):
    a, w, b = _gemm_values(case, seed)
    c = a.double() @ w.double().T
    return [gelu(c + b.double()) if case["gelu"] else c]


def _exact_scores(case, seed):
    q, k = _scores_values(case, seed)
    return [torch.stack([q[h].double() @ k[h].double().T for h in range(case["heads"])])]


def _exact_exact(case, seed):
    a, b = _exact_values(case, seed)
    return [a.double() @ b.double()]


# ---- what a pass cannot do without, and how far two right answers are apart --------

def work(case):
    kind = case["kind"]
    if kind == "gemv":
        n, k, w = case["n"], case["k"], SIZE[case["dtype"]]
        act = 4 if case["dtype"][0] == "q" else w
        return {"bytes": n * k * w + (k + n) * act, "flops": 2 * n * k}
    if kind in ("token", "batch"):
        hidden, shapes = layer_shapes(case)
        M, w = case.get("m", 1), SIZE[case["dtype"]]
        mats = [nk for _ in range(case["layers"]) for nk in shapes.values()] + [(case["vocab"], hidden)]
        total = sum(n * k * w + 4 * M * (n + k) for n, k in mats)
        flops = sum(2 * M * n * k for n, k in mats)
        if kind == "token":
            total += case["layers"] * 2 * (case["cache"] + 1) * hidden * 2 + 4 * case["vocab"]
            flops += case["layers"] * 4 * (case["cache"] + 1) * hidden
        return {"bytes": total, "flops": flops}
    if kind == "block":
        S, hidden, inner = case["seq"], case["heads"] * case["head_dim"], case["inner"]
        weights = 4 * hidden * hidden + 2 * hidden * inner
        keys = (S + 1) / 2 if case["causal"] else S
        return {"bytes": 2 * (weights + S * (4 * hidden + 3 * hidden + hidden + hidden + inner + hidden)),
                "flops": 2 * S * weights + 4 * S * keys * hidden}
    if kind == "scores":
        H, S, D = case["heads"], case["seq"], case["head_dim"]
        return {"bytes": H * (2 * S * D * 2 + S * S * 4), "flops": 2 * H * S * S * D}
    M, N, K = case["m"], case["n"], case["k"]
    out = SIZE[case["out"]] if kind == "gemm" else 2
    return {"bytes": 2 * (M * K + N * K) + out * M * N, "flops": 2 * M * N * K}


def tolerance(case):
    """About four times what the path is off its 64-bit result in fp32 outputs
    (1e-7 to 4e-7 over K = 256 .. 8192).  Outputs rounded to 16 bits differ in
    the last place where two fp32 sums fall on either side of a rounding
    boundary: one place is 2^-10 (fp16) or 2^-7 (bf16) of a value at most, and
    few values are hit.  A block's attention rounds its probabilities to fp16,
    against a running maximum that depends on the order of the keys."""
    kind = case["kind"]
    flips = {"f16": {"rel": 2e-4, "max": 2e-3}, "bf16": {"rel": 1.6e-3, "max": 1.6e-2}}
    if kind == "exact":
        return "exact"                       # one order of summation, one rounding
    if kind == "gemv":
        return flips.get(case["dtype"], {"rel": 2e-6})
    if kind == "gemm":
        return flips.get(case["out"], {"rel": 2e-6})
    if kind == "token":                      # q, the new key and value are rounded to fp16
        return {"rel": 1e-4}
    if kind == "block":
        return {"rel": 1e-3, "max": 2e-2}
    return {"rel": 2e-6}
