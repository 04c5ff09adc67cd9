"""The calls whose time and results are watched, and how to make their inputs.

Each case is one pass through the public surface a user's program calls:
``ComputeEngine`` (the fused quantized linear, the SwiGLU MLP, the LoRA
linear, the f32 matmul family, the input gradient) or ``LlamaRunner`` (a whole
generation).  Buffers live on the GPU as torch tensors, handed over as
``UnifiedTensor`` views; weights are made once per state, as a program loads
them once.

Values: Linear weights have standard deviation 0.02 around zero (the usual
Llama init) as int8 codes with a scale per row or u8 codes with a scale and
bias per group; activations and gradients are normal.
"""
from __future__ import annotations

import math

import torch

from rusty_amd import ComputeEngine, DType, QuantizedTensor, UnifiedTensor, WgpuContext
from rusty_amd import lib as _library
from rusty_amd.llama import LLAMA_1B, LlamaConfig, LlamaHostWeights, LlamaRunner

W_STD = 0.02
CODE_STD = 73.3  # of codes uniform in [-127, 127]

_DTYPES = {"f16": (torch.float16, DType.FP16), "f32": (torch.float32, DType.FP32)}
_shared = {}


def _engine():
    """One context and engine for the process, as a program has."""
    if not _shared:
        _shared["ctx"] = WgpuContext(0)
        _shared["eng"] = ComputeEngine(_shared["ctx"])
    return _shared["ctx"], _shared["eng"]


# ---- the cases ---------------------------------------------------------------


def listed():
    return [
        # One token through one Linear of a 7B-shape block: the smallest call a
        # decoding program makes, latency and launch included.
        _linear("linear_one_token", 1, 4096, 4096, 0, "f16", "f16"),
        # A small ragged batch in the reference's own formats: affine codes
        # with a scale and bias per 64, f32 activations (13 sequences).
        _linear("linear_batch_affine_f32", 13, 4096, 4096, 64, "f32", "f32"),
        # A 7B-shape MLP for a decoding batch of 8 (11008 x 4096 weights).
        {"name": "mlp_batch", "op": "mlp", "m": 8, "hidden": 4096, "inner": 11008, "group": 0, "dtype": "f16"},
        # A long prompt through one Linear: the compute-bound end.
        _linear("linear_prompt", 2048, 4096, 4096, 0, "f16", "f16"),
        # A prompt of odd length through an MLP-up-sized Linear in the
        # reference's formats (affine codes, f32 in and out).
        _linear("linear_prompt_affine_f32", 777, 11008, 4096, 64, "f32", "f32"),
        # A short prompt through the MLP of a 1.1B-shape block.
        {"name": "mlp_prompt", "op": "mlp", "m": 300, "hidden": 2048, "inner": 5632, "group": 0, "dtype": "f16"},
        # The f32 matmul the reference publishes, and the small one of its
        # dequantize-then-multiply path (8 rows against a 1024 x 1024 weight).
        {"name": "matmul_large", "op": "matmul", "kind": "ab", "m": 4096, "k": 4096, "n": 4096},
        {"name": "matmul_small", "op": "matmul", "kind": "abt", "m": 8, "k": 1024, "n": 1024},
        # Backward through a frozen affine weight (the reference's format), in
        # the reference's arithmetic.
        {"name": "input_gradient", "op": "dx", "m": 512, "n": 4096, "k": 4096, "group": 64, "mfma": False},
        # One fine-tuning step of one Linear with a rank-16 adapter: forward,
        # input gradient, and the gradients of A and B.
        {"name": "lora_step", "op": "lora", "m": 512, "n": 4096, "k": 4096, "rank": 16, "group": 0},
        # A chat answer: 512 prompt tokens, 128 greedy tokens, 1.1B shape.
        _generate("generate", 512, 128, 0),
        # A long document and a short answer: 4096 prompt tokens, 32 tokens.
        _generate("generate_long", 4096, 32, 0),
    ]


def _linear(name, m, n, k, group, x, y):
    return {"name": name, "op": "linear", "m": m, "n": n, "k": k, "group": group, "x": x, "y": y}


def _generate(name, prompt, steps, group):
    return {"name": name, "op": "generate", "prompt": prompt, "steps": steps, "layers": LLAMA_1B.n_layers,
            "group": group}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, step):
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    """One more case of the same ranges: token counts 1..2048 and widths
    256..11008 over their logarithms (odd counts and ragged widths among
    them), every weight format and dtype, prompts of 16..4096 tokens."""
    op = rng.choices(["linear", "mlp", "matmul", "dx", "lora", "generate"], [40, 14, 18, 9, 11, 8])[0]
    group = rng.choice([0, 0, 64, 64, 128, 32])
    if op == "linear":
        k = _width(rng, 256, 11008, max(group, rng.choice([64, 64, 64, 32, 16])))
        n = _width(rng, 256, 11008, rng.choice([64, 64, 64, 16, 8, 1]))
        x, y = rng.choice([("f16", "f16"), ("f16", "f16"), ("f32", "f32"), ("f16", "f32")])
        # a large weight that the matrix-core kernels refuse takes long per token
        m = _log(rng, 1, 2048 if group != 32 and k % 64 == 0 else 256)
        c = _linear("", m, n, k, group, x, y)
    elif op == "mlp":
        c = {"op": "mlp", "m": _log(rng, 1, 1024 if group != 32 else 128),
             "hidden": _width(rng, 512, 4096, 128), "inner": _width(rng, 1024, 11008, 128),
             "group": group, "dtype": rng.choice(["f16", "f16", "f32"])}
    elif op == "matmul":
        step = rng.choice([64, 16, 4, 1])
        c = {"op": "matmul", "kind": rng.choice(["ab", "abt", "atb"]), "m": _width(rng, 1, 4096, rng.choice([1, 8])),
             "k": _width(rng, 16, 4096, step), "n": _width(rng, 8, 4096, step)}
    elif op == "dx":
        c = {"op": "dx", "m": _log(rng, 1, 1024), "n": _width(rng, 256, 11008, 64),
             "k": _width(rng, 256, 4096, max(group, 64)), "group": group, "mfma": group == 0 and rng.random() < 0.5}
    elif op == "lora":
        c = {"op": "lora", "m": _log(rng, 16, 1024), "n": _width(rng, 256, 8192, 64), "k": _width(rng, 256, 4096, 128),
             "rank": rng.choice([4, 8, 16, 32, 64]), "group": rng.choice([0, 0, 64])}
    else:
        c = _generate("", _log(rng, 16, 4096), _log(rng, 4, 64), rng.choice([0, 64]))
        c["layers"] = rng.choice([4, 8, 16])
    c.pop("name", None)
    return c


# ---- inputs --------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, dtype, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(dtype)


def _codes(g, n, k, group):
    """A weight as torch tensors: (q, scale) per row, or (u, scale, bias, group)."""
    if not group:
        q = torch.randint(-127, 128, (n, k), generator=g, device="cuda", dtype=torch.int8)
        s = (torch.rand(n, generator=g, device="cuda") + 0.5) * (W_STD / CODE_STD)
        return q, s
    u = torch.randint(0, 256, (n, k), generator=g, device="cuda", dtype=torch.uint8)
    s = (torch.rand((n, k // group), generator=g, device="cuda") + 0.5) * (W_STD / CODE_STD)
    b = -128.0 * s * (0.98 + 0.04 * torch.rand(s.shape, generator=g, device="cuda"))
    return u, s, b, group


def _view(t):
    kind = {torch.float16: DType.FP16, torch.float32: DType.FP32, torch.int8: DType.I8, torch.uint8: DType.U8}[t.dtype]
    return UnifiedTensor(_engine()[0], t.data_ptr(), t.shape, kind, owner=False)


def _weight(state, w):
    """The QuantizedTensor of codes on the GPU, with its load-time table."""
    state["keep"].append(w)
    n, k = w[0].shape
    if len(w) == 2:
        return QuantizedTensor(_view(w[0]), _view(w[1]), None, n, k, 0, 0)
    qt = QuantizedTensor(_view(w[0]), _view(w[1]), _view(w[2]), n, k, 1, w[3])
    torch.cuda.synchronize()  # the codes are there before the table is made from them
    qt.prepare(_engine()[0])
    return qt


def _deq(w):
    """The weight a quantized Linear stands for, in 64 bits."""
    if len(w) == 2:
        return w[0].double() * w[1].double()[:, None]
    return w[0].double() * w[1].double().repeat_interleave(w[3], 1) + w[2].double().repeat_interleave(w[3], 1)


def _inputs(case, seed):
    """The tensors of a case, by name, made from the seed alone."""
    g = _gen(seed)
    op = case["op"]
    if op == "linear":
        t = {"w": _codes(g, case["n"], case["k"], case["group"]),
             "x": _normal(g, (case["m"], case["k"]), _DTYPES[case["x"]][0])}
    elif op == "mlp":
        h, i, gr = case["hidden"], case["inner"], case["group"]
        t = {"gate": _codes(g, i, h, gr), "up": _codes(g, i, h, gr), "down": _codes(g, h, i, gr),
             "x": _normal(g, (case["m"], h), _DTYPES[case["dtype"]][0])}
    elif op == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        t = {"a": _normal(g, (k, m) if case["kind"] == "atb" else (m, k), torch.float32),
             "b": _normal(g, (n, k) if case["kind"] == "abt" else (k, n), torch.float32, W_STD)}
    elif op == "dx":
        t = {"w": _codes(g, case["n"], case["k"], case["group"]),
             "dy": _normal(g, (case["m"], case["n"]), torch.float32, 1e-2)}
    elif op == "lora":
        m, n, k, r = case["m"], case["n"], case["k"], case["rank"]
        t = {"w": _codes(g, n, k, case["group"]), "x": _normal(g, (m, k), torch.float32),
             "a": _normal(g, (k, r), torch.float32, 1.0 / math.sqrt(k)), "b": _normal(g, (r, n), torch.float32, W_STD),
             "dy": _normal(g, (m, n), torch.float32, 1e-2)}
    else:
        t = _model(case, g)
    return t


def _model(case, g):
    """A 1.1B-shape model (of `layers` blocks) and a prompt.  The lm_head's
    rows are the embedding's, quantized and permuted, so that the model is as
    sure of its next token as a trained one is (random rows would leave the
    greedy pick to the last bits of the logits)."""
    cfg = _config(case)
    gr = case["group"]
    norm = lambda: (0.9 + 0.2 * torch.rand(cfg.hidden, generator=g, device="cuda")).half()  # noqa: E731
    embed = _normal(g, (cfg.vocab, cfg.hidden), torch.float16)
    layers = []
    for _ in range(cfg.n_layers):
        layer = {name: _codes(g, n, k, gr) for name, (n, k) in cfg.linear_shapes().items()}
        layers.append({"attn_norm": norm(), "mlp_norm": norm(), **layer})
    rows = embed[torch.randperm(cfg.vocab, generator=g, device="cuda")].float()
    if gr:
        part = rows.view(cfg.vocab, cfg.hidden // gr, gr)
        top = part.abs().amax(2)
        s = top / 127
        head = ((part / s[:, :, None]).round() + 128).to(torch.uint8).view(cfg.vocab, cfg.hidden), s * W_STD, \
            -128.0 * s * W_STD, gr
    else:
        s = rows.abs().amax(1) / 127
        head = (rows / s[:, None]).round().to(torch.int8), s * W_STD
    tokens = torch.randint(0, cfg.vocab, (case["prompt"],), generator=g, device="cuda", dtype=torch.int32)
    return {"embed": embed, "layers": layers, "final_norm": norm(), "lm_head": head, "tokens": tokens}


def _config(case):
    c = LLAMA_1B
    return LlamaConfig(n_layers=case["layers"], hidden=c.hidden, n_heads=c.n_heads, n_kv_heads=c.n_kv_heads,
                       head_dim=c.head_dim, intermediate=c.intermediate, vocab=c.vocab,
                       max_seq=-(-(case["prompt"] + case["steps"]) // 64) * 64)


def prepare(case, seed):
    ctx, _ = _engine()
    t = _inputs(case, seed)
    s = {"op": case["op"], "keep": [t]}
    op = case["op"]
    new = lambda shape, dtype: torch.empty(shape, dtype=dtype, device="cuda")  # noqa: E731
    if op == "linear":
        y = new((case["m"], case["n"]), _DTYPES[case["y"]][0])
        s.update(w=_weight(s, t["w"]), x=_view(t["x"]), y=_view(y), out=y)
    elif op == "mlp":
        y = new((case["m"], case["hidden"]), _DTYPES[case["dtype"]][0])
        h = new((2, case["m"], case["inner"]), torch.float16)
        s["keep"].append(h)
        s.update({k: _weight(s, t[k]) for k in ("gate", "up", "down")}, x=_view(t["x"]), y=_view(y), h=_view(h), out=y)
    elif op == "matmul":
        y = new((case["m"], case["n"]), torch.float32)
        s.update(kind=case["kind"], a=_view(t["a"]), b=_view(t["b"]), y=_view(y), out=y)
    elif op == "dx":
        dx = new((case["m"], case["k"]), torch.float32)
        s.update(w=_weight(s, t["w"]), dy=_view(t["dy"]), dx=_view(dx), mfma=case["mfma"], work=None, out=dx)
        if case["mfma"]:
            _dx_buffers(s, ctx, case["m"], case["n"])
    elif op == "lora":
        m, n, k, r = case["m"], case["n"], case["k"], case["rank"]
        s.update(w=_weight(s, t["w"]), x=_view(t["x"]), a=_view(t["a"]), b=_view(t["b"]), dy=_view(t["dy"]),
                 mfma=not case["group"], work=None)
        out = {"y": new((m, n), torch.float32), "xa": new((m, r), torch.float32), "db": new((r, n), torch.float32),
               "dxa": new((m, r), torch.float32), "da": new((k, r), torch.float32), "dx": new((m, k), torch.float32),
               "dx_adapter": new((m, k), torch.float32)}
        need = _library().rq_qmatmul_lora_workspace(m, k, n, r, 0, 0)
        lw = new(max(int(need), 1), torch.uint8)
        s["keep"].append(lw)
        s.update(out=out, v={name: _view(o) for name, o in out.items()}, lwork=_view(lw))
        if s["mfma"]:
            _dx_buffers(s, ctx, m, n)
    else:
        host = lambda v: tuple(x.cpu().numpy() if torch.is_tensor(x) else x for x in v) if isinstance(v, tuple) \
            else v.cpu().numpy()  # noqa: E731
        w = LlamaHostWeights(embed=host(t["embed"]), final_norm=host(t["final_norm"]), lm_head=host(t["lm_head"]))
        w.layers = [{name: host(v) for name, v in layer.items()} for layer in t["layers"]]
        s.update(keep=[], steps=case["steps"], prompt=host(t["tokens"]), model=LlamaRunner(ctx, _config(case), w))
    torch.cuda.synchronize()
    return s


def _dx_buffers(s, ctx, m, n):
    """What a training loop keeps for the matrix-core input gradient: the
    weight's transposed table and the workspace."""
    torch.cuda.synchronize()
    s["w"].dx_table(ctx)
    work = torch.empty(max(int(_library().rq_qmatmul_dx_mfma_workspace(m, n)), 1), dtype=torch.uint8, device="cuda")
    s["keep"].append(work)
    s["work"] = _view(work)


# ---- one pass -------------------------------------------------------------------


def run(state):
    ctx, eng = _engine()
    s, op = state, state["op"]
    if op == "linear":
        eng.qmatmul(ctx, s["x"], s["w"], s["y"])
    elif op == "mlp":
        eng.mlp_swiglu(ctx, s["x"], s["gate"], s["up"], s["down"], s["y"], s["h"])
    elif op == "matmul":
        {"ab": eng.matmul, "abt": eng.matmul_bt, "atb": eng.matmul_at}[s["kind"]](ctx, s["a"], s["b"], s["y"])
    elif op == "dx":
        eng.qmatmul_dx(ctx, s["dy"], s["w"], s["dx"], mfma=s["mfma"], workspace=s["work"])
    elif op == "lora":
        v = s["v"]
        eng.qmatmul_lora(ctx, s["x"], s["w"], s["a"], s["b"], v["y"], s["lwork"])
        eng.matmul(ctx, s["x"], s["a"], v["xa"])              # kept for the backward pass
        eng.matmul_at(ctx, v["xa"], s["dy"], v["db"])         # dB = (x A)^T dY
        eng.matmul_bt(ctx, s["dy"], s["b"], v["dxa"])         # d(x A) = dY B^T
        eng.matmul_at(ctx, s["x"], v["dxa"], v["da"])         # dA = x^T d(x A)
        eng.qmatmul_dx(ctx, s["dy"], s["w"], v["dx"], mfma=s["mfma"], workspace=s["work"])
        eng.matmul_bt(ctx, v["dxa"], s["a"], v["dx_adapter"])  # the adapter's share of dX
    else:
        model = s["model"]
        model.prefill(s["prompt"])
        model.decode(s["steps"])
        return {"tokens": model.tokens(), "logits": model.logits()}
    return s["out"]


# ---- what a pass cannot do without --------------------------------------------------


def _weight_bytes(n, k, group):
    return n * k + (8 * n * (k // group) if group else 4 * n)


def work(case):
    op = case["op"]
    size = {"f16": 2, "f32": 4}
    if op == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _weight_bytes(n, k, case["group"]) + m * k * size[case["x"]] + m * n * size[case["y"]],
                "flops": 2 * m * n * k}
    if op == "mlp":
        m, h, i, gr = case["m"], case["hidden"], case["inner"], case["group"]
        return {"bytes": 2 * _weight_bytes(i, h, gr) + _weight_bytes(h, i, gr) + 2 * m * h * size[case["dtype"]],
                "flops": 6 * m * h * i}
    if op == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if op == "dx":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _weight_bytes(n, k, case["group"]) + 4 * m * (n + k), "flops": 2 * m * n * k}
    if op == "lora":
        m, n, k, r = case["m"], case["n"], case["k"], case["rank"]
        # x, dY, the weight, A and B read once; y, dX (both shares), dA, dB, x A and its gradient written once
        return {"bytes": _weight_bytes(n, k, case["group"]) + 4 * (2 * m * (k + n) + m * k + 2 * r * (k + n) + 2 * m * r),
                "flops": 4 * m * n * k + 2 * m * r * (4 * k + 3 * n)}
    cfg = _config(case)
    p, d = case["prompt"], case["steps"]
    linears = sum(n * k for n, k in cfg.linear_shapes().values()) * cfg.n_layers
    head = cfg.vocab * cfg.hidden
    weights = cfg.weight_bytes(case["group"])
    pairs = p * (p + 1) // 2 + sum(p + i + 1 for i in range(d))  # (query, key) pairs of one head
    row = cfg.n_layers * cfg.n_kv_heads * cfg.head_dim * 2 * 2  # bytes of one position's K and V
    return {"bytes": (1 + d) * weights + row * (2 * p + sum(p + i + 1 for i in range(d))),
            "flops": 2 * linears * (p + d) + 2 * head * (1 + d) + 4 * cfg.head_dim * cfg.n_heads * cfg.n_layers * pairs}


# ---- how close, and the true result ----------------------------------------------------


def tolerance(case):
    op = case["op"]
    if op == "matmul" or (op == "dx" and not case["mfma"]):
        return "exact"  # one fma per term in a stated order: the entry points' contract
    if op == "dx":
        return {"rel": 5e-6}  # f32 sums in another order
    if op == "linear":
        # Sums are f32 everywhere.  fp16 outputs round once (2^-11); f32 activations stay f32 up to 16 rows and enter the
        # matrix cores as fp16 above, affine weights as fp16 from 3 rows on.
        if case["y"] == "f16" or case["m"] > 16 or (case["group"] and case["x"] == "f16"):
            return {"rel": 1e-3}
        return {"rel": 5e-6}
    if op == "mlp":
        return {"rel": 2e-3}  # the intermediate is fp16 too
    if op == "lora":
        return {"rel": 1e-3}  # the frozen product of m > 16 rows: fp16 inputs
    # Whole calls: fp16 activations through every layer; the greedy tokens are
    # far from ties (see _model), one in a hundred may differ.
    return {"rel": 5e-3, "differ": 0.01}


def exact(case, seed):
    t = _inputs(case, seed)
    op = case["op"]
    if op == "linear":
        return t["x"].double() @ _deq(t["w"]).T.contiguous()
    if op == "mlp":
        x = t["x"].double()
        g, u = x @ _deq(t["gate"]).T.contiguous(), x @ _deq(t["up"]).T.contiguous()
        return (g * torch.sigmoid(g) * u) @ _deq(t["down"]).T.contiguous()
    if op == "matmul":
        a, b = t["a"].double(), t["b"].double()
        return (a.T.contiguous() if case["kind"] == "atb" else a) @ (b.T.contiguous() if case["kind"] == "abt" else b)
    if op == "dx":
        return t["dy"].double() @ _deq(t["w"])
    if op == "lora":
        w, x, a, b, dy = _deq(t["w"]), t["x"].double(), t["a"].double(), t["b"].double(), t["dy"].double()
        xa, dxa = x @ a, dy @ b.T.contiguous()
        return {"y": x @ w.T.contiguous() + xa @ b, "xa": xa, "db": xa.T.contiguous() @ dy, "dxa": dxa,
                "da": x.T.contiguous() @ dxa, "dx": dy @ w, "dx_adapter": dxa @ a.T.contiguous()}
    return _exact_generation(case, t)


def _exact_generation(case, t):
    """The model's arithmetic in 64 bits with a KV cache: logits of the last
    step, on the tokens it picks greedily itself."""
    cfg = _config(case)
    hd, nh, nkv = cfg.head_dim, cfg.n_heads, cfg.n_kv_heads
    names = list(cfg.linear_shapes())
    layers = [{**{n: _deq(w[n]).T.contiguous() for n in names}, "an": w["attn_norm"].double(),
               "mn": w["mlp_norm"].double()} for w in t["layers"]]
    head, embed, final = _deq(t["lm_head"]).T.contiguous(), t["embed"], t["final_norm"].double()
    cache = [[None, None] for _ in layers]
    freq = cfg.rope_theta ** (-2.0 * torch.arange(hd // 2, device="cuda", dtype=torch.float64) / hd)

    def norm(x, w):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + cfg.norm_eps) * w

    def rope(x, pos):
        ang = pos.double()[:, None] * freq[None, :]
        c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
        a, b = x[..., : hd // 2], x[..., hd // 2:]
        return torch.cat([a * c - b * s, a * s + b * c], -1)

    def forward(ids, first):
        T = ids.numel()
        pos = torch.arange(first, first + T, device="cuda")
        x = embed[ids].double()
        for L, kv in zip(layers, cache):
            xn = norm(x, L["an"])
            q = rope((xn @ L["q"]).view(T, nh, hd), pos)
            k, v = rope((xn @ L["k"]).view(T, nkv, hd), pos), (xn @ L["v"]).view(T, nkv, hd)
            if kv[0] is not None:
                k, v = torch.cat([kv[0], k]), torch.cat([kv[1], v])
            kv[0], kv[1] = k, v
            mask = torch.arange(first + T, device="cuda")[None, :] > pos[:, None]
            out = torch.empty((T, nh, hd), dtype=torch.float64, device="cuda")
            for h in range(nh):
                j = h // (nh // nkv)
                sc = (q[:, h].contiguous() @ k[:, j].T.contiguous()) / math.sqrt(hd)
                out[:, h] = torch.softmax(sc.masked_fill(mask, -math.inf), 1) @ v[:, j].contiguous()
            x = x + out.reshape(T, nh * hd) @ L["o"]
            xn = norm(x, L["mn"])
            g = xn @ L["gate"]
            x = x + (g * torch.sigmoid(g) * (xn @ L["up"])) @ L["down"]
        return (norm(x[-1:], final) @ head)[0]

    ids, n = t["tokens"].long(), case["prompt"]
    logits = forward(ids, 0)
    for i in range(case["steps"]):
        logits = forward(logits.argmax()[None], n + i)
    return {"logits": logits, "tokens": None}
