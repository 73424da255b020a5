"""Performance cases of the backend: the calls a serving program makes, over the sizes it makes them at.

Each kind below is one part of running the model shapes this repository configures (GPT-2 small in fp32, TinyLlama-1.1B
and a Gemma-style layer in bf16, a 128-expert MoE block), through `sandyrt_amd.ops`, `HipDevice` and the decoders:

  fused_groups        residual add + RMSNorm, RoPE of q and k, SiLU gate: one token row up to a 4096-token prompt
  prefill_attention   causal attention of a prompt or prompt chunk, bf16, dense K/V or the engine's page list,
                      full or sliding window
  projection          one weight matrix applied to a prompt's rows, bf16
  gpt2                the whole GPT-2 prompt pass (or some of its layers) in fp32, logits out
  moe_block           router softmax + top-k, permute, expert GEMMs, SwiGLU, weighted combine
  paged_decode        decode attention over paged K/V with mixed context lengths, bf16
  decode_step         a whole TinyLlama step from one captured graph, given tokens in, logits out
"""
from __future__ import annotations

import math

import torch

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64

# TinyLlama-1.1B
HIDDEN, HEADS, KV_HEADS, HEAD_DIM, FFN, VOCAB, LAYERS = 2048, 32, 4, 64, 5632, 32000, 22
# GPT-2 small
G_HIDDEN, G_HEADS, G_DIM, G_FFN, G_VOCAB, G_POSITIONS, G_LAYERS = 768, 12, 64, 3072, 50257, 1024, 12
# MoE block
M_EXPERTS, M_TOP, M_HIDDEN, M_WIDTH = 128, 8, 2816, 704
PAGE = 16
EPS = 1e-5


def listed():
    return [
        # one decode row's element-wise chain: launches and latency are all there is
        {"name": "fused_groups_row", "kind": "fused_groups", "tokens": 1, "past": 777},
        # the same groups over a long prompt: memory streams
        {"name": "fused_groups_4096", "kind": "fused_groups", "tokens": 4096, "past": 0},
        # the attention of a 2048-token prompt chunk (the engine's default chunk length)
        {"name": "prefill_attention_2048", "kind": "prefill_attention", "batch": 1, "heads": HEADS, "kv_heads": KV_HEADS,
         "dim": HEAD_DIM, "tokens": 2048, "past": 0, "window": 0, "paged": False},
        # a later, ragged chunk of a Gemma-style sliding-window layer, K/V read from the engine's pages
        {"name": "prefill_attention_window", "kind": "prefill_attention", "batch": 1, "heads": 8, "kv_heads": 2,
         "dim": 256, "tokens": 777, "past": 1500, "window": 1024, "paged": True},
        # gate and up projection of a prompt chunk: compute-bound
        {"name": "projection_2048", "kind": "projection", "rows": 2048, "cols": 2 * FFN, "depth": HIDDEN},
        # down projection of a short ragged prompt: few tiles, long contraction
        {"name": "projection_ragged", "kind": "projection", "rows": 333, "cols": HIDDEN, "depth": FFN},
        # the GPT-2 prompt of the greedy benchmark
        {"name": "gpt2_prompt_64", "kind": "gpt2", "tokens": 64, "layers": G_LAYERS},
        # two blocks and the head of a prompt that nearly fills GPT-2's positions
        {"name": "gpt2_blocks_1000", "kind": "gpt2", "tokens": 1000, "layers": 2},
        # the MoE block at a batched step's token count, and at a few decoded tokens
        {"name": "moe_block_512", "kind": "moe_block", "tokens": 512},
        {"name": "moe_block_5", "kind": "moe_block", "tokens": 5},
        # batched decode attention of mixed contexts
        {"name": "paged_decode_32", "kind": "paged_decode", "batch": 32, "heads": HEADS, "kv_heads": KV_HEADS,
         "dim": HEAD_DIM, "ctx_low": 512, "ctx_high": 4096, "window": 0},
        # one whole step of a batch
        {"name": "decode_step_16", "kind": "decode_step", "batch": 16, "ctx_low": 256, "ctx_high": 2048},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["fused_groups", "prefill_attention", "prefill_attention", "projection", "projection", "gpt2",
                       "moe_block", "paged_decode", "decode_step"])
    if kind == "fused_groups":
        return {"kind": kind, "tokens": _log_int(rng, 1, 4096), "past": rng.randrange(0, 2000)}
    if kind == "prefill_attention":
        heads, kv_heads, dim = rng.choice([(HEADS, KV_HEADS, HEAD_DIM), (8, 2, 256), (16, 2, 128)])
        batch = rng.choice([1, 1, 2])
        return {"kind": kind, "batch": batch, "heads": heads, "kv_heads": kv_heads, "dim": dim,
                "tokens": _log_int(rng, 16, 2000 // batch // (2 if dim == 256 else 1)),
                "past": rng.choice([0, rng.randrange(1, 1500)]), "window": rng.choice([0, 0, 512, 1024]),
                "paged": rng.random() < 0.5}
    if kind == "projection":
        cols, depth = rng.choice([((HEADS + 2 * KV_HEADS) * HEAD_DIM, HIDDEN), (HIDDEN, HIDDEN), (2 * FFN, HIDDEN),
                                  (HIDDEN, FFN), (VOCAB, HIDDEN), (2560, 10240)])
        return {"kind": kind, "rows": _log_int(rng, 1, 1024 if cols == VOCAB else 2040), "cols": cols, "depth": depth}
    if kind == "gpt2":
        tokens = _log_int(rng, 5, 1000)
        return {"kind": kind, "tokens": tokens, "layers": rng.randrange(1, 3) if tokens > 100 else rng.randrange(1, 12)}
    if kind == "moe_block":
        return {"kind": kind, "tokens": _log_int(rng, 1, 2048)}
    if kind == "paged_decode":
        heads, kv_heads, dim = rng.choice([(HEADS, KV_HEADS, HEAD_DIM), (8, 2, 256), (16, 2, 128)])
        low = _log_int(rng, 16, 1500)
        return {"kind": kind, "batch": _log_int(rng, 1, 64), "heads": heads, "kv_heads": kv_heads, "dim": dim,
                "ctx_low": low, "ctx_high": low + _log_int(rng, 16, 4000), "window": rng.choice([0, 0, 1024])}
    low = _log_int(rng, 16, 1000)
    return {"kind": kind, "batch": _log_int(rng, 1, 32), "ctx_low": low, "ctx_high": low + _log_int(rng, 16, 1500)}


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0, mean=0.0, dtype=BF16):
    t = torch.randn(*shape, generator=g, device="cuda")
    if std != 1.0:
        t *= std
    if mean:
        t += mean
    return t.to(dtype)


def _contexts(case, seed):
    g = torch.Generator()
    g.manual_seed(seed)
    return torch.randint(case["ctx_low"], case["ctx_high"] + 1, (case["batch"],), generator=g)


def _inputs(case, seed):
    """The tensors of a case, from the seed alone (shared by prepare and exact)."""
    g, kind = _generator(seed), case["kind"]
    if kind == "fused_groups":
        n = case["tokens"]
        return {"x": _randn(g, n, HIDDEN), "h": _randn(g, n, HIDDEN), "w": _randn(g, HIDDEN, std=0.1, mean=1.0),
                "q": _randn(g, 1, HEADS, n, HEAD_DIM), "k": _randn(g, 1, KV_HEADS, n, HEAD_DIM),
                "gate": _randn(g, n, FFN), "up": _randn(g, n, FFN),
                "pos": torch.full((1,), case["past"], dtype=torch.int64, device="cuda")}
    if kind == "prefill_attention":
        b, n, d = case["batch"], case["tokens"], case["dim"]
        keys = case["past"] + n
        s = {"q": _randn(g, b, case["heads"], n, d),
             "pos": torch.full((b,), case["past"], dtype=torch.int64, device="cuda")}
        if case["paged"]:  # [pages, batch * kv heads, page rows, dim], one page list for the batch
            pages = -(-keys // PAGE)
            s["k"] = _randn(g, pages, b * case["kv_heads"], PAGE, d)
            s["v"] = _randn(g, pages, b * case["kv_heads"], PAGE, d)
            s["order"] = torch.randperm(pages, generator=g, device="cuda")
        else:
            s["k"] = _randn(g, b, case["kv_heads"], keys, d)
            s["v"] = _randn(g, b, case["kv_heads"], keys, d)
        return s
    if kind == "projection":
        return {"x": _randn(g, case["rows"], case["depth"]), "w": _randn(g, case["cols"], case["depth"], std=0.02)}
    if kind == "gpt2":
        w = {"wte": _randn(g, G_VOCAB, G_HIDDEN, std=0.02, dtype=F32),
             "wpe": _randn(g, G_POSITIONS, G_HIDDEN, std=0.02, dtype=F32)}
        for i in range(case["layers"]):
            for n, o, k in (("q", G_HIDDEN, G_HIDDEN), ("k", G_HIDDEN, G_HIDDEN), ("v", G_HIDDEN, G_HIDDEN),
                            ("proj", G_HIDDEN, G_HIDDEN), ("fc", G_FFN, G_HIDDEN), ("out", G_HIDDEN, G_FFN)):
                w[f"{i}.{n}.w"] = _randn(g, o, k, std=0.02, dtype=F32)
                w[f"{i}.{n}.b"] = _randn(g, o, std=0.02, dtype=F32)
            for n in ("ln1", "ln2"):
                w[f"{i}.{n}.w"] = _randn(g, G_HIDDEN, std=0.02, mean=1.0, dtype=F32)
                w[f"{i}.{n}.b"] = _randn(g, G_HIDDEN, std=0.02, dtype=F32)
        w["lnf.w"], w["lnf.b"] = _randn(g, G_HIDDEN, std=0.02, mean=1.0, dtype=F32), _randn(g, G_HIDDEN, std=0.02, dtype=F32)
        w["ids"] = torch.randint(0, G_VOCAB, (1, case["tokens"]), generator=g, device="cuda")
        return w
    if kind == "moe_block":
        n = case["tokens"]
        return {"x": _randn(g, n, M_HIDDEN), "router": _randn(g, n, M_EXPERTS, dtype=F32),
                "gate": _randn(g, M_EXPERTS, M_WIDTH, M_HIDDEN, std=0.02),
                "up": _randn(g, M_EXPERTS, M_WIDTH, M_HIDDEN, std=0.02),
                "down": _randn(g, M_EXPERTS, M_HIDDEN, M_WIDTH, std=0.02)}
    if kind == "paged_decode":
        b, d, hk = case["batch"], case["dim"], case["kv_heads"]
        ctx = _contexts(case, seed)
        blocks = (ctx + PAGE - 1) // PAGE
        pool = int(blocks.sum())
        s = {"q": _randn(g, b, case["heads"], 1, d), "k": _randn(g, pool, hk, PAGE, d), "v": _randn(g, pool, hk, PAGE, d),
             "ctx": ctx, "pos": (ctx - 1).cuda()}
        order = torch.randperm(pool, generator=g, device="cuda").int().cpu()
        table = torch.zeros(b, int(blocks.max()), dtype=torch.int32)
        at = 0
        for i, m in enumerate(blocks.tolist()):
            table[i, :m] = order[at:at + m]
            at += m
        s["table"] = table.cuda()
        return s
    ctx = _contexts(case, seed)  # decode_step
    s = {"ctx": ctx, "token": torch.randint(0, VOCAB, (case["batch"],), generator=g, device="cuda")}
    rows = int(ctx.max())  # every sequence's context is the head of one set of rows a layer
    s["k"] = [_randn(g, 1, KV_HEADS, rows, HEAD_DIM) for _ in range(LAYERS)]
    s["v"] = [_randn(g, 1, KV_HEADS, rows, HEAD_DIM) for _ in range(LAYERS)]
    return s


_device = None


def _hip_device():
    """The program's one device: its stream orders the steps of every decoder."""
    global _device
    if _device is None:
        from sandyrt_amd.device import HipDevice
        _device = HipDevice(0)
    return _device


class _Decoder:
    """A decoder with its contexts cached, its step captured, and room for `room` more tokens a sequence."""

    room = 1024

    def __init__(self, case, seed):
        from sandyrt_amd.decode import DecodeConfig, TinyLlamaDecoder, random_weights

        self.inputs = _inputs(case, seed)
        self.tokens = self.inputs["token"].view(-1, 1)
        self.cfg = DecodeConfig(page_size=PAGE, max_context=int(self.inputs["ctx"].max()) + self.room + 2)
        self.weights = random_weights(self.cfg, seed)
        self.dev = _hip_device()
        self.dec = TinyLlamaDecoder(self.dev, self.cfg, self.weights, batch=case["batch"])
        torch.cuda.synchronize()
        self._fill()
        self.dec.step()  # generated kernels and workspaces exist before the capture
        self.dev.synchronize()
        self.dec.capture()
        self.rewind()

    def _fill(self):
        for b, n in enumerate(self.inputs["ctx"].tolist()):
            self.dec.prefill_cache([t[:, :, :n].contiguous() for t in self.inputs["k"]],
                                   [t[:, :, :n].contiguous() for t in self.inputs["v"]], seq=b)
        self.dec.set_token(self.inputs["token"].tolist())
        self.steps = 0

    def rewind(self):
        """The sequences end and new ones with the same contexts take their slots (the captured step stays)."""
        self.dev.synchronize()
        pages = (self.cfg.max_context + PAGE - 1) // PAGE
        for pools, seqs in ((self.dec.k_pools, self.dec.k_seq), (self.dec.v_pools, self.dec.v_seq)):
            for layer, ids in enumerate(seqs):
                for t in ids:
                    self.dev.dealloc_paged(t)
                new = [self.dev.alloc_paged(pools[layer]) for _ in ids]
                ids[:] = sorted(new, key=lambda t: self.dev.paged_meta(t).slot)  # sequence b in slot b
                for t in ids:
                    self.dev.reserve_paged(t, pages)
        self._fill()

    def __del__(self):
        try:
            torch.cuda.synchronize()
            self.dec.close()
            for pool, ids in zip(self.dec.k_pools + self.dec.v_pools, self.dec.k_seq + self.dec.v_seq):
                for t in ids:
                    self.dev.dealloc_paged(t)
                self.dev.destroy_paged_pool(pool)
        except Exception:  # the interpreter is going down
            pass


def prepare(case, seed):
    from sandyrt_amd import ops

    kind = case["kind"]
    if kind == "decode_step":
        return {"kind": kind, "decoder": _Decoder(case, seed)}
    s = _inputs(case, seed)
    s["kind"], s["case"] = kind, case
    if kind in ("fused_groups", "moe_block"):
        s["silu"] = ops.silu_mul_nodes()
    if kind == "moe_block":
        s["copy"] = [ops.ScalarNode(0, ops.LOAD, 0)]
    if kind == "gpt2":
        s["gelu"], s["add"], s["copy"] = ops.gelu_nodes(), ops.residual_add_nodes(), [ops.ScalarNode(0, ops.LOAD, 0)]
        s["pos"] = torch.arange(case["tokens"], dtype=torch.int64, device="cuda").view(1, -1)
        s["offsets"] = torch.zeros(1, dtype=torch.int64, device="cuda")
    if kind == "paged_decode":
        s["k_cache"], s["v_cache"] = ops.PagedCache(s["k"]), ops.PagedCache(s["v"])
    if kind == "prefill_attention" and case["paged"]:
        dims = [case["batch"], case["kv_heads"], case["past"] + case["tokens"], case["dim"]]
        for name in ("k", "v"):
            pool = s[name]
            at = pool.data_ptr() + s["order"] * (pool.stride(0) * pool.element_size())
            s[name + "_view"] = ops.PagedView(at, dims, PAGE, BF16)
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    from sandyrt_amd import ops

    kind = s["kind"]
    if kind == "fused_groups":
        total, normed = ops.add_rms_norm(s["x"], s["h"], s["w"], EPS)
        q, k = ops.rope_pair(s["q"], s["k"], 1e4, split_half=True, position_ids=s["pos"])
        nodes, result = s["silu"]
        return {"sum": total, "norm": normed, "q": q, "k": k, "act": ops.elementwise(nodes, result, [s["gate"], s["up"]])}
    if kind == "prefill_attention":
        case = s["case"]
        if case["paged"]:
            return ops.attention_paged_view(s["q"], s["k_view"], s["v_view"], s["pos"], window=case["window"])
        return ops.attention(s["q"], s["k"], s["v"], s["pos"], window=case["window"])
    if kind == "projection":
        return ops.matmul(s["x"], s["w"], transpose_rhs=True)
    if kind == "gpt2":
        return _gpt2(ops, s)
    if kind == "moe_block":
        n = s["case"]["tokens"]
        weights, ids = ops.topk(ops.softmax(s["router"]), M_TOP)
        weights = ops.elementwise(s["copy"], 0, [weights], out_dtype=BF16)
        packed, packed_w, tokens, offsets = ops.moe_gather(s["x"], ids, weights, M_EXPERTS)
        gate = ops.moe_matmul(packed, offsets, s["gate"])
        up = ops.moe_matmul(packed, offsets, s["up"])
        nodes, result = s["silu"]
        down = ops.moe_matmul(ops.elementwise(nodes, result, [gate, up]), offsets, s["down"])
        return {"out": ops.moe_scatter_sum(down, packed_w, tokens, n), "ids": ids}
    if kind == "paged_decode":
        return ops.paged_attention(s["q"], s["k_cache"], s["v_cache"], s["table"], s["pos"], window=s["case"]["window"])
    d = s["decoder"]
    if d.steps == d.room:
        d.rewind()
    with torch.cuda.stream(d.dev.torch_stream()):  # the next tokens are given, as in scoring a text
        d.dec.token.copy_(d.tokens)
    d.dec.replay()
    d.steps += 1
    return d.dec.logits


def _gpt2(ops, s):
    """The prompt pass of sandyrt_amd.gpt2 (its K/V appends left out): the last row's logits."""
    case = s["case"]
    n = case["tokens"]
    add, add_res = s["add"]
    gelu, gelu_res = s["gelu"]

    def heads(t):
        return t.view(n, G_HEADS, G_DIM).permute(1, 0, 2).unsqueeze(0)

    x = ops.elementwise(add, add_res, [ops.embedding(s["ids"], s["wte"]), ops.embedding(s["pos"], s["wpe"])])
    x = x.view(n, G_HIDDEN)
    for i in range(case["layers"]):
        h = ops.layer_norm(x, s[f"{i}.ln1.w"], s[f"{i}.ln1.b"], EPS)
        q, k, v = (ops.linear(h, s[f"{i}.{p}.w"], s[f"{i}.{p}.b"]) for p in "qkv")
        kh, vh = (ops.elementwise(s["copy"], 0, [heads(t)]) for t in (k, v))
        ctx = torch.empty(n, G_HIDDEN, dtype=F32, device="cuda")
        ops.attention(heads(q), kh, vh, s["offsets"], out=heads(ctx))
        x = ops.elementwise(add, add_res, [x, ops.linear(ctx, s[f"{i}.proj.w"], s[f"{i}.proj.b"])])
        h = ops.layer_norm(x, s[f"{i}.ln2.w"], s[f"{i}.ln2.b"], EPS)
        f = ops.elementwise(gelu, gelu_res, [ops.linear(h, s[f"{i}.fc.w"], s[f"{i}.fc.b"])])
        x = ops.elementwise(add, add_res, [x, ops.linear(f, s[f"{i}.out.w"], s[f"{i}.out.b"])])
    h = ops.layer_norm(x[n - 1:n], s["lnf.w"], s["lnf.b"], EPS)
    return {"x": x, "logits": ops.matmul(h, s["wte"], transpose_rhs=True)}


# ------------------------------------------------------------------ what a pass cannot do without
def _pairs(tokens, past, window):
    """Causal (query, key) pairs of one head."""
    total = 0
    for i in range(tokens):
        p = past + i + 1
        total += min(p, window) if window else p
    return total


def work(case):
    kind = case["kind"]
    if kind == "fused_groups":
        n = case["tokens"]
        kv = (HEADS + KV_HEADS) * HEAD_DIM
        return {"bytes": 2 * n * (4 * HIDDEN + 2 * kv + 3 * FFN) + 2 * HIDDEN, "flops": n * (6 * HIDDEN + 4 * kv + 6 * FFN)}
    if kind == "prefill_attention":
        b, n, d = case["batch"], case["tokens"], case["dim"]
        keys = case["past"] + n
        if case["window"]:
            keys = min(keys, n + case["window"] - 1)
        return {"bytes": 2 * b * d * (2 * case["heads"] * n + 2 * case["kv_heads"] * keys),
                "flops": 4 * b * case["heads"] * d * _pairs(n, case["past"], case["window"])}
    if kind == "projection":
        m, n, k = case["rows"], case["cols"], case["depth"]
        return {"bytes": 2 * (m * k + n * k + m * n), "flops": 2 * m * n * k}
    if kind == "gpt2":
        n, layers = case["tokens"], case["layers"]
        per_layer = 4 * G_HIDDEN * G_HIDDEN + 2 * G_HIDDEN * G_FFN
        return {"bytes": 4 * (layers * per_layer + G_VOCAB * G_HIDDEN + 4 * n * G_HIDDEN),
                "flops": 2 * n * layers * per_layer + 4 * layers * G_HIDDEN * _pairs(n, 0, 0) + 2 * G_VOCAB * G_HIDDEN}
    if kind == "moe_block":
        n = case["tokens"]
        experts = M_EXPERTS * (1 - (1 - M_TOP / M_EXPERTS) ** n)  # experts that get a row, for even routing
        return {"bytes": 2 * (experts * 3 * M_HIDDEN * M_WIDTH + 2 * n * M_HIDDEN) + 4 * n * M_EXPERTS,
                "flops": 6 * n * M_TOP * M_HIDDEN * M_WIDTH}
    mean = (case["ctx_low"] + case["ctx_high"]) / 2
    if kind == "paged_decode":
        keys = min(mean, case["window"]) if case["window"] else mean
        b = case["batch"]
        return {"bytes": 2 * b * case["dim"] * (2 * keys * case["kv_heads"] + 2 * case["heads"]),
                "flops": 4 * b * case["heads"] * case["dim"] * keys}
    b = case["batch"]
    weights = LAYERS * ((HEADS + 2 * KV_HEADS) * HEAD_DIM * HIDDEN + HIDDEN * HIDDEN + 3 * FFN * HIDDEN) + VOCAB * HIDDEN
    return {"bytes": 2 * (weights + b * LAYERS * mean * 2 * KV_HEADS * HEAD_DIM + b * VOCAB),
            "flops": 2 * b * (weights + LAYERS * 2 * HEADS * HEAD_DIM * mean)}


def tolerance(case):
    kind = case["kind"]
    if kind == "gpt2":
        return {"rel": 1e-5, "max": 1e-4}  # 32-bit sums through the layers
    if kind == "moe_block":
        return {"rel": 4e-3, "max": 6e-2, "differ": 1e-4}  # roundings of gate, up and down meet in the combine
    if kind == "decode_step":
        # bf16 roundings through 22 layers: other K splits of the projections give 0.019 and 0.11
        return {"rel": 3e-2, "max": 4e-1}
    # one bf16 rounding of a 32-bit sum: other orders of the sum give 6e-5 and one last place of a value
    return {"rel": 4e-4, "max": 3.2e-2}


# ------------------------------------------------------------------ the same in 64 bits
def _exact_attention(q, k, v, past, window, scale):
    """q [H, T, D] against k, v [H, K, D] in float64, a head at a time."""
    n, keys = q.shape[1], k.shape[1]
    at = past + torch.arange(n, device=q.device).view(-1, 1)
    key = torch.arange(keys, device=q.device).view(1, -1)
    seen = key <= at
    if window:
        seen &= key >= at + 1 - window
    out = torch.empty_like(q, dtype=F64)
    group = q.shape[0] // k.shape[0]
    for h in range(q.shape[0]):
        scores = (q[h].to(F64) @ k[h // group].to(F64).t().contiguous()) * scale
        out[h] = torch.softmax(scores.masked_fill(~seen, -math.inf), -1) @ v[h // group].to(F64)
    return out


def _exact_rope(x, pos, split_dim):
    """Split-half RoPE, theta 1e4; pos broadcasts against x's vectors."""
    half = split_dim // 2
    i = torch.arange(half, dtype=F64, device=x.device)
    angle = pos.to(F64).unsqueeze(-1) / (1e4 ** (2 * i / split_dim))
    a, b = x[..., :half].to(F64), x[..., half:].to(F64)
    return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1)


def _exact_rms(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.to(F64)


def _exact_norm(x, w, b):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), w.to(F64), b.to(F64), EPS)


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode_step":
        return _exact_step(case, seed)
    s = _inputs(case, seed)
    silu = torch.nn.functional.silu
    if kind == "fused_groups":
        total = s["x"].to(F64) + s["h"].to(F64)
        pos = s["pos"] + torch.arange(case["tokens"], device="cuda")
        # the norm reads the rounded sum, which is itself an output
        return {"sum": total, "norm": _exact_rms(total.to(BF16).to(F64), s["w"]), "q": _exact_rope(s["q"], pos, HEAD_DIM),
                "k": _exact_rope(s["k"], pos, HEAD_DIM), "act": silu(s["gate"].to(F64)) * s["up"].to(F64)}
    if kind == "prefill_attention":
        b, hk, keys = case["batch"], case["kv_heads"], case["past"] + case["tokens"]
        k, v = s["k"], s["v"]
        if case["paged"]:
            k, v = (t[s["order"]].transpose(0, 1).reshape(b, hk, -1, case["dim"])[:, :, :keys] for t in (k, v))
        return torch.stack([_exact_attention(s["q"][i], k[i], v[i], case["past"], case["window"], case["dim"] ** -0.5)
                            for i in range(b)])
    if kind == "projection":
        return s["x"].to(F64) @ s["w"].to(F64).t().contiguous()
    if kind == "gpt2":
        return _exact_gpt2(case, s)
    if kind == "moe_block":
        weights, ids = torch.topk(torch.softmax(s["router"].to(F64), -1), M_TOP)
        out = torch.zeros(case["tokens"], M_HIDDEN, dtype=F64, device="cuda")
        x = s["x"].to(F64)
        for e in range(M_EXPERTS):
            row, slot = torch.nonzero(ids == e, as_tuple=True)
            if row.numel():
                rows = x[row]
                act = silu(rows @ s["gate"][e].to(F64).t().contiguous()) * (rows @ s["up"][e].to(F64).t().contiguous())
                out.index_add_(0, row, act @ s["down"][e].to(F64).t().contiguous() * weights[row, slot, None])
        return {"out": out, "ids": None}
    out = torch.empty(case["batch"], case["heads"], 1, case["dim"], dtype=F64, device="cuda")
    for b, n in enumerate(s["ctx"].tolist()):
        blocks = s["table"][b, :-(-n // PAGE)].long()
        k, v = (s[t][blocks].transpose(0, 1).reshape(case["kv_heads"], -1, case["dim"])[:, :n] for t in ("k", "v"))
        out[b] = _exact_attention(s["q"][b], k, v, n - 1, case["window"], case["dim"] ** -0.5)
    return out


def _exact_gpt2(case, s):
    n = case["tokens"]

    def linear(t, name):
        return t @ s[name + ".w"].to(F64).t().contiguous() + s[name + ".b"].to(F64)

    def heads(t):
        return t.view(n, G_HEADS, G_DIM).transpose(0, 1).contiguous()

    x = s["wte"][s["ids"][0]].to(F64) + s["wpe"][:n].to(F64)
    for i in range(case["layers"]):
        h = _exact_norm(x, s[f"{i}.ln1.w"], s[f"{i}.ln1.b"])
        q, k, v = (heads(linear(h, f"{i}.{p}")) for p in "qkv")
        ctx = _exact_attention(q, k, v, 0, 0, G_DIM ** -0.5).transpose(0, 1).reshape(n, G_HIDDEN)
        x = x + linear(ctx, f"{i}.proj")
        f = linear(_exact_norm(x, s[f"{i}.ln2.w"], s[f"{i}.ln2.b"]), f"{i}.fc")
        x = x + linear(torch.nn.functional.gelu(f, approximate="tanh"), f"{i}.out")
    h = _exact_norm(x[n - 1:], s["lnf.w"], s["lnf.b"])
    return {"x": x, "logits": h @ s["wte"].to(F64).t().contiguous()}


def _exact_step(case, seed):
    from sandyrt_amd.decode import DecodeConfig, random_weights  # the weights alone

    s, w = _inputs(case, seed), random_weights(DecodeConfig(), seed)
    b, q_cols, kv_cols = case["batch"], HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
    pos = s["ctx"].cuda()

    def times(t, name, rows=slice(None)):
        return t @ w[name][rows].to(F64).t().contiguous()

    x = w["embed"][s["token"]].to(F64)
    for i in range(LAYERS):
        h = _exact_rms(x, w[f"{i}.in_norm"])
        qkv = times(h, f"{i}.qkv")
        q = _exact_rope(qkv[:, :q_cols].view(b, HEADS, HEAD_DIM), pos.view(b, 1), HEAD_DIM)
        k = _exact_rope(qkv[:, q_cols:q_cols + kv_cols].view(b, KV_HEADS, HEAD_DIM), pos.view(b, 1), HEAD_DIM)
        v = qkv[:, q_cols + kv_cols:].view(b, KV_HEADS, HEAD_DIM)
        ctx = torch.empty(b, q_cols, dtype=F64, device="cuda")
        group = HEADS // KV_HEADS
        for j, n in enumerate(s["ctx"].tolist()):
            keys = torch.cat([s["k"][i][0, :, :n].to(F64), k[j].unsqueeze(1)], 1)
            values = torch.cat([s["v"][i][0, :, :n].to(F64), v[j].unsqueeze(1)], 1)
            scores = torch.bmm(q[j].view(KV_HEADS, group, HEAD_DIM), keys.transpose(1, 2).contiguous()) * HEAD_DIM ** -0.5
            ctx[j] = torch.bmm(torch.softmax(scores, -1), values).reshape(q_cols)
        x = x + times(ctx, f"{i}.o")
        h = _exact_rms(x, w[f"{i}.post_norm"])
        act = torch.nn.functional.silu(times(h, f"{i}.gate_up", slice(0, FFN))) * times(h, f"{i}.gate_up", slice(FFN, None))
        x = x + times(act, f"{i}.down")
    return times(_exact_rms(x, w["norm"]), "lm_head")
