"""Performance cases: the work a user of this package has it do, through its public entry points.

Kinds (a case's ``"kind"``; its other entries are that kind's sizes and options):

``gemv``      one projection of a decode step over packed weights (``ops.w4_gemv`` / ``w8_gemv``): RMSNorm
              prologue, bias or residual epilogue, or the paired gate/up form
``head``      the end of a decode step: final norm, language-model head, greedy argmax (logits and token)
``decode_attention``   one ring step of static-cache attention: RoPE, cache write, one query over the window
``attention`` the causal, left-padded prompt attention of a prefill
``qkv`` / ``mlp`` / ``out``   the prefill projections with the epilogues a layer runs them with
``pack``      quantizing one weight matrix, as compiling a checkpoint does for each of its projections
``block``     a transformer block compiled by ``compile_module`` and called
``prefill_decode`` / ``generate``   whole calls of a compiled decoder

Sizes are those of the two decoder shapes the benchmark runs (896-wide with 24 layers, 4096-wide) and generic
ones between and beyond them; weights N(0, 0.03), activations N(0, 1), norms 1 + N(0, 0.1), as the
benchmark's random-init states have them.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

BF16 = torch.bfloat16


# ----------------------------------------------------------------------------- the listed cases
def listed():
    return [
        # one q/k/v projection of the 896-wide decoder's decode step: the smallest call, latency and launch
        dict(name="gemv_qkv_896", kind="gemv", bits=4, k=896, n=1152, group=64, norm=True, epilogue="bias"),
        # the paired gate/up projection of a decode step at a width between and beyond the benchmarked ones
        dict(name="gemv_gate_up_5120", kind="gemv", bits=4, k=5120, n=13824, group=64, norm=True, epilogue="paired"),
        # the int8 decoder's last launches of every token: a 151936-row head and its argmax
        dict(name="head_w8_896", kind="head", bits=8, k=896, n=151936, group=64),
        # one layer's attention late in a long generation of the 4096-wide decoder
        dict(name="decode_attention_8192", kind="decode_attention", heads=32, kv_heads=8, dim=128, capacity=8192,
             valid=8000, offset=4321),
        # a 1900-token prompt in the 2048 bucket
        dict(name="attention_2048", kind="attention", heads=32, kv_heads=8, dim=128, tokens=2048, start=148,
             mask=False),
        # a 1024-token prompt on the 896-wide decoder: q/k/v with bias, RoPE and the cache fill
        dict(name="qkv_896_1024", kind="qkv", bits=4, k=896, heads=14, kv_heads=2, dim=64, group=64, tokens=1024,
             extra=64, bias=True),
        # the largest prefill projection pair (2048 tokens through the 4096-wide decoder's gate and up)
        dict(name="mlp_4096_2048", kind="mlp", bits=4, k=4096, n=14336, group=64, tokens=2048),
        # an odd prompt length on the int8 decoder: the down projection, the residual and the next norm
        dict(name="out_w8_14336_333", kind="out", bits=8, k=14336, n=4096, group=64, tokens=333),
        # packing one projection of the 4096-wide decoder from its bf16 checkpoint
        dict(name="pack_w4_14336", kind="pack", bits=4, rows=14336, cols=4096, group=64, f32=False),
        # a bf16 transformer block through the graph compiler, 512 tokens
        dict(name="block_bf16_896_512", kind="block", dtype="bf16", hidden=896, heads=14, kv_heads=2, inter=4864,
             tokens=512),
        # a 100-token prompt in the 128 bucket, then one step of the functional decode plan
        dict(name="prefill_decode_896", kind="prefill_decode", bits=4, layers=24, hidden=896, inter=4864, heads=14,
             kv_heads=2, dim=64, vocab=151936, bucket=128, length=100, new=64),
        # the greedy loop: 128-token prompt, 32 tokens
        dict(name="generate_896", kind="generate", bits=4, layers=24, hidden=896, inter=4864, heads=14, kv_heads=2,
             dim=64, vocab=151936, bucket=128, length=128, new=32),
    ]


def _spread(rng, low, high, step=1):
    """A multiple of ``step`` in [low, high], spread over the logarithm."""

    value = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(value / step)) * step))


def draw(rng):
    kind = rng.choice(("gemv", "gemv", "head", "decode_attention", "attention", "qkv", "mlp", "out", "pack", "block",
                       "prefill_decode", "generate"))
    bits = rng.choice((4, 4, 8))
    group = rng.choice((64, 64, 64, 32, 128))
    if kind == "gemv":
        epilogue = rng.choice(("none", "bias", "residual", "paired"))
        return dict(kind=kind, bits=bits, k=_spread(rng, 512, 16384, max(64, group)), n=_spread(rng, 256, 16384, 16),
                    group=group, norm=epilogue in ("none", "bias", "paired"), epilogue=epilogue)
    if kind == "head":
        return dict(kind=kind, bits=bits, k=_spread(rng, 512, 5120, max(64, group)), n=_spread(rng, 8192, 151936, 2),
                    group=group)
    if kind in ("decode_attention", "attention", "qkv"):
        dim, kv = rng.choice((64, 128)), rng.choice((1, 2, 4, 8))
        heads = kv * rng.choice((1, 2, 4, 7))
        if kind == "decode_attention":
            capacity = _spread(rng, 64, 16384)
            return dict(kind=kind, heads=heads, kv_heads=kv, dim=dim, capacity=capacity,
                        valid=max(1, int(capacity * rng.uniform(0.3, 1.0))), offset=rng.randrange(capacity))
        tokens = _spread(rng, 16, 2048)
        if kind == "attention":
            return dict(kind=kind, heads=heads, kv_heads=kv, dim=dim, tokens=tokens,
                        start=rng.choice((0, rng.randrange(max(1, tokens // 2)))), mask=rng.random() < 0.2)
        return dict(kind=kind, bits=bits, k=_spread(rng, 512, 5120, max(64, group)), heads=heads, kv_heads=kv, dim=dim,
                    group=group, tokens=tokens, extra=rng.choice((0, 64, 200)), bias=rng.random() < 0.5)
    if kind == "mlp":
        return dict(kind=kind, bits=bits, k=_spread(rng, 512, 4096, max(64, group)), n=_spread(rng, 512, 14336, 16),
                    group=group, tokens=_spread(rng, 16, 2048))
    if kind == "out":
        return dict(kind=kind, bits=bits, k=_spread(rng, 512, 14336, max(64, group)), n=_spread(rng, 512, 4096, 16),
                    group=group, tokens=_spread(rng, 16, 2048))
    if kind == "pack":
        return dict(kind=kind, bits=bits, rows=_spread(rng, 64, 14336), cols=_spread(rng, 512, 8192, max(64, group)),
                    group=group, f32=rng.random() < 0.25)
    if kind == "block":
        kv = rng.choice((1, 2, 4))
        heads = kv * rng.choice((1, 2, 4))
        return dict(kind=kind, dtype=rng.choice(("bf16", "bf16", "f32")), hidden=64 * heads, heads=heads, kv_heads=kv,
                    inter=_spread(rng, 128, 4096, 8), tokens=_spread(rng, 4, 768))
    kv = rng.choice((1, 2, 4))
    heads = kv * rng.choice((2, 4, 7))
    bucket = _spread(rng, 16, 512)
    return dict(kind=kind, bits=bits, layers=rng.choice((2, 4, 8)), hidden=_spread(rng, 256, 1024, 128),
                inter=_spread(rng, 512, 4096, 128), heads=heads, kv_heads=kv, dim=64, vocab=_spread(rng, 2048, 65536, 16),
                bucket=bucket, length=max(1, bucket - rng.choice((0, bucket // 3))), new=rng.choice((8, 24)))


# ----------------------------------------------------------------------------- inputs
class _Draws:
    """Seeded device tensors, made in the order they are asked for."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=BF16):
        values = torch.randn(*shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return values.mul_(std).add_(mean).to(dtype)

    def norm(self, n):
        return self.normal(n, std=0.1, mean=1.0)

    def ids(self, n, vocab):
        return torch.randint(0, vocab, (1, n), generator=self.gen, device="cuda")

    def packed(self, n, k, group, bits):
        """A packed ``[n, k]`` weight: (words, scales)."""

        return _pack(self.normal(n, k, std=0.03), group, bits)


def _pack(weight, group, bits):
    """Symmetric group codes of a weight in int32 words, and bf16 scales (the packed format's own rule)."""

    n, k = weight.shape
    top = 7 if bits == 4 else 127
    words, scales = [], []
    for part in weight.split(max(1, (1 << 26) // k)):  # bounded temporaries
        w = part.float().view(part.shape[0], k // group, group)
        widest = w.abs().amax(-1, keepdim=True)
        scale = torch.where(widest > 0, widest, torch.ones_like(widest)) / top
        codes = torch.clamp(torch.round(w / scale), -top - 1, top).to(torch.int32).view(part.shape[0], -1, 32 // bits)
        word = torch.zeros(codes.shape[:2], dtype=torch.int32, device=weight.device)
        for i in range(32 // bits):
            word |= (codes[:, :, i] & ((1 << bits) - 1)) << (bits * i)
        words.append(word)
        scales.append(scale.view(part.shape[0], -1).to(BF16))
    return torch.cat(words).contiguous(), torch.cat(scales).contiguous()


def _dequantized(words, scales, bits, rounded):
    """The weight of a pack in 64 bits; ``rounded``: the products code * scale as bf16 holds them."""

    shifts = torch.arange(0, 32, bits, device=words.device, dtype=torch.int32)
    codes = (words[:, :, None] >> shifts) & ((1 << bits) - 1)
    codes = torch.where(codes >= 1 << (bits - 1), codes - (1 << bits), codes).view(words.shape[0], -1)
    values = codes.double() * scales.double().repeat_interleave(codes.shape[1] // scales.shape[1], dim=1)
    return values.to(BF16).double() if rounded else values


def _tables(rows, dim, theta=1e6):
    """bf16 cos / sin tables ``[rows, dim]``: f32 angles rounded to bf16 before cos and sin."""

    angles = torch.arange(rows, dtype=torch.float32)[:, None] / torch.pow(
        torch.tensor(theta), torch.arange(0, dim, 2, dtype=torch.float32)[None, :] / dim)
    angles = torch.cat((angles, angles), dim=-1).to(BF16)
    return angles.cos().cuda().contiguous(), angles.sin().cuda().contiguous()


def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), dim=-1) * sin


def _rms(x, weight, eps=1e-6):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * weight


class Block(torch.nn.Module):
    """A pre-norm transformer block with rotary grouped-query attention and a gated MLP."""

    def __init__(self, hidden, heads, kv_heads, inter):
        super().__init__()
        self.heads, self.kv_heads, self.dim = heads, kv_heads, hidden // heads
        width = self.dim * kv_heads
        self.q = torch.nn.Linear(hidden, hidden)
        self.k, self.v = torch.nn.Linear(hidden, width), torch.nn.Linear(hidden, width)
        self.o = torch.nn.Linear(hidden, hidden, bias=False)
        self.gate, self.up = torch.nn.Linear(hidden, inter, bias=False), torch.nn.Linear(hidden, inter, bias=False)
        self.down = torch.nn.Linear(inter, hidden, bias=False)
        self.norm1, self.norm2 = torch.nn.Parameter(torch.ones(hidden)), torch.nn.Parameter(torch.ones(hidden))

    @staticmethod
    def norm(x, weight):
        y = x.float()
        y = y * torch.rsqrt(y.pow(2).mean(-1, keepdim=True) + 1e-6)
        return weight * y.to(x.dtype)

    def forward(self, x, cos, sin):
        b, t, h = x.shape
        n = self.norm(x, self.norm1)
        q = _rotate(self.q(n).view(b, t, self.heads, self.dim).transpose(1, 2), cos, sin)
        k = _rotate(self.k(n).view(b, t, self.kv_heads, self.dim).transpose(1, 2), cos, sin)
        v = self.v(n).view(b, t, self.kv_heads, self.dim).transpose(1, 2)
        a = F.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=self.heads != self.kv_heads)
        x = x + self.o(a.transpose(1, 2).reshape(b, t, h))
        n = self.norm(x, self.norm2)
        return x + self.down(F.silu(self.gate(n)) * self.up(n))


def _block(case, draws):
    dtype = BF16 if case["dtype"] == "bf16" else torch.float32
    module = Block(case["hidden"], case["heads"], case["kv_heads"], case["inter"]).eval().requires_grad_(False)
    module = module.to(device="cuda", dtype=dtype)
    for name, parameter in module.named_parameters():
        one = name.startswith("norm")
        parameter.copy_(draws.normal(*parameter.shape, std=0.1 if one else 0.03, mean=float(one), dtype=dtype))
    x = draws.normal(1, case["tokens"], case["hidden"], dtype=dtype)
    cos, sin = (t.to(dtype) for t in _tables(case["tokens"], case["hidden"] // case["heads"]))
    return module, x, cos, sin


def _weights(case, draws):
    """A decoder's tensors: embedding, per-layer packs and norms, and a head that follows a fixed successor of each
    token with a wide margin (as a trained model's does), so that greedy tokens do not hang on the last bit."""

    h, i, g, bits = case["hidden"], case["inter"], 64, case["bits"]
    qd, kd = case["heads"] * case["dim"], case["kv_heads"] * case["dim"]

    def pack(n, k, std):
        return _pack(draws.normal(n, k, std=std), g, bits)

    layers = [dict(qkv=pack(qd + 2 * kd, h, 0.03), bias=draws.normal(qd + 2 * kd, std=0.03), o=pack(h, qd, 0.01),
                   gate=pack(i, h, 0.03), up=pack(i, h, 0.03), down=pack(h, i, 0.005), norm1=draws.norm(h),
                   norm2=draws.norm(h)) for _ in range(case["layers"])]
    embed = draws.normal(case["vocab"], h)
    head = _pack(embed.roll(7, dims=0).mul(0.03), g, bits)
    ids = draws.ids(case["length"], case["vocab"])
    return dict(layers=layers, embed=embed, head=head, norm=draws.norm(h), ids=ids,
                token=draws.ids(1, case["vocab"]).view(1))


def _inputs(case, seed):
    """The tensors of a single-operation case, in the order :func:`prepare` and :func:`exact` both make them."""

    kind, draws = case["kind"], _Draws(seed)
    if kind == "gemv":
        n, k, g, bits = case["n"], case["k"], case["group"], case["bits"]
        paired = case["epilogue"] == "paired"
        return dict(x=draws.normal(k), w=draws.packed(n, k, g, bits), up=draws.packed(n, k, g, bits) if paired else None,
                    norm=draws.norm(k) if case["norm"] else None,
                    bias=draws.normal(n, std={"bias": 0.03}.get(case["epilogue"], 1.0))
                    if case["epilogue"] in ("bias", "residual") else None)
    if kind == "head":
        x, weight = draws.normal(case["k"]), draws.normal(case["n"], case["k"], std=0.03)
        weight[case["n"] * 5 // 7] = x * 0.03  # one token well ahead of the others, as a trained model's logits have it
        return dict(x=x, w=_pack(weight, case["group"], case["bits"]), norm=draws.norm(case["k"]), up=None, bias=None)
    if kind == "decode_attention":
        width = (case["heads"] + 2 * case["kv_heads"]) * case["dim"]
        cos, sin = _tables(case["capacity"], case["dim"])
        return dict(row=draws.normal(1, width), cos=cos, sin=sin,
                    pair=draws.normal(2, 1, case["kv_heads"], case["capacity"], case["dim"]))
    if kind == "attention":
        t, d = case["tokens"], case["dim"]
        return dict(q=draws.normal(1, case["heads"], t, d), k=draws.normal(1, case["kv_heads"], t, d),
                    v=draws.normal(1, case["kv_heads"], t, d))
    if kind == "pack":
        return dict(w=draws.normal(case["rows"], case["cols"], std=0.03,
                                   dtype=torch.float32 if case["f32"] else BF16))
    x = draws.normal(case["tokens"], case["k"])
    if kind == "mlp":
        n = case["n"]
        return dict(x=x, w=draws.packed(n, case["k"], case["group"], case["bits"]),
                    up=draws.packed(n, case["k"], case["group"], case["bits"]))
    if kind == "out":
        return dict(x=x, w=draws.packed(case["n"], case["k"], case["group"], case["bits"]),
                    residual=draws.normal(case["tokens"], case["n"]), norm=draws.norm(case["n"]))
    n = (case["heads"] + 2 * case["kv_heads"]) * case["dim"]
    cos, sin = _tables(case["tokens"] + case["extra"], case["dim"])
    return dict(x=x, w=draws.packed(n, case["k"], case["group"], case["bits"]), cos=cos, sin=sin,
                bias=draws.normal(n, std=0.03) if case["bias"] else None,
                positions=torch.arange(case["tokens"], device="cuda"))


def _spec(case):
    from aotolith_amd.decoder import DecoderSpec

    return DecoderSpec(family="qwen2", vocab=case["vocab"], hidden=case["hidden"], intermediate=case["inter"],
                       layers=case["layers"], heads=case["heads"], kv_heads=case["kv_heads"], head_dim=case["dim"],
                       eps=1e-6, theta=1e6, qkv_bias=True)


def _runtime(case, weights):
    from aotolith_amd.decoder import DecoderState, LayerState, PackedWeight, compile_decoder_state

    def packed(pair):
        return PackedWeight(*pair, 64, case["bits"])

    layers = [LayerState(qkv=packed(w["qkv"]), o=packed(w["o"]), gate=packed(w["gate"]), up=packed(w["up"]),
                         down=packed(w["down"]), input_norm=w["norm1"], post_norm=w["norm2"], qkv_bias=w["bias"])
              for w in weights["layers"]]
    state = DecoderState(embed=weights["embed"], final_norm=weights["norm"], lm_head=packed(weights["head"]),
                         layers=layers)
    return compile_decoder_state(_spec(case), state, prompt_length=case["bucket"], max_new_tokens=case["new"],
                                 group_size=64)


def prepare(case, seed):
    from aotolith_amd import compile_module, ops

    kind = case["kind"]
    state = dict(case=case)
    if kind == "block":
        module, x, cos, sin = _block(case, _Draws(seed))
        plan = compile_module(module, (x, cos, sin))
        return dict(state, plan=plan, x=x, cos=cos, sin=sin)
    if kind in ("prefill_decode", "generate"):
        weights = _weights(case, _Draws(seed))
        return dict(state, runtime=_runtime(case, weights), ids=weights["ids"], token=weights["token"])
    state.update(_inputs(case, seed))
    # the buffers a decode loop or a prefill keeps from call to call
    if kind == "decode_attention":
        state["workspace"] = ops.decode_attention_workspace(1, case["heads"], case["kv_heads"], case["capacity"],
                                                            case["dim"], device="cuda")
    if kind == "qkv":
        state["pair"] = torch.zeros(2, 1, case["kv_heads"], case["tokens"] + case["extra"], case["dim"], dtype=BF16,
                                    device="cuda")
    if kind == "attention" and case["mask"]:
        at = torch.arange(case["tokens"], device="cuda")
        state["mask"] = (at[None, :] <= at[:, None]) & (at[None, :] >= case["start"])
    return state


def run(state):
    from aotolith_amd import ops

    case = state["case"]
    kind = case["kind"]
    if kind == "gemv":
        gemv = ops.w4_gemv if case["bits"] == 4 else ops.w8_gemv
        return gemv(state["x"], *state["w"], case["group"], norm_weight=state["norm"], bias=state["bias"],
                    up=state["up"])
    if kind == "head":
        gemv = ops.w4_gemv if case["bits"] == 4 else ops.w8_gemv
        logits = gemv(state["x"], *state["w"], case["group"], norm_weight=state["norm"])
        return logits, ops.argmax(logits)
    if kind == "decode_attention":
        heads, kv, dim, cap = case["heads"], case["kv_heads"], case["dim"], case["capacity"]
        out = ops.decode_rope_attention(
            state["row"], state["cos"], state["sin"], state["pair"], query_heads=heads, query_start=0,
            key_start=heads * dim, value_start=(heads + kv) * dim, position=case["valid"] - 1,
            slot=(case["offset"] - 1) % cap, valid=case["valid"], ring_offset=case["offset"],
            workspace=state["workspace"])
        return out, state["pair"]
    if kind == "attention":
        if case["mask"]:
            return ops.prefill_attention(state["q"], state["k"], state["v"], mask=state["mask"])
        return ops.prefill_attention(state["q"], state["k"], state["v"], key_start=case["start"])
    if kind == "qkv":
        out, q = ops.matmul_qkv_rope(
            state["x"], *state["w"], case["group"], state["positions"], state["cos"], state["sin"], state["pair"],
            query_heads=case["heads"], kv_heads=case["kv_heads"], head_dim=case["dim"], slot0=case["extra"],
            bias=state["bias"], bits=case["bits"])
        return out, q, state["pair"]
    if kind == "mlp":
        matmul = ops.w4_matmul_gate_up if case["bits"] == 4 else ops.w8_matmul_gate_up
        return matmul(state["x"], *state["w"], *state["up"], case["group"])
    if kind == "out":
        return ops.matmul_residual_norm(state["x"], *state["w"], case["group"], state["residual"], state["norm"],
                                        1e-6, bits=case["bits"])
    if kind == "pack":
        return ops.quantize(state["w"], case["group"], case["bits"])
    if kind == "block":
        return state["plan"](state["x"], state["cos"], state["sin"])
    runtime = state["runtime"]
    if kind == "generate":
        tokens = runtime.greedy_generate(state["ids"])
        return tokens, runtime.engine.logits, runtime.engine.ring  # the ring: the generation's cache
    logits, compact = runtime.prefill_padded(state["ids"])
    step, cache = runtime.decode_token(state["token"], runtime.pad_cache(compact), case["length"] + 1)
    return logits, step, cache


# ----------------------------------------------------------------------------- work, tolerance, 64 bits
def _packed_bytes(n, k, case):
    return n * k * case["bits"] // 8 + n * (k // case["group"]) * 2


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        copies = 2 if case["epilogue"] == "paired" else 1
        n, k = case["n"], case["k"]
        return {"bytes": copies * _packed_bytes(n, k, case) + 2 * (k * (1 + case["norm"]) + n), "flops": 2 * copies * n * k}
    if kind == "head":
        n, k = case["n"], case["k"]
        return {"bytes": _packed_bytes(n, k, case) + 4 * k + 2 * n, "flops": 2 * n * k}
    if kind == "decode_attention":
        heads, kv, dim, valid = case["heads"], case["kv_heads"], case["dim"], case["valid"]
        return {"bytes": 4 * kv * valid * dim + 4 * heads * dim, "flops": 4 * heads * valid * dim}
    if kind == "attention":
        live = case["tokens"] - case["start"]
        heads, kv, dim, t = case["heads"], case["kv_heads"], case["dim"], case["tokens"]
        return {"bytes": 4 * t * heads * dim + 4 * t * kv * dim, "flops": 2 * live * (live + 1) * heads * dim}
    if kind in ("qkv", "mlp", "out"):
        t, k = case["tokens"], case["k"]
        if kind == "qkv":
            n, copies = (case["heads"] + 2 * case["kv_heads"]) * case["dim"], 1
            held = 2 * 2 * t * n + 4 * case["kv_heads"] * case["extra"] * case["dim"]
        else:
            n, copies = case["n"], 2 if kind == "mlp" else 1
            held = 2 * t * n * (1 if kind == "mlp" else 3)
        return {"bytes": copies * _packed_bytes(n, k, case) + 2 * t * k + held, "flops": 2 * copies * t * n * k}
    if kind == "pack":
        size = case["rows"] * case["cols"]
        return {"bytes": size * (4 if case["f32"] else 2) + _packed_bytes(case["rows"], case["cols"], case),
                "flops": 2 * size}
    if kind == "block":
        h, i, t = case["hidden"], case["inter"], case["tokens"]
        size = 2 if case["dtype"] == "bf16" else 4
        kv = h // case["heads"] * case["kv_heads"]
        weights = 2 * h * h + 2 * h * kv + 3 * h * i
        return {"bytes": size * (weights + 2 * t * h), "flops": 2 * t * weights + 2 * t * (t + 1) * h}
    h, i, dim = case["hidden"], case["inter"], case["dim"]
    qd, kd = case["heads"] * dim, case["kv_heads"] * dim
    layer, head = h * (qd + 2 * kd) + h * qd + 3 * h * i, h * case["vocab"]
    packed = (case["layers"] * layer + head) * (case["bits"] / 8 + 2 / 64)
    window = case["layers"] * 4 * kd * (case["bucket"] + case["new"])
    steps = 2 if kind == "prefill_decode" else case["new"]
    return {"bytes": steps * packed + (steps - 1) * window * (2 if kind == "prefill_decode" else 1),
            "flops": 2 * (case["length"] + steps - 1) * case["layers"] * layer + 2 * steps * head}


def tolerance(case):
    kind = case["kind"]
    if kind == "pack":
        return "exact"
    if kind == "block":
        return {"rel": 2e-2} if case["dtype"] == "bf16" else {"rel": 1e-5}
    if kind in ("prefill_decode", "generate"):  # 24 layers of bf16 roundings: 1.3e-2 to 1.4e-2 off 64 bits
        return {"rel": 3e-2, "max": 0.5, "differ": 0.0}
    if kind == "head":
        return {"rel": 8e-3, "differ": 0.0}
    if kind == "mlp" or case.get("epilogue") == "paired":  # the gate is rounded once more than the others' sums
        return {"rel": 1.2e-2}
    return {"rel": 8e-3}


def _attend(q, k, v, keep, scale):
    """``q [H, T, D]`` over ``k``, ``v`` ``[Hkv, S, D]`` with the keep mask ``[T, S]``; a row of none gives zeros."""

    out = torch.empty_like(q)
    for head in range(q.shape[0]):
        at = head * k.shape[0] // q.shape[0]
        scores = (q[head] @ k[at].T * scale).masked_fill(~keep, -math.inf)
        out[head] = torch.nan_to_num(torch.softmax(scores, -1)) @ v[at]
    return out


def _forward(case, weights, ids, cos, sin):
    """A decoder in 64 bits over ``ids [T]``: (logits of the last token, [keys, values] of each layer)."""

    heads, kv, dim = case["heads"], case["kv_heads"], case["dim"]
    t = ids.shape[0]
    keep = torch.ones(t, t, dtype=torch.bool, device="cuda").tril()
    x = weights["embed"][ids].double()
    caches = []

    def project(y, pair):
        return y @ _dequantized(*pair, case["bits"], True).T

    for w in weights["layers"]:
        qkv = project(_rms(x, w["norm1"].double()), w["qkv"]) + w["bias"].double()
        q, k, v = (part.view(t, -1, dim).transpose(0, 1) for part in qkv.split((heads * dim, kv * dim, kv * dim), 1))
        q, k = _rotate(q, cos[:t], sin[:t]), _rotate(k, cos[:t], sin[:t])
        caches.append(torch.stack((k, v)))
        x = x + project(_attend(q, k, v, keep, dim ** -0.5).transpose(0, 1).reshape(t, -1), w["o"])
        n = _rms(x, w["norm2"].double())
        x = x + project(F.silu(project(n, w["gate"])) * project(n, w["up"]), w["down"])
    return project(_rms(x[-1:], weights["norm"].double()), weights["head"]), caches


def exact(case, seed):
    kind = case["kind"]
    if kind == "block":
        module, x, cos, sin = _block(case, _Draws(seed))
        module, t, dim = module.double(), case["tokens"], case["hidden"] // case["heads"]
        x, cos, sin = x[0].double(), cos.double(), sin.double()
        n = _rms(x, module.norm1)
        q, k, v = (f(n).view(t, -1, dim).transpose(0, 1) for f in (module.q, module.k, module.v))
        keep = torch.ones(t, t, dtype=torch.bool, device="cuda").tril()
        a = _attend(_rotate(q, cos, sin), _rotate(k, cos, sin), v, keep, dim ** -0.5)
        x = x + module.o(a.transpose(0, 1).reshape(t, -1))
        n = _rms(x, module.norm2)
        return ((x + module.down(F.silu(module.gate(n)) * module.up(n)))[None],)
    if kind in ("prefill_decode", "generate"):
        weights = _weights(case, _Draws(seed))
        cos, sin = (table.double() for table in _tables(case["bucket"] + case["new"], case["dim"]))
        ids = weights["ids"][0]
        if kind == "generate":
            logits, _ = _forward(case, weights, ids, cos, sin)
            tokens = [int(logits.argmax())]
            while len(tokens) < case["new"]:  # the head's successor of each token
                tokens.append((tokens[-1] + 7) % case["vocab"])
            tokens = torch.tensor(tokens, device="cuda")
            logits, _ = _forward(case, weights, torch.cat((ids, tokens[:-1])), cos, sin)
            return tokens[None], logits[None], None  # the ring is rotated, and its unused slots hold no such value
        first, _ = _forward(case, weights, ids, cos, sin)
        step, caches = _forward(case, weights, torch.cat((ids, weights["token"])), cos, sin)
        capacity, length = case["bucket"] + case["new"], case["length"]
        cache = torch.zeros(case["layers"], 2, 1, case["kv_heads"], capacity, case["dim"], device="cuda",
                            dtype=torch.float64)
        for layer, pair in enumerate(caches):
            cache[layer, :, 0, :, capacity - length - 1:] = pair
        return first[None], step[None], None if length < case["bucket"] else cache  # pad slots hold no such value
    at = _inputs(case, seed)
    if kind in ("gemv", "head"):
        x = at["x"].double()
        if at["norm"] is not None:
            x = _rms(x, at["norm"].double())
        y = _dequantized(*at["w"], case["bits"], False) @ x
        if kind == "head":
            return y, y.argmax().view(1)
        if at["up"] is not None:
            return F.silu(y) * (_dequantized(*at["up"], case["bits"], False) @ x)
        return y if at["bias"] is None else y + at["bias"].double()
    if kind == "decode_attention":
        heads, kv, dim, cap, valid = (case[n] for n in ("heads", "kv_heads", "dim", "capacity", "valid"))
        q, k, v = (p.view(-1, dim) for p in at["row"][0].double().split((heads * dim, kv * dim, kv * dim)))
        cos, sin = at["cos"][valid - 1].double(), at["sin"][valid - 1].double()
        pair = at["pair"].double()
        pair[0, 0, :, (case["offset"] - 1) % cap] = _rotate(k, cos, sin)
        pair[1, 0, :, (case["offset"] - 1) % cap] = v
        order = (torch.arange(cap - valid, cap, device="cuda") + case["offset"]) % cap
        keep = torch.ones(1, valid, dtype=torch.bool, device="cuda")
        out = _attend(_rotate(q, cos, sin)[:, None], pair[0, 0][:, order], pair[1, 0][:, order], keep, dim ** -0.5)
        return out.view(1, heads, dim), pair
    if kind == "attention":
        spot = torch.arange(case["tokens"], device="cuda")
        keep = (spot[None, :] <= spot[:, None]) & (spot[None, :] >= case["start"])
        out = _attend(at["q"][0].double(), at["k"][0].double(), at["v"][0].double(), keep, case["dim"] ** -0.5)
        return out.transpose(0, 1).reshape(1, case["tokens"], -1)
    if kind == "pack":
        return _pack(at["w"], case["group"], case["bits"])
    y = at["x"].double() @ _dequantized(*at["w"], case["bits"], True).T
    if kind == "mlp":
        return F.silu(y) * (at["x"].double() @ _dequantized(*at["up"], case["bits"], True).T)
    if kind == "out":
        y = y + at["residual"].double()
        return y, _rms(y, at["norm"].double())
    if at["bias"] is not None:
        y = y + at["bias"].double()
    heads, kv, dim, t, start = (case[n] for n in ("heads", "kv_heads", "dim", "tokens", "extra"))
    q, k, v = (p.view(t, -1, dim).transpose(0, 1) for p in y.split((heads * dim, kv * dim, kv * dim), 1))
    cos, sin = at["cos"][:t].double(), at["sin"][:t].double()
    pair = torch.zeros(2, 1, kv, t + start, dim, dtype=torch.float64, device="cuda")
    pair[0, 0, :, start:], pair[1, 0, :, start:] = _rotate(k, cos, sin), v
    return y, _rotate(q, cos, sin)[None], pair
