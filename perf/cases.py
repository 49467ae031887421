"""Performance cases of the framework: what its users have it do, through its public entry points.

  matmul    QMatMul.forward of one GGUF weight: a token, a served batch, a prompt
  moe       FusedMoeGGUF.forward, a layer of a mixture of quantized experts
  llama     ModelWeights of the Q4_K_M llama decoder: a prompt, or a prompt and greedy generation
  venizen   the decoder of talking-head attention, retention and the generalized delta rule (bfloat16 weights)
  kudurax   the decoder of latent attention and mixtures of experts (bfloat16 weights)

Weights are made as a file would bring them: GGUF blocks of normally distributed codes, or bfloat16 tensors.  ``exact`` evaluates the same definitions
in 64 bits with plain torch.  GGUF products are defined on activations rounded to int8 blocks (Q8_K for the K formats, Q8_0 otherwise), which
``exact`` does as well, in f32 as the definition says.
"""
import math
import zlib

import numpy as np
import torch

from candle_amd import kudurax, venizen
from candle_amd.fused_moe import FusedMoeGGUF
from candle_amd.quantized import GgmlDType, QMatMul, QStorage, QTensor
from candle_amd.quantized_llama import Config as LlamaConfig
from candle_amd.quantized_llama import ModelWeights

DEV = "cuda:0"
FORMATS = {"q4_0": GgmlDType.Q4_0, "q8_0": GgmlDType.Q8_0, "q4_k": GgmlDType.Q4K, "q5_k": GgmlDType.Q5K, "q6_k": GgmlDType.Q6K}
BLOCK_BYTES = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210)}
FLOATS = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# a Q4_K_M file: attn_v and ffn_down in Q6_K, the rest in Q4_K
Q4_K_M = {"attention_wq": "q4_k", "attention_wk": "q4_k", "attention_wv": "q6_k", "attention_wo": "q4_k", "feed_forward_w1": "q4_k", "feed_forward_w3": "q4_k",
          "feed_forward_w2": "q6_k", "output": "q4_k"}


def listed():
    return [
        # one projection of one token: the smallest call there is (8-bit attention projection of a 4096-wide model)
        {"name": "token_q8_0", "kind": "matmul", "fmt": "q8_0", "n": 4096, "k": 4096, "rows": 1, "dtype": "f32"},
        # sixteen sequences served together: the gate projection of an 8B model over a token of each
        {"name": "batch16_q4_k", "kind": "matmul", "fmt": "q4_k", "n": 14336, "k": 4096, "rows": 16, "dtype": "f32"},
        # a short prompt of odd length through the feed-forward of a 5120-wide layer, half-precision activations
        {"name": "prompt131_q4_0", "kind": "matmul", "fmt": "q4_0", "n": 13824, "k": 5120, "rows": 131, "dtype": "f16"},
        # an ordinary prompt through a gate projection, bfloat16 activations
        {"name": "prompt512_q5_k", "kind": "matmul", "fmt": "q5_k", "n": 14336, "k": 4096, "rows": 512, "dtype": "bf16"},
        # a full context through the down projection of an 8B model
        {"name": "prompt2048_q6_k", "kind": "matmul", "fmt": "q6_k", "n": 4096, "k": 14336, "rows": 2048, "dtype": "f32"},
        # mixture of 128 experts of which a token takes 8 (30B-A3B layer shape): decoding for sixteen sequences, and a prompt
        {"name": "moe_decode16", "kind": "moe", "fmt": "q4_k", "experts": 128, "top": 8, "hidden": 2048, "inter": 768, "tokens": 16, "dtype": "f32"},
        {"name": "moe_prompt1500", "kind": "moe", "fmt": "q4_k", "experts": 128, "top": 8, "hidden": 2048, "inter": 768, "tokens": 1500, "dtype": "bf16"},
        # the 8B decoder at an eighth of its depth and a quarter of its vocabulary: a chat turn (prompt, then tokens one by one), and a long prompt
        {"name": "llama_chat", "kind": "llama", "layers": 4, "hidden": 4096, "heads": 32, "kv_heads": 8, "ffn": 14336, "vocab": 32768, "prompt": 300, "new": 64},
        {"name": "llama_prompt1000", "kind": "llama", "layers": 4, "hidden": 4096, "heads": 32, "kv_heads": 8, "ffn": 14336, "vocab": 32768, "prompt": 1000, "new": 0},
        # the bfloat16 decoders: long prompts, and a chat turn
        {"name": "venizen_prompt2048", "kind": "venizen", "width": 2048, "vocab": 32768, "prompt": 2048, "new": 0},
        {"name": "kudurax_prompt1500", "kind": "kudurax", "width": 2048, "vocab": 32768, "prompt": 1500, "new": 0},
        {"name": "kudurax_chat", "kind": "kudurax", "width": 2048, "vocab": 32768, "prompt": 100, "new": 48},
    ]


def log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "matmul", "matmul", "matmul", "moe", "moe", "llama", "llama", "venizen", "kudurax", "kudurax"])
    if kind == "matmul":
        while True:
            n, k, rows = log_uniform(rng, 1024, 16384), 256 * log_uniform(rng, 4, 56), log_uniform(rng, 1, 2048)
            if n * k <= 14336 * 5120 and n * k * rows <= 4096 * 14336 * 2048:
                break
        if rng.random() < 0.7:
            n = n // 64 * 64
        return {"kind": kind, "fmt": rng.choice(sorted(FORMATS)), "n": n, "k": k, "rows": rows, "dtype": rng.choice(["f32", "f32", "f32", "bf16", "f16"])}
    if kind == "moe":
        return {"kind": kind, "fmt": rng.choice(["q4_k", "q4_k", "q5_k", "q6_k", "q8_0"]), "experts": rng.choice([64, 128]), "top": rng.choice([4, 6, 8]),
                "hidden": rng.choice([1024, 2048]), "inter": rng.choice([512, 768, 1024]), "tokens": log_uniform(rng, 1, 1500), "dtype": rng.choice(["f32", "f32", "bf16"])}
    if kind == "llama":
        hidden = rng.choice([2048, 4096])
        return {"kind": kind, "layers": rng.choice([2, 3, 4]), "hidden": hidden, "heads": hidden // 128, "kv_heads": hidden // 512, "ffn": hidden * 7 // 2, "vocab": 32768,
                "prompt": log_uniform(rng, 20, 1000), "new": rng.choice([0, 8, 24, 64])}
    return {"kind": kind, "width": rng.choice([1024, 2048]), "vocab": rng.choice([8192, 32768]), "prompt": log_uniform(rng, 20, 1500), "new": rng.choice([0, 0, 8, 24])}


# ------------------------------------------------------------------------------------------------- weights
def generator(seed, name):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) << 32) + zlib.crc32(name.encode()))
    return g


def normal(seed, name, *shape):
    return torch.randn(shape, generator=generator(seed, name), device=DEV)


def halves(x):
    """f32 [blocks] -> the two bytes of each as f16."""
    return x.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def nibbles(low, high):
    return low | (high << 4)


def six_bits(sc, m):
    """Scales and minimums [blocks, 8] of a K block in its 12 bytes."""
    return torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), m[:, :4] | ((m[:, 4:] >> 4) << 6), nibbles(sc[:, 4:] & 15, m[:, 4:] & 15)], 1)


def blocks(fmt, seed, name, *shape):
    """GGUF block bytes [blocks, bytes] of a weight of standard deviation 0.02: normally distributed codes under scales that vary from block to block."""
    size, nbytes = BLOCK_BYTES[fmt]
    nb = math.prod(shape) // size
    g = generator(seed, name)
    out = torch.empty((nb, nbytes), dtype=torch.uint8, device=DEV)
    part = 1 << 20
    for lo in range(0, nb, part):
        m = min(part, nb - lo)
        rand = lambda *s: torch.randn(s, generator=g, device=DEV)
        codes = lambda mean, dev, top: (rand(m, size) * dev + mean).round_().clamp_(0, top).to(torch.uint8)
        d = torch.exp(0.1 * rand(m))
        if fmt == "q8_0":
            out[lo:lo + m] = torch.cat([halves(d * (0.02 / 45)), codes(127, 45, 254).to(torch.int16).sub_(127).to(torch.int8).view(torch.uint8)], 1)
            continue
        if fmt == "q4_0":
            c = codes(8, 3, 15)
            out[lo:lo + m] = torch.cat([halves(d * (0.02 / 3)), nibbles(c[:, :16], c[:, 16:])], 1)
            continue
        if fmt == "q6_k":
            c = codes(32, 10, 63).reshape(m, 2, 4, 32)
            ql = torch.stack([nibbles(c[:, :, 0] & 15, c[:, :, 2] & 15), nibbles(c[:, :, 1] & 15, c[:, :, 3] & 15)], 2).reshape(m, 128)
            qh = sum((c[:, :, i] >> 4) << (2 * i) for i in range(4)).to(torch.uint8).reshape(m, 64)
            sc = (rand(m, 16) * 15 + 90).round_().clamp_(40, 127).to(torch.uint8)
            out[lo:lo + m] = torch.cat([ql, qh, sc, halves(d * (0.02 / 10 / 90))], 1)
            continue
        dev, top = (3, 15) if fmt == "q4_k" else (6, 31)
        c = codes(0.5 * top, dev, top)
        sc = (rand(m, 8) * 6 + 48).round_().clamp_(24, 63).to(torch.uint8)
        mn = (sc + rand(m, 8) * 2).round_().clamp_(20, 63).to(torch.uint8)
        step = d * (0.02 / dev / 48)
        c4 = (c & 15).reshape(m, 4, 2, 32)
        parts = [halves(step), halves(step * (0.5 * top)), six_bits(sc, mn)]
        if fmt == "q5_k":
            parts.append(sum((c.reshape(m, 8, 32)[:, i] >> 4) << i for i in range(8)).to(torch.uint8))
        out[lo:lo + m] = torch.cat(parts + [nibbles(c4[:, :, 0], c4[:, :, 1]).reshape(m, 128)], 1)
    return out


def values(fmt, b, *shape):
    """The weights that block bytes stand for, in 64 bits."""
    f = lambda lo: b[:, lo:lo + 2].contiguous().view(torch.float16).to(torch.float64)
    if fmt == "q8_0":
        w = f(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "q4_0":
        w = f(0) * (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8)
    elif fmt == "q6_k":
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
        c = torch.stack([(ql[:, :, i % 2] >> (4 * (i // 2)) & 15) | ((qh >> (2 * i) & 3) << 4) for i in range(4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        w = f(208) * (sc.repeat_interleave(16, 1) * (c.reshape(-1, 256).double() - 32))
    else:
        s, qs = b[:, 4:16], b[:, -128:].reshape(-1, 4, 32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        c = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
        if fmt == "q5_k":
            c = c | torch.stack([(b[:, 16:48] >> i & 1) << 4 for i in range(8)], 1)
        w = ((f(0) * sc)[:, :, None] * c.double() - (f(2) * mn)[:, :, None]).reshape(-1, 256)
    return w.reshape(shape)


def weight(fmt, b, *shape):
    return QTensor.new(QStorage.from_data(b, DEV, FORMATS[fmt]), shape)


def rounded(fmt, x):
    """Activation rows as their int8 blocks hold them."""
    size = BLOCK_BYTES[fmt][0]
    z = x.to(torch.float32).reshape(-1, size)
    first = torch.arange(size, device=DEV)
    at = torch.where(z.abs() == z.abs().amax(1, keepdim=True), first, size - 1).amin(1, keepdim=True)
    if size == 256:
        top = z.gather(1, at)
        scale = torch.where(top != 0, torch.full_like(top, -127.0) / top, 0.0)      # one division: a reciprocal times -127 rounds twice
        d = torch.where(top != 0, torch.ones_like(top) / scale, 0.0).double()
    else:
        top = z.gather(1, at).abs()
        d32 = top / torch.full_like(top, 127.0)
        scale = torch.where(d32 != 0, torch.ones_like(top) / d32, 0.0)
        d = d32.to(torch.float16).double()
    v = (z * scale).double()
    return ((v.sign() * (v.abs() + 0.5).floor()).clamp(-128, 127) * d).reshape(x.shape)


def product(fmt, x, w):
    return rounded(fmt, x) @ w.T


# ------------------------------------------------------------------------------------------------- one weight
def matmul_weight(case, seed):
    return blocks(case["fmt"], seed, "w", case["n"], case["k"])


def matmul_input(case, seed):
    return normal(seed, "x", 1, case["rows"], case["k"]).to(FLOATS[case["dtype"]])


# ------------------------------------------------------------------------------------------------- a mixture layer
def moe_shapes(case):
    E, h, i = case["experts"], case["hidden"], case["inter"]
    return {"gate": (E, i, h), "up": (E, i, h), "down": (E, h, i)}


def moe_router(case, seed):
    return normal(seed, "router", case["experts"], case["hidden"]) * 2 / math.sqrt(case["hidden"])


def moe_input(case, seed):
    return normal(seed, "x", 1, case["tokens"], case["hidden"]).to(FLOATS[case["dtype"]])


def moe_exact(case, seed):
    fmt, x = case["fmt"], moe_input(case, seed)[0].double()
    p, ids = torch.softmax(x @ moe_router(case, seed).double().T, -1).topk(case["top"], -1)
    p = p / p.sum(-1, keepdim=True)
    b = {name: blocks(fmt, seed, name, *shape).reshape(case["experts"], -1, BLOCK_BYTES[fmt][1]) for name, shape in moe_shapes(case).items()}
    out = torch.zeros_like(x)
    for e in range(case["experts"]):
        t, slot = (ids == e).nonzero(as_tuple=True)
        if len(t):
            w = {name: values(fmt, b[name][e], *shape[1:]) for name, shape in moe_shapes(case).items()}
            h = torch.nn.functional.silu(product(fmt, x[t], w["gate"])) * product(fmt, x[t], w["up"])
            out.index_add_(0, t, product(fmt, h, w["down"]) * p[t, slot, None])
    return out[None]


# ------------------------------------------------------------------------------------------------- the llama decoder
def llama_config(case):
    return LlamaConfig(n_layer=case["layers"], hidden=case["hidden"], n_head=case["heads"], n_kv_head=case["kv_heads"], head_dim=case["hidden"] // case["heads"],
                       ffn=case["ffn"], vocab=case["vocab"], ctx=case["prompt"] + case["new"] + 28)


def llama_blocks(case, seed):
    """(name, format, shape, block bytes) of every quantized tensor."""
    h, kv, f = case["hidden"], case["kv_heads"] * (case["hidden"] // case["heads"]), case["ffn"]
    shapes = {"attention_wq": (h, h), "attention_wk": (kv, h), "attention_wv": (kv, h), "attention_wo": (h, h), "feed_forward_w1": (f, h), "feed_forward_w3": (f, h),
              "feed_forward_w2": (h, f)}
    every = [("output", "output", (case["vocab"], h))] + [(f"blk.{i}.{name}", name, shape) for i in range(case["layers"]) for name, shape in shapes.items()]
    for full, name, shape in every:
        yield full, Q4_K_M[name], shape, blocks(Q4_K_M[name], seed, full, *shape)


def following(case, seed):
    """The token that the models' heads favour after each token: a trained model is mostly sure of what follows, and so are these."""
    return torch.randperm(case["vocab"], generator=generator(seed, "following"), device=DEV)


def embedding_for(head, case, seed):
    """An embedding under which the head's largest logit belongs to the following token, eight times as large as what a layer adds to it: as in a trained
    model, no single layer turns the residual stream round."""
    return (head[following(case, seed)] * 400).float()


def norm_weight(case, seed, name):
    return 1 + 0.1 * normal(seed, name, case["hidden"])


def prompt_of(case, seed):
    return torch.randint(0, case["vocab"], (case["prompt"],), generator=generator(seed, "prompt"), device=DEV)


def llama_exact(case, seed):
    """Logits of the last position and the caches, of the prompt and of the tokens that follow it."""
    cfg, eps = llama_config(case), 1e-5
    H, G, D = cfg.n_head, cfg.n_kv_head, cfg.head_dim
    w = {name: (fmt, shape, b) for name, fmt, shape, b in llama_blocks(case, seed)}
    mm = lambda x, name: product(w[name][0], x, values(w[name][0], w[name][2], *w[name][1]))
    norm = lambda x, name: x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * norm_weight(case, seed, name).double()
    tokens, after = prompt_of(case, seed).tolist(), following(case, seed).tolist()
    for _ in range(case["new"]):
        tokens.append(after[tokens[-1]])
    new, tokens = tokens[case["prompt"]:], tokens[:max(case["prompt"], len(tokens) - 1)]
    T = len(tokens)
    # the angles are f32 products by definition: at position 1000 they are off by up to 3e-5, which the rounding to int8 behind them would turn into more
    theta = np.float32(1.0) / np.power(np.float32(cfg.rope_theta), np.arange(0, D, 2, dtype=np.float32) / np.float32(D))
    angle = torch.from_numpy(np.arange(T, dtype=np.float32)[:, None] * theta).to(DEV).double()
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def turned(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    head = values(*[w["output"][i] for i in (0, 2)], *w["output"][1])
    x = embedding_for(head, case, seed)[torch.tensor(tokens, device=DEV)].double()
    later = torch.ones(T, T, dtype=torch.bool, device=DEV).triu(1)
    caches = []
    for i in range(cfg.n_layer):
        h = norm(x, f"blk.{i}.attention_norm")
        q, k, v = (mm(h, f"blk.{i}.attention_{n}").reshape(T, -1, D) for n in ("wq", "wk", "wv"))
        q, k, v = turned(q).transpose(0, 1), turned(k).transpose(0, 1), v.transpose(0, 1)
        for c in (k, v):
            caches.append(torch.cat([c, c.new_zeros(G, cfg.ctx - T, D)], 1))
        s = q.reshape(G, H // G, T, D) @ k[:, None].transpose(-1, -2) / math.sqrt(D)
        o = torch.softmax(s.masked_fill_(later, -math.inf), -1) @ v[:, None]
        x = x + mm(o.reshape(H, T, D).transpose(0, 1).reshape(T, H * D), f"blk.{i}.attention_wo")
        h = norm(x, f"blk.{i}.ffn_norm")
        x = x + mm(torch.nn.functional.silu(mm(h, f"blk.{i}.feed_forward_w1")) * mm(h, f"blk.{i}.feed_forward_w3"), f"blk.{i}.feed_forward_w2")
    logits = product(w["output"][0], norm(x[-1:], "norm"), head)
    return {"logits": logits, "cache": caches, **({"tokens": torch.tensor(new)} if new else {})}


# ------------------------------------------------------------------------------------------------- the bfloat16 decoders
def design_config(case):
    """Widths of 1024 and 2048 with heads of 128 / 64, as the repository's benchmark lays these decoders out."""
    w = case["width"]
    heads = w // 128
    top = {"vocab": case["vocab"], "width": w, "norm": {"eps": 1e-5}}
    if case["kind"] == "venizen":
        parallel = {"type": "parallel", "mlp": {"kind": "dense", "ff": w * 7 // 2},
                    "mixer": {"left": {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": 1024, "keep_first": 4},
                                       "rot": {"base": 500000.0, "dims": 128}},
                              "right": {"heads": heads // 2, "dim": 128, "vdim": 128, "rot": {"base": 10000.0, "dims": 128},
                                        "decay": [1.0 - 2.0 ** -(5 + 5.0 * h / (heads // 2 - 1)) for h in range(heads // 2)]},
                              "left_scale": 1.0, "right_scale": 1.0}}
        delta = {"type": "general_delta", "mixer": {"heads": w // 64, "dim": 64}, "mlp": None}
        return dict(top, layers=[parallel, delta, parallel, delta], loop={"start": 2, "stop": 4, "times": 2})
    mixer = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5,
             "rot": {"base": 10000.0, "dims": 64, "scaling": {"factor": 40.0, "fast": 32.0, "slow": 1.0, "original": 4096}}}
    dense = {"kind": "dense", "ff": w * 7 // 2}
    mixture = {"kind": "moe", "router": {"experts": 64, "top": 6}, "expert": {"ff": w * 11 // 16}, "shared": {"ff": w * 11 // 8}}
    layer = lambda mlp, source=None: {"type": "latent_attention", "mlp": mlp, "mixer": mixer if source is None else dict(mixer, kv_from=source)}
    return dict(top, embedding={"scale": 1.0}, layers=[layer(dense), layer(mixture), layer(dense, 1), layer(mixture, 1)])


def design(case):
    module = venizen if case["kind"] == "venizen" else kudurax
    return module, module.Config.from_dict(design_config(case), case["prompt"] + case["new"] + 28)


def design_tensor(case, seed, shapes, name):
    """A tensor of the checkpoint, in bfloat16 where it is a matrix."""
    shape = shapes[name]
    if name == "embed":
        return (design_tensor(case, seed, shapes, "head")[following(case, seed)] * math.sqrt(case["width"])).to(torch.bfloat16)
    if name.endswith("act"):
        return torch.tensor([0.7, 0.2, 0.1, 0.0], device=DEV)
    if len(shape) == 1:
        centre = 0.0 if name.endswith((".b", "w0")) else 1.0
        return (centre + 0.1 * normal(seed, name, *shape)).to(torch.bfloat16)
    return (normal(seed, name, *shape) * shape[-1] ** -0.5).to(torch.bfloat16)


def rms(x, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt()


def attend(q, k, v, scale, hidden, talk=None):
    """q [T, H, d], k [T, G, d], v [T, G, e] -> [T, H e]."""
    r = q.shape[1] // k.shape[1]
    q, k, v = q.transpose(0, 1), k.transpose(0, 1).repeat_interleave(r, 0), v.transpose(0, 1).repeat_interleave(r, 0)
    s = q @ k.transpose(1, 2) * scale
    if talk is not None:
        s = (talk @ s.flatten(1)).reshape(s.shape)
    return (torch.softmax(s.masked_fill_(hidden, -math.inf), -1) @ v).transpose(0, 1).flatten(1)


def venizen_exact(case, seed, get, tokens):
    cfg, T, eps, t = design_config(case), len(tokens), 1e-5, torch.arange(len(tokens), device=DEV)
    back = t[:, None] - t[None]

    def turned(x, rot):
        a, b = x.chunk(2, -1)
        angle = t[:, None] * float(rot["base"]) ** (-2.0 * torch.arange(rot["dims"] // 2, device=DEV).double() / rot["dims"])
        c, s = angle.cos()[:, None], angle.sin()[:, None]
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    def parallel(h, pre, m):
        a, r = m["left"], m["right"]
        heads = lambda name, n: (h @ get(pre + name).T).reshape(T, n, -1)
        q = turned(rms(heads("left.q", a["heads"]), eps) * get(pre + "left.q.norm"), a["rot"])
        k = turned(rms(heads("left.k", a["kv_heads"]), eps) * get(pre + "left.k.norm"), a["rot"])
        hidden = (back < 0) | ((back >= a["mask"]["size"]) & (t[None] >= a["mask"]["keep_first"]))
        left = attend(q, k, heads("left.v", a["kv_heads"]), a["scale"], hidden, get(pre + "left.talk")) @ get(pre + "left.o").T
        q, k = turned(heads("right.q", r["heads"]), r["rot"]), turned(heads("right.k", r["heads"]), r["rot"]) * r["dim"] ** -0.5
        v, outs = heads("right.v", r["heads"]), []
        for i, decay in enumerate(r["decay"]):
            outs.append((q[:, i] @ k[:, i].T * torch.where(back >= 0, decay ** back.clamp(min=0).double(), 0.0)) @ v[:, i])
        o = rms(torch.stack(outs, 1), eps).flatten(1) * torch.nn.functional.silu(h @ get(pre + "right.g").T)
        return left + o @ get(pre + "right.o").T

    def delta(h, pre, m):
        heads = lambda x: x.reshape(T, m["heads"], m["dim"])
        r, k, v = (heads(h @ get(pre + n).T) for n in "rkv")
        w = heads(torch.exp(-math.exp(-0.5) * torch.sigmoid(torch.tanh(h @ get(pre + "w1").T) @ get(pre + "w2").T + get(pre + "w0"))))
        u = k / (k.square().sum(-1, keepdim=True) + 1e-6).sqrt()
        au = heads(torch.sigmoid(h @ get(pre + "a").T + get(pre + "a.b"))) * u
        S, outs = h.new_zeros(m["heads"], m["dim"], m["dim"]), []
        for i in range(T):
            S = w[i, :, :, None] * S - au[i, :, :, None] * (u[i, :, None] @ S) + k[i, :, :, None] * v[i, :, None]
            outs.append((r[i, :, None] @ S)[:, 0])
        o = rms(torch.stack(outs), eps).flatten(1) * get(pre + "norm") * torch.sigmoid(h @ get(pre + "g").T)
        return o @ get(pre + "o").T

    order = [(0, False), (1, False), (2, False), (3, False), (2, True), (3, False)]
    x = emb = get("embed")[tokens]
    for i, again in order:
        x = x + emb if again else x
        layer, pre = cfg["layers"][i], f"l{i}."
        x = x + (parallel if layer["type"] == "parallel" else delta)(rms(x, eps) * get(pre + "norm1"), pre + "mix.", layer["mixer"])
        if layer["mlp"]:
            z, c = (rms(x, eps) * get(pre + "norm2")) @ get(pre + "mlp.up").T, get(pre + "mlp.act")
            x = x + (sum(c[p - 1] * rms(z ** p, eps) for p in (1, 2, 3)) + c[3]) @ get(pre + "mlp.down").T
    return (rms(x[-1:], eps) * get("final.norm")) @ get("head").T


def kudurax_exact(case, seed, get, tokens):
    cfg, T, eps, F = design_config(case), len(tokens), 1e-5, torch.nn.functional
    norm = lambda x, name: F.layer_norm(x, x.shape[-1:], get(name), get(name + ".b"), eps)
    rot = cfg["layers"][0]["mixer"]["rot"]
    s, dims = rot["scaling"], rot["dims"]
    turns = lambda n: dims * math.log(s["original"] / (2 * math.pi * n)) / (2 * math.log(rot["base"]))
    lo, hi = max(math.floor(turns(s["fast"])), 0), min(math.ceil(turns(s["slow"])), dims - 1)
    i = torch.arange(dims // 2, device=DEV).double()
    slowed = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    angle = torch.arange(T, device=DEV)[:, None] * (rot["base"] ** (-2 * i / dims) * (slowed / s["factor"] + 1 - slowed))
    grown = 0.1 * math.log(s["factor"]) + 1
    cos, sin = grown * angle.cos()[:, None], grown * angle.sin()[:, None]

    def turned(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    gated = lambda h, pre: (F.silu(h @ get(pre + "gate").T) * (h @ get(pre + "up").T)) @ get(pre + "down").T
    later = torch.ones(T, T, dtype=torch.bool, device=DEV).triu(1)
    x, kept = get("embed")[tokens], {}
    for i, layer in enumerate(cfg["layers"]):
        pre, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
        h = norm(x, pre + "norm1")
        if m.get("kv_from") is None:
            z = h @ get(pre + "mix.dkv").T
            kept[i] = rms(z[:, :m["kv_rank"]], eps) * get(pre + "mix.dkv.norm"), turned(z[:, None, m["kv_rank"]:])
        c, kr = kept[i if m.get("kv_from") is None else m["kv_from"]]
        H, d = m["heads"], m["dim"]
        q = (h @ get(pre + "mix.q").T).reshape(T, H, -1)
        q = torch.cat([q[..., :d], turned(q[..., d:])], -1)
        k = torch.cat([(c @ get(pre + "mix.uk").T).reshape(T, H, d), kr.expand(T, H, -1)], -1)
        o = attend(q, k, (c @ get(pre + "mix.uv").T).reshape(T, H, -1), m["scale"], later).reshape(T, H, -1)
        x = x + (o * torch.sigmoid(h @ get(pre + "mix.g").T)[..., None]).flatten(1) @ get(pre + "mix.o").T
        h = norm(x, pre + "norm2")
        if mlp["kind"] == "dense":
            x = x + F.relu(h @ get(pre + "mlp.up").T).square() @ get(pre + "mlp.down").T
            continue
        p, ids = (h @ get(pre + "mlp.router").T).topk(mlp["router"]["top"], -1)
        p, y = torch.softmax(p, -1), torch.sigmoid(h @ get(pre + "mlp.shared.sg").T) * gated(h, pre + "mlp.shared.")
        for e in range(mlp["router"]["experts"]):
            t, slot = (ids == e).nonzero(as_tuple=True)
            if len(t):
                y.index_add_(0, t, gated(h[t], f"{pre}mlp.e{e}.") * p[t, slot, None])
        x = x + y
    return norm(x[-1:], "final.norm") @ get("head").T


# ------------------------------------------------------------------------------------------------- what is measured
def prepare(case, seed):
    kind = case["kind"]
    if kind == "matmul":
        return {"case": case, "mm": QMatMul.from_qtensor(weight(case["fmt"], matmul_weight(case, seed), case["n"], case["k"])), "x": matmul_input(case, seed)}
    if kind == "moe":
        experts = [weight(case["fmt"], blocks(case["fmt"], seed, name, *shape), *shape) for name, shape in moe_shapes(case).items()]
        return {"case": case, "layer": FusedMoeGGUF(moe_router(case, seed), *experts, True, case["top"]), "x": moe_input(case, seed)}
    if kind == "llama":
        tensors = {}
        for name, fmt, shape, b in llama_blocks(case, seed):
            tensors[name] = (FORMATS[fmt], b.cpu().numpy().tobytes())
            if name == "output":
                tensors["tok_embeddings"] = embedding_for(values(fmt, b, *shape), case, seed)
        for name in ["norm"] + [f"blk.{i}.{n}_norm" for i in range(case["layers"]) for n in ("attention", "ffn")]:
            tensors[name] = norm_weight(case, seed, name)
        model = ModelWeights.from_blocks(llama_config(case), tensors, DEV)
    else:
        module, cfg = design(case)
        shapes = module.tensor_shapes(cfg)
        model = module.Model(cfg, lambda name: design_tensor(case, seed, shapes, name), DEV, "bfloat16")
    prompt = prompt_of(case, seed).to(torch.int32)
    return {"case": case, "model": model, "prompt": prompt[None], "prompt_list": prompt.tolist()}


def run(state):
    case = state["case"]
    if case["kind"] == "matmul":
        return state["mm"].forward(state["x"])
    if case["kind"] == "moe":
        return state["layer"].forward(state["x"], case["tokens"] > 16)
    model, cache = state["model"], state["model"].cache
    out = {}
    if case["new"]:
        out["tokens"] = torch.tensor(model.generate_greedy(state["prompt_list"], case["new"])["tokens"])
        if case["kind"] == "llama":
            out["logits"] = model.logits
    else:
        out["logits"] = model.forward(state["prompt"], 0)
    out["cache"] = [t for pair in cache.kv for t in pair] + cache.rows + cache.states
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "matmul":
        return product(case["fmt"], matmul_input(case, seed), values(case["fmt"], matmul_weight(case, seed), case["n"], case["k"]))
    if kind == "moe":
        return moe_exact(case, seed)
    if kind == "llama":
        return llama_exact(case, seed)
    # the caches are laid out as their kernels read them, and generated tokens bring no logits
    shapes = design(case)[0].tensor_shapes(design(case)[1])
    get = lambda name: design_tensor(case, seed, shapes, name).double()
    if case["new"]:
        return None
    return {"logits": (venizen_exact if kind == "venizen" else kudurax_exact)(case, seed, get, prompt_of(case, seed)), "cache": None}


def weight_bytes(fmt, elements):
    size, nbytes = BLOCK_BYTES[fmt]
    return elements // size * nbytes


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        n, k, rows, wide = case["n"], case["k"], case["rows"], 4 if case["dtype"] == "f32" else 2
        return {"bytes": weight_bytes(case["fmt"], n * k) + wide * rows * (n + k), "flops": 2.0 * rows * n * k}
    if kind == "moe":
        E, top, h, i, t = (case[key] for key in ("experts", "top", "hidden", "inter", "tokens"))
        hit = E * (1 - (1 - top / E) ** t)
        return {"bytes": int(hit * 3 * weight_bytes(case["fmt"], i * h)) + 4 * E * h + 2 * (4 if case["dtype"] == "f32" else 2) * t * h, "flops": 2.0 * t * h * (3 * top * i + E)}
    prompt, steps = case["prompt"], max(case["new"] - 1, 0)
    if kind == "llama":
        h, f, layers, kv = case["hidden"], case["ffn"], case["layers"], case["kv_heads"] * (case["hidden"] // case["heads"])
        q4, q6 = h * (2 * h + kv + 2 * f), h * (kv + f)
        per_pass = layers * (weight_bytes("q4_k", q4) + weight_bytes("q6_k", q6)) + weight_bytes("q4_k", case["vocab"] * h)
        keys = prompt * (prompt + 1) / 2 + sum(prompt + 1 + s for s in range(steps))
        cached = layers * 2 * 4 * kv * (prompt + sum(prompt + 1 + s for s in range(steps)))
        return {"bytes": per_pass * (1 + steps) + cached, "flops": 2.0 * (prompt + steps) * layers * (q4 + q6) + 2.0 * (1 + steps) * case["vocab"] * h + 4.0 * layers * h * keys}
    w, head = case["width"], case["vocab"] * case["width"]
    if kind == "venizen":
        # per layer run: left q, k, v, o and right q, k, v, g, o of the parallel mixer and its feed-forward; r, k, v, g, a, o of the delta mixer
        dense, attended = 3 * (2.5 * w * w + 2.5 * w * w + 7 * w * w) + 3 * 6 * w * w, 3 * 4.0 * w
        token = reached = dense
    else:
        kept = w * 576
        mixers = 4 * (w // 128 * 192 * w + 2 * w * 512 + w * w) + 2 * kept
        ff, shared, expert = 2 * 7 * w * w, 2 * 3 * w * (w * 11 // 8), 2 * 3 * w * (w * 11 // 16)
        token, attended = mixers + ff + shared + 6 * expert, 4 * (w // 128) * 2.0 * (192 + 128)
        reached = mixers + ff + shared + 64 * (1 - (1 - 6 / 64) ** prompt) * expert
    keys = prompt * (prompt + 1) / 2 + sum(prompt + 1 + s for s in range(steps))
    return {"bytes": int(2 * (reached + head) + steps * 2 * (token + head)), "flops": 2.0 * (prompt + steps) * token + 2.0 * (1 + steps) * head + attended * keys}


def tolerance(case):
    """About four times what the path is off from ``exact`` or from itself with its sums in another order."""
    if case["kind"] == "matmul":
        return {"f32": {"rel": 2e-6, "max": 2e-5}, "f16": {"rel": 1e-3, "max": 2e-3}, "bf16": {"rel": 7e-3, "max": 1.6e-2}}[case["dtype"]]
    if case["kind"] == "moe":
        # a last bit of an f32 sum now and then moves a value between two int8 in front of the down projection
        return {"rel": 6e-4, "max": 0.03} if case["dtype"] == "f32" else {"rel": 7e-3, "max": 0.04}
    if case["kind"] == "llama":
        # ... and here in front of every product of every layer: 1.4e-2 after four layers
        return {"rel": 0.03, "max": 0.25}
    # bfloat16 between products: 0.5e-2; where two experts' logits are equal to that, a token may take the other expert
    return {"rel": 0.02, "max": 0.1} if case["kind"] == "venizen" else {"rel": 0.03, "max": 0.9}
