"""The work that users of this framework have it do, as cases that can be timed and compared.

The framework replaces the kernel path of a GPT-2 trainer, so the cases are that trainer's steps at
its own sizes, evaluation forwards, and the operators that callers import one by one:

  step       one optimisation step: t_loss_bkwd3_t with fresh dropout seeds, then adam_w_in_place
  forward    t_gpt2_forward_t without dropout: evaluation, scoring
  attention  attention forward and backward on [B, H, 3, T, 64]
  rowwise    LayerNorm, GELU and dropout, each forward and backward
  head       LM head product, cross-entropy forward and backward, the head's two gradient products
  ffn        feed-forward block, forward and backward
  matmul     t_matmul_t

The model is GPT-2 small (12 blocks, 768 wide, 12 heads, feed-forward 3072).  Token ids follow Zipf's
law over the vocabulary, as words of a text do; id 0 is padding.  Masks are the collator's: lower
triangular ("causal"), with padded tails ("padded"), or with several documents per row ("packed").
"""
import importlib
import math

import torch

mt = importlib.import_module("pre-tjax_amd.model_triton")
lo = importlib.import_module("pre-tjax_amd.loss_and_optimizer_triton")

D, HEADS, F, LAYERS, DH = 768, 12, 3072, 12, 64
VOCABS = (50257, 35374)          # GPT-2's own, and that of the trainer's corpus
MASKS = ("causal", "padded", "packed")
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # The benchmark's step: batch 16 at the full context, bf16 on fp32 master weights.
        {"name": "step_bf16_b16_t1024", "kind": "step", "dtype": "bf16", "b": 16, "t": 1024, "v": 50257, "mask": "causal"},
        # The trainer's own configuration: fp32, batch 8 of 512 tokens, one padded document per row.
        {"name": "step_fp32_b8_t512", "kind": "step", "dtype": "fp32", "b": 8, "t": 512, "v": 35374, "mask": "padded"},
        # A batch of packed documents whose row count fills no tile evenly.
        {"name": "step_bf16_b7_t448", "kind": "step", "dtype": "bf16", "b": 7, "t": 448, "v": 35374, "mask": "packed"},
        # A micro-batch as fine-tuning and debugging runs use it: launches count.
        {"name": "step_bf16_b2_t256", "kind": "step", "dtype": "bf16", "b": 2, "t": 256, "v": 50257, "mask": "causal"},
        # Scoring one short text: the smallest call of the whole model.
        {"name": "forward_bf16_b1_t64", "kind": "forward", "dtype": "bf16", "b": 1, "t": 64, "v": 50257, "mask": "causal"},
        # An evaluation batch.
        {"name": "forward_bf16_b8_t512", "kind": "forward", "dtype": "bf16", "b": 8, "t": 512, "v": 50257, "mask": "padded"},
        # Attention alone at the full context, and at the trainer's size in fp32 with dropout.
        {"name": "attention_bf16_b8_t1024", "kind": "attention", "dtype": "bf16", "b": 8, "t": 1024, "mask": "causal", "train": False},
        {"name": "attention_fp32_b8_t512", "kind": "attention", "dtype": "fp32", "b": 8, "t": 512, "mask": "padded", "train": True},
        # The row-wise operators on the activations of 8192 tokens.
        {"name": "rowwise_bf16_8192x768", "kind": "rowwise", "dtype": "bf16", "rows": 8192, "cols": 768},
        # LM head and loss on 8192 tokens, logits in rows padded to whole 128-byte lines.
        {"name": "head_bf16_8192", "kind": "head", "dtype": "bf16", "rows": 8192, "v": 50257, "pitch": 50304},
        # A feed-forward block on an odd number of tokens.
        {"name": "ffn_bf16_3001", "kind": "ffn", "dtype": "bf16", "rows": 3001},
        # The operator's own benchmark: one fp32 product.
        {"name": "matmul_fp32_4096x3072x768", "kind": "matmul", "dtype": "fp32", "n": 4096, "m": 3072, "k": 768, "b_t": False},
    ]


def _log(rng, lo_, hi):
    """A whole number from lo_ to hi, spread evenly over the logarithm."""
    return min(hi, max(lo_, round(math.exp(rng.uniform(math.log(lo_), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("step",) * 4 + ("forward",) * 2 + ("attention",) * 2 + ("rowwise", "head", "ffn", "matmul"))
    dtype = rng.choice(("bf16", "bf16", "fp32"))
    c = {"kind": kind, "dtype": dtype}
    if kind in ("step", "forward", "attention"):
        t = 64 * rng.randint(1, 16)
        most = {"step": 4096, "forward": 8192, "attention": 8192}[kind] if dtype == "fp32" else 16384
        c.update(b=_log(rng, 1, min(64, most // t)), t=t, mask=rng.choice(MASKS))
        if kind == "attention":
            c["train"] = rng.random() < 0.5
        else:
            c["v"] = rng.choice(VOCABS)
    elif kind == "rowwise":
        c.update(rows=_log(rng, 64, 16384), cols=rng.choice((768, 768, _log(rng, 64, 4096))))
    elif kind == "head":
        v = rng.choice(VOCABS)
        # either padded rows or the pitch of a plain [rows, V] tensor
        c.update(rows=_log(rng, 64, 8192), v=v, pitch=rng.choice(((v + 63) // 64 * 64, (v + 63) // 64 * 64, v)))
    elif kind == "ffn":
        c.update(rows=_log(rng, 64, 16384 if dtype == "bf16" else 8192))
    else:
        c.update(n=_log(rng, 64, 4096), m=_log(rng, 64, 4096), k=_log(rng, 64, 4096), b_t=rng.random() < 0.5)
    return c


# ---- inputs ---------------------------------------------------------------------------------------

def _zipf(gen, shape, v):
    """Token ids 1 .. v-1 with probability about 1 / (id + 1)."""
    u = torch.rand(shape, generator=gen, device="cuda")
    return (torch.exp(u * math.log(v)).long()).clamp_(1, v - 1)


def _tokens_and_mask(gen, b, t, v, kind):
    """(tokens [b, t+1], mask bool [b, t, t]) as the collator builds them."""
    y = _zipf(gen, (b, t + 1), v)
    pos = torch.arange(t, device="cuda")
    mask = (pos[None, :] <= pos[:, None]).expand(b, t, t)
    if kind == "padded":         # documents of half to all of the row's length
        length = torch.randint(t // 2, t + 2, (b, 1), generator=gen, device="cuda")
        y[torch.arange(t + 1, device="cuda")[None, :] >= length] = 0
        real = y[:, :-1] != 0
        mask = mask & real[:, :, None] & real[:, None, :]
    elif kind == "packed":       # about four documents a row
        doc = torch.cumsum((torch.rand((b, t), generator=gen, device="cuda") < 3.0 / t).int(), 1)
        mask = mask & (doc[:, :, None] == doc[:, None, :])
    return y, mask.contiguous()


def _visible(c):
    """Expected number of visible (query, key) pairs of one row of the batch."""
    t = c["t"]
    return t * (t + 1) / 2 * {"causal": 1.0, "padded": 0.58, "packed": 0.37}[c["mask"]]


def _shapes(v, t):
    block = [(D,), (D,), (HEADS, 3, DH, D), (D, D), (D,), (D,), (F, D), (F,), (D, F), (D,)]
    return [[(v, D), (v,)], [(t, D)]] + [list(block) for _ in range(LAYERS)] + [[(D,), (D,)]]


def _n_params(v, t):
    return sum(math.prod(s) for grp in _shapes(v, t) for s in grp)


def _buffers(shapes, dtype):
    """The nest of parameters as views of two flat buffers (tables; blocks and final norm), every
    tensor starting at a multiple of 128 elements: what a trainer keeps to clear, save and count its
    state in one go."""
    nest, flat = [], {}
    sizes = {"tables": 0, "blocks": 0}
    part = ["tables", "tables"] + ["blocks"] * (len(shapes) - 2)
    at = []
    for p, grp in zip(part, shapes):
        for s in grp:
            at.append(sizes[p])
            sizes[p] += (math.prod(s) + 127) // 128 * 128
    for p in sizes:
        flat[p] = torch.zeros(sizes[p], dtype=dtype, device="cuda")
    at = iter(at)
    for p, grp in zip(part, shapes):
        nest.append([])
        for s in grp:
            o = next(at)
            nest[-1].append(flat[p][o:o + math.prod(s)].view(s))
    return nest, flat


def _fill(gen, nest):
    """Weights as GPT-2 is initialised, with gains and biases a little off 1 and 0."""
    for gi, grp in enumerate(nest):
        for pi, p in enumerate(grp):
            small = 2 <= gi < len(nest) - 1 and pi in (3, 8)       # projections onto the residual stream
            p.normal_(0.0, 0.02 / (math.sqrt(2 * LAYERS) if small else 1.0), generator=gen)
            if (2 <= gi < len(nest) - 1 and pi in (0, 4)) or (gi == len(nest) - 1 and pi == 0):
                p.add_(1.0)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rn = lambda *shape, scale=1.0: torch.randn(*shape, generator=gen, device="cuda").mul_(scale).to(dt)
    kind, dt = case["kind"], DTYPES[case["dtype"]]
    s = {"kind": kind}
    if kind == "step":
        shapes = _shapes(case["v"], case["t"])
        s["master"], s["master_flat"] = _buffers(shapes, torch.float32)
        _fill(gen, s["master"])
        m, s["m_flat"] = _buffers(shapes, torch.float32)
        v, s["v_flat"] = _buffers(shapes, torch.float32)
        s["moments"] = [m, v]
        s["params"], s["shadow_flat"] = s["master"], {}
        if dt != torch.float32:
            s["params"], s["shadow_flat"] = _buffers(shapes, dt)
            for p in s["shadow_flat"]:
                s["shadow_flat"][p].copy_(s["master_flat"][p])
        s["decay"] = [[p.dim() > 1 for p in grp] for grp in s["master"]]
        s["y"], s["mask"] = _tokens_and_mask(gen, case["b"], case["t"], case["v"], case["mask"])
        s["seeds"] = torch.Generator().manual_seed(seed + 1)
        s["i"] = 0
    elif kind == "forward":
        s["params"], flat = _buffers(_shapes(case["v"], case["t"]), torch.float32)
        _fill(gen, s["params"])
        if dt != torch.float32:
            s["params"] = [[p.to(dt) for p in grp] for grp in s["params"]]
        y, s["mask"] = _tokens_and_mask(gen, case["b"], case["t"], case["v"], case["mask"])
        s["y"] = y[:, :-1].contiguous()
    elif kind == "attention":
        s["qkv"] = rn(case["b"], HEADS, 3, case["t"], DH)
        s["do"] = rn(case["b"], HEADS, case["t"], DH)
        _, s["mask"] = _tokens_and_mask(gen, case["b"], case["t"], 1000, case["mask"])
        s["train"], s["seed"] = case["train"], seed % 1_000_000
    elif kind == "rowwise":
        rows, cols = case["rows"], case["cols"]
        s["x"], s["dy"] = rn(rows, cols), rn(rows, cols, scale=0.1)
        s["ln"] = (rn(cols, scale=0.1) + 1, rn(cols, scale=0.1))
        s["xf"], s["dyf"] = rn(rows, 4 * cols), rn(rows, 4 * cols, scale=0.1)
        s["seed"] = seed % 1_000_000
    elif kind == "head":
        rows, v = case["rows"], case["v"]
        s["x"], s["w"], s["b"] = rn(rows, D), rn(v, D, scale=0.02), rn(v, scale=0.02)
        s["labels"] = _zipf(gen, (rows,), v)
        s["labels"][torch.rand(rows, generator=gen, device="cuda") < 0.1] = 0     # padding
        s["logits"] = torch.empty((rows, case["pitch"]), dtype=dt, device="cuda")[:, :v]
    elif kind == "ffn":
        s["x"], s["dy"] = rn(case["rows"], D), rn(case["rows"], D, scale=0.1)
        s["w"] = (rn(F, D, scale=0.02), rn(F, scale=0.02), rn(D, F, scale=0.02), rn(D, scale=0.02))
    else:
        s["a"] = rn(case["n"], case["k"])
        s["b"] = rn(case["m"], case["k"]).t() if case["b_t"] else rn(case["k"], case["m"])
    return s


# ---- one pass -------------------------------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "step":
        i = s["i"]
        s["i"] = i + 1
        seeds = lo.sample_p_gen_aux(s["master"], s["seeds"])
        grads, (loss, acc, frac) = lo.t_loss_bkwd3_t(s["params"], s["y"], s["mask"], None, True, seeds)
        shadow = s["params"] if s["shadow_flat"] else None
        lr = 6e-4 * min(1.0, (i + 1) / 2000)                       # warm-up
        lo.adam_w_in_place(s["master"], grads, lr, (0.9, 0.95), 1e-8, s["moments"], i, 0.1, s["decay"], shadow=shadow)
        # the moments start at zero: after the first step m is a tenth of the gradient of every parameter
        return {"loss": loss, "acc": acc, "frac": frac, "w": s["master_flat"], "m": s["m_flat"], "v": s["v_flat"],
                "shadow": s["shadow_flat"]}
    if kind == "forward":
        return mt.t_gpt2_forward_t(s["params"], s["y"], s["mask"], None, False)
    if kind == "attention":
        o, acts = mt.t_scaled_dot_prod_attn_fwd3_t(s["qkv"], s["mask"], s["train"], s["seed"])
        dq, dk, dv = mt.t_scaled_dot_prod_attn_bkwd3_t(s["do"], acts, s["qkv"], s["mask"], s["train"], s["seed"])
        return {"o": o, "dq": dq, "dk": dk, "dv": dv}
    if kind == "rowwise":
        x, dy, xf, dyf, ln = s["x"], s["dy"], s["xf"], s["dyf"], s["ln"]
        return {"ln": mt.t_layernorm_fwd_t(ln, x), "ln_dx": mt.t_layernorm_bkwd2_x_t(dy, ln, x),
                "ln_dp": mt.t_layernorm_bkwd2_p_t(dy, ln, x), "gelu": mt.t_gelu_fwd_t(xf),
                "gelu_dx": mt.t_gelu_bkwd2_t(dyf, xf), "drop": mt.t_dropout_fwd_t(x, True, s["seed"]),
                "drop_dx": mt.t_dropout_bkwd2_t(dy, x, True, s["seed"])}
    if kind == "head":
        logits = mt.matmul_t(s["x"], s["w"].t(), s["b"], out=s["logits"])
        loss, count, d = lo.t_avg_cross_entropy_loss_bkwd3_t(s["labels"], logits)
        return {"logits": logits, "loss": loss, "count": count, "dlogits": d, "dx": mt.matmul_t(d, s["w"]),
                "dw": mt.matmul_t(d.t(), s["x"])}
    if kind == "ffn":
        return {"y": mt.t_tlayer_ffn_fwd_t(s["w"], s["x"]), "d": mt.t_tlayer_ffn_bkwd2_t(s["dy"], s["w"], s["x"])}
    return mt.t_matmul_t(s["a"], s["b"])


# ---- what one pass cannot do without ----------------------------------------------------------------

def work(case):
    kind, e = case["kind"], 2 if case["dtype"] == "bf16" else 4
    if kind in ("step", "forward"):
        n, v, t = case["b"] * case["t"], case["v"], case["t"]
        products = 2 * n * D * (3 * D + D + 2 * F) * LAYERS + 2 * n * D * v
        pairs = LAYERS * DH * HEADS * case["b"] * _visible(case)
        p = _n_params(v, t)
        if kind == "forward":
            return {"bytes": p * e + n * v * e + 8 * n + n * t, "flops": products + 4 * pairs}
        # weights, moments and (in bf16) the working copies read and written once; tokens and mask read
        return {"bytes": 24 * p + (4 * p if e == 2 else 0) + 8 * n + n * t, "flops": 3 * products + 14 * pairs}
    if kind == "attention":
        n = case["b"] * case["t"]
        return {"bytes": 8 * n * HEADS * DH * e + n * case["t"], "flops": 14 * DH * HEADS * case["b"] * _visible(case)}
    if kind == "rowwise":
        x = case["rows"] * case["cols"] * e
        return {"bytes": x * (2 + 3 + 2 + 2) + 4 * x * 3, "flops": 40 * case["rows"] * case["cols"]}
    if kind == "head":
        n, v = case["rows"], case["v"]
        return {"bytes": (2 * n * D + 2 * v * D + 2 * n * v) * e + 8 * n, "flops": 6 * n * v * D}
    if kind == "ffn":
        n = case["rows"]
        return {"bytes": (4 * n * D + 4 * D * F) * e, "flops": 6 * 2 * n * D * F + 2 * n * D * F}
    n, m, k = case["n"], case["m"], case["k"]
    return {"bytes": (n * k + k * m + n * m) * e, "flops": 2 * n * m * k}


def tolerance(case):
    """bf16 carries 8 bits and fp32 24; the second moments of a step are squares of its gradients,
    which come through twelve blocks."""
    if case["kind"] == "step":
        return {"rel": 2e-2} if case["dtype"] == "bf16" else {"rel": 5e-5}
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 1e-5}
