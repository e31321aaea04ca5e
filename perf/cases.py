"""
The work a program gives this package, as a list of measurable cases: the MoE block from one
decoded token to a long prefill, forward and forward + backward, in each dtype it takes; the
prefill's attention; the tied head's loss; and the whole decoder's prefill.

Every case uses nanoSpeaker's own sizes (d_model 576, 76 routed + 2 shared SwiGLU experts of
width 128, top-6; 9 query and 3 key/value heads of 64; vocabulary 32768; 20 layers, window
512 with every fourth layer global).  What varies over the real range is the number of
tokens, the dtype, the direction, the routing's skew and how the call is issued: programs
with fixed shapes (a decode loop, a training step) keep a captured graph of the call and
replay it, the others call the module.

    listed()            the cases, plain dicts
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs, weights and handles a program holds before the call
    run(state)          one pass through the public entry points, returning its outputs whole
    exact(case, seed)   the same outputs in 64 bits, in plain torch
    work(case)          the bytes and operations a pass cannot do without
    tolerance(case)     how far another correct implementation may be off
"""

import math

import torch

from nanospeaker_amd import MoEBlock, moe_kernel
from nanospeaker_amd.decoder import Attention, Decoder, DecoderConfig, RMSNorm, Rotary
from nanospeaker_amd.head import linear_cross_entropy

D, E, S, K, H = 576, 76, 2, 6, 128      # d_model, routed, shared, top-k, expert width
HQ, HKV, DH = 9, 3, 64                  # query heads, key/value heads, head width
VOCAB, LAYERS, WINDOW = 32768, 20, 512
AUX_COEF, EPS, STD = 1e-2, 1e-6, 0.02
DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
MAX_TOKENS = {"decode": 256, "prompt": 32768, "train": 16384}
# fp32 runs at a tenth of the 16-bit matrix rate and is used for checks and small runs.
MAX_TOKENS_FP32 = 2048


def _block_case(kind, tokens, dtype="bf16", graph=False, skew=False, master=False, name=None):
    """kind: "decode" (eval forward), "prompt" (eval forward of x + block(norm(x))) or
    "train" (forward + backward, every gradient); graph: the call is captured once and
    replayed; skew: Zipf-like expert load; master: fp32 parameters under 16-bit tokens."""
    c = {"what": kind, "tokens": tokens, "dtype": dtype, "graph": graph, "skew": skew,
         "master": master}
    return {"name": name, **c} if name else c


def listed():
    return [
        # One sequence being generated: one token per call, issued from Python.
        _block_case("decode", 1, name="decode_1"),
        # A serving loop's decode step over 64 sequences, captured once with the weights'
        # packed copies shared into the graph.
        _block_case("decode", 64, graph=True, name="decode_64_graph"),
        # A prompt of ragged length through one layer's FFN half.
        _block_case("prompt", 1531, name="prompt_1531"),
        # A small micro-batch in fp16, one token short of a whole number of tiles.
        _block_case("train", 2047, "fp16", graph=True, name="train_2047_fp16_graph"),
        # The training shape (8 sequences of 1024), bf16, as a captured step.
        _block_case("train", 8192, graph=True, name="train_8192_graph"),
        # The same step with fp32 master weights under bf16 tokens, as mixed-precision
        # training keeps them: the casts and the gradients' casts back belong to the step.
        _block_case("train", 8192, graph=True, master=True, name="train_8192_master_graph"),
        # A double batch with a skewed router (the hottest expert takes ~15 % of the pairs).
        _block_case("train", 16384, skew=True, name="train_16384_skew"),
        # Full fp32, as the checks and small experiments of a training project run it.
        _block_case("train", 2048, "fp32", name="train_2048_fp32"),
        # One layer's FFN half in the long prefill: 4 sequences of 8192 tokens.
        _block_case("prompt", 32768, name="prompt_32768"),
        # A global-attention layer of a prefill, two prompts of ragged length.
        {"name": "attention_2x5003", "what": "attention", "batch": 2, "seq": 5003, "window": 0,
         "dtype": "bf16"},
        # The training loss of one long sequence: tied head, cross-entropy, both gradients.
        {"name": "head_8191", "what": "head", "tokens": 8191, "dtype": "bf16"},
        # The whole decoder: a prefill of 4 x 8192 tokens to logits.
        {"name": "prefill_4x8192", "what": "decoder", "batch": 4, "seq": 8192,
         "layers": LAYERS, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    what = rng.choice(["decode", "decode", "prompt", "prompt", "train", "train", "train",
                       "attention", "head", "decoder"])
    if what == "decode":
        return _block_case("decode", _log_int(rng, 1, MAX_TOKENS["decode"]),
                           rng.choice(["bf16", "bf16", "fp16"]), graph=rng.random() < 0.5)
    if what == "prompt":
        return _block_case("prompt", _log_int(rng, 16, MAX_TOKENS["prompt"]),
                           rng.choice(["bf16", "bf16", "fp16"]))
    if what == "train":
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        most = MAX_TOKENS_FP32 if dtype == "fp32" else MAX_TOKENS["train"]
        kind = rng.choice(["plain", "plain", "skew", "master"]) if dtype != "fp32" else "plain"
        # a step too short to hide its own launches is captured
        tokens = _log_int(rng, 128, most)
        return _block_case("train", tokens, dtype, graph=dtype != "fp32" and tokens <= 8192,
                           skew=kind == "skew", master=kind == "master")
    if what == "attention":
        seq = _log_int(rng, 64, 8192)
        return {"what": "attention", "batch": rng.randint(1, 4), "seq": seq,
                "window": rng.choice([0, WINDOW]), "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    if what == "head":
        return {"what": "head", "tokens": _log_int(rng, 128, 8191),
                "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    return {"what": "decoder", "batch": rng.randint(1, 4), "seq": _log_int(rng, 128, 8192),
            "layers": LAYERS, "dtype": "bf16"}


# ---- inputs -------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(1_000_003 * int(seed) + 17)


def _randn(gen, *shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=gen, device=DEV) * scale).to(dtype)


def _block_inputs(case, seed):
    """Parameters ~ N(0, 0.02) in the block's order, x and the upstream gradient ~ N(0, 1),
    a norm gain near one, and for a skewed router the experts' offsets: logits that fall by
    0.36 per e-fold of popularity rank give the load Zipf(1.2) has when no token may take
    one expert twice; which expert is popular differs from seed to seed."""
    gen, dt = _gen(seed), DTYPES[case["dtype"]]
    pdt = torch.float32 if case["master"] else dt
    n = case["tokens"]
    shapes = {"W_r": (D, E), "W_in": (E, D, 2 * H), "W_out": (E, H, D),
              "W_sh_in": (S, D, 2 * H), "W_sh_out": (S, H, D)}
    p = {k: _randn(gen, *s, dtype=pdt, scale=STD) for k, s in shapes.items()}
    x, g = _randn(gen, n, D, dtype=dt), _randn(gen, n, D, dtype=dt)
    gamma = (1.0 + _randn(gen, D, dtype=torch.float32, scale=0.1)).to(dt)
    bias = None
    if case["skew"]:
        rank = torch.randperm(E, generator=gen, device=DEV).float() + 1.0
        bias = 1.2 - 0.36 * rank.log()
    return p, x, g, gamma, bias


def _captured(fn):
    """fn() captured once in a HIP graph, after a warm-up on a side stream: (graph, outputs)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def _prepare_block(case, seed):
    p, x, g, gamma, bias = _block_inputs(case, seed)
    with torch.device(DEV):
        m = MoEBlock(D, E, d_ff=3 * H // 2, top_k=K, n_shared=S, capacity_factor=None,
                     aux_loss_coef=AUX_COEF, std=STD, fused=False)
    m = m.to(torch.float32 if case["master"] else x.dtype)
    with torch.no_grad():
        m.router.W.copy_(p["W_r"])
        for name in ("W_in", "W_out", "W_sh_in", "W_sh_out"):
            getattr(m, name).copy_(p[name])
    params = [m.router.W, m.W_in, m.W_out, m.W_sh_in, m.W_sh_out]
    norm = None
    if case["what"] == "train":
        m.train()
        xg = x.requires_grad_(True)
        one = torch.ones((), dtype=torch.float32, device=DEV)

        def call():
            if bias is None:
                out, aux = m(xg), m.aux_loss
                counts = m.expert_counts
            else:
                out, aux, counts, _, _ = moe_kernel.block_forward(
                    xg, *params, None, None, None, None, K, True, True, "silu", AUX_COEF,
                    logit_bias=bias)
            grads = torch.autograd.grad([out, aux], [xg] + params, [g, one])
            return {"out": out.detach(), "aux": aux.detach(), "counts": counts,
                    "grads": list(grads)}
    else:
        m.eval()
        if case["what"] == "prompt":
            norm = RMSNorm(D, EPS).to(device=DEV, dtype=x.dtype)
            with torch.no_grad():
                norm.gamma.copy_(gamma)

        def call():
            with torch.no_grad():
                out = m(x) if norm is None else m.forward_residual(x, norm)
            return {"out": out, "counts": m.expert_counts}

    state = {"call": call, "keep": (m, norm)}
    if case["graph"]:
        if case["what"] == "train":
            graph, out = _captured(call)
        else:
            # the weights do not change while a decode loop runs: its graph reads the packs
            call()
            before = moe_kernel.PACKS.share_with_graphs
            moe_kernel.PACKS.share_with_graphs = True
            try:
                graph, out = _captured(call)
            finally:
                moe_kernel.PACKS.share_with_graphs = before
        state.update(graph=graph, out=out)
    return state


def _attention_inputs(case, seed):
    gen, dt = _gen(seed), DTYPES[case["dtype"]]
    w = {"W_q": (D, HQ * DH), "W_k": (D, HKV * DH), "W_v": (D, HKV * DH)}
    p = {k: _randn(gen, *s, dtype=dt, scale=STD) for k, s in w.items()}
    p["W_O"] = _randn(gen, HQ * DH, D, dtype=dt, scale=STD / math.sqrt(2 * LAYERS))
    for k in ("q", "k"):
        p[k] = (1.0 + _randn(gen, DH, dtype=torch.float32, scale=0.1)).to(dt)
    shape = (case["batch"], case["seq"], D)
    x, z = _randn(gen, *shape, dtype=dt), _randn(gen, *shape, dtype=dt)
    return p, x, z


def _prepare_attention(case, seed):
    p, x, z = _attention_inputs(case, seed)
    cfg = DecoderConfig()
    with torch.device(DEV):
        att = Attention(cfg, Rotary(DH, cfg.rope_base), case["window"] or None)
    att = att.to(x.dtype).eval()
    with torch.no_grad():
        for name in ("W_q", "W_k", "W_v", "W_O"):
            getattr(att, name).copy_(p[name])
        att.q_norm.gamma.copy_(p["q"])
        att.k_norm.gamma.copy_(p["k"])

    def call():
        with torch.no_grad():
            return {"out": att.forward_residual(x, z)}

    return {"call": call, "keep": att}


def _head_inputs(case, seed):
    """Normed hidden states (unit rows), the embedding matrix and the next tokens."""
    gen, dt = _gen(seed), DTYPES[case["dtype"]]
    h = _randn(gen, case["tokens"], D, dtype=dt)
    W = _randn(gen, VOCAB, D, dtype=dt, scale=STD)
    y = torch.randint(0, VOCAB, (case["tokens"],), generator=gen, device=DEV)
    return h, W, y


def _prepare_head(case, seed):
    h, W, y = _head_inputs(case, seed)
    h.requires_grad_(True)
    W.requires_grad_(True)

    def call():
        loss = linear_cross_entropy(h, W, y)
        dh, dW = torch.autograd.grad(loss, [h, W])
        return {"loss": loss.detach(), "dh": dh, "dW": dW}

    return {"call": call}


def _prepare_decoder(case, seed):
    torch.manual_seed(1_000_003 * int(seed) + 29)
    cfg = DecoderConfig(n_layers=case["layers"])
    with torch.device(DEV):
        model = Decoder(cfg)
        idx = torch.randint(0, VOCAB, (case["batch"], case["seq"]))
        # Embedding rows of unit scale: a trained residual stream is large beside one
        # layer's update, a freshly initialised one (0.02) is smaller than it.
        torch.nn.init.normal_(model.embed.weight)
    model = model.to(DTYPES[case["dtype"]]).eval()

    def call():
        with torch.no_grad():
            return {"logits": model(idx)}

    return {"call": call, "keep": model}


_PREPARE = {"attention": _prepare_attention, "head": _prepare_head, "decoder": _prepare_decoder}


def prepare(case, seed):
    return _PREPARE.get(case["what"], _prepare_block)(case, seed)


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return state["call"]()


# ---- the same results in 64 bits ------------------------------------------------------------

def _f64(t):
    return t.detach().double()


def _rms64(x, gamma):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gamma


def _exact_block(case, seed):
    """The router's logits are rounded to the tokens' dtype, as the block's definition has
    it; everything after them is in 64 bits.  Equal logits are taken in CPU topk's order."""
    p, x, g, gamma, bias = _block_inputs(case, seed)
    dt = x.dtype
    train, prompt = case["what"] == "train", case["what"] == "prompt"
    W_r, W_in, W_out, W_si, W_so = (
        _f64(p[k].to(dt)).requires_grad_(train)
        for k in ("W_r", "W_in", "W_out", "W_sh_in", "W_sh_out"))
    x64 = _f64(x).requires_grad_(train)
    xn = x64
    if prompt:
        xn = _rms64(x64, _f64(gamma))
    raw = (xn.to(dt).double() if prompt else xn) @ W_r
    if bias is not None:
        raw = raw + bias.double()
    logits = raw + (raw.detach().to(dt).double() - raw.detach())
    idx = logits.detach().float().cpu().topk(K, dim=-1).indices.to(DEV)
    probs = logits.softmax(-1)
    w = probs.gather(1, idx)
    w = w / w.sum(-1, keepdim=True)
    counts = torch.bincount(idx.reshape(-1), minlength=E)

    def glu(v, a, b):
        gate, up = (v @ a).chunk(2, dim=-1)
        return (torch.nn.functional.silu(gate) * up) @ b

    out = torch.zeros_like(x64)
    for s in range(S):
        out = out + glu(xn, W_si[s], W_so[s])
    for e in range(E):
        tok, slot = (idx == e).nonzero(as_tuple=True)
        if tok.numel():
            y = glu(xn.index_select(0, tok), W_in[e], W_out[e]) * w[tok, slot][:, None]
            out = out.index_add(0, tok, y)
    if prompt:
        out = out + x64
    if not train:
        return {"out": out, "counts": None}
    aux = AUX_COEF * E * (counts / counts.sum() * probs.mean(0)).sum()
    grads = torch.autograd.grad((out * g.double()).sum() + aux, [x64, W_r, W_in, W_out, W_si, W_so])
    return {"out": out.detach(), "aux": aux.detach(), "counts": None, "grads": list(grads)}


def _exact_attention(case, seed):
    p, x, z = _attention_inputs(case, seed)
    B, T, w = case["batch"], case["seq"], case["window"]
    p = {k: _f64(v) for k, v in p.items()}
    z, half = _f64(z), DH // 2
    inv = DecoderConfig().rope_base ** (
        -torch.arange(half, dtype=torch.float32, device=DEV) * 2.0 / DH)
    ang = torch.arange(T, dtype=torch.float32, device=DEV)[:, None] * inv[None, :]
    cos, sin = ang.double().cos(), ang.double().sin()

    def heads(W, n, gain=None):
        v = (z @ W).view(B, T, n, DH).transpose(1, 2)
        if gain is None:
            return v
        v = _rms64(v, gain)
        a, b = v[..., :half], v[..., half:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)

    q, k, v = heads(p["W_q"], HQ, p["q"]), heads(p["W_k"], HKV, p["k"]), heads(p["W_v"], HKV)
    o = torch.empty(B, T, HQ * DH, dtype=torch.float64, device=DEV)
    step = 2048
    for b in range(B):
        for h in range(HQ):
            kv = h // (HQ // HKV)
            for s in range(0, T, step):
                e = min(T, s + step)
                lo = max(0, s - w + 1) if w else 0
                qi = torch.arange(s, e, device=DEV)[:, None]
                kj = torch.arange(lo, e, device=DEV)[None, :]
                sc = q[b, h, s:e] @ k[b, kv, lo:e].t() / math.sqrt(DH)
                dead = (kj > qi) | ((qi - kj >= w) if w else torch.zeros_like(kj > qi))
                sc = sc.masked_fill(dead, float("-inf")).softmax(-1)
                o[b, s:e, h * DH:(h + 1) * DH] = sc @ v[b, kv, lo:e]
    return {"out": _f64(x) + o @ p["W_O"]}


def _exact_head(case, seed):
    h, W, y = _head_inputs(case, seed)
    h, W = _f64(h), _f64(W)
    n, step = h.shape[0], 1024
    loss = torch.zeros((), dtype=torch.float64, device=DEV)
    dh, dW = torch.empty_like(h), torch.zeros_like(W)
    for s in range(0, n, step):
        hc, yc = h[s:s + step], y[s:s + step]
        logits = hc @ W.t()
        lse = logits.logsumexp(-1, keepdim=True)
        loss = loss + (lse[:, 0] - logits.gather(1, yc[:, None])[:, 0]).sum()
        pr = (logits - lse).exp()
        pr.scatter_add_(1, yc[:, None], torch.full_like(lse, -1.0))
        dh[s:s + step] = pr @ W / n
        dW += pr.t() @ hc / n
    return {"loss": loss / n, "dh": dh, "dW": dW}


def exact(case, seed):
    if case["what"] == "attention":
        return _exact_attention(case, seed)
    if case["what"] == "head":
        return _exact_head(case, seed)
    if case["what"] == "decoder":
        # Rounding decides which experts a token takes from the second layer on: the whole
        # decoder has no 64-bit counterpart.
        return None
    return _exact_block(case, seed)


# ---- what a pass cannot do without ----------------------------------------------------------

def _attention_flops(B, T, window):
    """4 x head width operations per (head, query, visible key)."""
    keys = T * (T + 1) // 2
    if window and window < T:
        keys = window * (window + 1) // 2 + (T - window) * window
    return float(B * HQ * keys * 4 * DH)


_EXPERT_WEIGHTS = (E + S) * 3 * D * H
_QKVO_WEIGHTS = 2 * D * (HQ + HKV) * DH


def _block_work(tokens, es, train, residual, master=False):
    rows = tokens * (K + S)
    flops = rows * 6.0 * D * H + 2.0 * tokens * D * E
    # a short call needs only the experts that its tokens take
    routed = min(E, tokens * K)
    weights = ((routed + S) * 3 * D * H + D * E) * (4 if master else es)
    nbytes = weights + 2 * tokens * D * es
    if train:
        flops *= 3
        nbytes += (_EXPERT_WEIGHTS + D * E) * (4 if master else es) + 2 * tokens * D * es
    return nbytes, flops


def work(case):
    es = 4 if case["dtype"] == "fp32" else 2
    if case["what"] == "attention":
        B, T = case["batch"], case["seq"]
        return {"bytes": float(3 * B * T * D * es + _QKVO_WEIGHTS * es),
                "flops": 2.0 * B * T * _QKVO_WEIGHTS + _attention_flops(B, T, case["window"])}
    if case["what"] == "head":
        n = case["tokens"]
        return {"bytes": float(2 * (n + VOCAB) * D * es + 8 * n), "flops": 6.0 * n * VOCAB * D}
    if case["what"] == "decoder":
        B, T = case["batch"], case["seq"]
        n = B * T
        moe_bytes, moe_flops = _block_work(n, es, False, True)
        moe_weights = moe_bytes - 2 * n * D * es
        att = sum(_attention_flops(B, T, 0 if i % 4 == 0 else WINDOW)
                  for i in range(case["layers"]))
        flops = case["layers"] * (moe_flops + 2.0 * n * _QKVO_WEIGHTS) + att
        return {"bytes": float(case["layers"] * (moe_weights + _QKVO_WEIGHTS * es) + 8 * n
                               + VOCAB * D * es + n * VOCAB * es),
                "flops": flops + 2.0 * n * VOCAB * D}
    nbytes, flops = _block_work(case["tokens"], es, case["what"] == "train",
                                case["what"] == "prompt", case["master"])
    return {"bytes": float(nbytes), "flops": flops}


def tolerance(case):
    """About four times what a pass is off from the same inputs in 64 bits: 3.9e-3 in bf16,
    4.8e-4 in fp16, 8.7e-7 in fp32 (the largest over a pass's outputs), and for single
    values 0.06, 4e-3 and 7e-6 of the output's scale.  The whole decoder: its
    logits move by 6.4e-3 and 0.08 when every attention layer sums in another order."""
    if case["what"] == "decoder":
        return {"rel": 2.5e-2, "max": 0.35}
    if case["dtype"] == "fp32":
        return {"rel": 4e-6, "max": 5e-5}
    if case["dtype"] == "fp16":
        return {"rel": 2e-3, "max": 4e-2}
    return {"rel": 1.5e-2, "max": 0.25}
