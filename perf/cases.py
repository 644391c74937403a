"""The work whose time is measured: a QLoRA training step of a Qwen2-shaped model on one GPU and
the blocks it is made of, each through the package's public entry points.

A case is a dict of plain values; its "kind" names the block, the other keys its sizes:

  dequant    NF4 double-quant weights to fp16, one launch (ops.dequant_many)
  mlp        the gate|up product with the SwiGLU, the down product with the residual, and back
             to the MLP input (linear.*, ops._glu_bwd), the weights' dequant included
  attn_input input norm with the two LoRA-dropout copies, qkv projection, LoRA, RoPE, and back
             (engine.attn_input_fwd / attn_input_bwd)
  attention  varlen causal attention over packed sequences, forward and backward
             (ops._attn_fwd / _attn_bwd)
  head       the lm_head loss with the hidden and embedding gradients, over whole rows or
             vocabulary pieces (head.full_head / chunked_head)
  step       a whole training step, forward and backward (engine.FusedQwen2.step)
  graph      the same step replayed from a HIP graph on a padded batch (engine.StepGraph)

Model widths are those of the repository's tests and benchmark: (hidden, intermediate, q heads,
kv heads, head_dim, vocabulary) of WIDTHS.
"""

import importlib
import math

import torch
from torch.utils.checkpoint import checkpoint

PKG = importlib.import_module("hack-fe30cb28-opus-5-5-ultracode_amd")
DEV = torch.device("cuda", 0)

WIDTHS = {
    "0.5B": (896, 4864, 14, 2, 64, 151936),
    "1.5B": (1536, 8960, 12, 2, 128, 151936),
    "7B": (3584, 18944, 28, 4, 128, 152064),
}
DROPOUT = 0.05   # LoRA dropout of the benchmark's step
GRAD = 0.05      # standard deviation of incoming fp16 gradients (loss-scaled)
LOSS_SCALE = 1024.0
PIECE = 8192


# ---------------------------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------------------------
def listed():
    return [
        # one projection's weight, decoded on its own: the smallest call there is
        {"name": "dequant_q_proj", "kind": "dequant", "shapes": "1536x1536"},
        # a decoder layer's four weights in one launch, as the step does once per layer
        {"name": "dequant_layer", "kind": "dequant",
         "shapes": "2048x1536,1536x1536,17920x1536,1536x8960"},
        # the MLP on one short prompt of a small model (few rows, ragged)
        {"name": "mlp_short", "kind": "mlp", "width": "0.5B", "tokens": 97},
        # the MLP on a usual micro-batch of packed tokens
        {"name": "mlp_batch", "kind": "mlp", "width": "1.5B", "tokens": 2048},
        # the MLP of a large model on a long micro-batch: the largest products
        {"name": "mlp_large", "kind": "mlp", "width": "7B", "tokens": 4001},
        # the attention-input block on four packed sequences
        {"name": "attn_input", "kind": "attn_input", "width": "1.5B",
         "lengths": "128,733,1024,406"},
        # attention over a usual micro-batch: four sequences of 256 to 1024 tokens
        {"name": "attention_batch", "kind": "attention", "width": "1.5B",
         "lengths": "611,997,283,744"},
        # attention over long sequences (long-context fine-tuning)
        {"name": "attention_long", "kind": "attention", "width": "1.5B",
         "lengths": "4096,3001"},
        # the lm_head's loss and gradients over whole rows
        {"name": "head_rows", "kind": "head", "width": "1.5B", "tokens": 2048, "pieces": False},
        # the same with the logits in vocabulary pieces (little memory), ragged rows
        {"name": "head_pieces", "kind": "head", "width": "1.5B", "tokens": 1027,
         "pieces": True},
        # the whole training step on a usual micro-batch, as the benchmark runs it
        {"name": "step_batch", "kind": "step", "width": "1.5B", "layers": 28,
         "lengths": "611,997,283,744"},
        # the step on a small batch of short prompts, where launches count: a captured graph
        {"name": "graph_short", "kind": "graph", "width": "1.5B", "layers": 28,
         "lengths": "119,64,97,30"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _lengths(rng, rows, lo, hi, most):
    got = [_log_int(rng, lo, hi) for _ in range(rows)]
    while sum(got) > most:
        got = [max(1, g // 2) for g in got]
    return ",".join(str(g) for g in got)


def draw(rng):
    kind = rng.choice(["dequant", "mlp", "mlp", "attn_input", "attention", "attention", "head",
                       "step", "graph"])
    if kind == "dequant":
        shapes = []
        for _ in range(rng.randint(1, 4)):
            shapes.append("%dx%d" % (_log_int(rng, 32, 18000), 64 * _log_int(rng, 1, 140)))
        return {"kind": kind, "shapes": ",".join(shapes)}
    if kind == "mlp":
        return {"kind": kind, "width": rng.choice(["0.5B", "1.5B", "7B"]),
                "tokens": _log_int(rng, 1, 4000)}
    if kind == "attn_input":
        return {"kind": kind, "width": rng.choice(["0.5B", "1.5B", "7B"]),
                "lengths": _lengths(rng, rng.randint(1, 8), 1, 1024, 4000)}
    if kind == "attention":
        return {"kind": kind, "width": rng.choice(["0.5B", "1.5B", "7B"]),
                "lengths": _lengths(rng, rng.randint(1, 8), 16, 4096, 7000)}
    if kind == "head":
        return {"kind": kind, "width": rng.choice(["0.5B", "1.5B"]),
                "tokens": _log_int(rng, 16, 2048), "pieces": rng.random() < 0.5}
    if kind == "step":
        return {"kind": kind, "width": rng.choice(["0.5B", "1.5B"]),
                "layers": rng.randint(2, 12),
                "lengths": _lengths(rng, rng.randint(1, 6), 32, 1024, 3000)}
    return {"kind": kind, "width": rng.choice(["0.5B", "1.5B"]), "layers": rng.randint(2, 12),
            "lengths": _lengths(rng, rng.randint(1, 4), 16, 256, 1000)}


def _ints(text):
    return [int(x) for x in text.split(",")]


def _shapes(case):
    return [tuple(int(d) for d in s.split("x")) for s in case["shapes"].split(",")]


# ---------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(1000003 * seed + 17)


def _randn(g, shape, std=1.0, dtype=torch.float16):
    return (torch.randn(shape, generator=g, device=DEV) * std).to(dtype)


def _nf4(g, shape):
    return PKG.ops.NF4Weight(PKG.quant.quantize_nf4(_randn(g, shape, 0.02)))


def _config(width, layers=1, vocab=None):
    H, I, HQ, HKV, D, V = WIDTHS[width]
    return PKG.engine.Qwen2Config(
        hidden_size=H, intermediate_size=I, num_hidden_layers=layers, num_attention_heads=HQ,
        num_key_value_heads=HKV, head_dim=D, vocab_size=V if vocab is None else vocab,
        lora_dropout=DROPOUT)


def _batch(g, lengths, vocab, T=None):
    """A right-padded batch as a collator makes it: random ids, the first quarter of each
    sequence without labels; the supervised next-token count on the host."""
    B, T = len(lengths), T or max(lengths)
    ids = torch.randint(0, vocab, (B, T), generator=g, device=DEV)
    lens = torch.tensor(lengths, device=DEV)
    real = torch.arange(T, device=DEV)[None] < lens[:, None]
    ids = torch.where(real, ids, 0)
    prompt = torch.arange(T, device=DEV)[None] < torch.div(lens, 4, rounding_mode="floor")[:, None]
    labels = torch.where(real & ~prompt, ids, -100)
    n_sup = sum(n - max(1, n // 4) for n in lengths)
    return ids, real.long(), labels, n_sup


def _packed(model, lengths):
    n, T = len(lengths), max(lengths)
    real = torch.arange(T)[None] < torch.tensor(lengths)[:, None]
    ids = torch.zeros((n, T), dtype=torch.int64, device=DEV)
    return PKG.engine.Packed(ids, real.long().to(DEV), torch.full_like(ids, -100), model.rope,
                             model.dropout, model.dropout_p, lengths=lengths, n_supervised=0)


def _qkv(case, seed):
    _, _, HQ, HKV, D, _ = WIDTHS[case["width"]]
    n = sum(_ints(case["lengths"]))
    g = _gen(seed)
    return (_randn(g, (n, HQ, D)), _randn(g, (n, HKV, D)), _randn(g, (n, HKV, D)),
            _randn(g, (n, HQ, D), GRAD))


def _mlp_inputs(case, seed):
    H, I = WIDTHS[case["width"]][:2]
    T = case["tokens"]
    g = _gen(seed)
    gate, up, down = _nf4(g, (I, H)), _nf4(g, (I, H)), _nf4(g, (H, I))
    return (PKG.ops.NF4Group.of([gate, up]), down, _randn(g, (T, H)),
            _randn(g, (T, H), 1.0, torch.float32), _randn(g, (T, H), GRAD))


def _head_inputs(case, seed):
    H, V, T = WIDTHS[case["width"]][0], WIDTHS[case["width"]][5], case["tokens"]
    g = _gen(seed)
    hn = _randn(g, (T, H))
    E = _randn(g, (V, H), 0.02)
    targets = torch.randint(0, V, (T,), generator=g, device=DEV)
    targets[torch.rand(T, generator=g, device=DEV) < 0.25] = -100
    targets[0] = 5
    return hn, E, targets, float((targets >= 0).sum())


def _attn_input_state(case, seed):
    lengths = _ints(case["lengths"])
    model = PKG.engine.random_qwen2(_config(case["width"], vocab=1024), DEV, seed=seed)
    spec = model.layers[0]
    model.dropout.gen.manual_seed(seed)
    packed = _packed(model, lengths)
    seeds = (packed.draw(spec.H), packed.draw(spec.H))
    lora = [t.detach().half() for t in spec.lora_params()]
    g = _gen(seed)
    n = packed.n
    return dict(spec=spec, packed=packed, seeds=seeds, lora=lora,
                lora_t=[t.t().contiguous() for t in lora],
                h=_randn(g, (n, spec.H), 1.0, torch.float32),
                dq=_randn(g, (n, spec.HQ, spec.D), GRAD),
                dk=_randn(g, (n, spec.HQ, spec.D), GRAD),
                dv=_randn(g, (n, spec.HQ, spec.D), GRAD),
                dres=_randn(g, (n, spec.H), GRAD, torch.float32))


def _step_state(case, seed, padded):
    cfg = _config(case["width"], layers=case["layers"])
    lengths = _ints(case["lengths"])
    model = PKG.engine.random_qwen2(cfg, DEV, seed=seed)
    T = -(-max(lengths) // 8) * 8 if padded else None
    ids, mask, labels, n_sup = _batch(_gen(seed), lengths, cfg.vocab_size, T)
    return dict(model=model, ids=ids, mask=mask, labels=labels, n_sup=n_sup, lengths=lengths,
                denom=float(max(1, n_sup)), gen=model.dropout.gen, seed=seed)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dequant":
        g = _gen(seed)
        return kind, [_nf4(g, s) for s in _shapes(case)]
    if kind == "mlp":
        return kind, _mlp_inputs(case, seed)
    if kind == "attn_input":
        return kind, _attn_input_state(case, seed)
    if kind == "attention":
        lengths = _ints(case["lengths"])
        width = WIDTHS[case["width"]]
        rope = PKG.engine.RopeTable(1e6, width[4], DEV)
        n, T = len(lengths), max(lengths)
        real = torch.arange(T)[None] < torch.tensor(lengths)[:, None]
        ids = torch.zeros((n, T), dtype=torch.int64, device=DEV)
        packed = PKG.engine.Packed(ids, real.long().to(DEV), torch.full_like(ids, -100), rope,
                                   None, 0.0, lengths=lengths, n_supervised=0)
        return kind, (packed, width[4] ** -0.5, *_qkv(case, seed))
    if kind == "head":
        fn = PKG.head.chunked_head if case["pieces"] else PKG.head.full_head
        return kind, (fn, *_head_inputs(case, seed))
    if kind == "step":
        return kind, _step_state(case, seed, False)
    s = _step_state(case, seed, True)
    s["gen"].manual_seed(seed)  # the graph's dropout counters belong to the seed it captures
    s["graph"] = PKG.engine.StepGraph(s["model"], *s["ids"].shape)
    return kind, s


# ---------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------
def _run_mlp(gu_w, down, x, resid, dy):
    L, ops = PKG.linear, PKG.ops
    I = gu_w.shape[0] // 2
    with L.reuse_dequant():
        L.dequant_layer([gu_w, down])
        m, gu = L.nf4_linear_swiglu_keep(x, gu_w, I)
        y = L.nf4_linear_resid(m, down, resid)
        dm = L.nf4_linear_t(dy, down)
        ops._glu_bwd(dm, gu, I)
        dx = L.nf4_linear_t(gu, gu_w)
    return m, y, gu, dx  # gu now holds [dg | du]


def run(state):
    kind, s = state
    if kind == "dequant":
        return PKG.ops.dequant_many(s, DEV)
    if kind == "mlp":
        return _run_mlp(*s)
    if kind == "attn_input":
        E = PKG.engine
        with PKG.linear.reuse_dequant():
            q, k, v, saved = E.attn_input_fwd(s["spec"], s["h"], s["packed"], s["lora"],
                                              s["seeds"], keep_bits=True)
            dh, dh16, grads = E.attn_input_bwd(s["spec"], s["dq"], s["dk"], s["dv"], s["h"],
                                               saved, s["packed"], s["lora_t"], s["seeds"],
                                               dres=s["dres"])
        return q, k, v, dh, dh16, grads
    if kind == "attention":
        packed, scale, q, k, v, dout = s
        out, lse, _, _ = PKG.ops._attn_fwd(q, k, v, packed, scale)
        dq, dk, dv = PKG.ops._attn_bwd(dout, q, k, v, out, lse, None, None, packed, scale)
        return out, lse, dq, dk, dv
    if kind == "head":
        fn, hn, emb, targets, denom = s
        r = fn(hn, emb, targets, denom)
        return r.loss, r.dhn, r.dE, r.tok_loss, r.correct
    # the dropout generator is put where the state's seed puts it (a host-side number), so that
    # a pass can be repeated with the same masks
    model = s["model"]
    s["gen"].manual_seed(s["seed"])
    if kind == "step":
        loss, _, _ = model.step(s["ids"], s["mask"], s["labels"], s["denom"],
                                lengths=s["lengths"], n_supervised=s["n_sup"])
        (loss * LOSS_SCALE).backward()
        loss = loss.detach()
    else:
        loss = s["graph"].replay(s["ids"], s["mask"], s["labels"], s["denom"], LOSS_SCALE)
    params = model.parameters()
    grads = torch.cat([p.grad.reshape(-1) for p in params])  # one flat gradient, all of it
    for p in params:
        p.grad = None
    return loss, grads


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------
def _weight_bytes(numel):
    return numel * (0.5 + 1 / 64 + 4 / 16384)


def _pairs(lengths):
    return sum(n * (n + 1) // 2 for n in lengths)


def _layer_params(width):
    H, I, HQ, HKV, D, _ = WIDTHS[width]
    return H * (HQ + 2 * HKV) * D + H * HQ * D + 3 * H * I


def work(case):
    kind = case["kind"]
    if kind == "dequant":
        numel = sum(r * c for r, c in _shapes(case))
        return {"bytes": _weight_bytes(numel) + 2 * numel, "flops": 2 * numel}
    H, I, HQ, HKV, D, V = WIDTHS[case["width"]]
    C = (HQ + 2 * HKV) * D
    if kind == "mlp":
        T = case["tokens"]
        # x, resid, dy in; m, y, [dg|du], dx out
        return {"bytes": _weight_bytes(3 * H * I) + T * (2 * H + 4 * H + 2 * H + 2 * I + 4 * H
                                                         + 4 * I + 2 * H),
                "flops": 12 * T * H * I}
    if kind == "head":
        T = case["tokens"]
        return {"bytes": 2 * V * H + 4 * V * H + T * (2 * H + 4 * H),
                "flops": 2 * T * V * H + 2 * 2 * 0.75 * T * V * H}
    lengths = _ints(case["lengths"])
    n = sum(lengths)
    if kind == "attn_input":
        # h, dq, dk, dv, dres in; q, k, v, dh, dh16 out
        return {"bytes": _weight_bytes(H * C) + n * (4 * H + 3 * 2 * HQ * D + 4 * H + 2 * C
                                                     + 4 * H + 2 * H),
                "flops": 4 * n * H * C + 6 * 2 * n * 16 * (2 * H + (HQ + HKV) * D)}
    if kind == "attention":
        # q, k, v, dout in; out, lse, dq, dk, dv out
        return {"bytes": n * (2 * 2 * HQ * D + 2 * 2 * HKV * D + 2 * HQ * D + 4 * HQ
                              + 3 * 2 * HQ * D),
                "flops": 14 * D * HQ * _pairs(lengths)}
    layers = case["layers"]
    flops = layers * (4 * n * _layer_params(case["width"]) + 14 * D * HQ * _pairs(lengths)) \
        + 2 * n * V * H + 2 * 0.75 * n * V * H
    # the frozen weights twice (forward and backward), each layer's input and its gradient
    return {"bytes": layers * (2 * _weight_bytes(_layer_params(case["width"])) + n * 4 * 4 * H)
            + 2 * 2 * V * H, "flops": flops}


def tolerance(case):
    """About four times the difference from the same path in 64 bits, as measured on the listed
    and on drawn sizes (fp16 operands and outputs, fp32 sums)."""
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind == "mlp":
        return {"rel": 1.7e-3, "max": 0.012}
    if kind == "attn_input":
        return {"rel": 1.5e-3, "max": 0.008}
    if kind == "attention":
        return {"rel": 1.3e-3, "max": 0.06}
    if kind == "head":
        # the pieces' hidden gradient is rounded to fp16, the whole rows' is fp32
        return {"rel": 9e-4 if case["pieces"] else 6e-5, "max": 0.002, "differ": 0.005}
    return {"rel": 2e-2, "max": 0.95}


# ---------------------------------------------------------------------------------------------
# The same in 64 bits, plain torch
# ---------------------------------------------------------------------------------------------
def _weight64(w):
    """The fp16 weight an NF4 weight stands for (bitsandbytes' rounding), as float64."""
    codes = torch.stack([w.packed.reshape(-1) >> 4, w.packed.reshape(-1) & 15], 1).reshape(-1)
    scale = w.code2[w.absmax.long()] * w.absmax2.repeat_interleave(w.bs2)[:w.absmax.numel()] \
        + w.offset
    vals = w.code[codes.long()].view(-1, w.bs1) * scale[:, None]
    return vals.half().double().view(w.shape)


def _rms64(x, w, eps):
    return w.double() * x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _rope64(x, pos, theta):
    half = x.shape[-1] // 2
    inv = theta ** (-torch.arange(half, device=DEV, dtype=torch.float64) / half)
    ang = (pos.double()[:, None] * inv[None])[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)


def _attend64(q, k, v, lengths, scale):
    """(out [n, HQ, D], lse [HQ, n]) of q, k, v all with HQ heads."""
    outs, lses, start = [], [], 0
    for n in lengths:
        sl = slice(start, start + n)
        heads_o, heads_l = [], []
        dead = torch.ones((n, n), device=DEV, dtype=torch.bool).triu(1)
        for h in range(q.shape[1]):  # one head at a time: [n, n] in 64 bits is large
            s = (q[sl, h] @ k[sl, h].t() * scale).masked_fill(dead, -math.inf)
            lse = torch.logsumexp(s, -1)
            heads_l.append(lse)
            heads_o.append(torch.exp(s - lse[:, None]) @ v[sl, h])
        outs.append(torch.stack(heads_o, 1))
        lses.append(torch.stack(heads_l))
        start += n
    return torch.cat(outs), torch.cat(lses, 1)


def _masks(seed, B, T, H, tok, count):
    """The keep masks of `count` LoRA dropout calls on a [B, T, H] input, as nn.Dropout draws
    them, at the packed tokens."""
    gen = torch.cuda.default_generators[DEV.index]
    gen.manual_seed(seed)
    ones = torch.ones((B, T, H), device=DEV)
    return [torch.nn.functional.dropout(ones, DROPOUT, True).view(B * T, H).index_select(0, tok)
            != 0 for _ in range(count)]


def _attn_input64(h, spec, masks, lora, pos, weights):
    n = h.shape[0]
    a = _rms64(h, spec.ln1, spec.eps)
    aq, av = (torch.where(m, a / (1 - DROPOUT), torch.zeros_like(a)) for m in masks)
    Aq, Bq, Av, Bv = lora
    s = spec.lora["q"][2]
    qkv = a @ weights.t() + spec.bias_qkv.double()
    nq, nk = spec.HQ * spec.D, spec.HKV * spec.D
    q = (qkv[:, :nq] + s * (aq @ Aq.t()) @ Bq.t()).view(n, spec.HQ, spec.D)
    k = qkv[:, nq:nq + nk].view(n, spec.HKV, spec.D)
    v = (qkv[:, nq + nk:] + s * (av @ Av.t()) @ Bv.t()).view(n, spec.HKV, spec.D)
    return _rope64(q, pos, 1e6), _rope64(k, pos, 1e6), v


def _positions(lengths):
    return torch.cat([torch.arange(n, device=DEV) for n in lengths])


def _step64(s, T, seed):
    model, lengths = s["model"], s["lengths"]
    B, H = len(lengths), model.cfg.hidden_size
    pos = _positions(lengths)
    tok = torch.cat([torch.arange(n, device=DEV) + T * r for r, n in enumerate(lengths)])
    masks = _masks(seed, B, T, H, tok, 2 * len(model.layers))
    leaves = [t.detach().double().requires_grad_() for t in model.parameters()]
    E = model.embed.double()
    h = E[s["ids"].reshape(-1)[tok]]

    def layer(i, h, *lora):
        spec = model.layers[i]
        w = {k: _weight64(x) for k, x in spec.w.items()}
        q, k, v = _attn_input64(h, spec, masks[2 * i:2 * i + 2], lora, pos,
                                torch.cat([w["q_proj"], w["k_proj"], w["v_proj"]]))
        rep = spec.HQ // spec.HKV
        o, _ = _attend64(q, k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1), lengths,
                         spec.scale)
        h = h + o.reshape(h.shape[0], -1) @ w["o_proj"].t()
        b = _rms64(h, spec.ln2, spec.eps)
        m = torch.nn.functional.silu(b @ w["gate_proj"].t()) * (b @ w["up_proj"].t())
        return h + m @ w["down_proj"].t()

    for i in range(len(model.layers)):
        h = checkpoint(layer, i, h, *leaves[4 * i:4 * i + 4], use_reentrant=False,
                       preserve_rng_state=False)
    nxt = torch.nn.functional.pad(s["labels"], (0, 1), value=-100)[:, 1:].reshape(-1)[tok]
    sup = nxt >= 0
    logits = _rms64(h[sup], model.norm_w, model.eps) @ E.t()
    loss = torch.nn.functional.cross_entropy(logits, nxt[sup], reduction="sum") / s["denom"]
    grads = torch.autograd.grad(loss * LOSS_SCALE, leaves)
    return loss.detach(), torch.cat([g.reshape(-1) for g in grads])


def exact(case, seed):
    kind = case["kind"]
    if kind == "dequant":
        g = _gen(seed)
        return [_weight64(_nf4(g, s)) for s in _shapes(case)]
    if kind == "mlp":
        gu_w, down, x, resid, dy = _mlp_inputs(case, seed)
        gate, up = (_weight64(w) for w in gu_w.weights)
        w_d = _weight64(down)
        x, dy = x.double(), dy.double()
        g, u = x @ gate.t(), x @ up.t()
        sig = torch.sigmoid(g)
        m = g * sig * u
        dm = dy @ w_d
        dg, du = dm * u * sig * (1 + g * (1 - sig)), dm * g * sig
        return m, resid.double() + m @ w_d.t(), torch.cat([dg, du], 1), dg @ gate + du @ up
    if kind == "attn_input":
        s = _attn_input_state(case, seed)
        spec, lengths = s["spec"], _ints(case["lengths"])
        masks = _masks(seed, len(lengths), max(lengths), spec.H, s["packed"].tok, 2)
        w = torch.cat([_weight64(spec.w[k]) for k in ("q_proj", "k_proj", "v_proj")])
        lora = [t.double().requires_grad_() for t in s["lora"]]
        h = s["h"].double().requires_grad_()
        q, k, v = _attn_input64(h, spec, masks, lora, _positions(lengths), w)
        rep = spec.HQ // spec.HKV
        group = [t.double().view(-1, spec.HKV, rep, spec.D).sum(2) for t in (s["dk"], s["dv"])]
        dh, dAq, dBq, dAv, dBv = torch.autograd.grad(
            (q, k, v), (h, *lora), (s["dq"].double(), *group))
        dh = dh + s["dres"].double()
        return q.detach(), k.detach(), v.detach(), dh, dh, (dAq, dBq, dAv, dBv)
    if kind == "attention":
        width = WIDTHS[case["width"]]
        q, k, v, dout = (t.double() for t in _qkv(case, seed))
        rep = width[2] // width[3]
        q, k, v = (t.detach().requires_grad_() for t in (
            q, k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)))
        out, lse = _attend64(q, k, v, _ints(case["lengths"]), width[4] ** -0.5)
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), dout)
        return out.detach(), lse.detach(), dq, dk, dv
    if kind == "head":
        hn, emb, targets, denom = _head_inputs(case, seed)
        hn, emb = hn.double(), emb.double()
        sup = targets >= 0
        logits = hn @ emb.t()
        lse = torch.logsumexp(logits, 1)
        safe = targets.clamp(min=0)
        tok = torch.where(sup, lse - logits.gather(1, safe[:, None])[:, 0], 0.0)
        correct = (sup & (logits.argmax(1) == targets)).to(torch.int32)
        grad = logits.sub_(lse[:, None]).exp_()
        grad[torch.arange(grad.shape[0], device=DEV), safe] -= 1
        grad.mul_(sup[:, None] / denom)
        return tok.sum() / denom, grad @ emb, grad.t() @ hn, tok, correct
    s = _step_state(case, seed, kind == "graph")
    return _step64(s, s["ids"].shape[1], seed)
