"""The workloads whose speed counts: the layers of a LLaDA2-shaped block
diffusion model as a program runs them on the GPU, and one whole step.

A block-diffusion sampler calls every layer once per denoising step over its
whole window, N = 32 (block + 1) tokens: from one block up to a window of
2048.  The other sampler and a prompt bring any number of tokens (no block
routing then).  Each case is one call of one entry point on device buffers
(`step`: the calls of a whole step), with weights in the GGUF block layouts.

Kinds
  moe    the block-routed MoE layer (Context.forward_device)
  attn   the attention half of a layer (Context.attn_forward_device)
  dense  the dense MLP of the first layer (Context.forward_device)
  head   final norm, LM head, argmax and confidence (Context.head_forward_device)
  step   attention + dense MLP, then attention + MoE per further layer with the
         residual adds between them, then the LM head
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "diffuse-cpp_amd"))

import dmoe  # noqa: E402

DEV = "cuda:0"
EPS = 1e-6
EXPERTS, TOP_K, CAPACITY, BLOCK, SCALING = 256, 8, 48, 32, 2.5
VOCAB = 157184
HEAD_DIM, ROTARY, ROPE_BASE = 128, 64, 3e6

# per hidden size: the experts' (and the shared expert's) width, the dense
# MLP's width, attention heads and KV heads
SHAPES = {4096: dict(ff=1024, n_ff=9216, heads=32, kv=4),
          2048: dict(ff=512, n_ff=5120, heads=16, kv=4)}

TYPES = {"q4_k": dmoe.TYPE_Q4_K, "q8_0": dmoe.TYPE_Q8_0, "f16": dmoe.TYPE_F16, "q6_k": 14}
BLOCK_BYTES = {"q4_k": (256, 144), "q8_0": (32, 34), "f16": (1, 2), "q6_k": (256, 210)}


def row_bytes(wtype, n):
    elems, size = BLOCK_BYTES[wtype]
    return n // elems * size


def listed():
    def c(name, kind, wtype, n, hidden=4096, **more):
        return dict(name=name, kind=kind, wtype=wtype, n=n, hidden=hidden, **more)
    return [
        # the sampler's first block: the smallest window, and the headline
        c("moe_q4k_n32", "moe", "q4_k", 32, hot=False),
        # the same call of a model half as wide: the smallest work per call
        c("moe_q4k_h2048_n32", "moe", "q4_k", 32, hidden=2048, hot=False),
        # a window of eight blocks, the middle of a generation
        c("moe_q4k_n256", "moe", "q4_k", 256, hot=False),
        # the longest window
        c("moe_q4k_n2048", "moe", "q4_k", 2048, hot=False),
        # 8-bit experts on a ragged number of tokens: plain top-k over all experts
        c("moe_q8_0_n77", "moe", "q8_0", 77, hot=False),
        # unquantised experts over a long prompt whose blocks agree on a hot set
        c("moe_f16_n2048", "moe", "f16", 2048, hot=True),
        # the attention half of the same windows
        c("attn_q4k_n32", "attn", "q4_k", 32),
        c("attn_q4k_n2048", "attn", "q4_k", 2048),
        c("attn_q8_0_n200", "attn", "q8_0", 200),
        # the first layer's MLP
        c("dense_q4k_n160", "dense", "q4_k", 160),
        # the LM head over a window: Q6_K is what the 4-bit schemes give it
        c("head_q6k_n256", "head", "q6_k", 256),
        # a denoising step over the first block through a model cut to three
        # layers: every entry point in turn, down to the logits
        c("step_n32", "step", "q4_k", 32, layers=3),
    ]


def draw(rng):
    """One more case: any kind, type and size of the ranges above."""
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    wtypes = {"moe": ("q4_k", "q4_k", "q8_0", "f16"), "attn": ("q4_k", "q4_k", "q8_0"),
              "dense": ("q4_k", "q4_k", "q6_k"), "head": ("q6_k", "q6_k", "q4_k")}
    top = {"moe": 2048, "attn": 2048, "dense": 512, "head": 256}
    while True:
        kind = rng.choice(("moe", "moe", "moe", "attn", "attn", "dense", "head"))
        wtype = rng.choice(wtypes[kind])
        n = int(round(math.exp(rng.uniform(math.log(16), math.log(top[kind])))))
        if n >= 64 and rng.random() < 0.6:
            n = n // 32 * 32                        # whole blocks
        elif n % 32 == 0:
            n -= 1
        case = dict(kind=kind, wtype=wtype, n=n, hidden=rng.choice((4096, 4096, 2048)))
        if kind == "moe":
            case["hot"] = rng.random() < 0.3
        if case not in known:
            return case


# ---------------------------------------------------------------------------
# Inputs.  Weights ~ N(0, 0.02) as the quantisers leave them: quants centred
# and bell-shaped, scales of each block spread around their mean.

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _bell(g, rows, n, mean, std, top):
    """Whole values around `mean`, 0 .. top, as uint8."""
    z = torch.empty((rows, n), dtype=torch.float16, device=DEV).normal_(mean, std, generator=g)
    return z.round_().clamp_(0, top).to(torch.uint8)


def _bytes_of(half):
    return half.view(torch.uint8)


def _chunks(rows, n):
    step = max(1, (1 << 28) // n)
    return [(r, min(rows, r + step)) for r in range(0, rows, step)]


def _fill_q4k(g, out, n):
    rows, nb = out.shape[0], n // 256
    q = _bell(g, rows, n, 7.5, 3.6, 15).view(rows, nb, 4, 2, 32)
    b = out.view(rows, nb, 144)
    sc = torch.randint(40, 64, (rows, nb, 8), generator=g, device=DEV, dtype=torch.uint8)
    m = torch.randint(40, 64, (rows, nb, 8), generator=g, device=DEV, dtype=torch.uint8)
    d = torch.empty((rows, nb, 1), device=DEV).uniform_(0.9, 1.1, generator=g).mul_(0.02 / 3.6 / 51.5)
    b[..., 0:2] = _bytes_of(d.half())
    b[..., 2:4] = _bytes_of((7.5 * d).half())
    b[..., 4:8] = sc[..., :4] | (sc[..., 4:] >> 4 << 6)
    b[..., 8:12] = m[..., :4] | (m[..., 4:] >> 4 << 6)
    b[..., 12:16] = (sc[..., 4:] & 15) | (m[..., 4:] << 4)
    b[..., 16:] = (q[..., 0, :] | (q[..., 1, :] << 4)).reshape(rows, nb, 128)


def _fill_q6k(g, out, n):
    rows, nb = out.shape[0], n // 256
    q = _bell(g, rows, n, 32.0, 11.0, 63).view(rows, nb, 2, 4, 32)
    b = out.view(rows, nb, 210)
    lo, hi = q & 15, q >> 4
    ql = torch.stack((lo[..., 0, :] | (lo[..., 2, :] << 4), lo[..., 1, :] | (lo[..., 3, :] << 4)), dim=3)
    b[..., :128] = ql.reshape(rows, nb, 128)
    qh = hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)
    b[..., 128:192] = qh.reshape(rows, nb, 64)
    sc = torch.randint(70, 128, (rows, nb, 16), generator=g, device=DEV, dtype=torch.int8)
    sign = torch.randint(0, 2, (rows, nb, 16), generator=g, device=DEV, dtype=torch.int8)
    b[..., 192:208] = (sc * (1 - 2 * sign)).view(torch.uint8)
    d = torch.empty((rows, nb, 1), device=DEV).uniform_(0.9, 1.1, generator=g).mul_(0.02 / 11.0 / 98.0)
    b[..., 208:] = _bytes_of(d.half())


def _fill_q8_0(g, out, n):
    rows, nb = out.shape[0], n // 32
    q = torch.empty((rows, nb, 32), dtype=torch.float16, device=DEV).normal_(0.0, 48.0, generator=g)
    b = out.view(rows, nb, 34)
    b[..., 2:] = q.round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
    d = torch.empty((rows, nb, 1), device=DEV).uniform_(0.85, 1.15, generator=g).mul_(0.02 / 48.0)
    b[..., :2] = _bytes_of(d.half())


def _fill_f16(g, out, n):
    out.view(torch.float16).normal_(0.0, 0.02, generator=g)


_FILL = {"q4_k": _fill_q4k, "q6_k": _fill_q6k, "q8_0": _fill_q8_0, "f16": _fill_f16}


def _weight(g, wtype, rows, n):
    out = torch.empty((rows, row_bytes(wtype, n)), dtype=torch.uint8, device=DEV)
    for r0, r1 in _chunks(rows, n):
        _FILL[wtype](g, out[r0:r1], n)
    return out


def _uniform(g, lo, hi, n):
    return torch.empty(n, device=DEV).uniform_(lo, hi, generator=g)


def _normal(g, *shape, std=1.0):
    return torch.empty(shape, device=DEV).normal_(0.0, std, generator=g)


def _moe_inputs(case, g):
    H, ff = case["hidden"], SHAPES[case["hidden"]]["ff"]
    t = case["wtype"]
    w = dict(gate_w=_normal(g, EXPERTS, H, std=0.02))
    if case.get("hot"):
        # a quarter of the experts favoured, so that the blocks agree on most
        bias = _uniform(g, -0.05, 0.05, EXPERTS)
        bias[torch.randperm(EXPERTS, generator=g, device=DEV)[:EXPERTS // 4]] += 0.05
    else:
        bias = _uniform(g, -0.1, 0.1, EXPERTS)
    w["gate_bias"] = bias
    w["exp_gate"] = _weight(g, t, EXPERTS * ff, H).view(EXPERTS, ff, -1)
    w["exp_up"] = _weight(g, t, EXPERTS * ff, H).view(EXPERTS, ff, -1)
    w["exp_down"] = _weight(g, t, EXPERTS * H, ff).view(EXPERTS, H, -1)
    w["sh_gate"] = _weight(g, t, ff, H)
    w["sh_up"] = _weight(g, t, ff, H)
    w["sh_down"] = _weight(g, t, H, ff)
    return w


def _attn_inputs(case, g):
    H, s = case["hidden"], SHAPES[case["hidden"]]
    q_dim, qkv_dim = s["heads"] * HEAD_DIM, (s["heads"] + 2 * s["kv"]) * HEAD_DIM
    return dict(attn_norm=_uniform(g, 0.5, 1.5, H), qkv=_weight(g, case["wtype"], qkv_dim, H),
                wo=_weight(g, case["wtype"], H, q_dim), post_norm=_uniform(g, 0.5, 1.5, H),
                q_norm=_uniform(g, 0.5, 1.5, HEAD_DIM), k_norm=_uniform(g, 0.5, 1.5, HEAD_DIM))


def _dense_inputs(case, g):
    H, n_ff = case["hidden"], SHAPES[case["hidden"]]["n_ff"]
    return dict(gate=_weight(g, case["wtype"], n_ff, H), up=_weight(g, case["wtype"], n_ff, H),
                down=_weight(g, case["wtype"], H, n_ff))


def _head_inputs(case, g):
    return dict(norm=_uniform(g, 0.5, 1.5, case["hidden"]),
                output=_weight(g, case["wtype"], VOCAB, case["hidden"]))


_INPUTS = {"moe": _moe_inputs, "attn": _attn_inputs, "dense": _dense_inputs, "head": _head_inputs}


def _parts(case):
    """(kind, case of that kind) of the layers a case runs, in order."""
    if case["kind"] != "step":
        return [(case["kind"], case)]
    parts = [("attn", case), ("dense", case)]
    for _ in range(case["layers"] - 1):
        parts += [("attn", case), ("moe", dict(case, hot=False))]
    return parts + [("head", dict(case, wtype="q6_k"))]


def _part_inputs(case, seed, i):
    kind, part = _parts(case)[i]
    return _INPUTS[kind](part, _gen(seed * 1009 + 31 * i + 7))


def _x(case, seed):
    """The layer's input rows (a normed residual stream for the MLPs, the
    stream itself for the others): unit variance."""
    return _normal(_gen(seed * 1009 + 5), case["n"], case["hidden"])


# ---------------------------------------------------------------------------
# The framework's side.

_ctx = None


def _context():
    """One context per process, as a program that serves one GPU keeps."""
    global _ctx
    if _ctx is None:
        _ctx = dmoe.Context(0)
    return _ctx


def _wrap(ctx, kind, case, w):
    H, s, t = case["hidden"], SHAPES[case["hidden"]], TYPES[case["wtype"]]
    if kind == "moe":
        layer = ctx.wrap_device(dmoe.LayerWeights(
            n_embd=H, n_experts=EXPERTS, top_k=TOP_K, capacity=CAPACITY, block_size=BLOCK, moe_ff=s["ff"], wtype=t,
            n_shared=1, shared_ff=s["ff"], stype=t, routed_scaling=SCALING, **w))
        # the library holds its own tiled copy of the experts by now
        for k in ("exp_gate", "exp_up", "exp_down", "sh_gate", "sh_up", "sh_down"):
            setattr(layer.weights, k, None)
        return layer
    if kind == "attn":
        return ctx.attn_wrap_device(dmoe.AttnWeights(
            n_embd=H, n_head=s["heads"], n_head_kv=s["kv"], head_dim=HEAD_DIM, rotary_dim=ROTARY, block_length=BLOCK,
            rope_base=ROPE_BASE, rms_eps=EPS, wtype=t, **w))
    if kind == "dense":
        return ctx.dense_wrap_device(dmoe.DenseWeights(n_embd=H, n_ff=s["n_ff"], wtype=t, **w))
    return ctx.head_wrap_device(dmoe.HeadWeights(n_embd=H, n_vocab=VOCAB, wtype=t, **w))


def prepare(case, seed):
    ctx, N, H = _context(), case["n"], case["hidden"]
    layers = []
    for i, (kind, part) in enumerate(_parts(case)):
        w = _part_inputs(case, seed, i)
        torch.cuda.synchronize()                    # the upload runs on the context's own stream
        layers.append((kind, _wrap(ctx, kind, part, w)))
    x = _x(case, seed)
    st = dict(ctx=ctx, kind=case["kind"], layers=layers, n=N, hidden=H, x=x, y=torch.empty_like(x))
    if case["kind"] in ("attn", "step"):
        st["moe_in"] = torch.empty_like(x)
    if case["kind"] == "step":
        st["scratch"] = torch.empty_like(x)
        st["h"] = torch.empty_like(x)
    if case["kind"] in ("head", "step"):
        st["tokens"] = torch.empty(N, dtype=torch.int32, device=DEV)
        st["probs"] = torch.empty(N, device=DEV)
        st["logits"] = torch.empty((N, VOCAB), device=DEV)
    return st


def run(st):
    ctx, kind, N, H = st["ctx"], st["kind"], st["n"], st["hidden"]
    s = torch.cuda.current_stream().cuda_stream
    if kind in ("moe", "dense"):
        ctx.forward_device(st["layers"][0][1], st["x"], N, st["y"], s)
        return st["y"]
    if kind == "attn":
        ctx.attn_forward_device(st["layers"][0][1], st["x"], N, st["y"], st["moe_in"], s)
        return st["y"], st["moe_in"]
    if kind == "head":
        ctx.head_forward_device(st["layers"][0][1], st["x"], N, EPS, st["tokens"], st["probs"], st["logits"], s)
        return dict(logits=st["logits"], probs=st["probs"], tokens=st["tokens"])
    src = st["x"]                                   # the embedded tokens
    for k, layer in st["layers"]:
        if k == "attn":
            ctx.attn_forward_device(layer, src, N, st["h"], st["moe_in"], s)
            src = st["h"]
        elif k == "head":
            ctx.head_forward_device(layer, st["h"], N, EPS, st["tokens"], st["probs"], st["logits"], s)
        else:
            ctx.forward_device(layer, st["moe_in"], N, st["y"], s)
            ctx.residual_rmsnorm(st["h"], st["y"], st["scratch"], N, H, EPS, stream=s)
    return dict(h=st["h"], logits=st["logits"], probs=st["probs"])


# ---------------------------------------------------------------------------
# What a pass cannot do without.

def _touched(case):
    """Experts a forward is expected to reach: 48 in one block; further blocks
    add what their own choice leaves out, a ragged call draws from all."""
    n = case["n"]
    if n % BLOCK == 0:
        hit = {32: 48, 256: 100, 2048: 125}.get(n, 48 + 15 * math.log2(n / BLOCK))
        if case.get("hot"):
            hit *= 1.3
    else:
        hit = EXPERTS * (1 - (1 - TOP_K / EXPERTS) ** (0.6 * n))
    return min(float(EXPERTS), hit)


def _part_work(kind, case):
    N, H, s, t = case["n"], case["hidden"], SHAPES[case["hidden"]], case["wtype"]
    io = 4 * N * H
    if kind == "moe":
        one = 2 * s["ff"] * row_bytes(t, H) + H * row_bytes(t, s["ff"])
        return (_touched(case) * one + one + 4 * EXPERTS * H + 2 * io,
                2.0 * N * ((TOP_K + 1) * 3 * H * s["ff"] + H * EXPERTS))
    if kind == "attn":
        q_dim, qkv_dim = s["heads"] * HEAD_DIM, (s["heads"] + 2 * s["kv"]) * HEAD_DIM
        seen = sum(min(N, (q // BLOCK + 1) * BLOCK) for q in range(N))
        return (qkv_dim * row_bytes(t, H) + H * row_bytes(t, q_dim) + 3 * io,
                2.0 * N * H * (qkv_dim + q_dim) + 4.0 * HEAD_DIM * s["heads"] * seen)
    if kind == "dense":
        return 2 * s["n_ff"] * row_bytes(t, H) + H * row_bytes(t, s["n_ff"]) + 2 * io, 6.0 * N * H * s["n_ff"]
    return VOCAB * row_bytes(t, H) + io + 4 * N * VOCAB, 2.0 * N * H * VOCAB


def work(case):
    b = f = 0.0
    for kind, part in _parts(case):
        pb, pf = _part_work(kind, part)
        b, f = b + pb, f + pf
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Relative error that another correct implementation shows.

    moe      the expert products take x and h as 8-bit (Q4_K, Q8_0) or 16-bit
             (F16) values; summing in another order moves an f32 h by an ulp
             and now and then one of those values by a step
    attn, dense, head   f32 activations as 16-bit integers relative to their
             block's largest value: 1e-5 to 1e-4 of the result against 64 bits
             (the dense MLP, whose gated h is the most uneven, the 1e-4)
    step     what the layers' differences grow to over three layers: it is 2e-2
             off in 64 bits, most of it the experts' 8-bit activations
    """
    if case["kind"] == "moe":
        return {"rel": 2e-3, "max": 0.05} if case["wtype"] != "f16" else {"rel": 4e-4, "max": 0.02}
    if case["kind"] == "step":
        return {"rel": 1e-2, "max": 0.5}
    return {"rel": 4e-4 if case["kind"] == "dense" else 2e-4, "max": 1e-2, "differ": 0.01}


# ---------------------------------------------------------------------------
# The same results in 64 bits, from the block layouts and the formulas alone.

def _decode(wtype, raw, n):
    """GGUF block bytes [rows][row_bytes] -> f64 [rows][n]."""
    rows = raw.shape[0]
    if wtype == "f16":
        return raw.view(torch.float16).double()
    elems, size = BLOCK_BYTES[wtype]
    b = raw.view(rows, n // elems, size)

    def half(lo):
        return b[..., lo:lo + 2].contiguous().view(torch.float16).double()

    if wtype == "q8_0":
        return (b[..., 2:].contiguous().view(torch.int8).double() * half(0)).reshape(rows, n)
    if wtype == "q4_k":
        s = b[..., 4:16].int()
        sc = torch.cat((s[..., :4] & 63, (s[..., 8:] & 15) | (s[..., :4] >> 6 << 4)), -1).double()
        m = torch.cat((s[..., 4:8] & 63, (s[..., 8:] >> 4) | (s[..., 4:8] >> 6 << 4)), -1).double()
        qs = b[..., 16:].reshape(rows, -1, 4, 32)
        q = torch.stack((qs & 15, qs >> 4), 3).reshape(rows, -1, 8, 32).double()
        return (q * (half(0) * sc).unsqueeze(-1) - (half(2) * m).unsqueeze(-1)).reshape(rows, n)
    ql = b[..., :128].reshape(rows, -1, 2, 2, 32).int()
    qh = b[..., 128:192].reshape(rows, -1, 2, 32).int()
    q = torch.stack([(ql[..., 0, :] & 15) | ((qh & 3) << 4), (ql[..., 1, :] & 15) | ((qh >> 2 & 3) << 4),
                     (ql[..., 0, :] >> 4) | ((qh >> 4 & 3) << 4), (ql[..., 1, :] >> 4) | ((qh >> 6 & 3) << 4)], 3)
    q = (q - 32).double().reshape(rows, -1, 16, 16)
    sc = b[..., 192:208].contiguous().view(torch.int8).double()
    return (q * (half(208) * sc).unsqueeze(-1)).reshape(rows, n)


def _norm64(x, gain=None):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return y if gain is None else y * gain.double()


def _times(x, wtype, raw, n):
    """x [N][n] times the rows of a weight, some rows at a time."""
    out = torch.empty((x.shape[0], raw.shape[0]), dtype=torch.float64, device=DEV)
    for r0 in range(0, raw.shape[0], 8192):
        out[:, r0:r0 + 8192] = x @ _decode(wtype, raw[r0:r0 + 8192], n).T
    return out


def _mlp64(x, t, gate, up, down):
    H, ff = x.shape[1], gate.shape[0]
    h = torch.nn.functional.silu(_times(x, t, gate, H)) * _times(x, t, up, H)
    return _times(h, t, down, ff)


def _moe64(case, w, x):
    N, t = x.shape[0], case["wtype"]
    p = torch.sigmoid(x @ w["gate_w"].double().T)
    sel = p + w["gate_bias"].double()
    if N % BLOCK == 0:
        top = sel.view(N // BLOCK, BLOCK, EXPERTS).amax(1)
        thr = top.sort(-1, descending=True).values[:, CAPACITY - 1:CAPACITY]
        keep = (top > thr - 1e-6).repeat_interleave(BLOCK, 0)
        sel = torch.where(keep, sel, torch.full_like(sel, -1e30))
    idx = sel.topk(TOP_K, -1).indices
    wt = p.gather(1, idx)
    wt = wt / wt.sum(-1, keepdim=True) * SCALING
    y = _mlp64(x, t, w["sh_gate"], w["sh_up"], w["sh_down"])
    for e in idx.unique().tolist():
        tok, slot = (idx == e).nonzero(as_tuple=True)
        out = _mlp64(x[tok], t, w["exp_gate"][e], w["exp_up"][e], w["exp_down"][e])
        y.index_add_(0, tok, out * wt[tok, slot].unsqueeze(-1))
    return y


def _attn64(case, w, h):
    N, H, s, t = h.shape[0], case["hidden"], SHAPES[case["hidden"]], case["wtype"]
    nh, kv = s["heads"], s["kv"]
    qkv = _times(_norm64(h, w["attn_norm"]), t, w["qkv"], H).view(N, nh + 2 * kv, HEAD_DIM)
    q, k, v = qkv.split((nh, kv, kv), 1)
    q, k = _norm64(q, w["q_norm"]), _norm64(k, w["k_norm"])
    at = torch.arange(N, device=DEV, dtype=torch.float64).unsqueeze(1)
    ang = at * ROPE_BASE ** (-2.0 / ROTARY * torch.arange(ROTARY // 2, device=DEV, dtype=torch.float64))
    cos, sin = ang.cos().unsqueeze(1), ang.sin().unsqueeze(1)

    def rope(z):
        a, b = z[..., :ROTARY // 2], z[..., ROTARY // 2:ROTARY]
        return torch.cat((a * cos - b * sin, a * sin + b * cos, z[..., ROTARY:]), -1)

    q, k = rope(q), rope(k)
    blk = torch.arange(N, device=DEV) // BLOCK
    hidden = blk.unsqueeze(0) > blk.unsqueeze(1)
    out = torch.empty((N, nh, HEAD_DIM), dtype=torch.float64, device=DEV)
    for i in range(nh):
        g = i // (nh // kv)
        score = (q[:, i] @ k[:, g].T / math.sqrt(HEAD_DIM)).masked_fill(hidden, -math.inf)
        out[:, i] = torch.softmax(score, -1) @ v[:, g]
    h_out = h + _times(out.reshape(N, -1), t, w["wo"], nh * HEAD_DIM)
    return h_out, _norm64(h_out, w["post_norm"])


def _head64(case, w, h):
    logits = _times(_norm64(h, w["norm"]), case["wtype"], w["output"], case["hidden"])
    return logits, torch.softmax(logits, -1).amax(-1)


def exact(case, seed):
    x = _x(case, seed).double()
    kind = case["kind"]
    if kind != "step":
        w = _part_inputs(case, seed, 0)
        if kind == "moe":
            return _moe64(case, w, x)
        if kind == "dense":
            return _mlp64(x, case["wtype"], w["gate"], w["up"], w["down"])
        if kind == "attn":
            return _attn64(case, w, x)
        logits, probs = _head64(case, w, x)
        return dict(logits=logits, probs=probs, tokens=None)
    h = x
    for i, (k, part) in enumerate(_parts(case)):
        w = _part_inputs(case, seed, i)
        if k == "attn":
            h, moe_in = _attn64(part, w, h)
        elif k == "head":
            logits, probs = _head64(part, w, h)
        elif k == "dense":
            h = h + _mlp64(moe_in, part["wtype"], w["gate"], w["up"], w["down"])
        else:
            h = h + _moe64(part, w, moe_in)
    return dict(h=h, logits=logits, probs=probs)
