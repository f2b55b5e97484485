"""The calls whose speed counts: the layers and operators of the LFM2.5-8B-A1B decoder at its own
sizes (hidden 2048, 32 experts of 1792 with top-4, dense FFN 7168, 32 query and 8 kv heads of 64,
a 128,000-row vocabulary), each through the entry point a program calls, and two whole calls.

Weights are synthetic blocks in the GGUF byte layouts, their scales set so that a weight has about
the standard deviation 1/sqrt(2048) of a trained matrix and a zero mean, so the router's logits,
the gates and the residual stream have the sizes they have in a trained model.

Outputs are compared bit for bit: the library promises the reference CPU path's bits (integer
dots, f32 epilogues in a fixed order), so another correct implementation shows no difference.
`exact` states the same operations in float64; the 8-bit activations are part of each operation.
"""
import math

import numpy as np
import torch

from bebelm_amd import kernels, synth
from bebelm_amd.model import AttnOp, Context, ConvOp, DenseLayer, FfnStack, Model, MoeLayer

Q4, Q6 = synth.Q4_K, synth.Q6_K
H, F, E, K = synth.HIDDEN, synth.MOE_FF, synth.N_EXPERTS, synth.N_USED
DENSE_F, L_CACHE = synth.DENSE_FF, synth.CONV_L_CACHE
NH, NKV, HD = synth.N_HEADS, synth.N_KV_HEADS, synth.HEAD_DIM
VOCAB, EPS, THETA = synth.VOCAB, synth.RMS_EPS, synth.ROPE_THETA
CHUNK = 512            # the agent absorbs a prompt in chunks of this many tokens
STACK_LAYERS = 8       # layers 0 .. 7 of the schedule: two dense, six MoE
CHAT_LAYERS = 6        # layers 0 .. 5: two dense FFNs, four MoE, attention at layer 2
MAX_CONTEXT = 4096


def listed():
    return [
        # one conversation generating: every MoE layer of every token is this call
        {"name": "moe_decode_1", "kind": "moe", "tokens": 1, "down": Q4, "zipf": False},
        # a handful of conversations stepping together; Q6_K down, as half of the layers have
        {"name": "moe_decode_6_q6k", "kind": "moe", "tokens": 6, "down": Q6, "zipf": False},
        # a decode batch of 16 independent conversations
        {"name": "moe_decode_16", "kind": "moe", "tokens": 16, "down": Q4, "zipf": False},
        # a short user turn, or a larger decode batch: fewer entries per expert than a matrix tile
        {"name": "moe_turn_49_q6k", "kind": "moe", "tokens": 49, "down": Q6, "zipf": False},
        # one full chunk of a prompt
        {"name": "moe_prefill_512", "kind": "moe", "tokens": 512, "down": Q4, "zipf": False},
        # a long prompt in one call with a few experts taking most of it
        {"name": "moe_prefill_4096_zipf_q6k", "kind": "moe", "tokens": 4096, "down": Q6, "zipf": True},
        # a dense layer's FFN on a ragged prompt
        {"name": "dense_130", "kind": "dense", "tokens": 130, "dtype": Q4},
        # a short-conv operator on a user turn
        {"name": "conv_77", "kind": "conv", "tokens": 77, "in": Q4, "out": Q6},
        # an attention operator absorbing a long prompt chunk by chunk, the last one ragged
        {"name": "attn_prompt_4000", "kind": "attn", "tokens": 4000},
        # one token attending over a long conversation
        {"name": "attention_9001", "kind": "attention", "positions": 9001},
        # the FFN path of several layers for one token, layer boundaries included
        {"name": "ffn_stack_1", "kind": "stack", "tokens": 1},
        # a whole turn: a prompt absorbed, then a reply token by token with logits on the host
        {"name": "chat_100_12", "kind": "chat", "prompt": 100, "reply": 12},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "moe", "dense", "conv", "attn", "attention", "stack", "chat"])
    if kind == "moe":
        return {"kind": kind, "tokens": _log(rng, 1, 4096), "down": rng.choice([Q4, Q6]), "zipf": rng.random() < 0.3}
    if kind == "dense":
        return {"kind": kind, "tokens": _log(rng, 1, 1024), "dtype": rng.choice([Q4, Q4, Q6])}
    if kind == "conv":
        return {"kind": kind, "tokens": _log(rng, 1, CHUNK), "in": rng.choice([Q4, Q6]), "out": rng.choice([Q4, Q6])}
    if kind == "attn":
        return {"kind": kind, "tokens": _log(rng, 16, 4000)}
    if kind == "attention":
        return {"kind": kind, "positions": _log(rng, 16, 32768)}
    if kind == "stack":
        return {"kind": kind, "tokens": _log(rng, 1, 16)}
    return {"kind": kind, "prompt": _log(rng, 1, 100), "reply": rng.randint(1, 12)}


# ---- inputs ------------------------------------------------------------------------------------
def _gen(seed, *stream):
    g = torch.Generator(device="cuda")
    s = 1_000_003 * int(seed) + 17
    for v in stream:
        s = (s * 6364136223846793005 + int(v) + 1442695040888963407) % (1 << 63)
    g.manual_seed(s)
    return g


def _normal(seed, stream, *shape):
    return torch.randn(*shape, generator=_gen(seed, *stream), device="cuda", dtype=torch.float32)


def _blocks(seed, stream, dtype, n_in, n_out, n_mat=1):
    """Quantised rows u8 [n_mat * n_out, n_in / 256, block bytes] on the GPU."""
    g = _gen(seed, *stream)
    rows, nb, size = n_mat * n_out, n_in // 256, 144 if dtype == Q4 else 210
    b = torch.randint(0, 256, (rows, nb, size), generator=g, device="cuda", dtype=torch.uint8)
    spread = torch.exp(0.3 * torch.randn(rows, nb, generator=g, device="cuda"))
    if dtype == Q4:
        # w = d·sc·q - dmin·m with sc, m in 0..63 and q in 0..15: dmin = 7.5·d centres it
        d = (8.7e-5 * spread).to(torch.float16)
        b[..., 0:2] = d.unsqueeze(-1).view(torch.uint8)
        b[..., 2:4] = (7.5 * d).unsqueeze(-1).view(torch.uint8)
    else:
        # w = d·sc·(q - 32) with sc in -64..63 and q in 0..63
        sc = b[..., 192:208].view(torch.int8)
        b[..., 192:208] = (sc >> 1).view(torch.uint8)
        b[..., 208:210] = (3.2e-5 * spread).to(torch.float16).unsqueeze(-1).view(torch.uint8)
    return b


def _host(b):
    return b.reshape(-1).cpu().numpy()


def _gain(seed, *stream, n=H):
    return 1.0 + 0.05 * _normal(seed, stream, n)


def _moe_parts(seed, layer, down, zipf):
    """(router, bias, gate, up, down rows) of one MoE layer on the GPU."""
    s = (layer, 1)
    bias = synth.zipf_bias(seed) if zipf else np.zeros(E, np.float32)
    return (0.02 * _normal(seed, s + (0,), E, H), bias, _blocks(seed, s + (1,), Q4, H, F, E),
            _blocks(seed, s + (2,), Q4, H, F, E), _blocks(seed, s + (3,), down, F, H, E))


def _dense_parts(seed, layer, dtype):
    s = (layer, 2)
    return (_blocks(seed, s + (0,), dtype, H, DENSE_F), _blocks(seed, s + (1,), dtype, H, DENSE_F),
            _blocks(seed, s + (2,), dtype, DENSE_F, H))


def _conv_parts(seed, layer, d_in, d_out):
    s = (layer, 3)
    return (_blocks(seed, s + (0,), d_in, H, 3 * H), 0.5 * _normal(seed, s + (1,), H * L_CACHE),
            _blocks(seed, s + (2,), d_out, H, H))


ATTN_TYPES = (Q4, Q4, Q6, Q4)  # q, k, v, o


def _attn_parts(seed, layer):
    s = (layer, 4)
    outs = (NH * HD, NKV * HD, NKV * HD, H)
    w = [_blocks(seed, s + (i,), t, H, n) for i, (t, n) in enumerate(zip(ATTN_TYPES, outs))]
    return (*w, _gain(seed, *s, 8, n=HD), _gain(seed, *s, 9, n=HD))


def _moe_weights(seed, layer, down, zipf=False):
    router, bias, gate, up, dn = _moe_parts(seed, layer, down, zipf)
    return synth.MoeWeights(H, F, E, K, router.cpu().numpy(), bias, Q4, Q4, down, _host(gate), _host(up), _host(dn))


def _dense_weights(seed, layer, dtype):
    gate, up, dn = _dense_parts(seed, layer, dtype)
    return synth.DenseWeights(H, DENSE_F, dtype, dtype, dtype, _host(gate), _host(up), _host(dn))


def _conv_weights(seed, layer, d_in, d_out):
    w_in, taps, w_out = _conv_parts(seed, layer, d_in, d_out)
    return synth.ConvWeights(H, L_CACHE, d_in, d_out, _host(w_in), _host(w_out), taps.cpu().numpy())


def _attn_weights(seed, layer):
    q, k, v, o, qn, kn = _attn_parts(seed, layer)
    return synth.AttnWeights(H, NH, NKV, HD, *ATTN_TYPES, _host(q), _host(k), _host(v), _host(o), qn.cpu().numpy(),
                             kn.cpu().numpy())


def _down_type(layer):
    return Q4 if layer % 2 == 0 else Q6


def _chat_weights(seed):
    layers = []
    for i in range(CHAT_LAYERS):
        op = _attn_weights(seed, i) if i in synth.ATTENTION_LAYERS else _conv_weights(seed, i, Q4, _down_type(i))
        ffn = _dense_weights(seed, i, Q4) if i < synth.N_DENSE else _moe_weights(seed, i, _down_type(i))
        layers.append(synth.DecoderLayerWeights(_gain(seed, i, 5).cpu().numpy(), _gain(seed, i, 6).cpu().numpy(), op,
                                                ffn))
    embd = _host(_blocks(seed, (90,), Q6, H, VOCAB))
    return synth.ModelWeights(H, VOCAB, Q6, embd, _gain(seed, 91).cpu().numpy(), layers)


def _chat_tokens(case, seed):
    n = case["prompt"] + case["reply"]
    return torch.randint(0, VOCAB, (n,), generator=_gen(seed, 92), device="cuda").cpu().numpy().astype(np.uint32)


# ---- the program ---------------------------------------------------------------------------------
class _Program:
    """What a process keeps: one context, its work on one torch stream."""
    ctx = None
    stream = None

    @classmethod
    def context(cls):
        if cls.ctx is None:
            cls.stream = torch.cuda.Stream()
            cls.ctx = Context(torch.cuda.current_device())
            cls.ctx.set_stream(cls.stream.cuda_stream)
        return cls.ctx


class _State(dict):
    """A case's inputs and handles; the handles are closed, last made first, when it goes."""

    def __init__(self, *handles, **items):
        super().__init__(**items)
        self.handles = handles

    def __del__(self):
        for h in reversed(self.handles):
            h.close()


def prepare(case, seed):
    ctx, kind = _Program.context(), case["kind"]
    if kind == "attention":
        n = case["positions"]
        return _State(case=case, q=_normal(seed, (1,), NH * HD), k=_normal(seed, (2,), n * NKV * HD),
                      v=_normal(seed, (3,), n * NKV * HD), out=torch.empty(NH * HD, device="cuda"))
    if kind == "chat":
        model = Model(ctx, _chat_weights(seed))
        cache = model.new_cache(MAX_CONTEXT)
        return _State(model, cache, case=case, model=model, cache=cache, tokens=_chat_tokens(case, seed))
    t = case["tokens"]
    io = {"case": case, "x": _normal(seed, (1,), t, H), "out": torch.empty(t, H, device="cuda")}
    if kind == "moe":
        layer = MoeLayer(ctx, _moe_weights(seed, 0, case["down"], case["zipf"]))
        return _State(layer, layer=layer, **io)
    if kind == "dense":
        layer = DenseLayer(ctx, _dense_weights(seed, 0, case["dtype"]))
        return _State(layer, layer=layer, **io)
    if kind == "conv":
        op = ConvOp(ctx, _conv_weights(seed, 0, case["in"], case["out"]))
        return _State(op, layer=op, state=torch.zeros((L_CACHE - 1) * H, device="cuda"), **io)
    if kind == "attn":
        op = AttnOp(ctx, _attn_weights(seed, 0))
        cache = op.new_cache(MAX_CONTEXT)
        return _State(op, cache, layer=op, cache=cache, **io)
    layers = []
    for i in range(STACK_LAYERS):
        ffn = (DenseLayer(ctx, _dense_weights(seed, i, Q4)) if i < synth.N_DENSE else
               MoeLayer(ctx, _moe_weights(seed, i, _down_type(i))))
        layers.append((_gain(seed, i, 6).cpu().numpy(), ffn))
    stack = FfnStack(ctx, layers, EPS)
    return _State(*(ffn for _, ffn in layers), stack, layer=stack, **io)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attention":
        return kernels.attention_decode(_Program.ctx, state["q"], state["k"], state["v"], case["positions"], NH, NKV,
                                        HD, state["out"])
    if kind == "chat":
        model, cache, tokens, p = state["model"], state["cache"], state["tokens"], case["prompt"]
        cache.reset()
        model.absorb(cache, tokens[:p], MAX_CONTEXT)
        return [model.forward_step(tok, cache) for tok in tokens[p:]]
    layer, x, out, t = state["layer"], state["x"], state["out"], case["tokens"]
    if kind == "conv":  # a new conversation: a cleared conv cache
        with torch.cuda.stream(_Program.stream):
            state["state"].zero_()
        layer.forward(state["state"], x, t, out)
        return out, state["state"]
    if kind == "attn":
        cache = state["cache"]
        for i in range(0, t, CHUNK):
            n = min(CHUNK, t - i)
            layer.forward(cache, i, x[i:i + n], n, out[i:i + n])
        cache.evict_front(t)  # the conversation is dropped
        return out
    return layer.forward(x, t, out)


# ---- what a pass cannot do without ---------------------------------------------------------------
def _w(dtype, *dims):
    return synth.byte_size(dtype, math.prod(dims))


def _moe_work(t, down):
    hit = E * (1.0 - (1.0 - K / E) ** t)  # experts chosen at least once
    return hit * (2 * _w(Q4, H, F) + _w(down, F, H)) + 4 * E * H, 2 * t * (3 * K * H * F + E * H)


def _dense_work(t, dtype):
    return 2 * _w(dtype, H, DENSE_F) + _w(dtype, DENSE_F, H), 6 * t * H * DENSE_F


def _conv_work(t, d_in, d_out):
    return _w(d_in, H, 3 * H) + _w(d_out, H, H) + 4 * H * (3 * L_CACHE - 2), 2 * t * H * (4 * H + L_CACHE + 2)


def _attn_work(t, n0=0):
    outs = (NH * HD, NKV * HD, NKV * HD, H)
    kv = 4 * 2 * NKV * HD * (n0 + t)
    seen = t * n0 + t * (t + 1) // 2
    return sum(_w(d, H, n) for d, n in zip(ATTN_TYPES, outs)) + kv, 2 * t * H * sum(outs) + 4 * NH * HD * seen


def work(case):
    kind = case["kind"]
    if kind == "attention":
        n = case["positions"]
        return {"bytes": 8 * n * NKV * HD + 8 * NH * HD, "flops": 4 * NH * HD * n}
    if kind == "chat":
        p, r = case["prompt"], case["reply"]
        nbytes, flops = 0, 2 * r * H * VOCAB
        for t, n0 in [(min(CHUNK, p - i), i) for i in range(0, p, CHUNK)] + [(1, p + i) for i in range(r)]:
            for i in range(CHAT_LAYERS):
                op = _attn_work(t, n0) if i in synth.ATTENTION_LAYERS else _conv_work(t, Q4, _down_type(i))
                ffn = _dense_work(t, Q4) if i < synth.N_DENSE else _moe_work(t, _down_type(i))
                nbytes, flops = nbytes + op[0] + ffn[0], flops + op[1] + ffn[1]
            nbytes += t * _w(Q6, H)
        return {"bytes": nbytes + r * (_w(Q6, H, VOCAB) + 4 * VOCAB), "flops": flops}
    t = case["tokens"]
    nbytes, flops = 8 * t * H, 0
    if kind == "moe":
        parts = [_moe_work(t, case["down"])]
    elif kind == "dense":
        parts = [_dense_work(t, case["dtype"])]
    elif kind == "conv":
        parts = [_conv_work(t, case["in"], case["out"])]
    elif kind == "attn":
        parts = [_attn_work(t)]
    else:
        parts = [_dense_work(t, Q4) if i < synth.N_DENSE else _moe_work(t, _down_type(i)) for i in range(STACK_LAYERS)]
    return {"bytes": nbytes + sum(b for b, _ in parts), "flops": flops + sum(f for _, f in parts)}


def tolerance(case):
    return "exact"


# ---- the same operations in 64 bits --------------------------------------------------------------
def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(b, dtype):
    """float64 [rows, n_in] of quantised rows."""
    rows, nb, _ = b.shape
    if dtype == Q4:
        d, dmin, s = _f16(b[..., 0:2]), _f16(b[..., 2:4]), b[..., 4:16].int()
        lo, mid, hi = s[..., 0:4], s[..., 4:8], s[..., 8:12]
        sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], -1).double()
        m = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], -1).double()
        q = b[..., 16:].reshape(rows, nb, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 3).reshape(rows, nb, 8, 32).double()
        w = (d * sc).unsqueeze(-1) * q - (dmin * m).unsqueeze(-1)
        return w.reshape(rows, nb * 256)
    ql = b[..., 0:128].int().reshape(rows, nb, 2, 2, 32)
    qh = b[..., 128:192].int().reshape(rows, nb, 2, 1, 32)
    quarters = [(ql[..., i % 2:i % 2 + 1, :] >> (4 * (i // 2))) & 15 | (((qh >> (2 * i)) & 3) << 4) for i in range(4)]
    q = torch.cat(quarters, 3).reshape(rows, nb, 16, 16).double() - 32
    sc = b[..., 192:208].contiguous().view(torch.int8).double()
    w = (_f16(b[..., 208:210]) * sc).unsqueeze(-1) * q
    return w.reshape(rows, nb * 256)


def _q8(x):
    v = x.reshape(*x.shape[:-1], -1, 256)
    scale = v.abs().amax(-1, keepdim=True) / 127
    return (torch.round(v / torch.where(scale > 0, scale, 1)) * scale).reshape(x.shape)


def _project(x, b, dtype):
    return _q8(x) @ _dequant(b, dtype).T


def _norm(x, gain):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gain.double()


def _swiglu(gate, up):
    return gate * torch.sigmoid(gate) * up


def _moe64(x, parts, down):
    """(output, each token's margin between the last chosen expert and the next one)."""
    router, bias, gate, up, dn = parts
    score = torch.sigmoid(x @ router.double().T)
    keys, sel = torch.topk(score + torch.from_numpy(bias).cuda().double(), K + 1, dim=-1)
    sel = sel[:, :K]
    w = score.gather(1, sel)
    w = w / (w.sum(-1, keepdim=True) + 1e-6)
    out = torch.zeros_like(x)
    for e in range(E):
        t, slot = torch.where(sel == e)
        if len(t):
            act = _swiglu(_project(x[t], gate[e * F:(e + 1) * F], Q4), _project(x[t], up[e * F:(e + 1) * F], Q4))
            out.index_add_(0, t, w[t, slot].unsqueeze(1) * _project(act, dn[e * H:(e + 1) * H], down))
    return out, keys[:, K - 1] - keys[:, K]


def _dense64(x, parts, dtype):
    gate, up, dn = parts
    return _project(_swiglu(_project(x, gate, dtype), _project(x, up, dtype)), dn, dtype)


def _conv64(x, parts, d_in, d_out):
    """(output, the conv cache's last columns) from a cleared cache."""
    w_in, taps, w_out = parts
    b, c, gate = _project(x, w_in, d_in).split(H, 1)
    bx = torch.cat([torch.zeros(L_CACHE - 1, H, device="cuda", dtype=torch.float64), b * gate])
    taps = taps.double().reshape(H, L_CACHE)
    y = sum(bx[k:k + len(x)] * taps[:, k] for k in range(L_CACHE))
    return _project(c * y, w_out, d_out), bx[len(x):].reshape(-1)


def _rope64(x):
    half = HD // 2
    angle = torch.arange(len(x), device="cuda").double().unsqueeze(1) * THETA ** (
        -torch.arange(half, device="cuda").double() / half)
    cos, sin = angle.cos().unsqueeze(1), angle.sin().unsqueeze(1)
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _attend64(q, k, v, causal):
    """q [T, NH, HD], k and v [N, NKV, HD] -> [T, NH * HD]."""
    out = torch.empty_like(q)
    for h in range(NH):
        kv = h // (NH // NKV)
        s = q[:, h] @ k[:, kv].T / math.sqrt(HD)
        if causal:
            s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, kv]
    return out.reshape(len(q), NH * HD)


def _attn64(x, parts):
    q, k, v, o, qn, kn = parts
    qr = _rope64(_norm(_project(x, q, ATTN_TYPES[0]).reshape(-1, NH, HD), qn))
    kr = _rope64(_norm(_project(x, k, ATTN_TYPES[1]).reshape(-1, NKV, HD), kn))
    vr = _project(x, v, ATTN_TYPES[2]).reshape(-1, NKV, HD)
    return _project(_attend64(qr, kr, vr, True), o, ATTN_TYPES[3])


def _chat64(case, seed):
    """The 8-bit rounding of one layer's activations moves the next layer's by about a percent of
    their size, so a reply token with a close choice of experts may go to others: it has no
    64-bit counterpart (None)."""
    margin = torch.full((case["prompt"] + case["reply"],), math.inf, device="cuda", dtype=torch.float64)
    embd = _blocks(seed, (90,), Q6, H, VOCAB)
    h = _dequant(embd[torch.from_numpy(_chat_tokens(case, seed).astype(np.int64)).cuda()], Q6)
    for i in range(CHAT_LAYERS):
        x = _norm(h, _gain(seed, i, 5))
        if i in synth.ATTENTION_LAYERS:
            h = h + _attn64(x, _attn_parts(seed, i))
        else:
            h = h + _conv64(x, _conv_parts(seed, i, Q4, _down_type(i)), Q4, _down_type(i))[0]
        y, m = _ffn64(_norm(h, _gain(seed, i, 6)), seed, i)
        h, margin = h + y, torch.minimum(m, margin)
    hidden = _q8(_norm(h[case["prompt"]:], _gain(seed, 91)))
    logits = torch.cat([hidden @ _dequant(embd[r:r + 16000], Q6).T for r in range(0, VOCAB, 16000)], 1)
    rows = [row if m > 0.01 else None for row, m in zip(logits.cpu().numpy(), margin[case["prompt"]:].tolist())]
    return rows if any(r is not None for r in rows) else None


def _ffn64(x, seed, i):
    if i < synth.N_DENSE:
        return _dense64(x, _dense_parts(seed, i, Q4), Q4), x.new_full((len(x),), math.inf)
    return _moe64(x, _moe_parts(seed, i, _down_type(i), False), _down_type(i))


def exact(case, seed):
    kind = case["kind"]
    if kind == "attention":
        s = prepare(case, seed)
        kv = [s[n].double().reshape(-1, NKV, HD) for n in ("k", "v")]
        return _attend64(s["q"].double().reshape(1, NH, HD), *kv, False).reshape(-1)
    if kind == "chat":
        return _chat64(case, seed)
    x = _normal(seed, (1,), case["tokens"], H).double()
    if kind == "moe":
        return _moe64(x, _moe_parts(seed, 0, case["down"], case["zipf"]), case["down"])[0]
    if kind == "dense":
        return _dense64(x, _dense_parts(seed, 0, case["dtype"]), case["dtype"])
    if kind == "conv":
        return _conv64(x, _conv_parts(seed, 0, case["in"], case["out"]), case["in"], case["out"])
    if kind == "attn":
        return _attn64(x, _attn_parts(seed, 0))
    for i in range(STACK_LAYERS):
        x = x + _ffn64(_norm(x, _gain(seed, i, 6)), seed, i)[0]
    return x
