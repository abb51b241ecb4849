"""The work that a program has this library do, as cases that can be timed and checked.

A case is a plain dict; prepare() makes what a program holds before the call (weights, caches, inputs,
output buffers), run() is one pass through the public entry points, work() the bytes and operations that
the pass cannot do without, and exact() the same outputs in 64 bits from plain torch.  The dimensions are the
125B-A6B model's (hidden 2560, 512 experts top-10 + shared, 24/2 attention heads of 256, GDN heads 16/48,
hyper-connections 4 x 2560, rank-320 mixers, vocabulary 248320) in both checkpoint formats (group sizes 64 and
32); whole targets have one interval of the layer schedule (three GDN layers, one attention layer)."""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "mlxfast-qwen38-125b-a6b-engine_amd"))

import mtpx  # noqa: E402

H, E, TOPK, F = 2560, 512, 10, 640
HQ, HK, D, ROT, INDEX = 24, 2, 256, 64, 128
GK, GV, TAPS = 16, 48, 4
HC, RANK, VOCAB = 4, 320, 248320
W = HC * H
SHORT_LOW, SHORT_FROM = 98304, 248044
EPS, MAX_POS, LAYERS = 1e-6, 2048, 4
QKV = 2 * HQ * D + 2 * HK * D + INDEX                 # q | gate | k | v | index key
CONV = (2 * GK + GV) * 128
GDN_IN = CONV + GV * 128 + 2 * GV                     # qkv | z | b | a
SHORTLIST = (SHORT_LOW + VOCAB - SHORT_FROM + 7) // 8 * 8
# the dense projections of the model: GDN in, attention qkv, the two output projections, lm_head
DENSE = ((GDN_IN, H), (QKV, H), (H, HQ * D), (VOCAB, H))


def listed():
    return [
        # the greedy accept of a round of draft depth 3: the smallest device call of every round
        dict(name="accept_3", kind="accept", k=3),
        # one token through an output projection: serial decode, 48 times per token
        dict(name="out_proj_1", kind="proj", n=H, k=HQ * D, gs=64, m=1),
        # the verify window's logits: the largest dense matrix of a round
        dict(name="lm_head_4", kind="proj", n=VOCAB, k=H, gs=64, m=4),
        # a projection over a whole prefill batch
        dict(name="in_proj_512", kind="proj", n=GDN_IN, k=H, gs=64, m=512),
        # the MoE block of one token in the checkpoint's own format (group size 32): a draft step, serial decode
        dict(name="moe_1_gs32", kind="moe", m=1, gs=32),
        # the MoE block of the verify window of draft depth 3
        dict(name="moe_4", kind="moe", m=4, gs=64),
        # a gated-deltanet sublayer over a verify window, half of the window committed each round
        dict(name="gdn_4", kind="gdn", s=4, keep=2, gs=64),
        # an attention + MoE layer over a verify window behind a thousand cached positions
        dict(name="layer_4", kind="layer", s=4, context=1024, gs=64),
        # a draft step of the MTP head
        dict(name="draft_1", kind="head", s=1, context=1027, gs=64),
        # the verify forward of draft depth 3
        dict(name="verify_4", kind="verify", s=4, context=1024, gs=64),
        # a short chat turn as a prompt, in the checkpoint's own format
        dict(name="prefill_75_gs32", kind="prefill", s=75, gs=32),
        # a long prompt that is no multiple of the batch or the window
        dict(name="prefill_1003", kind="prefill", s=1003, gs=64),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("accept", "proj", "proj", "moe", "gdn", "layer", "head", "verify", "prefill", "prefill"))
    gs = rng.choice((64, 64, 32))
    if kind == "accept":
        return dict(kind=kind, k=rng.randint(0, 6), vocab=_log(rng, 30011, VOCAB))
    if kind == "proj":
        if rng.random() < 0.5:
            n, k = rng.choice(DENSE)
            m = rng.randint(1, 8)
        else:
            n, k = rng.choice(DENSE[:3])
            m = _log(rng, 9, 512)
        return dict(kind=kind, n=n, k=k, gs=gs, m=m)
    if kind == "moe":
        return dict(kind=kind, m=rng.randint(1, 8), gs=gs)
    if kind == "gdn":
        s = rng.randint(1, 8)
        return dict(kind=kind, s=s, keep=rng.randint(0, s), gs=gs)
    if kind in ("layer", "verify"):
        return dict(kind=kind, s=rng.randint(1, 6), context=rng.randint(1, 1900), gs=gs)
    if kind == "head":
        return dict(kind=kind, s=1 if rng.random() < 0.5 else _log(rng, 2, 256), context=rng.randint(1, 1700), gs=gs)
    return dict(kind=kind, s=_log(rng, 9, 1003), gs=gs)


# ---- what a program holds before the call -------------------------------------------------------------------

_CTX = []


def _ctx():
    if not _CTX:
        _CTX.append(mtpx.Context(0))
    return _CTX[0]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, sigma=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * sigma).bfloat16()


def _empty(*shape, dtype=torch.bfloat16):
    return torch.zeros(*shape, dtype=dtype, device="cuda")


def _q4(g, rows, k, gs):
    """A random N(0, 0.02) matrix in the weight format: nibbles, scales, biases, packed scale/bias rows."""
    c = _ctx()
    wq = torch.empty(rows, k // 8, dtype=torch.int32, device="cuda")
    s = torch.empty(rows, k // gs, dtype=torch.bfloat16, device="cuda")
    b = torch.empty_like(s)
    step = max(1, (1 << 27) // k)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        c.affine_quantize(_randn(g, n, k, sigma=0.02), gs, wq[r:r + n], s[r:r + n], b[r:r + n])
    return wq, s, b, c.pack_sb(s, b, k, gs)


def _layer_config(gs):
    return mtpx.LayerConfig(H, E, TOPK, F, gs, HQ, HK, D, ROT, INDEX, 1e7, EPS, MAX_POS)


def _bytes_at(ptr, nbytes):
    """Device memory that the library owns (weights, caches), as a byte tensor without a copy."""
    class Mem:
        __cuda_array_interface__ = dict(shape=(nbytes,), typestr="|u1", data=(ptr, False), version=3)
    return torch.as_tensor(Mem(), device="cuda")


def _at(ptr, shape, dtype=torch.bfloat16):
    size = torch.empty((), dtype=dtype).element_size()
    return _bytes_at(ptr, math.prod(shape) * size).view(dtype).view(*shape)


def _fill_cache(kv, g, n):
    k, v, tmax = kv.buffers()
    for p in (k, v):
        _at(p, (HK, tmax, D))[:, :n] = _randn(g, HK, n, D)


def _moe_weights(g, gs):
    t = dict(router=_randn(g, E, H, sigma=0.02), shared_gate=_randn(g, H, sigma=0.02))
    for name, rows, k in (("gate", E * F, H), ("up", E * F, H), ("down", E * H, F),
                          ("sh_gate", F, H), ("sh_up", F, H), ("sh_down", H, F)):
        for part, x in zip(("_w", "_s", "_b", "_sb"), _q4(g, rows, k, gs)):
            t[name + part] = x
    return t


def prepare(case, seed):
    ctx, g, kind, gs = _ctx(), _gen(seed), case["kind"], case.get("gs")
    st = dict(case, ctx=ctx)
    if kind == "accept":
        k, v = case["k"], case.get("vocab", VOCAB)
        logits = _randn(g, k + 1, v, sigma=2.0)
        drafts = logits.float().argmax(1)[:k].int()  # a drafter that is right about seven times in ten
        miss = torch.rand(k, generator=g, device="cuda") > 0.7
        st.update(logits=logits, drafts=torch.where(miss, (drafts + 1) % v, drafts).int().contiguous(),
                  out=_empty(3, dtype=torch.int32), top=_empty(k + 1, dtype=torch.int32),
                  tokens=_empty(k + 1, dtype=torch.int32))
    elif kind == "proj":
        st.update(w=_q4(g, case["n"], case["k"], gs), x=_randn(g, case["m"], case["k"]),
                  y=_empty(case["m"], case["n"]))
    elif kind == "moe":
        m = case["m"]
        t = _moe_weights(g, gs)
        st.update(t=t, w=mtpx.moe_weights_from(t, H, E, TOPK, F, gs), x=_randn(g, m, H), y=_empty(m, H),
                  idx=_empty(m, TOPK, dtype=torch.int32), wts=_empty(m, TOPK, dtype=torch.float32),
                  logits=_empty(m, E, dtype=torch.float32))
    elif kind == "gdn":
        cfg = mtpx.GDNConfig(H, GK, GV, TAPS, gs, EPS)
        s = case["s"]
        state = mtpx.GDNState(ctx, cfg)
        st.update(conv0=_randn(g, TAPS - 1, CONV), ssm0=torch.randn(GV, 128, 128, generator=g, device="cuda") * 0.05)
        state.load(st["conv0"], st["ssm0"])
        st.update(gdn=mtpx.GDN(ctx, cfg, seed), state=state, x=_randn(g, s, H), y=_empty(s, H),
                  gated=_empty(s, GV * 128))
    elif kind == "layer":
        kv = mtpx.KVCache(ctx, HK, D, MAX_POS)
        _fill_cache(kv, g, case["context"])
        st.update(layer=mtpx.DecoderLayer(ctx, _layer_config(gs), seed), kv=kv, x=_randn(g, case["s"], H),
                  y=_empty(case["s"], H))
    elif kind == "head":
        s = case["s"]
        kv = mtpx.KVCache(ctx, HK, D, MAX_POS)
        _fill_cache(kv, g, case["context"])
        head = mtpx.MTPHead(ctx, mtpx.HeadConfig(_layer_config(gs), HC, RANK, VOCAB, SHORT_LOW, SHORT_FROM), seed)
        st.update(head=head, kv=kv, ids=torch.randint(VOCAB, (s,), generator=g, device="cuda", dtype=torch.int32),
                  multi=_randn(g, s, W), multi_next=_empty(s, W), sample=_empty(s, H),
                  draft=_empty(1, dtype=torch.int32))
    else:
        cfg = mtpx.TargetConfig(_layer_config(gs), GK, GV, TAPS, LAYERS, 4, HC, RANK, VOCAB)
        cfg.ple_layer = -1
        target = mtpx.Target(ctx, cfg, seed)
        s = case["s"]
        ids = torch.randint(VOCAB, (s,), generator=g, device="cuda", dtype=torch.int32)
        st.update(target=target, state=mtpx.TargetState(ctx, target), ids=ids, multi=_empty(s, W))
        if kind == "verify":
            st.update(logits=_empty(s, VOCAB), mixed=_empty(s, H))
            prompt = torch.randint(VOCAB, (case["context"],), generator=g, device="cuda", dtype=torch.int32)
            target.prefill(st["state"], prompt)
        else:
            st.update(logits=_empty(VOCAB))
    return st


# ---- one pass -----------------------------------------------------------------------------------------------

def run(st):
    ctx, kind = st["ctx"], st["kind"]
    if kind == "accept":
        ctx.accept_greedy_bf16(st["logits"], st["drafts"] if st["k"] else None, 1024, st["out"], st["top"],
                               st["tokens"])
        return dict(out=st["out"], top=st["top"], tokens=st["tokens"])  # past the accepted count: zeros
    if kind == "proj":
        ctx.qmv(*st["w"][:3], st["gs"], st["x"], st["y"], sb=st["w"][3])
        return st["y"]
    if kind == "moe":
        ctx.moe_forward(st["w"], st["x"], st["y"], st["idx"], st["wts"], st["logits"])
        return dict(y=st["y"], idx=st["idx"], weights=st["wts"], logits=st["logits"])
    if kind == "gdn":
        st["gdn"].forward(st["state"], st["x"], st["y"], st["gated"])
        st["state"].commit(st["keep"])
        return dict(y=st["y"], gated=st["gated"])
    if kind == "layer":
        st["kv"].offset = st["context"]
        st["layer"].forward(st["kv"], st["x"], st["y"])
        return st["y"]
    if kind == "head":
        st["kv"].offset = st["context"]
        st["head"].forward(st["kv"], st["ids"], st["multi"], st["multi_next"], st["sample"], st["draft"])
        return dict(multi=st["multi_next"], sample=st["sample"], draft=st["draft"])
    if kind == "verify":  # the window is discarded by the next one
        st["target"].verify(st["state"], st["ids"], st["logits"], st["multi"], st["mixed"])
        return dict(logits=st["logits"], multi=st["multi"], mixed=st["mixed"])
    st["state"].reset()  # a new request's prompt
    st["target"].prefill(st["state"], st["ids"], st["logits"], st["multi"])
    return dict(logits=st["logits"], multi=st["multi"])


# ---- what a pass cannot do without --------------------------------------------------------------------------

def _w_bytes(n, k, gs):
    return n * k // 2 + 4 * n * k // gs


def _touched(m):
    return E * (1 - (1 - TOPK / E) ** m)


def _proj_work(m, gs, *mats):
    return sum(_w_bytes(n, k, gs) for n, k in mats), sum(2 * m * n * k for n, k in mats)


def _moe_work(m, gs):
    one_b, one_f = _proj_work(1, gs, (F, H), (F, H), (H, F))
    return (_touched(m) + 1) * one_b + 2 * E * H, m * (TOPK + 1) * one_f + 2 * m * E * H


def _attn_work(m, gs, context):
    b, f = _proj_work(m, gs, (QKV, H), (H, HQ * D))
    keys = context + (m + 1) / 2
    return b + 4 * HK * D * (context + m), f + 4 * m * keys * HQ * D


def _gdn_work(m, gs):
    b, f = _proj_work(m, gs, (GDN_IN, H), (H, GV * 128))
    return b + 2 * 4 * GV * 128 * 128, f + m * GV * 128 * 128 * 7


def _mixer_work(m, gs, n):
    b, f = _proj_work(m, gs, (RANK + HC, W), (W, RANK))
    return n * b, n * f


def work(case):
    kind, gs = case["kind"], case.get("gs")
    if kind == "accept":
        n = (case["k"] + 1) * case.get("vocab", VOCAB)
        return dict(bytes=2 * n, flops=n)
    m = case.get("m", case.get("s"))
    if kind == "proj":
        parts = [_proj_work(m, gs, (case["n"], case["k"])), (2 * m * (case["n"] + case["k"]), 0)]
    elif kind == "moe":
        parts = [_moe_work(m, gs), (4 * m * H + 4 * m * E, 0)]
    elif kind == "gdn":
        parts = [_gdn_work(m, gs), (4 * m * H + 2 * m * GV * 128, 0)]
    elif kind == "layer":
        parts = [_attn_work(m, gs, case["context"]), _moe_work(m, gs), (4 * m * H, 0)]
    elif kind == "head":
        parts = [_attn_work(m, gs, case["context"]), _moe_work(m, gs), _mixer_work(m, gs, 3),
                 _proj_work(m, gs, (H, H)), _proj_work(HC * m, gs, (H, H)), _proj_work(1, gs, (SHORTLIST, H)),
                 (m * (H // 2 + 4 * W + 2 * H), 0)]
    else:
        verify = kind == "verify"
        attn = _attn_work(m, gs, case["context"] if verify else 0)
        parts = [_gdn_work(m, gs)] * 3 + [attn] + [_moe_work(m, gs)] * 4 + [_mixer_work(m, gs, 9)]
        rows = m if verify else 1
        parts += [_proj_work(rows, gs, (VOCAB, H)), (m * (H // 2 + 2 * W) + 2 * rows * VOCAB, 0)]
    return dict(bytes=sum(b for b, _ in parts), flops=sum(f for _, f in parts))


def tolerance(case):
    # four times the distance from exact() that the 64-bit comparison shows: a projection rounds once (1.7e-3),
    # the MoE block and the GDN sublayer at every step between (6e-3), a layer adds its input (2.8e-3), the head
    # carries streams through three mixers (6e-3) and a whole target through four layers and their routers' choices
    kind = case["kind"]
    if kind == "accept":
        return "exact"
    if kind == "proj":
        return dict(rel=6e-3)
    if kind == "layer":
        return dict(rel=1.2e-2)
    if kind in ("moe", "gdn", "head"):
        return dict(rel=2.5e-2, differ=0.0)
    return dict(rel=3e-2, max=0.9)


# ---- the same in 64 bits ------------------------------------------------------------------------------------

def _deq(w, s, b, gs):
    """float64 of packed rows [..., k/8] with scales and biases [..., k/gs]."""
    sh = torch.arange(0, 32, 4, device=w.device, dtype=torch.int32)
    q = ((w.unsqueeze(-1) >> sh) & 15).flatten(-2).double()
    q = q.unflatten(-1, (-1, gs))
    return (q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).flatten(-2)


class _Q:
    """A q4 matrix [rows, k] on the device, from tensors or from the library's pointers."""

    def __init__(self, w, s, b, rows, k, gs):
        if isinstance(w, int):
            w, s, b = (_at(w, (rows, k // 8), torch.int32), _at(s, (rows, k // gs)), _at(b, (rows, k // gs)))
        self.w, self.s, self.b, self.gs = w, s, b, gs

    def rows(self, r0, n):
        return _deq(self.w[r0:r0 + n], self.s[r0:r0 + n], self.b[r0:r0 + n], self.gs)

    def at(self, ids):
        ids = ids.long()
        return _deq(self.w[ids], self.s[ids], self.b[ids], self.gs)

    def __call__(self, x):
        return torch.cat([x @ self.rows(r, min(16384, self.w.shape[0] - r)).T
                          for r in range(0, self.w.shape[0], 16384)], -1)


def _field(m, name, rows, k, gs):
    return _Q(getattr(m, name + "_w"), getattr(m, name + "_s"), getattr(m, name + "_b"), rows, k, gs)


def _struct(q, rows, k, gs):
    return _Q(q.w, q.s, q.b, rows, k, gs)


def _rms(x, eps=EPS):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt()


def _silu(x):
    return x * torch.sigmoid(x)


def _x_moe(m, x, gs):
    """(y, idx, weights, logits) of the MoE block; m: the weights struct."""
    logits = x @ _at(m.router, (E, H)).double().T
    top, idx = logits.topk(TOPK, -1)
    wts = top.softmax(-1)
    gate, up = _field(m, "gate", E * F, H, gs), _field(m, "up", E * F, H, gs)
    down = _field(m, "down", E * H, F, gs)
    if m.shared_gate_w:
        sg = _field(m, "shared_gate", 1, H, gs)(x)
    else:
        sg = (x @ _at(m.shared_gate, (H,)).double()).unsqueeze(-1)
    sh = [_field(m, "sh_" + n, r, k, gs) for n, r, k in (("gate", F, H), ("up", F, H), ("down", H, F))]
    y = torch.sigmoid(sg) * sh[2](_silu(sh[0](x)) * sh[1](x))
    for e in idx.unique().tolist():
        tok, rank = (idx == e).nonzero(as_tuple=True)
        a = _silu(x[tok] @ gate.rows(e * F, F).T) * (x[tok] @ up.rows(e * F, F).T)
        y.index_add_(0, tok, wts[tok, rank].unsqueeze(-1) * (a @ down.rows(e * H, H).T))
    return y, idx, wts, logits


def _x_attn(lw, x, gs, pos, keys, values):
    """Attention sublayer on x at position pos behind keys/values [HK, pos, D] (grown by the window)."""
    s = x.shape[0]
    qkv = _Q(lw.qkv_w, lw.qkv_s, lw.qkv_b, QKV, H, gs)(x)
    q, gate = qkv[:, :HQ * D].reshape(s, HQ, D), qkv[:, HQ * D:2 * HQ * D]
    k, v = qkv[:, 2 * HQ * D:2 * HQ * D + 2 * HK * D].reshape(s, 2, HK, D).unbind(1)
    cos, sin = (_at(p, (MAX_POS, ROT)).double()[pos:pos + s].unsqueeze(1) for p in (lw.rope_cos, lw.rope_sin))

    def rope(t, w):
        t = _rms(t) * _at(w, (D,)).double()
        r, h = t[..., :ROT], ROT // 2
        return torch.cat([r * cos + torch.cat([-r[..., h:], r[..., :h]], -1) * sin, t[..., ROT:]], -1)

    q, k = rope(q, lw.q_norm), rope(k, lw.k_norm)
    keys, values = torch.cat([keys, k.transpose(0, 1)], 1), torch.cat([values, v.transpose(0, 1)], 1)
    sc = torch.matmul(q.reshape(s, HK, HQ // HK, D).permute(1, 2, 0, 3).reshape(HK, -1, D),
                      keys.transpose(1, 2).contiguous()).reshape(HK, HQ // HK, s, -1) / math.sqrt(D)
    seen = torch.arange(pos + s, device="cuda") <= torch.arange(pos, pos + s, device="cuda").unsqueeze(1)
    p = sc.masked_fill(~seen, -math.inf).softmax(-1)
    o = torch.matmul(p.reshape(HK, -1, pos + s), values).reshape(HK, HQ // HK, s, D).permute(2, 0, 1, 3)
    return _Q(lw.o_w, lw.o_s, lw.o_b, H, HQ * D, gs)(o.reshape(s, HQ * D) * torch.sigmoid(gate))


def _x_gdn(gw, x, gs, conv, ssm):
    """(y, gated) of the GDN sublayer behind conv rows [TAPS-1, CONV] and state [GV, 128, 128]."""
    s = x.shape[0]
    proj = _struct(gw.in_proj, GDN_IN, H, gs)(x)
    rows = torch.cat([conv, proj[:, :CONV]])
    taps = _at(gw.conv_w, (CONV, TAPS)).double()
    u = _silu(sum(rows[j:j + s] * taps[:, j] for j in range(TAPS)))
    q, k = (_rms(t.reshape(s, GK, 128)).repeat_interleave(GV // GK, 1) for t in (u[:, :GK * 128],
                                                                                 u[:, GK * 128:2 * GK * 128]))
    q, k, v = q / 128, k / math.sqrt(128), u[:, 2 * GK * 128:].reshape(s, GV, 128)
    z, b, a = proj[:, CONV:CONV + GV * 128], proj[:, CONV + GV * 128:][:, :GV], proj[:, CONV + GV * 128 + GV:]
    decay = (_at(gw.neg_exp_alog, (GV,), torch.float32).double()
             * torch.nn.functional.softplus(a + _at(gw.dt_bias, (GV,)).double())).exp()
    beta, out = torch.sigmoid(b), []
    for t in range(s):
        ssm = ssm * decay[t, :, None, None]
        delta = (v[t] - (ssm * k[t].unsqueeze(1)).sum(-1)) * beta[t].unsqueeze(-1)
        ssm = ssm + delta.unsqueeze(-1) * k[t].unsqueeze(1)
        out.append((ssm * q[t].unsqueeze(1)).sum(-1))
    o = _rms(torch.stack(out)) * _at(gw.norm_w, (128,)).double()
    gated = o.reshape(s, GV * 128) * torch.sigmoid(z)
    return _struct(gw.out_proj, H, GV * 128, gs)(gated), gated


def _x_norm(m, stream, gs, last=False):
    """The mixer m on the streams [S, HC, H]: (x [S, H], inject [S, HC])."""
    n = (_rms(stream) * _at(m.norm_scale, (HC, H)).double()).flatten(1)
    up = _struct(m.up, W, RANK, gs)(_silu(_struct(m.down, RANK, W, gs)(n)))
    x = (torch.sigmoid(up) * n).unflatten(1, (HC, H)).sum(1)
    return x, None if last else 2 * torch.sigmoid(_struct(m.inject, HC, W, gs)(n))


def _inject(stream, out, j):
    return stream + out.unsqueeze(1) * j.unsqueeze(-1)


def _x_layer(st, x, gs):
    lw, c = st["layer"].weights(), st["context"]
    k, v, tmax = st["kv"].buffers()
    kc, vc = (_at(p, (HK, tmax, D))[:, :c].double() for p in (k, v))
    s_ = x + _x_attn(lw, _rms(x) * _at(lw.attn_norm, (H,)).double(), gs, c, kc, vc)
    return s_ + _x_moe(lw.moe, _rms(s_) * _at(lw.post_norm, (H,)).double(), gs)[0]


def _x_head(st, gs):
    hw, c = st["head"].weights(), st["context"]
    k, v, tmax = st["kv"].buffers()
    kc, vc = (_at(p, (HK, tmax, D))[:, :c].double() for p in (k, v))
    e = _rms(_struct(hw.embed, VOCAB, H, gs).at(st["ids"])) * _at(hw.pre_norm_embedding, (H,)).double()
    m = _rms(st["multi"].double()) * _at(hw.pre_norm_hidden, (W,)).double()
    stream = _struct(hw.fc_hidden, H, H, gs)(m.reshape(-1, H)).reshape(-1, HC, H)
    stream = stream + _struct(hw.fc_embedding, H, H, gs)(e).unsqueeze(1)
    x, j = _x_norm(hw.attn_hc, stream, gs)
    stream = _inject(stream, _x_attn(hw.layer, x, gs, c, kc, vc), j)
    x, j = _x_norm(hw.mlp_hc, stream, gs)
    stream = _inject(stream, _x_moe(hw.layer.moe, x, gs)[0], j)
    return dict(multi=stream.flatten(1), sample=_x_norm(hw.final_hc, stream, gs, last=True)[0], draft=None)


def _x_target(st, gs):
    target, prefill = st["target"], st["kind"] == "prefill"
    c = 0 if prefill else st["context"]
    tw = target.weights()
    stream = _struct(tw.embed, VOCAB, H, gs).at(st["ids"]).unsqueeze(1).expand(-1, HC, -1)
    for i in range(LAYERS):
        lw = target.layer_weights(i)
        x, j = _x_norm(lw.attn_hc, stream, gs)
        if lw.kind == 1:
            kc = vc = torch.zeros(HK, 0, D, dtype=torch.float64, device="cuda")
            if not prefill:
                k, v, tmax = st["state"].kv(i).buffers()
                kc, vc = (_at(p, (HK, tmax, D))[:, :c].double() for p in (k, v))
            out = _x_attn(lw.attn, x, gs, c, kc, vc)
        else:
            conv, ssm = _empty(TAPS - 1, CONV), _empty(GV, 128, 128, dtype=torch.float32)
            if not prefill:
                st["state"].gdn(i).store(conv, ssm)
            out = _x_gdn(lw.gdn, x, gs, conv.double(), ssm.double())[0]
        stream = _inject(stream, out, j)
        x, j = _x_norm(lw.mlp_hc, stream, gs)
        stream = _inject(stream, _x_moe(lw.attn.moe, x, gs)[0], j)
    mixed, _ = _x_norm(tw.final_hc, stream, gs, last=True)
    logits = _struct(tw.lm_head, VOCAB, H, gs)(mixed[-1:] if prefill else mixed)
    multi = stream.flatten(1)
    return dict(logits=logits[0], multi=multi) if prefill else dict(logits=logits, multi=multi, mixed=mixed)


def exact(case, seed):
    st = prepare(case, seed)
    kind, gs = case["kind"], case.get("gs")
    if kind == "accept":
        return None
    if kind == "proj":
        return _Q(*st["w"][:3], case["n"], case["k"], gs)(st["x"].double())
    if kind == "moe":
        y, _, wts, logits = _x_moe(st["w"], st["x"].double(), gs)
        return dict(y=y, idx=None, weights=wts, logits=logits)
    if kind == "gdn":
        y, gated = _x_gdn(st["gdn"].weights(), st["x"].double(), gs, st["conv0"].double(), st["ssm0"].double())
        return dict(y=y, gated=gated)
    if kind == "layer":
        return _x_layer(st, st["x"].double(), gs)
    if kind == "head":
        return _x_head(st, gs)
    return _x_target(st, gs)
