"""The workloads this framework is timed on: what a program that uses it has it do, each through a public entry point.

Kinds of case (the "op" field):
  linear   one bf16 or W8A8 Linear with its epilogue, at the widths of the three models' layers and 1 .. 186,624 rows
  sdpa     one attention call: the tower's (16 heads x 72, views of the fused qkv output), the text decoder's prefill
           (32 heads x 64, prefix + causal mask, keys read from the cache), the tracker's (12 heads x 64)
  rglru    one RG-LRU layer step on its own
  tower    the vision tower (its first `layers` blocks and the final LayerNorm) on a batch of crops, as its HIP graph
  prefill  the text decoder's prompt prefill, as its HIP graph
  query    the text decoder's yes / no questions over a prefix that is in the cache, as its HIP graph
  decode   one decode step at the end of a prefilled cache
  track    the tracker on one streamed frame (its HIP graph) or on a clip of frames at once

Weights are N(0, 0.02), LayerNorms have gamma 1 and beta 0, pixels are uniform: the synthetic models that the tests and
the benchmark use, drawn on the GPU from the seed.
"""
import math

import torch
import torch.nn.functional as F

from strix_halo_maxx_amd import md2, md2text, ops, trecvit
from strix_halo_maxx_amd.synth import TRV, TXT, VIS, freqs_cis

BF, F64 = torch.bfloat16, torch.float64

# (N, K) of the models' Linears: the tower's qkv, proj, fc1, fc2 and projection MLP; the text layers' qkv, proj, fc1,
# fc2; the tracker's yx, out, gated up, down, qkv
LINEARS = ((3456, 1152), (1152, 1152), (4304, 1152), (1152, 4304), (8192, 2304), (2048, 8192), (6144, 2048),
           (2048, 2048), (8192, 2048), (1536, 768), (768, 768), (6144, 768), (768, 3072), (2304, 768))


def listed():
    return [
        # the tracker's recurrence as a layer of its own on one frame's tokens: the smallest call that programs make
        dict(name="rglru_frame", op="rglru", t=1280),
        # the tower's attention at its throughput batch of 256 crops
        dict(name="sdpa_b256", op="sdpa", form="vision", b=256, t=729),
        # the largest single product: fc1 + GELU on 256 crops
        dict(name="fc1_b256", op="linear", m=186624, n=4304, k=1152, act="tanh", res=False, w8a8=False),
        # the W8A8 text Linear on a prefill's 794 rows, quantisation of its input included
        dict(name="fc1_w8a8", op="linear", m=794, n=8192, k=2048, act="tanh", res=False, w8a8=True),
        # the whole tower on one image: the latency of a frame
        dict(name="tower_b1", op="tower", b=1, layers=27),
        # three blocks on one global and twelve local crops: the tower's rate on a large image
        dict(name="blocks_b13", op="tower", b=13, layers=3),
        # image tokens and a prompt of 64 ids through text layers
        dict(name="prefill", op="prefill", n_img=729, n_ids=64, layers=4, ctx=1024, w8a8=False),
        # one 32-id yes / no question over an image that is in the cache
        dict(name="query", op="query", n_img=729, nq=1, l=32, layers=8, ctx=832, w8a8=False),
        # one generated token after an image and a prompt
        dict(name="decode", op="decode", n_img=729, n_ids=64, layers=24, ctx=1024, w8a8=False),
        # the same far into the longest context the model has, int8 weights
        dict(name="decode_long", op="decode", n_img=729, n_ids=771, layers=4, ctx=2048, w8a8=True),
        # one frame of a 480p video through the tracker: its latency
        dict(name="track_frame", op="track", frames=1, h=480, w=854, layers=4),
        # sixteen frames at once: its rate on recorded video
        dict(name="track_clip", op="track", frames=16, h=256, w=256, layers=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("linear", "linear", "sdpa", "rglru", "tower", "prefill", "query", "decode", "track"))
    w8a8 = rng.random() < 0.3
    if op == "linear":
        if w8a8:
            n, k = rng.choice(LINEARS[5:9])
            return dict(op=op, m=_log(rng, 1, 8000), n=n, k=k, act=rng.choice(("none", "tanh")),
                        res=rng.random() < 0.5, w8a8=True)
        n, k = rng.choice(LINEARS)
        return dict(op=op, m=_log(rng, 1, min(186624, 9 * 10 ** 11 // (n * k))), n=n, k=k,
                    act=rng.choice(("none", "tanh", "erf")), res=rng.random() < 0.4, w8a8=False)
    if op == "sdpa":
        form = rng.choice(("vision", "text", "track"))
        t = _log(rng, 64, 1500) if rng.random() < 0.6 else dict(vision=729, text=794, track=1280)[form]
        hi = max(1, min(256, int(256 * (729 / t) ** 2 * (1.0 if form == "vision" else 0.5))))
        return dict(op=op, form=form, b=_log(rng, 1, hi), t=t)
    if op == "rglru":
        return dict(op=op, t=_log(rng, 1, 100000))
    if op == "tower":
        layers = rng.randint(1, 4)
        return dict(op=op, b=_log(rng, 1, 40 // layers), layers=layers)
    if op == "prefill":
        n_img, n_ids = _log(rng, 16, 1200), _log(rng, 1, 300)
        return dict(op=op, n_img=n_img, n_ids=n_ids, layers=rng.randint(1, 3 if w8a8 else 4),
                    ctx=-(-(n_img + max(n_ids, 32) + 1) // 64) * 64, w8a8=w8a8)
    if op == "query":
        n_img, l = _log(rng, 64, 1200), _log(rng, 4, 64)
        return dict(op=op, n_img=n_img, nq=rng.randint(1, 6), l=l, layers=rng.randint(1, 2 if w8a8 else 6),
                    ctx=-(-(n_img + l + 1) // 64) * 64, w8a8=w8a8)
    if op == "decode":
        n_img, n_ids = _log(rng, 16, 1200), _log(rng, 1, 700)
        return dict(op=op, n_img=n_img, n_ids=n_ids, layers=rng.randint(1, 4 if w8a8 else 12),
                    ctx=rng.choice([c for c in (512, 1024, 1536, 2048) if c > n_img + max(n_ids, 32) + 8]), w8a8=w8a8)
    frames = rng.choice((1, 1, 2, 4, 7, 16))
    h = rng.choice((256, rng.randint(180, 1080)))
    return dict(op=op, frames=frames, h=h, w=256 if h == 256 else h * 16 // 9, layers=rng.randint(1, 4))


class _Draws:
    """Seeded tensors on the GPU, in the order they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=0.02, dtype=BF):
        return (torch.randn(*shape, generator=self.g, device="cuda") * std).to(dtype)

    def ids(self, n, hi):
        return torch.randint(0, hi, (n,), generator=self.g, device="cuda")

    def pixels(self, *shape):
        return torch.randint(0, 256, shape, generator=self.g, device="cuda", dtype=torch.uint8)

    def linear(self, w, name, n, k):
        w[name + ".weight"], w[name + ".bias"] = self.normal(n, k), self.normal(n)

    def norm(self, w, name, d):
        w[name + ".weight"] = torch.ones(d, device="cuda", dtype=BF)
        w[name + ".bias"] = torch.zeros(d, device="cuda", dtype=BF)


def _vision_weights(d, layers):
    D, ff, w = VIS["dim"], VIS["ff"], {}
    d.linear(w, "patch_emb", D, 3 * VIS["patch"] ** 2)
    w["pos_emb"] = d.normal(1, VIS["ntok"], D)
    for i in range(layers):
        p = f"blocks.{i}."
        d.norm(w, p + "ln1", D)
        d.norm(w, p + "ln2", D)
        for name, n, k in (("attn.qkv", 3 * D, D), ("attn.proj", D, D), ("mlp.fc1", ff, D), ("mlp.fc2", D, ff)):
            d.linear(w, p + name, n, k)
    d.norm(w, "post_ln", D)
    return w


def _text_weights(d, layers):
    D, ff, V = TXT["dim"], TXT["ff"], TXT["vocab"]
    w = {"wte": d.normal(V, D)}
    for i in range(layers):
        p = f"blocks.{i}."
        d.norm(w, p + "ln", D)
        for name, n, k in (("attn.qkv", 3 * D, D), ("attn.proj", D, D), ("mlp.fc1", ff, D), ("mlp.fc2", D, ff)):
            d.linear(w, p + name, n, k)
    d.norm(w, "post_ln", D)
    d.linear(w, "lm_head", V, D)
    return w


def _rglru_weights(d):
    H = TRV["heads"]
    return dict(input_gate_w=d.normal(H, 64, 64), input_gate_b=d.normal(H, 64), a_gate_w=d.normal(H, 64, 64),
                a_gate_b=d.normal(H, 64), a_param=d.normal(TRV["dim"], std=1.0))


def _track_weights(d, layers):
    D, w = TRV["dim"], {}
    for i in range(layers):
        sb, vb = f"blocks.{i}.ssm_block.", f"blocks.{i}.vit_block."
        rb = sb + "recurrent_block."
        w[sb + "temporal_pre_norm.scale"], w[sb + "channel_pre_norm.scale"] = d.normal(D, std=0.1), d.normal(D, std=0.1)
        for name, n, k in ((rb + "linear_yx", 2 * D, D), (rb + "linear_out", D, D),
                           (sb + "mlp_block.ffw_up", 2 * TRV["ff_gated"], D),
                           (sb + "mlp_block.ffw_down", D, TRV["ff_gated"]), (vb + "self_attention.out_proj", D, D),
                           (vb + "mlp.0", TRV["ff_vit"], D), (vb + "mlp.3", D, TRV["ff_vit"])):
            d.linear(w, name, n, k)
        w[vb + "self_attention.in_proj_weight"] = d.normal(3 * D, D)
        w[vb + "self_attention.in_proj_bias"] = d.normal(3 * D)
        w[rb + "conv_1d.w"], w[rb + "conv_1d.b"] = d.normal(TRV["conv_taps"], D), d.normal(D)
        r = _rglru_weights(d)
        w[rb + "rg_lru.a_param"] = r["a_param"]
        for gate in ("input_gate", "a_gate"):
            w[rb + f"rg_lru.{gate}.w"], w[rb + f"rg_lru.{gate}.b"] = r[gate + "_w"], r[gate + "_b"]
        d.norm(w, vb + "ln_1", D)
        d.norm(w, vb + "ln_2", D)
    d.norm(w, "encoder_norm", D)
    w["lin_proj.weight"], w["lin_proj.bias"] = d.normal(D, 3, TRV["patch"], TRV["patch"]), d.normal(D)
    w["image_pos_emb"] = d.normal(1, TRV["n_img"], D)
    d.linear(w, "query_proj", D, 2)
    Hh = TRV["head_hidden"]
    for hn, no in (("coordinate_head", 2 * TRV["img"]), ("visible_head", 1)):
        for i, n, k in ((0, Hh, D), (3, Hh, Hh), (6, no, Hh)):
            w[f"{hn}.{i}.weight"] = d.normal(n, k, std=0.05, dtype=torch.float32)
            w[f"{hn}.{i}.bias"] = d.normal(n, dtype=torch.float32)
        for i in (1, 4):
            w[f"{hn}.{i}.weight"] = 1 + d.normal(Hh, std=0.1, dtype=torch.float32)
            w[f"{hn}.{i}.bias"] = d.normal(Hh, std=0.1, dtype=torch.float32)
    return w


def _inputs(c, seed):
    """The weights and inputs of a case, as plain tensors."""
    d, op = _Draws(seed), c["op"]
    if op == "linear":
        s = {}
        d.linear(s, "lin", c["n"], c["k"])
        s["x"] = d.normal(c["m"], c["k"], std=1.0)  # a normalised activation
        s["res"] = d.normal(c["m"], c["n"], std=1.0) if c["res"] else None
        return s
    if op == "sdpa":
        b, t = c["b"], c["t"]
        h, hd = _heads(c)
        if c["form"] == "text":  # queries of their own, keys and values in a longer cache
            return dict(q=d.normal(b, h, t, hd, std=0.9), kc=d.normal(b, h, t + 64, hd, std=0.9),
                        vc=d.normal(b, h, t + 64, hd, std=0.9))
        return dict(qkv=d.normal(b, t, 3, h, hd, std=0.7))
    if op == "rglru":
        return dict(w=_rglru_weights(d), x=d.normal(c["t"], TRV["dim"], std=0.5),
                    h0=d.normal(c["t"], TRV["dim"], std=0.5, dtype=torch.float32))
    if op == "tower":
        return dict(w=_vision_weights(d, c["layers"]), img=d.pixels(c["b"], VIS["img"], VIS["img"], 3))
    if op == "track":
        return dict(w=_track_weights(d, c["layers"]), frames=d.pixels(2 * c["frames"], c["h"], c["w"], 3),
                    q=torch.rand(TRV["n_q"], 2, generator=d.g, device="cuda").to(BF))
    s = dict(w=_text_weights(d, c["layers"]), img=d.normal(c["n_img"], TXT["dim"], std=0.5))
    if op == "query":
        s["ids"] = d.ids(c["nq"] * c["l"], TXT["vocab"]).view(c["nq"], c["l"])
        s["last"] = [c["l"] - (b % c["l"]) for b in range(c["nq"])]  # ids of each question; the rest is padding
    else:
        s["ids"], s["next"] = d.ids(c["n_ids"], TXT["vocab"]), int(d.ids(1, TXT["vocab"]))
    return s


def _heads(c):
    return dict(vision=(VIS["heads"], VIS["hd"]), text=(TXT["heads"], TXT["hd"]), track=(TRV["heads"], TRV["hd"]))[c["form"]]


YES, NO = (5297, 3363, 3763), (1400, 645, 3919)


def prepare(c, seed):
    s, op = _inputs(c, seed), c["op"]
    s["c"] = c
    if op == "linear":
        s["lin"] = (ops.MxI8Lin if c["w8a8"] else ops.MxLin)(s["lin.weight"], s["lin.bias"])
    elif op == "sdpa":
        s["attn"] = ops.Attn(*_heads(c)[:1], c["t"], _heads(c)[1])
        if c["form"] != "text":
            s["q"], s["k"], s["v"] = (s["qkv"][:, :, i].transpose(1, 2) for i in range(3))
        else:
            s["k"], s["v"] = s["kc"][:, :, :c["t"]], s["vc"][:, :, :c["t"]]
    elif op == "rglru":
        s["layer"] = trecvit.RGLRU(**s["w"])
    elif op == "tower":
        s["vt"], s["buf"] = md2.VisionTower(s["w"]), torch.zeros_like(s["img"])
        s["graph"], s["out"] = s["vt"].capture(s["buf"])
    elif op == "track":
        m = s["model"] = trecvit.TRecViT(s["w"])
        n = c["frames"]
        if n == 1:
            m.step(s["frames"][0], s["q"])  # picks every kernel before the graphs are recorded
            m.capture()
            m.reset()
            m.step(s["frames"][0], s["q"], use_graph=True)
        else:
            m.clip_state(n)
            m.forward_clip(s["frames"][:n], s["q"])
    else:
        kw = dict(ctx=c["ctx"], w8a8=c["w8a8"])
        if op == "query":
            td = md2text.TextDecoder(s["w"], nq=c["nq"], L=c["l"], yes_ids=YES, no_ids=NO, **kw)
            td.encode(s["img"])
            td.set_questions([s["ids"][b, :n].tolist() for b, n in enumerate(s["last"])])
            td.capture_query()
        else:
            td = md2text.TextDecoder(s["w"], **kw)
            if op == "prefill":
                td.capture_prefill(c["n_img"], c["n_ids"])
            else:
                td.prefill(s["img"], s["ids"])
                s["row"] = td.wte[s["next"]].clone()
        s["td"] = td
    if op != "track":
        s.pop("w", None)
    return s


def run(s):
    c = s["c"]
    op = c["op"]
    if op == "linear":
        return s["lin"](s["x"], act=None if c["act"] == "none" else c["act"], res=s["res"])
    if op == "sdpa":
        if c["form"] == "text":  # the last 64 rows (or the last of few) are the prompt, the others the image prefix
            return ops.sdpa(s["q"], s["k"], s["v"], causal_from=_prefix(c["t"]))
        return s["attn"](s["q"], s["k"], s["v"])
    if op == "rglru":
        return s["layer"].forward(s["x"], s["h0"])
    if op == "tower":
        s["buf"].copy_(s["img"])
        s["graph"].replay()
        return s["out"]
    if op == "track":
        m, n = s["model"], c["frames"]
        if n == 1:
            # the graph reads out tracks too; they are not returned, since with random weights they hang on an argmax
            out = m.step(s["frames"][1], s["q"], use_graph=True)
            return dict(tokens=out, logits=m.logits, vis=m.vis, h=m.h)
        return dict(tokens=m.forward_clip(s["frames"][n:], s["q"]), h=m.h)
    td = s["td"]
    if op == "prefill":
        out, n = td.prefill(s["img"], s["ids"]), 1 + c["n_img"] + c["n_ids"]
    elif op == "query":
        out, n = td.query(), 1 + c["n_img"] + c["l"]
        return dict(logits=out, k=[k[:, :, :n] for k in td.kc], v=[v[:, :, :n] for v in td.vc])
    else:
        # the token is given, as in teacher forcing or rescoring: an argmax would hang on near ties
        td.start_decode()
        td.xd[0].copy_(s["row"])
        td.decode_step(logits=True)
        out, n = None, 2 + c["n_img"] + c["n_ids"]
    return dict(hidden=out, logits=td.logits, k=[k[:, :, :n] for k in td.kc], v=[v[:, :, :n] for v in td.vc])


def _prefix(t):
    return t - min(64, t // 2)


def _linear_params(op):
    D, ff = {"tower": (VIS["dim"], VIS["ff"])}.get(op, (TXT["dim"], TXT["ff"]))
    return 4 * D * D + 2 * D * ff


def work(c):
    op = c["op"]
    if op == "linear":
        m, n, k, wb = c["m"], c["n"], c["k"], 1 if c["w8a8"] else 2
        return dict(bytes=2 * m * k + wb * n * k + 2 * m * n * (2 if c["res"] else 1), flops=2.0 * m * n * k)
    if op == "sdpa":
        (h, d), b, t = _heads(c), c["b"], c["t"]
        p = _prefix(t) if c["form"] == "text" else t
        return dict(bytes=8 * b * h * t * d, flops=4.0 * b * h * d * (t * p + (t - p) * (t - p + 1) / 2))
    if op == "rglru":
        D = TRV["dim"]
        return dict(bytes=c["t"] * D * 12 + 4 * D * 64, flops=4.0 * c["t"] * D * 64)
    if op == "tower":
        m, D, L = c["b"] * VIS["ntok"], VIS["dim"], c["layers"]
        K = 3 * VIS["patch"] ** 2
        return dict(bytes=2 * (L * _linear_params(op) + K * D + VIS["ntok"] * D + m * D) + c["b"] * VIS["img"] ** 2 * 3,
                    flops=2.0 * m * (L * (_linear_params(op) + 2 * VIS["ntok"] * D) + K * D))
    if op == "track":
        D, T, L, n = TRV["dim"], TRV["n_img"] + TRV["n_q"], c["layers"], c["frames"]
        params = 7 * D * D + 3 * D * TRV["ff_gated"] + 2 * D * TRV["ff_vit"] + 2 * D * 64
        return dict(bytes=L * (2 * params + T * D * (8 + 2 * 4)) + n * (c["h"] * c["w"] * 3 + 2 * T * D),
                    flops=2.0 * n * T * L * (params + 2 * T * D))
    D, L, V = TXT["dim"], c["layers"], TXT["vocab"]
    params, wb = L * _linear_params(op), 1 if c["w8a8"] else 2
    P = 1 + c["n_img"]
    if op == "decode":
        keys = P + c["n_ids"] + 1
        return dict(bytes=wb * params + 2 * V * D + 4 * L * keys * D, flops=2.0 * (params + V * D + 2 * L * keys * D))
    if op == "query":
        rows = c["nq"] * c["l"]
        return dict(bytes=wb * params + 4 * L * c["nq"] * (P + c["l"]) * D,
                    flops=2.0 * rows * (params + 2 * L * (P + c["l"] / 2) * D))
    n, ids = P + c["n_ids"], c["n_ids"]
    return dict(bytes=wb * params + 2 * V * D + 4 * L * n * D + 4 * n * D,
                flops=2.0 * (n * params + V * D + 2 * L * D * (n * P + ids * (ids + 1) / 2)))


def tolerance(c):
    """About four times what the path differs by when its sums are taken in another order or split. Measured against
    torch's fp32 products rounded at the same places: a Linear 8e-5 (one in some hundred values takes the other bf16
    neighbour), attention 2.5e-3 (its probabilities in bf16 or not). Against the same model with that attention in
    every layer: 5e-3 .. 1e-2 over three or four bf16 layers, 1.4e-2 over the tower's 27, 1.7e-2 .. 2.2e-2 over four
    to six W8A8 layers, where a changed bit moves whole int8 steps of the next layer's input."""
    op = c["op"]
    if op == "linear":
        return dict(rel=1e-3, max=0.05)
    if op in ("sdpa", "rglru"):
        return dict(rel=5e-3, max=0.05)
    return dict(rel=0.03, max=0.5)


# ---- the same in 64 bits, plain torch


def _lin(w, name, x):
    return x @ w[name + ".weight"].to(F64).t() + w[name + ".bias"].to(F64)


def _ln(w, name, x, eps):
    return F.layer_norm(x, x.shape[-1:], w[name + ".weight"].to(F64), w[name + ".bias"].to(F64), eps)


def _tanh(x):
    return F.gelu(x, approximate="tanh")


def _attend(q, k, v, mask=None):
    """(B, H, T, D) in 64 bits, a few heads' scores at a time."""
    out = torch.empty_like(q)
    step = max(1, int(2e9 // (8 * q.shape[1] * q.shape[2] * k.shape[2])))
    for b in range(0, q.shape[0], step):
        e = b + step
        s = q[b:e].contiguous() @ k[b:e].transpose(2, 3).contiguous() * q.shape[3] ** -0.5
        if mask is not None:
            s = s.masked_fill(~mask, float("-inf"))
        out[b:e] = torch.softmax(s, -1) @ v[b:e].contiguous()
    return out


def _merge(a):
    return a.transpose(1, 2).reshape(a.shape[0], a.shape[2], -1)


def _quant(x, least):
    """Rows of x as int8 values and their scales."""
    s = x.abs().amax(-1, keepdim=True).clamp_min(least) / 127
    return torch.trunc(x / s + torch.where(x >= 0, 0.5, -0.5)), s


def _lin8(w, name, x):
    q, s = _quant(x, 1e-5)
    wq, ws = _quant(w[name + ".weight"].to(F64), 1e-8)
    return (q @ wq.t()) * s * ws[:, 0] + w[name + ".bias"].to(F64)


def _exact_tower(c, s):
    w, B, T, H = s["w"], c["b"], VIS["ntok"], VIS["heads"]
    P, G = VIS["patch"], VIS["grid"]
    x = (s["img"].permute(0, 3, 1, 2).to(F64) / 255 - 0.5) / 0.5
    x = x.reshape(B, 3, G, P, G, P).permute(0, 2, 4, 1, 3, 5).reshape(B, T, -1)
    x = _lin(w, "patch_emb", x) + w["pos_emb"].to(F64)
    for i in range(c["layers"]):
        p = f"blocks.{i}."
        qkv = _lin(w, p + "attn.qkv", _ln(w, p + "ln1", x, VIS["ln_eps"])).view(B, T, 3, H, -1).permute(2, 0, 3, 1, 4)
        x = x + _lin(w, p + "attn.proj", _merge(_attend(*qkv)))
        x = x + _lin(w, p + "mlp.fc2", _tanh(_lin(w, p + "mlp.fc1", _ln(w, p + "ln2", x, VIS["ln_eps"]))))
    return _ln(w, "post_ln", x, VIS["ln_eps"])


def _rope(x, cs):
    """Rotates the first 32 dims of each head: the two halves of 16 in, interleaved pairs out."""
    r = TXT["rot"]
    a, b, cos, sin = x[..., :r // 2], x[..., r // 2:r], cs[:, :, 0], cs[:, :, 1]
    return torch.cat([torch.stack((a * cos - b * sin, a * sin + b * cos), -1).flatten(-2), x[..., r:]], -1)


class _Text:
    def __init__(self, c, w):
        self.c, self.w, self.lin = c, w, _lin8 if c["w8a8"] else _lin
        self.cs = freqs_cis(TXT["rot"], 4096, TXT["theta"]).cuda().to(F64)
        self.k, self.v = [None] * c["layers"], [None] * c["layers"]

    def layers(self, x, prefix):
        """x (B, n, D) after the keys that are held; a key before `prefix` is seen by every row."""
        w, B, n, H = self.w, x.shape[0], x.shape[1], TXT["heads"]
        pos = 0 if self.k[0] is None else self.k[0].shape[2]
        at = torch.arange(pos + n, device="cuda")
        mask = (at[None] < prefix) | (at[None] <= pos + torch.arange(n, device="cuda")[:, None])
        for i in range(self.c["layers"]):
            p = f"blocks.{i}."
            h = _ln(w, p + "ln", x, TXT["ln_eps"])
            q, k, v = self.lin(w, p + "attn.qkv", h).view(B, n, 3, H, -1).permute(2, 0, 3, 1, 4)
            q, k = _rope(q, self.cs[pos:pos + n]), _rope(k, self.cs[pos:pos + n])
            if pos:
                k, v = (torch.cat([o.expand(B, -1, -1, -1), t], 2) for o, t in ((self.k[i], k), (self.v[i], v)))
            self.k[i], self.v[i] = k, v
            a = self.lin(w, p + "attn.proj", _merge(_attend(q, k, v, mask)))
            x = x + a + self.lin(w, p + "mlp.fc2", _tanh(self.lin(w, p + "mlp.fc1", h)))
        return x

    def embed(self, ids):
        return self.w["wte"][ids].to(F64)

    def logits(self, x, rows=slice(None)):
        h = _ln(self.w, "post_ln", x, TXT["ln_eps"])
        return h @ self.w["lm_head.weight"][rows].to(F64).t() + self.w["lm_head.bias"][rows].to(F64)


def _exact_text(c, s):
    t, P, none = _Text(c, s["w"]), 1 + c["n_img"], [None] * c["layers"]
    x = torch.cat([t.embed(torch.tensor([md2text.BOS], device="cuda")), s["img"].to(F64)])[None]
    if c["op"] == "query":
        t.layers(x, P)
        ids = s["ids"].clone()
        for b, n in enumerate(s["last"]):
            ids[b, n:] = 0
        x = t.layers(t.embed(ids), P)
        last = torch.stack([x[b, n - 1] for b, n in enumerate(s["last"])])
        return dict(logits=t.logits(last, list(YES + NO)), k=t.k, v=t.v)
    x = t.layers(torch.cat([x, t.embed(s["ids"])[None]], 1), P)
    if c["op"] == "prefill":
        return dict(hidden=x[0, P:], logits=t.logits(x[0, -1]), k=t.k, v=t.v)
    x = t.layers(t.embed(torch.tensor([[s["next"]]], device="cuda")), P)
    return dict(hidden=None, logits=t.logits(x[0, -1]), k=t.k, v=t.v)


def _gates(w, x):
    """Decay a and the gated input of the RG-LRU; x (..., 768)."""
    H = TRV["heads"]
    xh = x.reshape(-1, H, 64).transpose(0, 1).contiguous()

    def gate(n):
        g = xh @ w[n + "_w"].to(F64) + w[n + "_b"].to(F64)[:, None]
        return torch.sigmoid(g).transpose(0, 1).reshape(x.shape)

    log_a = -8 * gate("a_gate") * F.softplus(w["a_param"].to(F64))
    return log_a, x * gate("input_gate")


def _exact_track(c, s):
    w, n, T, H = s["w"], 2 * c["frames"], TRV["n_img"] + TRV["n_q"], TRV["heads"]
    x = s["frames"].permute(0, 3, 1, 2).to(F64)
    x = F.interpolate(x, size=(TRV["img"], TRV["img"]), mode="bilinear", align_corners=False) / 127.5 - 1
    P, G = TRV["patch"], TRV["img"] // TRV["patch"]
    x = x.reshape(n, 3, G, P, G, P).permute(0, 2, 4, 1, 3, 5).reshape(n, G * G, -1)
    x = x @ w["lin_proj.weight"].to(F64).flatten(1).t() + w["lin_proj.bias"].to(F64) + w["image_pos_emb"].to(F64)
    x = torch.cat([x, _lin(w, "query_proj", s["q"].to(F64)).expand(n, -1, -1)], 1)
    rms = lambda v, scale: v * torch.rsqrt((v * v).mean(-1, keepdim=True) + TRV["rms_eps"]) * (1 + w[scale].to(F64))
    hs = []
    for i in range(c["layers"]):
        sb, vb = f"blocks.{i}.ssm_block.", f"blocks.{i}.vit_block."
        rb = sb + "recurrent_block."
        y, xx = _lin(w, rb + "linear_yx", rms(x, sb + "temporal_pre_norm.scale")).chunk(2, -1)
        pad = torch.cat([torch.zeros_like(xx[:1]).expand(3, -1, -1), xx])
        xc = sum(pad[k:k + n] * w[rb + "conv_1d.w"][k].to(F64) for k in range(4)) + w[rb + "conv_1d.b"].to(F64)
        log_a, gated = _gates({g + v: w[rb + f"rg_lru.{g}.{v[1]}"] for g in ("input_gate", "a_gate") for v in ("_w", "_b")}
                              | {"a_param": w[rb + "rg_lru.a_param"]}, xc)
        h, states = gated[0], [gated[0]]
        for t in range(1, n):
            h = torch.exp(log_a[t]) * h + gated[t] * torch.sqrt(1 - torch.exp(2 * log_a[t]))
            states.append(h)
        hs.append(h)
        x = x + _lin(w, rb + "linear_out", torch.stack(states) * _tanh(y))
        g, u = _lin(w, sb + "mlp_block.ffw_up", rms(x, sb + "channel_pre_norm.scale")).chunk(2, -1)
        x = x + _lin(w, sb + "mlp_block.ffw_down", _tanh(g) * u)
        qkv = _ln(w, vb + "ln_1", x, TRV["ln_eps"]) @ w[vb + "self_attention.in_proj_weight"].to(F64).t()
        qkv = (qkv + w[vb + "self_attention.in_proj_bias"].to(F64)).view(n, T, 3, H, -1).permute(2, 0, 3, 1, 4)
        x = x + _lin(w, vb + "self_attention.out_proj", _merge(_attend(*qkv)))
        x = x + _lin(w, vb + "mlp.3", F.gelu(_lin(w, vb + "mlp.0", _ln(w, vb + "ln_2", x, TRV["ln_eps"]))))
    out = _ln(w, "encoder_norm", x, TRV["ln_eps"])
    if c["frames"] > 1:
        return dict(tokens=out[c["frames"]:], h=hs)

    def head(name):
        v = out[1, TRV["n_img"]:]
        for i in (0, 3):
            v = F.gelu(_ln(w, f"{name}.{i + 1}", _lin(w, f"{name}.{i}", v), TRV["head_ln_eps"]))
        return _lin(w, f"{name}.6", v)

    return dict(tokens=out[1], logits=head("coordinate_head"), vis=head("visible_head")[:, 0], h=hs)


def exact(c, seed):
    s, op = _inputs(c, seed), c["op"]
    if op == "linear":
        out = torch.empty(c["m"], c["n"], device="cuda", dtype=F64)
        act = dict(none=lambda v: v, tanh=_tanh, erf=F.gelu)[c["act"]]
        for m in range(0, c["m"], 16384):
            y = act((_lin8 if c["w8a8"] else _lin)(s, "lin", s["x"][m:m + 16384].to(F64)))
            out[m:m + 16384] = y if s["res"] is None else y + s["res"][m:m + 16384].to(F64)
        return out
    if op == "sdpa":
        t = c["t"]
        if c["form"] == "text":
            at = torch.arange(t, device="cuda")
            mask = (at[None] < _prefix(t)) | (at[None] <= at[:, None])
            return _merge(_attend(s["q"].to(F64), s["kc"][:, :, :t].to(F64), s["vc"][:, :, :t].to(F64), mask))
        return _merge(_attend(*s["qkv"].to(F64).permute(2, 0, 3, 1, 4)))
    if op == "rglru":
        log_a, gated = _gates(s["w"], s["x"].to(F64))
        h = torch.exp(log_a) * s["h0"].to(F64) + gated * torch.sqrt(1 - torch.exp(2 * log_a))
        return h, h
    return dict(tower=_exact_tower, track=_exact_track).get(op, _exact_text)(c, s)
