"""The work that programs built on this framework have it do, as cases that can be timed.

Four kinds of work:

  token   one decode step of a dense transformer on GGUF weights (cut_amd.decode.DecodeStep): from a token id to the
          logits and the next token id, KV cache included.  A serving loop captures the step into a HIP graph once and
          replays it per token; a program that experiments runs it launch by launch.
  rows    the norms, projections and feed-forward of a few layers for several activation rows: a decode batch (2 to 32
          sequences, replayed as a graph) or the rows of a prompt (up to 2048, launched as they come).  The attention
          over several rows is the caller's own, so its output is an input here.
  load    a model's tensors on their way in: GGUF blocks to fp16 / fp32 (dequantize), or to the separated [K, N] layout
          (prepare_sep).
  sep     matmuls on weights that are kept in the separated [K, N] layout, fp32 in and out.

Sizes are those of this repository's configurations, tests and benchmark (hidden 4096, 32 / 8 heads of 128, feed-forward
14336, vocabulary 128256; the two-layer model of the tests), or generic ones around them.
"""
import math

import torch

from cut_amd import lib, ops
from cut_amd.decode import DecodeConfig, DecodeStep

FORMATS = {"Q8_0": (32, 34), "Q4_0": (32, 18), "Q4_K": (256, 144), "Q6_K": (256, 210)}   # elements and bytes of a block
# formats of a model's tensors: attention projections, v projection, feed-forward, output head
MIXES = {"K": ("Q4_K", "Q6_K", "Q4_K", "Q6_K"), "Q6_K": ("Q6_K",) * 4, "Q8_0": ("Q8_0",) * 4, "Q4_0": ("Q4_0",) * 4}
DEVICE = "cuda:0"
EPS = 1e-5
MAX_BYTES, MAX_FLOPS = 4.5e9, 1.7e12   # a drawn case stays below the largest listed ones


def listed():
    full = dict(hidden=4096, heads=32, kv_heads=8, head_dim=128, ffn=14336)
    small = dict(hidden=2048, heads=32, kv_heads=8, head_dim=64, ffn=8192)
    return [
        # a chat turn on the 8B shape: the step of the benchmark, weights and a context of 2048 read once per token
        dict(full, name="token_ctx2k", kind="token", layers=32, vocab=128256, ctx=2048, pos=2047, mix="K", graph=True),
        # the same model deep inside a long document: the KV cache is a third of what a token reads
        dict(full, name="token_ctx16k", kind="token", layers=32, vocab=128256, ctx=16384, pos=15999, mix="K", graph=True),
        # a small assistant at 8 bits, heads of 64, in the middle of its context
        dict(small, name="token_small_q8", kind="token", layers=16, vocab=32000, ctx=1024, pos=700, mix="Q8_0", graph=True),
        # the tests' two-layer model stepped launch by launch: latency, and nothing else
        dict(name="token_tiny_eager", kind="token", hidden=512, heads=8, kv_heads=2, head_dim=64, ffn=1024, layers=2,
             vocab=2048, ctx=64, pos=40, mix="K", graph=False),
        # eight sequences decoded together
        dict(full, name="rows_8", kind="rows", layers=4, rows=8, mix="K", act="f16", graph=True),
        # a fuller decode batch on an 8-bit model
        dict(full, name="rows_24_q8", kind="rows", layers=4, rows=24, mix="Q8_0", act="f16", graph=True),
        # a short question as a prompt, of a length that fits no tile
        dict(full, name="rows_100", kind="rows", layers=4, rows=100, mix="K", act="f16", graph=False),
        # a page of text on a small 4-bit model whose host keeps fp32 activations
        dict(hidden=2048, heads=32, kv_heads=8, head_dim=64, ffn=5632, name="rows_300_f32", kind="rows", layers=8, rows=300,
             mix="Q4_0", act="f32", graph=False),
        # a long prompt, in the chunks of 2048 rows that the benchmark's prefill uses
        dict(full, name="rows_2048", kind="rows", layers=2, rows=2048, mix="K", act="f16", graph=False),
        # a loader that keeps fp16 weights: one feed-forward matrix of each format
        dict(name="load_f16", kind="load", to="f16", rows=14336, cols=4096, formats="Q8_0 Q4_0 Q4_K Q6_K"),
        # a loader that keeps the separated layout
        dict(name="load_sep", kind="load", to="sep", rows=14336, cols=4096, formats="Q8_0 Q4_0 Q4_K"),
        # one token through a layer's matrices on that layout
        dict(full, name="sep_1", kind="sep", rows=1, layout="q8"),
    ]


def _spread(rng, low, high, step=1):
    """A multiple of step between low and high, even over the logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high))) / step)) * step))


def _draw_one(rng):
    kind = rng.choices(("token", "rows", "load", "sep"), (3, 5, 2, 2))[0]
    if kind == "load":
        to = rng.choice(("f16", "f32", "sep"))
        formats = [f for f in FORMATS if to != "sep" or f != "Q6_K"]
        return dict(kind=kind, to=to, rows=2 * _spread(rng, 500, 16000), cols=_spread(rng, 512, 14336, 256),
                    formats=" ".join(rng.sample(formats, rng.randint(1, len(formats)))))
    head_dim = rng.choice((64, 128))
    heads = rng.choice([n for n in range(4, 65, 4) if 512 <= n * head_dim <= 5120])
    hidden = -(-heads * head_dim // 256) * 256
    heads = hidden // head_dim
    kv_heads = heads // rng.choice([r for r in (1, 2, 4, 8) if heads % r == 0])
    mix = rng.choice(list(MIXES))
    ffn = _spread(rng, 2 * hidden, min(4 * hidden, 14336), 256 if "K" in mix else 64)
    dims = dict(kind=kind, hidden=hidden, heads=heads, kv_heads=kv_heads, head_dim=head_dim, ffn=ffn)
    if kind == "token":
        ctx = _spread(rng, 64, 16384)
        return dict(dims, layers=_spread(rng, 2, 32), vocab=_spread(rng, 2000, 128256), ctx=ctx, pos=rng.randint(ctx // 2, ctx - 1),
                    mix=mix, graph=rng.random() < 0.75)
    if kind == "rows":
        rows = _spread(rng, 2, 2048)
        return dict(dims, layers=_spread(rng, 2, 8), rows=rows, mix=mix, act=rng.choice(("f16", "f16", "f32")),
                    graph=rows <= 32)
    return dict(dims, rows=_spread(rng, 1, 512), layout=rng.choice(("q8", "q4", "affine") if ffn % 256 == 0 else ("q8", "q4")))


def draw(rng):
    while True:
        case = _draw_one(rng)
        w = work(case)
        if w["bytes"] <= MAX_BYTES and w["flops"] <= MAX_FLOPS:
            return case


# ---- weights: GGUF blocks of Gaussian matrices, encoded on the GPU ----------------------------------------------------
def _half_bytes(v):
    return v.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _pack_8bit(x):
    d = (x.abs().amax(-1) / 127).half()
    q = (x / d.float().clamp_min(1e-8).unsqueeze(-1)).round_().clamp_(-127, 127).to(torch.int8)
    return torch.cat((_half_bytes(d), q.view(torch.uint8)), -1)


def _pack_4bit(x):
    d = (x.abs().amax(-1) / 8).half()
    q = (x / d.float().clamp_min(1e-8).unsqueeze(-1)).round_().add_(8).clamp_(0, 15).to(torch.uint8)
    return torch.cat((_half_bytes(d), q[..., :16] | q[..., 16:] << 4), -1)


def _pack_q4_k(x):
    s = x.view(*x.shape[:-1], 8, 32)
    low = (-s.amin(-1)).clamp_min_(0)
    step = (s.amax(-1) + low) / 15
    d, dmin = (step.amax(-1) / 63).half(), (low.amax(-1) / 63).half()
    df, mf = d.float().clamp_min(1e-8).unsqueeze(-1), dmin.float().clamp_min(1e-8).unsqueeze(-1)
    sc, mn = (step / df).round_().clamp_(1, 63), (low / mf).round_().clamp_(0, 63)
    q = ((s + (mf * mn).unsqueeze(-1)) / (df * sc).unsqueeze(-1)).round_().clamp_(0, 15).to(torch.uint8)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    packed = torch.cat((sc[..., :4] | (sc[..., 4:] >> 4) << 6, mn[..., :4] | (mn[..., 4:] >> 4) << 6,
                        (sc[..., 4:] & 15) | (mn[..., 4:] & 15) << 4), -1)
    return torch.cat((_half_bytes(d), _half_bytes(dmin), packed, (q[..., 0::2, :] | q[..., 1::2, :] << 4).flatten(-2)), -1)


def _pack_q6_k(x):
    s = x.view(*x.shape[:-1], 16, 16)
    step = s.abs().amax(-1) / 31
    d = (step.amax(-1) / 127).half()
    df = d.float().clamp_min(1e-8).unsqueeze(-1)
    sc = (step / df).round_().clamp_(1, 127)
    q = (s / (df * sc).unsqueeze(-1)).round_().add_(32).clamp_(0, 63).to(torch.uint8).view(*x.shape[:-1], 2, 4, 32)
    ql = torch.cat((q[..., 0, :] & 15 | (q[..., 2, :] & 15) << 4, q[..., 1, :] & 15 | (q[..., 3, :] & 15) << 4), -1)
    qh = q[..., 0, :] >> 4 | q[..., 1, :] >> 4 << 2 | q[..., 2, :] >> 4 << 4 | q[..., 3, :] >> 4 << 6
    return torch.cat((ql.flatten(-2), qh.flatten(-2), sc.to(torch.uint8), _half_bytes(d)), -1)


_PACK = {"Q8_0": _pack_8bit, "Q4_0": _pack_4bit, "Q4_K": _pack_q4_k, "Q6_K": _pack_q6_k}


def _blocks(gen, fmt, n, k, spread=0.0):
    """n rows of k Gaussian weights that keep the scale of what they multiply; spread: log-normal factor of a row."""
    out = []
    for n0 in range(0, n, 16384):   # a few hundred MB of fp32 at a time
        w = torch.randn((min(16384, n - n0), k), generator=gen, device=DEVICE).mul_(k ** -0.5)
        if spread:
            w *= torch.exp(spread * torch.randn((w.shape[0], 1), generator=gen, device=DEVICE))
        out.append(_PACK[fmt](w.view(-1, FORMATS[fmt][0])).flatten())
    return torch.cat(out) if len(out) > 1 else out[0]


def _norm_weight(gen, n):
    return 0.5 + torch.rand(n, generator=gen, device=DEVICE)


# ---- the kinds ----------------------------------------------------------------------------------------------------------
def _layer_shapes(case):
    """name -> (format, rows, columns) of a layer's matrices."""
    attn, v, ffn, _ = MIXES[case["mix"]]
    h, q, kv, f = case["hidden"], case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["ffn"]
    return {"qk": (attn, q + kv, h), "v": (v, kv, h), "o": (attn, h, q), "gate_up": (ffn, 2 * f, h), "down": (ffn, h, f)}


def _layer(gen, case):
    L = {k: _blocks(gen, *s) for k, s in _layer_shapes(case).items()}
    L["attn_norm"], L["ffn_norm"] = _norm_weight(gen, case["hidden"]), _norm_weight(gen, case["hidden"])
    return L


def _captured(fn):
    fn()   # once outside the capture, as the first pass of any program is
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


def _prepare_token(case, gen):
    attn, v, ffn, head = MIXES[case["mix"]]
    h, kv = case["hidden"], case["kv_heads"] * case["head_dim"]
    cfg = DecodeConfig(hidden=h, n_layers=case["layers"], n_heads=case["heads"], n_kv_heads=case["kv_heads"], head_dim=case["head_dim"],
                       ffn=case["ffn"], vocab=case["vocab"], max_ctx=case["ctx"], eps=EPS, fmt_attn=attn, fmt_v=v, fmt_ffn=ffn,
                       fmt_head=head, fmt_embd=attn)
    step = DecodeStep(cfg, [_layer(gen, case) for _ in range(cfg.n_layers)], _norm_weight(gen, h),
                      _blocks(gen, head, cfg.vocab, h, spread=1.0), DEVICE, embedding=_blocks(gen, attn, cfg.vocab, h))
    # the context so far: both caches in one piece, a layer's in each slice of it
    keys = torch.randn((cfg.n_layers, cfg.max_ctx, kv), generator=gen, device=DEVICE).half()
    values = torch.randn((cfg.n_layers, cfg.max_ctx, kv), generator=gen, device=DEVICE).half()
    step.k_cache, step.v_cache = list(keys.unbind(0)), list(values.unbind(0))
    step.set_position(case["pos"])
    token = torch.randint(cfg.vocab, (1,), generator=gen, device=DEVICE, dtype=torch.int32)
    step.token.copy_(token)
    return dict(step=step, token=token, keys=keys, values=values, graph=_captured(step.step) if case["graph"] else None)


def _run_token(s):
    step = s["step"]
    step.token.copy_(s["token"])
    if s["graph"] is not None:
        s["graph"].replay()
    else:
        step.step()
    return {"logits": step.logits, "token": step.token, "keys": s["keys"], "values": s["values"]}


def _prepare_rows(case, gen):
    M, h, f = case["rows"], case["hidden"], case["ffn"]
    q, kv = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    act = torch.float16 if case["act"] == "f16" else torch.float32
    layers = [_layer(gen, case) for _ in range(case["layers"])]
    shapes = _layer_shapes(case)
    pairs = M <= 8   # gate and up rows interleaved for the SwiGLU epilogue, as far as it goes
    if pairs:
        from cut_amd.decode import interleave_gate_up
        for L in layers:
            L["gate_up"] = interleave_gate_up(L["gate_up"], f)
    ws = max((ops.matmul_gguf_workspace(fmt, M, k, n // 2 if name == "gate_up" and not pairs else n, act, DEVICE)
              for name, (fmt, n, k) in shapes.items()), key=lambda t: t.numel())

    def buf(*shape, dtype=act):
        return torch.empty(shape, dtype=dtype, device=DEVICE)
    s = dict(case=case, layers=layers, shapes=shapes, pairs=pairs, ws=ws, xn=buf(M, h), gate_up=buf(2, M, f), hidden=buf(M, f),
             x=buf(M, h, dtype=torch.float32), qk=[buf(M, q + kv) for _ in layers], v=[buf(M, kv) for _ in layers],
             x_in=torch.randn((M, h), generator=gen, device=DEVICE),
             attn=[torch.randn((M, q), generator=gen, device=DEVICE).to(act) for _ in layers])
    s["graph"] = _captured(lambda: _layers_of_rows(s)) if case["graph"] else None
    return s


def _layers_of_rows(s):
    x, xn, ws, f = s["x_in"], s["xn"], s["ws"], s["case"]["ffn"]
    for i, L in enumerate(s["layers"]):
        def mm(a, name, out, w=None, n=None, **more):
            fmt, rows, k = s["shapes"][name]
            ops.matmul_gguf(a, L[name] if w is None else w, fmt, n or rows, k, out=out, workspace=ws, **more)
        ops.rmsnorm(x, L["attn_norm"], EPS, out=xn)
        mm(xn, "qk", s["qk"][i])
        mm(xn, "v", s["v"][i])
        mm(s["attn"][i], "o", s["x"], binary="add", d=x)
        x = s["x"]
        ops.rmsnorm(x, L["ffn_norm"], EPS, out=xn)
        if s["pairs"]:
            mm(xn, "gate_up", s["hidden"], swiglu_pairs=True)
        else:
            gate, up = L["gate_up"].view(2, -1)
            mm(xn, "gate_up", s["gate_up"][0], gate, f)
            mm(xn, "gate_up", s["gate_up"][1], up, f)
            ops.silu_mul(s["gate_up"], s["hidden"])
        mm(s["hidden"], "down", x, binary="add", d=x)


def _run_rows(s):
    if s["graph"] is not None:
        s["graph"].replay()
    else:
        _layers_of_rows(s)
    return {"x": s["x"], "qk": s["qk"], "v": s["v"]}


def _prepare_load(case, gen):
    return dict(case=case, tensors=[(f, _blocks(gen, f, case["rows"], case["cols"])) for f in case["formats"].split()])


def _run_load(s):
    n, k, to = s["case"]["rows"], s["case"]["cols"], s["case"]["to"]
    if to == "sep":
        return [ops.prepare_sep(w, f, n, k) for f, w in s["tensors"]]
    return [ops.dequantize(w, f, n, k, torch.float16 if to == "f16" else torch.float32) for f, w in s["tensors"]]


def _sep_shapes(case):
    h, q, kv, f = case["hidden"], case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["ffn"]
    return [(q, h), (kv, h), (kv, h), (h, q), (f, h), (f, h), (h, f)]


def _prepare_sep(case, gen):
    fmt = {"q8": "Q8_0", "q4": "Q4_0", "affine": "Q4_K"}[case["layout"]]
    mats = []
    for n, k in _sep_shapes(case):
        b, scales = ops.prepare_sep(_blocks(gen, fmt, n, k), fmt, n, k)
        mats.append((torch.randn((case["rows"], k), generator=gen, device=DEVICE), b, scales, n))
    return dict(mats=mats, q4=case["layout"] != "q8", affine=case["layout"] == "affine")


def _run_sep(s):
    return [ops.matmul_sep(a, b, scales, n, q4=s["q4"], affine=s["affine"]) for a, b, scales, n in s["mats"]]


_KINDS = {"token": (_prepare_token, _run_token), "rows": (_prepare_rows, _run_rows), "load": (_prepare_load, _run_load),
          "sep": (_prepare_sep, _run_sep)}


def prepare(case, seed):
    lib.check(lib.load().cuthip_init(0))
    gen = torch.Generator(DEVICE).manual_seed(seed)
    return _KINDS[case["kind"]][0](case, gen), case["kind"]


def run(state):
    return _KINDS[state[1]][1](state[0])


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------
def _weight_bytes(fmt, n, k):
    return n * k / FORMATS[fmt][0] * FORMATS[fmt][1]


def work(case):
    kind = case["kind"]
    if kind == "load":
        n, k = case["rows"], case["cols"]
        out = {"f16": dict.fromkeys(FORMATS, 2.0), "f32": dict.fromkeys(FORMATS, 4.0),
               "sep": {"Q8_0": 1 + 2 / 32, "Q4_0": 0.5 + 2 / 32, "Q4_K": 0.5 + 4 / 32}}[case["to"]]
        return {"bytes": sum(_weight_bytes(f, n, k) + out[f] * n * k for f in case["formats"].split()), "flops": 0}
    if kind == "sep":
        M, per = case["rows"], {"q8": 1 + 2 / 32, "q4": 0.5 + 2 / 32, "affine": 0.5 + 4 / 32}[case["layout"]]
        return {"bytes": sum(per * n * k + 4.0 * M * (n + k) for n, k in _sep_shapes(case)),
                "flops": sum(2.0 * M * n * k for n, k in _sep_shapes(case))}
    shapes, L, h = _layer_shapes(case).values(), case["layers"], case["hidden"]
    weights = L * (sum(_weight_bytes(*s) for s in shapes) + 8.0 * h)
    macs = L * sum(float(n) * k for _, n, k in shapes)
    q, kv = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    if kind == "token":
        head, length = MIXES[case["mix"]][3], case["pos"] + 1
        macs += float(case["vocab"]) * h + L * 2.0 * length * q
        return {"bytes": weights + _weight_bytes(head, case["vocab"], h) + 4.0 * case["vocab"] + L * 2 * length * kv * 2.0, "flops": 2 * macs}
    M, a = case["rows"], 2.0 if case["act"] == "f16" else 4.0
    return {"bytes": weights + M * (8.0 * h + L * a * (2 * q + 2 * kv)), "flops": 2.0 * M * macs}


def tolerance(case):
    """About four times what was measured, seeded cases against another order of the same arithmetic (tokens: the step
    with every operator a launch of its own) or against fp64 products between the same roundings (rows, sep)."""
    if case["kind"] == "load":
        return "exact"
    if case["kind"] == "token":   # fp16 activations through the depth of the model: 0.0010, 0.0025, 0.0041 at 2, 16, 32 layers
        rel = 0.003 * math.sqrt(case["layers"])
        return {"rel": rel, "max": 20 * rel}   # (of logits of rows of very different norms: 0.08 for one at 32 layers)
    if case["kind"] == "rows":    # fp16 products and intermediates, one value up to 0.0028 off
        return {"rel": 0.0025, "max": 0.012}
    if case["rows"] < 32:         # fp32 throughout
        return {"rel": 2e-6, "max": 1e-5}
    return {"rel": 0.0012, "max": 0.006}   # weights and activations rounded to fp16 once
