"""The work this library is used for, as timed cases: the MoE layer at decode and prompt sizes, and its router.

A case is one layer shape, a weight format, a routing and a token count, run through xsmoe's public calls: MoeLayer
(decode or prefill form), router_logits_f32 and router_top10.  Shapes are the layer shapes of bench.py and the tests:

  shape    hidden  experts  top-k  expert width
  small      1024        8      2           512
  qwen30     2048      128      8           768
  qwen235    4096      128      8          1536
  dsv3       7168      256      8          2048    group-limited sigmoid routing, one shared Q8_0 expert

Weights are N(0, 0.02) quantized here, in plain torch, to the GGUF blocks; exact() reads the same blocks back in 64 bits.
"""
import math
import pathlib
import sys

import numpy as np
import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "xestrata-win_amd"))
import xsmoe  # noqa: E402

DEV = "cuda"
Q8_0, Q4_K, Q6_K, IQ4_XS = 8, 12, 14, 23
BLOCK = {Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210), IQ4_XS: (256, 136)}   # values, bytes
FORMATS = {"q8_0": (Q8_0, Q8_0), "q4_k+q6_k": (Q4_K, Q6_K), "q4_k": (Q4_K, Q4_K), "iq4_xs": (IQ4_XS, IQ4_XS)}
SHAPES = {   # hidden, experts, top-k, expert width
    "small": (1024, 8, 2, 512),
    "qwen30": (2048, 128, 8, 768),
    "qwen235": (4096, 128, 8, 1536),
    "dsv3": (7168, 256, 8, 2048),
}
GROUPS, TOP_GROUPS, ROUTED_SCALE = 8, 4, 2.5   # the dsv3 router
DRAWN = 16   # experts drawn of a layer; the others repeat them with their gate and up rows rotated


# ---------------------------------------------------------------------------------------------------- the cases

def _case(name, do, shape, fmt, tokens, layers=1, routing="uniform", shared="none", project=False):
    """do: decode, prefill or router.  layers: so many layers in a row, each with its own weights, x and routing, the
    residual carried through.  routing: uniform or zipf (softmax), or sigmoid.  shared: none, plain or gated.  project:
    the call starts with the router's projection of x (else the logits are given)."""
    return dict(name=name, do=do, shape=shape, format=fmt, tokens=tokens, layers=layers, routing=routing, shared=shared,
                project=project)


def listed():
    return [
        # the smallest call: one layer of a small model, a few tokens; launch latency is most of it
        _case("decode_small_4", "decode", "small", "q8_0", 4),
        # generating one sequence: the MoE sections of 16 layers, from x to the residual, the weights out of HBM
        _case("step_qwen30_1", "decode", "qwen30", "q4_k+q6_k", 1, layers=16, project=True),
        # checking a few draft tokens, routed unevenly as trained routers do
        _case("verify_qwen30_5", "decode", "qwen30", "q4_k+q6_k", 5, layers=4, routing="zipf"),
        # a small batch of sequences
        _case("decode_qwen30_16", "decode", "qwen30", "q4_k+q6_k", 16),
        # a serving batch: nearly every expert is read, each for a few tokens; a shared expert with its gate
        _case("decode_qwen30_64", "decode", "qwen30", "q4_k", 64, shared="gated"),
        # a wide layer in 4-bit codebook weights
        _case("decode_qwen235_8", "decode", "qwen235", "iq4_xs", 8),
        # the widest layer, one token, the sigmoid router and the shared expert in the call
        _case("decode_dsv3_1", "decode", "dsv3", "q4_k", 1, routing="sigmoid", shared="plain"),
        # a prompt chunk, from x to the residual
        _case("prompt_qwen30_2048", "prefill", "qwen30", "q4_k+q6_k", 2048, routing="zipf", project=True),
        # a short prompt of odd length, every expert read for a few rows
        _case("prompt_qwen235_333", "prefill", "qwen235", "iq4_xs", 333),
        # a prompt through a small 8-bit layer with a gated shared expert
        _case("prompt_small_700", "prefill", "small", "q8_0", 700, shared="gated"),
        # the largest: a prompt chunk of the widest layer
        _case("prompt_dsv3_1024", "prefill", "dsv3", "q4_k", 1024, routing="sigmoid", shared="plain"),
        # the router alone at prompt size, for callers that place the experts themselves
        _case("router_qwen30_2048", "router", "qwen30", "none", 2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(("decode", "decode", "prefill", "prefill", "router"))
    if do == "router":
        shape = rng.choice(("qwen30", "qwen235", "dsv3"))
        return _drop(_case("", do, shape, "none", _log_int(rng, 1, 4096)))
    shape = rng.choice(("small", "qwen30", "qwen30", "qwen235", "dsv3"))
    if shape == "dsv3":
        fmt, routing, shared = "q4_k", "sigmoid", "plain"
        tokens = _log_int(rng, 1, 6) if do == "decode" else _log_int(rng, 65, 1000)
    else:
        fmt = "q8_0" if shape == "small" else rng.choice(("q4_k+q6_k", "q4_k+q6_k", "q4_k", "iq4_xs", "q8_0"))
        routing = rng.choice(("uniform", "zipf"))
        shared = rng.choice(("none", "none", "plain", "gated"))
        most = {"small": 4000, "qwen30": 4000, "qwen235": 1000}[shape]
        tokens = _log_int(rng, 1, 64 if shape != "qwen235" else 24) if do == "decode" else _log_int(rng, 65, most)
    layers = rng.choice((1, 1, 3)) if do == "decode" and shape in ("small", "qwen30") else 1
    return _drop(_case("", do, shape, fmt, tokens, layers, routing, shared, rng.random() < 0.3))


def _drop(case):
    del case["name"]
    return case


# ---------------------------------------------------------------------------------------------------- GGUF blocks

_IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _half(v):
    """[n] fp32 -> (its fp16 bytes [n, 2], the fp16 value as fp32)."""
    h = v.to(torch.float16)
    return h.view(torch.uint8).view(-1, 2), h.float()


def _pack(t, w):
    """w [rows, cols] fp32 -> `t` blocks [rows, row bytes]."""
    rows, cols = w.shape
    qk, nb = BLOCK[t]
    w = w.reshape(-1, qk)
    n = w.shape[0]
    out = torch.empty(n, nb, dtype=torch.uint8, device=w.device)
    if t == Q8_0:
        b, d = _half(w.abs().amax(1) / 127)
        q = (w / d.clamp_min(1e-10)[:, None]).round().clamp(-127, 127).to(torch.int8)
        out[:, 0:2] = b
        out[:, 2:] = q.view(torch.uint8)
    elif t == Q4_K:
        s = w.view(n, 8, 32)
        low = s.amin(2).clamp_max(0)
        scale = (s.amax(2) - low).clamp_min(1e-10) / 15
        bd, d = _half(scale.amax(1) / 63)
        bm, dmin = _half((-low).amax(1) / 63)
        sc = (scale / d.clamp_min(1e-10)[:, None]).round().clamp(1, 63)
        mn = (-low / dmin.clamp_min(1e-10)[:, None]).round().clamp(0, 63)
        q = ((s + (dmin[:, None] * mn)[:, :, None]) / (d[:, None] * sc).clamp_min(1e-10)[:, :, None]).round()
        q = q.clamp(0, 15).to(torch.uint8)
        sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
        out[:, 0:2], out[:, 2:4] = bd, bm
        out[:, 4:8] = sc[:, :4] | (sc[:, 4:] >> 4) << 6
        out[:, 8:12] = mn[:, :4] | (mn[:, 4:] >> 4) << 6
        out[:, 12:16] = (sc[:, 4:] & 15) | (mn[:, 4:] & 15) << 4
        out[:, 16:] = (q[:, 0::2] | q[:, 1::2] << 4).reshape(n, 128)
    elif t == Q6_K:
        s = w.view(n, 16, 16)
        scale = s.abs().amax(2).clamp_min(1e-10) / 31
        b, d = _half(scale.amax(1) / 127)
        sc = (scale / d.clamp_min(1e-10)[:, None]).round().clamp(1, 127)
        q = ((s / (d[:, None] * sc).clamp_min(1e-10)[:, :, None]).round().clamp(-32, 31) + 32).to(torch.uint8)
        q = q.view(n, 2, 4, 32)
        out[:, 0:128] = torch.stack((q[:, :, 0] & 15 | (q[:, :, 2] & 15) << 4, q[:, :, 1] & 15 | (q[:, :, 3] & 15) << 4),
                                    2).reshape(n, 128)
        h = q >> 4
        out[:, 128:192] = (h[:, :, 0] | h[:, :, 1] << 2 | h[:, :, 2] << 4 | h[:, :, 3] << 6).reshape(n, 64)
        out[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
        out[:, 208:210] = b
    else:
        s = w.view(n, 8, 32)
        scale = s.abs().amax(2).clamp_min(1e-10) / 120
        b, d = _half(scale.amax(1) / 31)
        ls = (scale / d.clamp_min(1e-10)[:, None]).round().clamp(1, 31)
        levels = torch.tensor(_IQ4, dtype=torch.float32, device=w.device)
        q = torch.bucketize(s / (d[:, None] * ls).clamp_min(1e-10)[:, :, None], (levels[1:] + levels[:-1]) / 2)
        q, ls = q.to(torch.uint8), ls.to(torch.int32) + 32
        high = ((ls >> 4) << torch.arange(0, 16, 2, device=w.device)).sum(1).to(torch.int32)
        out[:, 0:2] = b
        out[:, 2], out[:, 3] = (high & 255).to(torch.uint8), (high >> 8).to(torch.uint8)
        out[:, 4:8] = (ls[:, 0::2] & 15 | (ls[:, 1::2] & 15) << 4).to(torch.uint8)
        out[:, 8:] = (q[:, :, :16] | q[:, :, 16:] << 4).reshape(n, 128)
    return out.view(rows, cols // qk * nb)


def _unpack(t, b):
    """`t` blocks [rows, row bytes] -> the weights [rows, cols] in 64 bits."""
    rows, row = b.shape
    qk, nb = BLOCK[t]
    b = b.contiguous().view(-1, nb)
    n = b.shape[0]
    half = lambda i: b[:, i:i + 2].contiguous().view(torch.float16).double()   # noqa: E731  [n, 1]
    if t == Q8_0:
        v = b[:, 2:].contiguous().view(torch.int8).double() * half(0)
    elif t == Q4_K:
        a, m, c = b[:, 4:8], b[:, 8:12], b[:, 12:16]
        sc = torch.cat((a & 63, c & 15 | (a >> 6) << 4), 1).double() * half(0)
        mn = torch.cat((m & 63, c >> 4 | (m >> 6) << 4), 1).double() * half(2)
        q = b[:, 16:].view(n, 4, 32)
        q = torch.stack((q & 15, q >> 4), 2).view(n, 8, 32).double()
        v = q * sc[:, :, None] - mn[:, :, None]
    elif t == Q6_K:
        ql, qh = b[:, 0:128].view(n, 2, 2, 32), b[:, 128:192].view(n, 2, 32)
        q = torch.stack((ql[:, :, 0] & 15 | (qh & 3) << 4, ql[:, :, 1] & 15 | (qh >> 2 & 3) << 4,
                         ql[:, :, 0] >> 4 | (qh >> 4 & 3) << 4, ql[:, :, 1] >> 4 | (qh >> 6) << 4), 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * half(208)
        v = (q.view(n, 16, 16).double() - 32) * sc[:, :, None]
    else:
        high = b[:, 2].int() | b[:, 3].int() << 8
        low = torch.stack((b[:, 4:8] & 15, b[:, 4:8] >> 4), 2).view(n, 8).int()
        ls = low | (high[:, None] >> torch.arange(0, 16, 2, device=b.device) & 3) << 4
        q = b[:, 8:].view(n, 8, 16)
        q = torch.cat((q & 15, q >> 4), 2).long()
        levels = torch.tensor(_IQ4, dtype=torch.float64, device=b.device)
        v = levels[q] * ((ls - 32).double() * half(0))[:, :, None]
    return v.reshape(rows, row // nb * qk)


# ---------------------------------------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _experts(g, n, H, F, gu, dn):
    """n experts' (gate, up, down) blocks."""
    draw_rows = lambda rows, cols, t: _pack(t, _normal(g, rows, cols) * 0.02)   # noqa: E731
    return [(draw_rows(F, H, gu), draw_rows(F, H, gu), draw_rows(H, F, dn)) for _ in range(n)]


def _shift(e, layer):
    """How far expert e's gate and up rows are rotated from those of the drawn expert it repeats."""
    return e // DRAWN + 3 * layer


def _arena(drawn, E, layer):
    """E experts' blobs (gate rows, up rows, down rows) back to back."""
    gate, up, down = drawn[0]
    a, b = gate.numel(), gate.numel() + up.numel()
    arena = torch.empty(E, b + down.numel(), dtype=torch.uint8, device=DEV)
    for e in range(E):
        gate, up, down = drawn[e % len(drawn)]
        s = _shift(e, layer)
        arena[e, :a] = torch.roll(gate, s, 0).view(-1)
        arena[e, a:b] = torch.roll(up, s, 0).view(-1)
        arena[e, b:] = down.view(-1)
    return arena


def _inputs(case, seed):
    """What prepare() and exact() both start from: per layer x, router weights and logits, the residual, the bias, the
    drawn experts, the shared expert and its gate's weights."""
    H, E, k, F = SHAPES[case["shape"]]
    T, n = case["tokens"], case["layers"]
    g = _gen(seed)
    v = dict(x=_normal(g, n, T, H).bfloat16().float(), residual=_normal(g, T, H) * 0.1, router=None, logits=None, bias=None,
             drawn=None, shared=None, w_gate=None)
    popularity = torch.zeros(n, E, device=DEV)
    if case["routing"] == "zipf":   # an expert's share falls as rank ** -1.2, the ranks in another order in each layer
        rank = torch.stack([torch.randperm(E, generator=g, device=DEV) for _ in range(n)]) + 1
        popularity = -1.2 * rank.float().log()
    if case["project"] or case["do"] == "router":
        # the hidden states share a direction u, by which the router tells an expert's popularity
        u = _normal(g, n, 1, H).sign() * 0.5
        v["x"] = (v["x"] + u).bfloat16().float()
        v["router"] = _normal(g, n, E, H) * 0.02 + popularity[:, :, None] * u / (0.25 * H)
    else:
        gumbel = -torch.rand(n, T, E, generator=g, device=DEV).clamp(1e-7, 1 - 1e-7).log().neg().log()
        v["logits"] = popularity[:, None] + gumbel if case["routing"] != "sigmoid" else _normal(g, n, T, E)
    if case["routing"] == "sigmoid":
        v["bias"] = _normal(g, n, E) * 0.1
    if case["do"] != "router":
        gu, dn = FORMATS[case["format"]]
        v["drawn"] = _experts(g, min(DRAWN, E), H, F, gu, dn)
        if case["shared"] != "none":
            v["shared"] = _experts(g, 1, H, F, Q8_0, Q8_0)[0]
        if case["shared"] == "gated":
            v["w_gate"] = _normal(g, H) * 0.02
    return v


class State:
    pass


def prepare(case, seed):
    H, E, k, F = SHAPES[case["shape"]]
    T, n = case["tokens"], case["layers"]
    v = _inputs(case, seed)
    s = State()
    s.k, s.x, s.router, s.logits, s.residual, s.layers = k, v["x"], v["router"], v["logits"], v["residual"], []
    if case["do"] == "router":
        return s
    gu, dn = FORMATS[case["format"]]
    L = xsmoe.native_expert_layout(gu, dn, H, F)
    s.out = torch.empty(n, T, H, device=DEV)
    for i in range(n):
        shared = router = None
        if v["shared"] is not None:
            blob = torch.cat([part.reshape(-1) for part in v["shared"]])
            shared = (xsmoe.native_expert_layout(Q8_0, Q8_0, H, F), blob, v["w_gate"])
        if v["bias"] is not None:
            router = xsmoe.grouped_sigmoid_router(v["bias"][i], GROUPS, TOP_GROUPS, ROUTED_SCALE)
        s.layers.append(xsmoe.MoeLayer(L, _arena(v["drawn"], E, i), E, k, T, prefill=case["do"] == "prefill",
                                       shared=shared, router=router))
    return s


def run(s):
    if not s.layers:
        logits = xsmoe.router_logits_f32(s.x[0], s.router[0])
        ids, weights = xsmoe.router_top10(logits, s.k)
        return dict(logits=logits, ids=ids, weights=weights)
    residual, projected = s.residual, []
    for i, layer in enumerate(s.layers):
        if s.router is not None:
            logits = xsmoe.router_logits_f32(s.x[i], s.router[i])
            projected.append(logits)
        else:
            logits = s.logits[i]
        residual = layer(s.x[i], logits, residual, s.out[i])
    return dict(out=residual, logits=projected)


# ---------------------------------------------------------------------------------------------------- accounting

def _rows_read(case):
    """The number of distinct experts that a layer's tokens reach, expected."""
    _, E, k, _ = SHAPES[case["shape"]]
    r = np.random.default_rng(0)
    popularity = -1.2 * np.log(np.arange(1, E + 1)) if case["routing"] == "zipf" else np.zeros(E)
    z = popularity + r.gumbel(size=(8, min(case["tokens"], 512), E))
    top = np.argpartition(-z, k - 1, axis=2)[:, :, :k]
    return float(np.mean([len(np.unique(t)) for t in top]))


def work(case):
    H, E, k, F = SHAPES[case["shape"]]
    T, n = case["tokens"], case["layers"]
    nbytes = flops = 0.0
    if case["project"] or case["do"] == "router":
        nbytes += 4 * (E * H + T * H + T * E)
        flops += 2.0 * T * E * H
    if case["do"] == "router":
        return dict(bytes=nbytes + 8.0 * T * k, flops=flops)
    gu, dn = FORMATS[case["format"]]
    row = lambda t, cols: cols // BLOCK[t][0] * BLOCK[t][1]   # noqa: E731
    nbytes += _rows_read(case) * (2 * F * row(gu, H) + H * row(dn, F)) + 4 * (3 * T * H + T * E)
    flops += 6.0 * T * k * H * F
    if case["shared"] != "none":
        nbytes += 2 * F * row(Q8_0, H) + H * row(Q8_0, F)
        flops += 6.0 * T * H * F
    return dict(bytes=n * nbytes, flops=n * flops)


def tolerance(case):
    # Four times what was measured over these ranges.  router: fp32 sums of `hidden` products, 8e-7 off the 64-bit ones.
    # decode: x and h in 8 bits, so that a change of x in its last bits moves the result by 3e-3 (largest value 2e-2).
    # prefill: x, the weights and h in f16 with fp32 sums, 1.1e-3 off the 64-bit result (largest value 7e-3).
    if case["do"] == "router":
        return dict(rel=5e-6, differ=1e-4)
    return dict(rel=1.2e-2, max=9e-2) if case["do"] == "decode" else dict(rel=4e-3, max=3e-2)


# ---------------------------------------------------------------------------------------------------- in 64 bits

def _route(case, logits, bias):
    """logits [T, E] in 64 bits -> (expert ids [T, k], weights [T, k]), the largest first."""
    _, E, k, _ = SHAPES[case["shape"]]
    if case["routing"] != "sigmoid":
        w, ids = logits.softmax(1).topk(k, 1)
        return ids, w / w.sum(1, keepdim=True)
    score = logits.sigmoid()
    pick = score + bias.double()
    best = pick.view(-1, GROUPS, E // GROUPS).topk(2, 2)[0].sum(2).topk(TOP_GROUPS, 1)[1]
    open_ = torch.zeros(len(pick), GROUPS, dtype=torch.bool, device=DEV).scatter_(1, best, True)
    pick = pick.masked_fill(~open_.repeat_interleave(E // GROUPS, 1), -math.inf)
    ids = pick.topk(k, 1)[1]
    w = score.gather(1, ids)
    return ids, w / w.sum(1, keepdim=True) * ROUTED_SCALE


def exact(case, seed):
    v = _inputs(case, seed)
    logits = [x.double() @ w.double().T for x, w in zip(v["x"], v["router"])] if v["router"] is not None else \
        [z.double() for z in v["logits"]]
    if case["do"] == "router":
        return dict(logits=logits[0], ids=None, weights=_route(case, logits[0], None)[1])
    gu, dn = FORMATS[case["format"]]
    out, silu = v["residual"].double(), torch.nn.functional.silu
    for i in range(case["layers"]):
        x = v["x"][i].double()
        ids, weights = _route(case, logits[i], v["bias"][i] if v["bias"] is not None else None)
        moe = torch.zeros_like(out)
        for b, (gate, up, down) in enumerate(v["drawn"]):
            used = [int(e) for e in torch.unique(ids[ids % len(v["drawn"]) == b])]
            if not used:
                continue
            gate, up, down = _unpack(gu, gate), _unpack(gu, up), _unpack(dn, down)
            for e in used:
                t, j = (ids == e).nonzero(as_tuple=True)
                h = silu(x[t] @ gate.T) * (x[t] @ up.T)
                moe[t] += weights[t, j, None] * (torch.roll(h, _shift(e, i), 1) @ down.T)
        if v["shared"] is not None:
            gate, up, down = (_unpack(Q8_0, part) for part in v["shared"])
            y = (silu(x @ gate.T) * (x @ up.T)) @ down.T
            moe += y * (x @ v["w_gate"].double()).sigmoid()[:, None] if v["w_gate"] is not None else y
        out = out + moe
    return dict(out=out, logits=logits if v["router"] is not None else [])
