"""The calls whose time matters to a program built on stratametal_amd, over the range it makes them in.

A case is one call of a public operator of the package on one layer (or, for the stack, a few layers):

  moe       MoELayer.forward            the quantised mixture-of-experts block on a batch of tokens
  junction  MoELayer.forward_residual   the block with the residual junction before it, as a stack of layers calls it
  ffn       FfnLayer.run                the whole layer call: hyper-connection read, block, write back
  verify    VerifyWindow.begin / end    a window of draft tokens with part of the experts held, the rest evaluated from
                                        a second table (expert_group, expert_grouped)
  stack     forward_residual per layer  a token's way through several layers, each with its own weights

`prepare` makes a layer's weights and inputs on the GPU from the seed, `run` makes the call, `exact` restates the
call's arithmetic contract in 64 bits: activations of the decode contract are q8_1 blocks, those of the prefill contract
bf16, weights are the stored blocks' values (IQ2_S with its integer sub-block sum), all sums are float64.
"""
import math
import os

import numpy as np
import torch

import stratametal_amd as S

Q2_0, IQ2_S = S.Q2_0, S.IQ2_S
PREFILL = 128  # Q2_0 layers take the prefill contract from this many tokens on
EPS = 1e-6

# The layer of the package's benchmark.
BASE = dict(n_embd=2048, n_ff=512, n_ff_shared=512, n_expert=512, top_k=10, w_type=Q2_0, sh_type=Q2_0, router_dtype=0,
            sh_gate_type=0, sh_up_type=0, sh_down_type=0)
GEOM_KEYS = tuple(BASE)


def _case(name, op, tokens, geom=None, **kw):
    c = dict(name=name, op=op, tokens=tokens, zipf=False, hc=4, hc_lr=320, layers=1)
    c.update(BASE)
    c.update(geom or {})
    c.update(kw)
    return c


def listed():
    iq2 = dict(w_type=IQ2_S, sh_type=IQ2_S)
    wide = dict(n_embd=2560, n_ff=640, n_ff_shared=640)  # the width whose rows are five units of 128
    # a shared expert stored in its own types, as real layers have it: Q3_K gate and up, IQ4_NL down
    native = dict(sh_type=S.Q3_K, sh_down_type=S.IQ4_NL)
    return [
        # one sequence generating: the smallest call, latency and launches
        _case("decode_1", "moe", 1),
        # a small serving batch
        _case("decode_16", "moe", 16),
        # a larger, odd serving batch on the wider layer with the f32 router
        _case("decode_77_wide", "moe", 77, dict(wide, router_dtype=S.ROUTER_F32)),
        # an ordinary prompt, expert popularity Zipf(1.2)
        _case("prefill_512_zipf", "moe", 512, zipf=True),
        # a short odd prompt on a layer of other sizes: many experts, no shared expert, f32 router
        _case("prefill_301_f32_router", "moe", 301, dict(n_embd=1024, n_ff=1024, n_expert=1024, top_k=8, sh_type=-1,
                                                         router_dtype=S.ROUTER_F32)),
        # one layer of a long prompt's way through a stack
        _case("junction_4096", "junction", 4096),
        # a serving batch on IQ2_S experts
        _case("iq2s_64", "moe", 64, iq2),
        # a prompt on IQ2_S experts
        _case("iq2s_600", "moe", 600, iq2),
        # the whole layer call while generating
        _case("ffn_1", "ffn", 1, native),
        # the whole layer call on a prompt
        _case("ffn_1000", "ffn", 1000, native),
        # a speculative window of four tokens, three quarters of the experts held
        _case("verify_4", "verify", 4),
        # a token through eight layers
        _case("stack_8_layers", "stack", 1, layers=8),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    q2 = [dict(), dict(n_embd=2560, n_ff=640, n_ff_shared=640), dict(n_embd=1024, n_ff=1024, n_expert=1024, top_k=8, sh_type=-1),
          dict(n_embd=1536, n_ff=768, n_ff_shared=768, n_expert=128, top_k=8), dict(n_expert=600)]
    iq2 = [dict(w_type=IQ2_S, sh_type=IQ2_S), dict(w_type=IQ2_S, sh_type=IQ2_S, n_embd=1024, n_expert=128, top_k=6),
           dict(w_type=IQ2_S, sh_type=-1, n_expert=256, top_k=8)]
    ends = [dict(), dict(sh_type=S.Q3_K, sh_down_type=S.IQ4_NL), dict(sh_type=S.Q8_0), dict(sh_type=S.Q4_0),
            dict(n_embd=2560, n_ff=640, n_ff_shared=640, sh_type=S.Q3_K, sh_down_type=S.IQ4_NL)]
    op = rng.choice(["decode", "prefill", "junction", "iq2", "ffn", "ffn", "verify", "stack"])
    f32 = rng.random() < 0.25
    router = dict(router_dtype=S.ROUTER_F32) if f32 else {}
    if op == "decode":
        c = _case("", "moe", _log_int(rng, 1, PREFILL - 1), dict(rng.choice(q2), **router))
    elif op == "prefill":
        c = _case("", "moe", _log_int(rng, PREFILL, 2048), dict(rng.choice(q2), **router), zipf=rng.random() < 0.5)
    elif op == "junction":
        c = _case("", "junction", _log_int(rng, 1, 3000), dict(rng.choice(q2), **router))
    elif op == "iq2":
        c = _case("", "moe", _log_int(rng, 1, 600), dict(rng.choice(iq2), **router))
    elif op == "ffn":
        c = _case("", "ffn", _log_int(rng, 1, 900), rng.choice(ends), hc=rng.choice([2, 4, 4]),
                  hc_lr=rng.choice([64, 200, 320, 320]))
    elif op == "verify":
        c = _case("", "verify", _log_int(rng, 1, 16), rng.choice(q2 + iq2))
    else:
        c = _case("", "stack", _log_int(rng, 1, 16), rng.choice(q2), layers=rng.randint(2, 8))
    if c["zipf"] and c["sh_type"] < 0:
        c["zipf"] = False
    del c["name"]
    return c


def _geom(case):
    return S.Geom(**{k: case[k] for k in GEOM_KEYS})


# ------------------------------------------------------------------------------------------------ inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFFFFFF)


def _native_blocks(gen, wtype, n_values, sigma=0.02):
    """Random blocks of a native type: uniform codes, small positive fp16 scales."""
    qk, nb = S.NATIVE_BLOCKS[wtype]
    field, div = {S.Q8_0: (0, 64.0), S.Q4_0: (0, 4.0), S.IQ4_NL: (0, 64.0), S.Q3_K: (108, 32.0)}[wtype]
    n = n_values // qk
    b = torch.randint(0, 256, (n, nb), dtype=torch.uint8, device="cuda", generator=gen)
    d = torch.randn(n, device="cuda", generator=gen).abs_().mul_(sigma / div).half()
    b[:, field:field + 2] = d.view(torch.uint8).view(n, 2)
    return b.reshape(-1)


def _bf16(gen, n, sigma):
    return torch.randn(n, device="cuda", generator=gen).mul_(sigma).bfloat16().view(torch.int16)


def _layer(case, seed, gen):
    g = _geom(case)
    bias = None
    if case["zipf"]:
        b = S.zipf_bias(g.n_expert, 1.2, 1, n_tokens=512, top_k=g.top_k, n_embd=g.n_embd, sims=1024, iters=12)
        bias = torch.from_numpy(b).cuda()
    types = g.shared_types()
    if g.sh_type < 0 or all(t in (Q2_0, IQ2_S) for t in types):
        return g, S.synth_layer(g, seed, logit_bias=bias)
    plain = S.Geom(**dict(vars(g), sh_type=-1, sh_gate_type=0, sh_up_type=0, sh_down_type=0))
    w = S.synth_layer(plain, seed, logit_bias=bias)
    H, F = g.n_embd, g.n_ff_shared
    w.update(gate_sh=_native_blocks(gen, types[0], F * H), up_sh=_native_blocks(gen, types[1], F * H),
             down_sh=_native_blocks(gen, types[2], H * F), gate_inp_sh=_bf16(gen, H, 0.02))
    return g, w


def prepare(case, seed):
    gen = _generator(seed)
    T, H = case["tokens"], case["n_embd"]
    st = dict(op=case["op"], seed=seed)
    seeds = [(int(seed) * 64 + l) & 0x7FFFFFFF for l in range(case["layers"])]
    layers = [_layer(case, s, gen) for s in seeds]
    g, w = st["g"], st["w"] = layers[0]
    st["x"] = torch.randn((T, H), device="cuda", generator=gen)
    if case["op"] == "ffn":
        hc, lr, hd = case["hc"], case["hc_lr"], case["hc"] * H
        norm = torch.randn(hd, device="cuda", generator=gen).mul_(0.1).add_(1.0)
        st["ends"] = S.HyperConnection(H, hc, lr, norm, _bf16(gen, lr * hd, 0.2), _bf16(gen, hd * lr, 0.2),
                                       _bf16(gen, hc * hd, 0.05), eps=EPS)
        scale = 3.0 ** torch.arange(hc, device="cuda", dtype=torch.float32)
        st["x"] = torch.randn((T, hc, H), device="cuda", generator=gen) * scale[None, :, None]
        st["layer"] = S.FfnLayer(g, w, st["ends"], T)
    elif case["op"] == "verify":
        E = g.n_expert
        blobs = torch.cat([w[n].view(E, -1) for n in ("gate_exps", "up_exps", "down_exps")], dim=1)
        at = torch.arange(E, device="cuda") * blobs.shape[1] + blobs.data_ptr()
        held = torch.arange(E, device="cuda") % 4 != 0
        st["blobs"] = blobs
        st["held"], st["rest"] = torch.where(held, at, 0), torch.where(held, 0, at)
        st["layer"] = S.VerifyWindow(g, w, T)
    else:
        if case["op"] == "junction":
            st["r"] = torch.randn((T, H), device="cuda", generator=gen)
        st["layer"] = [S.MoELayer(lg, lw, T) for lg, lw in layers]
    return st


def run(st):
    op, x = st["op"], st["x"]
    if op == "moe":
        return st["layer"][0].forward(x)
    if op == "junction":
        xn = torch.empty_like(x)
        y = st["layer"][0].forward_residual(x, st["r"], xn, eps=EPS)
        return xn, y
    if op == "ffn":
        return st["layer"].run(x)
    if op == "verify":
        g, win = st["g"], st["layer"]
        r = win.begin(x, st["held"])
        # the experts the first table does not hold, as a second tier on the same GPU evaluates them
        groups = S.expert_group(r["ids"], g.top_k, g.n_expert, st["rest"])
        S.expert_grouped(g, groups, S.quantize_q8_1(x), x.shape[0], r["rows"])
        return win.end(r)
    cur, nxt = x.clone(), torch.empty_like(x)
    y = st["layer"][0].forward(cur)
    for layer in st["layer"][1:]:
        layer.forward_residual(cur, y, nxt, y, eps=EPS)
        cur, nxt = nxt, cur
    return S.residual_rmsnorm(cur, y, EPS, out=nxt)


# ------------------------------------------------------------------------------------------------ work

def work(case):
    """Compulsory traffic (every touched expert's blocks once, the router, x in, y out) and products."""
    g = _geom(case)
    T, H, F, E, k = case["tokens"], g.n_embd, g.n_ff, g.n_expert, g.top_k
    touched = E * (1.0 - (1.0 - k / E) ** T)  # distinct experts of T uniform tokens
    if case["zipf"]:
        touched = min(touched, float((S.zipf_targets(E, 1.2, T, k) >= 0.5).sum()))
    bytes_ = touched * g.expert_bytes() + g.shared_bytes() + E * H * (4 if g.router_dtype else 2) + 2 * T * H * 4
    flops = 2.0 * T * H * E + 6.0 * T * k * H * F + (6.0 * T * H * g.n_ff_shared if g.sh_type >= 0 else 0.0)
    if case["op"] == "junction":
        bytes_ += 2 * T * H * 4
    if case["op"] == "ffn":
        hd = case["hc"] * H
        bytes_ += 2 * hd * case["hc_lr"] * 2 + case["hc"] * hd * 2 + 2 * T * hd * 4 - 2 * T * H * 4
        flops += 2.0 * T * hd * (2 * case["hc_lr"] + case["hc"])
    n = case["layers"]
    return {"bytes": int(bytes_ * n), "flops": int(flops * n)}


def tolerance(case):
    # The sums are 32-bit.  What separates two correct evaluations is a rounding of an intermediate activation (q8_1
    # steps or bf16, of h and of the next layer's x) that falls to the other side where its 32-bit sum differs in the
    # last bits: one step in 127, or 2^-8 of the value, in a few of the row's values.  Against `exact`, measured over
    # listed and drawn cases, such steps amount to at most 4.3e-4 (decode: few tokens, so one step shows), 3.2e-5
    # (prefill) and 7.8e-5 (ffn, where the residual streams carry most of the norm); a stack repeats them per layer.
    return {"rel": TOLERANCE[_kind(case)]}


TOLERANCE = {"decode": 1.5e-3, "prefill": 1.5e-4, "ffn": 3e-4, "stack": 5e-3}


def _kind(case):
    if case["op"] in ("ffn", "stack"):
        return case["op"]
    return "prefill" if case["w_type"] == Q2_0 and case["tokens"] >= PREFILL and case["op"] != "verify" else "decode"


# ------------------------------------------------------------------------------------------------ 64-bit restatement

def _f16(blocks, at):
    return blocks[:, at:at + 2].contiguous().view(torch.float16).double()


_NL = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _values(wtype, data, rows, n):
    """The rows' weights in float64 (every type but IQ2_S)."""
    if wtype == Q2_0:
        b = data.view(-1, 18)
        q = torch.stack([(b[:, 2:] >> (2 * i)) & 3 for i in range(4)], dim=2).view(-1, 64)
        return (_f16(b, 0) * (q.double() - 1.0)).view(rows, n)
    qk, nb = S.NATIVE_BLOCKS[wtype]
    b = data.view(-1, nb)
    if wtype == S.Q8_0:
        return (_f16(b, 0) * b[:, 2:].contiguous().view(torch.int8).double()).view(rows, n)
    if wtype in (S.Q4_0, S.IQ4_NL):
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], dim=1)
        v = q.double() - 8.0 if wtype == S.Q4_0 else torch.tensor(_NL, device=b.device).double()[q.long()]
        return (_f16(b, 0) * v).view(rows, n)
    assert wtype == S.Q3_K
    hm, qs, sc8 = b[:, :32], b[:, 32:96], b[:, 96:108]
    sc = torch.stack([((sc8[:, i % 8] >> (4 * (i // 8))) & 15) | (((sc8[:, 8 + i % 4] >> (2 * (i // 4))) & 3) << 4)
                      for i in range(16)], dim=1).double() - 32.0
    parts = []
    for grp in range(8):
        low = (qs[:, 32 * (grp // 4):32 * (grp // 4) + 32] >> (2 * (grp % 4))) & 3
        parts.append(low.double() - 4.0 * (1 - ((hm >> grp) & 1)).double())
    v = torch.stack(parts, dim=1).view(-1, 16, 16) * sc[:, :, None]
    return (_f16(b, 108) * v.view(-1, 256)).view(rows, n)


_GRID = None


def _grid():
    """The IQ2_S format's 1024 magnitude groups, from the checker's copy of the table."""
    global _GRID
    if _GRID is None:
        root = os.path.dirname(os.path.dirname(os.path.abspath(S.__file__)))
        text = open(os.path.join(root, "oracle", "iq2s_grid_codes.inc")).read().split("*/")[-1]
        codes = np.array([int(t, 0) for t in text.replace(",", " ").split()], dtype=np.int64)
        mags = np.array([8, 25, 43, 0])[(codes[:, None] >> (2 * np.arange(8))) & 3]
        _GRID = torch.from_numpy(mags.astype(np.float64)).cuda()
    return _GRID


def _iq2(data):
    """Per block: signed magnitudes (blocks, 8 sub-blocks, 2 halves, 16), half scales (blocks, 8, 2), block scale."""
    b = data.view(-1, 82)
    shift = 2 * torch.arange(4, device=b.device)
    hi = (b[:, 66:74, None].int() >> shift) & 3
    idx = b[:, 2:34].view(-1, 8, 4).int() | (hi << 8)
    sign = 1.0 - 2.0 * ((b[:, 34:66].view(-1, 8, 4, 1).int() >> torch.arange(8, device=b.device)) & 1).double()
    v = _grid()[idx.long()] * sign
    ls = torch.stack([b[:, 74:82] & 15, b[:, 74:82] >> 4], dim=2).double()
    return v.view(-1, 8, 2, 16), ls, _f16(b, 0)


def _q8(x):
    """q8_1 of float64 rows: integer values and the fp16 scale of each 32."""
    v = x.view(x.shape[0], -1, 32)
    d = v.abs().amax(dim=2) / 127.0
    r = v / torch.where(d > 0, d, torch.ones_like(d))[:, :, None]
    return torch.sign(r) * torch.floor(r.abs() + 0.5), d.half().double()


def _product(wtype, data, rows, n, x, contract):
    """x (c, n) times the rows, as the contract rounds x: float64 (c, rows)."""
    if contract == "bf16":
        return x.bfloat16().double() @ _values(wtype, data, rows, n).T
    q, d = _q8(x)
    if wtype != IQ2_S:
        return (q * d[:, :, None]).view(x.shape) @ _values(wtype, data, rows, n).T
    v, ls, dw = _iq2(data)
    subs, c = n // 32, x.shape[0]
    w2 = v.view(rows, subs * 2, 16).permute(1, 2, 0).contiguous()
    s = torch.bmm(q.view(c, subs * 2, 16).permute(1, 0, 2).contiguous(), w2).view(subs, 2, c, rows)
    ls = ls.view(rows, subs, 2).permute(1, 2, 0)
    i = torch.trunc((s[:, 0] * ls[:, 0, None] + s[:, 1] * ls[:, 1, None] + torch.trunc((s[:, 0] + s[:, 1]) / 2)) / 4)
    i = i.view(n // 256, 8, c, rows) * d.T.reshape(n // 256, 8, c, 1)
    return (i.sum(dim=1) * dw.view(rows, -1).T[:, None, :]).sum(dim=0)


def _expert(types, data, H, F, x, contract):
    gate, up = (_product(types[i], data[i], F, H, x, contract) for i in (0, 1))
    return _product(types[2], data[2], H, F, gate / (1.0 + torch.exp(-gate)) * up, contract)


def _block(g, w, x, prefill):
    """The block's y of float64 x."""
    T, H, F, E = x.shape[0], g.n_embd, g.n_ff, g.n_expert
    contract = "bf16" if prefill and g.w_type == Q2_0 else "q8_1"
    xb = x.bfloat16().double()
    if g.router_dtype == S.ROUTER_F32:
        logits = x @ w["router"].view(E, H).double().T
    else:
        logits = xb @ w["router"].view(torch.bfloat16).view(E, H).double().T
    if w.get("logit_bias") is not None:
        logits = logits + w["logit_bias"].double()
    top, ids = torch.topk(torch.softmax(logits, dim=1), g.top_k, dim=1)
    wts = top / top.sum(dim=1, keepdim=True).clamp_min(2.0 ** -14)
    y = torch.zeros((T, H), dtype=torch.float64, device=x.device)
    planes = [w[n].view(E, -1) for n in ("gate_exps", "up_exps", "down_exps")]
    step = 64 if g.w_type == IQ2_S else 1 << 30  # (the IQ2_S sums hold every sub-block: few columns at a time)
    order = torch.argsort(ids.view(-1), stable=True)
    counts = torch.bincount(ids.view(-1), minlength=E).tolist()
    at = 0
    for e in range(E):
        mine = order[at:at + counts[e]]
        at += counts[e]
        for pairs in mine.split(step) if counts[e] else ():
            tok = pairs // g.top_k
            out = _expert((g.w_type,) * 3, [p[e] for p in planes], H, F, x[tok], contract)
            y.index_add_(0, tok, out * wts.view(-1)[pairs][:, None])
    if g.sh_type >= 0:
        types = g.shared_types()
        if any(t != g.w_type for t in types):
            contract = "q8_1"  # a shared expert in its own types is always on q8_1 activations
        data = [w[n] for n in ("gate_sh", "up_sh", "down_sh")]
        gate = torch.sigmoid(xb @ w["gate_inp_sh"].view(torch.bfloat16).double())
        for tok in torch.arange(T, device=x.device).split(step):
            y[tok] += _expert(types, data, H, g.n_ff_shared, x[tok], contract) * gate[tok, None]
    return y


def _norm(v):
    return v / torch.sqrt((v * v).mean(dim=-1, keepdim=True) + EPS)


def exact(case, seed):
    if case["op"] == "stack":
        return None  # each layer's roundings decide the next layer's: no 64-bit value to hold it to
    st = prepare(case, seed)
    g, w, x = st["g"], st["w"], st["x"].double()
    prefill = case["tokens"] >= PREFILL
    if case["op"] == "junction":
        xn = _norm(x + st["r"].double())
        return xn, _block(g, w, xn, prefill)
    if case["op"] != "ffn":
        return _block(g, w, x, prefill and case["op"] == "moe")
    hc, lr, H = case["hc"], case["hc_lr"], g.n_embd
    norm, down, up, inj = st["ends"].tensors
    down, up, inj = (t.view(torch.bfloat16).double() for t in (down, up, inj))
    xn = _norm(x) * norm.view(hc, H).double()
    act = xn.view(-1, hc * H).bfloat16().double()
    z = act @ down.view(lr, hc * H).T / hc
    lq = (z / (1.0 + torch.exp(-z))).bfloat16().double()
    gate = torch.sigmoid(lq @ up.view(hc * H, lr).T).view(-1, hc, H)
    y = _block(g, w, (xn * gate).sum(dim=1) / hc, prefill)
    inject = act @ inj.view(hc, hc * H).T
    return x + y[:, None, :] * (2.0 * torch.sigmoid(inject / hc))[:, :, None]
