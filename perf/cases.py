"""The calls that a user of this library makes, as cases that can be timed and checked.

The user is an inference engine of one sequence at a time: a context of up to 8192 positions
(it_validate_geometry), prompts in calls of 64, 128, 256 or 512 tokens (it_prefill_chunks) or in one
call, then one token at a time, or a few with an MTP draft (verify). Its model mixes Gated-DeltaNet
layers and softmax attention layers, here in the two head geometries that the tests and the benchmark
use: 16 query / 2 KV heads with 32 value / 16 key heads in the recurrence, and 24 / 4 with 48 / 16.
One pass of a case is the calls of `layers` such layers, each with its own weights, cache and state.

ops of a case:
  attn         pre-pass (norm, rope, f16 append) and attention of `nt` tokens after `pos0` cached ones, in
               calls of at most `ubatch` tokens (0: one call); `q16`: the pre-pass also hands over the
               query in f16
  mtp          the MTP head's pre-pass and attention over its own f32 cache
  gdn_decode   two consecutive steps of `nt` tokens (the conv state alternates between two buffers) and
               the gated norm; `ckpt`: with the verify checkpoint, and the second step rolled back
  gdn_prefill  the recurrent layer over `nt` prompt tokens, and the gated norm
`graph`: the pass is captured once and replayed, as a layer loop whose launches are short is run; the
others are called each time.
"""
from __future__ import annotations

import math

import torch

from irontimber_amd import ops
from irontimber_amd._lib import lib

HD, S, KC = 256, 128, 4            # head_dim, recurrent state size, conv taps
EPS = 1e-6
N_ROT, SECTIONS, BASE = 64, (11, 11, 10, 0), 1e7
CTX = 8192


def _attn(name, nt, pos0, nh=16, nkv=2, ubatch=0, q16=False, layers=1, graph=False, op="attn"):
    return dict(name=name, op=op, nt=nt, pos0=pos0, nh=nh, nkv=nkv, ubatch=ubatch, q16=q16, layers=layers, graph=graph)


def _gdn(name, op, nt, nv=32, nk=16, layers=1, graph=False, ckpt=False):
    return dict(name=name, op=op, nt=nt, nv=nv, nk=nk, layers=layers, graph=graph, ckpt=ckpt)


def listed():
    return [
        # the smallest call: one token of a short chat, one layer, called directly: latency and launches
        _attn("decode_512_direct", 1, 511),
        # a token of a long conversation through the attention layers of a model: the KV cache's bytes
        _attn("decode_8191", 1, 8191, layers=8, graph=True),
        # checking an MTP draft of three tokens, the larger geometry, an odd context
        _attn("verify4_2997_24h", 4, 2997, nh=24, nkv=4, layers=8, graph=True),
        # a long prompt in the engine's smallest calls: 128 dependent calls whose context grows
        _attn("prompt_8192_by_64", 8192, 0, ubatch=64, q16=True, graph=True),
        # a long question appended to a conversation, in the engine's largest calls with a ragged end
        _attn("prompt_3001_at_5000_by_512", 3001, 5000, ubatch=512, q16=True),
        # a middle-sized prompt in one call, the query handed over in f32
        _attn("prompt_1531", 1531, 0),
        # the longest prompt in one call: the largest amount of matrix work
        _attn("prompt_8192", 8192, 0, q16=True),
        # a token through the recurrent layers of a model: the states' bytes and the launches
        _gdn("gdn_decode", "gdn_decode", 1, layers=24, graph=True),
        # a draft of one token checked by the recurrent layers, then rejected
        _gdn("gdn_verify2_48v", "gdn_decode", 2, nv=48, layers=24, graph=True, ckpt=True),
        # one of the engine's largest prompt calls through a few recurrent layers, a ragged length
        _gdn("gdn_prompt_500_48v", "gdn_prefill", 500, nv=48, layers=3),
        # the longest prompt through a recurrent layer
        _gdn("gdn_prompt_8192", "gdn_prefill", 8192),
        # the MTP head catching up on 64 prompt tokens over its f32 cache
        _attn("mtp_64_at_4096", 64, 4096, op="mtp"),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["decode", "prompt", "prompt", "mtp", "gdn_decode", "gdn_prefill", "gdn_prefill"])
    if kind.startswith("gdn"):
        nv = rng.choice([32, 48])
        if kind == "gdn_decode":
            nt = rng.randint(1, 4)
            c = _gdn("", kind, nt, nv=nv, layers=rng.randint(8, 24), graph=True, ckpt=nt > 1 and rng.random() < 0.5)
        else:
            c = _gdn("", kind, _log(rng, 16, CTX), nv=nv, layers=rng.randint(1, 3))
    else:
        nh, nkv = rng.choice([(16, 2), (24, 4)])
        if kind == "decode":
            nt = rng.choice([1, 1, 2, 3, 4])
            c = _attn("", nt, _log(rng, 16, CTX - nt), nh, nkv, layers=rng.randint(2, 8), graph=True)
        elif kind == "mtp":
            nt = rng.choice([1, 2, rng.randint(3, 64)])
            c = _attn("", nt, _log(rng, 16, CTX - nt), nh, nkv, layers=1 if nt > 2 else 4, graph=nt <= 2, op="mtp")
        else:
            nt = _log(rng, 16, CTX if nh == 16 else CTX // 2)
            pos0 = rng.choice([0, _log(rng, 16, max(16, CTX - nt))])
            ubatch = rng.choice([0, 64, 128, 256, 512])
            c = _attn("", nt, min(pos0, CTX - nt), nh, nkv, ubatch=ubatch, q16=rng.random() < 0.5, graph=ubatch == 64)
    c.pop("name")
    return c


# ---- inputs: those of a model's projections, normal values; K unit-RMS per head as a norm leaves it

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _attn_inputs(c, g):
    n = lambda *s: torch.randn(*s, device="cuda", generator=g)
    nt, pos0, nh, kvd = c["nt"], c["pos0"], c["nh"], c["nkv"] * HD
    rows = pos0 + nt
    k = n(rows, c["nkv"], HD)
    k = (k * torch.rsqrt(k.square().mean(-1, keepdim=True) + EPS)).reshape(rows, kvd)
    v = n(rows, kvd)
    kind = torch.float32 if c["op"] == "mtp" else torch.float16
    return dict(kc=k.to(kind), vc=v.to(kind), q=2 * n(nt, nh * 2 * HD), k=2 * n(nt, kvd), v=n(nt, kvd),
                qn=1 + 0.1 * n(HD), kn=1 + 0.1 * n(HD))


def _gdn_inputs(c, g, steps):
    n = lambda *s: torch.randn(*s, device="cuda", generator=g)
    nt, nv, nk = c["nt"], c["nv"], c["nk"]
    cd = (2 * nk + nv) * S
    return dict(state=0.02 * n(nv, S, S), w=0.5 * n(cd, KC), conv=n(KC - 1, cd),
                x=[n(nt, cd) for _ in range(steps)], beta=[n(nt, nv) for _ in range(steps)],
                alpha=[n(nt, nv) for _ in range(steps)], z=[n(nt, nv * S) for _ in range(steps)],
                a=-torch.exp(2 * torch.rand(nv, device="cuda", generator=g) - 1), dt=torch.zeros(nv, device="cuda"),
                nw=1 + 0.1 * n(S))


def _steps(c):
    return 2 if c["op"] == "gdn_decode" else 1


def _inputs(c, seed):
    g = _gen(seed)
    make = (lambda: _gdn_inputs(c, g, _steps(c))) if c["op"].startswith("gdn") else (lambda: _attn_inputs(c, g))
    return [make() for _ in range(c["layers"])]


def _calls(c):
    """(first token, tokens) of the calls that a prompt is processed in."""
    if not c.get("ubatch"):
        return [(0, c["nt"])]
    import ctypes
    cap = c["nt"] // 64 + 2
    starts, lens = (ctypes.c_size_t * cap)(), (ctypes.c_size_t * cap)()
    n = lib().it_prefill_chunks(c["nt"], c["ubatch"], ctypes.addressof(starts), ctypes.addressof(lens), cap)
    return [(starts[i], lens[i]) for i in range(n)]


def prepare(case, seed):
    c = dict(case)
    layers = _inputs(c, seed)
    calls = _calls(c)
    st = dict(case=c, layers=layers, calls=calls, graph=None)
    nt = c["nt"]
    # outputs and scratch as an engine's arena holds them: scratch is shared by the layers
    if c["op"].startswith("gdn"):
        # the layers' states as slices of one buffer each
        for name in ("state", "conv"):
            st[name] = torch.stack([d[name] for d in layers])
        st["out"] = torch.empty(len(layers), _steps(c), nt, c["nv"] * S, device="cuda")
        for i, d in enumerate(layers):
            d["out"], d["state"], d["conv"] = st["out"][i], st["state"][i], st["conv"][i]
            d["conv2"] = torch.empty_like(d["conv"])
            if c["ckpt"]:
                d["ck_state"], d["ck_conv"] = torch.empty_like(d["state"]), torch.empty_like(d["conv"])
        need = lib().it_gdn_prefill_scratch_bytes(nt, c["nv"], c["nk"], S) if c["op"] == "gdn_prefill" else 0
    else:
        for d in layers:
            d["out"] = torch.empty(nt, c["nh"] * HD, device="cuda")
        if c["op"] == "mtp":
            need = lib().it_attn_f32kv_scratch_bytes(c["pos0"], nt, HD, c["nh"], c["nkv"])
        else:
            need = max(ops.attn_scratch_bytes(c["pos0"] + t0, n, c["nh"], c["nkv"]) for t0, n in calls)
    st["scratch"] = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    if c["graph"]:
        moved = ("q", "kc", "vc", "state", "conv")
        kept = [{k: d[k].clone() for k in moved if k in d} for d in layers]
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            _pass(st)                      # loads the kernels: not possible under capture
        torch.cuda.current_stream().wait_stream(s)
        for d, k in zip(layers, kept):
            for name, t in k.items():
                d[name].copy_(t)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"], stream=s):
            _pass(st)
        torch.cuda.synchronize()
    return st


def _pass(st):
    c, scratch = st["case"], st["scratch"]
    if c["op"] == "gdn_decode":
        for i in range(2):
            for d in st["layers"]:
                src, dst = (d["conv"], d["conv2"]) if i == 0 else (d["conv2"], d["conv"])
                ck = dict(ckpt_state=d["ck_state"], ckpt_conv=d["ck_conv"]) if c["ckpt"] else {}
                o = ops.gdn_decode_fused(d["x"][i], d["w"], src, dst, d["beta"][i], d["alpha"][i], d["dt"], d["a"],
                                         d["state"], c["nv"], c["nk"], EPS, out=d["out"][i], **ck)
                ops.gdn_gated_rmsnorm(o, d["z"][i], d["nw"], c["nv"], EPS, out=o)
        if c["ckpt"]:
            for d in st["layers"]:
                ops.gdn_rollback(d["ck_conv"], d["conv"], d["ck_state"], d["state"])
    elif c["op"] == "gdn_prefill":
        for d in st["layers"]:
            o = ops.gdn_prefill(d["x"][0], d["w"], d["conv"], d["beta"][0], d["alpha"][0], d["dt"], d["a"], d["state"],
                                c["nv"], c["nk"], EPS, out=d["out"][0], scratch=scratch)
            ops.gdn_gated_rmsnorm(o, d["z"][0], d["nw"], c["nv"], EPS, out=o)
    elif c["op"] == "mtp":
        # slot p of the head's cache holds position p + 1
        for d in st["layers"]:
            ops.attn_prep_f32kv(d["q"], d["k"], d["v"], d["kc"], d["vc"], c["pos0"] + 1, c["pos0"], c["nh"], c["nkv"],
                                d["qn"], d["kn"], EPS)
            ops.attn_f32kv(d["q"], d["kc"], d["vc"], c["pos0"], c["nh"], c["nkv"], out=d["out"], scratch=scratch)
    else:
        nh, nkv = c["nh"], c["nkv"]
        for t0, n in st["calls"]:
            pos, t1 = c["pos0"] + t0, t0 + n
            for d in st["layers"]:
                q, k, v, out = d["q"][t0:t1], d["k"][t0:t1], d["v"][t0:t1], d["out"][t0:t1]
                if c["q16"]:
                    q16 = ops.attn_prep_f16_q16(q, k, v, d["kc"], d["vc"], pos, nh, nkv, q_norm=d["qn"], k_norm=d["kn"],
                                                eps=EPS)
                    ops.attn_f16_q16(q, q16, d["kc"], d["vc"], pos, nh, nkv, out=out, scratch=scratch)
                else:
                    ops.attn_prep_f16(q, k, v, d["kc"], d["vc"], pos, nh, nkv, d["qn"], d["kn"], EPS)
                    ops.attn_f16(q, d["kc"], d["vc"], pos, nh, nkv, out=out, scratch=scratch)


def run(st):
    if st["graph"] is not None:
        st["graph"].replay()
    else:
        _pass(st)
    c = st["case"]
    if c["op"].startswith("gdn"):
        return dict(out=st["out"], state=st["state"], conv=st["conv"])
    return [dict(out=d["out"], k=d["kc"][c["pos0"]:], v=d["vc"][c["pos0"]:]) for d in st["layers"]]


def work(case):
    """Each input read once and each output written once; products over the keys a token sees, and the
    recurrence token by token."""
    c, nt = case, case["nt"]
    if c["op"].startswith("gdn"):
        nv, cd = c["nv"], (2 * c["nk"] + c["nv"]) * S
        steps = _steps(c)
        per_step = nt * (cd + 2 * nv + 2 * nv * S) * 4        # x, gates, z in; out
        once = 2 * (nv * S * S + (KC - 1) * cd) * 4 + cd * KC * 4   # both states in and out, taps
        flops = steps * nt * (nv * 7 * S * S + 2 * KC * cd)
        if c["ckpt"]:                                         # a checkpoint a step, and the rollback's read
            once += 3 * (nv * S * S + (KC - 1) * cd) * 4
        return {"bytes": c["layers"] * (steps * per_step + once), "flops": c["layers"] * flops}
    size = 4 if c["op"] == "mtp" else 2
    kvd, keys = c["nkv"] * HD, c["pos0"] + nt
    seen = nt * c["pos0"] + nt * (nt + 1) // 2
    # q (normed in place) and gate in, out; k and v rows in and to the cache; the earlier rows in
    b = nt * c["nh"] * HD * 4 * 4 + 2 * nt * kvd * (4 + size) + 2 * c["pos0"] * kvd * size
    return {"bytes": c["layers"] * b, "flops": c["layers"] * 4 * HD * c["nh"] * seen}


def tolerance(case):
    """About four times what the calls differ by from exact()."""
    if case["op"] == "gdn_prefill":
        return {"rel": 2e-3}               # f16 products of a chunk, f32 state
    if case["op"] == "gdn_decode":
        return {"rel": 5e-6, "max": 2e-4}  # f32 arithmetic throughout
    if case["op"] == "attn" and case["nt"] >= 16:
        return {"rel": 1.2e-3}             # f16 query and probabilities
    if case["op"] == "attn":
        return {"rel": 3e-5, "max": 2e-3}  # f32 arithmetic; an appended f16 value may round the other way
    return {"rel": 5e-6, "max": 2e-4}      # f32 arithmetic throughout, cache included


# ---- the same in 64 bits

def _rope64(x, pos):
    """Rotates the first N_ROT dims of x [nt, heads, HD] at positions pos [nt]."""
    half = N_ROT // 2
    i = torch.arange(half, device=x.device)
    scale = float(torch.tensor(BASE, dtype=torch.float32) ** torch.tensor(-2.0 / N_ROT, dtype=torch.float32))
    ang = pos.double()[:, None] * (scale ** i.double())[None, :]
    sec = i % sum(SECTIONS)
    text = torch.zeros_like(sec, dtype=torch.bool)
    for r, s in ((1, SECTIONS[1]), (2, SECTIONS[2]), (0, SECTIONS[0])):
        text |= (sec % 3 == r) & (sec < 3 * s)
    ang = torch.where(text[None, :], ang, torch.zeros_like(ang))[:, None, :]
    lo, hi = x[..., :half], x[..., half:N_ROT]
    y = x.clone()
    y[..., :half] = lo * ang.cos() - hi * ang.sin()
    y[..., half:N_ROT] = hi * ang.cos() + lo * ang.sin()
    return y


def _norm64(x, w):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _attn64(c, d):
    nt, pos0, nh, nkv = c["nt"], c["pos0"], c["nh"], c["nkv"]
    pos = pos0 + (1 if c["op"] == "mtp" else 0) + torch.arange(nt, device="cuda")
    qg = d["q"].double().view(nt, nh, 2 * HD)
    q = _rope64(_norm64(qg[..., :HD], d["qn"]), pos)
    gate = torch.sigmoid(qg[..., HD:])
    k = _rope64(_norm64(d["k"].double().view(nt, nkv, HD), d["kn"]), pos).reshape(nt, -1)
    v = d["v"].double()
    # an f16 cache holds f16 values
    held = (lambda x: x) if c["op"] == "mtp" else (lambda x: x.float().half().double())
    k, v = held(k), held(v)
    kk = torch.cat([d["kc"][:pos0].double(), k]).view(-1, nkv, HD)
    vv = torch.cat([d["vc"][:pos0].double(), v]).view(-1, nkv, HD)
    out = torch.empty(nt, nh, HD, dtype=torch.float64, device="cuda")
    G = nh // nkv
    at = torch.arange(pos0 + nt, device="cuda")
    for t0 in range(0, nt, 256):
        t1 = min(nt, t0 + 256)
        hidden = at[None, :pos0 + t1] > (pos0 + torch.arange(t0, t1, device="cuda"))[:, None]
        for h in range(nh):
            s = q[t0:t1, h] @ kk[:pos0 + t1, h // G].T.contiguous() / math.sqrt(HD)
            out[t0:t1, h] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ vv[:pos0 + t1, h // G].contiguous()
    return dict(out=(out * gate).reshape(nt, -1), k=k, v=v)


def _gdn64(c, d):
    nt, nv, nk = c["nt"], c["nv"], c["nk"]
    state, conv, w = d["state"].double(), d["conv"].double(), d["w"].double()
    outs, back = [], None
    for i in range(_steps(c)):
        x = torch.cat([conv, d["x"][i].double()])
        y = sum(x[j:j + nt] * w[:, j] for j in range(KC))
        y = (y * torch.sigmoid(y)).view(nt, -1, S)
        qk = y[:, :2 * nk]
        qk = qk / qk.norm(dim=-1, keepdim=True).clamp_min(EPS)
        heads = torch.arange(nv, device="cuda") % nk
        q, k, v = qk[:, :nk][:, heads], qk[:, nk:][:, heads], y[:, 2 * nk:]
        beta = torch.sigmoid(d["beta"][i].double())
        decay = torch.exp(torch.nn.functional.softplus(d["alpha"][i].double() + d["dt"].double()) * d["a"].double())
        o = torch.empty(nt, nv, S, dtype=torch.float64, device="cuda")
        for t in range(nt):
            state = state * decay[t][:, None, None]
            delta = (v[t] - (state * k[t][:, :, None]).sum(1)) * beta[t][:, None]
            state = state + k[t][:, :, None] * delta[:, None, :]
            o[t] = (state * q[t][:, :, None]).sum(1)
            if c["ckpt"] and t == 0:
                back = (x[1:KC], state)    # the states after the step's first token
        o = o / math.sqrt(S)
        z = d["z"][i].double().view(nt, nv, S)
        outs.append((_norm64(o, d["nw"]) * z * torch.sigmoid(z)).reshape(nt, -1))
        conv = x[nt:]
    if c["ckpt"]:
        conv, state = back
    return dict(out=torch.stack(outs), state=state, conv=conv)


def exact(case, seed):
    c = dict(case)
    if not c["op"].startswith("gdn"):
        return [_attn64(c, d) for d in _inputs(c, seed)]
    each = [_gdn64(c, d) for d in _inputs(c, seed)]
    return {name: torch.stack([e[name] for e in each]) for name in each[0]}
