"""The work that a user of this framework has it do, as cases to measure.

Four kinds of call, each through the public entry points of the SGLang
binding (``mac_attention.integrations.sglang.bridge``):

* ``decode``: one fused decode step (``mac_persistent_decode_bf16``).  Serving
  captures it in a graph (``graph``); an eager server calls it directly.
* ``prefix``: the full prefill state (o, lse) of the rows the ring keeps, as
  the ROCm backends' prefill hook asks for it (``window_attention_return_lse``
  with no window).
* ``three_calls``: windowed attention over every row of a chunk, the
  downdate, and the ring write -- the composition of separate calls.
* ``rectify``: the fused form of that composition
  (``mac_prefill_rectify_update_cache``).
* ``rope``: decode RoPE with the pre-RoPE query kept and K/V written.

The decode cases decide hits by the documented synthetic override
(``bench_mode`` 1, exact quota): a step writes its query into the ring, so the
real scan would match that row when the same step is repeated, and the work
would not stay what the case says.  The scan itself runs as always, and the
ring holds near copies of the hit heads' queries where the override puts its
matches, so both would decide the same on a first pass.
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mac-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from mac_attention import synthetic as syn  # noqa: E402
from mac_attention.integrations.sglang import bridge  # noqa: E402

D = 128
SM = 1.0 / math.sqrt(D)
MAX_CONTEXT = 131072  # the serving default, which sizes the decode workspaces
TILE, MATCH_TILE = 32, 32  # serving defaults
LAG = 24  # matched tokens back from the current one (inside every ring used)
BENCH_SEED = 1
DEV = "cuda"


# ------------------------------------------------------------------ cases ---


def _decode(name, batch, hq, hkv, ctx, ring, hit, *, ragged=False, S=256, F=0, gated=False, graph=True,
            partial="f32", loc64=False):
    c = dict(kind="decode", batch=batch, hq=hq, hkv=hkv, ctx=ctx, ring=ring, hit=hit, ragged=ragged, S=S, F=F,
             gated=gated, graph=graph, partial=partial, loc64=loc64)
    return dict(c, name=name) if name else c


def _prefix(name, batch, rows, kv, hq, hkv, ragged=False):
    c = dict(kind="prefix", batch=batch, rows=rows, kv=kv, hq=hq, hkv=hkv, ragged=ragged)
    return dict(c, name=name) if name else c


def _three(name, batch, rows, prefix, hq, hkv, S, ring):
    c = dict(kind="three_calls", batch=batch, rows=rows, prefix=prefix, hq=hq, hkv=hkv, S=S, ring=ring)
    return dict(c, name=name) if name else c


def _rectify(name, batch, rows, prefix, hq, hkv, S, ring, F=0, sink_mode=0):
    c = dict(kind="rectify", batch=batch, rows=rows, prefix=prefix, hq=hq, hkv=hkv, S=S, ring=ring, F=F,
             sink_mode=sink_mode)
    return dict(c, name=name) if name else c


def _rope(name, batch, hq, hkv, rot, neox, loc64):
    c = dict(kind="rope", batch=batch, hq=hq, hkv=hkv, rot=rot, neox=neox, loc64=loc64)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one request at a short context on an eager server, default ring:
        # the smallest step, where the call itself and the launches count
        _decode("decode_eager_b1_4k", 1, 32, 8, 4096, 512, 0.5, graph=False),
        # a single long chat (32K context, front sink), half of the heads hit
        _decode("decode_b1_32k_sink", 1, 32, 8, 32768, 4096, 0.5, F=64),
        # a single request at the longest context with nothing to reuse, on
        # the 2048-slot ring of the published curves, bf16 partials
        _decode("decode_b1_127k_exact", 1, 32, 4, 126976, 2048, 0.0, partial="bf16"),
        # a small batch of medium contexts of unequal length with the default
        # ring: the everyday step of a server
        _decode("decode_b16_default", 16, 32, 8, 16384, 512, 0.9, ragged=True, loc64=True),
        # a large-ring deployment: 32768 cached queries per request to search
        _decode("decode_b16_ring32768", 16, 32, 4, 65536, 32768, 0.9, F=128),
        # a serving mix: ragged contexts, rings that are not ready or stale,
        # front sink, rows scattered over the pool
        _decode("decode_ragged_gated", 64, 32, 4, 126976, 32, 0.8, ragged=True, F=128, gated=True, loc64=True),
        # the headline step: 64 requests of 127K context, hit ratio 0.8
        _decode("decode_b64_127k", 64, 32, 8, 130048, 32, 0.8),
        # ring filling after one request's chunk: its last 512 rows over a
        # 32K context
        _prefix("prefix_b1_32k", 1, 512, 32768, 32, 8),
        # a batch of requests with short kept suffixes over long contexts
        _prefix("prefix_b8_ragged", 8, 32, 65536, 32, 4, ragged=True),
        # the three separate calls on whole chunks
        _three("three_calls_8x8192", 8, 8192, 2048, 32, 4, 256, 512),
        # the fused ring update of a batch's chunks, default ring
        _rectify("rectify_b8_ring512", 8, 2048, 1024, 32, 8, 256, 512),
        # RoPE and K/V write of a decode batch, from the fused qkv buffer
        _rope("rope_b64", 64, 32, 8, 128, True, True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["decode", "decode", "decode", "decode", "prefix", "prefix", "three_calls", "rectify", "rope"])
    hkv = rng.choice([1, 2, 4, 8, 8, 4])
    if kind == "decode":
        g = rng.choice([1, 2, 3, 4, 4, 5, 6, 7, 8, 8])
        ring = rng.choice([32, 48, 64, 100, 128, 256, 333, 512, 512, 1024, 2048, 4096])
        batch = _log(rng, 1, 64)
        # (at most the headline step's bytes, if nothing is reused)
        top = min(130048, (7_000_000_000 - batch * ring * g * hkv * D) // (batch * hkv * 4 * D))
        ctx = _log(rng, 2048, top)
        return _decode(None, batch, g * hkv, hkv, ctx, ring, round(rng.choice([0.0, 0.5, 0.8, 0.9, 1.0, rng.random()]), 3),
                       ragged=rng.random() < 0.6, S=rng.choice([64, 256, 256]), F=rng.choice([0, 0, 5, 64, 128]),
                       gated=rng.random() < 0.3, graph=rng.random() < 0.75,
                       partial=rng.choice(["f32", "f32", "bf16"]), loc64=rng.random() < 0.5)
    g = rng.choice([1, 2, 4, 4, 8, 8, 7])
    if kind == "prefix":
        batch = _log(rng, 1, 32)
        rows = _log(rng, 1, 2048 if batch < 8 else 512)
        # (at most the largest listed prefill's operations, and the headline step's bytes)
        top = min(126976, 270_000_000_000 // (4 * D * g * hkv * rows * batch), 6_900_000_000 // (4 * D * hkv * batch))
        kv = max(rows + 1, _log(rng, 300, max(top, 400)))
        return _prefix(None, batch, rows, kv, g * hkv, hkv, ragged=rng.random() < 0.6)
    if kind == "three_calls":
        batch = _log(rng, 1, 8)
        rows = _log(rng, 17, 8192)
        g = min(g, 32 // hkv)
        return _three(None, batch, rows, rng.randrange(1024, 4096), g * hkv, hkv, rng.choice([64, 128, 256, 256]),
                      rng.choice([32, 100, 512, 2048]))
    if kind == "rectify":
        batch = _log(rng, 1, 32)
        return _rectify(None, batch, _log(rng, 1, 2048), rng.randrange(1024, 4096), g * hkv, hkv,
                        rng.choice([64, 128, 256, 256]), rng.choice([32, 100, 512, 1024]), F=rng.choice([0, 0, 64]),
                        sink_mode=rng.choice([0, 1]))
    return _rope(None, _log(rng, 1, 512), g * hkv, hkv, rng.choice([64, 128, 128]), rng.random() < 0.7,
                 rng.random() < 0.5)


def _rng(case):
    """The case's own choices (lengths, readiness): the same for every seed,
    captured in a graph or not."""
    key = ",".join(f"{k}={case[k]}" for k in sorted(case) if k not in ("name", "graph"))
    return random.Random(key)


def _ragged(rng, n, top, low):
    return [max(low, _log(rng, max(top / 8, low), top)) for _ in range(n)]


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape, dtype=torch.bfloat16):
    """N(0, 1), filled in slices (a fill draws its numbers in float32)."""
    t = torch.empty(*shape, device=DEV, dtype=dtype)
    flat = t.view(-1)
    for i in range(0, flat.numel(), 1 << 28):
        flat[i:i + (1 << 28)].normal_(generator=g)
    return t


def _i32(xs):
    return torch.tensor(xs, device=DEV, dtype=torch.int32)


# ----------------------------------------------------------------- decode ---


def _decode_plan(case):
    """Past lengths, readiness, and per (request, head) whether the override
    makes it a hit and the head is reused (None: a miss, else the matched
    position)."""
    b, hq, S, F = case["batch"], case["hq"], case["S"], case["F"]
    g = hq // case["hkv"]
    rng = _rng(case)
    past = _ragged(rng, b, case["ctx"], 2048) if case["ragged"] else [case["ctx"]] * b
    state = [rng.random() for _ in range(b)] if case["gated"] else [1.0] * b
    # 20% of the requests have no ready ring, 10% a stale one
    ready = [0 if s < 0.2 else (2 if s < 0.3 else 1) for s in state]
    units = b * hq
    miss_units = min(max(int(math.floor(min(max(1.0 - case["hit"], 0.0), 1.0) * units + 0.5)), 0), units)
    match = []
    for n in range(b):
        base = (BENCH_SEED ^ ((past[n] * 0x85EBCA6B) & 0xFFFFFFFF)) & 0xFFFFFFFF
        row = []
        for h in range(hq):
            rot = n * hq + h + base % units
            rot -= units if rot >= units else 0
            pos = max(past[n] - min(LAG, case["ring"], past[n]), 0)
            hit = ready[n] == 1 and rot >= miss_units and past[n] + 1 - S > 0
            if hit and F > 0 and max(pos + 1 - S, 0) < F:
                hit = False
            row.append(pos if hit else None)
        match.append(row)
    return past, ready, match, g


def _slot(past, m, pos):
    if past < m:
        return pos
    return (pos - (past - m) + past % m) % m


def _decode_prepare(case, seed):
    b, hq, hkv, m, S = case["batch"], case["hq"], case["hkv"], case["ring"], case["S"]
    past, ready, match, _ = _decode_plan(case)
    g = _gen(seed)
    rows = sum(past) + b
    k, v = _normal(g, rows, hkv, D), _normal(g, rows, hkv, D)
    # requests' rows: back to back, or (ragged cases) scattered over the pool
    order = (torch.randperm(rows, generator=g, device=DEV) if case["ragged"] else torch.arange(rows, device=DEV)).int()
    r2t = torch.zeros(b, max(past) + 1, device=DEV, dtype=torch.int32)
    cur, at = [], 0
    for n, p in enumerate(past):
        r2t[n, :p + 1] = order[at:at + p + 1]
        at += p + 1
        cur.append(at - 1)
    loc = order[torch.tensor(cur, device=DEV)].to(torch.int64 if case["loc64"] else torch.int32).contiguous()
    q_pre, q_post = _normal(g, b, hq, D), _normal(g, b, hq, D)
    qc, ac = _normal(g, b, m, hq, D), _normal(g, b, m, hq, D)
    ac.mul_(1.0 / 16)  # prefix states average many values: small outputs,
    lc = _normal(g, b, m, hq, dtype=torch.float32) * 0.1  # lse near the log of their lengths
    lc += _i32(past).float().log().view(b, 1, 1)
    where = [(n, _slot(past[n], m, pos), h) for n, row in enumerate(match) for h, pos in enumerate(row) if pos is not None]
    if where:  # a hit head's query came by LAG tokens ago, slightly different
        ni, si, hi = torch.tensor(where, device=DEV).unbind(1)
        qc[ni, si, hi] = (0.98 * q_pre[ni, hi].float() + 0.2 * torch.randn(len(where), D, device=DEV, generator=g)).bfloat16()
    if case["gated"]:
        cr = torch.tensor([r != 0 for r in ready], device=DEV)
        ce = torch.tensor([1 if r == 2 else 2 for r in ready], device=DEV, dtype=torch.int64)
        re_ = torch.full((b,), 2, device=DEV, dtype=torch.int64)
    else:
        cr = ce = re_ = torch.empty(0, device=DEV)
    ws = syn.workspace(torch, batch=b, hq=hq, hkv=hkv, capacity=m, max_context=MAX_CONTEXT, tile_tokens=TILE,
                       match_tile_slots=MATCH_TILE, semantic_pos_ahead=S, front_sink_tokens=case["F"],
                       partial_dtype=torch.float32 if case["partial"] == "f32" else torch.bfloat16)
    out = torch.empty(b, hq, D, device=DEV, dtype=torch.bfloat16)
    out_lse = torch.empty(b, hq, device=DEV)
    ext = bridge.load_mac_persistent_decode_extension(False)
    args = (q_post, q_pre, k, v, r2t, torch.arange(b, device=DEV, dtype=torch.int32), _i32(past), loc, qc, ac, lc,
            out, out_lse, *ws, MAX_CONTEXT, TILE, MATCH_TILE, S, case["F"], 0, 0, 0, 0.45, SM, 0, 1,
            float(case["hit"]), 0.0, -1.0, 0.0, float(LAG), 0.0, BENCH_SEED, -1, 0, qc, cr, ce, re_)
    s = dict(kind="decode", ext=ext, args=args, outputs=(out, out_lse, qc, ac, lc, ws[3], ws[15]), graph=None)
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            ext.mac_persistent_decode_bf16(*args)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            ext.mac_persistent_decode_bf16(*args)
        s["graph"] = graph
    return s


def _attend(q, k, v):
    """Softmax attention state in 64 bits: q [G, 128], k and v [T, 128]."""
    x = (q.double() @ k.double().t()) * SM
    lse = torch.logsumexp(x, -1)
    return torch.exp(x - lse[:, None]) @ v.double(), lse


def _merge(a, b):
    """Two attention states of the same heads as one."""
    lse = torch.logaddexp(a[1], b[1])
    return a[0] * torch.exp(a[1] - lse)[:, None] + b[0] * torch.exp(b[1] - lse)[:, None], lse


def _decode_exact(case, seed):
    past, ready, match, g = _decode_plan(case)
    s = _decode_prepare(dict(case, graph=False), seed)
    q_post, q_pre, k, v, r2t, _, _, _, qc, ac, lc = s["args"][:11]
    b, hq, hkv, m, S, F = (case[x] for x in ("batch", "hq", "hkv", "ring", "S", "F"))
    out = torch.zeros(b, hq, D, device=DEV, dtype=torch.float64)
    out_lse = torch.zeros(b, hq, device=DEV, dtype=torch.float64)
    qc, ac, lc = qc.clone(), ac.double(), lc.double()
    hit = torch.zeros(b, hq, dtype=torch.int32, device=DEV)
    mode = torch.zeros(b, hkv, dtype=torch.int32, device=DEV)
    for n in range(b):
        P = past[n]
        rows = r2t[n, :P + 1].long()
        ne = max(P + 1 - S, 0)
        fs = min(F, ne)
        dest = P % m
        new_rows = []
        for kv in range(hkv):
            reuse = [match[n][kv * g + i] is not None for i in range(g)]
            mode[n, kv] = 0 if all(reuse) else (2 if any(reuse) else 1)
            need_all = not all(reuse)
            kk, vv = (k[rows, kv], v[rows, kv]) if need_all else (None, None)
            for begin in sorted({max(p + 1 - S, 0) if p is not None else fs for p in match[n][kv * g:(kv + 1) * g]}):
                heads = [i for i in range(g) if (max(match[n][kv * g + i] + 1 - S, 0) if reuse[i] else fs) == begin]
                h = torch.tensor([kv * g + i for i in heads], device=DEV)
                q = q_post[n, h]

                def part(lo, hi):
                    if hi <= lo:
                        return (torch.zeros(len(heads), D, device=DEV, dtype=torch.float64),
                                torch.full((len(heads),), -math.inf, device=DEV, dtype=torch.float64))
                    if need_all:
                        return _attend(q, kk[lo:hi], vv[lo:hi])
                    return _attend(q, k[rows[lo:hi], kv], v[rows[lo:hi], kv])

                ring = part(begin, ne)
                taken = torch.tensor([match[n][x] is not None for x in h.tolist()], device=DEV)
                if bool(taken.any()):
                    slots = torch.tensor([_slot(P, m, match[n][x]) if match[n][x] is not None else 0 for x in h.tolist()],
                                         device=DEV)
                    e = (ac[n, slots, h], torch.where(taken, lc[n, slots, h], -math.inf))
                    ring = _merge(ring, e) if ne > begin else e
                if ready[n] == 1:
                    new_rows.append((h, ring))
                o = _merge(ring, part(ne, P + 1)) if bool(torch.isfinite(ring[1]).all()) else part(ne, P + 1)
                if fs > 0:
                    o = _merge(o, part(0, fs))
                out[n, h], out_lse[n, h] = o
                hit[n, h] = taken.int()
        for h, (o, lse) in new_rows:
            qc[n, dest, h], ac[n, dest, h], lc[n, dest, h] = q_pre[n, h], o, lse
    return out, out_lse, qc, ac, lc, hit, mode


def _decode_work(case):
    past, ready, match, g = _decode_plan(case)
    b, hq, hkv, m, S, F = (case[x] for x in ("batch", "hq", "hkv", "ring", "S", "F"))
    tokens = flops = slots = 0
    for n in range(b):
        P = past[n]
        ne = max(P + 1 - S, 0)
        fs = min(F, ne)
        for kv in range(hkv):
            row = match[n][kv * g:(kv + 1) * g]
            begins = [max(p + 1 - S, 0) if p is not None else fs for p in row]
            begin = min(begins)
            t = fs + (ne - begin) + (P + 1 - ne)
            tokens += t
            flops += 4 * D * sum(fs + (ne - x) + (P + 1 - ne) for x in begins)
        slots += min(m, P)
    # a slot far from the query can be told from half of its row
    scan = slots * hq * D
    small = b * hq * (D * 2 * 5 + 3 * 4) + 4 * sum(past)
    return dict(bytes=tokens * 2 * 2 * D + scan + small, flops=flops)


# ---------------------------------------------------------------- prefill ---


def _ragged_batch(case, qlens, kvlens, seed):
    """Queries and scattered K/V rows of a ragged chunk, with its offsets."""
    g = _gen(seed)
    hq, hkv, total = case["hq"], case["hkv"], sum(kvlens)
    pool = total + 16
    acc = lambda xs: [sum(xs[:i]) for i in range(len(xs) + 1)]  # noqa: E731
    return g, dict(q=_normal(g, sum(qlens), hq, D), k=_normal(g, pool, hkv, D), v=_normal(g, pool, hkv, D),
                   qo=_i32(acc(qlens)), kvp=_i32(acc(kvlens)),
                   kvi=torch.randperm(pool, generator=g, device=DEV)[:total].int().contiguous())


def _prefix_lens(case):
    rng = _rng(case)
    b = case["batch"]
    rows = [rng.randint(max(1, case["rows"] // 2), case["rows"]) for _ in range(b)] if case["ragged"] else [case["rows"]] * b
    kv = _ragged(rng, b, case["kv"], case["rows"]) if case["ragged"] else [case["kv"]] * b
    return rows, kv


def _windowed(q, k, v, qlens, kvlens, kvi, window):
    """Causal (windowed: the last `window` keys up to a row's own) attention
    of a ragged batch in 64 bits; window None: every key up to a row's own."""
    hq, hkv = q.shape[1], k.shape[1]
    g = hq // hkv
    o = torch.zeros(q.shape, device=DEV, dtype=torch.float64)
    lse = torch.zeros(q.shape[:2], device=DEV, dtype=torch.float64)
    q0 = k0 = 0
    for ql, kl in zip(qlens, kvlens):
        step = max(1, min(512, (1 << 25) // (kl * g))) if window is None else 512
        for i in range(0, ql, step):
            n = min(step, ql - i)
            p0 = kl - ql + i
            lo = 0 if window is None else max(p0 + 1 - window, 0)
            keys = kvi[k0 + lo:k0 + p0 + n].long()
            pos = torch.arange(p0, p0 + n, device=DEV)[:, None]
            at = torch.arange(lo, p0 + n, device=DEV)[None, :]
            seen = (at <= pos) if window is None else (at <= pos) & (at > pos - window)
            for kv in range(hkv):
                kk, vv = k[keys, kv].double(), v[keys, kv].double()
                x = q[q0 + i:q0 + i + n, kv * g:(kv + 1) * g].double().reshape(n * g, D) @ kk.t().contiguous() * SM
                x = x.view(n, g, -1).masked_fill_(~seen[:, None, :], -math.inf)
                l = torch.logsumexp(x, -1)
                o[q0 + i:q0 + i + n, kv * g:(kv + 1) * g] = (torch.exp(x - l[..., None]).view(n * g, -1) @ vv).view(n, g, D)
                lse[q0 + i:q0 + i + n, kv * g:(kv + 1) * g] = l
        q0 += ql
        k0 += kl
    return o, lse


def _seen_keys(rows, kv, window):
    """Sum over the last `rows` positions of kv of the keys each attends to."""
    first = kv - rows + 1
    if window is None:
        return rows * (first + kv) // 2
    short = max(0, min(window, kv + 1) - first)
    return short * (2 * first + short - 1) // 2 + (rows - short) * window


def _full_state(g, qlens, kvlens, hq):
    """A full prefill state as such inputs give it: values N(0, 1) averaged
    with softmax weights of N(0, 1) scores over the row's keys."""
    n = torch.cat([torch.arange(kl - ql + 1, kl + 1, device=DEV) for ql, kl in zip(qlens, kvlens)]).float()
    lse = n.log()[:, None] + 0.5 + 0.05 * torch.randn(n.numel(), hq, device=DEV, generator=g)
    o = _normal(g, n.numel(), hq, D)
    o.mul_((math.e / n).sqrt()[:, None, None])
    return o, lse.contiguous()


def _ring_state(case, g, b):
    """Rings of twice the batch's requests; the batch takes every other one."""
    r, m, hq = 2 * b, case["ring"], case["hq"]
    return (_normal(g, r, m, hq, D), _normal(g, r, m, hq, D), _normal(g, r, m, hq, dtype=torch.float32),
            torch.arange(0, r, 2, device=DEV, dtype=torch.int32))


def _chunk_prepare(case, seed):
    b, rows, prefix = case["batch"], case["rows"], case["prefix"]
    qlens, kvlens = [rows] * b, [rows + prefix] * b
    g, s = _ragged_batch(case, qlens, kvlens, seed)
    s["o"], s["lse"] = _full_state(g, qlens, kvlens, case["hq"])
    s["src_q"] = _normal(g, b * rows, case["hq"], D)
    s["qc"], s["ac"], s["lc"], s["ids"] = _ring_state(case, g, b)
    s["length"] = torch.full((2 * b,), prefix, device=DEV, dtype=torch.int32)
    s["lens"] = _i32(qlens)
    s.update(kind=case["kind"], S=case["S"], F=case.get("F", 0), sink_mode=case.get("sink_mode", 0), ring=case["ring"],
             hq=case["hq"])
    return s


def _downdate(o, lse, ow, lw):
    rest = lse + torch.log1p(-torch.exp(lw - lse) + 1e-7)
    return (o.double() - torch.exp(lw - lse)[..., None] * ow) * torch.exp(lse - rest)[..., None], rest


def _chunk_exact(case, seed):
    s = _chunk_prepare(case, seed)
    b, rows, prefix, m, S = (case[x] for x in ("batch", "rows", "prefix", "ring", "S"))
    qlens, kvlens = [rows] * b, [rows + prefix] * b
    keep = min(rows, m)
    fused = case["kind"] == "rectify"
    calc = keep if fused else rows  # rows of each request whose window is needed
    last = torch.cat([torch.arange((i + 1) * rows - calc, (i + 1) * rows, device=DEV) for i in range(b)])
    q, o, lse = s["q"][last], s["o"][last], s["lse"][last].double()
    ow, lw = _windowed(q, s["k"], s["v"], [calc] * b, kvlens, s["kvi"], S)
    F, with_sink = case.get("F", 0), fused and case["sink_mode"] == 1 and case["F"] > 0
    if with_sink:  # (the prefix is longer than sink and window: every row has the whole sink)
        ls, os_ = torch.zeros_like(lw), torch.zeros_like(ow)
        g = case["hq"] // case["hkv"]
        for i in range(b):
            at = s["kvi"][i * (rows + prefix):i * (rows + prefix) + F].long()
            for h in range(case["hq"]):
                r = slice(i * calc, (i + 1) * calc)
                os_[r, h], ls[r, h] = _attend(q[r, h], s["k"][at, h // g], s["v"][at, h // g])
        both = torch.logaddexp(lw, ls)
        ow = ow * torch.exp(lw - both)[..., None] + os_ * torch.exp(ls - both)[..., None]
        lw = both
    od, ld = _downdate(o, lse, ow, lw)
    qc, ac, lc, length = s["qc"].clone(), s["ac"].double(), s["lc"].double(), s["length"].clone()
    slots = (prefix + rows - keep + torch.arange(keep, device=DEV)) % m
    for i in range(b):
        mine = slice((i + 1) * calc - keep, (i + 1) * calc)
        qc[2 * i, slots] = s["src_q"][(i + 1) * rows - keep:(i + 1) * rows]
        ac[2 * i, slots] = od[mine]
        lc[2 * i, slots] = -math.inf if fused and F > 0 and case["sink_mode"] == 0 else ld[mine]
        length[2 * i] += rows
    if fused:
        return qc, ac, lc, length
    return od, ld, qc, ac, lc, length


def _chunk_work(case):
    b, rows, prefix, m, S, hq, hkv = (case[x] for x in ("batch", "rows", "prefix", "ring", "S", "hq", "hkv"))
    keep = min(rows, m)
    calc = keep if case["kind"] == "rectify" else rows
    seen = _seen_keys(calc, rows + prefix, S)
    row = hq * D * 2
    kv = (min(calc + S - 1, rows + prefix)) * hkv * D * 4
    if case["kind"] == "rectify":
        f = case["F"] if case["sink_mode"] == 1 else 0
        return dict(bytes=b * (kv + f * hkv * D * 4 + keep * (5 * row + 8 * hq)), flops=4 * D * hq * b * (seen + calc * f))
    # queries and the full state read, the rectified state written, then the
    # kept rows' queries read and the rings written
    return dict(bytes=b * (kv + rows * (3 * row + 8 * hq) + keep * (3 * row + 4 * hq)), flops=4 * D * hq * b * seen)


# ------------------------------------------------------------------- rope ---


def _rope_prepare(case, seed):
    b, hq, hkv, rot = case["batch"], case["hq"], case["hkv"], case["rot"]
    g = _gen(seed)
    pool, positions = 8192, 131072
    qkv = _normal(g, b, (hq + 2 * hkv) * D)
    q, k, v = qkv.split([hq * D, hkv * D, hkv * D], dim=1)
    inv = 1.0 / (10000.0 ** (torch.arange(0, rot, 2, device=DEV, dtype=torch.float64) / rot))
    angle = torch.arange(positions, device=DEV, dtype=torch.float64)[:, None] * inv[None, :]
    cs = torch.cat([angle.cos(), angle.sin()], 1).float().contiguous()
    it = torch.int64 if case["loc64"] else torch.int32
    return dict(kind="rope", q=q, k=k, v=v, q_pre=torch.empty(b, hq, D, device=DEV, dtype=torch.bfloat16),
                kb=_normal(g, pool, hkv, D), vb=_normal(g, pool, hkv, D), cs=cs,
                pos=torch.randint(0, positions, (b,), generator=g, device=DEV).to(it),
                loc=torch.randperm(pool, generator=g, device=DEV)[:b].to(it), neox=case["neox"], hq=hq, hkv=hkv,
                ext=bridge.load_mac_decode_rope_preserve_extension(False))


def _rope_exact(case, seed):
    s = _rope_prepare(case, seed)
    b, rot, half = case["batch"], case["rot"], case["rot"] // 2
    cs = s["cs"][s["pos"].long()].double()
    c, si = cs[:, None, :half], cs[:, None, half:]

    def turned(x, heads):
        y = x.reshape(b, heads, D).double().clone()
        r = y[..., :rot].clone()
        x0, x1 = (r[..., :half], r[..., half:]) if case["neox"] else (r[..., 0::2], r[..., 1::2])
        y0, y1 = x0 * c - x1 * si, x1 * c + x0 * si
        y[..., :rot] = torch.cat([y0, y1], -1) if case["neox"] else torch.stack([y0, y1], -1).flatten(-2)
        return y

    q_pre = s["q"].reshape(b, case["hq"], D).clone()
    q, k = turned(s["q"], case["hq"]), turned(s["k"], case["hkv"])
    kb, vb = s["kb"].double(), s["vb"].clone()
    kb[s["loc"].long()] = k
    vb[s["loc"].long()] = s["v"].reshape(b, case["hkv"], D)
    return q.view(b, -1), k.view(b, -1), q_pre, kb, vb


# ----------------------------------------------------------- entry points ---


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return _decode_prepare(case, seed)
    if kind == "rope":
        return _rope_prepare(case, seed)
    ext = bridge.load_mac_prefill_rectify_extension(False)
    if kind == "prefix":
        s = _ragged_batch(case, *_prefix_lens(case), seed)[1]
        return dict(s, kind=kind, ext=ext)
    s = _chunk_prepare(case, seed)
    return dict(s, ext=ext, down=bridge.load_mac_merge_downdate_cache_extension(False),
                update=bridge.load_mac_prefill_update_cache_extension(False))


def run(s):
    kind = s["kind"]
    if kind == "decode":
        if s["graph"] is not None:
            s["graph"].replay()
        else:
            s["ext"].mac_persistent_decode_bf16(*s["args"])
        return s["outputs"]
    if kind == "rope":
        s["ext"].mac_decode_rope_preserve_q_bf16(s["q"], s["k"], s["v"], s["q_pre"], s["kb"], s["vb"], s["cs"], s["pos"],
                                                 s["loc"], D, s["neox"])
        return s["q"], s["k"], s["q_pre"], s["kb"], s["vb"]
    if kind == "prefix":
        return s["ext"].window_attention_return_lse(s["q"], s["k"], s["v"], s["qo"], s["kvp"], s["kvi"], -1, SM)
    if kind == "three_calls":
        o, lse = s["ext"].window_attention_return_lse(s["q"], s["k"], s["v"], s["qo"], s["kvp"], s["kvi"], s["S"] - 1, SM)
        s["down"].mac_update_then_downdate_bf16_inplace(s["o"], s["lse"], o, lse)
        s["update"].mac_prefill_update_cache(s["qc"], s["ac"], s["lc"], s["length"], s["ids"], s["src_q"], o, lse, s["qo"],
                                             s["lens"], s["ring"], s["hq"], D, None)
        return o, lse, s["qc"], s["ac"], s["lc"], s["length"]
    s["ext"].mac_prefill_rectify_update_cache(s["q"], s["src_q"], s["o"], s["lse"], s["k"], s["v"], s["qo"], s["kvp"],
                                              s["kvi"], s["qc"], s["ac"], s["lc"], s["length"], s["ids"], s["S"], s["F"],
                                              SM, sink_mode=s["sink_mode"])
    return s["qc"], s["ac"], s["lc"], s["length"]


def work(case):
    kind = case["kind"]
    if kind == "decode":
        return _decode_work(case)
    hq, hkv, b = case["hq"], case["hkv"], case["batch"]
    if kind == "rope":
        row = (hq + 2 * hkv) * D * 2
        return dict(bytes=b * (row + (hq + hkv) * D * 2 + hq * D * 2 + 2 * hkv * D * 2 + case["rot"] * 4),
                    flops=b * (hq + hkv) * case["rot"] * 3)
    if kind == "prefix":
        rows, kv = _prefix_lens(case)
        return dict(bytes=sum(rows) * hq * (D * 4 + 4) + sum(kv) * (hkv * D * 4 + 4),
                    flops=4 * D * hq * sum(_seen_keys(r, k, None) for r, k in zip(rows, kv)))
    return _chunk_work(case)


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return _decode_exact(case, seed)
    if kind == "rope":
        return _rope_exact(case, seed)
    if kind == "prefix":
        rows, kv = _prefix_lens(case)
        s = _ragged_batch(case, rows, kv, seed)[1]
        return _windowed(s["q"], s["k"], s["v"], rows, kv, s["kvi"], None)
    return _chunk_exact(case, seed)


def tolerance(case):
    """bf16 results: a correctly rounded one is 1.7e-3 from its value in the
    2-norm.  Attention over a chunk also rounds its weights to bf16 (2.4e-3
    in all, measured against 64 bits).  Four times each."""
    return {"rel": 1e-2 if case["kind"] in ("prefix", "three_calls") else 7e-3}
