"""The work this library is measured by, through its public entry points.

One full-attention layer of the engine makes three kinds of calls, and the cases are those calls at the sizes the
engine runs them: a decode step or MTP verify window (attn_decode with split-K partials), a prefill chunk (attn_decode
with one split) and the dense projections on either side of the attention (gemv / gemm of the qkv and o matrices).
The model's sizes are fixed (16 query heads, 2 kv heads, head dim 256, hidden 2048); the number of tokens, the context,
the cache's capacity, the cache format and the weight form vary.

  listed()  the named cases        draw(rng)  one more of the same ranges
  prepare() inputs on the GPU      run()      one pass through the entry points
  work()    bytes and flops that one pass cannot do without
  exact()   the same outputs in 64 bits by plain torch
"""
import math

import torch

import moex_amd as M

H, KV, D = 16, 2, 256
HIDDEN = 2048
LQ = H * 2 * D + 2 * KV * D  # one token's row of the fused qkv projection: (query, gate) per head, then k, then v
ROT, THETA, EPS = 64, 1e7, 1e-6
MAX_CONTEXT = 262144
CAPACITIES = (8192, 32768, 131072, MAX_CONTEXT)  # positions a session's cache is allocated for
FORMS = ("int8", "int4", "int6", "f16")
QKV, O = (LQ, HIDDEN), (HIDDEN, H * D)  # the two dense matrices, [outputs][inputs]


def _step(T, pos, cap, turbo):
    return {"kind": "step", "T": T, "pos": pos, "cap": cap, "turbo": turbo}


def _chunk(T, pos, cap, turbo):
    return {"kind": "chunk", "T": T, "pos": pos, "cap": cap, "turbo": turbo}


def _dense(S, form):
    return {"kind": "dense", "T": S, "form": form}


def listed():
    return [
        # one generated token early in a chat: a short context in a small cache, all latency and launches
        dict(_step(1, 700, 8192, False), name="step_short"),
        # one generated token over a long document, the int8 cache read once
        dict(_step(1, 89999, 131072, False), name="step_90k"),
        # an MTP verify window: four tokens over the same context
        dict(_step(4, 89996, 131072, False), name="window4_90k"),
        # one generated token at the model's full context, in the compressed (TurboQuant) cache made for it
        dict(_step(1, MAX_CONTEXT - 1, MAX_CONTEXT, True), name="step_turbo_262k"),
        # the first prefill chunk of a prompt, nothing cached before it
        dict(_chunk(2048, 0, 32768, False), name="chunk_first"),
        # the ragged last chunk of a prompt of a few thousand tokens
        dict(_chunk(213, 6144, 8192, False), name="chunk_tail"),
        # a full chunk in the middle of a long prompt
        dict(_chunk(2048, 32768, MAX_CONTEXT, False), name="chunk_32k"),
        # the last chunk of the longest prompt, compressed cache: the largest call
        dict(_chunk(2048, MAX_CONTEXT - 2048, MAX_CONTEXT, True), name="chunk_turbo_262k"),
        # the projections around a decode step
        dict(_dense(1, "int8"), name="dense_1"),
        # the projections around an MTP verify window
        dict(_dense(4, "int8"), name="dense_4"),
        # the projections of a ragged chunk, weights in the small form
        dict(_dense(300, "int4"), name="dense_300_int4"),
        # the projections of a full prefill chunk
        dict(_dense(2048, "int8"), name="dense_2048"),
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("step", "step", "chunk", "dense"))
    if kind == "dense":
        return _dense(_log_uniform(rng, 1, 2048), rng.choice(FORMS))
    turbo = rng.random() < 0.4
    if kind == "step":
        T = rng.choice((1, 1, 1, 2, 3, 4, 6, 8))
        pos = _log_uniform(rng, 16, MAX_CONTEXT - T)
    else:
        T = _log_uniform(rng, 9, 2048)
        pos = 0 if rng.random() < 0.25 else _log_uniform(rng, 32, MAX_CONTEXT - T)
    cap = rng.choice([c for c in CAPACITIES if c >= pos + T])
    return (_step if kind == "step" else _chunk)(T, pos, cap, turbo)


# ---- the TurboQuant format (data of the format): sign tables, centroid codes, thresholds ----
_S1 = ("-++--+-+--+++++++-+-+--+++-++----++-++-+-++--+-++++-----+-++++-+"
       "--+---+---+---+++--+++--++-++-+--++-+-+-++++-+-++-++-----++-++-+")
_S2 = ("++++-++-+---+---++--+-+-+--+-+++++---+------+++-+-+++--+------++"
       "+-+----+-+-+--++-+-++-+----+--+-+-+++--+-+-++--+-+-++-+-+-----+-")


def _signs(text):
    return torch.tensor([1.0 if c == "+" else -1.0 for c in text], dtype=torch.float64, device="cuda")


_I4 = (-127, -96, -75, -58, -44, -31, -18, -6, 6, 18, 31, 44, 58, 75, 96, 127)
_I3 = (-127, -79, -45, -14, 14, 45, 79, 127)
_M4 = (-0.212203, -0.162947, -0.127026, -0.097164, -0.070671, -0.046174, -0.022824, 0.0,
       0.022824, 0.046174, 0.070671, 0.097164, 0.127026, 0.162947, 0.212203)
_M3 = (-0.154496, -0.092804, -0.044243, 0.0, 0.044243, 0.092804, 0.154496)
_K4, _K3 = 0.241529 / 127, 0.190207 / 127


def _pack_turbo(ik, iv):
    """codes [.., 256] -> the cache's K bytes [.., 128] and V bytes [.., 96]"""
    k = (ik[..., 0::2] | ik[..., 1::2] << 4).to(torch.uint8)
    low = sum((iv[..., j::4] & 3) << 2 * j for j in range(4)).to(torch.uint8)
    high = sum((iv[..., j::8] >> 2) << j for j in range(8)).to(torch.uint8)
    return k, torch.cat([low, high], -1)


def _unpack_turbo(k, v):
    k, v = k.int(), v.int()
    ik = torch.stack([k & 15, k >> 4], -1).flatten(-2)
    low = torch.stack([v[..., :64] >> 2 * j & 3 for j in range(4)], -1).flatten(-2)
    high = torch.stack([v[..., 64:] >> j & 1 for j in range(8)], -1).flatten(-2)
    return ik, low | high << 2


# ---- inputs ----
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _cached(case, g):
    """The cache before the call: rows [0, pos) of keys and values of unit variance, as appends of them leave it."""
    n, cap, turbo = case["pos"], case["cap"], case["turbo"]
    c = M.DeviceKVCache(KV, cap, turbo)
    for a in (c.k, c.v, c.ks, c.vs):
        a.zero_()
    for h in range(KV):
        for p in range(0, n, 65536):
            m = min(65536, n - p)
            kr = torch.randn((m, D), generator=g, device="cuda")
            vr = torch.randn((m, D), generator=g, device="cuda")
            if turbo:  # the rotated halves of unit-variance rows are again normal: codes by the thresholds
                ik = torch.bucketize(kr, torch.tensor(_M4, device="cuda") * math.sqrt(128), right=True).int()
                iv = torch.bucketize(vr, torch.tensor(_M3, device="cuda") * math.sqrt(128), right=True).int()
                c.k[h, p:p + m], c.v[h, p:p + m] = _pack_turbo(ik, iv)
                c.ks[h, p:p + m] = kr.view(m, 2, 128).norm(dim=-1)
                c.vs[h, p:p + m] = vr.view(m, 2, 128).norm(dim=-1)
            else:
                for rows, codes, scales in ((kr, c.k, c.ks), (vr, c.v, c.vs)):
                    s = rows.abs().amax(-1) / 127
                    codes[h, p:p + m] = (rows / s[:, None]).round().to(torch.int8)
                    scales[h, p:p + m] = s
    return c


def _codes(shape, spread, lo, hi, g):
    return (torch.randn(shape, generator=g, device="cuda") * spread).round().clamp(lo, hi).to(torch.int32)


def _matrix(form, O_, I, g):
    """(fields of M.Mat, codes or values, scales) of one matrix with rows of about 1/sqrt(I) per weight"""
    size = 1 / math.sqrt(I)
    jitter = torch.rand(O_ if form in ("int8", "f16") else (O_, I // 64), generator=g, device="cuda") * 0.4 + 0.8
    if form == "f16":
        w = (torch.randn((O_, I), generator=g, device="cuda") * size).half()
        return {"f16": w}, w, None
    spread = {"int8": 36.0, "int4": 2.8, "int6": 11.0}[form]
    s = (jitter * (size / spread)).float().contiguous()
    if form == "int8":
        q = _codes((O_, I), spread, -127, 127, g).to(torch.int8)
        return {"q": q, "s": s}, q, s
    if form == "int4":
        q = _codes((O_, I), spread, -8, 7, g)
        return {"q4": (q[:, 0::2] & 15 | (q[:, 1::2] & 15) << 4).to(torch.uint8), "s": s}, q, s
    q = _codes((O_, I), spread, -32, 31, g)
    u = q + 32
    low = (u[:, 0::2] & 15 | (u[:, 1::2] & 15) << 4).to(torch.uint8)
    high = sum((u[:, j::4] >> 4) << 2 * j for j in range(4)).to(torch.uint8)
    return {"q6": low, "q6h": high, "s": s}, q, s


def _dense_inputs(case, seed):
    g = _gen(seed)
    S, got = case["T"], []
    for O_, I in (QKV, O):
        fields, q, s = _matrix(case["form"], O_, I, g)
        x = torch.randn((S, I), generator=g, device="cuda")  # normalised activations
        got.append((fields, q, s, x, O_, I))
    return got


def _attn_inputs(case, seed):
    g = _gen(seed)
    cache = _cached(case, g)
    T = case["T"]
    qkv = torch.randn((T, LQ), generator=g, device="cuda")  # rows of the fused projection
    qn = (torch.randn(D, generator=g, device="cuda") * 0.1).half()
    kn = (torch.randn(D, generator=g, device="cuda") * 0.1).half()
    return cache, qkv, qn, kn


def prepare(case, seed):
    if case["kind"] == "dense":
        st = {"kind": "dense", "S": case["T"], "mats": []}
        for fields, _, _, x, O_, I in _dense_inputs(case, seed):
            st["mats"].append((M.Mat(**fields), fields, x, torch.empty((case["T"], O_), device="cuda"), I, O_))
        return st
    cache, qkv, qn, kn = _attn_inputs(case, seed)
    T = case["T"]
    ns = M.decode_splits(case["cap"]) if case["kind"] == "step" else 1
    return {"kind": case["kind"], "T": T, "cap": case["cap"], "cache": cache, "qkv": qkv, "qn": qn, "kn": kn, "ns": ns,
            "part": torch.empty(T * H * ns * (D + 2), device="cuda") if ns > 1 else None,
            "pos": torch.tensor([case["pos"]], dtype=torch.int32, device="cuda"),
            "qo": torch.empty((T, H, D), device="cuda"), "out": torch.empty((T, H, D), device="cuda")}


def run(state):
    if state["kind"] == "dense":
        for mat, _, x, y, I, O_ in state["mats"]:
            if state["S"] == 1:
                M.gemv(mat, x, y, I, O_)
            else:
                M.gemm(mat, x, y, state["S"], I, O_)
        return {"qkv": state["mats"][0][3], "o": state["mats"][1][3]}
    qkv, c = state["qkv"], state["cache"]
    M.attn_decode(qkv, qkv[:, H * 2 * D:], qkv[:, H * 2 * D + KV * D:], state["qn"], state["kn"], state["qo"], c,
                  state["out"], H, KV, state["pos"], state["cap"], ROT, THETA, EPS, state["T"], LQ, None,
                  state["part"], state["ns"])
    # the output, the query the call leaves behind, and the cache it has appended to
    return {"out": state["out"], "qo": state["qo"], "k": c.k, "v": c.v, "ks": c.ks, "vs": c.vs}


def work(case):
    T = case["T"]
    if case["kind"] == "dense":
        per = {"int8": 1.0, "int4": 0.5 + 4 / 64, "int6": 0.75 + 4 / 64, "f16": 2.0}[case["form"]]
        return {"bytes": sum(O_ * I * per + (4.0 * O_ if case["form"] == "int8" else 0.0) + 4.0 * T * (I + O_)
                             for O_, I in (QKV, O)),
                "flops": sum(2.0 * T * O_ * I for O_, I in (QKV, O))}
    row = 240 if case["turbo"] else 520
    keys = case["pos"] * T + T * (T + 1) // 2
    return {"bytes": float(KV * case["pos"] * row + KV * T * row + 4 * T * (LQ + 2 * H * D)),
            "flops": 4.0 * H * D * keys}


def tolerance(case):
    if case["kind"] == "dense":
        # fp32 sums of 2048 to 4096 products, or one rounding of the inputs (and scaled weights) to fp16 before them
        gemv = case["T"] <= (8 if case["form"] in ("int8", "int6") else 2)
        return {"rel": 1e-6, "max": 2e-5} if gemv else {"rel": 1e-3, "max": 1e-2}
    # the cache codes: a row whose value lies on a rounding border may fall to the other side
    if case["kind"] == "step":
        return {"rel": 2e-5, "max": 1e-3, "differ": 1e-5}  # attention in fp32
    return {"rel": 2e-3, "max": 5e-2, "differ": 1e-5}  # queries and probabilities rounded to fp16


# ---- the same in 64 bits ----
def _hadamard():
    h = torch.ones((1, 1), dtype=torch.float64, device="cuda")
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(128)


def _rotate(x, inverse=False):
    first, last = (_signs(_S2), _signs(_S1)) if inverse else (_signs(_S1), _signs(_S2))
    y = x.reshape(-1, 128) * first
    return (y @ _hadamard() * last).reshape(x.shape)


def _front(x, w, pos):
    """RMSNorm(1 + w) and rotary embedding of rows [T][heads][256] at positions pos + t"""
    x = x.double()
    y = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * (1 + w.double())
    half = ROT // 2
    j = torch.arange(half, dtype=torch.float64, device="cuda")
    freq = (torch.tensor(THETA, dtype=torch.float64, device="cuda") ** (-2 * j / ROT)).float()
    p = torch.arange(pos, pos + x.shape[0], device="cuda").float()
    a = (p[:, None, None] * freq).double()  # the format's angle is a product in 32 bits
    u, v = y[..., :half], y[..., half:ROT]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), y[..., ROT:]], -1)


def _int8_rows(x):
    s = x.abs().amax(-1) / 127
    return (x / s[..., None]).round(), s


def _turbo_rows(x, thresholds, centroids, unit):
    t = torch.tensor(thresholds, dtype=torch.float64, device="cuda")
    c = torch.tensor(centroids, dtype=torch.float64, device="cuda")
    halves = x.reshape(*x.shape[:-1], 2, 128)
    n = halves.norm(dim=-1)
    ix = torch.bucketize(_rotate(halves / n[..., None]).contiguous(), t, right=True)
    return c[ix].reshape(x.shape), n / (c[ix] * unit).norm(dim=-1)


def exact(case, seed):
    if case["kind"] == "dense":
        got = []
        for _, q, s, x, O_, I in _dense_inputs(case, seed):
            w = q.double()
            if s is not None:
                w = w * s.double()[:, None] if s.dim() == 1 else (w.view(O_, I // 64, 64) * s.double()[..., None]).view(O_, I)
            got.append(x.double() @ w.t().contiguous())
        return {"qkv": got[0], "o": got[1]}
    cache, qkv, qn, kn = _attn_inputs(case, seed)
    T, pos, turbo = case["T"], case["pos"], case["turbo"]
    n = pos + T
    q = qkv[:, :H * 2 * D].reshape(T, H, 2, D)
    k = _front(qkv[:, H * 2 * D:H * 2 * D + KV * D].reshape(T, KV, D), kn, pos)
    v = qkv[:, H * 2 * D + KV * D:].reshape(T, KV, D).double()
    qo = _front(q[:, :, 0], qn, pos)
    gate = torch.sigmoid(q[:, :, 1].double())
    if turbo:
        qo = _rotate(qo)
    ks, vs = cache.ks.double(), cache.vs.double()
    out = torch.empty((T, H, D), dtype=torch.float64, device="cuda")
    for h in range(KV):
        if turbo:
            ik, iv = _unpack_turbo(cache.k[h, :pos], cache.v[h, :pos])
            kc = torch.tensor(_I4, dtype=torch.float64, device="cuda")[ik]
            vc = torch.tensor(_I3, dtype=torch.float64, device="cuda")[iv]
            nk, ks[h, pos:n] = _turbo_rows(k[:, h], _M4, _I4, _K4)
            nv, vs[h, pos:n] = _turbo_rows(v[:, h], _M3, _I3, _K3)
            spread = lambda s: s.repeat_interleave(128, -1)  # noqa: E731  one norm per half
            kd = torch.cat([kc, nk]) * spread(ks[h, :n]) * _K4
            vd = torch.cat([vc, nv]) * spread(vs[h, :n]) * _K3
            del ik, iv, kc, vc
        else:
            nk, ks[h, pos:n] = _int8_rows(k[:, h])
            nv, vs[h, pos:n] = _int8_rows(v[:, h])
            kd = torch.cat([cache.k[h, :pos].double(), nk]) * ks[h, :n, None]
            vd = torch.cat([cache.v[h, :pos].double(), nv]) * vs[h, :n, None]
        kt = kd.t().contiguous()
        del kd
        heads = slice(h * (H // KV), (h + 1) * (H // KV))
        step = max(1, min(T, int(1.6e8) // (n * (H // KV))))
        for t in range(0, T, step):
            e = min(T, t + step)
            m = pos + e
            s = qo[t:e, heads].reshape(-1, D) @ kt[:, :m] / math.sqrt(D)
            late = torch.arange(m, device="cuda")[None, :] > pos + torch.arange(t, e, device="cuda")[:, None]
            s.view(e - t, H // KV, m).masked_fill_(late[:, None, :], -math.inf)
            out[t:e, heads] = (torch.softmax(s, -1) @ vd[:m]).view(e - t, H // KV, D)
    if turbo:
        out = _rotate(out, inverse=True)
    return {"out": out * gate, "qo": qo, "k": None, "v": None, "ks": ks, "vs": vs}
