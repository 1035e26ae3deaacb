"""The work that a program has this library do, as cases that can be timed.

Kinds (a case's "kind"), each through the package's public calls:

  linear       quantise one activation vector and multiply a packed matrix with it (the decode
               projections and the head): quant.quantize_act + quant.matvec_packed
  rows         the same with the matrix in the reference's row layout (the drop-in call for weights
               that were not packed): quant.quantize_act + quant.matvec_rows
  tokens       quantise T vectors and multiply a packed matrix with all of them (a prompt's
               projections): quant.quantize_act + quant.matmul_tokens
  moe          one routed MoE block for one token, every expert resident: MoeBlock.__call__
  moe_prefill  the same block for T tokens of a prompt: MoeBlock.prefill
  decode       a whole model of few layers: eight greedy tokens from a context of `context`
               positions, the last one's logits on the host: Model.decode + Model.step
  prefill      the same kind of model given a prompt of `tokens` tokens behind a context of
               `context` positions, the last one's logits on the host: Model.prefill

Geometries: "c1" is the small synthetic model (4 layers, hidden 512, 32 experts top-4 and a shared
expert), "30b" a layer of Qwen3-30B-A3B, "235b" a layer of Qwen3-235B-A22B.  Block formats are the
library's (Q8_0 dense weights; Q4_K, Q5_K and Q6_K experts).  The library promises the same bits
for every order of its work (one exact integer sum per block, then one chain per row), so every
tolerance is "exact"."""
import math

import torch

from tierlm_amd import MoeBlock
from tierlm_amd import quant as hq
from tierlm_amd.model import QWEN3_30B_A3B, QWEN3_235B_A22B, Model

DT = {"q8_0": hq.Q8_0, "q4_k": hq.Q4_K, "q5_k": hq.Q5_K, "q6_k": hq.Q6_K}
C1 = dict(n_layers=4, d_model=512, n_heads=8, n_kv_heads=2, head_dim=64, vocab=4096, n_experts=32, top_k=4,
          d_expert=256, n_shared=1, d_shared=256, max_ctx=40960, router=0, rope_theta=1e6, norm_eps=1e-6,
          routed_scale=1.0)
GEOM = {"c1": C1, "30b": QWEN3_30B_A3B, "235b": QWEN3_235B_A22B}
STEPS = 8          # tokens of a decode pass
_ready = []


def listed():
    return [
        # the smallest projection of the small model: two launches and nothing to hide them behind
        {"name": "linear_q8_0_512x512", "kind": "linear", "dt": "q8_0", "rows": 512, "n": 512},
        # the head of a 151936-word model: the largest matrix that a decode step reads
        {"name": "linear_q8_0_head", "kind": "linear", "dt": "q8_0", "rows": 151936, "n": 2048},
        # the reference's own kernel figure (4096 x 4096 Q6_K), weights as they lie in a store
        {"name": "rows_q6_k_4096x4096", "kind": "rows", "dt": "q6_k", "rows": 4096, "n": 4096},
        # a full prompt chunk through the query projection
        {"name": "tokens_q8_0_1024", "kind": "tokens", "dt": "q8_0", "rows": 4096, "n": 2048, "tokens": 1024},
        # the routed block at batch 1, both model sizes: most of a decode step's bytes
        {"name": "moe_q6_k_30b", "kind": "moe", "geom": "30b", "dt": "q6_k"},
        {"name": "moe_q4_k_235b", "kind": "moe", "geom": "235b", "dt": "q4_k"},
        # the routed block for a prompt: a full chunk, and a short one that leaves most tiles part empty
        {"name": "moe_prefill_q6_k_30b_512", "kind": "moe_prefill", "geom": "30b", "dt": "q6_k", "tokens": 512},
        {"name": "moe_prefill_q4_k_235b_77", "kind": "moe_prefill", "geom": "235b", "dt": "q4_k", "tokens": 77},
        # greedy decoding: the small model (latency alone) and a large one late in its context
        {"name": "decode_c1_64", "kind": "decode", "geom": "c1", "dt": "q6_k", "layers": 4, "context": 64, "cache": 0},
        {"name": "decode_30b_2000", "kind": "decode", "geom": "30b", "dt": "q6_k", "layers": 4, "context": 2000,
         "cache": 0},
        # experts behind the slot cache, as a model larger than the card's share is served
        {"name": "decode_235b_cached_300", "kind": "decode", "geom": "235b", "dt": "q4_k", "layers": 2,
         "context": 300, "cache": 1},
        # a long prompt
        {"name": "prefill_30b_2047", "kind": "prefill", "geom": "30b", "dt": "q6_k", "layers": 4, "tokens": 2047,
         "context": 0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "rows", "tokens", "tokens", "moe", "moe_prefill", "moe_prefill", "decode",
                       "decode", "prefill", "prefill"])
    if kind in ("linear", "rows", "tokens"):
        dt = rng.choice(["q8_0", "q8_0", "q4_k", "q5_k", "q6_k"])
        step = 32 if dt == "q8_0" and kind != "tokens" else 256
        n = step * max(1, _log(rng, 256, 8192) // step)
        rows = _log(rng, 200, 40000 if kind == "linear" else 10000)
        c = {"kind": kind, "dt": dt, "rows": rows, "n": n}
        if kind == "tokens":
            c["tokens"] = _log(rng, 2, 1024)
        return c
    dt = rng.choice(["q4_k", "q5_k", "q6_k"])
    geom = rng.choice(["c1", "30b", "30b", "235b"])
    if kind == "moe":
        return {"kind": kind, "geom": geom, "dt": dt}
    if kind == "moe_prefill":
        return {"kind": kind, "geom": geom, "dt": dt, "tokens": _log(rng, 2, 512 if geom == "235b" else 1024)}
    layers = {"c1": 4, "30b": 2, "235b": 1}[geom]
    if kind == "decode":
        return {"kind": kind, "geom": geom, "dt": dt, "layers": layers, "context": _log(rng, 16, 8000),
                "cache": rng.choice([0, 0, 1])}
    return {"kind": kind, "geom": geom, "dt": dt, "layers": layers, "tokens": _log(rng, 5, 2047),
            "context": rng.choice([0, 0, _log(rng, 16, 2000)])}


# ---- inputs ------------------------------------------------------------------------------------

class _Rand:
    """Tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed * 7919 + 17)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32)

    def rows(self, dt, rows, n):
        """Block rows as a store holds them: uniform codes, scales that give weights of about 0.02."""
        bv, bb = hq.BLOCK[dt]
        nb = n // bv
        w = torch.randint(0, 256, (rows, nb, bb), generator=self.g, device="cuda", dtype=torch.uint8)
        fields = {hq.Q8_0: [(0, 2.7e-4, 1)], hq.Q6_K: [(208, 1.5e-5, 1)], hq.Q4_K: [(0, 7e-5, 0), (2, 5e-4, 0)],
                  hq.Q5_K: [(0, 3.5e-5, 0), (2, 5e-4, 0)]}[dt]
        for off, s, signed in fields:
            v = self.normal(rows, nb) * s
            v = (v if signed else v.abs()).to(torch.float16)
            w[:, :, off:off + 2] = v.view(torch.uint8).reshape(rows, nb, 2)
        return w.reshape(rows, nb * bb)


def _pack(dt, w, n):
    return hq.pack(dt, w.reshape(-1), w.shape[1], w.shape[0], n)


class _Matrix:
    pass


def _matrix(case, seed):
    dt, r = DT[case["dt"]], _Rand(seed)
    m = _Matrix()
    m.dt, m.kind, m.n, m.nrows, m.T = dt, hq.act_kind_for(dt), case["n"], case["rows"], case.get("tokens", 0)
    m.rows = r.rows(dt, m.nrows, m.n)
    m.x = r.normal(max(m.T, 1), m.n).reshape(-1)
    return m


class _Moe:
    pass


def _moe(case, seed, packed=True):
    g, dt, r = GEOM[case["geom"]], DT[case["dt"]], _Rand(seed)
    D, de, E, k = g["d_model"], g["d_expert"], g["n_experts"], g["top_k"]
    m = _Moe()
    m.D, m.de, m.E, m.k, m.dt, m.eps = D, de, E, k, dt, g["norm_eps"]
    m.norm = 1.0 + 0.1 * r.normal(D)
    m.router = r.normal(E, D) / math.sqrt(D)
    m.ds = g["d_shared"] if g["n_shared"] else 0
    m.T = case.get("tokens", 1)
    m.h0 = r.normal(m.T, D)
    m.shared = [r.rows(hq.Q8_0, *s) for s in ((m.ds, D), (m.ds, D), (D, m.ds))] if m.ds else None
    m.experts = []
    for _ in range(E):
        e = [r.rows(dt, de, D), r.rows(dt, de, D), r.rows(dt, D, de)]
        m.experts.append([_pack(dt, w, n) for w, n in zip(e, (D, D, de))] if packed else e)
    if packed:
        if m.ds:
            m.shared = tuple(_pack(hq.Q8_0, w, n) for w, n in zip(m.shared, (D, D, m.ds)))
        m.block = MoeBlock(D=D, de=de, E=E, k=k, expert_dt=dt, ffn_norm=m.norm, router_w=m.router,
                           expert_ptrs=[p.data_ptr() for e in m.experts for p in e], eps=m.eps, ds=m.ds,
                           shared_dt=hq.Q8_0, shared=m.shared)
        m.h = torch.empty_like(m.h0)
        m.ids = torch.zeros(m.T, k, dtype=torch.int32, device="cuda")
        m.w = torch.zeros(m.T, k, dtype=torch.float32, device="cuda")
    return m


class _Run:
    pass


def _model(case, seed):
    g = dict(GEOM[case["geom"]], n_layers=case["layers"])
    ctx, T = case["context"], case.get("tokens", 0)
    more = {}
    if case.get("cache"):       # every expert fits; a pool of payloads stands for the host copy
        bv, bb = hq.BLOCK[DT[case["dt"]]]
        per = 3 * g["d_model"] * g["d_expert"] // bv * bb
        more = dict(expert_cache=int((g["n_layers"] * g["n_experts"] + 1) * per * 1.01), expert_pool=16)
    s = _Run()
    s.m = Model.synth(g, expert_dt=DT[case["dt"]], seed=seed + 1, max_ctx=ctx + max(T, STEPS) + 8, **more)
    r = torch.Generator()
    r.manual_seed(seed * 7919 + 17)
    tok = torch.randint(0, g["vocab"], (ctx + max(T, 2),), generator=r).tolist()
    if ctx:
        s.m.prefill(tok[:ctx], logits=False)
    s.ctx, s.prompt, s.tok = ctx, tok[ctx:], tok[ctx + 1]
    if case["kind"] == "decode":   # the first step's token lies at the context's end
        s.m.step(tok[ctx], logits=False)
    return s


def prepare(case, seed):
    if not _ready:
        hq.init(0)
        _ready.append(True)
    kind = case["kind"]
    if kind in ("linear", "rows", "tokens"):
        m = _matrix(case, seed)
        m.case_kind, m.rb = kind, m.rows.shape[1]
        if kind != "rows":
            m.W = _pack(m.dt, m.rows, m.n)
            m.rows = None
        m.act = torch.empty(hq.qact_bytes(m.kind, m.x.numel()), dtype=torch.uint8, device="cuda")
        m.y = torch.empty((m.T, m.nrows) if kind == "tokens" else m.nrows, dtype=torch.float32, device="cuda")
        return m
    m = _moe(case, seed) if kind in ("moe", "moe_prefill") else _model(case, seed)
    m.case_kind = kind
    return m


def run(s):
    kind = s.case_kind
    if kind == "linear":
        hq.quantize_act(s.kind, s.x, s.act)
        return hq.matvec_packed(s.dt, s.W, s.nrows, s.n, s.act, s.y)
    if kind == "rows":
        hq.quantize_act(s.kind, s.x, s.act)
        return hq.matvec_rows(s.dt, s.rows, s.rb, s.act, s.n, 0, s.nrows, s.y)
    if kind == "tokens":
        hq.quantize_act(s.kind, s.x, s.act)
        return hq.matmul_tokens(s.dt, s.W, s.nrows, s.n, s.act, s.T, s.y)
    if kind == "moe":
        s.h.copy_(s.h0)
        s.block(s.h)
        return s.h, s.block.ids, s.block.w
    if kind == "moe_prefill":
        s.h.copy_(s.h0)
        s.block.prefill(s.h, s.ids, s.w)
        return s.h, s.ids, s.w
    if kind == "decode":
        s.m.rewind(s.ctx)
        s.m.decode(STEPS - 1)
        logits, nxt = s.m.step(s.tok)
        return logits, nxt
    s.m.rewind(s.ctx)
    return s.m.prefill(s.prompt)


# ---- what a pass cannot do without ---------------------------------------------------------------

def _mat_bytes(dt, rows, n):
    bv, bb = hq.BLOCK[dt]
    return rows * (n // bv) * bb


def _moe_work(g, dt, T):
    """Routed block for T tokens: every selected expert's matrices once (all of them for a long
    prompt: the expected number of distinct experts), the router, h in and out."""
    D, de, E, k, ds = g["d_model"], g["d_expert"], g["n_experts"], g["top_k"], g["d_shared"] if g["n_shared"] else 0
    used = k if T == 1 else E * (1.0 - (1.0 - k / E) ** T)
    b = used * 3 * _mat_bytes(dt, de, D) + 4 * E * D + 4 * D + 8 * T * D + 8 * T * k
    f = T * (6.0 * k * de * D + 2.0 * E * D + 6.0 * ds * D)
    return b + (3 * _mat_bytes(hq.Q8_0, ds, D) if ds else 0), f


def _model_work(case, T, ctx):
    """T tokens behind ctx positions in one pass over the weights; the logits of the last."""
    g = GEOM[case["geom"]]
    D, hd, H, KV, V = g["d_model"], g["head_dim"], g["n_heads"], g["n_kv_heads"], g["vocab"]
    mb, mf = _moe_work(g, DT[case["dt"]], T)
    pairs = T * ctx + T * (T + 1) / 2.0
    b = mb + _mat_bytes(hq.Q8_0, H * hd + 2 * KV * hd, D) + _mat_bytes(hq.Q8_0, D, H * hd)
    b += 8 * KV * hd * (ctx + T) + 8 * KV * hd * T
    f = mf + T * 4.0 * D * hd * (H + KV) + 4.0 * pairs * H * hd
    return case["layers"] * b + _mat_bytes(hq.Q8_0, V, D) + 4 * V, case["layers"] * f + 2.0 * V * D


def work(case):
    kind = case["kind"]
    if kind in ("linear", "rows", "tokens"):
        T = case.get("tokens", 1)
        return {"bytes": _mat_bytes(DT[case["dt"]], case["rows"], case["n"]) + 4 * T * (case["n"] + case["rows"]),
                "flops": 2.0 * T * case["rows"] * case["n"]}
    if kind in ("moe", "moe_prefill"):
        b, f = _moe_work(GEOM[case["geom"]], DT[case["dt"]], case.get("tokens", 1))
    elif kind == "decode":
        one = [_model_work(case, 1, case["context"] + i) for i in range(STEPS)]
        b, f = sum(x[0] for x in one), sum(x[1] for x in one)
    else:
        b, f = _model_work(case, case["tokens"], case["context"])
    return {"bytes": b, "flops": f}


def tolerance(case):
    return "exact"


# ---- the same results in 64 bits ------------------------------------------------------------------

def _unpack(dt, w, n):
    """Block rows -> float64 weights."""
    bv, bb = hq.BLOCK[dt]
    w = w.reshape(w.shape[0], n // bv, bb)

    def f16(off):
        return w[:, :, off:off + 2].contiguous().view(torch.float16).to(torch.float64)

    if dt == hq.Q8_0:
        q = w[:, :, 2:].contiguous().view(torch.int8).to(torch.float64)
        return (q * f16(0)).reshape(w.shape[0], n)
    i = w.to(torch.int32)
    if dt == hq.Q6_K:
        parts = []
        for h in range(2):
            ql, qh = i[:, :, 64 * h:64 * h + 64], i[:, :, 128 + 32 * h:160 + 32 * h]
            for q in range(4):
                nib = (ql[:, :, 32 * (q & 1):32 * (q & 1) + 32] >> (4 * (q >> 1))) & 15
                parts.append((nib | (((qh >> (2 * q)) & 3) << 4)) - 32)
        code = torch.cat(parts, 2).reshape(w.shape[0], n // bv, 16, 16).to(torch.float64)
        sc = w[:, :, 192:208].contiguous().view(torch.int8).to(torch.float64)
        return (code * sc[..., None] * f16(208)[..., None]).reshape(w.shape[0], n)
    s, qs = i[:, :, 4:16], i[:, :, 48 if dt == hq.Q5_K else 16:]
    lo, mi, hi = s[:, :, 0:4], s[:, :, 4:8], s[:, :, 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 2).to(torch.float64)
    mn = torch.cat([mi & 63, (hi >> 4) | ((mi >> 6) << 4)], 2).to(torch.float64)
    parts = []
    for b in range(8):
        c = (qs[:, :, 32 * (b >> 1):32 * (b >> 1) + 32] >> (4 * (b & 1))) & 15
        if dt == hq.Q5_K:
            c = c | (((i[:, :, 16:48] >> b) & 1) << 4)
        parts.append(c)
    code = torch.stack(parts, 2).to(torch.float64)
    v = code * (sc * f16(0))[..., None] - (mn * f16(2))[..., None]
    return v.reshape(w.shape[0], n)


def _act(kind, x):
    """What the activation quantiser keeps of x (rows of float32), as float64: codes of
    round(x 127 / amax) per block of 256 (Q8_K) or 32 values, times amax / 127."""
    bv = 256 if kind == hq.Q8_K else 32
    b = x.to(torch.float32).reshape(x.shape[0], -1, bv)
    amax = b.abs().amax(2, keepdim=True)
    some = torch.where(amax > 0, amax, torch.ones_like(amax))
    hundred = torch.full_like(amax, 127.0)
    code = torch.clamp(torch.round(b * (hundred / some)), -127, 127) * (amax > 0)
    return (code.to(torch.float64) * (amax / hundred).to(torch.float64)).reshape(x.shape)


def _ffn(mats, dt, x):
    """down(quantised silu(gate x) * (up x)) for quantised rows x, in float64."""
    kind, D = hq.act_kind_for(dt), x.shape[1]
    g, u = x @ _unpack(dt, mats[0], D).T, x @ _unpack(dt, mats[1], D).T
    h = _act(kind, (g * torch.sigmoid(g) * u).to(torch.float32))
    return h @ _unpack(dt, mats[2], h.shape[1]).T


def exact(case, seed):
    kind = case["kind"]
    if kind in ("linear", "rows", "tokens"):
        m = _matrix(case, seed)
        x = _act(m.kind, m.x.reshape(max(m.T, 1), m.n))
        y = torch.cat([x @ _unpack(m.dt, m.rows[i:i + 8192], m.n).T for i in range(0, m.nrows, 8192)], 1)
        return y if kind == "tokens" else y[0]
    if kind not in ("moe", "moe_prefill"):
        return None
    m = _moe(case, seed, packed=False)
    h = m.h0.to(torch.float64)
    xb = h / torch.sqrt((h * h).mean(1, keepdim=True) + m.eps) * m.norm.to(torch.float64)
    p = torch.softmax(xb @ m.router.to(torch.float64).T, 1)
    w, ids = torch.topk(p, m.k, 1)
    w = w / w.sum(1, keepdim=True)
    out = h.clone()
    x = _act(hq.act_kind_for(m.dt), xb.to(torch.float32))
    for e in torch.unique(ids).tolist():
        t, r = (ids == e).nonzero(as_tuple=True)
        out.index_add_(0, t, w[t, r][:, None] * _ffn(m.experts[e], m.dt, x[t]))
    if m.ds:
        out += _ffn(m.shared, hq.Q8_0, _act(hq.Q8_0, xb.to(torch.float32)))
    ids = ids.to(torch.int32)
    return (out[0:1], ids[0], w[0]) if kind == "moe" else (out, ids, w)
