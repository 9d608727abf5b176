"""Workloads of the Qwen3 attention path: what a program that uses this library has it do.

Four kinds, each through the public entry points:

  decode   one new token: the fused step (QK-norm + RoPE, cache append, split-K attention) over
           every layer's own KV cache, called layer by layer or replayed as one HIP graph
  batch    one new token for each of several sequences of different lengths, from one pool
           (contiguous ranges, or blocks of a paged pool)
  prefill  one prompt chunk of one layer: key norm + RoPE + append, then causal attention over the
           chunk and the cached keys before it (contiguous cache or paged pool)
  project  attention RMSNorm + the fused [Wq | Wk | Wv] product of a decode step, over every
           layer's own weights (F32, F16, or Q8_0 / Q4_K / Q6_K blocks)

Inputs follow the benchmark's configurations: Q/K/V ~ N(0,1), gammas 1 + 0.1 N(0,1), RoPE theta
1e6, softmax scale 1/sqrt(128).
"""
from __future__ import annotations

import math

import torch

from exactinfer_amd import _capi
from exactinfer_amd import attention as A

D = 128
EPS = 1e-6
THETA = 1e6
SCALE = 1.0 / math.sqrt(D)

W_TYPES = {"f32": 0, "f16": 1, "q8_0": 8, "q4_k": 12, "q6_k": 14}
BLOCKS = {"q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}  # values, bytes


def listed():
    return [
        # the smallest call: one layer of a small model early in a conversation, planned for a long one
        dict(name="decode_short", kind="decode", heads=16, kv_heads=8, layers=1, ctx=300, max_kv=4096, spike=0,
             graph=False),
        # one token of a 4B-shaped model at context 4096, the layers in one HIP graph (the headline workload)
        dict(name="decode_token_graph", kind="decode", heads=32, kv_heads=8, layers=36, ctx=4096, max_kv=4096,
             spike=0, graph=True),
        # one token of a 0.6B-shaped model at an odd length, layer after layer without a graph
        dict(name="decode_token_eager", kind="decode", heads=16, kv_heads=8, layers=28, ctx=1733, max_kv=2048,
             spike=0, graph=False),
        # long context with sharp softmax peaks (every 512th key scaled by 4)
        dict(name="decode_long", kind="decode", heads=16, kv_heads=8, layers=4, ctx=32768, max_kv=32768, spike=512,
             graph=False),
        # a serving batch of ragged sequences in a paged pool
        dict(name="batch_paged", kind="batch", heads=16, kv_heads=8, n_seq=64, min_len=256, max_len=8192, block=64),
        # a handful of sequences, five query heads to a KV head, contiguous ranges
        dict(name="batch_small", kind="batch", heads=40, kv_heads=8, n_seq=5, min_len=100, max_len=3000, block=0),
        # a whole 2048-token prompt of a 4B-shaped layer
        dict(name="prefill_2048", kind="prefill", heads=32, kv_heads=8, rows=2048, pos0=0, block=0),
        # a 512-token chunk late in a prompt of a 0.6B-shaped layer
        dict(name="prefill_chunk", kind="prefill", heads=16, kv_heads=8, rows=512, pos0=7680, block=0),
        # a ragged tail of a prompt after a cached prefix, paged, five query heads to a KV head
        dict(name="prefill_paged_tail", kind="prefill", heads=40, kv_heads=8, rows=300, pos0=777, block=64),
        # the largest: an 8192-token prompt in one call
        dict(name="prefill_8192", kind="prefill", heads=32, kv_heads=8, rows=8192, pos0=0, block=0),
        # the projection of one token, 4-bit blocks, every layer of a 4B-shaped model
        dict(name="project_q4_k", kind="project", n_embd=2560, n_out=6144, rows=1, layers=36, weights="q4_k"),
        # the projection of four sequences' tokens, binary16 weights
        dict(name="project_f16_rows4", kind="project", n_embd=4096, n_out=6144, rows=4, layers=12, weights="f16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "batch", "prefill", "prefill", "project"])
    heads, kv_heads = rng.choice([(16, 8), (16, 8), (32, 8), (32, 8), (40, 8), (64, 8), (8, 8)])
    if kind == "decode":
        ctx = _log_int(rng, 100, 32768)
        layers = max(1, min(rng.choice([1, 4, 28, 36]), 150000 // ctx))
        max_kv = min(32768, ctx + rng.randrange(1, 2000))
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, layers=layers, ctx=ctx, max_kv=max_kv,
                    spike=rng.choice([0, 0, 512]), graph=rng.random() < 0.5)
    if kind == "batch":
        max_len = _log_int(rng, 300, 8192)
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, n_seq=_log_int(rng, 2, 64),
                    min_len=rng.randrange(64, 257), max_len=max_len, block=rng.choice([0, 32, 64, 128]))
    if kind == "prefill":
        rows = _log_int(rng, 16, 4096)
        pos0 = rng.choice([0, rng.randrange(1, 512), _log_int(rng, 64, 16384)])
        most = 32 * 8192 * 8192 // 2 // heads  # query-key pairs per head of the largest listed case
        pos0 = max(0, min(pos0, most // rows - rows))
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, rows=rows, pos0=pos0, block=rng.choice([0, 0, 0, 64]))
    n_embd, n_out = rng.choice([(1024, 4096), (2048, 4096), (2560, 6144), (4096, 6144), (5120, 7168)])
    return dict(kind=kind, n_embd=n_embd, n_out=n_out, rows=rng.choice([1, 1, 2, 3, 4]), layers=rng.choice([1, 4, 12]),
                weights=rng.choice(["f32", "f16", "q8_0", "q4_k", "q6_k"]))


# ------------------------------------------------------------------------------ inputs
class _Rng:
    """Normal and integer tensors on the GPU, from the seed alone."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)

    def gamma(self, n):
        return 1.0 + 0.1 * self.normal(n)

    def ints(self, lo, hi, *shape, dtype=torch.int32):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=dtype)


_tables = {}


def _rope_table(n):
    """The RoPE table a program builds once for its longest context (n rounded up, at least 4096)."""
    n = max(4096, 1 << (n - 1).bit_length())
    if n not in _tables:
        _tables[n] = A.rope_table(n, D, THETA)
    return _tables[n]


def _decode_inputs(c, seed):
    r = _Rng(seed)
    kd = (c["kv_heads"], D)
    k = r.normal(c["layers"], c["max_kv"], *kd)
    if c["spike"]:
        k[:, ::c["spike"]] *= 4.0
    v = r.normal(c["layers"], c["max_kv"], *kd)
    qkv = r.normal(c["layers"], 1, (c["heads"] + 2 * c["kv_heads"]) * D)
    return k, v, qkv, r.gamma(D), r.gamma(D)


def _batch_inputs(c, seed):
    r = _Rng(seed)
    lens = r.ints(min(c["min_len"], c["max_len"]), c["max_len"] + 1, c["n_seq"])
    if c["block"]:
        bs = c["block"]
        max_blocks = (c["max_len"] + bs - 1) // bs
        perm = torch.randperm(c["n_seq"] * max_blocks, generator=r.g, device="cuda")
        table = perm.view(c["n_seq"], max_blocks).to(torch.int32).contiguous()
        rows, where = c["n_seq"] * max_blocks * bs, table
    else:
        where = torch.cumsum(lens.to(torch.int64), 0) - lens  # first row of each sequence
        rows = c["n_seq"] * c["max_len"]
    k, v = r.normal(rows, c["kv_heads"], D), r.normal(rows, c["kv_heads"], D)
    qkv = r.normal(c["n_seq"], (c["heads"] + 2 * c["kv_heads"]) * D)
    return lens, where, k, v, qkv, r.gamma(D), r.gamma(D)


def _prefill_inputs(c, seed):
    r = _Rng(seed)
    n = c["pos0"] + c["rows"]
    if c["block"]:
        blocks = (n + c["block"] - 1) // c["block"]
        table = torch.randperm(blocks, generator=r.g, device="cuda").to(torch.int32)
        n = blocks * c["block"]
    else:
        table = None
    k, v = r.normal(n, c["kv_heads"], D), r.normal(n, c["kv_heads"], D)
    qkv = r.normal(c["rows"], (c["heads"] + 2 * c["kv_heads"]) * D)
    return table, k, v, qkv, r.gamma(D), r.gamma(D)


def _f16_bytes(x):
    return x.to(torch.float16).view(torch.uint8).view(*x.shape, 2)


def _project_inputs(c, seed):
    r = _Rng(seed)
    E, N, L = c["n_embd"], c["n_out"], c["layers"]
    x = 3.0 * r.normal(L, c["rows"], E)
    gamma = 1.0 + 0.1 * r.normal(L, E)
    t = c["weights"]
    if t == "f32":
        w = 0.05 * r.normal(L, N, E)
    elif t == "f16":
        w = (0.05 * r.normal(L, N, E)).to(torch.float16)
    else:
        vals, nbytes = BLOCKS[t]
        nb = E // vals
        w = r.ints(0, 256, L, N, nb, nbytes, dtype=torch.uint8)
        scale = 1.0 + 0.5 * torch.rand((L, N, nb, 2), generator=r.g, device="cuda")
        if t == "q8_0":  # d, 32 int8
            w[..., 0:2] = _f16_bytes(scale[..., 0] * 7e-4)
        elif t == "q4_k":  # d, dmin, 12 bytes of 6-bit scales and minima, 128 bytes of nibbles
            w[..., 0:2] = _f16_bytes(scale[..., 0] * 2e-4)
            w[..., 2:4] = _f16_bytes(scale[..., 1] * 1.5e-3)
        else:  # 128 low nibbles, 64 high bit pairs, 16 int8 scales, d
            w[..., 208:210] = _f16_bytes(scale[..., 0] * 4e-5)
        w = w.view(L, N, nb * nbytes)
    return x, gamma, w


def prepare(case, seed):
    c = case
    if c["kind"] == "project":
        x, gamma, w = _project_inputs(c, seed)
        out = torch.empty((c["layers"], c["rows"], c["n_out"]), dtype=torch.float32, device="cuda")
        return dict(c=c, x=x, gamma=gamma, w=w, out=out)
    shape = A.AttnShape(c["heads"], c["kv_heads"])
    s = dict(c=c, shape=shape)
    if c["kind"] == "decode":
        k, v, qkv, qg, kg = _decode_inputs(c, seed)
        ws = A.DecodeWorkspace(1, c["heads"], c["kv_heads"], c["max_kv"])
        s.update(k=k, v=v, qkv=qkv, qg=qg, kg=kg, ws=ws, cs=_rope_table(c["max_kv"]))
        s["pos"] = torch.tensor([c["ctx"] - 1], dtype=torch.int32, device="cuda")
        if c["graph"]:
            torch.cuda.synchronize()
            _decode_token(s)  # first launches outside the capture
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                s["outs"] = _decode_token(s)
            s["graph"] = graph
    elif c["kind"] == "batch":
        lens, where, k, v, qkv, qg, kg = _batch_inputs(c, seed)
        ws = A.DecodeWorkspace(c["n_seq"], c["heads"], c["kv_heads"], c["max_len"])
        s.update(lens=lens, where=where, k=k, v=v, qkv=qkv, qg=qg, kg=kg, ws=ws, cs=_rope_table(c["max_len"]))
    else:
        table, k, v, qkv, qg, kg = _prefill_inputs(c, seed)
        n = c["pos0"] + c["rows"]
        ws = A.PrefillWorkspace(c["rows"], c["heads"], c["kv_heads"], n)
        hd, kd = c["heads"] * D, c["kv_heads"] * D
        s.update(table=table, k=k, v=v, qkv=qkv, qg=qg, kg=kg, ws=ws, cs=_rope_table(n))
        s["k_cols"], s["raw_k"] = qkv[:, hd:hd + kd], qkv[:, hd:hd + kd].clone()
        s["pos"] = torch.tensor([c["pos0"]], dtype=torch.int32, device="cuda")
    return s


# ------------------------------------------------------------------------------ one pass
def _decode_token(s):
    return [A.decode_step(s["qkv"][i], s["k"][i], s["v"][i], s["shape"], s["qg"], s["kg"], s["cs"], s["ws"],
                          pos_dev=s["pos"]) for i in range(s["c"]["layers"])]


def run(s):
    c = s["c"]
    if c["kind"] == "decode":
        if c["graph"]:
            s["graph"].replay()
            outs = s["outs"]
        else:
            outs = _decode_token(s)
        return {"out": outs, "k": s["k"], "v": s["v"]}
    if c["kind"] == "batch":
        if c["block"]:
            out = A.decode_step_paged(s["qkv"], s["k"], s["v"], s["where"], c["block"], s["lens"], s["shape"], s["qg"],
                                      s["kg"], s["cs"], s["ws"])
        else:
            out = A.decode_step(s["qkv"], s["k"], s["v"], s["shape"], s["qg"], s["kg"], s["cs"], s["ws"],
                                kv_offset=s["where"], kv_len=s["lens"])
        return {"out": out, "k": s["k"], "v": s["v"]}
    if c["kind"] == "prefill":
        # the step norms the chunk's keys in place: the projection writes them afresh for each chunk
        s["k_cols"].copy_(s["raw_k"])
        out = A.prefill_step(s["qkv"], s["k"], s["v"], s["shape"], s["qg"], s["kg"], s["cs"], s["pos"], s["ws"],
                             block_table=s["table"], block_size=c["block"])
        return {"out": out, "k": s["k"], "v": s["v"]}
    x, gamma, w, out = s["x"], s["gamma"], s["w"], s["out"]
    stream = torch.cuda.current_stream().cuda_stream
    E, N, rows = c["n_embd"], c["n_out"], c["rows"]
    for i in range(c["layers"]):
        _capi.call("ei_qkv_project", stream, x[i].data_ptr(), E, rows, E, gamma[i].data_ptr(), EPS, w[i].data_ptr(),
                   W_TYPES[c["weights"]], N, out[i].data_ptr(), N)
    return {"out": out}


# ------------------------------------------------------------------------------ what a pass cannot do without
def work(case):
    c = case
    if c["kind"] == "project":
        vals, nbytes = BLOCKS.get(c["weights"], (1, 4 if c["weights"] == "f32" else 2))
        w = c["n_out"] * c["n_embd"] // vals * nbytes
        rows = c["rows"] * (c["n_embd"] + c["n_out"]) * 4 + c["n_embd"] * 4
        return {"bytes": c["layers"] * (w + rows), "flops": 2 * c["layers"] * c["rows"] * c["n_out"] * c["n_embd"]}
    H, HKV = c["heads"], c["kv_heads"]
    row = (2 * H + 2 * HKV) * D * 4  # a token's Q, K, V read and its output written
    if c["kind"] == "decode":
        return {"bytes": c["layers"] * (2 * c["ctx"] * HKV * D * 4 + row), "flops": c["layers"] * 4 * D * H * c["ctx"]}
    if c["kind"] == "batch":
        keys = c["n_seq"] * (min(c["min_len"], c["max_len"]) + c["max_len"]) // 2  # the mean over the seeds
        return {"bytes": 2 * keys * HKV * D * 4 + c["n_seq"] * row, "flops": 4 * D * H * keys}
    B, p = c["rows"], c["pos0"]
    return {"bytes": 2 * (p + 2 * B) * HKV * D * 4 + 2 * B * H * D * 4, "flops": 4 * D * H * (B * p + B * (B + 1) // 2)}


def tolerance(case):
    # four times the largest distance from the 64-bit result measured over the listed cases: 7e-7 for
    # attention (32-bit sums over up to 32768 keys), 1.8e-7 for the projection
    return {"rel": 7.2e-7} if case["kind"] == "project" else {"rel": 2.8e-6}


# ------------------------------------------------------------------------------ in 64 bits
def _norm_rope(x, gamma, pos):
    """RMS norm and rotate-half RoPE of x [..., rows, heads, 128] at positions pos [rows]."""
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()
    inv = THETA ** (-2.0 * torch.arange(D // 2, device=x.device, dtype=torch.float64) / D)
    th = pos.double()[:, None, None] * inv
    co, si = torch.cos(th), torch.sin(th)
    a, b = y[..., :D // 2], y[..., D // 2:]
    return torch.cat([a * co - b * si, a * si + b * co], -1)


def _split(qkv, H, HKV):
    rows = qkv.double().view(qkv.shape[0], H + 2 * HKV, D)
    return rows[:, :H], rows[:, H:H + HKV], rows[:, H + HKV:]


def _attend_one(q, k, v):
    """q [H, 128] over keys k, v [T, HKV, 128]."""
    g = q.shape[0] // k.shape[1]
    out = torch.empty_like(q)
    for h in range(k.shape[1]):
        s = torch.matmul(q[h * g:(h + 1) * g], k[:, h].double().t()) * SCALE
        out[h * g:(h + 1) * g] = torch.matmul(torch.softmax(s, -1), v[:, h].double())
    return out


def exact(case, seed):
    c = case
    if c["kind"] == "project":
        x, gamma, w = _project_inputs(c, seed)
        outs = []
        for i in range(c["layers"]):
            xd = x[i].double()
            h = xd * torch.rsqrt((xd * xd).mean(-1, keepdim=True) + EPS) * gamma[i].double()
            wd = w[i].double() if c["weights"] in ("f32", "f16") else _decode_blocks(w[i], c["weights"], c["n_embd"])
            outs.append(torch.matmul(h, wd.t()))
        return {"out": torch.stack(outs)}
    H, HKV = c["heads"], c["kv_heads"]
    if c["kind"] == "decode":
        k, v, qkv, qg, kg = _decode_inputs(c, seed)
        pos = torch.tensor([c["ctx"] - 1], device="cuda")
        outs, k64, v64 = [], k.double(), v.double()
        for i in range(c["layers"]):
            q, kn, vn = _split(qkv[i], H, HKV)
            k64[i, c["ctx"] - 1], v64[i, c["ctx"] - 1] = _norm_rope(kn, kg, pos)[0], vn[0]
            q = _norm_rope(q, qg, pos)[0]
            outs.append(_attend_one(q, k64[i, :c["ctx"]], v64[i, :c["ctx"]])[None])
        return {"out": outs, "k": k64, "v": v64}
    if c["kind"] == "batch":
        lens, where, k, v, qkv, qg, kg = _batch_inputs(c, seed)
        q, kn, vn = _split(qkv, H, HKV)
        pos = lens.long() - 1
        q, kn = _norm_rope(q, qg, pos), _norm_rope(kn, kg, pos)
        k64, v64, outs = k.double(), v.double(), []
        for i, n in enumerate(lens.tolist()):
            t = torch.arange(n, device="cuda")
            rows = where[i].long()[t // c["block"]] * c["block"] + t % c["block"] if c["block"] else where[i] + t
            k64[rows[-1]], v64[rows[-1]] = kn[i], vn[i]
            outs.append(_attend_one(q[i], k64[rows], v64[rows]))
        return {"out": torch.stack(outs), "k": k64, "v": v64}
    table, k, v, qkv, qg, kg = _prefill_inputs(c, seed)
    B, p = c["rows"], c["pos0"]
    q, kn, vn = _split(qkv, H, HKV)
    pos = p + torch.arange(B, device="cuda")
    q, kn = _norm_rope(q, qg, pos), _norm_rope(kn, kg, pos)
    t = torch.arange(p + B, device="cuda")
    rows = table.long()[t // c["block"]] * c["block"] + t % c["block"] if c["block"] else t
    k64, v64 = k.double(), v.double()
    k64[rows[p:]], v64[rows[p:]] = kn, vn
    out = torch.empty((B, H, D), dtype=torch.float64, device="cuda")
    g = H // HKV
    for h in range(H):
        kh, vh = k64[rows, h // g], v64[rows, h // g]
        for b in range(0, B, 2048):
            n = min(B, b + 2048)
            T = p + n
            s = torch.matmul(q[b:n, h], kh[:T].t()) * SCALE
            s.masked_fill_(t[None, :T] > pos[b:n, None], float("-inf"))
            out[b:n, h] = torch.matmul(torch.softmax(s, -1), vh[:T])
    return {"out": out, "k": k64, "v": v64}


def _f16_at(b, at):
    return b[..., at:at + 2].contiguous().view(torch.float16).double()  # [..., 1]


def _decode_blocks(w, kind, n_embd):
    """The values of GGML blocks: w [rows, bytes] -> [rows, n_embd] in 64 bits."""
    vals, nbytes = BLOCKS[kind]
    b = w.view(w.shape[0], n_embd // vals, nbytes)
    if kind == "q8_0":
        y = b[..., 2:34].contiguous().view(torch.int8).double() * _f16_at(b, 0)
    elif kind == "q4_k":
        d, dmin = _f16_at(b, 0), _f16_at(b, 2)
        s = b[..., 4:16].int()
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1)
        q = b[..., 16:144].int().view(*b.shape[:2], 4, 32)
        q = torch.stack([q & 15, q >> 4], -2).view(*b.shape[:2], 8, 32).double()
        y = (d * sc.double())[..., None] * q - (dmin * mn.double())[..., None]
    else:
        d = _f16_at(b, 208)
        lo = b[..., 0:128].int().view(*b.shape[:2], 2, 2, 32)
        hi = b[..., 128:192].int().view(*b.shape[:2], 2, 32)
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        parts = [((lo[..., g & 1, :] >> (4 * (g >> 1))) & 15) | (((hi >> (2 * g)) & 3) << 4) for g in range(4)]
        q = torch.stack(parts, -2).view(*b.shape[:2], 16, 16).double() - 32.0
        y = (d * sc)[..., None] * q
    return y.reshape(w.shape[0], n_embd)
