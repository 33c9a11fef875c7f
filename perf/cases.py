"""The workloads that the INT4 KV path is timed on: decode attention with the append of the new
token, chunked prefill, and whole attention blocks (QKV projection with the append, attention,
output projection) over the model shapes, batch sizes, context lengths and weight formats of
this repository's benchmark and tests.

A case is a dict of plain values:
  kind      "decode"   attn_decode_append of one token per sequence
            "prefill"  append_quant of a chunk, then attn_prefill over it
            "block"    qkv_append / qkv_append_gguf, attn_decode (one token) or attn_prefill,
                       attn_out_proj / attn_out_proj_gguf.  The output projection takes an
                       attention output of its own: a key or value that the QKV projection puts
                       next to the edge of a 4-bit code falls on either side of it with the last
                       bit of a correct sum, and what that does to the attention would hide the
                       projection's own rounding.
  layers    layers of one pass, each with a cache (and weights) of its own
  graph     the pass is captured once as a HIP graph and replayed, as a serving loop does with
            a decode step; otherwise every layer is called eagerly
  n_seq, n_head, n_kv, head_dim; ctx_lo, ctx_hi: cached positions per sequence, spread evenly
  tokens    new tokens per sequence
  dim, weights ("f16", "f16x2", "q4_k", "q5_k", "q8_0", "q4_0", "q5_0"): the block's
  softcap, qk_norm: attention options (Gemma-2, Qwen3)
"""
import math

import torch

from airframe_amd import weights as W
from airframe_amd.kv_cache import KVCache, RopeTable, attn_out_proj, attn_out_proj_gguf

THETA = 500000.0
EPS = 1e-6
GGML = {"q4_k": W.Q4_K, "q5_k": W.Q5_K, "q8_0": W.Q8_0, "q4_0": W.Q4_0, "q5_0": W.Q5_0}
#: bytes of 256 weights of one row
ROW256 = {"f16": 512, "f16x2": 1024, "q4_k": 144, "q5_k": 176, "q8_0": 272, "q4_0": 144, "q5_0": 176}


def _case(kind, n_seq, n_head, n_kv, head_dim, ctx_lo, ctx_hi, tokens=1, layers=1, graph=False,
          dim=0, weights="", softcap=0.0, qk_norm=False, **named):
    return dict(named, kind=kind, n_seq=n_seq, n_head=n_head, n_kv=n_kv, head_dim=head_dim, ctx_lo=ctx_lo,
                ctx_hi=ctx_hi, tokens=tokens, layers=layers, graph=graph, dim=dim, weights=weights,
                softcap=softcap, qk_norm=qk_norm)


def listed():
    return [
        # One layer of a chat turn on the smallest model (Llama-3.2-1B shape), called from Python:
        # the cost of one call.
        _case("decode", 1, 32, 8, 64, 512, 512, name="decode_b1_ctx512"),
        # Single-user generation: the attention of a whole decode step of a Llama-3.2-3B shape.
        _case("decode", 1, 24, 8, 128, 4171, 4171, layers=28, graph=True, name="decode_step_b1_ctx4k"),
        # Saturated serving, the headline shape (Qwen3-8B, batch 32, 8K cached tokens each).
        _case("decode", 32, 32, 8, 128, 8192, 8192, name="decode_b32_ctx8k"),
        # Long documents of different lengths (Llama-3-8B shape, 16K to 32K cached tokens).
        _case("decode", 8, 32, 8, 128, 16389, 32767, name="decode_b8_ragged32k"),
        # 256-dim heads with softcap (Gemma-2-9B shape), a medium batch of medium contexts.
        _case("decode", 16, 16, 8, 256, 2801, 4403, softcap=50.0, name="decode_b16_hd256"),
        # Eight query heads per kv head (Llama-3-70B's grouping), short ragged chats.
        _case("decode", 24, 64, 8, 128, 411, 3077, name="decode_b24_gqa8"),
        # Local single-user generation from a Q4_K GGUF (Llama-3.2-3B shape): projections and
        # attention of 8 layers.
        _case("block", 1, 24, 8, 128, 1533, 1533, layers=8, graph=True, dim=3072, weights="q4_k",
              name="block_decode_b1_q4k"),
        # Batched serving with f16 weights and QK norm (Qwen3-8B shape), 4 layers.
        _case("block", 32, 32, 8, 128, 700, 1531, layers=4, graph=True, dim=4096, weights="f16", qk_norm=True,
              name="block_decode_b32_f16"),
        # Chunked prefill of four sequences (Qwen3-4B shape): the last of four 512-token chunks.
        _case("prefill", 4, 32, 8, 128, 1536, 1536, tokens=512, name="prefill_chunk_b4"),
        # A long prompt of one user (Llama-3-8B shape), a 2048-token chunk behind 6100 tokens.
        _case("prefill", 1, 32, 8, 128, 6103, 6103, tokens=2048, name="prefill_long_b1"),
        # The second chunk of four prompts through a whole attention block (Qwen3-4B shape).
        _case("block", 4, 32, 8, 128, 512, 512, tokens=512, dim=2560, weights="f16", qk_norm=True,
              name="block_prefill_b4_f16"),
        # A second prompt of odd length from a Q4_K GGUF (Llama-3.2-3B shape).
        _case("block", 1, 24, 8, 128, 301, 301, tokens=777, dim=3072, weights="q4_k", name="block_prefill_b1_q4k"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ranges: batch 1 to 32, contexts up to 32K, chunks up to 2048 tokens,
    the listed head shapes and every weight format."""
    most_b = max(work(c)["bytes"] for c in listed())
    most_f = max(work(c)["flops"] for c in listed())
    while True:
        kind = rng.choice(["decode", "decode", "prefill", "block", "block", "block"])
        heads = [(32, 8, 64), (24, 8, 128), (32, 8, 128), (64, 8, 128)]
        if kind != "block":
            heads.append((16, 8, 256))
        n_head, n_kv, hd = rng.choice(heads)
        prompt = kind == "prefill" or (kind == "block" and rng.random() < 0.5)
        n_seq = _log_int(rng, 1, 4 if prompt else 32)
        tokens = _log_int(rng, 40, 2048) if prompt else 1
        ctx = _log_int(rng, 512 if kind == "block" else 60, 32000 if kind == "decode" else 8000)
        if kind == "prefill" and rng.random() < 0.4:
            ctx = 0
        lo = ctx if rng.random() < 0.4 else max(ctx // 2, min(ctx, 1))
        c = _case(kind, n_seq, n_head, n_kv, hd, lo, ctx, tokens=tokens, softcap=rng.choice([0.0, 0.0, 0.0, 50.0]),
                  qk_norm=rng.random() < 0.3)
        if kind == "block":
            c["dim"] = rng.choice([2048, 2560, 3072, 4096])
            c["weights"] = rng.choice(sorted(ROW256))
        if not prompt and (kind == "block" or n_seq == 1):
            c["layers"], c["graph"] = rng.choice([2, 4, 8]), True
        w = work(c)
        if w["bytes"] <= most_b and w["flops"] <= most_f:
            return c


# ---- inputs ---------------------------------------------------------------------------------

def _lens(c):
    n = c["n_seq"]
    return [c["ctx_lo"] + (c["ctx_hi"] - c["ctx_lo"]) * ((5 * s + n - 1) % n) // max(1, n - 1) if n > 1 else c["ctx_hi"]
            for s in range(n)]


def _dev():
    return torch.device("cuda", torch.cuda.current_device())


class _Draws:
    """Every random input of a case, from the seed alone: a stream per layer and name, so that
    a reader can make one of them again without the others."""

    def __init__(self, c, seed):
        self.c, self.seed = c, seed

    def gen(self, layer, what):
        g = torch.Generator(device=_dev())
        g.manual_seed((self.seed * 1000003 + layer * 101 + what) % (1 << 62))
        return g

    def normal(self, layer, what, *shape):
        return torch.randn(shape, generator=self.gen(layer, what), device=_dev())

    def outliers(self, layer):
        """[n_kv, head_dim] factors: 2% of a kv head's channels are 8 times as large."""
        c = self.c
        f = torch.ones(c["n_kv"], c["head_dim"], device=_dev())
        k = max(1, math.ceil(0.02 * c["head_dim"]))
        pick = torch.rand(c["n_kv"], c["head_dim"], generator=self.gen(layer, 1), device=_dev()).topk(k, dim=1).indices
        return f.scatter_(1, pick, 8.0)

    def cached(self, layer, upto):
        """K and V of the positions before the call, in pieces (first position, k, v)."""
        c, step = self.c, 1024
        f = self.outliers(layer)
        gk, gv = self.gen(layer, 2), self.gen(layer, 3)
        for p in range(0, upto, step):
            shape = (c["n_seq"], min(step, upto - p), c["n_kv"], c["head_dim"])
            yield p, torch.randn(shape, generator=gk, device=_dev()) * f, torch.randn(shape, generator=gv, device=_dev()) * f

    def new(self, layer):
        """q, k, v of the new tokens (decode and prefill cases)."""
        c = self.c
        f = self.outliers(layer)
        g = c["n_head"] // c["n_kv"]
        q = self.normal(layer, 4, c["n_seq"], c["tokens"], c["n_head"], c["head_dim"]) * f.repeat_interleave(g, 0)
        k = self.normal(layer, 5, c["n_seq"], c["tokens"], c["n_kv"], c["head_dim"]) * f
        v = self.normal(layer, 6, c["n_seq"], c["tokens"], c["n_kv"], c["head_dim"]) * f
        return q, k, v

    def norms(self, layer):
        hd = self.c["head_dim"]
        return 1.0 + 0.2 * self.normal(layer, 7, hd), 1.0 + 0.2 * self.normal(layer, 8, hd)

    def x(self, layer):
        c = self.c
        return self.normal(layer, 9, c["n_seq"], c["tokens"], c["dim"])

    def act(self, layer):
        c = self.c
        return self.normal(layer, 10, c["n_seq"] * c["tokens"], c["dim"])

    def attn(self, layer):
        c = self.c
        return 0.2 * self.normal(layer, 15, c["n_seq"] * c["tokens"], c["n_head"] * c["head_dim"])

    def weight(self, layer, what, rows, cols):
        """The weight matrix in its stored form: f16 rows, or the bytes of its GGUF blocks."""
        fmt = self.c["weights"]
        if fmt == "f16":
            return (self.normal(layer, what, rows, cols) * 0.02).half()
        if fmt == "f16x2":
            w = self.normal(layer, what, rows, cols) * 0.02
            hi = w.half()
            return torch.cat([hi, (w - hi.float()).half()], 1)
        g = self.gen(layer, what)
        per = 256 if fmt in ("q4_k", "q5_k") else 32
        n, size = rows * cols // per, ROW256[fmt] * per // 256
        b = torch.randint(0, 256, (n, size), generator=g, device=_dev(), dtype=torch.uint8)
        # block scales that give weights of about 0.02, and for the K formats mins that centre them
        top = {"q4_k": 1.5e-4, "q5_k": 7e-5, "q8_0": 3e-4, "q4_0": 5e-3, "q5_0": 2.5e-3}[fmt]
        d = top * (0.5 + torch.rand(n, 1, generator=g, device=_dev()))
        b[:, 0:2] = d.half().view(torch.uint8).reshape(n, 2)
        if per == 256:
            b[:, 2:4] = (d * {"q4_k": 7.5, "q5_k": 15.5}[fmt]).half().view(torch.uint8).reshape(n, 2)
        return b.reshape(-1)

    def weights(self, layer):
        c = self.c
        qr, kr = c["n_head"] * c["head_dim"], c["n_kv"] * c["head_dim"]
        return (self.weight(layer, 11, qr, c["dim"]), self.weight(layer, 12, kr, c["dim"]),
                self.weight(layer, 13, kr, c["dim"]), self.weight(layer, 14, c["dim"], qr))


def _passes(st):
    """One pass: every layer's calls, as a host loop makes them."""
    c, kv, rope = st["case"], st["kv"], st["rope"]
    for layer, io in enumerate(st["io"]):
        if c["kind"] == "decode":
            kv.attn_decode_append(layer, io["k"], io["v"], io["q"], rope, out=io["out"], softcap=c["softcap"],
                                  workspace=st["ws"])
            continue
        if c["kind"] == "prefill":
            kv.append_quant(layer, io["k"], io["v"], rope)
            kv.attn_prefill(layer, io["q"], rope, out=io["out"], softcap=c["softcap"])
            continue
        wq, wk, wv, wo = io["w"]
        planes = 2 if c["weights"] == "f16x2" else 1
        if c["weights"] in GGML:
            kv.qkv_append_gguf(layer, io["x"], GGML[c["weights"]], wq, wk, wv, rope, q_out=io["q"])
        else:
            kv.qkv_append(layer, io["x"], wq, wk, wv, rope, q_out=io["q"], planes=planes)
        if c["tokens"] == 1:
            kv.attn_decode(layer, io["q1"], rope, out=io["out"], softcap=c["softcap"], workspace=st["ws"])
        else:
            kv.attn_prefill(layer, io["q"], rope, out=io["out"], softcap=c["softcap"])
        if c["weights"] in GGML:
            attn_out_proj_gguf(io["attn"], GGML[c["weights"]], wo, c["dim"], io["act"])
        else:
            attn_out_proj(io["attn"], wo, io["act"], planes=planes)


def prepare(case, seed):
    c, d, dev = case, _Draws(case, seed), _dev()
    lens, tok, hd = _lens(c), c["tokens"], c["head_dim"]
    room = max(lens) + tok
    rope = RopeTable(room, hd, THETA)
    kv = KVCache.new_int4(c["layers"], c["n_kv"], hd, room, c["n_seq"])
    io = []
    for layer in range(c["layers"]):
        if c["qk_norm"]:
            kv.set_qk_norm(layer, *d.norms(layer), EPS)
        b = {}
        if c["kind"] == "block":
            b["x"], b["act"], b["w"] = d.x(layer), d.act(layer), d.weights(layer)
            b["q"] = torch.empty(c["n_seq"], tok, c["n_head"], hd, device=dev)
            b["out"] = torch.empty_like(b["q"])
            b["attn"] = d.attn(layer)
        else:
            b["q"], b["k"], b["v"] = d.new(layer)
            b["out"] = torch.empty_like(b["q"])
        if tok == 1:
            b["q1"], b["out"] = b["q"].view(c["n_seq"], c["n_head"], hd), b["out"].view(c["n_seq"], c["n_head"], hd)
            if c["kind"] == "decode":
                b["q"] = b["q1"]
        io.append(b)
    pieces = [d.cached(layer, max(lens)) for layer in range(c["layers"])]
    for p in range(0, max(lens), 1024):
        for layer, piece in enumerate(pieces):
            _, k, v = next(piece)
            kv.append_quant(layer, k, v, rope)
        kv.increment(k.shape[1])
    for s, n in enumerate(lens):
        if n != max(lens):
            kv.set_seq_len(n, seq=s)
    st = {"case": c, "kv": kv, "rope": rope, "io": io, "ws": kv.workspace(c["n_head"])}
    if c["graph"]:
        acts = [b["act"].clone() for b in io if "act" in b]
        _passes(st)  # the library's workspaces exist before the capture
        torch.cuda.synchronize()
        for b, a in zip(io, acts):
            b["act"].copy_(a)
        graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.graph(graph, stream=side):
            _passes(st)
        st["graph"] = graph
    return st


def run(state):
    if "graph" in state:
        state["graph"].replay()
    else:
        _passes(state)
    if state["case"]["kind"] == "block":
        return [(b["q"], b["out"], b["act"]) for b in state["io"]]
    return [b["out"] for b in state["io"]]


# ---- what a pass cannot do without ----------------------------------------------------------

def work(case):
    c = case
    lens, tok, hd = _lens(c), c["tokens"], c["head_dim"]
    rows = c["n_seq"] * tok
    row = c["n_kv"] * (hd + 8)  # packed K and V and the scales of one position
    keys = sum(n * tok + tok * (tok + 1) // 2 for n in lens)
    by = sum(lens) * row + rows * row  # the cached positions read, the new ones written
    by += 4 * rows * c["n_head"] * hd  # the attention output
    fl = 4.0 * keys * c["n_head"] * hd
    if c["kind"] == "block":
        qr, kr = c["n_head"] * hd, c["n_kv"] * hd
        by += (2 * qr + 2 * kr) * c["dim"] * ROW256[c["weights"]] / 256.0
        by += 4 * rows * (c["dim"] + 2 * qr + 2 * c["dim"])  # x, attn read, q written, act read and written
        fl += 2.0 * rows * c["dim"] * (2 * qr + 2 * kr)
    else:
        by += 4 * rows * (c["n_head"] + 2 * c["n_kv"]) * hd  # q, k, v read
    return {"bytes": by * c["layers"], "flops": fl * c["layers"]}


def tolerance(case):
    # Attention over given keys and values: the codes are the same bits, and what is left is
    # the f32 of the scores, the softmax and the sums (seen: up to 2.7e-6 off 64 bits).
    if case["kind"] != "block":
        return {"rel": 1e-5, "max": 1e-3}
    # Through the projection a code next to an edge may fall to its other side (see the top);
    # at 250 cached positions or more one such code moves an attention output by a part in a
    # few hundred at most.  (The projections themselves: seen up to 5e-7 off 64 bits.)
    return {"rel": 1e-3, "max": 0.2}


# ---- the same in 64 bits --------------------------------------------------------------------

def _table(hd, pos):
    """cos and sin of the f32 angles of the given positions, [len(pos), hd / 2]."""
    i = torch.arange(hd // 2, dtype=torch.float64, device=_dev())
    theta = (1.0 / (torch.tensor(THETA, dtype=torch.float64, device=_dev()) ** (2 * i / hd)).float()).float()
    angle = (pos.float()[:, None] * theta[None, :]).double()
    return angle.cos().float(), angle.sin().float()


def _rotate(x, cos, sin):
    """Adjacent pairs of x [..., heads, hd], in x's type; cos, sin [..., hd / 2]."""
    cos, sin = cos[..., None, :].to(x.dtype), sin[..., None, :].to(x.dtype)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)


def _norm_q(x, w):
    y = x.double()
    return y * torch.rsqrt((y * y).mean(-1, keepdim=True) + EPS) * w.double()


def _norm_k(x, w):
    """The norm of K in the f32 steps that the cache defines (the squares summed in order), as
    the codes depend on every bit of it."""
    total = torch.zeros_like(x[..., 0])
    for i in range(x.shape[-1]):
        total = total + x[..., i] * x[..., i]
    # torch's f32 square root and division on the CPU round correctly
    scale = (1.0 / torch.sqrt((total / x.shape[-1] + EPS).cpu())).to(x.device)
    return (x * scale[..., None]) * w


def _stored(x):
    """What the cache gives back for f32 head vectors: f32 scale, 4-bit codes, rounded half
    away from zero; in 64 bits."""
    top = x.abs().amax(-1, keepdim=True)
    # (divided by a tensor: torch multiplies by the reciprocal of a number)
    scale = torch.where(top > 0, top / torch.full_like(top, 7.0), torch.ones_like(top))
    q = (x / scale).double()
    code = torch.sign(q) * torch.floor(q.abs() + 0.5)
    return code.clamp(-7, 7) * scale.double()


def _dequant(fmt, b, rows, cols):
    """GGUF blocks to values in 64 bits."""
    if fmt == "f16":
        return b.double()
    if fmt == "f16x2":
        return b[:, :cols].double() + b[:, cols:].double()

    def half(x):
        return x.contiguous().view(torch.float16).double()

    if fmt in ("q4_0", "q5_0", "q8_0"):
        b = b.view(rows * cols // 32, -1)
        d = half(b[:, 0:2])
        if fmt == "q8_0":
            return (d * b[:, 2:].view(torch.int8).double()).view(rows, cols)
        qs = b[:, -16:]
        n = torch.cat([qs & 15, qs >> 4], 1).double()
        if fmt == "q4_0":
            return (d * (n - 8)).view(rows, cols)
        bit = torch.arange(8, device=b.device, dtype=torch.uint8)
        high = ((b[:, 2:6, None] >> bit) & 1).reshape(-1, 32).double()
        return (d * (n + 16 * high - 16)).view(rows, cols)
    b = b.view(rows * cols // 256, -1)
    d, dmin = half(b[:, 0:2]), half(b[:, 2:4])
    s = b[:, 4:16].to(torch.int32)
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    qs = b[:, -128:].view(-1, 4, 1, 32)
    n = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
    if fmt == "q5_k":
        bit = torch.arange(8, device=b.device, dtype=torch.uint8)
        n = n + 16 * ((b[:, None, 16:48] >> bit[None, :, None]) & 1).double()
    return ((d * sc)[:, :, None] * n - (dmin * mn)[:, :, None]).view(rows, cols)


def _block_exact(c, d, layer):
    qr = c["n_head"] * c["head_dim"]
    stored = d.weights(layer)
    wq = _dequant(c["weights"], stored[0], qr, c["dim"])
    q = d.x(layer).double().view(-1, c["dim"]) @ wq.t().contiguous()
    wo = _dequant(c["weights"], stored[3], c["dim"], qr)
    act = d.act(layer).double() + d.attn(layer).double() @ wo.t().contiguous()
    # no value in 64 bits for the attention between them: its keys and values are 4-bit codes
    # of projections, on either side of an edge (see the top)
    return q.view(c["n_seq"], c["tokens"], c["n_head"], c["head_dim"]), None, act


def exact(case, seed):
    c, d = case, _Draws(case, seed)
    if c["kind"] == "block":
        return [_block_exact(c, d, layer) for layer in range(c["layers"])]
    lens, tok, hd, g = _lens(c), c["tokens"], c["head_dim"], c["n_head"] // c["n_kv"]
    found = []
    for layer in range(c["layers"]):
        qn, kn = d.norms(layer) if c["qk_norm"] else (None, None)
        room = max(lens) + tok
        ks = torch.zeros(c["n_seq"], room, c["n_kv"], hd, device=_dev())
        vs = torch.zeros_like(ks)
        for p, k, v in d.cached(layer, max(lens)):
            ks[:, p:p + k.shape[1]], vs[:, p:p + k.shape[1]] = k, v
        q, kx, vx = d.new(layer)
        q = q.double()
        cos, sin = _table(hd, torch.arange(room, device=_dev()))
        out = torch.empty_like(q)
        for s, n in enumerate(lens):
            ks[s, n:n + tok], vs[s, n:n + tok] = kx[s], vx[s]
            k, v = ks[s, :n + tok], vs[s, :n + tok]
            if kn is not None:
                k = _norm_k(k, kn)
            k = _stored(_rotate(k, cos[:n + tok], sin[:n + tok]))
            v = _stored(v)
            qq = _norm_q(q[s], qn) if qn is not None else q[s]
            qq = _rotate(qq, cos[n:n + tok], sin[n:n + tok])
            qq = qq.view(tok, c["n_kv"], g, hd).permute(1, 0, 2, 3).reshape(c["n_kv"], tok * g, hd).contiguous()
            sc = torch.bmm(qq, k.permute(1, 2, 0).contiguous()) / math.sqrt(hd)
            if c["softcap"] > 0:
                sc = torch.tanh(sc / c["softcap"]) * c["softcap"]
            if tok > 1:
                at = torch.arange(n + tok, device=_dev())
                mask = at[None, :] > at[n:, None]
                sc.masked_fill_(mask.repeat_interleave(g, 0)[None], -math.inf)
            o = torch.bmm(torch.softmax(sc, -1), v.permute(1, 0, 2).contiguous())
            out[s] = o.view(c["n_kv"], tok, g, hd).permute(1, 0, 2, 3).reshape(tok, c["n_head"], hd)
            del sc, o
        found.append(out if tok > 1 else out[:, 0])
    return found
