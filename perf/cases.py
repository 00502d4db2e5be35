"""Timed workloads of the int4 x int8 linear-layer path, through webyiq_amd.ops
and webyiq_amd.layer.

A case is a dict of plain values.  Its "kind" names the call sequence that a
program runs:

  gemv    one decode product on activations that are already quantised
  head    final norm + quantiser, lm_head product, greedy argmax
  step    one recorded decode (or speculative verify) step: embedding lookup,
          decoder layers, head; replayed as a HIP graph
  linear  quantiser (or the MTP input stage) and one prefill product
  mlp     a prefill MLP block: norm + quantiser, gate/up with SiLU, quantiser,
          down
  chunk   one recorded prefill chunk: embedding lookup, qkv, MLP block with the
          residual add; sized for `cap` tokens and covering the `m` of the
          device step parameters; replayed as a HIP graph

Weights are drawn N(0, 0.02) and rounded to int4 with an f16 scale and minimum
per group of G codes; inputs are N(0, 1) with 8 outlier channels x 20.  GA = 0
means one activation scale per token, 32 one per 32 elements.
"""
import math

import torch

from webyiq_amd import ops
from webyiq_amd.layer import DecodeLayer

EPS = 1e-6
HEAD_DIM = 128
MAX_CTX = 4096


def listed():
    return [
        # the smallest call: one projection of one decoded token
        dict(name="gemv_token", kind="gemv", M=1, K=2048, N=6144, G=128, GA=0, mode=0),
        # a decoded token: the whole recorded step, full head
        dict(name="decode_step", kind="step", M=1, hidden=2048, ffn=6144, kv=512, layers=8, V=32768, G=128),
        # a speculative verify step of four tokens
        dict(name="verify_step", kind="step", M=4, hidden=2048, ffn=6144, kv=512, layers=4, V=32768, G=128),
        # the head over the full vocabulary, one token
        dict(name="head_token", kind="head", M=1, K=2048, V=151936, G=128, ids=False),
        # the reduced draft vocabulary for eight tokens, indices mapped
        dict(name="head_draft", kind="head", M=8, K=2048, V=32768, G=128, ids=True),
        # prompts of about a thousand tokens: an up-projection and a long-K down-projection
        dict(name="prefill_up", kind="linear", M=1024, K=2048, N=6144, G=128, GA=0, norm=True, mtp=False),
        dict(name="prefill_down", kind="linear", M=1024, K=6144, N=2048, G=128, GA=0, norm=False, mtp=False),
        # the converter's native group of 32, half a thousand tokens
        dict(name="prefill_mlp_g32", kind="mlp", M=512, hidden=2048, ffn=6144, G=32, GA=0),
        # the MTP input projection over a prompt of odd length, per-32 activations
        dict(name="mtp_fc", kind="linear", M=333, K=4096, N=2048, G=32, GA=32, norm=True, mtp=True),
        # a recorded chunk of up to 128 tokens, mostly filled
        dict(name="chunk", kind="chunk", cap=128, m=97, hidden=2048, ffn=6144, kv=512, G=128, GA=0),
        # the last chunk of a prompt: few tokens, the per-32 format
        dict(name="chunk_tail", kind="chunk", cap=128, m=19, hidden=2048, ffn=6144, kv=512, G=32, GA=32),
        # a long prompt
        dict(name="prefill_long", kind="mlp", M=4096, hidden=2048, ffn=6144, G=128, GA=0),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["gemv", "step", "head", "linear", "linear", "mlp", "mlp", "chunk", "chunk"])
    G = rng.choice([128, 128, 32])
    k128 = lambda lo, hi: 128 * max(1, _logu(rng, lo, hi) // 128)
    if kind == "gemv":
        return dict(kind=kind, M=rng.randint(1, 8), K=k128(512, 8192), N=_logu(rng, 256, 12288), G=G,
                    GA=rng.choice([0, 0, 32]), mode=rng.choice([0, 2]))
    if kind == "head":
        return dict(kind=kind, M=rng.randint(1, 8), K=k128(1024, 4096), V=_logu(rng, 8192, 65536), G=G,
                    ids=rng.random() < 0.5)
    if kind == "step":
        hidden = rng.choice([1024, 1536, 2048, 2560])
        return dict(kind=kind, M=rng.randint(1, 8), hidden=hidden, ffn=k128(2 * hidden, 4 * hidden),
                    kv=rng.choice([256, 512, 1024]), layers=rng.randint(2, 6), V=_logu(rng, 8192, 40000), G=G)
    if kind == "chunk":
        cap = rng.choice([64, 128, 128, 256])
        hidden = rng.choice([1024, 1536, 2048, 2560])
        return dict(kind=kind, cap=cap, m=rng.randint(9, cap), hidden=hidden, ffn=k128(2 * hidden, 4 * hidden),
                    kv=rng.choice([256, 512, 1024]), G=G, GA=rng.choice([0, 32]))
    GA = rng.choice([0, 0, 32])
    # multiply-adds up to the long prompt's (a quarter of them in the formats with a group of 32)
    budget = 3 * 4096 * 2048 * 6144 // (4 if 32 in (G, GA) else 1)
    if kind == "mlp":
        hidden = k128(1024, 4096)
        ffn = k128(2 * hidden, 4 * hidden)
        return dict(kind=kind, M=_logu(rng, 9, min(4096, budget // (3 * hidden * ffn))), hidden=hidden, ffn=ffn, G=G,
                    GA=GA)
    mtp = rng.random() < 0.2
    if mtp:
        G, GA = 32, 32
    K, N = k128(768, 8192), _logu(rng, 256, 12288)
    if mtp:
        K = 256 * max(3, K // 256)
    return dict(kind=kind, M=_logu(rng, 9, min(4096, budget // (K * N))), K=K, N=N, G=G, GA=GA,
                norm=rng.random() < 0.5, mtp=mtp)


# ------------------------------------------------------------------ inputs ----

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _weight(g, rows, K, G):
    """int4 rows of N(0, 0.02): code = round((w - m) / s), s = (max - m) / 15."""
    q = torch.empty((rows, K // 8), dtype=torch.int32, device="cuda")
    s = torch.empty((rows, K // G), dtype=torch.int32, device="cuda")
    shift = torch.tensor([0, 8, 16, 24, 4, 12, 20, 28], device="cuda")  # code i of a word's eight
    step = max(1, (1 << 26) // K)
    for r in range(0, rows, step):
        w = _randn(g, min(step, rows - r), K // G, G) * 0.02
        lo = w.amin(-1).half()
        sc = ((w.amax(-1) - lo.float()) / 15.0).half()
        c = torch.round((w - lo.float()[..., None]) / sc.float()[..., None]).clamp_(0, 15).to(torch.int64)
        words = (c.reshape(w.shape[0], K // 8, 8) << shift).sum(-1)
        q[r:r + step] = words.to(torch.int32)
        bits = (sc.view(torch.int16).to(torch.int32) & 0xFFFF) | (lo.view(torch.int16).to(torch.int32) << 16)
        s[r:r + step] = bits
    return ops.Q4Tensor(q, s, K, G)


def _inputs(g, M, K):
    x = _randn(g, M, K)
    hot = torch.randperm(K, generator=g, device="cuda")[:8]
    x[:, hot] *= 20.0
    return x


def _norm(g, K):
    return 1.0 + 0.2 * _randn(g, K)


def _tokens(g, n, V):
    return torch.randint(0, V, (n,), generator=g, device="cuda", dtype=torch.int32)


def _record(run):
    """Replayable recording of run(), its buffers warm."""
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    return graph


def _build(case, seed):
    """The operands of a case (what `prepare` and `exact` share)."""
    g = _gen(seed)
    kind = case["kind"]
    st = {"case": case}
    if kind == "gemv":
        rows = case["N"] * (2 if case["mode"] == 2 else 1)
        st["w"] = _weight(g, rows, case["K"], case["G"])
        st["x"] = _inputs(g, case["M"], case["K"])
    elif kind == "head":
        st["w"] = _weight(g, case["V"], case["K"], case["G"])
        st["x"] = _inputs(g, case["M"], case["K"])
        st["norm"] = _norm(g, case["K"])
        st["ids"] = None
        if case["ids"]:  # an ascending subset of a vocabulary four times as large
            st["ids"] = torch.randperm(4 * case["V"], generator=g, device="cuda")[:case["V"]].sort()[0].to(torch.int32)
    elif kind == "linear":
        K = case["K"] // (2 if case["mtp"] else 1)
        st["w"] = _weight(g, case["N"], case["K"], case["G"])
        st["x"] = _inputs(g, case["M"], K)
        st["norm"] = _norm(g, K) if case["norm"] or case["mtp"] else None
        if case["mtp"]:
            st["emb"] = 0.02 * _randn(g, case["M"], K)
            st["norm_e"], st["norm_h"] = _norm(g, K), _norm(g, K)
    elif kind == "mlp":
        st["x"] = _inputs(g, case["M"], case["hidden"])
        st["norm"] = _norm(g, case["hidden"])
        st["gate_up"] = _weight(g, 2 * case["ffn"], case["hidden"], case["G"])
        st["down"] = _weight(g, case["hidden"], case["ffn"], case["G"])
    elif kind == "chunk":
        h = case["hidden"]
        st["embed"] = _weight(g, 4096, h, case["G"])
        st["tok"] = _tokens(g, case["cap"], 4096)
        st["norm"], st["norm2"] = _norm(g, h), _norm(g, h)
        st["qkv"] = _weight(g, h + 2 * case["kv"], h, case["G"])
        st["gate_up"] = _weight(g, 2 * case["ffn"], h, case["G"])
        st["down"] = _weight(g, h, case["ffn"], case["G"])
    else:  # step
        h, M = case["hidden"], case["M"]
        st["head"] = _weight(g, case["V"], h, case["G"])
        st["tok"] = _tokens(g, M, case["V"])
        st["norm"] = _norm(g, h)
        st["pos"] = 200 + 37 * (seed % 61)
        st["layers"] = []
        for _ in range(case["layers"]):
            w = ops.Weights(qkv=_weight(g, h + 2 * case["kv"], h, case["G"]), o=_weight(g, h, h, case["G"]),
                            gate_up=_weight(g, 2 * case["ffn"], h, case["G"]),
                            down=_weight(g, h, case["ffn"], case["G"]), attn_norm=_norm(g, h), mlp_norm=_norm(g, h))
            # attention partials of a 4096-position context: output sums, maximum, weight sum per 32 positions
            part = _randn(g, M, h // HEAD_DIM, MAX_CTX // 32, HEAD_DIM + 2)
            part[..., HEAD_DIM + 1] = 1.0 + 31.0 * torch.rand(part.shape[:-1], generator=g, device="cuda")
            st["layers"].append((w, part))
    return st


def _ga(case, K):
    return case["GA"] or K


def prepare(case, seed):
    st = _build(case, seed)
    kind = case["kind"]
    f32 = dict(dtype=torch.float32, device="cuda")
    if kind == "gemv":
        st["acts"] = ops.quant(st["x"], GA=case["GA"] or None, G=case["G"])
        st["y"] = torch.zeros((case["M"], case["N"]), **f32)
    elif kind == "head":
        st["acts"] = ops.empty_acts(case["M"], case["K"], None, case["G"])
        st["logits"] = torch.zeros((case["M"], case["V"]), **f32)
        st["ws"] = ops.lm_head_workspace()
        st["out"] = torch.zeros(case["M"], dtype=torch.int32, device="cuda")
    elif kind == "linear":
        st["acts"] = ops.empty_acts(case["M"], case["K"], case["GA"] or None, case["G"])
        st["y"] = torch.zeros((case["M"], case["N"]), **f32)
        st["ws"] = ops.gemm_workspace(case["N"], case["K"], case["G"], case["M"], case["GA"] or None)
    elif kind == "mlp":
        h, f, M = case["hidden"], case["ffn"], case["M"]
        st["a1"] = ops.empty_acts(M, h, case["GA"] or None, case["G"])
        st["a2"] = ops.empty_acts(M, f, case["GA"] or None, case["G"])
        st["h"] = torch.zeros((M, f), **f32)
        st["y"] = torch.zeros((M, h), **f32)
        st["ws1"] = ops.gemm_workspace(f, h, case["G"], M, case["GA"] or None, ops.MODE_SILU_MUL)
        st["ws2"] = ops.gemm_workspace(h, f, case["G"], M, case["GA"] or None)
    elif kind == "chunk":
        h, f, cap = case["hidden"], case["ffn"], case["cap"]
        GA, G = case["GA"] or None, case["G"]
        st["params"] = ops.make_params(pos=0, seq_len=case["m"], m=case["m"])
        st["x"] = torch.zeros((cap, h), **f32)
        st["q"] = torch.zeros((cap, h + 2 * case["kv"]), **f32)
        st["h"] = torch.zeros((cap, f), **f32)
        st["a1"], st["a2"] = ops.empty_acts(cap, h, GA, G), ops.empty_acts(cap, f, GA, G)
        st["ws1"] = ops.gemm_workspace(h + 2 * case["kv"], h, G, cap, GA)
        st["ws2"] = ops.gemm_workspace(f, h, G, cap, GA, ops.MODE_SILU_MUL)
        st["ws3"] = ops.gemm_workspace(h, f, G, cap, GA, ops.MODE_ACCUMULATE)

        def run_chunk():
            p = st["params"]
            ops.embed(st["embed"], st["tok"], out=st["x"])
            ops.quant(st["x"], norm=st["norm"], eps=EPS, out=st["a1"])
            ops.gemm(st["qkv"], st["a1"], y=st["q"], params=p, workspace=st["ws1"])
            ops.quant(st["x"], norm=st["norm2"], eps=EPS, out=st["a1"])
            ops.gemm(st["gate_up"], st["a1"], mode=ops.MODE_SILU_MUL, y=st["h"], params=p, workspace=st["ws2"])
            ops.quant(st["h"], out=st["a2"])
            ops.gemm(st["down"], st["a2"], mode=ops.MODE_ACCUMULATE, y=st["x"], params=p, workspace=st["ws3"])
        st["graph"] = _record(run_chunk)
    else:
        h, M = case["hidden"], case["M"]
        st["x"] = torch.zeros((M, h), **f32)
        st["params"] = ops.make_params(pos=st["pos"], seq_len=st["pos"] + M, m=M)
        stack = []
        for w, part in st["layers"]:
            layer = DecodeLayer(w, M, hidden=h, q_dim=h, kv_dim=case["kv"], ffn=case["ffn"], G=case["G"], eps=EPS,
                                x=st["x"], attention="combine", head_dim=HEAD_DIM, max_ctx=MAX_CTX,
                                params=st["params"])
            layer.part = part
            stack.append(layer)
        st["stack"] = stack
        st["acts"] = ops.empty_acts(M, h, None, case["G"])
        st["logits"] = torch.zeros((M, case["V"]), **f32)
        st["out"] = torch.zeros(M, dtype=torch.int32, device="cuda")
        st["ws"] = ops.lm_head_workspace()

        def run_step():
            ops.embed(st["head"], st["tok"], out=st["x"])
            for layer in stack:
                layer.run()
            ops.quant(st["x"], norm=st["norm"], eps=EPS, out=st["acts"])
            ops.lm_head_argmax(st["head"], st["acts"], logits=st["logits"], workspace=st["ws"], out=st["out"])
        st["graph"] = _record(run_step)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "gemv":
        return ops.gemv(st["w"], st["acts"], mode=case["mode"], y=st["y"])
    if kind == "head":
        ops.quant(st["x"], norm=st["norm"], eps=EPS, out=st["acts"])
        ops.lm_head_argmax(st["w"], st["acts"], ids=st["ids"], logits=st["logits"], workspace=st["ws"],
                           out=st["out"])
        return st["logits"], st["out"]
    if kind == "linear":
        if case["mtp"]:
            ops.mtp_in(st["emb"], st["x"], st["norm"], st["norm_e"], st["norm_h"], eps=EPS, out=st["acts"])
        else:
            ops.quant(st["x"], norm=st["norm"], eps=EPS, out=st["acts"])
        return ops.gemm(st["w"], st["acts"], y=st["y"], workspace=st["ws"])
    if kind == "mlp":
        ops.quant(st["x"], norm=st["norm"], eps=EPS, out=st["a1"])
        ops.gemm(st["gate_up"], st["a1"], mode=ops.MODE_SILU_MUL, y=st["h"], workspace=st["ws1"])
        ops.quant(st["h"], out=st["a2"])
        ops.gemm(st["down"], st["a2"], y=st["y"], workspace=st["ws2"])
        return st["h"], st["y"]
    st["graph"].replay()
    if kind == "chunk":
        return st["q"], st["h"], st["x"]
    return st["logits"], st["x"], st["out"]


# --------------------------------------------------------------- accounting ----

def _lin(M, K, rows, N, G):
    """Weights and scales read once, f32 input rows read and output rows written once; 2 M K rows operations."""
    return rows * K // 2 + 4 * rows * (K // G) + 4 * M * K + 4 * M * N, 2 * M * K * rows


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        rows = case["N"] * (2 if case["mode"] == 2 else 1)
        b, f = _lin(case["M"], case["K"], rows, case["N"], case["G"])
        return {"bytes": b - 3 * case["M"] * case["K"], "flops": f}  # the input is int8
    if kind == "head":
        b, f = _lin(case["M"], case["K"], case["V"], case["V"], case["G"])
        return {"bytes": b, "flops": f}
    if kind == "linear":
        b, f = _lin(case["M"], case["K"], case["N"], case["N"], case["G"])
        return {"bytes": b, "flops": f}
    if kind == "mlp":
        b1, f1 = _lin(case["M"], case["hidden"], 2 * case["ffn"], case["ffn"], case["G"])
        b2, f2 = _lin(case["M"], case["ffn"], case["hidden"], case["hidden"], case["G"])
        return {"bytes": b1 + b2 - 4 * case["M"] * case["ffn"], "flops": f1 + f2}
    h = case["hidden"]
    M = case["m"] if kind == "chunk" else case["M"]
    parts = [(h, h + 2 * case["kv"], h + 2 * case["kv"]), (h, 2 * case["ffn"], case["ffn"]), (case["ffn"], h, h)]
    if kind == "chunk":
        each = [_lin(M, K, rows, N, case["G"]) for K, rows, N in parts]
        return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
    parts.append((h, h, h))
    each = [_lin(M, K, rows, N, case["G"]) for K, rows, N in parts]
    bh, fh = _lin(M, h, case["V"], case["V"], case["G"])
    ctx = 1000 // 32 * 4 * M * (h // HEAD_DIM) * (HEAD_DIM + 2)  # partials up to a position of about 1000
    return {"bytes": case["layers"] * (sum(b for b, _ in each) + ctx) + bh,
            "flops": case["layers"] * sum(f for _, f in each) + fh}


def tolerance(case):
    # About four times the measured distance from `exact`.  Sums differ by a few 1e-7; a value that falls next to a
    # rounding boundary of a quantiser takes the neighbouring code in another implementation, which moves the
    # product by about 1e-4, and by more after a second quantiser or through several layers.
    kind = case["kind"]
    if kind == "step":
        return {"rel": 2e-3, "differ": 0.5}
    if kind in ("mlp", "chunk"):
        return {"rel": 2e-3}
    if kind == "head":
        return {"rel": 4e-4, "differ": 0.0}
    return {"rel": 1e-5 if kind == "gemv" else 4e-4}


# -------------------------------------------------------------------- exact ----

def _codes(w):
    shift = torch.tensor([0, 8, 16, 24, 4, 12, 20, 28], device=w.q.device, dtype=torch.int32)
    return ((w.q[..., None] >> shift) & 15).reshape(w.q.shape[0], w.K)


def _dequant(w):
    """int4 rows as float64 [rows, K]."""
    s = (w.s & 0xFFFF).to(torch.int16).view(torch.float16).double()
    m = (w.s >> 16).to(torch.int16).view(torch.float16).double()
    q = _codes(w).reshape(w.q.shape[0], -1, w.G).double()
    return (q * s[..., None] + m[..., None]).reshape(w.q.shape[0], w.K)


def _rms(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _fq(x, GA):
    """Quantised to int8 with one scale per GA elements, and back."""
    v = x.double().reshape(x.shape[0], -1, GA)
    d = v.abs().amax(-1, keepdim=True) / 127.0
    return torch.where(d > 0, torch.round(v / torch.where(d > 0, d, 1.0)) * d, 0.0).reshape(x.shape)


def _mm(a, w):
    """a @ dequantised w^T, a slice of rows at a time."""
    out = torch.empty((a.shape[0], w.rows), dtype=torch.float64, device=a.device)
    step = max(1, (1 << 26) // w.K)
    for r in range(0, w.rows, step):
        part = ops.Q4Tensor(w.q[r:r + step], w.s[r:r + step], w.K, w.G)
        out[:, r:r + step] = a @ _dequant(part).T.contiguous()
    return out


def _swiglu(z):
    a, u = z.chunk(2, dim=1)
    return a / (1.0 + torch.exp(-a)) * u


def _merge(part, pos):
    """Attention output [M, H * D] of the chunk partials; token t covers positions 0 .. pos + t."""
    p = part.double()
    M, H, _, D2 = p.shape
    out = torch.empty((M, H, D2 - 2), dtype=torch.float64, device=p.device)
    for t in range(M):
        n = (pos + t) // 32 + 1
        mx = p[t, :, :n, D2 - 2]
        w = torch.exp(mx - mx.amax(-1, keepdim=True))
        out[t] = (w[..., None] * p[t, :, :n, :D2 - 2]).sum(1) / (w * p[t, :, :n, D2 - 1]).sum(1, keepdim=True)
    return out.reshape(M, -1)


def exact(case, seed):
    st = _build(case, seed)
    kind = case["kind"]
    if kind == "gemv":
        y = _mm(_fq(st["x"], _ga(case, case["K"])), st["w"])
        return _swiglu(y) if case["mode"] == 2 else y
    if kind == "head":
        return _mm(_fq(_rms(st["x"], st["norm"]), case["K"]), st["w"]), None
    if kind == "linear":
        if case["mtp"]:
            x = torch.cat([_rms(st["emb"], st["norm_e"]), _rms(_rms(st["x"], st["norm"]), st["norm_h"])], 1)
        else:
            x = _rms(st["x"], st["norm"]) if case["norm"] else st["x"]
        return _mm(_fq(x, _ga(case, case["K"])), st["w"])
    if kind == "mlp":
        hid, ffn = case["hidden"], case["ffn"]
        h = _swiglu(_mm(_fq(_rms(st["x"], st["norm"]), _ga(case, hid)), st["gate_up"]))
        return h, _mm(_fq(h, _ga(case, ffn)), st["down"])
    if kind == "chunk":
        hid, ffn, m = case["hidden"], case["ffn"], case["m"]
        x = _dequant(ops.Q4Tensor(st["embed"].q[st["tok"].long()], st["embed"].s[st["tok"].long()], hid, case["G"]))
        q = _mm(_fq(_rms(x, st["norm"]), _ga(case, hid)), st["qkv"])
        h = _swiglu(_mm(_fq(_rms(x, st["norm2"]), _ga(case, hid)), st["gate_up"]))
        q[m:] = 0.0  # rows past the chunk's tokens are not written
        h[m:] = 0.0
        x[:m] += _mm(_fq(h, _ga(case, ffn)), st["down"])[:m]
        return q, h, x
    h, ffn = case["hidden"], case["ffn"]
    head = st["head"]
    x = _dequant(ops.Q4Tensor(head.q[st["tok"].long()], head.s[st["tok"].long()], h, case["G"]))
    for w, part in st["layers"]:
        x = x + _mm(_fq(_merge(part, st["pos"]), 32), w["o"])
        x = x + _mm(_fq(_swiglu(_mm(_fq(_rms(x, w["mlp_norm"]), h), w["gate_up"])), ffn), w["down"])
    return _mm(_fq(_rms(x, st["norm"]), h), head), x, None
