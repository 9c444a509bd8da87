"""The work this framework is used for, as measurable cases over its public entry points.

Seven kinds, each a range of sizes, types and options (draw() samples them):

  gemv     one-to-32-row products with a packed matrix: a decode step's projections and head
           (quant.rwkvq_sb6_gemv / rwkvq_sym_gemv)
  gemm     the fp16 long pass of a packed matrix or r/k/v group: a prompt's projections
           (quant.rwkvq_sb6_gemm / rwkvq_sym_gemm)
  wkv      the WKV-7 forward over a sequence, step by step or in time chunks: a prompt's recurrence
           (kernel.wkv7_sequence_forward / wkv7_sequence_forward_chunked)
  train    the differentiable WKV-7 forward and its backward (kernel.wkv7_train_with_state)
  decode   tokens of the x070 model from a cached prompt state, one HIP graph per token
           (x070.X070Decoder.launch)
  prefill  prompts through the x070 model in one padded parallel pass (x070.X070Decoder.prefill_batch)
  tail     the group norm, bonus and gate behind the recurrence (kernel.wkv_tail)

Packed weights are quantised here from seeded Gaussian matrices; exact() is plain float64 torch.
"""
from __future__ import annotations

import math

import torch

from swiftrwkv_amd import kernel as K
from swiftrwkv_amd import quant as Q
from swiftrwkv_amd.synthetic import lora_ranks
from swiftrwkv_amd.x070 import Proj, RWKVState, X070Decoder

HEAD = 64
DEVICE = "cuda"
SB6 = {"sb6_4": 0, "sb6_5": 1, "sb6_6": 2}      # extra bits of the codes
SYM = {"sym_8": 8, "sym_6": 6}                  # bits of the codes
DTYPE = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


# ───────────────────────────── the cases ─────────────────────────────

def listed():
    return [
        # one token's attention projection of the smallest model: the smallest call there is
        {"name": "gemv_small", "kind": "gemv", "fmt": "sb6_4", "out": 768, "in": 768, "rows": 1},
        # the vocabulary head of the 1.5B model, one token: the largest matrix of a decode step
        {"name": "gemv_head", "kind": "gemv", "fmt": "sb6_4", "out": 65536, "in": 2048, "rows": 1},
        # an 8-bit (sym) ffn projection of eight sequences decoded together
        {"name": "gemv_batch_sym", "kind": "gemv", "fmt": "sym_8", "out": 8192, "in": 2048, "rows": 8},
        # one 128-token prompt through the 0.1B ffn key: few output tiles, a short sum
        {"name": "gemm_short", "kind": "gemm", "fmt": "sb6_4", "out": 3072, "in": 768, "groups": 1, "rows": 128,
         "epilogue": "store"},
        # a batch of ragged prompts (no multiple of any tile) through a 6-bit 0.4B r/k/v group
        {"name": "gemm_ragged", "kind": "gemm", "fmt": "sb6_6", "out": 3072, "in": 1024, "groups": 3, "rows": 1001,
         "epilogue": "store"},
        # an 8192-token prompt through the 7B-class ffn key: the largest product of a pass
        {"name": "gemm_long", "kind": "gemm", "fmt": "sb6_4", "out": 14336, "in": 4096, "groups": 1, "rows": 8192,
         "epilogue": "relu2_f16"},
        # one layer's recurrence of a 1024-token prompt, 0.1B heads, in time chunks
        {"name": "wkv_chunked", "kind": "wkv", "entry": "chunked", "batch": 1, "tokens": 1024, "heads": 12,
         "dtype": "f32", "state": False},
        # several prompts of an odd length continued from their states, step by step, 1.5B heads
        {"name": "wkv_steps", "kind": "wkv", "entry": "steps", "batch": 4, "tokens": 777, "heads": 32,
         "dtype": "f16", "state": True},
        # one layer's recurrence of a training step: 8 sequences of 4096 tokens, 1.5B heads, bf16
        {"name": "train", "kind": "train", "batch": 8, "tokens": 4096, "heads": 32, "dtype": "bf16", "state": False},
        # four tokens of the 1.5B model for one sequence: interactive decoding
        {"name": "decode_1.5B", "kind": "decode", "layers": 24, "width": 2048, "ffn": 8192, "vocab": 65536, "rows": 1,
         "tokens": 4},
        # a 128-token prompt through the 0.1B model: time to first token
        {"name": "prefill_0.1B", "kind": "prefill", "layers": 12, "width": 768, "ffn": 3072, "vocab": 65536, "rows": 1,
         "tokens": 128},
        # an 8192-token prompt through two 7B-class layers: the bulk of a long prompt
        {"name": "prefill_7B_layers", "kind": "prefill", "layers": 2, "width": 4096, "ffn": 14336, "vocab": 65536,
         "rows": 1, "tokens": 8192},
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], uniform in its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("gemv", "gemv", "gemm", "gemm", "wkv", "wkv", "train", "decode", "prefill", "prefill", "tail"))
    if kind == "gemv":
        # widths of 256 columns (the formats' super-block) and any 16-row count; batches up to 32
        while True:
            c = {"kind": kind, "fmt": rng.choice(sorted(SB6) + sorted(SYM)), "out": 16 * _log(rng, 4, 4096),
                 "in": 256 * _log(rng, 1, 56), "rows": 1 if rng.random() < 0.4 else _log(rng, 2, 32)}
            if c["out"] * c["in"] <= 1 << 27:
                return c
    if kind == "gemm":
        while True:
            groups = 3 if rng.random() < 0.3 else 1
            per = 128 * _log(rng, 2, 112)
            c = {"kind": kind, "fmt": rng.choice(sorted(SB6) + sorted(SYM)), "out": groups * per,
                 "in": 256 * _log(rng, 1, 56), "groups": groups, "rows": _log(rng, 3, 8192),
                 "epilogue": "store" if groups > 1 else rng.choice(("store", "add", "relu2_f16"))}
            if c["out"] * c["in"] <= 1 << 26 and c["out"] * c["in"] * c["rows"] <= 14336 * 4096 * 8192:
                return c
    if kind == "wkv":
        while True:
            c = {"kind": kind, "entry": rng.choice(("steps", "chunked")), "batch": _log(rng, 1, 16),
                 "tokens": _log(rng, 1, 8192), "heads": _log(rng, 1, 64), "dtype": rng.choice(sorted(DTYPE)),
                 "state": rng.random() < 0.5}
            if c["batch"] * c["tokens"] * c["heads"] <= 8192 * 64:
                return c
    if kind == "train":
        while True:
            c = {"kind": kind, "batch": _log(rng, 1, 16), "tokens": 16 * _log(rng, 1, 256), "heads": _log(rng, 1, 64),
                 "dtype": rng.choice(sorted(DTYPE)), "state": rng.random() < 0.5}
            if c["batch"] * c["tokens"] * c["heads"] <= 8 * 4096 * 32:
                return c
    if kind == "tail":
        return {"kind": kind, "rows": _log(rng, 1, 8192), "heads": _log(rng, 1, 64)}
    width = rng.choice((512, 768, 1024, 2048, 2560, 4096))
    layers = rng.randint(1, 4)
    vocab = rng.choice((2048, 16384, 65536))
    ffn = rng.choice((3, 4)) * width
    if kind == "decode":
        return {"kind": kind, "layers": layers, "width": width, "ffn": ffn, "vocab": vocab,
                "rows": 1 if rng.random() < 0.4 else _log(rng, 2, 32), "tokens": rng.randint(1, 4)}
    while True:
        c = {"kind": kind, "layers": layers, "width": width, "ffn": ffn, "vocab": vocab, "rows": _log(rng, 1, 8),
             "tokens": _log(rng, 5, 8192)}
        n = c["rows"] * c["tokens"] * layers
        if n <= 1 << 16 and n * width <= 8192 * 4096 * 2 and n * width * width <= 8192 * 4096 * 4096 * 2:
            return c


# ───────────────────────────── packed matrices ─────────────────────────────

def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _randn(g, *shape, std=1.0):
    return torch.randn(shape, generator=g, device=DEVICE) * std


def _uniform(g, lo, hi, *shape):
    return torch.rand(shape, generator=g, device=DEVICE) * (hi - lo) + lo


def _bits(plane):
    """0/1 values [..., 32] → the 4 bytes whose bit c is column c."""
    p = plane.reshape(*plane.shape[:-1], 4, 8).to(torch.int32)
    return (p << torch.arange(8, device=p.device, dtype=torch.int32)).sum(-1).to(torch.uint8)


def _pack_sb6(w, xbits):
    """Gaussian rows → (qblk, qsqm, ddm): per 32 columns a minimum and a step, both 6-bit under fp16 scales of
    256 columns; 4-bit codes in nibbles (columns c and c + 16) and a plane of bits per extra bit."""
    O, I = w.shape
    u = w.reshape(O, I // 256, 8, 32)
    mn, mx = u.amin(-1), u.amax(-1)
    step = (mx - mn) / (2 ** (4 + xbits) - 1)
    d = (step.amax(-1) / 63).half()
    dm = (mn.abs().amax(-1) / 31).half()
    qs = (step / d.float()[..., None]).round().clamp(1, 63)
    qm = (mn / dm.float()[..., None]).round().clamp(-31, 32)
    s = (qs * d.float()[..., None]).half().float()
    m = (qm * dm.float()[..., None]).half().float()
    code = ((u - m[..., None]) / s[..., None]).round().clamp(0, 2 ** (4 + xbits) - 1).to(torch.int32).reshape(O, -1, 32)
    parts = [((code[..., :16] & 15) | ((code[..., 16:] & 15) << 4)).to(torch.uint8)]
    parts += [_bits((code >> (4 + e)) & 1) for e in range(xbits)]
    qsqm = torch.stack((qs, qm), -1).to(torch.int32).to(torch.uint8).reshape(O, -1)
    return (torch.cat(parts, -1).reshape(O, -1).contiguous(), qsqm.contiguous(),
            torch.stack((d, dm), -1).reshape(O, -1).contiguous())


def _pack_sym(w, bits):
    """Gaussian rows → (qblk, qs, d): a signed 8-bit scale per 16 columns under an fp16 scale of 256."""
    O, I = w.shape
    top = 127 if bits == 8 else 31
    u = w.reshape(O, I // 256, 16, 16)
    step = u.abs().amax(-1) / top
    d = (step.amax(-1) / 127).half()
    qs = (step / d.float()[..., None]).round().clamp(1, 127)
    s = (qs * d.float()[..., None]).half().float()
    code = (u / s[..., None]).round().clamp(-top, top).to(torch.int32).reshape(O, I)
    if bits == 8:
        qblk = code.to(torch.int8).view(torch.uint8)
    else:
        c = (code + 32).reshape(O, I // 32, 2, 2, 8)
        nib = ((c[:, :, :, 0] & 15) | ((c[:, :, :, 1] & 15) << 4)).to(torch.uint8).reshape(O, I // 32, 16)
        c = c.reshape(O, I // 32, 32)
        qblk = torch.cat((nib, _bits((c >> 4) & 1), _bits((c >> 5) & 1)), -1).reshape(O, -1)
    return qblk.contiguous(), qs.to(torch.int8).view(torch.uint8).reshape(O, -1).contiguous(), d.contiguous()


def _pack(g, fmt, out, cols):
    """The packed buffers of a seeded N(0, 0.02) matrix, made in row blocks."""
    blocks = []
    for o in range(0, out, 16384):
        w = _randn(g, min(16384, out - o), cols, std=0.02)
        blocks.append(_pack_sb6(w, SB6[fmt]) if fmt in SB6 else _pack_sym(w, SYM[fmt]))
    return blocks[0] if len(blocks) == 1 else tuple(torch.cat(p) for p in zip(*blocks))


def _packed_bytes(fmt, out, cols):
    per = {"sb6_4": 18.5, "sb6_5": 22.5, "sb6_6": 26.5, "sym_8": 34.25, "sym_6": 26.25}[fmt]   # per 32 columns
    return out * cols / 32 * per


def _unbits(b):
    """4 bytes [..., 4] → 0/1 values of the 32 columns."""
    s = torch.arange(8, device=b.device, dtype=torch.int32)
    return ((b.to(torch.int32)[..., None] >> s) & 1).reshape(*b.shape[:-1], 32)


def _unpack64(fmt, bufs, out, cols):
    """The matrix that the packed bytes stand for, float64."""
    q = bufs[0]
    if fmt in SB6:
        b = q.reshape(out, cols // 32, -1)
        nib = b[..., :16].to(torch.int32)
        code = torch.cat((nib & 15, nib >> 4), -1)
        for e in range(SB6[fmt]):
            code = code | (_unbits(b[..., 16 + 4 * e:20 + 4 * e]) << (4 + e))
        sm = bufs[1].reshape(out, cols // 256, 8, 2)
        dd = bufs[2].view(torch.float16).float().reshape(out, cols // 256, 1, 2)
        s = (sm[..., 0].float() * dd[..., 0]).half().double().reshape(out, -1, 1)
        m = (sm[..., 1].contiguous().view(torch.int8).float() * dd[..., 1]).half().double().reshape(out, -1, 1)
        return (code.double() * s + m).reshape(out, cols)
    if fmt == "sym_8":
        code = q.view(torch.int8).double()
    else:
        b = q.reshape(out, cols // 32, 24)
        nib = b[..., :16].to(torch.int32).reshape(out, cols // 32, 2, 8)
        code = torch.stack((nib & 15, nib >> 4), 3).reshape(out, cols // 32, 32)
        code = (code | (_unbits(b[..., 16:20]) << 4) | (_unbits(b[..., 20:24]) << 5)).double() - 32
    s = (bufs[1].view(torch.int8).float().reshape(out, -1, 16) * bufs[2].float().reshape(out, -1, 1)).half().double()
    return (code.reshape(out, -1, 16) * s.reshape(out, -1, 1)).reshape(out, cols)


# ───────────────────────────── inputs ─────────────────────────────

def _wkv_inputs(g, B, T, H, dtype):
    """r, w, k, v, a, b as an x070 layer forms them: decays exp(-0.606531·σ), a = -kk, b = kk·σ with unit kk."""
    n = lambda std=1.0: _randn(g, B, T, H, HEAD, std=std)
    r, v, k = n(0.5), n(0.5), n(0.5)
    kk = torch.nn.functional.normalize(k, dim=-1)
    b = kk * torch.sigmoid(n())
    w = torch.exp(-0.606531 * torch.sigmoid(n()))
    return [x.to(dtype).contiguous() for x in (r, w, k, v, -kk, b)]


def _model_params(g, c):
    """The dense parameters of an x070 model (fp16 low-rank matrices and embedding) and its packed 4-bit projections."""
    D, F, V, L = c["width"], c["ffn"], c["vocab"], c["layers"]
    ranks = dict(zip("wavg", lora_ranks(D)))
    one = lambda: 1 + 0.1 * _randn(g, D)
    p = {"emb.weight": _randn(g, V, D, std=0.5).half()}
    for n in ("ln0", "ln_out"):
        p[n + ".weight"], p[n + ".bias"] = one(), _randn(g, D, std=0.1)
    proj = {}
    for l in range(L):
        b, t = f"blocks.{l}.", f"blocks.{l}.tmix."
        for n in ("ln1", "ln2"):
            p[b + n + ".weight"], p[b + n + ".bias"] = one(), _randn(g, D, std=0.1)
        for n in "rwkvag":
            p[t + "x_" + n] = _uniform(g, 0.0, 1.0, D)
        for n, r in ranks.items():
            p[t + n + "_lora_A.weight"] = _randn(g, r, D, std=D ** -0.5).half()
            p[t + n + "_lora_B.weight"] = _randn(g, D, r, std=0.5 * r ** -0.5).half()
            if n != "g":
                p[t + n + "_lora_B.bias"] = _randn(g, D, std=0.5)
        p[t + "k_k"], p[t + "k_a"], p[t + "r_k"] = one(), one(), _randn(g, D, std=0.1)
        p[t + "ln_x.weight"], p[t + "ln_x.bias"] = one(), _randn(g, D, std=0.1)
        p[b + "cmix.x_k"] = _uniform(g, 0.0, 1.0, D)
        for n in ("receptance", "key", "value", "output"):
            proj[f"{b}att.{n}.weight"] = (D, D)
        proj[b + "ffn.key.weight"], proj[b + "ffn.value.weight"] = (F, D), (D, F)
    proj["head.weight"] = (V, D)
    return p, {k: Proj("sb6", _pack(g, "sb6_4", o, i), o, i) for k, (o, i) in proj.items()}


def _model(c, seed):
    g = _gen(seed)
    dense, proj = _model_params(g, c)
    return g, dense, proj


def _prompts(c, g):
    """Prompts of ragged lengths, the first the longest."""
    lens = [c["tokens"]] + [max(1, c["tokens"] * (7 - i % 5) // 8 - i) for i in range(1, c["rows"])]
    return [torch.randint(0, c["vocab"], (n,), generator=g, device=DEVICE).tolist() for n in lens]


def _decode_inputs(c, g):
    """The cached state of the sequences' prompts and the tokens that follow."""
    L, N, D = c["layers"], c["rows"], c["width"]
    st = {"wkv": _randn(g, L, N, D // HEAD, HEAD, HEAD, std=0.3), "tmix_prev": _randn(g, L, N, D),
          "cmix_prev": _randn(g, L, N, D)}
    return st, torch.randint(0, c["vocab"], (c["tokens"], N), generator=g, device=DEVICE, dtype=torch.int32)


def _gemv_inputs(case, seed):
    g = _gen(seed)
    bufs = _pack(g, case["fmt"], case["out"], case["in"])
    return _randn(g, case["rows"], case["in"]), bufs


def _gemm_inputs(case, seed):
    g = _gen(seed)
    bufs = _pack(g, case["fmt"], case["out"], case["in"])
    x = _randn(g, case["groups"], case["rows"], case["in"]).half()
    y = _randn(g, case["rows"], case["out"]) if case["epilogue"] == "add" else None
    return x, bufs, y


def _seq_inputs(case, seed):
    g = _gen(seed)
    B, T, H = case["batch"], case["tokens"], case["heads"]
    xs = _wkv_inputs(g, B, T, H, DTYPE[case["dtype"]])
    h = _randn(g, B, H, HEAD, HEAD, std=0.1) if case["state"] else None
    gout = _randn(g, B, T, H, HEAD, std=0.5) if case["kind"] == "train" else None
    gh = _randn(g, B, H, HEAD, HEAD, std=0.1) if case["kind"] == "train" and case["state"] else None
    return xs, h, gout, gh


def _tail_inputs(case, seed):
    g = _gen(seed)
    N, H = case["rows"], case["heads"]
    rows = [_randn(g, N, H * HEAD, std=s) for s in (1.0, 0.5, 0.5, 0.5, 0.5)]       # wkv, r, k, v, gate
    return rows, [_randn(g, H * HEAD, std=0.1), 1 + 0.1 * _randn(g, H * HEAD), _randn(g, H * HEAD, std=0.1)]


# ───────────────────────────── one pass ─────────────────────────────

def prepare(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        x, bufs = _gemv_inputs(case, seed)
        return {"case": case, "x": x, "bufs": bufs}
    if kind == "gemm":
        x, bufs, y = _gemm_inputs(case, seed)
        return {"case": case, "x": x, "bufs": bufs, "y": y}
    if kind in ("wkv", "train"):
        xs, h, gout, gh = _seq_inputs(case, seed)
        if kind == "train":
            xs = [x.requires_grad_(True) for x in xs]
            h = None if h is None else h.requires_grad_(True)
        ws = None
        if case.get("entry") == "chunked":
            need = K.wkv7_chunked_workspace_bytes(case["batch"], case["tokens"], case["heads"])
            ws = torch.empty(need, dtype=torch.uint8, device=DEVICE)
        return {"case": case, "xs": xs, "h": h, "gout": gout, "gh": gh, "ws": ws}
    if kind == "tail":
        rows, vecs = _tail_inputs(case, seed)
        return {"case": case, "rows": rows, "vecs": vecs}
    g, dense, proj = _model(case, seed)
    dec = X070Decoder(case["layers"], case["width"], case["ffn"], case["vocab"], dense, proj, DEVICE)
    if kind == "prefill":
        return {"case": case, "dec": dec, "prompts": _prompts(case, g)}
    cached, tokens = _decode_inputs(case, g)
    start = dec.new_state(case["rows"])
    for n, t in cached.items():
        getattr(start, n).copy_(t)
    state, ids = start.clone(), tokens[0].clone()
    dec.launch(ids, state)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = dec.launch(ids, state)
    return {"case": case, "dec": dec, "start": start, "state": state, "ids": ids, "tokens": tokens, "graph": graph,
            "logits": logits}


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "gemv":
        if c["fmt"] in SB6:
            return Q.rwkvq_sb6_gemv(s["x"], *s["bufs"], c["out"], c["in"], SB6[c["fmt"]])
        return Q.rwkvq_sym_gemv(s["x"], *s["bufs"], c["out"], c["in"], SYM[c["fmt"]])
    if kind == "gemm":
        per = c["out"] // c["groups"]
        y = s["y"].clone() if s["y"] is not None else None       # the residual stream, added into
        if c["fmt"] in SB6:
            return Q.rwkvq_sb6_gemm(s["x"], *s["bufs"], c["out"], c["in"], SB6[c["fmt"]], per, c["epilogue"], y)
        return Q.rwkvq_sym_gemm(s["x"], *s["bufs"], c["out"], c["in"], SYM[c["fmt"]], per, c["epilogue"], y)
    if kind == "wkv":
        if c["entry"] == "chunked":
            return K.wkv7_sequence_forward_chunked(*s["xs"], s["h"], workspace=s["ws"])
        return K.wkv7_sequence_forward(*s["xs"], s["h"])
    if kind == "train":
        out, h_out = K.wkv7_train_with_state(*s["xs"], s["h"])
        wrt = s["xs"] + ([s["h"]] if s["h"] is not None else [])
        outs, cots = ((out, h_out), (s["gout"], s["gh"])) if s["gh"] is not None else ((out,), (s["gout"],))
        return out.detach(), h_out.detach(), list(torch.autograd.grad(outs, wrt, cots))
    if kind == "tail":
        wkv, r, k, v, gate = s["rows"]
        return K.wkv_tail(wkv, r, k, v, *s["vecs"], gate, c["heads"], HEAD, rows=c["rows"])
    if kind == "prefill":
        logits, st = s["dec"].prefill_batch(s["prompts"])
        return _model_out([logits], st)
    s["state"].copy_(s["start"])
    logits = []
    for tok in s["tokens"]:
        s["ids"].copy_(tok)
        s["graph"].replay()
        logits.append(s["logits"].clone())
    return _model_out(logits, s["state"])


def _model_out(logits, st: RWKVState):
    return {"logits": logits, "wkv": st.wkv, "tmix_prev": st.tmix_prev, "cmix_prev": st.cmix_prev}


# ───────────────────────────── what a pass cannot do without ─────────────────────────────

def _model_work(c, M, heads_out):
    """Bytes and operations of M token rows through the layers and `heads_out` rows through the head."""
    D, F, V, L = c["width"], c["ffn"], c["vocab"], c["layers"]
    lora = 2 * D * sum(lora_ranks(D))
    per_layer = _packed_bytes("sb6_4", 4 * D + 2 * F, D) + 2 * lora
    flops = M * L * (2 * D * (4 * D + 2 * F) + 2 * lora + 9 * HEAD * D) + 2 * heads_out * D * V
    state = 2 * L * c["rows"] * 4 * (D * HEAD + 2 * D)
    return L * per_layer + _packed_bytes("sb6_4", V, D) + 2 * M * D + state + 4 * heads_out * V, flops


def work(case):
    c, kind = case, case["kind"]
    if kind in ("gemv", "gemm"):
        M, o, i = c["rows"], c["out"], c["in"]
        if kind == "gemv":
            io = 4 * M * (i + o)
        else:
            io = 2 * c["groups"] * M * i + {"store": 4, "add": 8, "relu2_f16": 2}[c["epilogue"]] * M * o
        return {"bytes": _packed_bytes(c["fmt"], o, i) + io, "flops": 2 * M * o * i}
    if kind == "tail":
        n = c["rows"] * c["heads"] * HEAD
        return {"bytes": 4 * (6 * n + 3 * c["heads"] * HEAD), "flops": 14 * n}
    if kind in ("wkv", "train"):
        n = c["batch"] * c["tokens"] * c["heads"] * HEAD
        es = 4 if c["dtype"] == "f32" else 2
        st = 4 * c["batch"] * c["heads"] * HEAD * HEAD
        if kind == "wkv":
            return {"bytes": n * (6 * es + 4) + st * (2 if c["state"] else 1), "flops": 9 * HEAD * n}
        return {"bytes": n * (12 * es + 8) + st * (4 if c["state"] else 1), "flops": (9 + 24) * HEAD * n}
    if kind == "decode":
        b, f = _model_work(c, c["rows"], c["rows"])
        return {"bytes": c["tokens"] * b, "flops": c["tokens"] * f}
    rows = c["tokens"] + sum(max(1, c["tokens"] * (7 - i % 5) // 8 - i) for i in range(1, c["rows"]))
    b, f = _model_work(c, rows, c["rows"])
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times what another order of the same sums, or another correct rounding, was measured to change
    (the relative figures in the comments)."""
    kind = case["kind"]
    if kind == "gemv":       # 3e-7 off float64
        return {"rel": 1.2e-6}
    if kind == "gemm":       # fp32 sums rounded to fp16, now and then to the other neighbour: 1.2e-5 (doubled by relu²)
        return {"rel": 1e-4, "max": 4e-3}
    if kind == "wkv":        # steps against chunks: 4.2e-7
        return {"rel": 2e-6}
    if kind == "train":      # 1.3e-7 off float64; 16-bit gradients go to the other neighbour: 9e-5
        return {"rel": 1e-6} if case["dtype"] == "f32" else {"rel": 3e-4, "max": 1.6e-2}
    if kind == "tail":
        return {"rel": 1e-6}
    if kind == "decode":     # the low-rank branches round to fp16 at every layer: 1.6e-4 off float64
        return {"rel": 6e-4}
    return {"rel": 2.8e-3}   # every projection rounds to fp16: chunked against stepwise recurrence 6.9e-4


# ───────────────────────────── float64 ─────────────────────────────

def _wkv64(xs, h):
    """The recurrence S ← S·diag(w) + v kᵀ + (S a) bᵀ, y = S r over [B, T, H, 64] inputs; returns y and the last S."""
    B, T, H, D = xs[0].shape
    S = torch.zeros(B, H, D, D, dtype=torch.float64, device=xs[0].device) if h is None else h.detach().double()
    r, w, k, v, a, b = (x.detach() for x in xs)
    ys = []
    for t in range(T):
        S = _step64(S, *(x[:, t].double() for x in (w, k, v, a, b)))[0]
        ys.append((S @ r[:, t].double()[..., None])[..., 0])
    return torch.stack(ys, 1), S


def _step64(S, w, k, v, a, b):
    sa = S @ a[..., None]
    return S * w[..., None, :] + v[..., None] * k[..., None, :] + sa * b[..., None, :], sa[..., 0]


def _train64(xs, h, gout, gh):
    """y, the last state and the gradients of r, w, k, v, a, b (and of h), by the reverse recurrence over states
    recomputed in segments."""
    B, T, H, D = xs[0].shape
    xs = [x.detach() for x in xs]
    S = torch.zeros(B, H, D, D, dtype=torch.float64, device=xs[0].device) if h is None else h.detach().double()
    seg, starts, ys = 64, [], []
    at = lambda t: [x[:, t].double() for x in xs]
    for t in range(T):
        if t % seg == 0:
            starts.append(S)
        r, w, k, v, a, b = at(t)
        S = _step64(S, w, k, v, a, b)[0]
        ys.append((S @ r[..., None])[..., 0])
    last = S
    dS = torch.zeros_like(S) if gh is None else gh.double()
    grads = [[None] * T for _ in range(6)]
    for s0 in range((T - 1) // seg * seg, -1, -seg):
        states, sas = [starts[s0 // seg]], []
        for t in range(s0, min(T, s0 + seg)):
            _, w, k, v, a, b = at(t)
            S, sa = _step64(states[-1], w, k, v, a, b)
            states.append(S)
            sas.append(sa)
        for t in range(min(T, s0 + seg) - 1, s0 - 1, -1):
            r, w, k, v, a, b = at(t)
            before, after, sa = states[t - s0], states[t - s0 + 1], sas[t - s0]
            dy = gout[:, t].double()
            dr = (after * dy[..., None]).sum(-2)
            dS = dS + dy[..., None] * r[..., None, :]
            dsa = (dS @ b[..., None])[..., 0]
            got = (dr, (dS * before).sum(-2), (dS * v[..., None]).sum(-2), (dS @ k[..., None])[..., 0],
                   (before * dsa[..., None]).sum(-2), (dS * sa[..., None]).sum(-2))
            for n in range(6):
                grads[n][t] = got[n]
            dS = dS * w[..., None, :] + dsa[..., None] * a[..., None, :]
    return torch.stack(ys, 1), last, [torch.stack(x, 1) for x in grads] + ([dS] if h is not None else [])


def _tail64(wkv, r, k, v, r_k, lnw, lnb, gate, H):
    N = wkv.shape[0]
    y = wkv.double().reshape(N, H, HEAD)
    y = y - y.mean(-1, keepdim=True)
    y = (y / torch.sqrt((y * y).mean(-1, keepdim=True) + 64e-5)).reshape(N, -1) * lnw.double() + lnb.double()
    bonus = (r.double() * k.double() * r_k.double()).reshape(N, H, HEAD).sum(-1, keepdim=True)
    return (y + (bonus * v.double().reshape(N, H, HEAD)).reshape(N, -1)) * gate.double()


def _ln64(x, p, n):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * p[n + ".weight"].double() + p[n + ".bias"].double()


def _layer64(p, W, l, x, tprev, cprev, wkv, v_first):
    """One block over a sequence x [T, D] from its carried state: (x, the last shift rows, the state, v_first)."""
    T, D = x.shape
    H = D // HEAD
    b, t = f"blocks.{l}.", f"blocks.{l}.tmix."
    f = lambda n: p[t + n].double()
    xl = _ln64(x, p, b + "ln1")
    xx = torch.cat((tprev[None], xl[:-1])) - xl
    m = {n: xl + xx * f("x_" + n) for n in "rwkvag"}
    r, k0, v = (m[n] @ W(b + f"att.{key}.weight").T for n, key in (("r", "receptance"), ("k", "key"), ("v", "value")))
    act = {"w": torch.tanh, "a": lambda y: y, "v": lambda y: y, "g": torch.sigmoid}
    low = {n: act[n](m[n] @ f(n + "_lora_A.weight").T) @ f(n + "_lora_B.weight").T for n in "wavg"}
    if l == 0:
        v_first = v
    else:
        v = v + (v_first - v) * torch.sigmoid(low["v"] + f("v_lora_B.bias"))
    a = torch.sigmoid(low["a"] + f("a_lora_B.bias"))
    w = torch.exp(-0.606531 * torch.sigmoid(low["w"] + f("w_lora_B.bias")))
    kk = (k0 * f("k_k")).reshape(T, H, HEAD)
    kk = (kk / torch.sqrt((kk * kk).sum(-1, keepdim=True) + 1e-12)).reshape(T, D)
    k = k0 * (1 + (a - 1) * f("k_a"))
    y, wkv = _wkv64([z.reshape(1, T, H, HEAD) for z in (r, w, k, v, -kk, kk * a)], wkv[None])
    y = _tail64(y.reshape(T, D), r, k, v, f("r_k"), f("ln_x.weight"), f("ln_x.bias"), low["g"], H)
    x = x + y @ W(b + "att.output.weight").T
    xl2 = _ln64(x, p, b + "ln2")
    xk = xl2 + (torch.cat((cprev[None], xl2[:-1])) - xl2) * p[b + "cmix.x_k"].double()
    hk = torch.relu(xk @ W(b + "ffn.key.weight").T) ** 2
    return x + hk @ W(b + "ffn.value.weight").T, xl[-1], xl2[-1], wkv[0], v_first


def _model64(case, dense, proj, seqs, cached):
    """Every sequence of token ids from its cached state (None: zeros): logits of each token row asked for by the
    case (all of a decode, the last of a prompt) and the state."""
    L, D, N = case["layers"], case["width"], len(seqs)
    keep = {}

    def W(key):
        if key not in keep:
            q = proj[key]
            keep[key] = _unpack64("sb6_4", q.bufs, q.OUT, q.IN)
        return keep[key]

    z = lambda *s: torch.zeros(s, dtype=torch.float64, device=DEVICE)
    st = {"wkv": z(L, N, D // HEAD, HEAD, HEAD), "tmix_prev": z(L, N, D), "cmix_prev": z(L, N, D)}
    if cached is not None:
        st = {n: cached[n].double() for n in st}
    emb = dense["emb.weight"]
    xs = [_ln64(emb[torch.as_tensor(s, device=DEVICE, dtype=torch.long)].double(), dense, "ln0") for s in seqs]
    vf = [None] * N
    for l in range(L):
        for n in range(N):
            xs[n], st["tmix_prev"][l, n], st["cmix_prev"][l, n], st["wkv"][l, n], vf[n] = _layer64(
                dense, W, l, xs[n], st["tmix_prev"][l, n], st["cmix_prev"][l, n], st["wkv"][l, n], vf[n])
        keep.clear()
    rows = xs if case["kind"] == "decode" else [x[-1:] for x in xs]
    logits = torch.stack([_ln64(x, dense, "ln_out") @ W("head.weight").T for x in rows], 1)
    return {"logits": list(logits), **st}


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "gemv":
            x, bufs = _gemv_inputs(case, seed)
            return x.double() @ _unpack64(case["fmt"], bufs, case["out"], case["in"]).T
        if kind == "gemm":
            x, bufs, y = _gemm_inputs(case, seed)
            W = _unpack64(case["fmt"], bufs, case["out"], case["in"])
            out = torch.cat([xg.double() @ w.T for xg, w in zip(x, W.chunk(case["groups"]))], 1)
            if case["epilogue"] == "relu2_f16":
                return torch.relu(out) ** 2
            return out if y is None else out + y.double()
        if kind == "wkv":
            xs, h, _, _ = _seq_inputs(case, seed)
            return _wkv64(xs, h)
        if kind == "train":
            return _train64(*_seq_inputs(case, seed))
        if kind == "tail":
            (wkv, r, k, v, gate), vecs = _tail_inputs(case, seed)
            return _tail64(wkv, r, k, v, *vecs, gate, case["heads"])
        g, dense, proj = _model(case, seed)
        if kind == "prefill":
            return _model64(case, dense, proj, _prompts(case, g), None)
        cached, tokens = _decode_inputs(case, g)
        return _model64(case, dense, proj, tokens.T.tolist(), cached)
