"""The work that a program built on this library has it do, as cases to time.

A case is one pass through the public entry points, in the form a decoder runs
it, over one of five ranges:

  decode   one token through a few dense layers: the embedding row, then per
           layer RMSNORM -> QKV, ACT_Q8 -> O (added to the residual),
           RMSNORM -> gate/up, SILU_MUL -> ACT_Q8, down (added to the
           residual).  "eager": the frozen task table is issued on every
           token; otherwise the pass is captured once and replayed.
  verify   the layers' matrices for 2..16 columns at once (the tokens of a
           speculative verify step): ACT_Q8 and dots, one captured graph.
  head     the vocabulary projection of 1..16 columns.
  moe      1..16 tokens through mixture-of-experts layers: the F32 router
           matrix, ROUTER_SEL with the grouped gate/up, SILU_MUL -> ACT_Q8,
           the grouped down projection, WMERGE, one captured graph.
  dequant  rows of a quantized matrix to fp32 (embedding rows, or a whole
           matrix in front of a dense product over a long prompt).

Outputs accumulate (y += W x), so a pass clears its output slots first, all of
them with one call, as a decoder does before every token.
"""
import ctypes
import math

import torch

import __graft_entry__

flh = __graft_entry__._pkg()

FMT = {n: flh.Fmt[n] for n in ("F32", "Q8_0", "Q5_0", "Q4_K", "Q6_K", "IQ2_XXS", "IQ3_XXS")}
# the int8 routes of every format: the CPU's default masks, and the q8_1 bits
# that the reference's GPU masks add for the IQ formats
I8_MASK = flh.I8_MASK_DEFAULT | (1 << flh.Fmt.IQ2_XXS) | (1 << flh.Fmt.IQ3_XXS)
DEV = "cuda:0"
EPS = 1e-5
VOCAB_ROWS = 1024                                   # embedding rows that a decode case keeps

_stream = None


def _s():
    """The one stream that every pass is issued on."""
    global _stream
    if _stream is None:
        torch.cuda.init()
        flh.init(0)
        _stream = flh.Stream()
    return _stream


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # a draft model of a speculative decoder: every launch is a few
        # microseconds, the task table is issued from the host on every token
        {"name": "decode_draft_eager", "kind": "decode", "fmt": "Q4_K", "down": "Q4_K", "hidden": 1024, "ffn": 2816,
         "layers": 4, "eager": True},
        # one token through layers of the benchmark's shapes, Q4_K
        {"name": "decode_q4_K", "kind": "decode", "fmt": "Q4_K", "down": "Q4_K", "hidden": 4096, "ffn": 14336,
         "layers": 2, "eager": False},
        # the same in the 8-bit format that a user takes for accuracy
        {"name": "decode_q8_0", "kind": "decode", "fmt": "Q8_0", "down": "Q8_0", "hidden": 4096, "ffn": 14336,
         "layers": 1, "eager": False},
        # logits of one token
        {"name": "head_q6_K", "kind": "head", "fmt": "Q6_K", "rows": 128256, "hidden": 4096, "nx": 1},
        # logits of a verify step, an odd number of drafted tokens
        {"name": "head_q6_K_n5", "kind": "head", "fmt": "Q6_K", "rows": 128256, "hidden": 4096, "nx": 5},
        # verify steps of 4 and 8 tokens: one format throughout, and the usual
        # mix in which the down projection has 6 bits
        {"name": "verify4_q4_K", "kind": "verify", "fmt": "Q4_K", "down": "Q4_K", "hidden": 4096, "ffn": 14336,
         "layers": 1, "nx": 4},
        {"name": "verify8_q4_K_q6_K", "kind": "verify", "fmt": "Q4_K", "down": "Q6_K", "hidden": 4096, "ffn": 14336,
         "layers": 1, "nx": 8},
        # a verify step of a model whose sizes are no powers of two, 3 tokens
        {"name": "verify3_q8_0", "kind": "verify", "fmt": "Q8_0", "down": "Q8_0", "hidden": 5120, "ffn": 13824,
         "layers": 1, "nx": 3},
        # two of eight large experts: one token, and a batch of eight
        {"name": "moe1_q4_K", "kind": "moe", "fmt": "Q4_K", "down": "Q4_K", "hidden": 4096, "ffn": 14336, "experts": 8,
         "top_k": 2, "batch": 1, "layers": 1},
        {"name": "moe8_q4_K", "kind": "moe", "fmt": "Q4_K", "down": "Q4_K", "hidden": 4096, "ffn": 14336, "experts": 8,
         "top_k": 2, "batch": 8, "layers": 1},
        # six of 64 small experts, four tokens, the down projections in 8 bits
        {"name": "moe4_fine_q4_K_q8_0", "kind": "moe", "fmt": "Q4_K", "down": "Q8_0", "hidden": 2048, "ffn": 1536,
         "experts": 64, "top_k": 6, "batch": 4, "layers": 2},
        # a matrix to fp32, in front of a dense product over a long prompt
        {"name": "dequant_q4_K", "kind": "dequant", "fmt": "Q4_K", "rows": 14336, "cols": 4096},
    ]


def _log_int(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def draw(rng):
    """One more case of the same ranges: widths are any multiple of 256 (the
    K formats' superblock), row counts and columns are any number."""
    kind = rng.choice(["decode", "decode", "verify", "verify", "verify", "head", "moe", "moe", "dequant"])
    mixes = [("Q4_K", "Q4_K"), ("Q4_K", "Q6_K"), ("Q6_K", "Q6_K"), ("Q8_0", "Q8_0"), ("Q5_0", "Q5_0"), ("Q5_0", "Q8_0"),
             ("IQ2_XXS", "IQ3_XXS"), ("IQ3_XXS", "IQ3_XXS")]
    fmt, down = rng.choice(mixes)
    if kind in ("decode", "verify"):
        hidden = _log_int(rng, 1024, 8192, 256)
        ffn = min(16384, int(hidden * rng.uniform(2.25, 4.0) / 256) * 256)
        # enough layers that a pass reads about 60 MB or more
        per = hidden * hidden * 2.5 + 3 * hidden * ffn
        layers = max(1, min(8, int(110e6 / per)))
        c = {"kind": kind, "fmt": fmt, "down": down, "hidden": hidden, "ffn": ffn, "layers": layers}
        if kind == "decode":
            c["eager"] = rng.random() < 0.3
        else:
            c["nx"] = rng.randint(2, 16)
        return c
    if kind == "head":
        return {"kind": "head", "fmt": rng.choice(["Q6_K", "Q6_K", "Q8_0", "Q4_K"]), "rows": _log_int(rng, 32000, 152064),
                "hidden": _log_int(rng, 1024, 5120, 256), "nx": rng.choice([1, 1, 2, 3, 4, 5, 6, 8, 11, 16])}
    if kind == "moe":
        fine = rng.random() < 0.5
        hidden = _log_int(rng, 1024, 4096, 256)
        ffn = _log_int(rng, 512, 2048, 256) if fine else _log_int(rng, 4096, 14336, 256)
        # the experts' weights are at most about 0.8 GB
        bits = {"Q8_0": 8.5, "Q6_K": 6.6, "Q5_0": 5.5}.get(fmt, 4.5)
        ffn = max(256, min(ffn, int(1.4e9 * 4.5 / bits / (192 if fine else 24) / hidden / 256) * 256))
        return {"kind": "moe", "fmt": fmt, "down": down, "hidden": hidden, "ffn": ffn, "experts": 64 if fine else 8,
                "top_k": rng.randint(4, 8) if fine else 2, "batch": _log_int(rng, 1, 16), "layers": 2 if fine else 1}
    cols = _log_int(rng, 1024, 14336, 256)
    return {"kind": "dequant", "fmt": rng.choice(["Q8_0", "Q5_0", "Q4_K", "Q6_K", "IQ2_XXS", "IQ3_XXS"]),
            "rows": _log_int(rng, 64, 50000000 // cols), "cols": cols}


# ----------------------------------------------------------------- inputs --
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(seed, *shape):
    return torch.randn(*shape, generator=_gen(seed), device=DEV, dtype=torch.float32)


def _acts(seed, n, cols):
    """Activation columns: N(0, 1) with 1 % of the entries 20 times larger."""
    x = _normal(seed, n, cols)
    out = torch.rand(n, cols, generator=_gen(seed + 1), device=DEV) < 0.01
    return torch.where(out, 20.0 * x, x)


def _weights(seed, fmt, rows, cols):
    """Block bytes of a rows x cols matrix of N(0, 0.02^2) weights (Q8_0, Q4_K,
    Q6_K: the library's quantizer; Q5_0: each block scaled to its largest
    entry), or of random codebook entries, signs and group scales under block
    scales of that size (IQ2_XXS, IQ3_XXS)."""
    rb = flh.row_bytes(FMT[fmt], cols)
    if fmt in ("Q8_0", "Q4_K", "Q6_K"):
        w = torch.empty(rows * rb, dtype=torch.uint8, device=DEV)
        step = max(1, (64 << 20) // cols)
        for i, r0 in enumerate(range(0, rows, step)):
            n = min(step, rows - r0)
            src = _normal(seed + 7919 * i, n, cols).mul_(0.02)
            torch.cuda.synchronize()
            flh.quantize(FMT[fmt], src.data_ptr(), n, cols, w.data_ptr() + r0 * rb, _s())
            _s().sync()
        return w
    if fmt == "Q5_0":
        v = _normal(seed, rows * cols // 32, 32).mul_(0.02)
        top = v.gather(1, v.abs().argmax(1, keepdim=True))
        d = (top / -16.0).to(torch.float16)
        df = d.float()
        q = torch.where(df != 0, torch.round(v / df) + 16, torch.full_like(v, 16)).clamp_(0, 31).to(torch.int32)
        del v
        lo = ((q[:, :16] & 15) | ((q[:, 16:] & 15) << 4)).to(torch.uint8)
        sh = torch.arange(8, device=DEV, dtype=torch.int32)
        qh = (((q >> 4) & 1).view(-1, 4, 8) << sh).sum(2).to(torch.uint8)
        return torch.cat([d.view(torch.uint8), qh, lo], 1).reshape(-1).contiguous()
    bb = flh.BLK_BYTES[FMT[fmt]]
    b = torch.randint(0, 256, (rows * cols // 256, bb), generator=_gen(seed), device=DEV, dtype=torch.uint8)
    # an average weight is about 30 d (IQ2_XXS) or 100 d (IQ3_XXS)
    d = (torch.rand(b.shape[0], 1, generator=_gen(seed + 1), device=DEV) + 0.5).mul_(0.02 / 60).to(torch.float16)
    b[:, :2] = d.view(torch.uint8)
    return b.reshape(-1)


def _stride(cols):
    """Floats between activation columns, appendices included."""
    return ((flh.x_alloc_bytes(cols) + 127) & ~127) // 4


def _cols(x):
    """An activation buffer holding the columns x [n][cols]."""
    n, cols = x.shape
    buf = torch.zeros(n, _stride(cols), dtype=torch.float32, device=DEV)
    buf[:, :cols] = x
    return buf


class _Slots:
    """Output slots in one allocation, cleared with one call."""

    def __init__(self, sizes):
        self.at, total = {}, 0
        for name, shape in sizes:
            self.at[name] = (total, shape)
            total += (math.prod(shape) + 63) // 64 * 64
        self.mem = torch.zeros(total, dtype=torch.float32, device=DEV)

    def __getitem__(self, name):
        at, shape = self.at[name]
        return self.mem[at: at + math.prod(shape)].view(shape)

    def clear(self):
        flh.check(flh.lib().flh_zero(self.mem.data_ptr(), self.mem.numel() * 4, _s().handle))


class _State:
    """What the program keeps: buffers, and the pass as it issues it."""

    def __init__(self):
        self.graph, self.issue, self.out, self.keep = None, None, None, []

    def capture(self):
        with flh.Graph.capture(_s()) as g:
            self.issue()
        self.graph = g

    def __del__(self):
        if self.graph is not None:
            self.graph.close()


def _layer_shapes(c):
    h, f = c["hidden"], c["ffn"]
    return [("qkv", c["fmt"], h + h // 2, h), ("o", c["fmt"], h, h), ("gu", c["fmt"], 2 * f, h), ("down", c["down"], h, f)]


def _layer_seed(seed, layer, k):
    return (seed * 1009 + layer * 31 + k) * 104729 % (1 << 40)


def _decode_inputs(c, seed):
    h = c["hidden"]
    layers = []
    for l in range(c["layers"]):
        d = {n: _weights(_layer_seed(seed, l, k), fmt, r, cc) for k, (n, fmt, r, cc) in enumerate(_layer_shapes(c))}
        d["wn1"] = 1.0 + 0.1 * _normal(_layer_seed(seed, l, 10), h)
        d["wn2"] = 1.0 + 0.1 * _normal(_layer_seed(seed, l, 11), h)
        d["attn"] = _acts(_layer_seed(seed, l, 12), 1, h)
        layers.append(d)
    emb = _weights(_layer_seed(seed, 99, 0), "Q8_0", VOCAB_ROWS, h)
    return layers, emb, seed % VOCAB_ROWS


def _decode(c, seed):
    h, f = c["hidden"], c["ffn"]
    layers, emb, token = _decode_inputs(c, seed)
    st = _State()
    x = torch.zeros(h, dtype=torch.float32, device=DEV)
    slots = _Slots([(f"qkv{l}", (h + h // 2,)) for l in range(c["layers"])] +
                   [(f"gu{l}", (2 * f,)) for l in range(c["layers"])])
    xn = _cols(torch.zeros(1, h, device=DEV))
    hb = _cols(torch.zeros(1, f, device=DEV))
    attn = [_cols(d["attn"]) for d in layers]
    row = emb.data_ptr() + token * flh.row_bytes(FMT["Q8_0"], h)
    shapes = {n: (FMT[fmt], r, cc) for n, fmt, r, cc in _layer_shapes(c)}
    st.keep = [layers, emb, x, slots, xn, hb, attn]
    st.out = {"x": x}
    for l in range(c["layers"]):
        st.out[f"qkv{l}"], st.out[f"gu{l}"] = slots[f"qkv{l}"], slots[f"gu{l}"]

    def start():
        slots.clear()
        flh.dequant(FMT["Q8_0"], row, 1, h, x.data_ptr(), _s())

    if c["eager"]:
        # the table as the graph builder freezes it: row tiles of 512 rows
        tasks, params = [], []

        def task(kind, **kw):
            t = flh.Task(kind=int(kind), id=len(tasks))
            for k, v in kw.items():
                setattr(t, k, v)
            tasks.append(t)

        def param(p):
            b = flh.HostBuffer(256)
            ctypes.memmove(b.ptr, ctypes.addressof(p), ctypes.sizeof(p))
            params.append(b)
            return b.ptr

        def act(buf, cols):
            task(flh.TaskKind.ACT_Q8, x=buf.data_ptr(), y=buf.data_ptr() + flh.xq_offset(cols), cols=cols, rows=cols // 32)

        def dot(name, w, buf, y):
            fmt, r, cc = shapes[name]
            rb = flh.row_bytes(fmt, cc)
            for r0 in range(0, r, 512):
                n = min(512, r - r0)
                task(flh.TaskKind.STREAM_DOT, fmt=int(fmt), w=w.data_ptr() + r0 * rb, w_bytes=n * rb, x=buf.data_ptr(),
                     y=y.data_ptr() + 4 * r0, rows=n, cols=cc, nx=1)

        for l, d in enumerate(layers):
            qkv, gu = slots[f"qkv{l}"], slots[f"gu{l}"]
            for wn, name, y in (("wn1", "qkv", qkv), ("wn2", "gu", gu)):
                if name == "gu":
                    act(attn[l], h)
                    dot("o", d["o"], attn[l], x)
                task(flh.TaskKind.RMSNORM, aux=param(flh.RmsNormP(d[wn].data_ptr(), x.data_ptr(), xn.data_ptr(), EPS, h)))
                act(xn, h)
                dot(name, d[name], xn, y)
            task(flh.TaskKind.SILU_MUL, aux=param(flh.SiluMulP(gu.data_ptr(), gu.data_ptr() + 4 * f, hb.data_ptr(), f)))
            act(hb, f)
            dot("down", d["down"], hb, x)
        table = (flh.Task * len(tasks))(*tasks)
        st.keep += [table, params]

        def issue():
            start()
            flh.check(flh.lib().flh_exec_tasks(ctypes.addressof(table), len(table), 1, I8_MASK, flh.I8K_MASK_DEFAULT,
                                               _s().handle))
        st.issue = issue
        return st

    def issue():
        start()
        s = _s()
        for l, d in enumerate(layers):
            qkv, gu = slots[f"qkv{l}"], slots[f"gu{l}"]
            flh.rmsnorm_stream_dot(shapes["qkv"][0], d["qkv"].data_ptr(), *shapes["qkv"][1:], x.data_ptr(),
                                   d["wn1"].data_ptr(), EPS, xn.data_ptr(), qkv.data_ptr(), s, i8_mask=I8_MASK)
            flh.act_q8_stream_dot(shapes["o"][0], d["o"].data_ptr(), *shapes["o"][1:], attn[l].data_ptr(), x.data_ptr(),
                                  s, i8_mask=I8_MASK)
            flh.rmsnorm_stream_dot(shapes["gu"][0], d["gu"].data_ptr(), *shapes["gu"][1:], x.data_ptr(),
                                   d["wn2"].data_ptr(), EPS, xn.data_ptr(), gu.data_ptr(), s, i8_mask=I8_MASK)
            flh.silu_mul_act_q8(gu.data_ptr(), gu.data_ptr() + 4 * f, hb.data_ptr(), f, 1, 2 * f, _stride(f), s)
            flh.stream_dot(shapes["down"][0], d["down"].data_ptr(), *shapes["down"][1:], hb.data_ptr(), x.data_ptr(), s,
                           i8_mask=I8_MASK)
    st.issue = issue
    return st


def _verify_inputs(c, seed):
    layers = []
    for l in range(c["layers"]):
        d = {n: _weights(_layer_seed(seed, l, k), fmt, r, cc) for k, (n, fmt, r, cc) in enumerate(_layer_shapes(c))}
        for k, n in enumerate(("xq", "xo", "xg")):
            d[n] = _acts(_layer_seed(seed, l, 20 + 2 * k), c["nx"], c["hidden"])
        layers.append(d)
    return layers


def _verify(c, seed):
    h, f, nx = c["hidden"], c["ffn"], c["nx"]
    layers = _verify_inputs(c, seed)
    st = _State()
    sizes = []
    for l in range(c["layers"]):
        sizes += [(f"{n}{l}", (nx, r)) for n, _, r, _ in _layer_shapes(c)]
    slots = _Slots(sizes)
    bufs = [{n: _cols(d[n]) for n in ("xq", "xo", "xg")} for d in layers]
    hb = _cols(torch.zeros(nx, f, device=DEV))
    st.keep = [layers, slots, bufs, hb]
    st.out = {n: slots[n] for n, _ in sizes}

    def issue():
        slots.clear()
        s = _s()
        for l, d in enumerate(layers):
            for (n, fmt, r, cc), xn in zip(_layer_shapes(c), ("xq", "xo", "xg", None)):
                y = slots[f"{n}{l}"]
                if xn is None:
                    g = slots[f"gu{l}"]
                    flh.silu_mul_act_q8(g.data_ptr(), g.data_ptr() + 4 * f, hb.data_ptr(), f, nx, 2 * f, _stride(f), s)
                    b = hb
                else:
                    b = bufs[l][xn]
                    flh.act_q8(b.data_ptr(), cc, s, nx=nx, xstride=_stride(cc))
                flh.stream_dot(FMT[fmt], d[n].data_ptr(), r, cc, b.data_ptr(), y.data_ptr(), s, nx=nx, xstride=_stride(cc),
                               ystride=r, i8_mask=I8_MASK)
    st.issue = issue
    return st


def _head(c, seed):
    h, r, nx = c["hidden"], c["rows"], c["nx"]
    w = _weights(seed, c["fmt"], r, h)
    x = _acts(seed + 5, nx, h)
    wn = 1.0 + 0.1 * _normal(seed + 9, h)
    st = _State()
    xb, xn = _cols(x), _cols(torch.zeros(nx, h, device=DEV))
    slots = _Slots([("logits", (nx, r))])
    st.keep = [w, xb, xn, wn, slots]
    st.out = {"logits": slots["logits"]}

    def issue():
        slots.clear()
        s = _s()
        if nx == 1:
            flh.rmsnorm_stream_dot(FMT[c["fmt"]], w.data_ptr(), r, h, xb.data_ptr(), wn.data_ptr(), EPS, xn.data_ptr(),
                                   slots["logits"].data_ptr(), s)
        else:
            flh.act_q8(xb.data_ptr(), h, s, nx=nx, xstride=_stride(h))
            flh.stream_dot(FMT[c["fmt"]], w.data_ptr(), r, h, xb.data_ptr(), slots["logits"].data_ptr(), s, nx=nx,
                           xstride=_stride(h), ystride=r)
    st.issue = issue
    return st


def _moe_inputs(c, seed):
    h, f, e, n = c["hidden"], c["ffn"], c["experts"], c["batch"]
    layers = []
    for l in range(c["layers"]):
        layers.append({"router": _normal(_layer_seed(seed, l, 1), e, h).mul_(0.05),
                       "gu": _weights(_layer_seed(seed, l, 2), c["fmt"], e * 2 * f, h),
                       "down": _weights(_layer_seed(seed, l, 3), c["down"], e * h, f),
                       "x": _normal(_layer_seed(seed, l, 4), n, h),
                       "res": _normal(_layer_seed(seed, l, 5), n, h)})
    return layers


def _moe(c, seed):
    h, f, e, k, n = c["hidden"], c["ffn"], c["experts"], c["top_k"], c["batch"]
    layers = _moe_inputs(c, seed)
    st = _State()
    sizes = []
    for l in range(c["layers"]):
        sizes += [(f"logits{l}", (n, e)), (f"gu{l}", (n * k, 2 * f)), (f"down{l}", (n * k, h))]
    slots = _Slots(sizes)
    xb = [_cols(d["x"]) for d in layers]
    hb = _cols(torch.zeros(n * k, f, device=DEV))
    ids = [torch.zeros(n, k, dtype=torch.int32, device=DEV) for _ in layers]
    gates = [torch.zeros(n, k, dtype=torch.float32, device=DEV) for _ in layers]
    y = [torch.zeros(n, h, dtype=torch.float32, device=DEV) for _ in layers]
    st.keep = [layers, slots, xb, hb, ids, gates, y]
    st.out = {nm: slots[nm] for nm, _ in sizes}
    for l in range(c["layers"]):
        st.out.update({f"ids{l}": ids[l], f"gates{l}": gates[l], f"y{l}": y[l]})
    gb, db = 2 * f * flh.row_bytes(FMT[c["fmt"]], h), h * flh.row_bytes(FMT[c["down"]], f)

    def issue():
        slots.clear()
        s = _s()
        for l, d in enumerate(layers):
            lg, gu, dn = slots[f"logits{l}"], slots[f"gu{l}"], slots[f"down{l}"]
            flh.act_q8(xb[l].data_ptr(), h, s, nx=n, xstride=_stride(h))
            flh.stream_dot(FMT["F32"], d["router"].data_ptr(), e, h, xb[l].data_ptr(), lg.data_ptr(), s, nx=n,
                           xstride=_stride(h), ystride=e)
            flh.router_moe_dot(FMT[c["fmt"]], d["gu"].data_ptr(), gb, 2 * f, h, lg.data_ptr(), n, e, k, 1, 1.0,
                               ids[l].data_ptr(), gates[l].data_ptr(), xb[l].data_ptr(), _stride(h), False,
                               gu.data_ptr(), 2 * f, s)
            flh.silu_mul_act_q8(gu.data_ptr(), gu.data_ptr() + 4 * f, hb.data_ptr(), f, n * k, 2 * f, _stride(f), s)
            flh.moe_dot(FMT[c["down"]], d["down"].data_ptr(), db, h, f, ids[l].data_ptr(), n, k, e, hb.data_ptr(),
                        _stride(f), True, dn.data_ptr(), h, s)
            flh.wmerge(dn.data_ptr(), gates[l].data_ptr(), d["res"].data_ptr(), None, y[l].data_ptr(), 1.0, k, h, 0, n,
                       k * h, h, s)
    st.issue = issue
    return st


def _dequant(c, seed):
    w = _weights(seed, c["fmt"], c["rows"], c["cols"])
    st = _State()
    out = torch.zeros(c["rows"], c["cols"], dtype=torch.float32, device=DEV)
    st.keep, st.out = [w], {"w": out}
    st.issue = lambda: flh.dequant(FMT[c["fmt"]], w.data_ptr(), c["rows"], c["cols"], out.data_ptr(), _s())
    return st


def prepare(case, seed):
    _s()
    st = {"decode": _decode, "verify": _verify, "head": _head, "moe": _moe, "dequant": _dequant}[case["kind"]](case, seed)
    torch.cuda.synchronize()
    if case["kind"] != "dequant" and not case.get("eager"):
        st.capture()
    return st


def run(state):
    if state.graph is not None:
        state.graph.launch()
    else:
        state.issue()
    return state.out


# ------------------------------------------------------------------- work --
def work(case):
    def mat(fmt, r, cc):
        return r * flh.row_bytes(FMT[fmt], cc)

    kind = case["kind"]
    if kind in ("decode", "verify"):
        nx = case.get("nx", 1)
        shapes = _layer_shapes(case)
        by = sum(mat(fmt, r, cc) + 4 * nx * (r + cc) for _, fmt, r, cc in shapes)
        fl = sum(2 * nx * r * cc for _, _, r, cc in shapes)
        return {"bytes": by * case["layers"], "flops": fl * case["layers"]}
    if kind == "head":
        r, h, nx = case["rows"], case["hidden"], case["nx"]
        return {"bytes": mat(case["fmt"], r, h) + 4 * nx * (r + h), "flops": 2 * nx * r * h}
    if kind == "moe":
        h, f, e, k, n = (case[x] for x in ("hidden", "ffn", "experts", "top_k", "batch"))
        hit = e * (1 - (1 - k / e) ** n)                 # experts that some token takes, on average
        by = hit * (mat(case["fmt"], 2 * f, h) + mat(case["down"], h, f)) + 4 * e * h + 4 * n * (3 * h + e + k * (4 * f + 2 * h))
        return {"bytes": by * case["layers"], "flops": 2 * n * (e * h + k * 3 * f * h) * case["layers"]}
    n = case["rows"] * case["cols"]
    return {"bytes": mat(case["fmt"], case["rows"], case["cols"]) + 4 * n, "flops": 2 * n}


def tolerance(case):
    """Dots: 32-bit sums of exact integer products, about 4 times the 2-norm
    error of that against 64 bits.  Where a pass feeds one layer's sums into the
    next one's 8-bit activations, a last-bit difference moves some of them to
    the neighbouring step."""
    if case["kind"] == "dequant":
        return {"rel": 1e-6, "max": 1e-5}
    if case["kind"] == "head" and case["nx"] > 1:
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 1e-3, "max": 0.05}


# ------------------------------------------------- the same in 64 bits -----
def _halves(b):
    return b.contiguous().view(torch.float16).double()


def _unpack(w, fmt, rows, cols):
    """fp64 weights [rows][cols] of block bytes."""
    if fmt == "Q8_0":
        b = w.view(-1, 34)
        v = _halves(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "Q5_0":
        b = w.view(-1, 22)
        sh = torch.arange(8, device=w.device, dtype=torch.uint8)
        hi = ((b[:, 2:6].unsqueeze(2) >> sh) & 1).reshape(-1, 32).to(torch.int16) << 4
        lo = torch.cat([b[:, 6:] & 15, b[:, 6:] >> 4], 1).to(torch.int16)
        v = _halves(b[:, :2]) * ((lo | hi) - 16).double()
    elif fmt == "Q4_K":
        b = w.view(-1, 144)
        d, m, s = _halves(b[:, 0:2]), _halves(b[:, 2:4]), b[:, 4:16].to(torch.int16)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].view(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).view(-1, 8, 32).double()
        v = (d * sc).unsqueeze(2) * q - (m * mn).unsqueeze(2)
    else:                                                # Q6_K
        b = w.view(-1, 210)
        ql, qh = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)            # [block][half][4][32]
        hi = torch.cat([(qh >> (2 * g)) & 3 for g in range(4)], 2)
        q = (lo | (hi << 4)).to(torch.int16) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(-1, 16, 1)
        v = _halves(b[:, 208:210]).view(-1, 1, 1) * sc * q.reshape(-1, 16, 16).double()
    return v.reshape(rows, cols)


def _act(x, fmt):
    """The 8-bit activations that a dot of this format multiplies, as fp64."""
    n = 32 if fmt in ("Q8_0", "Q5_0") else 256
    v = x.float().reshape(-1, n)
    top = v.abs().amax(1, keepdim=True)
    d = top / 127.0
    y = v * torch.where(top > 0, 127.0 / top, torch.zeros_like(top))
    q = torch.sign(y) * torch.floor(y.abs().double() + 0.5)
    d = d.to(torch.float16).double() if n == 32 else d.double()
    return (q.clamp(-127, 127) * d).reshape(x.shape)


def _mul(w, fmt, rows, cols, x):
    """x [n][cols] (already 8-bit) times the matrix: [n][rows] in fp64."""
    rb = flh.row_bytes(FMT[fmt], cols)
    step = max(1, (32 << 20) // cols)
    return torch.cat([x @ _unpack(w[r0 * rb: min(rows, r0 + step) * rb], fmt, min(step, rows - r0), cols).T
                      for r0 in range(0, rows, step)], 1)


def _rms(x, wn):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * wn.double()


def _silu(g, u):
    return g / (1 + torch.exp(-g)) * u


def exact(case, seed):
    fmts = {case["fmt"], case.get("down", case["fmt"])}
    if fmts & {"IQ2_XXS", "IQ3_XXS"}:
        return None                                      # their codebooks are in the library only
    _s()
    kind, fmt = case["kind"], case["fmt"]
    if kind == "dequant":
        return {"w": _unpack(_weights(seed, fmt, case["rows"], case["cols"]), fmt, case["rows"], case["cols"])}
    out = {}
    if kind == "head":
        h, r, nx = case["hidden"], case["rows"], case["nx"]
        w, x = _weights(seed, fmt, r, h), _acts(seed + 5, nx, h).double()
        if nx == 1:
            x = _rms(x, 1.0 + 0.1 * _normal(seed + 9, h))
        return {"logits": _mul(w, fmt, r, h, _act(x, fmt))}
    f, h = case["ffn"], case["hidden"]
    if kind == "decode":
        layers, emb, token = _decode_inputs(case, seed)
        rb = flh.row_bytes(FMT["Q8_0"], h)
        x = _unpack(emb[token * rb: (token + 1) * rb], "Q8_0", 1, h)
        for l, d in enumerate(layers):
            q = _mul(d["qkv"], fmt, h + h // 2, h, _act(_rms(x, d["wn1"]), fmt))
            x = x + _mul(d["o"], fmt, h, h, _act(d["attn"], fmt))
            g = _mul(d["gu"], fmt, 2 * f, h, _act(_rms(x, d["wn2"]), fmt))
            x = x + _mul(d["down"], case["down"], h, f, _act(_silu(g[:, :f], g[:, f:]), case["down"]))
            out[f"qkv{l}"], out[f"gu{l}"] = q[0], g[0]
        out["x"] = x[0]
        return out
    if kind == "verify":
        for l, d in enumerate(_verify_inputs(case, seed)):
            for (n, ft, r, cc), xn in zip(_layer_shapes(case), ("xq", "xo", "xg", None)):
                if xn is None:
                    g = out[f"gu{l}"]
                    x = _silu(g[:, :f], g[:, f:])
                else:
                    x = d[xn]
                out[f"{n}{l}"] = _mul(d[n], ft, r, cc, _act(x, ft))
        return out
    e, k, n = case["experts"], case["top_k"], case["batch"]
    gb, db = 2 * f * flh.row_bytes(FMT[fmt], h), h * flh.row_bytes(FMT[case["down"]], f)
    for l, d in enumerate(_moe_inputs(case, seed)):
        lg = d["x"].double() @ d["router"].double().T
        p = torch.softmax(lg, 1)
        gate, ids = torch.topk(p, k, dim=1)
        gate = gate / gate.sum(1, keepdim=True)
        xq = _act(d["x"], fmt)
        gu = torch.zeros(n * k, 2 * f, dtype=torch.float64, device=DEV)
        dn = torch.zeros(n * k, h, dtype=torch.float64, device=DEV)
        flat = ids.reshape(-1)
        for ex in sorted(set(flat.tolist())):
            at = (flat == ex).nonzero().reshape(-1)
            gu[at] = _mul(d["gu"][ex * gb: (ex + 1) * gb], fmt, 2 * f, h, xq[at // k])
            hh = _silu(gu[at, :f], gu[at, f:])
            dn[at] = _mul(d["down"][ex * db: (ex + 1) * db], case["down"], h, f, _act(hh, case["down"]))
        y = d["res"].double() + (gate.unsqueeze(2) * dn.view(n, k, h)).sum(1)
        out.update({f"logits{l}": lg, f"gu{l}": gu, f"down{l}": dn, f"ids{l}": None, f"gates{l}": gate, f"y{l}": y})
    return out
