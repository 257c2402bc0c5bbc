"""Performance cases of the BFP8 W8A16 library: what its users have it do.

A case is a dict of plain values; its "kind" says which path of the library
it takes, the rest are sizes:

  gemv     one GEMV of a decode step through a plan (x float32 -> y float32)
  sweep    a decode token's independent GEMVs, and the fused lm_head, in one plan
  lm_head  the BFP8 lm_head with its top-k through a plan
  batch    B quantized activation vectors against one matrix
  bf16     the bf16 tied-embedding lm_head's top-k, then the sampler
  layer    the reference's forward_linear_layer / forward_mlp on host vectors
  token    forward_token_c over a few tokens, then the chat front end's
           final norm and top-k of the last one
  pack     the weight converter, reference planes -> GPU planes, or back

The shapes are the model's (hidden 1024, MLP 3584, conv channels 6144,
vocabulary 65536, 24 layers) where a case names one, else generic.  Every path
is bit-exact by contract (identical to the reference's arithmetic order), so
outputs are compared bit for bit.

exact() restates each path in 64 bits: the activation quantizer (int16 blocks
are part of the W8A16 format) followed by products and sums in double.
"""
import ctypes
import math
import mmap
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "qwen35-ax7020-edge-llm_amd"))
import qwen_kernels_gpu as qk  # noqa: E402

HIDDEN, MLP, CONV, HEADS, HEAD_DIM, VOCAB, LAYERS = 1024, 3584, 6144, 16, 128, 65536, 24
HD = HEADS * HEAD_DIM
EPS = 1e-6

# the GEMVs of one layer of the decode sweep, and of the forward's layers
SWEEP_LAYER = ((3584, 1024), (3584, 1024), (1024, 3584), (6144, 1024), (1024, 2048))
LINEAR = (("qkv", CONV, HIDDEN), ("z", HD, HIDDEN), ("o", HIDDEN, HD),
          ("gate", MLP, HIDDEN), ("up", MLP, HIDDEN), ("down", HIDDEN, MLP))
FULL = LINEAR[3:]
# the full-attention callback's own GEMVs (q with its gate, k, v, o)
CALLBACK = (("q", 4096, 1024), ("k", 512, 1024), ("v", 512, 1024), ("o", 1024, 2048))


def listed():
    return [
        # the smallest call: a lone down projection of a decode step
        {"name": "gemv_down", "kind": "gemv", "M": 1024, "K": 3584},
        # one decode token's weights: 24 layers' GEMVs and the lm_head's top-40
        {"name": "sweep_24", "kind": "sweep", "layers": 24, "k": 40},
        # greedy / top-40 sampling head on its own
        {"name": "lm_head_40", "kind": "lm_head", "vocab": 65536, "K": 1024, "k": 40},
        # wide sampling over an odd vocabulary (re-ranking, n-best)
        {"name": "lm_head_wide", "kind": "lm_head", "vocab": 50001, "K": 1024, "k": 200},
        # serving sixteen sequences: a gate projection, and the head's logits
        {"name": "batch16_gate", "kind": "batch", "M": 3584, "K": 1024, "B": 16},
        {"name": "batch16_head", "kind": "batch", "M": 65536, "K": 1024, "B": 16},
        # a handful of sequences on a long-K matrix with an odd row count
        {"name": "batch5_odd", "kind": "batch", "M": 2049, "K": 3584, "B": 5},
        # the chat front end's step on the device: scores, top-64, draw
        {"name": "bf16_head_64", "kind": "bf16", "vocab": 65536, "hidden": 1024, "k": 64, "layout": "tiles"},
        # one linear-attention layer over four tokens
        {"name": "linear_layer", "kind": "layer", "layers": 1, "linear": True, "tokens": 4, "resident": True},
        # a four-token prompt through the 24 layers
        {"name": "token_4", "kind": "token", "tokens": 4, "k": 64, "attention": False},
        # decode as the engine runs it: its full-attention layers call back
        {"name": "token_attention", "kind": "token", "tokens": 1, "k": 40, "attention": True},
        # loading: the largest tensor of the image to the GPU layout
        {"name": "pack_lm_head", "kind": "pack", "M": 65536, "K": 1024, "back": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("gemv", "sweep", "lm_head", "lm_head", "batch", "batch", "bf16", "layer", "token", "pack"))
    c = {"kind": kind}
    if kind == "gemv":
        c.update(M=_log(rng, 64, 65536), K=rng.choice((rng.randint(1, 64) * 64, rng.randint(64, 4096))))
    elif kind == "sweep":
        c.update(layers=rng.randint(1, 24), k=rng.choice((0, 1, rng.randint(2, 64))))
    elif kind == "lm_head":
        c.update(vocab=_log(rng, 1000, 65536), K=rng.choice((512, 768, 1024, 1024, 1536, 2048)),
                 k=rng.choice((1, rng.randint(2, 64), rng.randint(65, 500))))
    elif kind == "batch":
        c.update(M=_log(rng, 64, 65536), K=rng.choice((1024, rng.randint(1, 56) * 64, rng.randint(64, 3584))),
                 B=rng.randint(1, 16))
        if c["M"] > 16384:
            c["K"] = min(c["K"], 1024)
    elif kind == "bf16":
        c.update(vocab=_log(rng, 1000, 65536), hidden=1024, k=rng.randint(1, 64), layout=rng.choice(("tiles", "rows")))
        if c["layout"] == "rows":
            c["hidden"] = rng.choice((1024, rng.randint(128, 1200)))
    elif kind == "layer":
        c.update(layers=rng.randint(1, 6), linear=rng.random() < 0.7, tokens=rng.randint(1, 8),
                 resident=rng.random() < 0.7)
    elif kind == "token":
        c.update(tokens=rng.randint(1, 3), k=rng.randint(1, 64), attention=False)
        if rng.random() < 0.3:
            c.update(tokens=1, attention=True)
    else:
        c.update(M=_log(rng, 64, 65536), K=rng.randint(1, 16) * 64, back=rng.random() < 0.3)
    return c


# ---- inputs, from the seed alone -------------------------------------------------------
def _gen(seed, stream):
    return torch.Generator(device="cuda").manual_seed((seed * 1000003 + stream * 7919) & 0x7FFFFFFFFFFF)


def _planes(g, M, K, lo, hi):
    """Reference planes: mantissas uniform in [-127, 127], a block's exponent in
    [lo, hi] (scale 2^(e - 134): weights of a few hundredths)."""
    mant = torch.randint(-127, 128, (M, K), dtype=torch.int8, device="cuda", generator=g)
    exps = torch.randint(lo, hi + 1, (M, K // 64), dtype=torch.uint8, device="cuda", generator=g)
    return mant, exps


def _normal(g, *shape):
    return torch.randn(*shape, dtype=torch.float32, device="cuda", generator=g)


def _activation(g, K, swiglu):
    """A norm's output, or (down projections) a swiglu's with its outliers."""
    x = _normal(g, K)
    if swiglu:
        x = x / (1 + torch.exp(-x)) * _normal(g, K)
        far = torch.rand(K, device="cuda", generator=g) < 0.01
        x = torch.where(far, torch.sign(_normal(g, K)) * 20.0, x)
    return x.contiguous()


def _sweep_items(case):
    items = [(M, K, 124, 130) for _ in range(case["layers"]) for M, K in SWEEP_LAYER]
    return items + ([(VOCAB, HIDDEN, 122, 128)] if case["k"] else [])


class _Image:
    """A read-only mapping in host memory, as the engine's mmap of its weight
    image: tensors are placed at 64-byte offsets, then the pages protected.
    The mapping lives as long as the process, as the engine's does (the
    library keeps device copies by host address)."""

    live = []

    def __init__(self, nbytes):
        self.map = mmap.mmap(-1, nbytes)
        self.buf = np.frombuffer(self.map, dtype=np.uint8)
        self.at = 0
        _Image.live.append(self)

    def put(self, t):
        n = t.numel() * t.element_size()
        view = self.buf[self.at:self.at + n]
        torch.from_numpy(view).copy_(t.contiguous().view(torch.uint8).view(-1))
        self.at += (n + 63) & ~63
        return view.ctypes.data

    def protect(self):
        libc = ctypes.CDLL(None)
        libc.mprotect.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
        if libc.mprotect(self.buf.ctypes.data, len(self.buf), mmap.PROT_READ) != 0:
            raise OSError("mprotect of the weight image failed")


_host_keep = []  # parameters and states in host memory, which the library also knows by address


def _host(a):
    a = np.ascontiguousarray(a)
    _host_keep.append(a)
    return a


def _layer_inputs(seed, l, linear):
    """Planes and float parameters of one layer (device tensors / host arrays)."""
    g = _gen(seed, 100 + l)
    w = {n: _planes(g, M, K, 122, 126) for n, M, K in (LINEAR if linear else FULL)}
    p = {"post_ln_w": _normal(g, HIDDEN) * 0.1}
    if linear:
        p.update(in_ln_w=_normal(g, HIDDEN) * 0.1, conv_w=_normal(g, CONV, 4) * 0.5,
                 wa=_normal(g, HEADS, HIDDEN) * 0.03, wb=_normal(g, HEADS, HIDDEN) * 0.03,
                 nea=-(0.2 + 2.8 * torch.rand(HEADS, device="cuda", generator=g)),
                 dt=4 * torch.rand(HEADS, device="cuda", generator=g) - 2, norm_w=_normal(g, HEAD_DIM) * 0.5)
    return w, p


def _layer_bytes(linear):
    return sum(M * K + M * (K // 64) + 128 for _, M, K in (LINEAR if linear else FULL))


def _fill_plan(plan, image, w, p, linear):
    for n, M, K in (LINEAR if linear else FULL):
        setattr(plan, "mant_" + n, image.put(w[n][0]))
        setattr(plan, "exp_" + n, image.put(w[n][1]))
        setattr(plan, "M_" + n, M)
        setattr(plan, "K_" + n, K)
    for n, v in p.items():
        setattr(plan, n, _host(v.cpu().numpy()).ctypes.data)
    if not linear:
        return None
    conv, rec = _host(np.zeros((3, CONV), np.float32)), _host(np.zeros((HEADS, HEAD_DIM * HEAD_DIM), np.float32))
    plan.conv_s, plan.state = conv.ctypes.data, rec.ctypes.data
    return conv, rec


def _table(seed, vocab, hidden):
    """A bf16 embedding table's bits (int16), entries of a few hundredths."""
    return (_normal(_gen(seed, 7), vocab, hidden) * 0.05).to(torch.bfloat16).view(torch.int16)


def _is_full(l):
    return l % 4 == 3  # three linear-attention layers, then a full-attention one


# ---- prepare ---------------------------------------------------------------------------
def prepare(case, seed):
    lib = qk.load()
    lib.init_kernels()
    kind = case["kind"]
    if kind == "gemv":
        M, K = case["M"], case["K"]
        g = _gen(seed, 1)
        mat = qk.DeviceMatrix.from_soa(*_ragged(_planes(g, M, K // 64 * 64, 124, 130), K))
        x, y = _activation(g, K, K > 2048), torch.empty(M, dtype=torch.float32, device="cuda")
        return {"kind": kind, "plan": qk.SweepPlan([{"x": x, "mat": mat, "y": y}]), "y": y}
    if kind == "sweep":
        items, ys = [], torch.empty(sum(M for M, *_ in _sweep_items(case)), dtype=torch.float32, device="cuda")
        at = 0
        for i, (M, K, lo, hi) in enumerate(_sweep_items(case)):
            g = _gen(seed, 10 + i)
            it = {"mat": qk.DeviceMatrix.from_soa(*_planes(g, M, K, lo, hi)), "x": _activation(g, K, K > 2048)}
            if M == VOCAB:
                it["topk"] = case["k"]
            else:
                it["y"] = ys[at:at + M]
                at += M
            items.append(it)
        plan = qk.SweepPlan(items)
        return {"kind": kind, "plan": plan, "out": [ys[:at]] + list(plan.topk_out or ())}
    if kind == "lm_head":
        g = _gen(seed, 2)
        mat = qk.DeviceMatrix.from_soa(*_planes(g, case["vocab"], case["K"], 122, 128))
        plan = qk.SweepPlan([{"x": _activation(g, case["K"], False), "mat": mat, "topk": case["k"]}])
        return {"kind": kind, "plan": plan, "out": list(plan.topk_out)}
    if kind == "batch":
        M, K, B = case["M"], case["K"], case["B"]
        nb = K // 64
        g = _gen(seed, 3)
        mat = qk.DeviceMatrix.from_soa(*_ragged(_planes(g, M, nb * 64, 124, 130), K))
        xs = torch.empty((B, nb), dtype=torch.float32, device="cuda")
        xsp = torch.empty((B, nb * 32), dtype=torch.int32, device="cuda")
        for b in range(B):  # the vectors come quantized, as the layer before leaves them
            _, s, p = qk.quantize(_activation(g, K, K > 2048))
            xs[b], xsp[b] = s, p
        Y = torch.empty((B, M), dtype=torch.float32, device="cuda")
        return {"kind": kind, "mat": mat, "xs": xs, "xsp": xsp, "B": B, "Y": Y}
    if kind == "bf16":
        V, H, k = case["vocab"], case["hidden"], case["k"]
        t = _table(seed, V, H)
        if case["layout"] == "tiles":
            rows, t = t, torch.empty(lib.bf16_dev_tiles_bytes(V, H) // 2, dtype=torch.int16, device="cuda")
            qk.check(lib.bf16_dev_tile_table(t.data_ptr(), rows.data_ptr(), V, H, qk._stream()))
        i32 = lambda n: torch.zeros(n, dtype=torch.int32, device="cuda")  # noqa: E731
        return {"kind": kind, "case": case, "t": t, "h": _normal(_gen(seed, 8), H), "ids": i32(k),
                "sc": torch.zeros(k, dtype=torch.float32, device="cuda"), "cnt": i32(2), "out": i32(1),
                "rng": torch.full((1,), 12345 + seed % 1000, dtype=torch.int32, device="cuda"), "work": i32(2 * k)}
    if kind == "layer":
        L, linear = case["layers"], case["linear"]
        image = _Image(L * _layer_bytes(linear))
        plans, states = ((qk.LinearLayerPlan if linear else qk.MlpPlan) * L)(), []
        for l in range(L):
            states.append(_fill_plan(plans[l], image, *_layer_inputs(seed, l, linear), linear))
        image.protect()
        x = _normal(_gen(seed, 9), case["tokens"], HIDDEN).cpu().numpy()
        return {"kind": kind, "case": case, "plans": plans, "states": states, "x": x}
    if kind == "token":
        return _prepare_token(case, seed)
    M, K = case["M"], case["K"]
    ms, es = _planes(_gen(seed, 4), M, K, 122, 130)
    mat = qk.DeviceMatrix.from_soa(ms, es) if case["back"] else qk.DeviceMatrix.empty(M, K)
    return {"kind": kind, "case": case, "mat": mat, "ms": torch.empty_like(ms) if case["back"] else ms,
            "es": torch.empty_like(es) if case["back"] else es}


def _ragged(planes, K):
    """Planes of row stride K whose K % 64 trailing mantissas are in no block."""
    mant, exps = planes
    if K % 64:
        mant = torch.nn.functional.pad(mant, (0, K % 64))
    return mant, exps


def _prepare_token(case, seed):
    att = sum(M * K + M * (K // 64) + 128 for _, M, K in CALLBACK) if case["attention"] else 0
    nfull = sum(_is_full(l) for l in range(LAYERS))
    image = _Image((LAYERS - nfull) * _layer_bytes(True) + nfull * (_layer_bytes(False) + att) + VOCAB * HIDDEN * 2 + 64)
    lin, mlp = (qk.LinearLayerPlan * (LAYERS - nfull))(), (qk.MlpPlan * LAYERS)()
    full = _host(np.array([int(_is_full(l)) for l in range(LAYERS)], np.int32))
    li, attn = 0, {}
    for l in range(LAYERS):
        w, p = _layer_inputs(seed, l, not full[l])
        if full[l]:
            _fill_plan(mlp[l], image, w, p, False)
            if case["attention"]:
                g = _gen(seed, 300 + l)
                attn[l] = {n: (image.put(m), image.put(e), M, K)
                           for n, M, K in CALLBACK for m, e in (_planes(g, M, K, 122, 126),)}
                attn[l]["ln"] = _host((_normal(g, HIDDEN) * 0.1).cpu().numpy()).ctypes.data
        else:
            _fill_plan(lin[li], image, w, p, True)
            li += 1
    table = image.put(_table(seed, VOCAB, HIDDEN))
    image.protect()
    s = {"kind": "token", "case": case, "lin": lin, "mlp": mlp, "full": full, "table": table,
         "fnorm": _host((_normal(_gen(seed, 5), HIDDEN) * 0.1).cpu().numpy()),
         "ids": [int(i) for i in np.random.default_rng(seed).integers(0, VOCAB, case["tokens"])],
         "cb": qk.FULL_ATTN_CALLBACK()}
    if case["attention"]:
        s["cb"] = _callback(attn)
    return s


def _callback(attn):
    """The engine's full-attention callback around its attention step (which is
    another library's: stood in for by a scaled slice of q): rmsnorm, the q, k
    and v GEMVs, o, the residual, all through the host entry points."""
    lib = qk.load()
    normed, ys = np.empty(HIDDEN, np.float32), {n: np.empty(M, np.float32) for n, M, _ in CALLBACK}
    ctxv = np.empty(HD, np.float32)

    def gemv(layer, n, x):
        m, e, M, K = attn[layer][n]
        lib.bfp8_gemv(ys[n].ctypes.data, x.ctypes.data, m, e, M, K)

    def cb(layer, h_ptr, ctx):
        h = np.ctypeslib.as_array(ctypes.cast(h_ptr, ctypes.POINTER(ctypes.c_float)), shape=(HIDDEN,))
        lib.rmsnorm(normed.ctypes.data, h_ptr, attn[layer]["ln"], HIDDEN, EPS)
        for n in "qkv":
            gemv(layer, n, normed)
        np.multiply(ys["q"][:HD], np.float32(1e-3), out=ctxv)
        gemv(layer, "o", ctxv)
        np.add(h, ys["o"], out=h)

    return qk.FULL_ATTN_CALLBACK(cb)


# ---- run -------------------------------------------------------------------------------
def run(s):
    lib, kind = qk.load(), s["kind"]
    if kind == "gemv":
        s["plan"].run()
        return s["y"]
    if kind in ("sweep", "lm_head"):
        s["plan"].run()
        return s["out"]
    if kind == "batch":
        return qk.gemv_batch(s["mat"], s["xsp"], s["xs"], s["B"], s["Y"])
    if kind == "bf16":
        c, st = s["case"], qk._stream()
        ids, sc, cnt = s["ids"].data_ptr(), s["sc"].data_ptr(), s["cnt"].data_ptr()
        if c["layout"] == "tiles":
            qk.check(lib.bf16_dev_lm_head_tiles(ids, sc, cnt, cnt + 4, None, s["h"].data_ptr(), s["t"].data_ptr(),
                                                c["vocab"], c["hidden"], c["k"], st))
        else:
            qk.check(lib.bf16_dev_lm_head(ids, sc, cnt, cnt + 4, None, s["h"].data_ptr(), s["t"].data_ptr(),
                                          c["vocab"], c["hidden"], c["k"], 1, st))
        qk.check(lib.bfp8_dev_sample_from_topk(s["out"].data_ptr(), ids, sc, cnt, c["k"], 0.7, 50, 0.9,
                                               s["rng"].data_ptr(), s["work"].data_ptr(), st))
        return {"scores": s["sc"], "ids": s["ids"], "count": s["cnt"], "token": s["out"], "rng": s["rng"]}
    if kind == "layer":
        c = s["case"]
        lib.qwen_forward_state_resident(1 if c["resident"] else 0)
        out = s["x"].copy()
        fn = lib.forward_linear_layer if c["linear"] else lib.forward_mlp
        for t in range(c["tokens"]):
            for l in range(c["layers"]):
                fn(ctypes.addressof(s["plans"][l]), out[t].ctypes.data)
        states = [] if c["resident"] or not c["linear"] else [list(st) for st in s["states"]]
        return {"h": out, "states": states}
    if kind == "token":
        c = s["case"]
        lib.qwen_forward_state_resident(1)
        hs, ids = np.zeros((c["tokens"], HIDDEN), np.float32), []
        for t, tok in enumerate(s["ids"]):
            ids.append(lib.forward_token_c(tok, hs[t].ctypes.data, ctypes.addressof(s["lin"]),
                                           ctypes.addressof(s["mlp"]), s["full"].ctypes.data, s["fnorm"].ctypes.data,
                                           s["table"], s["cb"], None))
        normed = np.empty(HIDDEN, np.float32)
        lib.rmsnorm(normed.ctypes.data, hs[-1].ctypes.data, s["fnorm"].ctypes.data, HIDDEN, EPS)
        top, logits = np.full(c["k"], -1, np.int32), np.zeros(c["k"], np.float32)
        lib.qwen_lm_head_topk_bf16(normed.ctypes.data, s["table"], VOCAB, HIDDEN, c["k"], top.ctypes.data,
                                   logits.ctypes.data)
        return {"h": hs, "greedy": ids, "logits": logits, "top": top}
    c, m = s["case"], s["mat"]
    if c["back"]:
        qk.check(lib.bfp8_dev_unpack(s["ms"].data_ptr(), s["es"].data_ptr(), m.mant.data_ptr(), m.exps.data_ptr(),
                                     c["M"], c["K"], qk._stream()))
        return [s["ms"], s["es"]]
    qk.check(lib.bfp8_dev_pack(m.mant.data_ptr(), m.exps.data_ptr(), s["ms"].data_ptr(), s["es"].data_ptr(), c["M"],
                               c["K"], qk._stream()))
    return [m.mant, m.exps]


# ---- what a pass cannot do without ---------------------------------------------------------
def _w(M, K):
    return M * (K // 64) * 65


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        M, K = case["M"], case["K"]
        return {"bytes": _w(M, K) + 4 * K + 4 * M, "flops": 2 * M * K}
    if kind == "sweep":
        it = _sweep_items(case)
        return {"bytes": sum(_w(M, K) + 4 * K + (8 * case["k"] if M == VOCAB else 4 * M) for M, K, *_ in it),
                "flops": sum(2 * M * K for M, K, *_ in it)}
    if kind == "lm_head":
        M, K = case["vocab"], case["K"]
        return {"bytes": _w(M, K) + 4 * K + 8 * case["k"], "flops": 2 * M * K}
    if kind == "batch":
        M, K, B = case["M"], case["K"], case["B"]
        return {"bytes": _w(M, K) + B * (K // 64) * 132 + 4 * B * M, "flops": 2 * M * K * B}
    if kind == "bf16":
        V, H = case["vocab"], case["hidden"]
        return {"bytes": 2 * V * H + 4 * H + 8 * case["k"], "flops": 2 * V * H}
    lin = sum(_w(M, K) for _, M, K in LINEAR) + 4 * (2 * HIDDEN + 4 * CONV + 2 * HEADS * HIDDEN)
    lin += 2 * 4 * (3 * CONV + HEADS * HEAD_DIM * HEAD_DIM)  # states read and written
    mlp = sum(_w(M, K) for _, M, K in FULL) + 4 * HIDDEN
    macs = [sum(M * K for _, M, K in s) for s in (LINEAR, FULL, CALLBACK)]
    if kind == "layer":
        n = case["layers"] * case["tokens"]
        return {"bytes": n * (lin if case["linear"] else mlp) + 8 * HIDDEN * case["tokens"],
                "flops": 2 * n * macs[0 if case["linear"] else 1]}
    if kind == "token":
        T, nfull = case["tokens"], sum(_is_full(l) for l in range(LAYERS))
        head = 2 * VOCAB * HIDDEN
        b = T * ((LAYERS - nfull) * lin + nfull * mlp + head) + head
        f = 2 * (T * ((LAYERS - nfull) * macs[0] + nfull * macs[1] + VOCAB * HIDDEN) + VOCAB * HIDDEN)
        if case["attention"]:
            b += T * nfull * sum(_w(M, K) for _, M, K in CALLBACK)
            f += 2 * T * nfull * macs[2]
        return {"bytes": b, "flops": f}
    return {"bytes": 2 * _w(case["M"], case["K"]), "flops": 0}


def tolerance(case):
    # results are defined bit for bit (the reference's rounding order)
    return "exact"


# ---- 64-bit results ---------------------------------------------------------------------
def _dequant(x):
    """The activation quantizer (int16 per 64-block, scale amax / 16384) on a
    double or float tensor, dequantized in double; K % 64 trailing elements
    dropped."""
    xb = x[: x.numel() // 64 * 64].to(torch.float32).cpu().view(-1, 64)
    amax = xb.abs().amax(1, keepdim=True)
    live = amax > 1e-20
    q = torch.full_like(amax, 16384.0) / torch.where(live, amax, torch.ones_like(amax))
    xq = torch.where(live, torch.round(xb * q), torch.zeros_like(xb))
    xs = torch.where(live, amax / 16384, torch.zeros_like(amax))
    return (xq.double() * xs.double()).view(-1).cuda()


def _mul(planes, X):
    """Planes times the columns of X [K, B] in double, a slab of rows at a time."""
    mant, exps = planes
    out = []
    for r in range(0, mant.shape[0], 4096):
        w = mant[r:r + 4096].double().view(-1, exps.shape[1], 64) * torch.exp2(exps[r:r + 4096].double() - 134)[..., None]
        out.append(w.view(w.shape[0], -1) @ X)
    return torch.cat(out)


def _gemv64(planes, x):
    return _mul(planes, _dequant(x)[:, None])[:, 0]


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean() + EPS) * (1 + w.double())


def _mlp64(h, w, p):
    n = _norm64(h, p["post_ln_w"])
    a, b = _gemv64(w["gate"], n), _gemv64(w["up"], n)
    return h + _gemv64(w["down"], a / (1 + torch.exp(-a)) * b)


def _linear64(h, w, p, st):
    p = {k: v.double() for k, v in p.items()}
    n = _norm64(h, p["in_ln_w"])
    x, z = _gemv64(w["qkv"], n), _gemv64(w["z"], n)
    taps = torch.cat([st["conv"], x[None]])
    d = (p["conv_w"].T * taps).sum(0)
    st["conv"] = taps[1:]
    q, k, v = (d / (1 + torch.exp(-d))).view(3, HEADS, HEAD_DIM)
    k = k / torch.sqrt((k * k).sum(1, keepdim=True) + EPS)
    q = q / math.sqrt(HEAD_DIM) / torch.sqrt((q * q).sum(1, keepdim=True) + EPS)
    alpha = torch.exp(p["nea"] * torch.log1p(torch.exp(p["wa"] @ n + p["dt"])))[:, None]
    beta = torch.sigmoid(p["wb"] @ n)[:, None]
    S = st["rec"]
    dl = (v - (k[:, :, None] * S).sum(1) * alpha) * beta
    o = (q[:, :, None] * S).sum(1) * alpha + (q * k).sum(1, keepdim=True) * dl
    st["rec"] = S * alpha[..., None] + k[:, :, None] * dl[:, None, :]
    g = o / torch.sqrt((o * o).mean(1, keepdim=True) + EPS) * p["norm_w"] * (z / (1 + torch.exp(-z))).view(HEADS, -1)
    return _mlp64(h + _gemv64(w["o"], g.reshape(-1)), w, p)


def _state64():
    return {"conv": torch.zeros(3, CONV, dtype=torch.float64, device="cuda"),
            "rec": torch.zeros(HEADS, HEAD_DIM, HEAD_DIM, dtype=torch.float64, device="cuda")}


def _blocked(S):
    """[head][i][j] in the reference's blocked order: 4 x 4 tiles, columns
    outermost, a tile's rows innermost."""
    n = HEAD_DIM // 4
    return S.view(HEADS, n, 4, n, 4).permute(0, 3, 1, 4, 2).reshape(HEADS, -1)


def _scores64(table, h):
    t = table.view(torch.bfloat16)
    return torch.cat([t[r:r + 8192].double() @ h.double() for r in range(0, t.shape[0], 8192)])


def _best(scores, k):
    return torch.topk(scores, min(k, scores.numel())).values


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        g = _gen(seed, 1)
        planes = _planes(g, case["M"], case["K"] // 64 * 64, 124, 130)
        return _gemv64(planes, _activation(g, case["K"], case["K"] > 2048))
    if kind == "sweep":
        ys, top = [], []
        for i, (M, K, lo, hi) in enumerate(_sweep_items(case)):
            g = _gen(seed, 10 + i)
            planes = _planes(g, M, K, lo, hi)
            y = _gemv64(planes, _activation(g, K, K > 2048))
            if M == VOCAB:
                top = [None, _best(y, case["k"]), None]
            else:
                ys.append(y)
        return [torch.cat(ys)] + top
    if kind == "lm_head":
        g = _gen(seed, 2)
        planes = _planes(g, case["vocab"], case["K"], 122, 128)
        return [None, _best(_gemv64(planes, _activation(g, case["K"], False)), case["k"]), None]
    if kind == "batch":
        g, K = _gen(seed, 3), case["K"]
        planes = _planes(g, case["M"], K // 64 * 64, 124, 130)
        X = torch.stack([_dequant(_activation(g, K, K > 2048)) for _ in range(case["B"])], 1)
        return _mul(planes, X).T.contiguous()
    if kind == "bf16":
        s = _scores64(_table(seed, case["vocab"], case["hidden"]), _normal(_gen(seed, 8), case["hidden"]))
        return {"scores": _best(s, case["k"]), "ids": None, "count": None, "token": None, "rng": None}
    if kind == "layer":
        layers = [_layer_inputs(seed, l, case["linear"]) + (_state64(),) for l in range(case["layers"])]
        hs = _normal(_gen(seed, 9), case["tokens"], HIDDEN).double()
        out = []
        for h in hs:
            for w, p, st in layers:
                h = _linear64(h, w, p, st) if case["linear"] else _mlp64(h, w, p)
            out.append(h)
        states = [] if case["resident"] or not case["linear"] else [[st["conv"], _blocked(st["rec"])]
                                                                   for _, _, st in layers]
        return {"h": torch.stack(out), "states": states}
    if kind == "token":
        table = _table(seed, VOCAB, HIDDEN)
        layers = [_layer_inputs(seed, l, not _is_full(l)) + (_state64(),) for l in range(LAYERS)]
        out = []
        for tok in np.random.default_rng(seed).integers(0, VOCAB, case["tokens"]):
            h = table[int(tok)].view(torch.bfloat16).double()
            for l, (w, p, st) in enumerate(layers):
                if _is_full(l):
                    if case["attention"]:
                        g = _gen(seed, 300 + l)
                        a = {n: _planes(g, M, K, 122, 126) for n, M, K in CALLBACK}
                        n64 = _norm64(h, _normal(g, HIDDEN) * 0.1)
                        h = h + _gemv64(a["o"], _gemv64(a["q"], n64)[:HD] * 1e-3)
                    h = _mlp64(h, w, p)
                else:
                    h = _linear64(h, w, p, st)
            out.append(h)
        n64 = _norm64(out[-1], _normal(_gen(seed, 5), HIDDEN) * 0.1)
        return {"h": torch.stack(out), "greedy": None, "logits": _best(_scores64(table, n64), case["k"]), "top": None}
    return None  # bytes moved, nothing computed
