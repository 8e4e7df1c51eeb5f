"""The calls whose time on an MI355X counts for a user of this framework, as
data: listed() names them, draw() gives more of the same ranges, prepare()
and run() make one ready and run it, exact() is the same result in 64 bits.

Every call goes through the device-level C ABI (include/picolm_hip.h, bound in
picolm_amd) with device pointers, the way a decode loop or a prompt loop that
keeps its activations in HBM calls it:

  attn_decode   one token's attention block (RoPE, fp16 append, attention over
                the cached rows), layer by layer as a forward pass issues it
                or all layers in one launch; optionally with QK-norm
  attn_prefill  the same for a run of prompt tokens
  matvec        one weight matrix times one vector
  mlp           the SwiGLU block of one token: rmsnorm + gate/up + silu in one
                call, down + residual in another
  matmat        one weight matrix times the vectors of a prompt
  forward       one token through a whole model: logits, the final residual
                and the appended cache rows
  prompt        a prompt through a whole model, likewise

Weights are random GGUF blocks (Q4_K, Q6_K, Q8_0) whose outputs have order
one, activations N(0, 1), cache rows N(0, 1) rounded to fp16.
"""
import math
import types

import numpy as np
import torch

import picolm_amd as P

Q8_0, Q4_K, Q6_K = 8, 12, 14
BLOCK = {Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210)}  # weights, bytes
LLAMA, QWEN = 0, 1
EPS = 1e-5


def listed():
    return [
        # a short chat turn's token, the attention of every layer in turn
        # (TinyLlama-1.1B heads): launch latency
        _decode("decode_tinyllama_257_layers", 22, 32, 4, 64, 2048, 256, per_layer=True),
        # the same model at its full context, all layers in one launch
        _decode("decode_tinyllama_2048", 22, 32, 4, 64, 2048, 2047),
        # a long context, layer by layer (Llama-3.2-1B heads)
        _decode("decode_llama32_8192_layers", 16, 32, 8, 64, 8192, 8191, theta=5e5,
                per_layer=True),
        # a head size between the usual ones, as small models have (MHA, 80)
        _decode("decode_d80_1500_layers", 8, 32, 32, 80, 2048, 1499, per_layer=True),
        # a 512-token prompt's attention, all layers (TinyLlama heads)
        _prefill("prefill_tinyllama_512", 22, 32, 4, 64, 2048, 0, 512),
        # an odd-sized prompt, layer by layer, QK-norm and half-split rotation
        # (Qwen3-0.6B heads)
        _prefill("prefill_qwen3_509_layers", 28, 16, 8, 128, 2048, 0, 509, theta=1e6, rope=QWEN,
                 qk_norm=True, per_layer=True),
        # a prompt at another head size (GQA 4, 96), layer by layer
        _prefill("prefill_d96_300_layers", 8, 32, 8, 96, 1024, 0, 300, per_layer=True),
        # the logits of one token (TinyLlama's Q6_K output matrix)
        _case("matvec_head", "matvec", qtype=Q6_K, n=2048, d=32000),
        # one token's SwiGLU block (TinyLlama, Q4_K and a Q6_K down matrix)
        _case("mlp_tinyllama", "mlp", qtype=Q4_K, down=Q6_K, n=2048, f=5632),
        # a short turn's tokens through one Q8_0 matrix
        _case("matmat_q8_17", "matmat", qtype=Q8_0, n=2048, d=2048, tokens=17),
        # one generated token (TinyLlama-1.1B, Q4_K_M-style types)
        _model("forward_tinyllama", "forward", 22, 2048, 5632, 32, 4, 64, 32000, start=200,
               tokens=1),
        # a 128-token prompt of the same model
        _model("prompt_tinyllama_128", "prompt", 22, 2048, 5632, 32, 4, 64, 32000, start=0,
               tokens=128),
    ]


def _case(name, kind, **kw):
    return dict({"name": name} if name else {}, kind=kind, **kw)


def _decode(name, L, Hq, Hkv, D, S, pos, theta=1e4, rope=LLAMA, qk_norm=False, per_layer=False):
    return _case(name, "attn_decode", L=L, Hq=Hq, Hkv=Hkv, D=D, S=S, start=pos, n=1, theta=theta,
                 rope=rope, qk_norm=qk_norm, per_layer=per_layer)


def _prefill(name, L, Hq, Hkv, D, S, start, n, theta=1e4, rope=LLAMA, qk_norm=False,
             per_layer=False):
    return _case(name, "attn_prefill", L=L, Hq=Hq, Hkv=Hkv, D=D, S=S, start=start, n=n,
                 theta=theta, rope=rope, qk_norm=qk_norm, per_layer=per_layer)


def _model(name, kind, L, E, F, Hq, Hkv, D, vocab, start, tokens, rope=LLAMA, qtype=Q4_K):
    return _case(name, kind, L=L, E=E, F=F, Hq=Hq, Hkv=Hkv, D=D, vocab=vocab, S=2048, start=start,
                 tokens=tokens, theta=1e4, rope=rope, qtype=qtype)


# ---- more cases of the same ranges ------------------------------------------


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng):
    """A head layout: the usual head sizes twice as often as the others."""
    D = rng.choice([64, 64, 64, 128, 128, 128, 48, 80, 96])
    Hkv = rng.choice([2, 4, 8, 32])
    G = rng.choice([1, 2, 4, 7, 8]) if Hkv <= 8 else 1
    return Hkv * G, Hkv, D


def draw(rng):
    kind = rng.choice(["attn_decode", "attn_prefill", "matvec", "mlp", "matmat", "forward",
                       "prompt"])
    if kind == "attn_decode":
        Hq, Hkv, D = _heads(rng)
        pos = _log(rng, 16, 8191)
        return _decode(None, rng.randint(4, 28), Hq, Hkv, D, 8192 if pos >= 4096 else 4096, pos,
                       rope=rng.choice([LLAMA, QWEN]), qk_norm=rng.random() < 0.25,
                       per_layer=rng.random() < 0.7)
    if kind == "attn_prefill":
        Hq, Hkv, D = _heads(rng)
        n = _log(rng, 5, 1024 if D in (64, 128) else 400)
        start = rng.choice([0, 0, rng.randint(1, 1000)])
        return _prefill(None, rng.randint(2, 16), Hq, Hkv, D, 2048, start, n,
                        rope=rng.choice([LLAMA, QWEN]), qk_norm=rng.random() < 0.25,
                        per_layer=rng.random() < 0.7)
    qtype = rng.choice([Q4_K, Q4_K, Q6_K, Q8_0])
    unit = BLOCK[qtype][0]
    if kind == "matvec":
        return _case(None, kind, qtype=qtype, n=unit * max(1, _log(rng, 256, 11008) // unit),
                     d=_log(rng, 64, 32000))
    if kind == "mlp":
        n = 256 * rng.randint(2, 16)
        return _case(None, kind, qtype=qtype, down=rng.choice([qtype, Q6_K]), n=n,
                     f=256 * max(1, int(n * rng.uniform(2, 4)) // 256))
    if kind == "matmat":
        return _case(None, kind, qtype=qtype, n=unit * max(1, _log(rng, 256, 5632) // unit),
                     d=_log(rng, 64, 8192), tokens=_log(rng, 2, 256))
    D = rng.choice([64, 64, 128])
    Hkv = rng.choice([2, 4, 8])
    Hq = Hkv * rng.choice([1, 2, 4, 7])
    E = 256 * rng.randint(2, 9)
    Q = Hq * D
    if Q % 256:  # a row of the output projection is whole blocks
        Hq, Q = Hkv * 4, Hkv * 4 * D
    tokens = 1 if kind == "forward" else _log(rng, 4, 200)
    start = _log(rng, 1, 1800) if kind == "forward" else rng.choice([0, rng.randint(1, 300)])
    F = 256 * max(2, int(E * rng.uniform(2, 3)) // 256)
    L = rng.randint(3, 16)
    weights = 2 * E * (Q + Hkv * D) + 3 * E * F
    L = max(1, min(L, int(0.95e9 / weights), int(1.2e11 / (weights * tokens))))
    return _model(None, kind, L, E, F, Hq, Hkv, D, rng.randint(2000, 32000), start, tokens,
                  rope=rng.choice([LLAMA, QWEN]), qtype=rng.choice([Q4_K, Q4_K, Q8_0]))


# ---- what a pass cannot do without ------------------------------------------


def _bytes(qtype, n, d):
    w, b = BLOCK[qtype]
    return d * (n // w) * b


def _attn_work(L, Hq, Hkv, D, start, n):
    pairs = sum(start + i + 1 for i in range(n))
    rows = (start + n) * 2 * Hkv * D * 2  # cached rows read (the new ones once)
    act = n * (2 * Hq * D * 4 + 2 * Hkv * D * 4 + 2 * Hkv * D * 2)
    return L * (rows + act), L * Hq * 4 * D * pairs


def _model_matrices(c):
    q, kv = c["Hq"] * c["D"], c["Hkv"] * c["D"]
    t, hi = c["qtype"], Q6_K if c["qtype"] == Q4_K else c["qtype"]
    E, F = c["E"], c["F"]
    return {"q": (t, E, q), "k": (t, E, kv), "v": (hi, E, kv), "o": (t, q, E), "gate": (t, E, F),
            "up": (t, E, F), "down": (hi, F, E)}


def work(case):
    c = case
    k = c["kind"]
    if k in ("attn_decode", "attn_prefill"):
        b, f = _attn_work(c["L"], c["Hq"], c["Hkv"], c["D"], c["start"], c["n"])
        return {"bytes": b, "flops": f}
    if k in ("matvec", "matmat"):
        t = c.get("tokens", 1)
        return {"bytes": _bytes(c["qtype"], c["n"], c["d"]) + 4 * t * (c["n"] + c["d"]),
                "flops": 2 * t * c["n"] * c["d"]}
    if k == "mlp":
        n, f = c["n"], c["f"]
        return {"bytes": 2 * _bytes(c["qtype"], n, f) + _bytes(c["down"], f, n) + 4 * (4 * n + 2 * f),
                "flops": 2 * 3 * n * f}
    mats = _model_matrices(c)
    per = sum(_bytes(*m) for m in mats.values())
    wts = sum(m[1] * m[2] for m in mats.values())
    head = (Q6_K, c["E"], c["vocab"])
    b, f = _attn_work(c["L"], c["Hq"], c["Hkv"], c["D"], c["start"], c["tokens"])
    act = c["tokens"] * (2 * c["Hq"] * c["D"] * 4 + 2 * c["Hkv"] * c["D"] * 4)  # stay on the chip
    return {"bytes": b - c["L"] * act + c["L"] * per + _bytes(*head) + 4 * (c["vocab"] + c["E"]),
            "flops": f + 2 * c["tokens"] * c["L"] * wts + 2 * c["E"] * c["vocab"]}


# ---- inputs -------------------------------------------------------------------


def _rms_over_scale(qtype):
    """RMS of a weight over its block's fp16 scale when every quant is uniform."""
    return {Q4_K: 300.0, Q6_K: 1365.0, Q8_0: 74.0}[qtype]


def _quant_rows(rng, qtype, n, d):
    """d random GGUF rows of n weights whose products with a unit-RMS vector
    have order one."""
    w, b = BLOCK[qtype]
    nb = n // w
    rows = np.frombuffer(rng.bytes(d * nb * b), np.uint8).reshape(d, nb, b).copy()
    c = -math.log2(math.sqrt(n) * _rms_over_scale(qtype))

    def scales():
        return np.exp2(rng.uniform(c - 1, c + 1, size=(d, nb))).astype(np.float16)

    if qtype == Q4_K:
        rows[:, :, 0:2] = scales()[..., None].view(np.uint8)
        rows[:, :, 2:4] = scales()[..., None].view(np.uint8)
    else:
        at = 208 if qtype == Q6_K else 0
        rows[:, :, at:at + 2] = scales()[..., None].view(np.uint8)
    return rows.reshape(d, nb * b)


def _dequant(qtype, rows, n):
    """The rows' weights in float64 on the GPU."""
    w, b = BLOCK[qtype]
    r = torch.from_numpy(rows).cuda().reshape(-1, n // w, b)
    f16 = lambda lo: r[:, :, lo:lo + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if qtype == Q8_0:
        y = f16(0) * r[:, :, 2:].view(torch.int8).double()
    elif qtype == Q4_K:
        s = r[:, :, 4:16].int()
        lo, hi, up = s[..., 0:4], s[..., 4:8], s[..., 8:12]
        sc = torch.cat([lo & 63, (up & 15) | ((lo >> 6) << 4)], -1).double()
        mn = torch.cat([hi & 63, (up >> 4) | ((hi >> 6) << 4)], -1).double()
        qs = r[:, :, 16:].reshape(*r.shape[:2], 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 3).reshape(*r.shape[:2], 8, 32).double()
        y = (f16(0) * sc).unsqueeze(-1) * q - (f16(2) * mn).unsqueeze(-1)
    else:
        ql = r[:, :, :128].reshape(*r.shape[:2], 2, 2, 32).int()
        qh = r[:, :, 128:192].reshape(*r.shape[:2], 2, 1, 32).int()
        nib = torch.cat([ql & 15, ql >> 4], 3)  # quarters 0, 1 (low), 2, 3 (high)
        two = torch.cat([(qh >> (2 * i)) & 3 for i in range(4)], 3)
        q = ((nib | (two << 4)) - 32).reshape(*r.shape[:2], 16, 16).double()
        sc = r[:, :, 192:208].view(torch.int8).double()
        y = (f16(208) * sc).unsqueeze(-1) * q
    return y.reshape(-1, n)


def _np_rng(seed):
    return np.random.default_rng([seed, 20240917])


def _randn(gen, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _tables(S, D, theta):
    """RoPE tables [S][D/2], fp32."""
    i = np.arange(D // 2, dtype=np.float32)
    angle = np.arange(S, dtype=np.float32)[:, None] / np.float32(theta) ** (2 * i / D)
    return np.cos(angle), np.sin(angle)


def _attn_inputs(c, seed):
    g = _gen(seed)
    L, n, D = c["L"], c["n"], c["D"]
    kv = c["Hkv"] * D
    x = types.SimpleNamespace()
    x.q = _randn(g, L, n, c["Hq"] * D)
    x.k, x.v = _randn(g, L, n, kv), _randn(g, L, n, kv)
    x.kc, x.vc = (torch.zeros(L, c["S"], kv, device="cuda", dtype=torch.float16) for _ in "kv")
    for cache in (x.kc, x.vc):
        for li in range(L):
            cache[li, :c["start"]] = _randn(g, c["start"], kv, dtype=torch.float16)
    cos, sin = _tables(c["S"], D, c["theta"])
    x.cos, x.sin = torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()
    x.qn = x.kn = None
    if c["qk_norm"]:
        x.qn, x.kn = (torch.rand(L, D, generator=g, device="cuda") + 0.5 for _ in "qk")
    return x


def _model_host(c, seed):
    """A model's host buffers, one random layer's matrices for every layer
    (each gets its own device copy)."""
    rng = _np_rng(seed)
    E = c["E"]
    h = types.SimpleNamespace(
        n_layers=c["L"], n_embd=E, n_ffn=c["F"], n_heads=c["Hq"], n_kv_heads=c["Hkv"],
        head_dim=c["D"], vocab_size=c["vocab"], max_seq_len=c["S"], rope_type=c["rope"],
        rope_base=c["theta"], eps=EPS, q_dim=c["Hq"] * c["D"], kv_dim=c["Hkv"] * c["D"])
    h.cache_elems = lambda: h.n_layers * h.max_seq_len * h.kv_dim
    layer = {k: (m[0], _quant_rows(rng, *m)) for k, m in _model_matrices(c).items()}
    layer.update({k: None for k in ("q_bias", "k_bias", "v_bias", "o_bias", "q_norm", "k_norm")})
    h.layers = []
    for _ in range(h.n_layers):
        norms = {k: rng.uniform(0.5, 1.5, E).astype(np.float32) for k in ("attn_norm", "ffn_norm")}
        h.layers.append(dict(layer, **norms))
    # unit-RMS embedding rows, a small random table repeated over the vocabulary
    few = _quant_rows(rng, Q4_K, E, 512)
    h.embd_type = Q4_K
    h.token_embd = np.ascontiguousarray(few[np.arange(c["vocab"]) % 512])
    h.output_norm = rng.uniform(0.5, 1.5, E).astype(np.float32)
    h.output_type, h.output = Q6_K, _quant_rows(rng, Q6_K, E, c["vocab"])
    h.tokens = rng.integers(0, c["vocab"], c["tokens"]).astype(np.int32)
    return h


class _Device:
    """A buffer of a device model as torch sees it; keeps the model."""

    def __init__(self, model, ptr, shape, typestr):
        self.model = model
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False),
                                         "version": 2, "strides": None}


def _view(model, name, *shape, typestr="<f4"):
    ptr = getattr(model, name).ptr
    return torch.as_tensor(_Device(model, ptr, shape, typestr), device="cuda")


def _model_caches(c, seed):
    g = _gen(seed + 1)
    kv = c["Hkv"] * c["D"]
    return [_randn(g, c["L"], c["start"], kv, dtype=torch.float16) for _ in "kv"]


def prepare(case, seed):
    P.init(0)
    c = case
    k = c["kind"]
    s = types.SimpleNamespace(kind=k, keep=[])
    if k in ("attn_decode", "attn_prefill"):
        x = _attn_inputs(c, seed)
        out = torch.zeros(c["L"], c["n"], c["Hq"] * c["D"], device="cuda")
        rows = slice(c["start"], c["start"] + c["n"])
        s.out = {"out": out, "k_rows": x.kc[:, rows], "v_rows": x.vc[:, rows]}
        s.keep = [x, out]
        s.calls = []
        decode = k == "attn_decode"
        step = 1 if c["per_layer"] else c["L"]
        for l in range(0, c["L"], step):
            args = [c["L"], c["Hq"], c["Hkv"], c["D"], c["S"], c["rope"], l, step, c["start"]]
            args += [] if decode else [c["n"]]
            args += [t.data_ptr() for t in (x.q[l], x.k[l], x.v[l], x.kc, x.vc, x.cos, x.sin,
                                            out[l])]
            args += [] if decode else [c["Hq"] * c["D"]]
            if c["qk_norm"]:
                args += [x.qn[l].data_ptr(), x.kn[l].data_ptr(), EPS]
            s.calls.append(tuple(args))
        name = "plh_" + k + ("_qknorm" if c["qk_norm"] else "")
        s.fn = getattr(P.lib, name)
        return s
    if k in ("matvec", "matmat"):
        t = c.get("tokens", 1)
        s.W = P.QMatrix(c["qtype"], c["n"], c["d"], _quant_rows(_np_rng(seed), c["qtype"], c["n"],
                                                                c["d"]))
        s.x = _randn(_gen(seed), t, c["n"])
        s.out = torch.zeros(t, c["d"], device="cuda")
        s.fn = P.lib.plh_gemv if k == "matvec" else P.lib.plh_matmul_batch
        tok = () if k == "matvec" else (t,)
        s.calls = [(c["qtype"], c["n"], c["d"], s.W.ptr, s.x.data_ptr(), *tok, s.out.data_ptr())]
        return s
    if k == "mlp":
        n, f = c["n"], c["f"]
        gate, up, down, w = _mlp_host(c, seed)
        s.gate, s.up = (P.QMatrix(c["qtype"], n, f, r) for r in (gate, up))
        s.down = P.QMatrix(c["down"], f, n, down)
        s.x, s.w = _randn(_gen(seed), n), torch.from_numpy(w).cuda()
        s.h, s.y = torch.zeros(f, device="cuda"), torch.zeros(n, device="cuda")
        s.out = {"hidden": s.h, "out": s.y}
        s.swiglu = (c["qtype"], n, f, s.gate.ptr, s.up.ptr, s.x.data_ptr(), s.h.data_ptr(),
                    s.w.data_ptr(), EPS)
        s.down_args = (c["down"], f, n, s.down.ptr, s.h.data_ptr(), s.y.data_ptr(), None, 0.0,
                       None, 0, None, s.x.data_ptr())
        return s
    h = _model_host(c, seed)
    s.m = P.DeviceModel(h)
    for buf, table in zip((s.m.cos, s.m.sin), _tables(c["S"], c["D"], c["theta"])):
        buf.upload(table)
    kc, vc = (_view(s.m, b, c["L"], c["S"], h.kv_dim, typestr="<f2") for b in ("key", "val"))
    for cache, rows in zip((kc, vc), _model_caches(c, seed)):
        cache[:, :c["start"]] = rows
    s.start, s.tokens = c["start"], h.tokens
    rows = slice(c["start"], c["start"] + c["tokens"])
    s.out = {"logits": _view(s.m, "logits", c["vocab"]), "x": _view(s.m, "x_out", c["E"]),
             "k_rows": kc[:, rows], "v_rows": vc[:, rows]}
    s.token = int(h.tokens[0])
    return s


def _mlp_host(c, seed):
    rng = _np_rng(seed)
    gate, up = (_quant_rows(rng, c["qtype"], c["n"], c["f"]) for _ in "gu")
    down = _quant_rows(rng, c["down"], c["f"], c["n"])
    return gate, up, down, rng.uniform(0.5, 1.5, c["n"]).astype(np.float32)


def run(state):
    s = state
    if s.kind == "forward":
        s.m.forward(s.token, s.start)
    elif s.kind == "prompt":
        s.m.prefill(s.tokens, s.start)
    elif s.kind == "mlp":
        P.check(P.lib.plh_gemv_swiglu(*s.swiglu), "plh_gemv_swiglu")
        P.check(P.lib.plh_gemv_ex(*s.down_args), "plh_gemv_ex")
    else:
        for args in s.calls:
            if s.fn(*args):
                raise P.PicolmHipError(P.lib.plh_last_error())
    return s.out


# ---- how near two correct results are ----------------------------------------


def tolerance(case):
    k = case["kind"]
    # One layer's attention.  Its splits and tile orders differ by 1e-7 to
    # 5e-7; against 64 bits an appended element that lands on the other side
    # of an fp16 rounding boundary adds an fp16 step (1e-3 of it) here and
    # there: 1e-5 in all, 3e-3 of an early token's output at most.
    if k in ("attn_decode", "attn_prefill"):
        return {"rel": 4e-5, "max": 1.2e-2}
    # fp32 sums in another order: the two orders of the weight products differ
    # by 1e-7 to 4e-7, 1.6e-6 of a value at most
    if k in ("matvec", "mlp", "matmat"):
        return {"rel": 2e-6, "max": 1e-5}
    # A whole model: such a difference moves a cached element to the
    # neighbouring fp16 value now and then, and that travels through the later
    # layers: 2e-4 to 1e-3 of one token's logits over 22 layers.  A prompt's
    # first tokens attend over few rows and amplify it further: 1e-2 of the
    # cached rows, single elements by 0.4.
    if k == "forward":
        return {"rel": 4e-3, "max": 4e-2}
    return {"rel": 3e-2, "max": 0.9}


# ---- the same in 64 bits --------------------------------------------------------


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rope(x, cos, sin, rope):
    """x [n, heads, D] rotated with the tables' rows cos, sin [n, D/2]."""
    c, s = cos.double()[:, None], sin.double()[:, None]
    if rope == QWEN:
        a, b = x.chunk(2, -1)
        return torch.cat([a * c - b * s, a * s + b * c], -1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)


def _attend(q, k, v, start, c, cos, sin, kc, vc):
    """One layer: q [n, Hq*D], k, v [n, Hkv*D] in float64 (QK-norm done), the
    cached rows kc, vc [start, Hkv*D] fp16.  The attention output and the
    appended fp16 rows."""
    n, D, Hkv = q.shape[0], c["D"], c["Hkv"]
    rows = slice(start, start + n)
    q = _rope(q.view(n, -1, D), cos[rows], sin[rows], c["rope"])
    k16 = _rope(k.view(n, Hkv, D), cos[rows], sin[rows], c["rope"]).half()
    v16 = v.half().view(n, Hkv, D)
    K = torch.cat([kc.view(-1, Hkv, D), k16]).double()
    V = torch.cat([vc.view(-1, Hkv, D), v16]).double()
    G = c["Hq"] // Hkv
    t = torch.arange(start + n, device="cuda")
    mask = t[None] > (t[rows])[:, None]
    out = torch.empty(n, c["Hq"], D, device="cuda", dtype=torch.float64)
    for h in range(c["Hq"]):
        sc = q[:, h] @ K[:, h // G].T.contiguous() / math.sqrt(D)
        sc.masked_fill_(mask, -math.inf)
        out[:, h] = torch.softmax(sc, -1) @ V[:, h // G].contiguous()
    return out.reshape(n, -1), k16.reshape(n, -1), v16.reshape(n, -1)


def exact(case, seed):
    c = case
    k = c["kind"]
    if k in ("attn_decode", "attn_prefill"):
        x = _attn_inputs(c, seed)
        outs, ks, vs = [], [], []
        for l in range(c["L"]):
            q, kk = x.q[l].double(), x.k[l].double()
            if c["qk_norm"]:
                q = _rms(q.view(c["n"], -1, c["D"]), x.qn[l].double()).flatten(1)
                kk = _rms(kk.view(c["n"], -1, c["D"]), x.kn[l].double()).flatten(1)
            o, kr, vr = _attend(q, kk, x.v[l].double(), c["start"], c, x.cos, x.sin,
                                x.kc[l, :c["start"]], x.vc[l, :c["start"]])
            outs.append(o)
            ks.append(kr.double())
            vs.append(vr.double())
        return {"out": torch.stack(outs), "k_rows": torch.stack(ks), "v_rows": torch.stack(vs)}
    if k in ("matvec", "matmat"):
        W = _dequant(c["qtype"], _quant_rows(_np_rng(seed), c["qtype"], c["n"], c["d"]), c["n"])
        return _randn(_gen(seed), c.get("tokens", 1), c["n"]).double() @ W.T
    if k == "mlp":
        gate, up, down, w = _mlp_host(c, seed)
        x = _randn(_gen(seed), c["n"]).double()
        xn = _rms(x, torch.from_numpy(w).cuda().double())
        g, u = (_dequant(c["qtype"], r, c["n"]) @ xn for r in (gate, up))
        h = g * torch.sigmoid(g) * u
        return {"hidden": h, "out": x + _dequant(c["down"], down, c["f"]) @ h}
    h = _model_host(c, seed)
    start, n = c["start"], c["tokens"]
    mats = _model_matrices(c)
    W = {m: _dequant(mats[m][0], h.layers[0][m][1], mats[m][1]) for m in mats}
    cos, sin = (torch.from_numpy(t).cuda() for t in _tables(c["S"], c["D"], c["theta"]))
    caches = _model_caches(c, seed)
    x = _dequant(Q4_K, h.token_embd[h.tokens], c["E"])
    ks, vs = [], []
    for l, layer in enumerate(h.layers):
        f64 = lambda a: torch.from_numpy(a).cuda().double()  # noqa: E731
        xn = _rms(x, f64(layer["attn_norm"]))
        att, kr, vr = _attend(xn @ W["q"].T, xn @ W["k"].T, xn @ W["v"].T, start, c, cos, sin,
                              caches[0][l], caches[1][l])
        ks.append(kr.double())
        vs.append(vr.double())
        x = x + att @ W["o"].T
        xn = _rms(x, f64(layer["ffn_norm"]))
        g = xn @ W["gate"].T
        x = x + (g * torch.sigmoid(g) * (xn @ W["up"].T)) @ W["down"].T
    x = _rms(x[-1], torch.from_numpy(h.output_norm).cuda().double())
    logits = torch.cat([_dequant(Q6_K, h.output[r:r + 4096], c["E"]) @ x
                        for r in range(0, c["vocab"], 4096)])
    return {"logits": logits, "x": x, "k_rows": torch.stack(ks), "v_rows": torch.stack(vs)}
