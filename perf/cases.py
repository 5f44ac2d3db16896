"""The work this backend does for its users, as cases that can be timed and checked.

Every case goes through the public entry points: one kernel call (or a few) through
`HipBackend.dispatch` over a `DeviceWorkspace`, or one walk of a compiled graph through
`HipSession`. `listed()` holds the named cases, `draw(rng)` gives further ones from the same
ranges. The kinds:

  act          an activation over a 1-D 16-bit tensor (the table lookup of a model's SiLU / GELU)
  kv_append    a decode step's int8 quantize + append of new K and V rows
  matmul       a dense product, alone or with the loader's fused residual / activation, in every
               dtype a graph can hold; f32 weights also in the compiler's panel-packed layout
  attn_i8      one token per sequence against a ragged int8 cache (serving decode)
  attn_rows    a prompt's rows against the int8 cache they were appended to
  attn_valid   the compiler's own attention over a 16-bit / f32 cache, one row (decode) or many
               (prompt chunk); with `mask` its additive-mask form
  w8a8         a product with an int8 / int4 / codebook weight, activations quantized per token
  decode_step  a decoder's decode step: the graph captured once, one replay per token
  prompt_pass  a decoder's prompt pass: one eager walk per prompt
"""
import math

import numpy as np
import torch

from hologram_amd import DeviceWorkspace, HipBackend, HipSession
from hologram_amd import kernel_call as kc
from hologram_amd.decoder_graph import (DecoderConfig, build_decode_step, build_prefill,
                                        rope_tables, rope_tables_rows)
from hologram_amd.kernel_call import BufferRef, KernelCall

DTYPES = {"bf16": (kc.DTYPE_BF16, torch.bfloat16), "f16": (kc.DTYPE_F16, torch.float16),
          "f32": (kc.DTYPE_F32, torch.float32)}
ACTS = {"gelu": (KernelCall.Gelu, 2), "silu": (KernelCall.Silu, 3),
        "sigmoid": (KernelCall.Sigmoid, 4), "tanh": (KernelCall.Tanh, 5),
        "exp": (KernelCall.Exp, 8)}
TIERS = {"i8": kc.DTYPE_I8, "i4": kc.DTYPE_I4, "e8cb": kc.DTYPE_E8CB}


def listed():
    return [
        # an activation over a large tensor: a 2048-row prompt's FFN (8192 wide)
        dict(name="act_gelu_16m", kind="act", act="gelu", dtype="bf16", n=16777216),
        # the smallest call of a decode step: one new token for each of 16 sequences
        dict(name="kv_append_decode", kind="kv_append", dtype="bf16", batch=16, kv_heads=8,
             head_dim=128, bucket=4096, new_rows=1, in_place=True),
        # the large square product
        dict(name="gemm_bf16_4096", kind="matmul", dtype="bf16", m=4096, k=4096, n=4096,
             epilogue="none", packed=False),
        # a prompt of arbitrary length through a projection with its residual, in f16
        dict(name="gemm_f16_ragged", kind="matmul", dtype="f16", m=1009, k=2048, n=4096,
             epilogue="add", packed=False),
        # an f32 graph's constant weight, in the layout the compiler emits
        dict(name="gemm_f32_packed", kind="matmul", dtype="f32", m=500, k=1536, n=2000,
             epilogue="none", packed=True),
        # serving: a ragged batch of long contexts, one token each
        dict(name="attn_i8_decode", kind="attn_i8", dtype="bf16", batch=32, heads=32, kv_heads=8,
             head_dim=128, bucket=32768, shortest=512),
        # a prompt's attention against the int8 cache, after an earlier turn
        dict(name="attn_i8_prompt", kind="attn_rows", dtype="bf16", batch=4, rows=501, past=300,
             heads=32, kv_heads=8, head_dim=128, bucket=1024),
        # the compiler's attention op: a decode step over a bf16 cache
        dict(name="attn_valid_decode", kind="attn_valid", dtype="bf16", batch=8, heads=32,
             kv_heads=8, head_dim=128, past=8192, valid=7001, new=1, mask=False),
        # ... and a chunk of a prompt after what is already cached
        dict(name="attn_valid_prompt", kind="attn_valid", dtype="bf16", batch=2, heads=32,
             kv_heads=8, head_dim=128, past=2048, valid=1537, new=509, mask=False),
        # a quantized model's projection over a prompt
        dict(name="w8a8_prompt", kind="w8a8", tier="i8", m=512, k=4096, n=4096, act="none",
             residual=False),
        # one token for each of 8 sequences through a whole (two-layer) decoder
        dict(name="decode_step", kind="decode_step", layers=2, hidden=2048, heads=32, kv_heads=8,
             head_dim=64, ffn=8192, vocab=32000, batch=8, bucket=1024, pos=640),
        # the prompts of 8 sequences through a whole (one-layer) decoder; their length is no
        # multiple of any tile
        dict(name="prompt_pass", kind="prompt_pass", layers=1, hidden=2048, heads=32, kv_heads=8,
             head_dim=64, ffn=8192, vocab=32000, batch=8, bucket=1024, rows=509),
    ]


# ------------------------------------------------------------------ draws ----
def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dim(rng, lo, hi, odd=0.15):
    """A matrix dimension: mostly a multiple of 64, sometimes of 8, now and then any number."""
    v, p = _log(rng, lo, hi), rng.random()
    step = 1 if p < odd else 8 if p < odd + 0.25 else 64
    return max(step, v // step * step)


def _heads(rng):
    kv = rng.choice([2, 4, 8])
    return kv * rng.choice([1, 2, 4, 8]), kv


def _draw_act(rng):
    return dict(kind="act", act=rng.choice(sorted(ACTS)), dtype=rng.choice(["bf16", "bf16", "f16"]),
                n=_log(rng, 4096, 16777216))


def _draw_kv(rng):
    return dict(kind="kv_append", dtype=rng.choice(["bf16", "bf16", "f16", "f32"]),
                batch=_log(rng, 1, 32), kv_heads=rng.choice([2, 4, 8]),
                head_dim=rng.choice([64, 96, 128, 128]), bucket=rng.choice([512, 1024, 4096]),
                new_rows=rng.choice([1, 1, 1, 7, 64]), in_place=rng.random() < 0.75)


def _draw_matmul(rng):
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
    most = 2e9 if dtype == "f32" else 1.2e10
    k, n = _dim(rng, 128, 8192), _dim(rng, 128, 8192)
    m = _log(rng, 1, 2500)
    while m * k * n > most:
        m = max(1, m // 2)
        k, n = (k // 2, n) if m == 1 else (k, n)
    return dict(kind="matmul", dtype=dtype, m=m, k=k, n=n,
                epilogue=rng.choice(["none", "none", "add", "act", "add_act"]),
                packed=dtype == "f32" and rng.random() < 0.5)


def _draw_attn_i8(rng):
    heads, kv = _heads(rng)
    bucket = _log(rng, 128, 16384)
    return dict(kind="attn_i8", dtype=rng.choice(["bf16", "bf16", "f32"]), batch=_log(rng, 1, 48),
                heads=heads, kv_heads=kv, head_dim=rng.choice([64, 128, 128, 96]), bucket=bucket,
                shortest=max(1, bucket // 64))


def _draw_attn_rows(rng):
    heads, kv = _heads(rng)
    rows, past = _log(rng, 2, 700), rng.choice([0, 0, _log(rng, 1, 1000)])
    return dict(kind="attn_rows", dtype="bf16", batch=rng.randint(1, 4), rows=rows, past=past,
                heads=heads, kv_heads=kv, head_dim=rng.choice([64, 128, 128]),
                bucket=(rows + past + 255) // 256 * 256)


def _draw_attn_valid(rng):
    heads, kv = _heads(rng)
    decode = rng.random() < 0.5
    past = _log(rng, 64, 8192) if decode else _log(rng, 64, 2048)
    return dict(kind="attn_valid", dtype=rng.choice(["bf16", "bf16", "f16", "f32"]),
                batch=rng.randint(1, 8) if decode else rng.randint(1, 2), heads=heads, kv_heads=kv,
                head_dim=rng.choice([64, 128, 128, 80]), past=past, valid=rng.randint(0, past),
                new=1 if decode else _log(rng, 2, 400), mask=rng.random() < 0.3)


def _draw_w8a8(rng):
    k = max(64, _log(rng, 256, 8192) // 64 * 64)
    n = _dim(rng, 256, 8192)
    m = _log(rng, 1, 512)
    while m * k * n > 8.0e9:
        m //= 2
    return dict(kind="w8a8", tier=rng.choice(["i8", "i8", "i4", "e8cb"]), m=m, k=k, n=n,
                act=rng.choice(["none", "none", "silu", "gelu"]), residual=rng.random() < 0.3)


def _draw_decoder(rng, prompt):
    head_dim = rng.choice([64, 128])
    hidden = rng.choice([1024, 1536, 2048])
    heads = hidden // head_dim
    batch = rng.choice([1, 2, 3, 5, 8, 16]) if not prompt else rng.choice([1, 2, 3, 5, 8])
    bucket = rng.choice([512, 1024])
    c = dict(kind="prompt_pass" if prompt else "decode_step", layers=1 if prompt else 2,
             hidden=hidden, heads=heads, kv_heads=max(1, heads // rng.choice([2, 4])),
             head_dim=head_dim, ffn=rng.choice([2, 3, 4]) * hidden,
             vocab=rng.choice([8000, 16000, 32000]), batch=batch, bucket=bucket)
    if prompt:
        c["rows"] = _log(rng, 16, 509)
    else:
        c["pos"] = rng.randint(1, bucket - 1)
    return c


def draw(rng):
    return rng.choice([_draw_act, _draw_kv, _draw_matmul, _draw_matmul, _draw_attn_i8,
                       _draw_attn_rows, _draw_attn_valid, _draw_attn_valid, _draw_w8a8,
                       lambda r: _draw_decoder(r, False), lambda r: _draw_decoder(r, True)])(rng)


# ----------------------------------------------------------------- inputs ----
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype)


def _outliers(g, shape, dtype):
    """K / V rows as a model makes them: N(0, 1), a few channels 20 times as large."""
    x = torch.randn(shape, generator=g, device="cuda")
    big = torch.rand(shape[-1], generator=g, device="cuda") < 0.02
    return (x * torch.where(big, 20.0, 1.0)).to(dtype)


def _int8_cache(g, planes, rows, d):
    """A filled int8 cache and its scales: rows of N(0, 1) quantized to their largest value."""
    q = torch.empty((planes, rows, d), dtype=torch.int8, device="cuda")
    step = max(1, (1 << 27) // (rows * d))
    for p in range(0, planes, step):
        x = torch.randn((min(step, planes - p), rows, d), generator=g, device="cuda")
        q[p:p + step] = (x * (127.0 / 2.9)).round_().clamp_(-127, 127).to(torch.int8)
    s = (0.8 + 0.4 * torch.rand((planes, rows), generator=g, device="cuda")) * (2.9 / 127.0)
    return q, s


def _act_inputs(c, seed):
    return {"x": _randn(_gen(seed), c["n"], DTYPES[c["dtype"]][1], 2.5)}


def _kv_inputs(c, seed):
    g = _gen(seed)
    planes, dt = c["batch"] * c["kv_heads"], DTYPES[c["dtype"]][1]
    new = [_outliers(g, (planes, c["new_rows"], c["head_dim"]), dt) for _ in range(2)]
    caches = [_int8_cache(g, planes, c["bucket"], c["head_dim"]) for _ in range(2)]
    pos = torch.randint(0, 4 * c["bucket"], (1,), generator=g, device="cuda", dtype=torch.int32)
    return {"new": new, "caches": caches, "pos": pos}


def _matmul_inputs(c, seed):
    g = _gen(seed)
    dt = DTYPES[c["dtype"]][1]
    a = _randn(g, (c["m"], c["k"]), dt)
    b = _randn(g, (c["k"], c["n"]), dt, c["k"] ** -0.5)
    r = _randn(g, (c["m"], c["n"]), dt) if "add" in c["epilogue"] else None
    return {"a": a, "b": b, "r": r}


def _panels(b):
    """f32 [k, n] as the compiler's panels [ceil(n / 16)][k][16], zeros past n."""
    k, n = b.shape
    p = (n + 15) // 16
    wide = torch.zeros((k, p * 16), dtype=b.dtype, device=b.device)
    wide[:, :n] = b
    return wide.view(k, p, 16).permute(1, 0, 2).contiguous()


def _attn_i8_inputs(c, seed):
    g = _gen(seed)
    planes, rows = c["batch"] * c["kv_heads"], c.get("rows", 1)
    kq, ks = _int8_cache(g, planes, c["bucket"], c["head_dim"])
    vq, vs = _int8_cache(g, planes, c["bucket"], c["head_dim"])
    q = _randn(g, (c["batch"], rows, c["heads"], c["head_dim"]), DTYPES[c["dtype"]][1])
    if c["kind"] == "attn_i8":
        lens = torch.randint(c["shortest"], c["bucket"] + 1, (c["batch"],), generator=g,
                             device="cuda", dtype=torch.int32)
    else:      # every sequence's rows sit after its own part of the earlier turn
        lens = rows + torch.randint(0, c["past"] + 1, (c["batch"],), generator=g, device="cuda",
                                    dtype=torch.int32)
    return {"q": q, "kq": kq, "ks": ks, "vq": vq, "vs": vs, "lens": lens}


def _attn_valid_inputs(c, seed):
    g = _gen(seed)
    dt = DTYPES[c["dtype"]][1]
    planes, d, new = c["batch"] * c["kv_heads"], c["head_dim"], c["new"]
    x = {"q": _randn(g, (c["batch"], c["heads"], new, d), dt)}
    for name, rows in (("kp", c["past"]), ("vp", c["past"]), ("kn", new), ("vn", new)):
        x[name] = _randn(g, (planes, rows, d), dt)
    if c["mask"]:      # a causal mask over what is cached and the chunk itself
        total = c["past"] + new
        j = torch.arange(total, device="cuda")
        i = torch.arange(new, device="cuda")[:, None]
        seen = (j < c["valid"]) | ((j >= c["past"]) & (j <= c["past"] + i))
        x["mask"] = torch.where(seen, 0.0, -math.inf)
    else:
        x["valid"] = torch.tensor([c["valid"]], dtype=torch.int32, device="cuda")
    return x


def _w8a8_inputs(c, seed):
    g = _gen(seed)
    m, k, n = c["m"], c["k"], c["n"]
    x = {"a": _randn(g, (m, k)), "codebook": None}
    ints = lambda lo, hi, shape, dt: torch.randint(lo, hi, shape, generator=g, device="cuda",  # noqa: E731
                                                   dtype=dt)
    if c["tier"] == "i8":
        x["w"], level = ints(-127, 128, (n, k), torch.int8), 127
    elif c["tier"] == "i4":
        x["w"], level = ints(0, 256, (n, k // 2), torch.uint8), 7
    else:
        x["w"], level = ints(0, 256, (n, k // 8), torch.uint8), 32
        x["codebook"] = ints(-32, 33, (256, 8), torch.int8)
    x["scales"] = (0.5 + torch.rand(n, generator=g, device="cuda")) * (k ** -0.5 / level)
    x["zero_points"] = torch.zeros(n, dtype=torch.int32, device="cuda")
    x["r"] = _randn(g, (m, n)) if c["residual"] else None
    return x


def _config(c):
    return DecoderConfig(**{k: c[k] for k in ("layers", "hidden", "heads", "kv_heads", "head_dim",
                                              "ffn", "vocab", "batch", "bucket")})


def _weights(cfg, g):
    """Random weights N(0, 0.02), norm gains around 1, as bf16 tensors."""
    hd, kd, dm = cfg.heads * cfg.head_dim, cfg.kv_heads * cfg.head_dim, cfg.hidden
    w = lambda *shape: _randn(g, shape, torch.bfloat16, 0.02)  # noqa: E731
    gain = lambda: (1.0 + 0.1 * torch.randn(dm, generator=g, device="cuda")).to(torch.bfloat16)  # noqa: E731
    out = {"embedding": w(cfg.vocab, dm), "lm_head": w(dm, cfg.vocab), "final_norm": gain()}
    for layer in range(cfg.layers):
        out[f"l{layer}"] = {"attn_norm": gain(), "ffn_norm": gain(), "wq": w(dm, hd),
                            "wk": w(dm, kd), "wv": w(dm, kd), "wo": w(hd, dm),
                            "wg": w(dm, cfg.ffn), "wu": w(dm, cfg.ffn), "wd": w(cfg.ffn, dm)}
    return out


def _as_bytes(w):
    return {k: _as_bytes(v) if isinstance(v, dict) else v.view(torch.int16).cpu().numpy().tobytes()
            for k, v in w.items()}


def _decoder_inputs(c, seed):
    cfg, g = _config(c), _gen(seed)
    w = _weights(cfg, g)
    rows = c.get("rows", 1)
    prompt = c["kind"] == "prompt_pass"
    pos = 0 if prompt else c["pos"]
    tables = rope_tables_rows if prompt else rope_tables
    where = np.arange(pos, pos + rows)
    rope = [torch.frombuffer(bytearray(t), dtype=torch.bfloat16).cuda()
            for heads in (cfg.heads, cfg.kv_heads) for t in tables(cfg, where, heads)]
    tokens = torch.randint(0, cfg.vocab, (cfg.batch, rows), generator=g, device="cuda",
                           dtype=torch.int32)
    caches = []
    for _ in range(2 * cfg.layers):
        caches += _int8_cache(g, cfg.planes, cfg.bucket, cfg.head_dim)
    ports = [tokens, torch.tensor([pos], dtype=torch.int32, device="cuda"),
             torch.full((cfg.batch,), pos + rows, dtype=torch.int32, device="cuda"), *rope]
    return {"cfg": cfg, "weights": w, "rows": rows, "pos": pos, "ports": ports, "caches": caches}


# ---------------------------------------------------------------- prepare ----
def _backend():
    return HipBackend(device=0, stream=torch.cuda.current_stream().cuda_stream)


class _Calls:
    """A backend, a workspace with its slots bound, the calls of one pass and what they write."""

    def __init__(self):
        self.backend, self.ws, self.calls, self.out, self.slots = _backend(), DeviceWorkspace(), [], None, 0

    def slot(self, tensor):
        self.ws.bind(self.slots, tensor)
        self.slots += 1
        return BufferRef(self.slots - 1)

    def optional(self, tensor):
        return self.slot(tensor) if tensor is not None else kc.NO_BUFFER


def _prepare_act(c, seed):
    s, x = _Calls(), _act_inputs(c, seed)["x"]
    s.out = torch.empty_like(x)
    s.calls = [ACTS[c["act"]][0](kc.UnaryCall(s.slot(x), s.slot(s.out), c["n"], 16,
                                              DTYPES[c["dtype"]][0]))]
    return s


def _prepare_kv(c, seed):
    s, x = _Calls(), _kv_inputs(c, seed)
    pos = s.slot(x["pos"])
    s.out = []
    for new, (q, scales) in zip(x["new"], x["caches"]):
        nw, cq, cs = s.slot(new), s.slot(q), s.slot(scales)
        oq, os_ = cq, cs
        if not c["in_place"]:
            q, scales = torch.empty_like(q), torch.empty_like(scales)
            oq, os_ = s.slot(q), s.slot(scales)
        s.calls.append(KernelCall.KvQuantAppend(kc.KvQuantAppendCall(
            nw, pos, cq, cs, oq, os_, c["batch"] * c["kv_heads"], c["bucket"], c["new_rows"],
            c["head_dim"], DTYPES[c["dtype"]][0])))
        s.out += [q, scales]
    return s


def _prepare_matmul(c, seed):
    s, x = _Calls(), _matmul_inputs(c, seed)
    b = _panels(x["b"]) if c["packed"] else x["b"]
    s.out = torch.empty((c["m"], c["n"]), dtype=x["a"].dtype, device="cuda")
    mm = kc.MatMulCall(s.slot(x["a"]), s.slot(b), s.slot(s.out), c["m"], c["k"], c["n"],
                       DTYPES[c["dtype"]][0], b_packed=c["packed"])
    e = c["epilogue"]
    if e == "none":
        call = KernelCall.MatMul(mm)
    elif e == "act":
        call = KernelCall.MatMulActivation(kc.MatMulActivationCall(mm, ACTS["gelu"][1]))
    elif e == "add":
        call = KernelCall.MatMulAdd(kc.MatMulAddCall(mm, s.slot(x["r"])))
    else:
        call = KernelCall.MatMulAddActivation(kc.MatMulAddActivationCall(mm, s.slot(x["r"]),
                                                                         ACTS["silu"][1]))
    s.calls = [call]
    return s


def _prepare_attn_i8(c, seed):
    s, x = _Calls(), _attn_i8_inputs(c, seed)
    s.out = torch.empty_like(x["q"])
    attn = kc.DecodeAttentionI8Call(
        s.slot(x["q"]), s.slot(x["kq"]), s.slot(x["vq"]), s.slot(x["ks"]), s.slot(x["vs"]),
        s.slot(x["lens"]), s.slot(s.out), c["batch"], c["heads"], c["kv_heads"], c["bucket"],
        c["head_dim"], 0, DTYPES[c["dtype"]][0])
    s.calls = [KernelCall.DecodeAttentionI8(attn) if c["kind"] == "attn_i8" else
               KernelCall.AttentionI8Rows(kc.AttentionI8RowsCall(attn, c["rows"]))]
    return s


def _prepare_attn_valid(c, seed):
    s, x = _Calls(), _attn_valid_inputs(c, seed)
    s.out = torch.empty_like(x["q"])
    make, wrap = ((kc.DecodeAttentionCall, KernelCall.DecodeAttention) if c["mask"] else
                  (kc.DecodeAttentionValidCall, KernelCall.DecodeAttentionValid))
    s.calls = [wrap(make(s.slot(x["q"]), s.slot(x["kp"]), s.slot(x["vp"]), s.slot(x["kn"]),
                         s.slot(x["vn"]), s.slot(x["mask" if c["mask"] else "valid"]),
                         s.slot(s.out), c["batch"], c["heads"], c["kv_heads"], c["new"], c["past"],
                         c["new"], c["head_dim"], 0, DTYPES[c["dtype"]][0]))]
    return s


def _prepare_w8a8(c, seed):
    s, x = _Calls(), _w8a8_inputs(c, seed)
    s.out = torch.empty((c["m"], c["n"]), dtype=torch.float32, device="cuda")
    s.calls = [KernelCall.MatMulDequant(kc.MatMulDequantCall(
        a=s.slot(x["a"]), bq=s.slot(x["w"]), scales=s.slot(x["scales"]),
        zero_points=s.slot(x["zero_points"]), output=s.slot(s.out), m=c["m"], k=c["k"], n=c["n"],
        channels=c["n"], inner=1, quant_dtype=TIERS[c["tier"]], dtype=kc.DTYPE_F32, scale_bits=0,
        zero_point=0, bq_omajor=True, act_quant=1,
        act=ACTS[c["act"]][1] if c["act"] != "none" else 0, residual=s.optional(x["r"]),
        codebook=s.optional(x["codebook"])))]
    return s


class _DeviceBytes:
    """A device range a session owns, for torch.as_tensor: the tensor keeps this object, and this
    object the session, so the memory outlives every view of it."""

    def __init__(self, session, port):
        self.session = session
        ptr, nbytes = session.output_ptr(port)
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1",
                                         "data": (ptr, False), "version": 2}


class _Walk:
    """A loaded decoder archive with its input ports bound to device tensors."""

    def __init__(self, c, seed):
        x = _decoder_inputs(c, seed)
        cfg, w = x["cfg"], _as_bytes(x["weights"])
        del x["weights"]
        self.captured = c["kind"] == "decode_step"
        archive = build_decode_step(cfg, w) if self.captured else build_prefill(cfg, w, x["rows"])
        self.backend = _backend()
        self.session = HipSession(self.backend, archive)
        self.inputs = x["ports"] + x["caches"]
        for i, t in enumerate(self.inputs):
            self.session.bind_input(i, t)
        self.stream = torch.cuda.ExternalStream(self.session.stream())
        logits = torch.as_tensor(_DeviceBytes(self.session, 1), device="cuda")
        # The tokens are the logits' arg-maxima and stay out: a tie in bf16 logits is common and
        # either token is right. The caches are updated in place.
        self.out = {"logits": logits.view(torch.bfloat16).view(cfg.batch, cfg.vocab),
                    "caches": x["caches"]}
        if self.captured:
            torch.cuda.current_stream().synchronize()
            self.session.capture()
            self.session.synchronize()

    def run(self):
        now = torch.cuda.current_stream()
        self.stream.wait_stream(now)
        if self.captured:
            self.session.replay()
        else:
            self.session.run()
        now.wait_stream(self.stream)


_PREPARE = {"act": _prepare_act, "kv_append": _prepare_kv, "matmul": _prepare_matmul,
            "attn_i8": _prepare_attn_i8, "attn_rows": _prepare_attn_i8,
            "attn_valid": _prepare_attn_valid, "w8a8": _prepare_w8a8, "decode_step": _Walk,
            "prompt_pass": _Walk}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    if isinstance(state, _Walk):
        state.run()
    else:
        for call in state.calls:
            state.backend.dispatch(call, state.ws)
    return state.out


# ------------------------------------------------------- work, tolerances ----
def _seen(rows, past):
    """Keys seen by `rows` causal rows after `past` cached ones, summed over the rows."""
    return rows * past + rows * (rows + 1) // 2


def work(case):
    c, kind = case, case["kind"]
    es = {"bf16": 2, "f16": 2, "f32": 4}[c.get("dtype", "bf16")]
    if kind == "act":
        return {"bytes": 2 * es * c["n"], "flops": 0}
    if kind == "kv_append":
        planes, d = c["batch"] * c["kv_heads"], c["head_dim"]
        new = planes * c["new_rows"] * (d * es + d + 4)
        copied = 0 if c["in_place"] else 2 * planes * c["bucket"] * (d + 4)
        return {"bytes": 2 * (new + copied) + 4, "flops": 2 * planes * c["new_rows"] * d * 4}
    if kind == "matmul":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": es * (m * k + k * n + (2 if "add" in c["epilogue"] else 1) * m * n),
                "flops": 2 * m * k * n}
    if kind in ("attn_i8", "attn_rows"):
        b, h, kv, d, rows = c["batch"], c["heads"], c["kv_heads"], c["head_dim"], c.get("rows", 1)
        if kind == "attn_i8":
            mean = (c["shortest"] + c["bucket"]) / 2
            keys, seen = b * mean, b * mean
        else:
            keys, seen = b * (rows + c["past"] / 2), b * _seen(rows, c["past"] / 2)
        return {"bytes": keys * kv * (2 * d + 8) + 2 * es * b * rows * h * d + 4 * b,
                "flops": 4 * seen * h * d}
    if kind == "attn_valid":
        b, h, kv, d, new = c["batch"], c["heads"], c["kv_heads"], c["head_dim"], c["new"]
        keys = c["valid"] + new
        mask = 4 * new * (c["past"] + new) if c["mask"] else 4
        return {"bytes": es * (2 * b * kv * keys * d + 2 * b * h * new * d) + mask,
                "flops": 4 * b * h * d * _seen(new, c["valid"])}
    if kind == "w8a8":
        m, k, n = c["m"], c["k"], c["n"]
        weight = n * k // {"i8": 1, "i4": 2, "e8cb": 8}[c["tier"]]
        return {"bytes": weight + 4 * m * k + 8 * n + (8 if c["residual"] else 4) * m * n,
                "flops": 2 * m * k * n}
    dm, f, v, layers, b = c["hidden"], c["ffn"], c["vocab"], c["layers"], c["batch"]
    hd, kd, rows = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c.get("rows", 1)
    past = c.get("pos", 0)
    per_layer = dm * (2 * hd + 2 * kd) + 3 * dm * f
    cached = 2 * b * c["kv_heads"] * (past + rows) * (c["head_dim"] + 4)
    return {"bytes": 2 * (layers * (per_layer + 2 * dm) + dm * v + dm) + layers * cached +
            2 * b * rows * dm + 2 * b * v,
            "flops": 2 * b * rows * layers * per_layer + 2 * b * dm * v +
            4 * layers * b * hd * _seen(rows, past)}


def tolerance(case):
    kind = case["kind"]
    # a table lookup, a quantizer and exact integer sums: whole results are fixed
    if kind in ("act", "kv_append", "w8a8"):
        return "exact"
    if kind in ("decode_step", "prompt_pass"):
        # logits a few narrowing operations deep; a K / V value on an int8 rounding boundary
        # may move by one level
        return {"rel": 0.02, "max": 0.15, "differ": 0.005}
    return {"bf16": {"rel": 0.01}, "f16": {"rel": 0.0015}, "f32": {"rel": 1e-5}}[case["dtype"]]


# ------------------------------------------------------------ 64-bit values ----
_GELU_C = math.sqrt(2.0 / math.pi)


def _act64(name, x):
    if name == "gelu":
        return 0.5 * x * (1.0 + torch.tanh(_GELU_C * (x + 0.044715 * x * x * x)))
    if name == "silu":
        return x / (1.0 + torch.exp(-x))
    return {"sigmoid": torch.sigmoid, "tanh": torch.tanh, "exp": torch.exp}[name](x)


def _quant_rows(x):
    """The per-row symmetric int8 scheme, in the f32 operations that define it: levels, scales."""
    x = x.to(torch.float32)
    amax = x.abs().amax(-1, keepdim=True)
    inv = torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))
    t = x * inv
    q = torch.where(t >= 0, torch.trunc(t + 0.5), torch.trunc(t - 0.5)).clamp(-127, 127)
    return q, amax / 127.0


def _attention64(q, k, v, scale, limit):
    """q [rows, d], k and v [keys, d] in 64 bits; row i sees the first limit[i] keys."""
    s = (q @ k.t().contiguous()) / scale
    s = s.masked_fill(torch.arange(k.shape[0], device=q.device)[None, :] >= limit[:, None], -math.inf)
    p = torch.softmax(s, -1)
    return torch.where((limit > 0)[:, None], torch.nan_to_num(p) @ v, torch.zeros_like(q))


def _exact_attn_i8(c, seed):
    x = _attn_i8_inputs(c, seed)
    b, h, kv, d, rows = c["batch"], c["heads"], c["kv_heads"], c["head_dim"], c.get("rows", 1)
    out = torch.empty((b, rows, h, d), dtype=torch.float64, device="cuda")
    t = torch.arange(rows, device="cuda")
    for i, n in enumerate(x["lens"].tolist()):
        limit = (n - (rows - 1 - t)).clamp(0, c["bucket"])
        for p in range(kv):
            k = x["kq"][i * kv + p, :n].double() * x["ks"][i * kv + p, :n, None].double()
            v = x["vq"][i * kv + p, :n].double() * x["vs"][i * kv + p, :n, None].double()
            for g in range(p * h // kv, (p + 1) * h // kv):
                out[i, :, g] = _attention64(x["q"][i, :, g].double(), k, v, math.sqrt(d), limit)
    return out


def _exact_attn_valid(c, seed):
    x = _attn_valid_inputs(c, seed)
    b, h, kv, new = c["batch"], c["heads"], c["kv_heads"], c["new"]
    out = torch.empty(x["q"].shape, dtype=torch.float64, device="cuda")
    limit = c["valid"] + 1 + torch.arange(new, device="cuda")
    for i in range(b):
        for p in range(kv):
            k, v = (torch.cat([x[o][i * kv + p, :c["valid"]], x[w][i * kv + p]]).double()
                    for o, w in (("kp", "kn"), ("vp", "vn")))
            for g in range(p * h // kv, (p + 1) * h // kv):
                out[i, g] = _attention64(x["q"][i, g].double(), k, v, math.sqrt(c["head_dim"]), limit)
    return out


def _exact_w8a8(c, seed):
    x = _w8a8_inputs(c, seed)
    w = x["w"]
    if c["tier"] == "i4":
        w = torch.stack([w & 15, w >> 4], -1).view(c["n"], c["k"]).to(torch.int8)
        w = torch.where(w >= 8, w - 16, w)
    elif c["tier"] == "e8cb":
        w = x["codebook"][w.long()].view(c["n"], c["k"])
    q, scale = _quant_rows(x["a"])
    y = (q.double() @ w.double().t().contiguous()) * scale.double() * x["scales"].double()[None, :]
    y = y + x["r"].double() if x["r"] is not None else y
    return _act64(c["act"], y) if c["act"] != "none" else y


def _rms64(x, gain, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * gain.double()


def _rope64(x, cos, sin):
    half = x.shape[-1] // 2
    turned = torch.cat([-x[..., half:], x[..., :half]], -1)
    return x * cos.double().view(x.shape) + turned * sin.double().view(x.shape)


def _exact_decoder(c, seed):
    x = _decoder_inputs(c, seed)
    cfg, w, rows, pos = x["cfg"], x["weights"], x["rows"], x["pos"]
    b, h, kv, d = cfg.batch, cfg.heads, cfg.kv_heads, cfg.head_dim
    cos_q, sin_q, cos_k, sin_k = x["ports"][3:7]
    y = w["embedding"][x["ports"][0].long().view(-1)].double()
    limit = pos + 1 + torch.arange(rows, device="cuda")
    for layer in range(cfg.layers):
        lw = {k: v.double() for k, v in w[f"l{layer}"].items()}
        kq, ks, vq, vs = x["caches"][4 * layer:4 * layer + 4]
        n = _rms64(y, lw["attn_norm"], cfg.eps)
        q = _rope64((n @ lw["wq"]).view(b, rows, h, d), cos_q, sin_q)
        k = _rope64((n @ lw["wk"]).view(b, rows, kv, d), cos_k, sin_k)
        v = (n @ lw["wv"]).view(b, rows, kv, d)
        a = torch.empty((b, rows, h, d), dtype=torch.float64, device="cuda")
        for i in range(b):
            for p in range(kv):
                old = slice(0, pos)
                both = []
                for new, cq, cs in ((k, kq, ks), (v, vq, vs)):
                    nq, ns = _quant_rows(new[i, :, p])
                    before = cq[i * kv + p, old].double() * cs[i * kv + p, old, None].double()
                    both.append(torch.cat([before, nq.double() * ns.double()]))
                for g in range(p * h // kv, (p + 1) * h // kv):
                    a[i, :, g] = _attention64(q[i, :, g], both[0], both[1], math.sqrt(d), limit)
        y = y + a.view(b * rows, h * d) @ lw["wo"]
        n = _rms64(y, lw["ffn_norm"], cfg.eps)
        y = y + (_act64("silu", n @ lw["wg"]) * (n @ lw["wu"])) @ lw["wd"]
    y = _rms64(y.view(b, rows, -1)[:, -1], w["final_norm"], cfg.eps)
    # the caches hold levels, and levels have no 64-bit value
    return {"logits": y @ w["lm_head"].double(), "caches": [None] * len(x["caches"])}


def exact(case, seed):
    """What `run` returns for these inputs, in 64 bits; None where an output is whole numbers."""
    kind = case["kind"]
    if kind == "act":
        return _act64(case["act"], _act_inputs(case, seed)["x"].double())
    if kind == "kv_append":
        return None
    if kind == "matmul":
        x = _matmul_inputs(case, seed)
        y = x["a"].double() @ x["b"].double()
        if x["r"] is not None:
            y = y + x["r"].double()
        e = case["epilogue"]
        return y if e in ("none", "add") else _act64("gelu" if e == "act" else "silu", y)
    if kind in ("attn_i8", "attn_rows"):
        return _exact_attn_i8(case, seed)
    if kind == "attn_valid":
        return _exact_attn_valid(case, seed)
    if kind == "w8a8":
        return _exact_w8a8(case, seed)
    return _exact_decoder(case, seed)
