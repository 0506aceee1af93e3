"""Performance cases: the calls a program serving an INT4 model makes, each through its public entry point.

  listed()   twelve cases over the range in use
  draw(rng)  one more case of the same ranges
  prepare / run / work / tolerance / exact   one case's inputs, call, cost, allowed error and 64-bit value

The operations (a case's "op"):
  proj     one quantized projection: INT4 weights at f16, bf16 or fp8 matrix-core precision, INT4 weights on
           Q8 activations, or INT8 weights -- from a decode step's row to a prefill chunk's 2048
  ffn      a layer's FFN block (gate + up + SiLU, then down) with AWQ scales
  attend   K / V written to the cache and attention over it: TurboQuant or FP16 cache, decode (one token per
           sequence) or a prefill chunk, one sequence or a batch of sequences of different lengths
  decoder  a whole model: reset, prefill of a prompt, then decode steps; the logits of every call

Weights are N(0, 0.02) quantized in groups of 128, AWQ scales U[0.5, 2], activations N(0, 1) with 1 % of the
channels x20, K / V N(0, 1) with four channels per head x10.
"""
import math

import numpy as np
import torch

from ironmill_amd import Device, ops, quant

GROUP = 128
HEAD = 128
EPS = 1e-6
THETA = 1e6


def listed():
    return [
        # the smallest projection in use: one decode row over a 1024 x 1024 weight, where the launch counts
        dict(name="proj_1024_b1", op="proj", kind="int4_f16", m=1, n=1024, k=1024, awq=False),
        # the decode FFN of a 2560-wide model, one sequence: the call that a decode step spends most time in
        dict(name="ffn_b1", op="ffn", m=1, hidden=2560, inter=9728),
        # the same FFN for a dozen sequences decoded together
        dict(name="ffn_b12", op="ffn", m=12, hidden=2560, inter=9728),
        # the same FFN over a prompt chunk of an uneven length
        dict(name="ffn_m777", op="ffn", m=777, hidden=2560, inter=9728),
        # decode on Q8 activations, three sequences
        dict(name="q8_b3", op="proj", kind="int4_q8", m=3, n=9728, k=2560, awq=False),
        # a sensitive layer kept in INT8, over a short prompt
        dict(name="int8_m200", op="proj", kind="int8", m=200, n=2560, k=9728, awq=True),
        # prefill GEMMs: a full chunk at bf16, an uneven one at fp8
        dict(name="gemm_bf16_m2048", op="proj", kind="int4_bf16", m=2048, n=9728, k=2560, awq=True),
        dict(name="gemm_fp8_m509", op="proj", kind="int4_fp8", m=509, n=2560, k=9728, awq=True),
        # batched decode over long TurboQuant caches of different lengths
        dict(name="tq_decode_b16_32k", op="attend", cache="tq", batch=16, heads=32, kv_heads=8, ctx=32768, tokens=1,
             ragged=True),
        # a prefill chunk against a long TurboQuant cache
        dict(name="tq_prefill_t512_8k", op="attend", cache="tq", batch=1, heads=32, kv_heads=8, ctx=8192, tokens=512,
             ragged=False),
        # a prefill chunk of two sequences of different lengths on the FP16 cache, GQA 2
        dict(name="fp16_prefill_t301", op="attend", cache="fp16", batch=2, heads=16, kv_heads=8, ctx=2500, tokens=301,
             ragged=True),
        # a whole call: a 200-token prompt for two sequences, then eight decode steps (four layers, 151936 tokens)
        dict(name="generate", op="decoder", cache="tq", batch=2, hidden=2560, inter=9728, layers=4, heads=32,
             kv_heads=8, vocab=151936, prompt=200, steps=8),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _groups(rng, lo, hi):
    return GROUP * _log(rng, lo // GROUP, hi // GROUP)


def _draw(rng):
    op = rng.choice(["proj", "proj", "proj", "ffn", "ffn", "attend", "attend", "attend", "decoder"])
    if op == "proj":
        kind = rng.choice(["int4_f16", "int4_f16", "int4_bf16", "int4_fp8", "int4_q8", "int8"])
        return dict(op=op, kind=kind, m=_log(rng, 1, 2048), n=_log(rng, 512, 16384), k=_groups(rng, 512, 12288),
                    awq=kind != "int4_q8" and rng.random() < 0.6)
    if op == "ffn":
        return dict(op=op, m=_log(rng, 1, 1024), hidden=_groups(rng, 1024, 4096), inter=_groups(rng, 2048, 12288))
    if op == "attend":
        ctx = _log(rng, 100, 32768)
        tokens = 1 if rng.random() < 0.5 else min(ctx, _log(rng, 2, 1024))
        kv = rng.choice([4, 8])
        return dict(op=op, cache=rng.choice(["tq", "fp16"]), batch=_log(rng, 1, 16), heads=kv * rng.choice([1, 2, 4]),
                    kv_heads=kv, ctx=ctx, tokens=tokens, ragged=rng.random() < 0.5)
    kv = rng.choice([4, 8])
    return dict(op=op, cache=rng.choice(["tq", "fp16"]), batch=_log(rng, 1, 8), hidden=_groups(rng, 1024, 2560),
                inter=_groups(rng, 2048, 9728), layers=rng.randint(1, 3), heads=kv * rng.choice([2, 4]), kv_heads=kv,
                vocab=_log(rng, 8192, 65536), prompt=_log(rng, 8, 400), steps=_log(rng, 2, 12))


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= most:
            return c


# ------------------------------------------------------------------------------------------------- cost


def _weight_bytes(n, k, bits=4):
    return n * k * bits / 8 + 4 * n * (k // GROUP)


def _visible(case):
    """Positions attended to, summed over the query tokens of all sequences, and positions held."""
    seen = held = 0
    for length in _lengths(case):
        held += length
        t = case["tokens"]
        seen += t * length - t * (t - 1) // 2
    return seen, held


def work(case):
    if case["op"] == "proj":
        m, n, k = case["m"], case["n"], case["k"]
        bits = 8 if case["kind"] == "int8" else 4
        return dict(bytes=_weight_bytes(n, k, bits) + 2 * m * (n + k) + (2 * k if case["awq"] else 0),
                    flops=2 * m * n * k)
    if case["op"] == "ffn":
        m, h, f = case["m"], case["hidden"], case["inter"]
        return dict(bytes=3 * _weight_bytes(f, h) + 2 * (h + f) + 2 * m * (2 * h + f), flops=6 * m * h * f)
    if case["op"] == "attend":
        seen, held = _visible(case)
        row = (2 * HEAD + 12) if case["cache"] == "tq" else 4 * HEAD
        io = case["batch"] * case["tokens"] * HEAD * 2 * (2 * case["heads"] + 2 * case["kv_heads"])
        return dict(bytes=held * case["kv_heads"] * row + io, flops=4 * HEAD * case["heads"] * seen)
    b, h, f, layers = case["batch"], case["hidden"], case["inter"], case["layers"]
    qd, kvd = case["heads"] * HEAD, case["kv_heads"] * HEAD
    dense = h * (2 * qd + 2 * kvd) + 3 * h * f
    layer_bytes = _weight_bytes(2 * qd + 2 * kvd, h) + 3 * _weight_bytes(f, h)
    head_bytes = _weight_bytes(case["vocab"], h)
    t, steps = case["prompt"], case["steps"]
    row = (2 * HEAD + 12) if case["cache"] == "tq" else 4 * HEAD
    kv_rows = sum(t + i + 1 for i in range(steps)) + t
    seen = t * (t + 1) // 2 + sum(t + i + 1 for i in range(steps))
    return dict(
        bytes=(steps + 1) * (layers * layer_bytes + head_bytes + 2 * b * case["vocab"])
        + layers * b * kv_rows * case["kv_heads"] * row,
        flops=2 * b * (layers * dense * (t + steps) + h * case["vocab"] * (steps + 1))
        + layers * b * 4 * HEAD * case["heads"] * seen)


# ----------------------------------------------------------------------------------------------- inputs

_shared = {}


def _device():
    """The program's device and its one stream."""
    if not _shared:
        _shared["dev"] = Device(0)
        _shared["stream"] = _shared["dev"].stream()
    return _shared["dev"], _shared["stream"]


def _gen(seed):
    g = torch.Generator("cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _activations(g, m, k):
    x = _normal(g, m, k)
    x[:, torch.randperm(k, generator=g, device="cuda")[:max(1, k // 100)]] *= 20
    return x


def _awq(g, k):
    return (0.5 + 1.5 * torch.rand(k, generator=g, device="cuda")).half()


def _kv(g, b, t, heads):
    x = _normal(g, b, t, heads, HEAD)
    hot = torch.rand(heads, HEAD, generator=g, device="cuda").argsort(-1) < 4
    return torch.where(hot, 10 * x, x).half()


def _quantized(g, n, k, awq=None, levels=16):
    """Codes, scales, zero-points of W ~ N(0, 0.02) (times the AWQ scales), group by group, as arrays on the GPU."""
    codes = torch.empty(n, k, dtype=torch.uint8, device="cuda")
    scales = torch.empty(n, k // GROUP, dtype=torch.float16, device="cuda")
    zeros = torch.empty_like(scales)
    for i in range(0, n, 16384):   # by rows: the largest weights have 151936
        w = 0.02 * _normal(g, min(16384, n - i), k)
        if awq is not None:
            w *= awq.float()
        w = w.view(w.shape[0], -1, GROUP)
        lo, hi = w.amin(-1, keepdim=True), w.amax(-1, keepdim=True)
        s = (hi - lo) / (levels - 1)
        z = torch.round(-lo / s)
        codes[i:i + 16384] = torch.round(w / s + z).clamp(0, levels - 1).to(torch.uint8).view(-1, k)
        scales[i:i + 16384], zeros[i:i + 16384] = s.squeeze(-1).half(), z.squeeze(-1).half()
    return codes, scales, zeros


class _Int4:
    """An INT4 weight on the GPU, and the handle that the calls take."""

    def __init__(self, g, n, k, awq=None):
        codes, self.scales, self.zeros = _quantized(g, n, k, awq)
        self.data = codes[:, 0::2] | (codes[:, 1::2] << 4)
        self.awq = awq
        self.handle = ops.AffineQuantizedWeight.from_pointers(
            self.data.data_ptr(), self.scales.data_ptr(), self.zeros.data_ptr(),
            None if awq is None else awq.data_ptr(), n, k)

    def dense(self, start=0, stop=None):
        d = self.data[start:stop]
        codes = torch.stack((d & 15, d >> 4), -1).reshape(d.shape[0], -1, GROUP)
        w = (codes.double() - self.zeros[start:stop].double()[..., None]) * self.scales[start:stop].double()[..., None]
        return w.view(d.shape[0], -1)


def _lloyd_max(levels):
    """Lloyd-Max levels and boundaries of N(0, 1 / HEAD)."""
    p = (torch.arange(levels, dtype=torch.float64) + 0.5) / levels
    c = math.sqrt(2) * torch.erfinv(2 * p - 1)

    def density(x):
        return torch.exp(-x * x / 2) / math.sqrt(2 * math.pi)

    def below(x):
        return 0.5 * (1 + torch.erf(x / math.sqrt(2)))

    inf = torch.tensor([math.inf], dtype=torch.float64)
    for _ in range(300):
        b = torch.cat((-inf, (c[1:] + c[:-1]) / 2, inf))
        c = (density(b[:-1]) - density(b[1:])) / (below(b[1:]) - below(b[:-1]))
    c /= math.sqrt(HEAD)
    return c.float(), ((c[1:] + c[:-1]) / 2).float()


def _hadamard():
    h = torch.ones(1, 1, dtype=torch.float64)
    while h.shape[0] < HEAD:
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    return h


def _tables():
    """TurboQuant tables as a program that makes its own hands them over, and the same on the GPU in 64 bits."""
    if "tables" not in _shared:
        r = np.random.default_rng(42)
        kc, kb = _lloyd_max(128)
        vc, vb = _lloyd_max(256)
        host = dict(signs=np.where(r.random(HEAD) < 0.5, -1, 1).astype(np.float32), k_codebook=kc.numpy(),
                    k_bounds=kb.numpy(), v_codebook=vc.numpy(), v_bounds=vb.numpy(),
                    qjl=r.standard_normal((HEAD, HEAD)).astype(np.float32))
        t = {k: torch.from_numpy(v).cuda().double() for k, v in host.items()}
        t["rotate"] = t["signs"][:, None] * _hadamard().cuda() * t["signs"] / math.sqrt(HEAD)
        _shared["host_tables"], _shared["tables"] = host, t
    return _shared["host_tables"], _shared["tables"]


def _model_tables():
    if "tq" not in _shared:
        _shared["tq"] = ops.TurboQuantModel(_device()[0], HEAD, 8, 42, host_tables=_tables()[0])
    return _shared["tq"]


def _tq_codes(x, is_k):
    """Codes, scale and residual norm of rows x [..., HEAD]: rotated, scaled to length 1, nearest level; K also the
    signs of the residual's projection."""
    t = _tables()[1]
    u = x.double() @ t["rotate"]
    scale = u.norm(dim=-1, keepdim=True)
    u = u / scale
    if not is_k:
        return torch.bucketize(u, t["v_bounds"], right=True).to(torch.uint8), scale.squeeze(-1).float(), None
    index = torch.bucketize(u, t["k_bounds"], right=True)
    u = u - t["k_codebook"][index]
    signs = (u @ t["qjl"].T) >= 0
    return (index + 128 * signs).to(torch.uint8), scale.squeeze(-1).float(), u.norm(dim=-1).float()


def _tq_keys(codes, scale, norm):
    """The (rotated) keys that codes stand for."""
    t = _tables()[1]
    sign = (codes >= 128).double() * 2 - 1
    k = t["k_codebook"][(codes & 127).long()]
    k = k + math.sqrt(2 / math.pi) / HEAD * norm.double()[..., None] * (sign @ t["qjl"])
    return k * scale.double()[..., None]


def _tq_values(codes, scale):
    return _tables()[1]["v_codebook"][codes.long()] * scale.double()[..., None]


def _softmax_attention(q, k, v, first):
    """q [t, heads, d], k / v [kv_heads, n, d] in 64 bits; token i sees the first `first` + i + 1 positions."""
    t, heads, _ = q.shape
    group = heads // k.shape[0]
    seen = torch.arange(k.shape[1], device="cuda") <= first + torch.arange(t, device="cuda")[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        s = (q[:, h] @ k[h // group].T) / math.sqrt(HEAD)
        out[:, h] = s.masked_fill(~seen, -math.inf).softmax(-1) @ v[h // group]
    return out


def _lengths(case):
    """Positions of each sequence once the call's tokens are in the cache."""
    if not case["ragged"]:
        return [case["ctx"]] * case["batch"]
    least = max(case["tokens"], case["ctx"] // 4)
    r = np.random.default_rng(case["ctx"] + case["batch"])
    return [int(v) for v in r.integers(least, case["ctx"] + 1, case["batch"])]


class _State:
    pass


def _prepare_proj(case, g):
    s = _State()
    m, n, k = case["m"], case["n"], case["k"]
    wide = case["kind"] in ("int4_bf16", "int4_fp8")
    s.x = _activations(g, m, k).to(torch.bfloat16 if wide else torch.float16)
    s.awq = _awq(g, k) if case["awq"] else None
    if case["kind"] == "int8":
        s.w = _quantized(g, n, k, s.awq, levels=256)
        c, sc, z = (t.cpu().numpy() for t in s.w)
        s.handle = ops.AffineInt8Weight(_device()[0], quant.QuantizedInt8(
            data=c, scales=sc, zeros=z, scales_f32=sc.astype(np.float32), zeros_f32=z.astype(np.float32),
            awq=None if s.awq is None else s.awq.cpu().numpy(), n=n, k=k))
    else:
        s.w = _Int4(g, n, k, s.awq)
        s.handle = s.w.handle
    if case["kind"] == "int4_q8":
        s.q8 = torch.empty(m, k, dtype=torch.int8, device="cuda")
        s.q8_scales = torch.empty(m, k // GROUP, dtype=torch.float32, device="cuda")
    s.y = torch.empty(m, n, dtype=s.x.dtype, device="cuda")
    return s


def _run_proj(case, s):
    stream, m = _device()[1], case["m"]
    x, y = s.x.data_ptr(), s.y.data_ptr()
    if case["kind"] == "int8":
        ops.encode_projection_int8(stream, x, s.handle, y, m)
    elif case["kind"] == "int4_q8":
        ops.encode_projection_int4_q8(stream, x, s.handle, y, m, s.q8.data_ptr(), s.q8_scales.data_ptr())
        return s.y, s.q8, s.q8_scales
    elif case["kind"] == "int4_f16":
        ops.encode_projection(stream, x, s.handle, y, m)
    else:
        ops.encode_affine_gemm_int4(stream, x, m, s.handle, y,
                                    ops.GEMM_BF16 if case["kind"] == "int4_bf16" else ops.GEMM_FP8_E4M3)
    return s.y


def _project(x, w, awq):
    """x / awq times a weight's dense rows, some thousand rows at a time."""
    x = x.double() if awq is None else x.double() / awq.double()
    n = w.data.shape[0]
    return torch.cat([x @ w.dense(i, min(n, i + 8192)).T for i in range(0, n, 8192)], -1)


def _exact_proj(case, s):
    x, kind = s.x, case["kind"]
    if kind == "int8":
        codes, scales, zeros = (t.double() for t in s.w)
        w = (codes.view(case["n"], -1, GROUP) - zeros[..., None]) * scales[..., None]
        return (x.double() / (1 if s.awq is None else s.awq.double())) @ w.view(case["n"], -1).T
    if kind == "int4_f16":
        return _project(x, s.w, s.awq)
    if kind == "int4_q8":
        v = x.float().view(case["m"], -1, GROUP)
        top = v.abs().amax(-1, keepdim=True)
        q = torch.round(v * (127.0 / top)).clamp(-127, 127)
        y = (q.double() * (top / 127.0).double()).view(case["m"], -1)
        return _project(y, s.w, None), q.to(torch.int8).view(case["m"], -1), (top / 127.0).squeeze(-1)
    # x / awq is rounded once, to bf16 or (saturating) to fp8
    a = x.float() if s.awq is None else x.float() / s.awq.float()
    a = a.bfloat16() if kind == "int4_bf16" else a.clamp(-448, 448).to(torch.float8_e4m3fn).float()
    return _project(a, s.w, None)


def _prepare_ffn(case, g):
    s = _State()
    m, h, f = case["m"], case["hidden"], case["inter"]
    s.x = _activations(g, m, h).half()
    awq_h, awq_f = _awq(g, h), _awq(g, f)
    s.gate, s.up, s.down = _Int4(g, f, h, awq_h), _Int4(g, f, h, awq_h), _Int4(g, h, f, awq_f)
    s.act = torch.empty(m, f, dtype=torch.float16, device="cuda")
    s.y = torch.empty(m, h, dtype=torch.float16, device="cuda")
    return s


def _run_ffn(case, s):
    ops.encode_ffn_block_int4(_device()[1], s.x.data_ptr(), s.gate.handle, s.up.handle, s.down.handle,
                              s.act.data_ptr(), s.y.data_ptr(), case["m"])
    return s.act, s.y


def _exact_ffn(case, s):
    a = _project(s.x, s.gate, s.gate.awq)
    a = a * torch.sigmoid(a) * _project(s.x, s.up, s.gate.awq)
    return a, _project(a, s.down, s.down.awq)


def _prepare_attend(case, g):
    s = _State()
    dev, stream = _device()
    b, t, ctx, kv = case["batch"], case["tokens"], case["ctx"], case["kv_heads"]
    s.q = _normal(g, b, t, case["heads"], HEAD).half()
    s.k, s.v = _kv(g, b, t, kv), _kv(g, b, t, kv)
    s.out = torch.empty_like(s.q)
    s.lens = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")
    s.positions = s.lens - t
    # the positions before the call's own tokens; what the cache holds after them is not read
    s.old = _kv(g, b, ctx, kv), _kv(g, b, ctx, kv)
    torch.cuda.synchronize()
    old = [x.data_ptr() for x in s.old]
    if case["cache"] == "tq":
        s.tq = _model_tables()
        s.cache = ops.TurboQuantKvCache(dev, b, kv, HEAD, ctx)
        ops.encode_turboquant_cache_write_kv(stream, s.tq, s.cache, *old, ctx, 0)
    else:
        s.cache = ops.Fp16KvCache(dev, b, kv, HEAD, ctx)
        for x, is_k in zip(old, (True, False)):
            ops.encode_kv_scatter(stream, s.cache, x, ctx, 0, is_k)
    stream.sync()
    return s


def _run_attend(case, s):
    stream, t, c = _device()[1], case["tokens"], s.cache
    q, k, v, out = s.q.data_ptr(), s.k.data_ptr(), s.v.data_ptr(), s.out.data_ptr()
    heads, ctx = case["heads"], case["ctx"]
    if case["cache"] == "tq":
        if case["ragged"] or case["batch"] > 1 or t > 1:
            ops.encode_turboquant_cache_write_kv(stream, s.tq, c, k, v, t, 0, positions=s.positions.data_ptr())
            ops.encode_turboquant_attention(stream, s.tq, c, q, heads, ctx, out, seq_lens=s.lens.data_ptr(),
                                            token_count=t)
        else:
            ops.encode_kv_cache_and_attention(stream, s.tq, c, k, v, q, heads, ctx - 1, out)
    elif case["ragged"]:
        ops.encode_kv_scatter(stream, c, k, t, 0, True, positions=s.positions.data_ptr())
        ops.encode_kv_scatter(stream, c, v, t, 0, False, positions=s.positions.data_ptr())
        ops.encode_fp16_attention(stream, c, q, heads, ctx, out, token_count=t, seq_lens=s.lens.data_ptr())
    else:
        ops.encode_fp16_kv_cache_and_attention(stream, c, k, v, q, heads, ctx - t, out, token_count=t)
    return s.out


def _exact_attend(case, s):
    t, out, rotate = case["tokens"], [], _tables()[1]["rotate"]
    for i, length in enumerate(_lengths(case)):
        k, v = (torch.cat((old[i, :length - t], new[i])).transpose(0, 1)
                for old, new in zip(s.old, (s.k, s.v)))
        q = s.q[i].double()
        if case["cache"] == "fp16":
            out.append(_softmax_attention(q, k.double(), v.double(), length - t))
        else:
            o = _softmax_attention(q @ rotate, _tq_keys(*_tq_codes(k, True)), _tq_values(*_tq_codes(v, False)[:2]),
                                   length - t)
            out.append(o @ rotate.T)
    return torch.stack(out)


def _prepare_decoder(case, g):
    s = _State()
    dev = _device()[0]
    b, h, f = case["batch"], case["hidden"], case["inter"]
    qd, kvd = case["heads"] * HEAD, case["kv_heads"] * HEAD

    def norm(n):
        return (0.8 + 0.4 * torch.rand(n, generator=g, device="cuda")).half()

    s.layers = []
    for _ in range(case["layers"]):
        a, d = _awq(g, h), _awq(g, f)
        s.layers.append(dict(
            input_norm=norm(h), post_attn_norm=norm(h), q_norm=norm(HEAD), k_norm=norm(HEAD),
            q_proj=_Int4(g, qd, h, a), k_proj=_Int4(g, kvd, h, a), v_proj=_Int4(g, kvd, h, a), o_proj=_Int4(g, h, qd),
            gate_proj=_Int4(g, f, h, a), up_proj=_Int4(g, f, h, a), down_proj=_Int4(g, h, f, d)))
    s.embedding = _normal(g, case["vocab"], h).half()
    s.final_norm = norm(h)
    s.head = _Int4(g, case["vocab"], h)
    total = case["prompt"] + case["steps"]
    s.ids = torch.randint(case["vocab"], (b, total), generator=g, device="cuda").int()
    s.prompt = s.ids[:, :case["prompt"]].contiguous()
    s.steps = s.ids[:, case["prompt"]:].T.contiguous()
    s.logits = torch.empty(case["steps"] + 1, b, case["vocab"], dtype=torch.float16, device="cuda")
    s.decoder = ops.Decoder(dev, hidden_size=h, intermediate_size=f, num_layers=case["layers"],
                            num_heads=case["heads"], num_kv_heads=case["kv_heads"], head_dim=HEAD,
                            vocab_size=case["vocab"], max_seq_len=total, batch=b, rms_eps=EPS, rope_theta=THETA,
                            kv_cache="turboquant" if case["cache"] == "tq" else "fp16")
    for i, layer in enumerate(s.layers):
        s.decoder.set_layer(i, **{k: w.handle if isinstance(w, _Int4) else w.data_ptr() for k, w in layer.items()})
    s.decoder.set_model(s.embedding.data_ptr(), s.final_norm.data_ptr(), s.head.handle)
    if case["cache"] == "tq":
        s.decoder.set_tq_tables(_model_tables())
    return s


def _run_decoder(case, s):
    stream, b = _device()[1], case["batch"]
    logits, size = s.logits.data_ptr(), 2 * b * case["vocab"]
    s.decoder.reset(stream)
    s.decoder.prefill(stream, s.prompt.data_ptr(), case["prompt"], logits)
    for i in range(case["steps"]):
        s.decoder.step(stream, s.steps.data_ptr() + 4 * b * i, logits + size * (i + 1))
    return s.logits


def _rms_norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x):
    """x [tokens, heads, HEAD] at positions 0, 1, ..; the tables are f16."""
    half = HEAD // 2
    f = THETA ** (-torch.arange(half, device="cuda", dtype=torch.float64) * 2 / HEAD)
    a = torch.arange(x.shape[0], device="cuda", dtype=torch.float64)[:, None] * f
    c, s = (v.half().double()[:, None] for v in (a.cos(), a.sin()))
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat((lo * c - hi * s, lo * s + hi * c), -1)


def _exact_decoder(case, s):
    """Every token at once, causally: what prefill and the steps compute one after the other."""
    b, t = s.ids.shape
    x = s.embedding[s.ids.long().view(-1)].double()
    rotate = _tables()[1]["rotate"]
    for w in s.layers:
        a = _rms_norm(x, w["input_norm"])
        q, k, v = (_project(a, w[p], w[p].awq).view(b, t, -1, HEAD) for p in ("q_proj", "k_proj", "v_proj"))
        out = torch.empty_like(q)
        for i in range(b):
            qi, ki = _rope(_rms_norm(q[i], w["q_norm"])), _rope(_rms_norm(k[i], w["k_norm"]))
            ki, vi = ki.transpose(0, 1).half().double(), v[i].transpose(0, 1).half().double()
            if case["cache"] == "fp16":
                out[i] = _softmax_attention(qi, ki, vi, 0)
            else:
                o = _softmax_attention(qi @ rotate, _tq_keys(*_tq_codes(ki, True)),
                                       _tq_values(*_tq_codes(vi, False)[:2]), 0)
                out[i] = o @ rotate.T
        x = x + _project(out.view(b * t, -1), w["o_proj"], None)
        a = _rms_norm(x, w["post_attn_norm"])
        g = _project(a, w["gate_proj"], w["gate_proj"].awq)
        g = g * torch.sigmoid(g) * _project(a, w["up_proj"], w["gate_proj"].awq)
        x = x + _project(g, w["down_proj"], w["down_proj"].awq)
    x = x.view(b, t, -1)[:, case["prompt"] - 1:].transpose(0, 1)
    return _project(_rms_norm(x, s.final_norm), s.head, None)


_PREPARE = dict(proj=_prepare_proj, ffn=_prepare_ffn, attend=_prepare_attend, decoder=_prepare_decoder)
_RUN = dict(proj=_run_proj, ffn=_run_ffn, attend=_run_attend, decoder=_run_decoder)
_EXACT = dict(proj=_exact_proj, ffn=_exact_ffn, attend=_exact_attend, decoder=_exact_decoder)


def prepare(case, seed):
    s = _PREPARE[case["op"]](case, _gen(seed))
    s.case = case
    torch.cuda.synchronize()   # the calls run on the library's own stream
    return s


def run(state):
    return _RUN[state.case["op"]](state.case, state)


def tolerance(case):
    """Four times what the results are off by against exact(): the rounding of the outputs (f16 2e-4, bf16 1.7e-3),
    of the FFN's f16 activation, of the attention's f16 weights, and in a whole model of every stored row.  q8 codes
    are whole numbers: a value on a boundary may round either way."""
    if case["op"] == "decoder":
        return {"rel": 1.5e-2, "max": 0.2}
    if case["op"] == "proj" and case["kind"] in ("int4_bf16", "int4_fp8"):
        return {"rel": 7e-3, "max": 2e-2}
    if case["op"] == "proj" and case["kind"] == "int4_q8":
        return {"rel": 1e-3, "max": 4e-3, "differ": 1e-4}
    return {"rel": 1.5e-3, "max": 1e-2}


def exact(case, seed):
    return _EXACT[case["op"]](case, prepare(case, seed))
