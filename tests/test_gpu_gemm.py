"""GPU parity of the INT4 ops at prefill-sized token counts (the GEMM path:
superblock_matmul_int4, affine_matmul.metal:10-152, reached through
encode_projection at token_count > 1, projection.rs:227-312) against the CPU
oracle's dequantize-then-compute chain.

The GEMM multiplies the exact weight (the code minus its zero point in f16,
the f16 scale applied per group in f32) with x (exact f16) or, with AWQ,
with x / awq carried as f16 hi + lo (~22 bits; rounding it to f16 alone,
as the reference's prefill kernel does, moves outputs by several fp16 steps
where terms cancel).  Tolerance as on the decode path: rel-L2 <= 1e-3
and max-abs <= max(2e-2, 2 fp16 steps of the reference value)
(f16 scales on the GPU, f32 on the CPU path: one step, plus the output
rounding).
"""
import numpy as np
import pytest

import oracle as O
from conftest import assert_close
from ironmill_amd import ops, quant

pytestmark = pytest.mark.gpu


def ulps_for(awq):
    return 2


def weight(n, k, seed, awq):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float16).astype(np.float32)
    s = rng.uniform(0.5, 2.0, k).astype(np.float32) if awq else None
    return w, s


def acts(m, k, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((m, k)).astype(np.float32)
    idx = rng.choice(k, max(1, k // 100), replace=False)
    x[:, idx] *= 20.0
    return x.astype(np.float16)


def exact_weights(q):
    """The uploaded weight exactly, in f64: f16 scale x (code - f16 zero point)."""
    codes = np.empty((q.n, q.k), np.float64)
    codes[:, 0::2] = q.data & 0xF
    codes[:, 1::2] = q.data >> 4
    sc = np.repeat(q.scales.astype(np.float64), q.group_size, axis=1)
    zp = np.repeat(q.zeros.astype(np.float64), q.group_size, axis=1)
    return sc * (codes - zp)


def dense(w, s):
    wq = w if s is None else (w * s[None, :]).astype(np.float32)
    packed, sc, zp = O.quantize_tensor_int4(wq, 128)
    n, k = w.shape
    return O.dequant_affine_int4(packed, sc, zp, n, k, 128), (None if s is None else s.astype(np.float16))


@pytest.mark.parametrize("m,n,k,awq", [
    (32, 1000, 256, False),    # smallest GEMM token count, ragged N
    (64, 2560, 9728, True),    # Qwen3-4B down, split-K
    (200, 1000, 256, False),   # ragged M and N, one K split
    (128, 9728, 2560, True),   # Qwen3-4B gate shape, split-K over 76 x 1 tiles
    (512, 1024, 2560, True),   # BASELINE configs[3] M, smaller N
])
def test_gemm_projection(dev, stream, m, n, k, awq):
    w, s = weight(n, k, m + n, awq)
    x16 = acts(m, k, 3 * m + k)
    wt = ops.AffineQuantizedWeight(dev, quant.quantize_int4(w, awq_scales=s))
    xd, yd = dev.upload(x16), dev.empty((m, n), np.float16)
    ops.encode_projection(stream, xd, wt, yd, m)
    stream.sync()
    wdq, awq16 = dense(w, s)
    ref = O.matvec_f16w(wdq, x16, awq16, nthreads=8)
    assert_close(yd.read(), ref, what=f"gemm m={m} n={n} k={k} awq={awq}", ulps=ulps_for(awq))


@pytest.mark.parametrize("m,n,k", [(512, 9728, 2560), (512, 2560, 9728), (2048, 9728, 2560), (2048, 2560, 9728)])
def test_gemm_configs3_full_shapes(dev, stream, m, n, k):
    """BASELINE configs[3] at its full sizes (M = 512 / 2048, (K, N) = (2560, 9728) and
    (9728, 2560)), AWQ, every output against the oracle."""
    print(f"gemm configs[3] m={m} n={n} k={k}", flush=True)
    w, s = weight(n, k, 7 * m + n, True)
    x16 = acts(m, k, 11 * m + k)
    wt = ops.AffineQuantizedWeight(dev, quant.quantize_int4(w, awq_scales=s))
    xd, yd = dev.upload(x16), dev.empty((m, n), np.float16)
    ops.encode_projection(stream, xd, wt, yd, m)
    stream.sync()
    wdq, awq16 = dense(w, s)
    ref = O.matvec_f16w(wdq, x16, awq16, nthreads=16)
    assert_close(yd.read(), ref, what=f"gemm m={m} n={n} k={k}", ulps=ulps_for(True))


def test_gemm_matches_matvec_at_the_switch(dev, stream):
    """The same rows through the matvec (31 tokens) and the GEMM (32 tokens)."""
    n, k = 512, 1024
    w, s = weight(n, k, 5, True)
    wt = ops.AffineQuantizedWeight(dev, quant.quantize_int4(w, awq_scales=s))
    x16 = acts(32, k, 6)
    y31, y32 = dev.empty((31, n), np.float16), dev.empty((32, n), np.float16)
    ops.encode_projection(stream, dev.upload(x16[:31].copy()), wt, y31, 31)
    ops.encode_projection(stream, dev.upload(x16), wt, y32, 32)
    stream.sync()
    assert_close(y32.read()[:31], y31.read().astype(np.float32), what="gemm vs matvec", ulps=ulps_for(True))


@pytest.mark.parametrize("act", ["silu", "gelu"])
def test_gemm_fused_gate_up(dev, stream, act):
    m, n, k = 48, 9728, 2560
    wg, s = weight(n, k, 41, True)
    wu, _ = weight(n, k, 42, False)
    x16 = acts(m, k, 43)
    gate = ops.AffineQuantizedWeight(dev, quant.quantize_int4(wg, awq_scales=s))
    up = ops.AffineQuantizedWeight(dev, quant.quantize_int4(wu, awq_scales=s))
    xd, out = dev.upload(x16), dev.empty((m, n), np.float16)
    ops.encode_fused_ffn_gate_up_act_int4(stream, xd, gate, up, out, m, use_gelu=(act == "gelu"))
    stream.sync()
    got = out.read().astype(np.float64)
    wdq_g, awq16 = dense(wg, s)
    wdq_u, _ = dense(wu, s)
    ref = O.gate_up_act(wdq_g, wdq_u, x16, awq16, act=act)
    assert_close(got, ref, what=f"gemm fused gate+up {act} vs the CPU path", max_abs=np.inf)
    # Element-wise against the exact value of what the kernel computes: the
    # uploaded codes with their f16 scales and zero points, x / awq unrounded,
    # in f64.  The CPU path rounds each dequantized weight to f16; act(gate) *
    # up amplifies that, and at this shape it alone moves an output ~5 f16
    # steps (row 31, column 8523: exact -6.9241, CPU path -6.9079, 0.98 of
    # max(2e-2, 2 steps)), so the bound there would pass or fail on the
    # rounding direction of a correct result.  Bound: 2 f16 steps of the exact
    # value, plus 2^-16 of the summed magnitudes the f32 accumulation and the
    # hi / lo split of x / awq see, carried through act(gate) * up.
    qg = quant.quantize_int4(wg, awq_scales=s)
    qu = quant.quantize_int4(wu, awq_scales=s)
    xa = x16.astype(np.float64) / s.astype(np.float16).astype(np.float64)[None, :]
    Wg, Wu = exact_weights(qg), exact_weights(qu)
    g, u = xa @ Wg.T, xa @ Wu.T
    mg, mu = np.abs(xa) @ np.abs(Wg).T, np.abs(xa) @ np.abs(Wu).T
    if act == "silu":
        a = g / (1.0 + np.exp(-g))
    else:
        a = 0.5 * g * (1.0 + np.tanh(0.7978845608028654 * (g + 0.044715 * g ** 3)))
    exact = a * u
    slack = 2.0 ** -16 * 1.1 * (np.abs(u) * mg + np.abs(a) * mu)
    bound = 2.0 * np.spacing(np.abs(exact).astype(np.float16)).astype(np.float64) + slack
    err = np.abs(got - exact)
    worst = np.unravel_index(np.argmax(err / bound), err.shape)
    assert np.all(err <= bound), (f"gemm fused gate+up {act}: |got - exact| {err[worst]:.3e} > "
                                  f"{bound[worst]:.3e} at {worst} (exact {exact[worst]:.5f}, got {got[worst]:.5f})")


def test_gemm_batched_gate_up(dev, stream):
    m, n, k = 33, 2048, 1024
    wg, s = weight(n, k, 51, True)
    wu, _ = weight(n, k, 52, False)
    x16 = acts(m, k, 53)
    gate = ops.AffineQuantizedWeight(dev, quant.quantize_int4(wg, awq_scales=s))
    up = ops.AffineQuantizedWeight(dev, quant.quantize_int4(wu, awq_scales=s))
    xd = dev.upload(x16)
    go, uo = dev.empty((m, n), np.float16), dev.empty((m, n), np.float16)
    ops.encode_batched_affine_matvec_int4(stream, xd, gate, go, up, uo, m)
    stream.sync()
    wdq_g, awq16 = dense(wg, s)
    wdq_u, _ = dense(wu, s)
    assert_close(go.read(), O.matvec_f16w(wdq_g, x16, awq16, nthreads=8), what="gemm gate", ulps=ulps_for(True))
    assert_close(uo.read(), O.matvec_f16w(wdq_u, x16, awq16, nthreads=8), what="gemm up", ulps=ulps_for(True))


# the residual + norm rows kernel at 1, 2 and 8 register chunks per thread,
# and past those (K > 16384: the chunks beyond are read again)
@pytest.mark.parametrize("m,n,k", [(40, 4096, 2560), (33, 256, 1024), (32, 128, 16384), (34, 128, 16512)])
def test_gemm_fused_residual_norm(dev, stream, m, n, k):
    eps = 1e-6
    w, s = weight(n, k, 61, True)
    rng = np.random.default_rng(62)
    a = rng.standard_normal((m, k)).astype(np.float16)
    b = (rng.standard_normal((m, k)) * 0.5).astype(np.float16)
    gamma = rng.uniform(0.5, 1.5, k).astype(np.float16)
    wt = ops.AffineQuantizedWeight(dev, quant.quantize_int4(w, awq_scales=s))
    ad, bd, gd = dev.upload(a), dev.upload(b), dev.upload(gamma)
    y = dev.empty((m, n), np.float16)
    res = dev.empty((m, k), np.float16)
    nrm = dev.empty((m, k), np.float16)
    ops.encode_fused_residual_norm_affine_matvec_int4(stream, ad, bd, gd, res, wt, y, nrm, eps, m)
    stream.sync()
    wdq, awq16 = dense(w, s)
    y_ref, res_ref, nrm_ref = O.fused_residual_norm_matvec(a, b, gamma, wdq, eps, awq16)
    assert_close(y.read(), y_ref, what="gemm resnorm y", ulps=ulps_for(True))
    assert np.array_equal(res.read().view(np.uint16), res_ref.view(np.uint16))
    assert_close(nrm.read(), nrm_ref.astype(np.float32), rel=1e-3, max_abs=2e-3, what="gemm normed")


@pytest.mark.parametrize("m,n,k,awq", [
    (32, 256, 128, True),      # one group, the smallest tile, one column tile
    (33, 257, 1152, True),     # one row into a second tile half, one column past a tile, odd group count
    (65, 513, 1152, False),    # without AWQ: the activation straight from x, constants read in place
    (130, 31, 256, False),     # fewer columns than one fragment
])
def test_gemm_tile_edges(dev, stream, m, n, k, awq):
    """The GEMM at the edges of its tiles against the exact value of the uploaded weights
    (f64): one f16 step plus 2^-16 of the summed magnitudes (the f32 sums, and x / awq's ~22 bits)."""
    w, s = weight(n, k, m + n, awq)
    q = quant.quantize_int4(w, awq_scales=s)
    x16 = acts(m, k, 3 * m + k)
    xd, yd = dev.upload(x16), dev.empty((m, n), np.float16)
    ops.encode_projection(stream, xd, ops.AffineQuantizedWeight(dev, q), yd, m)
    stream.sync()
    a = x16.astype(np.float64) if s is None else x16.astype(np.float64) / s.astype(np.float16).astype(np.float64)
    W = exact_weights(q)
    exact = a @ W.T
    bound = np.spacing(np.abs(exact).astype(np.float16)).astype(np.float64) + 2.0 ** -16 * (np.abs(a) @ np.abs(W).T)
    err = np.abs(yd.read().astype(np.float64) - exact)
    assert np.all(err <= bound), f"m={m} n={n} k={k} awq={awq}: worst {np.max(err / bound):.2f} of the bound"


@pytest.mark.parametrize("m,n,k,awq", [
    (9, 12801, 1024, True),    # the fewest rows, one column past a tile, two blocks of groups
    (16, 7001, 1152, False),   # a full half tile, an odd group count, unsplit and split blocks
    (17, 6007, 1152, True),    # one row into the second half
    (31, 2560, 9728, True),    # split K
])
def test_gemm_rows_kernel(dev, stream, m, n, k, awq):
    """The one-launch kernel of 9 to 31 rows, to test_gemm_tile_edges' bound."""
    assert m * n * k >= 115e6
    test_gemm_tile_edges(dev, stream, m, n, k, awq)


@pytest.mark.parametrize("act", ["silu", "gelu"])
def test_gemm_rows_gate_up(dev, stream, act):
    """Gate and up of 12 rows in one launch, both epilogues: within 2 f16 steps of the exact
    value plus test_gemm_fused_gate_up's slack."""
    m, n, k = 12, 5121, 1024
    wg, s = weight(n, k, 141, True)
    wu, _ = weight(n, k, 142, False)
    x16 = acts(m, k, 143)
    qg, qu = quant.quantize_int4(wg, awq_scales=s), quant.quantize_int4(wu, awq_scales=s)
    out = dev.empty((m, n), np.float16)
    ops.encode_fused_ffn_gate_up_act_int4(stream, dev.upload(x16), ops.AffineQuantizedWeight(dev, qg),
                                          ops.AffineQuantizedWeight(dev, qu), out, m, use_gelu=(act == "gelu"))
    stream.sync()
    xa = x16.astype(np.float64) / s.astype(np.float16).astype(np.float64)
    Wg, Wu = exact_weights(qg), exact_weights(qu)
    g, u = xa @ Wg.T, xa @ Wu.T
    mg, mu = np.abs(xa) @ np.abs(Wg).T, np.abs(xa) @ np.abs(Wu).T
    a = g / (1.0 + np.exp(-g)) if act == "silu" else 0.5 * g * (1.0 + np.tanh(0.7978845608028654 * (g + 0.044715 * g ** 3)))
    bound = 2.0 * np.spacing(np.abs(a * u).astype(np.float16)).astype(np.float64) \
        + 2.0 ** -16 * 1.1 * (np.abs(u) * mg + np.abs(a) * mu)
    err = np.abs(out.read().astype(np.float64) - a * u)
    assert np.all(err <= bound), f"worst {np.max(err / bound):.2f} of the bound"


# zero-points as any f16 array may hold them: halves and smaller fractions, negative ones,
# odd whole numbers past 1024 and past 2048, and far ones (not so far that y passes the f16 range)
ZEROS = [7.5, 3.25, 0.1, -3.5, -1000.5, 1025.0, 1501.0, 2001.0, -1501.0, 3002.0, -5004.0, 8008.0, 8.0, 0.0]


def any_zeros(q, seed):
    """q with zero-points of ZEROS; every third column keeps its own, whole and small."""
    z = np.random.default_rng(seed).choice(np.asarray(ZEROS, np.float16), q.zeros.shape)
    z[::3] = q.zeros[::3]
    q.zeros = z
    return q


def magnitudes(q):
    """(|q| + |z|) s per weight: what sums of codes and of zero-points carry apart."""
    codes = np.empty((q.n, q.k), np.float64)
    codes[:, 0::2], codes[:, 1::2] = q.data & 0xF, q.data >> 4
    return (codes + np.repeat(np.abs(q.zeros.astype(np.float64)), q.group_size, axis=1)) \
        * np.repeat(q.scales.astype(np.float64), q.group_size, axis=1)


@pytest.mark.parametrize("awq", [False, True])
@pytest.mark.parametrize("m", [8, 9, 12, 17, 31, 32, 40, 65])
def test_any_zero_points(dev, stream, m, awq):
    """y = x . ((q - z) s) for every f16 z, on the matvec (8 rows), the one-launch kernel (9 to
    32) and the tiles above it, one matrix and a pair: 2 f16 steps plus 2^-16 of the magnitudes
    that sums of codes and zero-points carry (f32 sums; the activation's 22 bits against codes,
    in the matvec up to 16 times the code).  A zero-point half a code off is past the bound in
    the columns without a far one."""
    n, k = 12801, 1152
    w, s = weight(n, k, 17, awq)
    q0 = any_zeros(quant.quantize_int4(w, awq_scales=s), 18)
    q1 = any_zeros(quant.quantize_int4(weight(n, k, 19, False)[0], awq_scales=s), 20)
    x16 = acts(m, k, m)
    xd = dev.upload(x16)
    w0, w1 = ops.AffineQuantizedWeight(dev, q0), ops.AffineQuantizedWeight(dev, q1)
    y, g, u = (dev.empty((m, n), np.float16) for _ in range(3))
    ops.encode_projection(stream, xd, w0, y, m)
    ops.encode_batched_affine_matvec_int4(stream, xd, w0, g, w1, u, m)
    stream.sync()
    a = x16.astype(np.float64) if s is None else x16.astype(np.float64) / s.astype(np.float16).astype(np.float64)
    for what, got, q in (("one matrix", y, q0), ("gate", g, q0), ("up", u, q1)):
        exact = a @ exact_weights(q).T
        bound = 2.0 * np.spacing(np.abs(exact).astype(np.float16)).astype(np.float64) \
            + 2.0 ** -16 * (np.abs(a) @ magnitudes(q).T)
        err = np.abs(got.read().astype(np.float64) - exact)
        assert np.all(err <= bound), f"{what}: worst {np.max(err / bound):.2f} of the bound"


def test_gemm_capture_reads_constants_in_place(dev):
    """Under capture with scratch for the activation planes only, the GEMM reads scales and
    zero-points in place: the replays equal the eager result bit for bit."""
    m, k = 1024, 2048     # planes: 8 MiB, the first call's scratch with its constants just above
    w, s = weight(256, k, 91, True)
    small = ops.AffineQuantizedWeight(dev, quant.quantize_int4(w, awq_scales=s))
    w2, _ = weight(8192, k, 92, False)
    wide = ops.AffineQuantizedWeight(dev, quant.quantize_int4(w2, awq_scales=s))
    x16 = acts(m, k, 93)
    st = dev.stream()
    xd, y0 = dev.upload(x16), dev.empty((m, 256), np.float16)
    ye, yg = dev.empty((m, 8192), np.float16), dev.empty((m, 8192), np.float16)
    ops.encode_projection(st, xd, small, y0, m)
    g = st.capture(lambda: ops.encode_projection(st, xd, wide, yg, m))
    ops.encode_projection(st, xd, wide, ye, m)
    st.sync()
    want = ye.read().view(np.uint16)
    for _ in range(2):
        st.zero(yg)
        g.launch()
        st.sync()
        assert np.array_equal(yg.read().view(np.uint16), want)


@pytest.mark.parametrize("m", [32, 40])
def test_gemm_capture_without_partials(dev, m):
    """A capture on a stream without room for split partials runs the GEMM unsplit: each replay
    is within 2 f16 steps plus the sum-order slack of the exact value."""
    n, k = 1000, 4096
    w, _ = weight(n, k, 151, False)
    q = quant.quantize_int4(w)
    x16 = acts(m, k, 152)
    st = dev.stream()
    xd, y, wt = dev.upload(x16), dev.empty((m, n), np.float16), ops.AffineQuantizedWeight(dev, q)
    g = st.capture(lambda: ops.encode_projection(st, xd, wt, y, m))
    W = exact_weights(q)
    exact = x16.astype(np.float64) @ W.T
    bound = 2.0 * np.spacing(np.abs(exact).astype(np.float16)).astype(np.float64) \
        + 2.0 ** -16 * (np.abs(x16.astype(np.float64)) @ np.abs(W).T)
    for _ in range(2):
        st.zero(y)
        g.launch()
        st.sync()
        assert np.all(np.abs(y.read().astype(np.float64) - exact) <= bound)


def rows_splits(m, n, k, nmat=1, cus=256):
    """The K split of the one-launch kernel, as its host code picks it."""
    tiles, g = -(-n // (256 // nmat)), k // 128
    cost = {}
    for per in range(4, g + 4, 4):
        sp = -(-g // per)
        cost.setdefault(sp, -(-tiles * sp // (2 * cus)) * (4 + 1.05 * min(per, g))
                        + (3 + sp * m * nmat * n * 8 / 4.5e6 if sp > 1 else 0))
    return min(cost, key=cost.get)


@pytest.mark.parametrize("warm", [None, "gemm", "matvec"])
def test_gemm_rows_capture(dev, warm):
    """A capture of 12 rows whose stream lacks the split's partials -- with no scratch at all, with
    that of a smaller projection on the same kernel, or with the matvec's operand image -- records
    what needs none; each replay is within 2 f16 steps plus the sum-order slack of the exact value."""
    m, n, k = 12, 6144, 9728
    assert rows_splits(m, n, k) * m * n * 4 > 2 ** 20   # more than the smallest scratch block
    w, s = weight(n, k, 161, True)
    q = quant.quantize_int4(w, awq_scales=s)
    x16 = acts(m, k, 162)
    st = dev.stream()
    xd, y, wt = dev.upload(x16), dev.empty((m, n), np.float16), ops.AffineQuantizedWeight(dev, q)
    if warm:
        n0 = 1024 if warm == "gemm" else 64   # 64 x 9728 x 12 is the matvec's, 1024 x 9728 x 12 the GEMM's
        assert rows_splits(m, 1024, k) * m * 1024 * 4 <= 2 ** 20
        w0 = ops.AffineQuantizedWeight(dev, quant.quantize_int4(w[:n0].copy(), awq_scales=s))
        ops.encode_projection(st, xd, w0, dev.empty((m, n0), np.float16), m)
    g = st.capture(lambda: ops.encode_projection(st, xd, wt, y, m))
    a, W = x16.astype(np.float64) / s.astype(np.float16).astype(np.float64), exact_weights(q)
    exact = a @ W.T
    # the matvec's sums hold codes and zero-points apart
    bound = 2.0 * np.spacing(np.abs(exact).astype(np.float16)).astype(np.float64) + 2.0 ** -16 * (np.abs(a) @ magnitudes(q).T)
    for _ in range(2):
        st.zero(y)
        g.launch()
        st.sync()
        assert np.all(np.abs(y.read().astype(np.float64) - exact) <= bound)


def test_gemm_pair_capture_reads_constants_in_place(dev):
    """Gate and up with AWQ under capture, with scratch for the activation planes only: both
    matrices' scales and zero-points are read in place, and the replays equal the eager result bit
    for bit."""
    m, k = 1023, 2048
    ws, s = weight(256, k, 191, True)
    small = ops.AffineQuantizedWeight(dev, quant.quantize_int4(ws, awq_scales=s))
    gate, up = (ops.AffineQuantizedWeight(dev, quant.quantize_int4(weight(8200, k, seed, False)[0], awq_scales=s))
                for seed in (192, 193))
    x16 = acts(m, k, 194)
    st = dev.stream()
    xd, y0 = dev.upload(x16), dev.empty((m, 256), np.float16)
    outs = [dev.empty((m, 8200), np.float16) for _ in range(5)]

    def run(act, g, u):
        ops.encode_fused_ffn_gate_up_act_int4(st, xd, gate, up, act, m)
        ops.encode_batched_affine_matvec_int4(st, xd, gate, g, up, u, m)
    ops.encode_projection(st, xd, small, y0, m)
    graph = st.capture(lambda: run(*outs[:3]))
    st2 = dev.stream()
    ops.encode_fused_ffn_gate_up_act_int4(st2, xd, gate, up, outs[3], m)
    st2.sync()
    want_act = outs[3].read().view(np.uint16)
    ops.encode_batched_affine_matvec_int4(st2, xd, gate, outs[3], up, outs[4], m)
    st2.sync()
    want = [want_act, outs[3].read().view(np.uint16), outs[4].read().view(np.uint16)]
    for _ in range(2):
        for o in outs[:3]:
            st.zero(o)
        graph.launch()
        st.sync()
        for o, w in zip(outs, want):
            assert np.array_equal(o.read().view(np.uint16), w)
