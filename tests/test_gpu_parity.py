"""Parity of the gfx950 backend with the CPU oracle, through the C ABI.

Gates: KV slot/page indexing bit-exact; cached K/V within 1 f16 ulp;
attention output max-abs <= 2e-3 and cosine >= 0.99999. Inputs are the same
seeded host arrays for both sides. The reference's fixture tolerances apply to
the vendored fixtures.
"""
import numpy as np
import pytest

from conftest import FIXTURES, attention_f64, cosine, f16_ulp_diff
from qw3_amd import synth

pytestmark = pytest.mark.gpu

OUT_ATOL = 2e-3     # attention output, max-abs
OUT_COS = 0.99999   # attention output, cosine


def check_out(got, want, atol=OUT_ATOL, cos=OUT_COS):
    got = np.asarray(got, np.float32).ravel()
    want = np.asarray(want, np.float32).ravel()
    assert np.all(np.isfinite(got))
    err = float(np.max(np.abs(got - want)))
    c = cosine(got, want)
    print(f"  max_abs={err:.3e} cosine={c:.9f}", flush=True)
    assert err <= atol and c >= cos, (err, c)


def dev(ctx, a):
    return ctx.from_numpy(np.ascontiguousarray(a))


def host(ctx, buf, like):
    return ctx.to_numpy(buf, like.dtype, like.shape)


# ---------------------------------------------------------------------------
# single ops vs the reference fixtures and the oracle
# ---------------------------------------------------------------------------

def _cases(O, op):
    return [c for c in O.load_manifest(FIXTURES)["cases"] if c["op"] == op]


def _t(O, c, name):
    return O.load_ds5t(f"{FIXTURES}/{c['tensors'][name]}").data


@pytest.mark.parametrize("i", range(6))
def test_rmsnorm_fixtures_bit_exact(ctx, hip, oracle, i):
    c = _cases(oracle, "rmsnorm")[i]
    p, tol = c["params"], c["tolerance"]
    x, w, want = (_t(oracle, c, n) for n in ("input", "weight", "output"))
    xb = dev(ctx, x)
    hip.rmsNorm(ctx, hip.RmsNormArgs(xb, dev(ctx, w), xb, p["n_rows"], p["dim"], p["eps"]))  # out aliases x
    got = host(ctx, xb, x)
    assert oracle.compare(want, got, tol["atol"], tol["rtol"]).passed
    assert np.array_equal(got, oracle.rms_norm(x, w, p["eps"], p["n_rows"], p["dim"]))


@pytest.mark.parametrize("dim,scale", [(128, 1.0), (64, 1e-3), (128, 3e4), (4, 1.0)])
def test_rmsnorm_random_rows_bit_exact(ctx, hip, oracle, dim, scale):
    """rmsNorm over 5000 seeded rows of widely varying magnitude, bit-identical to
    the oracle (the scale 1/sqrt(mean + eps) must be correctly rounded)."""
    g = np.random.default_rng(dim + int(scale))
    n = 5000
    x = (g.standard_normal((n, dim)) * scale * np.exp(g.uniform(-4, 4, (n, 1)))).astype(np.float32)
    w = (1.0 + 0.02 * g.standard_normal(dim)).astype(np.float32)
    xb, out = dev(ctx, x), ctx.createBuffer(x.nbytes)
    hip.rmsNorm(ctx, hip.RmsNormArgs(xb, dev(ctx, w), out, n, dim, 1e-6))
    got = ctx.to_numpy(out, np.float32, x.shape)
    want = oracle.rms_norm(x, w, 1e-6, n, dim)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("dim", [257, 300, 512, 1000, 2048, 4096, 5000, 8192])
def test_rmsnorm_long_rows_tree_order(ctx, hip, oracle, dim):
    """Rows of more than 256 elements take the reference GPU kernel's reduction order
    (kernels_a.metal:127-165): bit-identical to the oracle's restatement of it, and within
    the fixtures' atol 1e-5 / rtol 1e-4 of the serial CPU order (the reference's own note
    on that kernel). 1, 3 and 67 rows, magnitudes over 8 decades, in place and not."""
    g = np.random.default_rng(dim)
    w = (1.0 + 0.02 * g.standard_normal(dim)).astype(np.float32)
    wb = dev(ctx, w)
    for n in (1, 3, 67):
        x = (g.standard_normal((n, dim)) * np.exp(g.uniform(-9, 9, (n, 1)))).astype(np.float32)
        xb, out = dev(ctx, x), ctx.createBuffer(x.nbytes)
        hip.rmsNorm(ctx, hip.RmsNormArgs(xb, wb, out, n, dim, 1e-6))
        got = ctx.to_numpy(out, np.float32, x.shape)
        want = oracle.rms_norm_tree(x, w, 1e-6, n, dim)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (dim, n)
        assert oracle.compare(oracle.rms_norm(x, w, 1e-6, n, dim), got, 1e-5, 1e-4).passed, (dim, n)
        hip.rmsNorm(ctx, hip.RmsNormArgs(xb, wb, xb, n, dim, 1e-6))  # out aliases x
        assert np.array_equal(host(ctx, xb, x).view(np.uint32), want.view(np.uint32)), (dim, n)


def test_rmsnorm_tree_order_special_row(ctx, hip, oracle):
    """The row whose f32 sum separates the orders (4096 at element 0, ones at elements 1
    and 3: 2^24 + 2 in the kernel's order, 2^24 serially) gives the oracle's tree result."""
    dim = 512
    x = np.zeros((1, dim), np.float32)
    x[0, 0], x[0, 1], x[0, 3] = 4096.0, 1.0, 1.0
    w = np.linspace(0.5, 1.5, dim).astype(np.float32)
    xb = dev(ctx, x)
    hip.rmsNorm(ctx, hip.RmsNormArgs(xb, dev(ctx, w), xb, 1, dim, 1e-6))
    got = host(ctx, xb, x)
    assert np.array_equal(got, oracle.rms_norm_tree(x, w, 1e-6))
    assert not np.array_equal(got, oracle.rms_norm(x, w, 1e-6))


@pytest.mark.parametrize("i", range(3))
def test_rope_fixtures(ctx, hip, oracle, i):
    c = _cases(oracle, "rope")[i]
    p, tol = c["params"], c["tolerance"]
    x, pos, want = (_t(oracle, c, n) for n in ("input", "positions", "output"))
    xb = dev(ctx, x)
    hip.rope(ctx, hip.RopeArgs(xb, dev(ctx, pos), p["n_tokens"], p["n_heads"], p["head_dim"], p["theta"],
                               p["freq_scale"]))
    got = host(ctx, xb, x)
    assert oracle.compare(want, got, tol["atol"], tol["rtol"]).passed
    ref = oracle.rope(x, pos, p["theta"], p["freq_scale"])
    assert np.max(np.abs(got - ref)) <= 4 * np.finfo(np.float32).eps * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("i", range(6))
@pytest.mark.parametrize("kv_dtype", [0, 1])
def test_attention_fixtures(ctx, hip, oracle, i, kv_dtype):
    """f32 caches: the reference fixture tolerance. f16 caches (MFMA decode and
    prefill at head_dim 64): against the oracle's f16 branch at the attention
    gate (max-abs 2e-3, cosine 0.99999); prefill rounds q and p to f16 for the
    MFMA products, which moves outputs by ~1e-4 on these fixtures."""
    c = _cases(oracle, "attention")[i]
    p, tol = c["params"], c["tolerance"]
    q, kc, vc, want = (_t(oracle, c, n) for n in ("q", "k_cache", "v_cache", "output"))
    if kv_dtype == 1:
        kc, vc = oracle.f32_to_f16_bits(kc), oracle.f32_to_f16_bits(vc)
        want = oracle.gqa_attention(q, kc, vc, 1, p["pos"], p["n_tokens"], p["n_q_heads"], p["n_kv_heads"],
                                    p["head_dim"], p["max_ctx"], p["scale"])
    out = ctx.createBuffer(want.nbytes)
    hip.gqaAttention(ctx, hip.AttnArgs(dev(ctx, q), dev(ctx, kc), dev(ctx, vc), kv_dtype, out, p["pos"],
                                       p["n_tokens"], p["n_q_heads"], p["n_kv_heads"], p["head_dim"], p["max_ctx"],
                                       p["scale"]))
    got = ctx.to_numpy(out, np.float32)
    if kv_dtype == 0:
        r = oracle.compare(want, got, tol["atol"], tol["rtol"])
        assert r.passed, r
    else:
        check_out(got, want)


@pytest.mark.parametrize("kv_dtype", [0, 1])
def test_kv_append_sentinel_bit_exact(ctx, hip, oracle, kv_dtype):
    hkv, hd, cap, pos, T = 4, 128, 40, 13, 5
    g = np.random.default_rng(11)
    kn = g.standard_normal((T, hkv, hd)).astype(np.float32)
    vn = g.standard_normal((T, hkv, hd)).astype(np.float32) * 300  # exercise f16 rounding far from 1
    kn[0, 0, :8] = [65504.0, 65520.0, 6.0e-8, -3.0e-8, 1e-6, -0.0, 1.0009765625, 70000.0]
    if kv_dtype == 0:
        kc = g.standard_normal((hkv, cap, hd)).astype(np.float32)
        vc = g.standard_normal((hkv, cap, hd)).astype(np.float32)
    else:
        kc = g.integers(0, 0x7C00, size=(hkv, cap, hd), dtype=np.uint64).astype(np.uint16)
        vc = g.integers(0, 0x7C00, size=(hkv, cap, hd), dtype=np.uint64).astype(np.uint16)
    kb, vb = dev(ctx, kc), dev(ctx, vc)
    hip.kvAppend(ctx, hip.KvAppendArgs(dev(ctx, kn), dev(ctx, vn), kb, vb, kv_dtype, pos, T, hkv, hd, cap))
    ko, vo = kc.copy(), vc.copy()
    oracle.kv_append(kn, vn, ko, vo, kv_dtype, pos, T, hkv, hd, cap)
    assert np.array_equal(host(ctx, kb, kc), ko)
    assert np.array_equal(host(ctx, vb, vc), vo)


def test_shape_errors_with_device(ctx, hip):
    b = ctx.createBuffer(256)
    with pytest.raises(hip.ShapeMismatch):  # kernels_b.zig:456-492
        hip.gqaAttention(ctx, hip.AttnArgs(b, b, b, 0, b, 8, 1, 2, 2, 4, 8, 0.5))
    with pytest.raises(hip.ShapeMismatch):
        hip.gqaAttention(ctx, hip.AttnArgs(b, b, b, 0, b, 0, 1, 3, 2, 4, 8, 0.5))
    with pytest.raises(hip.UnsupportedDtype):
        hip.kvAppend(ctx, hip.KvAppendArgs(b, b, b, b, 8, 0, 1, 1, 4, 2))
    with pytest.raises(hip.ShapeMismatch):
        hip.kvAppend(ctx, hip.KvAppendArgs(b, b, b, b, 0, 7, 2, 1, 4, 8))


# ---------------------------------------------------------------------------
# hand cases (kernels_b.zig:228-454) on both cache dtypes
# ---------------------------------------------------------------------------

def _f16_nan_cache(shape):
    return np.full(shape, 0x7E00, np.uint16)


@pytest.mark.parametrize("hd,kv_dtype", [(4, 0), (64, 1), (128, 1)])
def test_pos0_returns_v0_nan_tail(ctx, hip, oracle, hd, kv_dtype):
    hq, hkv, cap = 8, 2, 3
    g = np.random.default_rng(1)
    q = g.standard_normal(hq * hd).astype(np.float32)
    kf = np.full((hkv, cap, hd), np.nan, np.float32)
    vf = np.full((hkv, cap, hd), np.nan, np.float32)
    kf[:, 0] = g.standard_normal((hkv, hd))
    for kh in range(hkv):
        vf[kh, 0] = kh * 8 + np.arange(hd) / 8
    k, v = (kf, vf) if kv_dtype == 0 else (oracle.f32_to_f16_bits(kf), oracle.f32_to_f16_bits(vf))
    out = ctx.createBuffer(hq * hd * 4)
    hip.gqaAttention(ctx, hip.AttnArgs(dev(ctx, q), dev(ctx, k), dev(ctx, v), kv_dtype, out, 0, 1, hq, hkv, hd,
                                       cap, 0.5))
    got = ctx.to_numpy(out, np.float32).reshape(hq, hd)
    for h in range(hq):
        np.testing.assert_allclose(got[h], (h // 4) * 8 + np.arange(hd) / 8, atol=1e-6)


@pytest.mark.parametrize("hd,kv_dtype,T", [(8, 0, 2), (64, 1, 1), (128, 1, 1), (128, 1, 3), (64, 1, 40)])
def test_ragged_pos_packed_equivalence(ctx, hip, oracle, hd, kv_dtype, T):
    hq, hkv, pos = 8, 2, 37
    valid, big = pos + T, pos + T + 29
    g = np.random.default_rng(42)
    q = g.standard_normal((T, hq, hd)).astype(np.float32)
    kp = g.standard_normal((hkv, valid, hd)).astype(np.float32)
    vp = g.standard_normal((hkv, valid, hd)).astype(np.float32)
    if kv_dtype == 1:
        kp, vp = oracle.f32_to_f16_bits(kp), oracle.f32_to_f16_bits(vp)
        kb, vb = _f16_nan_cache((hkv, big, hd)), _f16_nan_cache((hkv, big, hd))
    else:
        kb, vb = np.full((hkv, big, hd), np.nan, np.float32), np.full((hkv, big, hd), np.nan, np.float32)
    kb[:, :valid], vb[:, :valid] = kp, vp
    scale = float(np.float32(1) / np.sqrt(np.float32(hd)))

    def run(k, v, cap):
        out = ctx.createBuffer(T * hq * hd * 4)
        hip.gqaAttention(ctx, hip.AttnArgs(dev(ctx, q), dev(ctx, k), dev(ctx, v), kv_dtype, out, pos, T, hq, hkv, hd,
                                           cap, scale))
        return ctx.to_numpy(out, np.float32)

    a, b = run(kp, vp, valid), run(kb, vb, big)
    assert np.array_equal(a, b)  # stride by max_ctx, never read past pos + t
    check_out(b, oracle.gqa_attention(q, kp, vp, kv_dtype, pos, T, hq, hkv, hd, valid, scale))
    if T > 1:  # perturb the last position: only the last query token changes
        kb2, vb2 = kb.copy(), vb.copy()
        if kv_dtype == 1:
            kb2[:, valid - 1] ^= 0x0400
            vb2[:, valid - 1] ^= 0x0400
        else:
            kb2[:, valid - 1] += 1.5
            vb2[:, valid - 1] -= 2.0
        c = run(kb2, vb2, big)
        row = (T - 1) * hq * hd
        assert np.array_equal(b[:row], c[:row]) and not np.array_equal(b[row:], c[row:])


@pytest.mark.parametrize("kv_dtype", [0, 1])
def test_softmax_stability(ctx, hip, oracle, kv_dtype):
    # scores +-200 (kernels_b.zig:424-454), widened to head_dim 64 for the MFMA path
    hd = 2 if kv_dtype == 0 else 64
    q = np.zeros(hd, np.float32)
    q[0] = 100
    k = np.zeros((1, 2, hd), np.float32)
    k[0, 0, 0], k[0, 1, 0] = -2, 2
    v = np.zeros((1, 2, hd), np.float32)
    v[0, 0, :2], v[0, 1, :2] = (7, -7), (3.5, -3.5)
    if kv_dtype == 1:
        k, v = oracle.f32_to_f16_bits(k), oracle.f32_to_f16_bits(v)
    out = ctx.createBuffer(hd * 4)
    hip.gqaAttention(ctx, hip.AttnArgs(dev(ctx, q), dev(ctx, k), dev(ctx, v), kv_dtype, out, 1, 1, 1, 1, hd, 2, 1.0))
    got = ctx.to_numpy(out, np.float32)
    np.testing.assert_allclose(got[:2], [3.5, -3.5], atol=1e-6)


# ---------------------------------------------------------------------------
# decode: split-K kernel over many lengths and group sizes (separate-op path)
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("L", [1, 2, 31, 32, 33, 127, 128, 129, 500, 1000, 4097])
@pytest.mark.parametrize("hq,hkv,hd", [(32, 4, 128), (64, 4, 128), (8, 8, 64), (64, 2, 128), (12, 4, 64)])
def test_decode_lengths_and_groups(ctx, hip, oracle, L, hq, hkv, hd):
    g = np.random.default_rng(L * 7 + hq)
    cap = L + 5
    q = g.standard_normal((1, hq, hd)).astype(np.float32)
    k = oracle.f32_to_f16_bits(g.standard_normal((hkv, cap, hd)).astype(np.float32))
    v = oracle.f32_to_f16_bits(g.standard_normal((hkv, cap, hd)).astype(np.float32))
    scale = float(np.float32(1) / np.sqrt(np.float32(hd)))
    out = ctx.createBuffer(hq * hd * 4)
    hip.gqaAttention(ctx, hip.AttnArgs(dev(ctx, q), dev(ctx, k), dev(ctx, v), 1, out, L - 1, 1, hq, hkv, hd, cap,
                                       scale))
    check_out(ctx.to_numpy(out, np.float32), oracle.gqa_attention(q, k, v, 1, L - 1, 1, hq, hkv, hd, cap, scale))


# ---------------------------------------------------------------------------
# the fused step at the benchmark configurations
# ---------------------------------------------------------------------------

def _run_step(ctx, hip, q, k, v, qn, kn, positions, kc, vc, pos, s, fused):
    """Runs one engine step on the GPU; returns (out, k_cache, v_cache)."""
    T, hq, hd = q.shape
    hkv, cap = kc.shape[0], kc.shape[1]
    qb, kb, vb = dev(ctx, q), dev(ctx, k), dev(ctx, v)
    qnb, knb, pb = dev(ctx, qn), dev(ctx, kn), dev(ctx, positions)
    kcb, vcb = dev(ctx, kc), dev(ctx, vc)
    out = ctx.createBuffer(T * hq * hd * 4)
    if fused:
        hip.attentionStep(ctx, hip.AttentionStepArgs(qb, kb, vb, qnb, knb, pb, kcb, vcb, out, 1, pos, T, hq, hkv, hd,
                                                     cap, s.eps, s.theta, 1.0, s.scale))
    else:  # forward.zig:345-412, op by op
        hip.rmsNorm(ctx, hip.RmsNormArgs(qb, qnb, qb, T * hq, hd, s.eps))
        hip.rmsNorm(ctx, hip.RmsNormArgs(kb, knb, kb, T * hkv, hd, s.eps))
        hip.rope(ctx, hip.RopeArgs(qb, pb, T, hq, hd, s.theta))
        hip.rope(ctx, hip.RopeArgs(kb, pb, T, hkv, hd, s.theta))
        hip.kvAppend(ctx, hip.KvAppendArgs(kb, vb, kcb, vcb, 1, pos, T, hkv, hd, cap))
        hip.gqaAttention(ctx, hip.AttnArgs(qb, kcb, vcb, 1, out, pos, T, hq, hkv, hd, cap, s.scale))
    return ctx.to_numpy(out, np.float32), host(ctx, kcb, kc), host(ctx, vcb, vc)


def _oracle_step(oracle, q, k, v, qn, kn, positions, kc, vc, pos, s):
    T, hq, hd = q.shape
    hkv, cap = kc.shape[0], kc.shape[1]
    kc, vc = kc.copy(), vc.copy()
    out, _, _ = oracle.attention_step(q, k, v, qn, kn, positions, kc, vc, kv_dtype=1, pos=pos, n_tokens=T,
                                      n_q_heads=hq, n_kv_heads=hkv, head_dim=hd, max_ctx=cap, eps=s.eps,
                                      theta=s.theta, scale=s.scale)
    return out, kc, vc


def check_cache(got_k, got_v, want_k, want_v, kc0, vc0, pos, T):
    # rows outside pos..pos+T-1 untouched (bit-exact), appended rows within 1 f16 ulp
    for got, want, old in ((got_k, want_k, kc0), (got_v, want_v, vc0)):
        assert np.array_equal(got[:, :pos], old[:, :pos])
        assert np.array_equal(got[:, pos + T:], old[:, pos + T:])
        ulp = f16_ulp_diff(got[:, pos:pos + T], want[:, pos:pos + T])
        print(f"  cache rows: max ulp {ulp.max()} ({int((ulp > 0).sum())} of {ulp.size} differ)", flush=True)
        assert ulp.max() <= 1


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("config,layer", [(0, 0), (1, 0), (1, 47), (3, 0)])
def test_decode_step_configs(ctx, hip, oracle, config, layer, fused):
    cfg = synth.CONFIGS[config]
    s, cap, pos = cfg["shape"], cfg["cap"], cfg["pos"]
    q, k, v, qn, kn = synth.step_inputs(config, layer, 1, s)
    kc, vc = synth.cache_f16(config, layer, s, cap, pos)
    positions = np.array([pos], np.int32)
    out, gk, gv = _run_step(ctx, hip, q, k, v, qn, kn, positions, kc, vc, pos, s, fused)
    wout, wk, wv = _oracle_step(oracle, q, k, v, qn, kn, positions, kc, vc, pos, s)
    check_cache(gk, gv, wk, wv, kc, vc, pos, 1)
    check_out(out, wout)


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("T,pos,hd,hq,hkv", [
    (300, 0, 128, 32, 4),   # 10 q tiles, masked last key tile
    (130, 100, 128, 32, 4),  # chunked continuation: the mask spans two key tiles
    (77, 5, 64, 32, 4),     # head_dim 64
    (2, 0, 128, 32, 4),     # one key tile: the second wavefront set idles
    (97, 0, 128, 32, 4),    # odd q-tile count: the middle tile runs once
    (160, 48, 128, 32, 4),  # middle tile whose first 16 rows see no key in set 1's key tiles
    (200, 31, 128, 64, 4),  # 16-head group: four head groups per kv head
    (96, 3, 128, 6, 3),     # 2-head group: half the wavefronts have no head
    (65, 0, 64, 8, 8),      # no grouping, head_dim 64
])
def test_prefill_step(ctx, hip, oracle, T, pos, hd, hq, hkv, fused):
    s = synth.Shape(n_q_heads=hq, n_kv_heads=hkv, head_dim=hd)
    cap = pos + T + 7
    q, k, v, qn, kn = synth.step_inputs(2, T, T, s, f16_exact=True)
    kc, vc = synth.cache_f16(2, T, s, cap, pos)
    positions = np.arange(pos, pos + T, dtype=np.int32)
    out, gk, gv = _run_step(ctx, hip, q, k, v, qn, kn, positions, kc, vc, pos, s, fused)
    wout, wk, wv = _oracle_step(oracle, q, k, v, qn, kn, positions, kc, vc, pos, s)
    check_cache(gk, gv, wk, wv, kc, vc, pos, T)
    check_out(out, wout)


@pytest.mark.parametrize("fused", [True, False])
def test_prefill_config2_full(ctx, hip, oracle, fused):
    """C2 at full size: every cache row checked; the attention output of every one
    of the 32 q heads checked against a float64 causal attention on the oracle's
    normalised and rotated q and cache rows, and one head of each kv group also
    against the oracle's own attention (~1 s per head)."""
    cfg = synth.CONFIGS[2]
    s, T = cfg["shape"], cfg["tokens"]
    q, k, v, qn, kn = synth.step_inputs(2, 0, T, s, f16_exact=True)
    kc, vc = synth.cache_f16(2, 0, s, T, 0)
    positions = np.arange(T, dtype=np.int32)
    out, gk, gv = _run_step(ctx, hip, q, k, v, qn, kn, positions, kc, vc, 0, s, fused)
    # oracle cache: k norm + rope + append (cheap), then per-head attention
    k_rot = oracle.rope(oracle.rms_norm(k, kn, s.eps), positions, s.theta)
    wk, wv = kc.copy(), vc.copy()
    oracle.kv_append(k_rot, v, wk, wv, 1, 0, T, s.n_kv_heads, s.head_dim, T)
    check_cache(gk, gv, wk, wv, kc, vc, 0, T)
    q_rot = oracle.rope(oracle.rms_norm(q, qn, s.eps), positions, s.theta)
    out = out.reshape(T, s.n_q_heads, s.head_dim)
    group = s.n_q_heads // s.n_kv_heads
    for h in range(s.n_q_heads):
        check_out(out[:, h], attention_f64(q_rot[:, h], wk[h // group], wv[h // group], s.scale))
    for h in (3, 10, 17, 29):  # one head of each kv group
        kh = h // group
        want = oracle.gqa_attention(np.ascontiguousarray(q_rot[:, h:h + 1]), np.ascontiguousarray(wk[kh:kh + 1]),
                                    np.ascontiguousarray(wv[kh:kh + 1]), 1, 0, T, 1, 1, s.head_dim, T, s.scale)
        check_out(out[:, h], want)


# ---------------------------------------------------------------------------
# paged decode (C4 layout)
# ---------------------------------------------------------------------------

def _paged_case(ctx, hip, oracle, n_seqs, lo, hi, seed, check_seqs=None, page_size=16):
    s = synth.Shape()
    lay = synth.paged_layout(n_seqs, lo, hi, page_size, seed=seed)
    hq, hkv, hd = s.n_q_heads, s.n_kv_heads, s.head_dim
    slots = lay.n_pages * page_size
    g = np.random.default_rng(seed)
    kpool = oracle.f32_to_f16_bits(g.standard_normal((hkv, slots, hd)).astype(np.float32))
    vpool = oracle.f32_to_f16_bits(g.standard_normal((hkv, slots, hd)).astype(np.float32))
    q, k, v, qn, kn = synth.step_inputs(4, seed, n_seqs, s)
    kpb, vpb = dev(ctx, kpool), dev(ctx, vpool)
    out = ctx.createBuffer(n_seqs * hq * hd * 4)
    max_len = int(lay.seq_lens.max())
    hip.pagedDecode(ctx, hip.PagedDecodeArgs(dev(ctx, q), dev(ctx, k), dev(ctx, v), dev(ctx, qn), dev(ctx, kn), kpb,
                                             vpb, dev(ctx, lay.page_table), dev(ctx, lay.seq_lens), out, n_seqs, hq,
                                             hkv, hd, page_size, lay.n_pages, lay.max_pages, max_len, s.eps, s.theta, 1.0,
                                             s.scale))
    got = ctx.to_numpy(out, np.float32).reshape(n_seqs, hq * hd)
    gk, gv = host(ctx, kpb, kpool), host(ctx, vpb, vpool)
    new_slots = [lay.slot(b, int(lay.seq_lens[b]) - 1) for b in range(n_seqs)]
    mask = np.ones(slots, bool)
    mask[new_slots] = False
    assert np.array_equal(gk[:, mask], kpool[:, mask]) and np.array_equal(gv[:, mask], vpool[:, mask])
    for b in (range(n_seqs) if check_seqs is None else check_seqs):
        L = int(lay.seq_lens[b])
        kc = oracle.paged_gather_f16(kpool, lay.page_table[b], page_size, L)
        vc = oracle.paged_gather_f16(vpool, lay.page_table[b], page_size, L)
        wout, wk, wv = _oracle_step(oracle, q[b:b + 1], k[b:b + 1], v[b:b + 1], qn, kn, np.array([L - 1], np.int32),
                                    kc, vc, L - 1, s)
        ulp_k = f16_ulp_diff(gk[:, new_slots[b]], wk[:, L - 1])
        ulp_v = f16_ulp_diff(gv[:, new_slots[b]], wv[:, L - 1])
        assert ulp_k.max() <= 1 and ulp_v.max() <= 1
        check_out(got[b], wout)


def test_paged_decode_small(ctx, hip, oracle):
    _paged_case(ctx, hip, oracle, 7, 1, 300, seed=5)


@pytest.mark.parametrize("page_size", [32, 64])
def test_paged_decode_larger_pages(ctx, hip, oracle, page_size):
    """Pages of 32 and 64 positions (the ABI takes any multiple of 16): a 32-position
    tile then lies inside one page, and page boundaries fall inside a split."""
    _paged_case(ctx, hip, oracle, 7, 1, 700, seed=11, page_size=page_size)


def test_paged_decode_config4_geometry(ctx, hip, oracle):
    """C4's geometry (32 sequences, lengths U[512, 16384], 16-token pages): every
    sequence's output and appended rows against the oracle on its gathered pages."""
    _paged_case(ctx, hip, oracle, 32, 512, 16384, seed=0)


def test_paged_decode_large_batch_unplanned(ctx, hip, oracle):
    """More sequences than the device-side plan stages (4096): the launch falls back to
    the (split, kv head, sequence) grid sized from the longest sequence, here one split
    per sequence whose workgroup writes the output itself. A sample of sequences
    against the oracle; every pool row outside the new slots byte-identical."""
    _paged_case(ctx, hip, oracle, 4100, 1, 40, seed=9, check_seqs=[0, 1, 777, 2048, 4095, 4096, 4099])


def test_paged_decode_large_batch_unplanned_splits(hip, oracle):
    """The unplanned grid with several splits: 4100 sequences of 1..300 positions with
    the split size fixed at 128 (DS5_HIP_DECODE_CHUNK, read when a context starts), so
    sequences of at most 128 positions have one split whose workgroup writes the output
    itself, and longer ones two or three splits that the merge combines, in the same
    launch. A sample of both kinds against the oracle."""
    import os
    os.environ["DS5_HIP_DECODE_CHUNK"] = "128"
    try:
        c = hip.Ctx.init(0)
    finally:
        del os.environ["DS5_HIP_DECODE_CHUNK"]
    try:
        lay = synth.paged_layout(4100, 1, 300, 16, seed=21)
        lens = lay.seq_lens
        short = [int(b) for b in np.nonzero(lens <= 128)[0][:4]]
        long_ = [int(b) for b in np.nonzero(lens > 256)[0][:4]] + [int(b) for b in np.nonzero((lens > 128) & (lens <= 256))[0][:2]]
        assert len(short) == 4 and len(long_) == 6
        print(f"[paged] unplanned splits: short {short}, long {long_}", flush=True)
        _paged_case(c, hip, oracle, 4100, 1, 300, seed=21, check_seqs=short + long_ + [4099])
    finally:
        c.deinit()


def test_paged_decode_invalid_entries(ctx, hip, oracle):
    """Device-side entries the host cannot check: a page id outside the pool and
    sequence lengths outside [1, max_seq_len] are never dereferenced; those
    sequences' outputs are NaN, every other sequence is unaffected."""
    s = synth.Shape()
    n_seqs, hq, hkv, hd = 5, s.n_q_heads, s.n_kv_heads, s.head_dim
    lay = synth.paged_layout(n_seqs, 40, 300, 16, seed=11)
    slots = lay.n_pages * 16
    g = np.random.default_rng(11)
    kpool = oracle.f32_to_f16_bits(g.standard_normal((hkv, slots, hd)).astype(np.float32))
    vpool = oracle.f32_to_f16_bits(g.standard_normal((hkv, slots, hd)).astype(np.float32))
    q, k, v, qn, kn = synth.step_inputs(4, 11, n_seqs, s)
    max_len = int(lay.seq_lens.max())
    table, lens = lay.page_table.copy(), lay.seq_lens.copy()
    table[1, 0] = lay.n_pages + 3          # page outside the pool
    lens[2] = 0                            # empty sequence
    lens[3] = max_len + 1                  # longer than max_seq_len
    out = ctx.createBuffer(n_seqs * hq * hd * 4)
    hip.pagedDecode(ctx, hip.PagedDecodeArgs(dev(ctx, q), dev(ctx, k), dev(ctx, v), dev(ctx, qn), dev(ctx, kn),
                                             dev(ctx, kpool), dev(ctx, vpool), dev(ctx, table), dev(ctx, lens), out,
                                             n_seqs, hq, hkv, hd, 16, lay.n_pages, lay.max_pages, max_len, s.eps,
                                             s.theta, 1.0, s.scale))
    got = ctx.to_numpy(out, np.float32).reshape(n_seqs, hq * hd)
    for b in (1, 2, 3):
        assert np.all(np.isnan(got[b])), b
    for b in (0, 4):
        L = int(lens[b])
        kc = oracle.paged_gather_f16(kpool, table[b], 16, L)
        vc = oracle.paged_gather_f16(vpool, table[b], 16, L)
        wout, _, _ = _oracle_step(oracle, q[b:b + 1], k[b:b + 1], v[b:b + 1], qn, kn, np.array([L - 1], np.int32),
                                  kc, vc, L - 1, s)
        check_out(got[b], wout)


# ---------------------------------------------------------------------------
# determinism
# ---------------------------------------------------------------------------

def test_decode_is_deterministic(ctx, hip):
    s = synth.Shape()
    q, k, v, qn, kn = synth.step_inputs(1, 3, 1, s)
    kc, vc = synth.cache_f16(1, 3, s, 2048, 2047)
    a = _run_step(ctx, hip, q, k, v, qn, kn, np.array([2047], np.int32), kc, vc, 2047, s, True)
    b = _run_step(ctx, hip, q, k, v, qn, kn, np.array([2047], np.int32), kc, vc, 2047, s, True)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("fused", [True, False])
def test_config0_golden(ctx, hip, oracle, fused):
    """The committed config-0 vectors (tests/golden/c0), run through the GPU."""
    import os
    from conftest import GOLDEN
    L = lambda n: oracle.load_ds5t(os.path.join(GOLDEN, "c0", f"{n}.ds5t")).data
    s = synth.CONFIGS[0]["shape"]
    q, k, v = L("q"), L("k"), L("v")
    kc, vc = L("k_cache_in"), L("v_cache_in")
    out, gk, gv = _run_step(ctx, hip, q, k, v, L("q_norm"), L("k_norm"), L("positions"), kc, vc, 31, s, fused)
    check_cache(gk, gv, L("k_cache_out"), L("v_cache_out"), kc, vc, 31, 1)
    check_out(out, L("output"))


# ---------------------------------------------------------------------------
# graph capture: every replay equals the eager call
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("kind,T,cap,hd", [
    ("decode", 1, 2048, 128),     # one tile per wavefront (16 splits + merge)
    ("decode", 1, 16384, 128),    # two tiles per wavefront (prefetch loop)
    ("prefill", 300, 307, 128),   # pre-pass + attention
    ("prefill", 77, 84, 64),
])
def test_graph_replays_match_eager(ctx, hip, kind, T, cap, hd):
    """The fused step captured into a HIP graph, replayed three times with eager
    work and synchronisations between the replays: each replay's output is
    bit-identical to the eager call's."""
    s = synth.Shape(n_q_heads=32, n_kv_heads=4, head_dim=hd)
    pos = cap - T if kind == "decode" else cap - T - 7
    config = 1 if kind == "decode" else 2
    q, k, v, qn, kn = synth.step_inputs(config, T, T, s, f16_exact=(kind == "prefill"))
    kc, vc = synth.cache_f16(config, T, s, cap, pos)
    positions = np.arange(pos, pos + T, dtype=np.int32)
    bufs = [dev(ctx, a) for a in (q, k, v, qn, kn, positions, kc, vc)]
    out, other = ctx.createBuffer(T * 32 * hd * 4), ctx.createBuffer(T * 32 * hd * 4)
    args = lambda o: hip.AttentionStepArgs(*bufs, o, 1, pos, T, 32, 4, hd, cap, s.eps, s.theta, 1.0, s.scale)
    hip.attentionStep(ctx, args(out))  # eager; also sizes the workspace before the capture
    want = ctx.to_numpy(out, np.float32)
    g = ctx.capture(lambda: hip.attentionStep(ctx, args(out)))
    try:
        zeros = np.zeros(T * 32 * hd, np.float32)
        for r in range(3):
            ctx.upload(out, 0, zeros)
            hip.attentionStep(ctx, args(other))  # eager work between replays
            ctx.submit()
            g.launch()
            ctx.submit()
            got = ctx.to_numpy(out, np.float32)
            print(f"  replay {r}: bit-identical={np.array_equal(got, want)}", flush=True)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        assert np.array_equal(ctx.to_numpy(other, np.float32).view(np.uint32), want.view(np.uint32))
    finally:
        g.destroy()


def test_capture_before_workspace_sized_fails_cleanly(hip):
    """A call whose workspace would have to grow inside a stream capture fails with a
    DeviceFailure that says to run it once first; the context stays usable."""
    c = hip.Ctx.init(0)
    try:
        s = synth.Shape()
        T, cap = 64, 64
        q, k, v, qn, kn = synth.step_inputs(2, T, T, s, f16_exact=True)
        kc, vc = synth.cache_f16(2, T, s, cap, 0)
        bufs = [c.from_numpy(np.ascontiguousarray(a)) for a in (q, k, v, qn, kn, np.arange(T, dtype=np.int32), kc, vc)]
        out = c.createBuffer(T * 32 * 128 * 4)
        args = hip.AttentionStepArgs(*bufs, out, 1, 0, T, 32, 4, 128, cap, s.eps, s.theta, 1.0, s.scale)
        with pytest.raises(hip.DeviceFailure, match="before capturing"):
            c.capture(lambda: hip.attentionStep(c, args))
        hip.attentionStep(c, args)  # eager: grows the workspace
        eager = c.to_numpy(out, np.float32)
        assert np.all(np.isfinite(eager))
        g = c.capture(lambda: hip.attentionStep(c, args))
        c.upload(out, 0, np.zeros_like(eager))
        g.launch()
        c.submit()
        assert np.array_equal(c.to_numpy(out, np.float32).view(np.uint32), eager.view(np.uint32))
        g.destroy()
    finally:
        c.deinit()


# ---------------------------------------------------------------------------
# matmul (the projection step before the path): kernels_a.zig:136-163
# ---------------------------------------------------------------------------

def _gpu_matmul(ctx, hip, x, w, w_dtype, m, n, k, x_off=0, w_off=0, out_off=0, w_pad=0):
    """Runs ds5_hip_matmul on views at the given byte offsets into fresh buffers."""
    xb = ctx.createBuffer(x.nbytes + x_off)
    wb = ctx.createBuffer(w.nbytes + w_off + w_pad)
    ob = ctx.createBuffer(m * n * 4 + out_off)
    ctx.upload(xb, x_off, np.ascontiguousarray(x))
    ctx.upload(wb, w_off, np.ascontiguousarray(w))
    view = lambda b, off, ln: hip.Buf(b.handle, b.offset + off, ln)
    hip.matmul(ctx, hip.MatmulArgs(view(xb, x_off, x.nbytes), view(wb, w_off, w.nbytes + w_pad), w_dtype,
                                   view(ob, out_off, m * n * 4), m, n, k))
    return ctx.to_numpy(ob, np.float32, (m, n), offset=out_off)


def _dot_bound(x, wf):
    """|a - b| allowed between two f32 evaluations of x . W^T in different orders."""
    return 1e-5 * (np.abs(x).astype(np.float64) @ np.abs(wf).astype(np.float64).T) + 1e-30


@pytest.mark.parametrize("i", range(4))
def test_matmul_quant_fixtures(ctx, hip, oracle, i):
    """kernels_a.zig:395-458 through the GPU: the case tolerance, and the oracle's
    value within the reordering bound."""
    c = _cases(oracle, "matmul_quant")[i]
    p, tol = c["params"], c["tolerance"]
    x, w, want = (_t(oracle, c, n) for n in ("input", "weight", "output"))
    got = _gpu_matmul(ctx, hip, x, w, hip.DTYPE_Q8_0, p["m"], p["n"], p["k"])
    r = oracle.compare(want, got, tol["atol"], tol["rtol"])
    print(f"  fixture max_abs={r.max_abs_diff:.3e} max_rel={r.max_rel_diff:.3e}", flush=True)
    assert r.passed, r
    orc = oracle.matmul(x, w, oracle.Q8_0, p["m"], p["n"], p["k"])
    assert np.all(np.abs(got - orc) <= _dot_bound(x, oracle.q8_0_dequantize(w, p["k"])))


def test_matmul_f32_hand_case(ctx, hip):
    """kernels_a.zig:524-553."""
    x = np.array([[1, 2, 3], [4, 5, 6]], np.float32)
    w = np.array([[1, 0, 2], [0, -1, 1]], np.float32)
    got = _gpu_matmul(ctx, hip, x, w, hip.DTYPE_F32, 2, 2, 3)
    assert np.array_equal(got, np.array([[7, 1], [16, 1]], np.float32))


@pytest.mark.parametrize("m,n,k", [
    (1, 5120, 2048),   # decode q/k/v projection, Qwen3-30B-A3B (hidden 2048 -> 32*128 + 2*4*128)
    (1, 2048, 4096),   # decode output projection (32*128 -> 2048)
    (3, 301, 4096),    # two blocks per lane, a 2-token pass plus a 1-token pass
    (2, 77, 8192),     # four blocks per lane
    (5, 33, 96),       # three blocks, odd row count, 4-token pass plus one
    (15, 40, 512),     # the most tokens the row kernel takes
    (16, 64, 32),      # matrix-core GEMM from 16 tokens: one block
    (17, 256, 256),    # fixture shape, small GEMM tile
    (33, 130, 4096),   # small tiles, ragged tokens and rows
    (128, 512, 2048),  # large tiles, exact
    (200, 300, 2080),  # large tiles, ragged tokens, rows and an odd block count
    (128, 256, 32),    # large tiles, one block: nothing loaded ahead
    (130, 128, 64),    # large tiles, two blocks: one block ahead only
    (256, 384, 96),    # large tiles, three blocks: the pipeline's first full iteration
    (136, 200, 160),   # large tiles, five blocks, ragged rows: each stage and raw area reused
])
def test_matmul_q8_0_and_f32_vs_oracle(ctx, hip, oracle, m, n, k):
    """Q8_0 rows and their dequantised f32 rows against the oracle, within the bound
    for summing the same products in another order."""
    g = np.random.default_rng(m * 7 + n + k)
    rows = oracle.q8_0_quantize(g.standard_normal((n, k)).astype(np.float32) * 0.05)
    wf = oracle.q8_0_dequantize(rows, k)
    x = g.standard_normal((m, k)).astype(np.float32)
    bound = _dot_bound(x, wf)
    for w, dt, odt in ((rows, hip.DTYPE_Q8_0, oracle.Q8_0), (wf, hip.DTYPE_F32, oracle.F32)):
        got = _gpu_matmul(ctx, hip, x, w, dt, m, n, k)
        want = oracle.matmul(x, w, odt, m, n, k)
        err = np.abs(got - want)
        print(f"  dtype {dt}: max |gpu - oracle| = {err.max():.3e} (bound {bound.min():.3e}..)", flush=True)
        assert np.all(np.isfinite(got)) and np.all(err <= bound)


def test_matmul_q8_0_wide_exponent_range(ctx, hip, oracle):
    """x rows from 1e-30 to 1e30 and mixed magnitudes inside rows: the GEMM's
    three-part bf16 split of x keeps f32 accuracy over the whole f32 range."""
    g = np.random.default_rng(5)
    m, n, k = 40, 96, 1024
    rows = oracle.q8_0_quantize(g.standard_normal((n, k)).astype(np.float32) * 0.05)
    wf = oracle.q8_0_dequantize(rows, k)
    x = g.standard_normal((m, k)) * 10.0 ** g.integers(-6, 7, (m, k))
    x = (x * 10.0 ** np.linspace(-24, 24, m)[:, None]).astype(np.float32)
    got = _gpu_matmul(ctx, hip, x, rows, hip.DTYPE_Q8_0, m, n, k)
    want = oracle.matmul(x, rows, oracle.Q8_0, m, n, k)
    assert np.all(np.isfinite(got)) and np.all(np.abs(got - want) <= _dot_bound(x, wf))


# (case, kernel that must run): views the fast kernels do not take (unaligned x or
# weights, a Q8_0 buffer whose last block would be over-read) run the serial
# kernel, bit-identical to the oracle; 2 bytes of slack after the weights, or
# k > 8192 (past the row kernel), take the fast kernels.
_PATH_CASES = [("x_unaligned", "matmul_generic_kernel"), ("w_unaligned", "matmul_generic_kernel"),
               ("q8_tail_no_slack", "matmul_generic_kernel"), ("q8_tail_slack", "matmul_rows_kernel"),
               ("k_gt_8192", "matmul_q8_mfma_kernel"), ("decode", "matmul_rows_kernel"),
               ("prefill", "matmul_q8_mfma_kernel")]


@pytest.mark.parametrize("case,kernel", _PATH_CASES, ids=[c for c, _ in _PATH_CASES])
def test_matmul_paths(ctx, hip, oracle, case, kernel):
    g = np.random.default_rng(len(case))
    m, n, k = {"k_gt_8192": (2, 5, 8224), "q8_tail_no_slack": (1, 3, 32), "q8_tail_slack": (1, 3, 32),
               "decode": (1, 24, 2048), "prefill": (16, 24, 2048)}.get(case, (3, 9, 256))
    rows = oracle.q8_0_quantize(g.standard_normal((n, k)).astype(np.float32))
    x = g.standard_normal((m, k)).astype(np.float32)
    kw = dict(x_off=4) if case == "x_unaligned" else dict(w_off=2) if case == "w_unaligned" else \
        dict(w_pad=2) if case in ("q8_tail_slack", "k_gt_8192") else {}
    ctx.set_kernel_timing(True)
    try:
        before = {kn: ctx.kernel_time(kn)[0] for _, kn in _PATH_CASES}
        got = _gpu_matmul(ctx, hip, x, rows, hip.DTYPE_Q8_0, m, n, k, **kw)
        ran = [kn for kn in before if ctx.kernel_time(kn)[0] > before[kn]]
    finally:
        ctx.set_kernel_timing(False)
    assert ran == [kernel]
    want = oracle.matmul(x, rows, oracle.Q8_0, m, n, k)
    if kernel == "matmul_generic_kernel":
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    else:
        assert np.all(np.abs(got - want) <= _dot_bound(x, oracle.q8_0_dequantize(rows, k)))


_GROUP_CASES = {
    # name: (m, k, rows per entry, weight dtype, byte offset of entry 1's weights, kernel launches)
    "decode_qkv": (1, 2048, (4096, 512, 512), "q8", 0, {"matmul_rows_kernel": 1}),
    "prefill_qkv": (40, 1024, (256, 64, 64), "q8", 0, {"matmul_x_split_kernel": 1, "matmul_q8_mfma_kernel": 1}),
    "prefill_large_tiles": (130, 512, (300, 100), "q8", 0, {"matmul_x_split_kernel": 1, "matmul_q8_mfma_kernel": 1}),
    "f32_passes": (6, 256, (40, 8, 8, 24), "f32", 0, {"matmul_rows_kernel": 2}),
    "empty_entry": (2, 512, (33, 0, 17), "q8", 0, {"matmul_rows_kernel": 1}),
    "mixed_kernels": (4, 256, (20, 9, 7), "q8", 2, {"matmul_rows_kernel": 2, "matmul_generic_kernel": 1}),
}


@pytest.mark.parametrize("case", list(_GROUP_CASES))
def test_matmul_group_equals_separate_calls(ctx, hip, oracle, case):
    """ds5_hip_matmul_group: every entry bit-identical to its own ds5_hip_matmul call;
    one launch when every entry takes the same kernel (the split x made once for the GEMM)."""
    m, k, ns, dt, w1_off, launches = _GROUP_CASES[case]
    g = np.random.default_rng(len(case) * 31 + m)
    x = g.standard_normal((m, k)).astype(np.float32)
    xb = ctx.from_numpy(x)
    dtype = hip.DTYPE_Q8_0 if dt == "q8" else hip.DTYPE_F32
    entries, ws = [], []
    for e, n in enumerate(ns):
        wf = g.standard_normal((n, k)).astype(np.float32) * 0.05
        w = oracle.q8_0_quantize(wf) if dt == "q8" else wf
        off = w1_off if e == 1 else 0
        wb = ctx.createBuffer(w.nbytes + off + 4)
        if w.nbytes:
            ctx.upload(wb, off, np.ascontiguousarray(w))
        wv = hip.Buf(wb.handle, wb.offset + off, w.nbytes)
        entries.append((wv, ctx.createBuffer(max(m * n * 4, 4)), n))
        ws.append(w)
    ctx.set_kernel_timing(True)
    try:
        hip.matmulGroup(ctx, hip.MatmulGroupArgs.of(xb, dtype, m, k, entries))
        ctx.submit()
        counts = {kn: ctx.kernel_time(kn)[0] for kn in ("matmul_rows_kernel", "matmul_x_split_kernel",
                                                         "matmul_q8_mfma_kernel", "matmul_generic_kernel")}
    finally:
        ctx.set_kernel_timing(False)
    assert {kn: c for kn, c in counts.items() if c} == launches
    for (wv, ob, n), w in zip(entries, ws):
        got = ctx.to_numpy(ob, np.float32, (m, n))
        sep = ctx.createBuffer(max(m * n * 4, 4))
        hip.matmul(ctx, hip.MatmulArgs(xb, wv, dtype, hip.Buf(sep.handle, sep.offset, m * n * 4), m, n, k))
        assert np.array_equal(got.view(np.uint32), ctx.to_numpy(sep, np.float32, (m, n)).view(np.uint32))
        if n:
            want = oracle.matmul(x, w, oracle.Q8_0 if dt == "q8" else oracle.F32, m, n, k)
            wf = oracle.q8_0_dequantize(w, k) if dt == "q8" else w
            assert np.all(np.abs(got - want) <= _dot_bound(x, wf))


@pytest.mark.parametrize("n,off", [(97, 0), (2048 * 3, 0), (1000, 2)])
def test_add_bit_exact(ctx, hip, oracle, n, off):
    """kernels_a.zig:703-724 through the GPU: out = x + y bit for bit (specials included),
    out aliasing x; views at a 2-byte offset take the byte-copy path."""
    g = np.random.default_rng(n + off)
    x = g.standard_normal(n).astype(np.float32)
    y = g.standard_normal(n).astype(np.float32)
    x[:5] = [np.inf, -np.inf, np.nan, -0.0, 3.4e38]
    y[:5] = [-np.inf, 1.0, 1.0, -0.0, 3.4e38]
    want = oracle.add(x, y)
    xb, yb = ctx.createBuffer(4 * n + off), ctx.createBuffer(4 * n + off)
    ctx.upload(xb, off, x)
    ctx.upload(yb, off, y)
    xv, yv = hip.Buf(xb.handle, xb.offset + off, 4 * n), hip.Buf(yb.handle, yb.offset + off, 4 * n)
    hip.add(ctx, hip.AddArgs(xv, yv, xv, n))
    got = ctx.to_numpy(xb, np.float32, (n,), offset=off)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("m,n,k,w_off", [(1, 2048, 4096, 0), (3, 300, 2048, 0), (40, 200, 1024, 0), (2, 17, 256, 2)])
def test_matmul_add_equals_matmul_then_add(ctx, hip, oracle, m, n, k, w_off):
    """forward.zig:416-418: residual + x . Wo^T in one call equals ds5_hip_matmul into a
    projection buffer then ds5_hip_add, bit for bit, in place on the residual (row
    kernel, GEMM, and the serial kernel for weights at a 2-byte offset)."""
    g = np.random.default_rng(m * 13 + n + w_off)
    rows = oracle.q8_0_quantize(g.standard_normal((n, k)).astype(np.float32) * 0.05)
    x = g.standard_normal((m, k)).astype(np.float32)
    r = g.standard_normal((m, n)).astype(np.float32)
    xb = ctx.from_numpy(x)
    wb = ctx.createBuffer(rows.nbytes + w_off + 4)
    ctx.upload(wb, w_off, rows)
    wv = hip.Buf(wb.handle, wb.offset + w_off, rows.nbytes)
    res = ctx.from_numpy(r)
    hip.matmulAdd(ctx, hip.MatmulAddArgs(xb, wv, hip.DTYPE_Q8_0, res, res, m, n, k))
    fused = ctx.to_numpy(res, np.float32, (m, n))
    proj, res2 = ctx.createBuffer(m * n * 4), ctx.from_numpy(r)
    hip.matmul(ctx, hip.MatmulArgs(xb, wv, hip.DTYPE_Q8_0, proj, m, n, k))
    hip.add(ctx, hip.AddArgs(res2, proj, res2, m * n))
    assert np.array_equal(fused.view(np.uint32), ctx.to_numpy(res2, np.float32, (m, n)).view(np.uint32))
    want = oracle.add(r, oracle.matmul(x, rows, oracle.Q8_0, m, n, k))
    assert np.all(np.abs(fused - want) <= _dot_bound(x, oracle.q8_0_dequantize(rows, k)) + 1e-6 * np.abs(r))


# ---------------------------------------------------------------------------
# MoE router and experts (kernels_c.zig)
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("i", range(3))
def test_router_fixtures(ctx, hip, oracle, i):
    """kernels_c.zig:250-318 through the GPU: ids exact, weights within the case tolerance,
    and ids equal to the oracle's, weights within 1e-6 of it (the device's expf against
    the C library's, through the softmax sum and the renormalisation)."""
    c = _cases(oracle, "router")[i]
    p, tol = c["params"], c["tolerance"]
    x, w = _t(oracle, c, "input"), _t(oracle, c, "weight")
    T, K = p["n_tokens"], p["top_k"]
    ids, wts = hip.routerTopK(ctx, ctx.from_numpy(x), ctx.from_numpy(w), hip.DTYPE_F32, T, p["dim"], p["n_experts"],
                              K, p["norm_topk_prob"])
    assert np.array_equal(ids.astype(np.int32), _t(oracle, c, "expert_ids").reshape(T, K))
    assert oracle.compare(_t(oracle, c, "gate_weights").reshape(T, K), wts, tol["atol"], tol["rtol"]).passed
    oi, ow = oracle.router_topk(x, w, oracle.F32, T, p["dim"], p["n_experts"], K, p["norm_topk_prob"])
    rel = np.abs(wts - ow) / np.abs(ow)
    print(f"  weights vs oracle: max rel {rel.max():.2e} ({(np.abs(wts - ow) / np.spacing(np.abs(ow))).max():.0f} ulp)")
    assert np.array_equal(ids, oi) and np.all(rel <= 1e-6)


@pytest.mark.parametrize("T,dim,E,dt", [(40, 2048, 128, "f32"), (2048, 2048, 128, "f32"), (70, 100, 200, "f16"),
                                         (1000, 196, 300, "f32")])
def test_router_tiles_equal_per_token(ctx, hip, oracle, T, dim, E, dt):
    """From 32 tokens the logits run in token x expert tiles (router_logits_tile_kernel:
    16 x 16, or 32 x 32 once those fill the chip); every logit is still dotRow's serial
    sum, so ids and weights equal, bit for bit, those of the per-token kernel (one call
    per token); for f32 rows the ids equal the oracle's. Ragged cases: tokens and experts
    not multiples of the tile, dim not a multiple of the 64-element chunk, f16 rows."""
    g = np.random.default_rng(T + dim)
    x = (g.standard_normal((T, dim)) * np.exp(g.uniform(-2, 2, (T, 1)))).astype(np.float32)
    w = (g.standard_normal((E, dim)) * 0.05).astype(np.float32)
    wv, wdt = (w, hip.DTYPE_F32) if dt == "f32" else (w.astype(np.float16), hip.DTYPE_F16)
    xb, wb = ctx.from_numpy(x), ctx.from_numpy(wv)
    K = 8
    ctx.set_kernel_timing(True)
    try:
        ids, wts = hip.routerTopK(ctx, xb, wb, wdt, T, dim, E, K, True)
        assert ctx.kernel_time("router_logits_tile_kernel")[0] == 1
    finally:
        ctx.set_kernel_timing(False)
    ids1, wts1 = np.zeros_like(ids), np.zeros_like(wts)
    for t in range(T):
        i1, w1 = hip.routerTopK(ctx, hip.Buf(xb.handle, xb.offset + t * dim * 4, dim * 4), wb, wdt, 1, dim, E, K, True)
        ids1[t], wts1[t] = i1[0], w1[0]
    assert np.array_equal(ids, ids1)
    assert np.array_equal(wts.view(np.uint32), wts1.view(np.uint32))
    if dt == "f32":
        oi, ow = oracle.router_topk(x, w, oracle.F32, T, dim, E, K, True)
        assert np.array_equal(ids, oi) and np.all(np.abs(wts - ow) <= 1e-6 * np.abs(ow))


@pytest.mark.parametrize("case", ["q8_rows", "dim_102"])
def test_router_many_tokens_untiled(ctx, hip, oracle, case):
    """Many tokens whose rows the tiles do not take -- Q8_0 router rows, or a dim that is not
    a multiple of 4 -- run the per-token kernel (no tile launch); ids equal the oracle's and
    weights are within 1e-6 of them."""
    g = np.random.default_rng(31 + len(case))
    T, dim, E, K = (40, 256, 64, 8) if case == "q8_rows" else (40, 102, 48, 4)
    x = g.standard_normal((T, dim)).astype(np.float32)
    wf = (g.standard_normal((E, dim)) * 0.05).astype(np.float32)
    w, wdt, odt = (oracle.q8_0_quantize(wf), hip.DTYPE_Q8_0, oracle.Q8_0) if case == "q8_rows" else \
        (wf, hip.DTYPE_F32, oracle.F32)
    ctx.set_kernel_timing(True)
    try:
        ids, wts = hip.routerTopK(ctx, ctx.from_numpy(x), ctx.from_numpy(w), wdt, T, dim, E, K, True)
        assert ctx.kernel_time("router_logits_tile_kernel")[0] == 0
        assert ctx.kernel_time("router_logits_kernel")[0] == 1
    finally:
        ctx.set_kernel_timing(False)
    oi, ow = oracle.router_topk(x, w, odt, T, dim, E, K, True)
    assert np.array_equal(ids, oi) and np.all(np.abs(wts - ow) <= 1e-6 * np.abs(ow))


def test_router_hand_cases(ctx, hip):
    """kernels_c.zig:403-477: raw probabilities without renormalisation; exact ties go to
    the lower id."""
    x = ctx.from_numpy(np.array([[1, 0, 0, 0]], np.float32))
    w = ctx.from_numpy(np.array([[2, 0, 0, 0], [0, 9, 9, 9], [1, 0, 0, 0], [-1, 0, 0, 0]], np.float32))
    ids, wts = hip.routerTopK(ctx, x, w, hip.DTYPE_F32, 1, 4, 4, 2, False)
    denom = sum(np.exp(np.float64(l) - 2.0) for l in (2, 0, 1, -1))
    assert ids.tolist() == [[0, 2]] and abs(wts[0, 0] - 1 / denom) <= 1e-6 and abs(wts[0, 1] - np.exp(-1) / denom) <= 1e-6
    w = ctx.from_numpy(np.array([[1, 0, 0, 0], [3, 0, 0, 0], [3, 0, 0, 0], [0, 0, 0, 0]], np.float32))
    ids, wts = hip.routerTopK(ctx, x, w, hip.DTYPE_F32, 1, 4, 4, 3, True)
    assert ids.tolist() == [[1, 2, 0]] and wts[0, 0] == wts[0, 1] and abs(wts.sum() - 1) <= 1e-6


@pytest.mark.parametrize("dt,off", [("f32", 0), ("f16", 0), ("q8", 0), ("f32", 2), ("f16", 1)])
def test_router_vs_oracle(ctx, hip, oracle, dt, off):
    """Qwen3-30B-A3B's router shape (dim 2048, 128 experts, top 8) on 5 tokens, every weight
    dtype, and views at odd offsets (bytewise reads): ids equal to the oracle's, weights
    within 1e-6; logits are the reference's serial dot, so only exp may differ."""
    g = np.random.default_rng(len(dt) * 7 + off)
    T, dim, E, K = 5, 2048, 128, 8
    wf = (g.standard_normal((E, dim)) * 0.03).astype(np.float32)
    if dt == "q8":
        wv, odt, hdt = oracle.q8_0_quantize(wf), oracle.Q8_0, hip.DTYPE_Q8_0
    elif dt == "f16":
        wv, odt, hdt = wf.astype(np.float16).view(np.uint16), oracle.F16, hip.DTYPE_F16
    else:
        wv, odt, hdt = wf, oracle.F32, hip.DTYPE_F32
    x = g.standard_normal((T, dim)).astype(np.float32)
    wb = ctx.createBuffer(wv.nbytes + off)
    ctx.upload(wb, off, np.ascontiguousarray(wv))
    ids, wts = hip.routerTopK(ctx, ctx.from_numpy(x), hip.Buf(wb.handle, wb.offset + off, wv.nbytes), hdt, T, dim, E,
                              K, True)
    oi, ow = oracle.router_topk(x, wv, odt, T, dim, E, K, True)
    assert np.array_equal(ids, oi)
    rel = np.abs(wts - ow) / np.abs(ow)
    print(f"  weights vs oracle: max rel {rel.max():.2e}", flush=True)
    assert np.all(rel <= 1e-6)


@pytest.mark.parametrize("E,K", [(300, 8), (128, 80), (16384, 8), (257, 64)])
def test_router_wide_selects(ctx, hip, oracle, E, K):
    """router_select_kernel beyond its register path (more than 256 experts or more than
    64 picks) and at the 16384-expert limit of its LDS: ids equal to the oracle's,
    weights within 1e-6."""
    g = np.random.default_rng(E + K)
    T, dim = 3, 64
    w = (g.standard_normal((E, dim)) * 0.05).astype(np.float32)
    x = g.standard_normal((T, dim)).astype(np.float32)
    ids, wts = hip.routerTopK(ctx, ctx.from_numpy(x), ctx.from_numpy(w), hip.DTYPE_F32, T, dim, E, K, True)
    oi, ow = oracle.router_topk(x, w, oracle.F32, T, dim, E, K, True)
    assert np.array_equal(ids, oi)
    rel = np.abs(wts - ow) / np.abs(ow)
    print(f"  E={E} K={K}: weights vs oracle max rel {rel.max():.2e}", flush=True)
    assert np.all(rel <= 1e-6)


@pytest.mark.parametrize("i", range(3))
def test_expert_mlp_fixtures(ctx, hip, oracle, i):
    """kernels_c.zig:320-401 through the GPU: Q8_0 banks, token-major pairs, the case tolerance."""
    c = _cases(oracle, "expert_mlp")[i]
    p, tol = c["params"], c["tolerance"]
    T, dim, ffn, E, K = p["n_tokens"], p["dim"], p["ffn_dim"], p["n_experts"], p["top_k"]
    x = _t(oracle, c, "input")
    banks = [ctx.from_numpy(_t(oracle, c, n)) for n in ("gate", "up", "down")]
    pairs = oracle.pairs_from_router(_t(oracle, c, "expert_ids").reshape(T, K), _t(oracle, c, "gate_weights").reshape(T, K))
    out = ctx.from_numpy(np.zeros((T, dim), np.float32))
    hip.expertMlpSwiglu(ctx, ctx.from_numpy(x), *banks, hip.DTYPE_Q8_0, pairs, out, T, dim, ffn, E)
    got = ctx.to_numpy(out, np.float32, (T, dim))
    assert oracle.compare(_t(oracle, c, "output").reshape(T, dim), got, tol["atol"], tol["rtol"]).passed


def test_expert_mlp_hand_cases(ctx, hip, oracle):
    """kernels_c.zig:550-623: no pairs leave out untouched; two f32 pairs accumulate."""
    bank = ctx.from_numpy(np.zeros((32, 34), np.uint8))
    out = ctx.from_numpy(np.full((2, 32), 7.0, np.float32))
    hip.expertMlpSwiglu(ctx, ctx.from_numpy(np.zeros((2, 32), np.float32)), bank, bank, bank, hip.DTYPE_Q8_0,
                        np.zeros(0, hip.PAIR_DTYPE), out, 2, 32, 32, 1)
    assert np.all(ctx.to_numpy(out, np.float32, (2, 32)) == 7.0)
    x = np.array([[1.0, -2.0]], np.float32)
    gate, up, down = (np.array(v, np.float32) for v in ([1, 0, 0, 1, 0, 1, 1, 0], [2, 0, 0, 2, 2, 0, 0, 2],
                                                        [1, 0, 0, 1, 0, 1, 1, 0]))
    pairs = np.array([(0, 0, 0.5), (0, 1, 2.0)], hip.PAIR_DTYPE)
    out = ctx.from_numpy(np.zeros((1, 2), np.float32))
    hip.expertMlpSwiglu(ctx, ctx.from_numpy(x), ctx.from_numpy(gate), ctx.from_numpy(up), ctx.from_numpy(down),
                        hip.DTYPE_F32, pairs, out, 1, 2, 2, 2)
    want = oracle.expert_mlp_swiglu(x, gate, up, down, oracle.F32, pairs.astype(oracle.PAIR_DTYPE), 1, 2, 2, 2)
    assert np.all(np.abs(ctx.to_numpy(out, np.float32, (1, 2)) - want) <= 1e-6)


def _expert_bound(x, G, U, D, pairs, T, dim, ffn):
    """Elementwise bound for two f32 evaluations of the expert MLP in different orders:
    1e-5 of the magnitudes the sums run over, through silu and the down projection."""
    ax = np.abs(x).astype(np.float64)
    b = np.zeros((T, dim))
    for t, e, wt in pairs.tolist():
        gm = np.abs(G[e * ffn:(e + 1) * ffn]) @ ax[t]
        um = np.abs(U[e * ffn:(e + 1) * ffn]) @ ax[t]
        hm = (gm + 1e-30) * (um + 1e-30) * 1.5
        b[t] += abs(wt) * (np.abs(D[e * dim:(e + 1) * dim]) @ hm)
    return 1e-5 * b + 1e-30


@pytest.mark.parametrize("case", ["decode_q8", "prefill_q8_interleaved", "f32", "serial_unaligned"])
def test_expert_mlp_vs_oracle(ctx, hip, oracle, case):
    """Qwen3-30B-A3B-shaped experts (dim 2048, ffn 768; fewer experts) against the oracle
    within a reordering bound: a decode token's 8 pairs; 6 tokens with their pairs
    interleaved (each token's contributions still added in list order); f32 banks; a bank
    view at a 2-byte offset (serial kernels)."""
    g = np.random.default_rng(len(case))
    E = 16
    T, dim, ffn = {"decode_q8": (1, 2048, 768), "prefill_q8_interleaved": (6, 2048, 768), "f32": (3, 256, 96),
                   "serial_unaligned": (2, 256, 96)}[case]
    q8 = case != "f32"
    mk = lambda rows, k: (g.standard_normal((rows, k)) * 0.05).astype(np.float32)
    Gf, Uf, Df = mk(E * ffn, dim), mk(E * ffn, dim), mk(E * dim, ffn)
    if q8:
        G, U, D = (oracle.q8_0_quantize(v) for v in (Gf, Uf, Df))
        Gf, Uf, Df = oracle.q8_0_dequantize(G, dim), oracle.q8_0_dequantize(U, dim), oracle.q8_0_dequantize(D, ffn)
    else:
        G, U, D = Gf, Uf, Df
    x = g.standard_normal((T, dim)).astype(np.float32)
    K = 8 if case == "decode_q8" else 3
    pairs = np.zeros(T * K, hip.PAIR_DTYPE)
    pairs["token"] = np.tile(np.arange(T), K) if case == "prefill_q8_interleaved" else np.repeat(np.arange(T), K)
    pairs["expert"] = g.integers(0, E, T * K)
    pairs["weight"] = g.random(T * K).astype(np.float32)
    off = 2 if case == "serial_unaligned" else 0
    bufs = []
    for arr in (G, U, D):
        b = ctx.createBuffer(arr.nbytes + off + 4)
        ctx.upload(b, off, np.ascontiguousarray(arr))
        bufs.append(hip.Buf(b.handle, b.offset + off, arr.nbytes))
    r = g.standard_normal((T, dim)).astype(np.float32)
    out = ctx.from_numpy(r)
    ctx.set_kernel_timing(True)
    try:
        hip.expertMlpSwiglu(ctx, ctx.from_numpy(x), *bufs, hip.DTYPE_Q8_0 if q8 else hip.DTYPE_F32, pairs, out, T, dim,
                            ffn, E)
        ctx.submit()
        serial = ctx.kernel_time("moe_gate_up_serial_kernel")[0]
    finally:
        ctx.set_kernel_timing(False)
    assert serial == (1 if case == "serial_unaligned" else 0)
    got = ctx.to_numpy(out, np.float32, (T, dim))
    want = oracle.expert_mlp_swiglu(x, G, U, D, oracle.Q8_0 if q8 else oracle.F32, pairs.astype(oracle.PAIR_DTYPE), T,
                                    dim, ffn, E, out=r)
    bound = _expert_bound(x, Gf.astype(np.float64), Uf.astype(np.float64), Df.astype(np.float64), pairs, T, dim, ffn)
    assert np.all(np.abs(got - want) <= bound + 2 * np.spacing(np.abs(want)))


@pytest.mark.parametrize("case", ["qwen_shape", "skewed", "narrow", "rows128", "many_experts"])
def test_expert_mlp_grouped_vs_oracle(ctx, hip, oracle, case):
    """Pair lists with at least two pairs per expert run grouped by expert on the matrix
    cores (moe_sort_kernel, the split x / h planes, one Q8_0 product per expert row tile),
    against the oracle within the reordering bound of the wavefront kernels' test, twice
    (the rows of one expert land in any order: the results must not depend on it).
    qwen_shape: dim 2048, ffn 768, 64 tokens x 8 pairs over 16 experts; skewed: most pairs
    on one expert (five 64-row tiles, the last partial), four experts without pairs;
    narrow: dim 256, ffn 96 (a partial column tile), pairs interleaved across tokens;
    rows128: 128 pairs per expert, the 128-row tiles; many_experts: 1100 experts (some of the
    sort's threads own two experts each in its scans)."""
    g = np.random.default_rng(500 + len(case))
    T, dim, ffn, E, K = {"qwen_shape": (64, 2048, 768, 16, 8), "skewed": (40, 512, 256, 12, 8),
                         "narrow": (24, 256, 96, 8, 3), "rows128": (256, 256, 96, 16, 8),
                         "many_experts": (300, 256, 64, 1100, 8)}[case]
    mk = lambda rows, k: oracle.q8_0_quantize((g.standard_normal((rows, k)) * 0.05).astype(np.float32))
    G, U, D = mk(E * ffn, dim), mk(E * ffn, dim), mk(E * dim, ffn)
    Gf, Uf, Df = (oracle.q8_0_dequantize(v, k).astype(np.float64) for v, k in ((G, dim), (U, dim), (D, ffn)))
    x = g.standard_normal((T, dim)).astype(np.float32)
    x[3] *= 1e-3  # rows of other magnitudes (their own plane exponents)
    x[5] = 0.0
    pairs = np.zeros(T * K, hip.PAIR_DTYPE)
    pairs["token"] = np.tile(np.arange(T), K) if case == "narrow" else np.repeat(np.arange(T), K)
    if case == "skewed":
        ex = g.integers(0, E - 4, T * K)
        ex[g.random(T * K) < 0.85] = 2  # ~272 of 320 pairs: tiles of 128, 128 and ~16 rows
        pairs["expert"] = ex
    else:
        pairs["expert"] = g.integers(0, E, T * K)
    pairs["weight"] = g.random(T * K).astype(np.float32)
    assert T * K >= 2 * E
    bufs = [ctx.from_numpy(v) for v in (G, U, D)]
    xb = ctx.from_numpy(x)
    r = g.standard_normal((T, dim)).astype(np.float32)
    want = oracle.expert_mlp_swiglu(x, G, U, D, oracle.Q8_0, pairs.astype(oracle.PAIR_DTYPE), T, dim, ffn, E, out=r)
    bound = _expert_bound(x, Gf, Uf, Df, pairs, T, dim, ffn)
    runs = []
    for _ in range(2):
        out = ctx.from_numpy(r)
        ctx.set_kernel_timing(True)
        try:
            hip.expertMlpSwiglu(ctx, xb, *bufs, hip.DTYPE_Q8_0, pairs, out, T, dim, ffn, E)
            ctx.submit()
            launches = {kn: ctx.kernel_time(kn)[0] for kn in ("moe_sort_kernel", "moe_gate_up_kernel",
                                                               "moe_h_split_kernel", "moe_combine_kernel")}
        finally:
            ctx.set_kernel_timing(False)
        assert launches == {"moe_sort_kernel": 1, "moe_gate_up_kernel": 0, "moe_h_split_kernel": 1,
                            "moe_combine_kernel": 1}, launches
        runs.append(ctx.to_numpy(out, np.float32, (T, dim)))
    got = runs[0]
    assert np.all(np.abs(got - want) <= bound + 2 * np.spacing(np.abs(want)))
    assert np.array_equal(runs[0].view(np.uint32), runs[1].view(np.uint32))


def test_expert_mlp_grouped_threshold(ctx, hip, oracle):
    """Below two pairs per expert on average the wavefront kernels run (no sort), from it
    the grouped path; both agree with the oracle within the reordering bound."""
    g = np.random.default_rng(7)
    dim, ffn, E = 256, 64, 8
    mk = lambda rows, k: oracle.q8_0_quantize((g.standard_normal((rows, k)) * 0.05).astype(np.float32))
    G, U, D = mk(E * ffn, dim), mk(E * ffn, dim), mk(E * dim, ffn)
    Gf, Uf, Df = (oracle.q8_0_dequantize(v, k).astype(np.float64) for v, k in ((G, dim), (U, dim), (D, ffn)))
    bufs = [ctx.from_numpy(v) for v in (G, U, D)]
    for P, sorts in ((2 * E - 1, 0), (2 * E, 1)):
        T = P
        x = g.standard_normal((T, dim)).astype(np.float32)
        pairs = np.zeros(P, hip.PAIR_DTYPE)
        pairs["token"] = np.arange(P)
        pairs["expert"] = np.arange(P) % E
        pairs["weight"] = 1.0
        out = ctx.createBuffer(T * dim * 4)
        ctx.zero(out, T * dim * 4)
        ctx.set_kernel_timing(True)
        try:
            hip.expertMlpSwiglu(ctx, ctx.from_numpy(x), *bufs, hip.DTYPE_Q8_0, pairs, out, T, dim, ffn, E)
            ctx.submit()
            n_sort = ctx.kernel_time("moe_sort_kernel")[0]
        finally:
            ctx.set_kernel_timing(False)
        assert n_sort == sorts
        want = oracle.expert_mlp_swiglu(x, G, U, D, oracle.Q8_0, pairs.astype(oracle.PAIR_DTYPE), T, dim, ffn, E)
        bound = _expert_bound(x, Gf, Uf, Df, pairs, T, dim, ffn)
        got = ctx.to_numpy(out, np.float32, (T, dim))
        assert np.all(np.abs(got - want) <= bound + 2 * np.spacing(np.abs(want)))


@pytest.mark.parametrize("case", ["f32_banks", "experts_2049"])
def test_expert_mlp_many_pairs_not_grouped(ctx, hip, oracle, case):
    """Many pairs per expert but banks the grouped path does not take: f32 banks (the
    matrix-core products read Q8_0 only), or more experts than the sort's LDS holds
    (2049): the wavefront kernels run (no sort), against the oracle within the
    reordering bound."""
    g = np.random.default_rng(11 + len(case))
    T, dim, ffn, E, K = {"f32_banks": (64, 256, 64, 8, 4), "experts_2049": (1025, 32, 32, 2049, 4)}[case]
    q8 = case != "f32_banks"
    mk = lambda rows, k: (g.standard_normal((rows, k)) * 0.05).astype(np.float32)
    Gf, Uf, Df = mk(E * ffn, dim), mk(E * ffn, dim), mk(E * dim, ffn)
    if q8:
        G, U, D = (oracle.q8_0_quantize(v) for v in (Gf, Uf, Df))
        Gf, Uf, Df = oracle.q8_0_dequantize(G, dim), oracle.q8_0_dequantize(U, dim), oracle.q8_0_dequantize(D, ffn)
    else:
        G, U, D = Gf, Uf, Df
    x = g.standard_normal((T, dim)).astype(np.float32)
    pairs = np.zeros(T * K, hip.PAIR_DTYPE)
    pairs["token"] = np.repeat(np.arange(T), K)
    pairs["expert"] = g.integers(0, E, T * K)
    pairs["weight"] = g.random(T * K).astype(np.float32)
    assert T * K >= 2 * E
    out = ctx.createBuffer(T * dim * 4)
    ctx.zero(out, T * dim * 4)
    ctx.set_kernel_timing(True)
    try:
        hip.expertMlpSwiglu(ctx, ctx.from_numpy(x), *(ctx.from_numpy(v) for v in (G, U, D)),
                            hip.DTYPE_Q8_0 if q8 else hip.DTYPE_F32, pairs, out, T, dim, ffn, E)
        ctx.submit()
        launches = {kn: ctx.kernel_time(kn)[0] for kn in ("moe_sort_kernel", "moe_gate_up_kernel")}
    finally:
        ctx.set_kernel_timing(False)
    assert launches == {"moe_sort_kernel": 0, "moe_gate_up_kernel": 1}, launches
    want = oracle.expert_mlp_swiglu(x, G, U, D, oracle.Q8_0 if q8 else oracle.F32, pairs.astype(oracle.PAIR_DTYPE), T,
                                    dim, ffn, E)
    bound = _expert_bound(x, Gf.astype(np.float64), Uf.astype(np.float64), Df.astype(np.float64), pairs, T, dim, ffn)
    got = ctx.to_numpy(out, np.float32, (T, dim))
    assert np.all(np.abs(got - want) <= bound + 2 * np.spacing(np.abs(want)))


def test_expert_mlp_bad_pair_leaves_out(ctx, hip):
    """A pair out of range is ShapeMismatch before anything runs (out unchanged)."""
    bank = ctx.from_numpy(np.zeros((2 * 32, 34), np.uint8))
    out = ctx.from_numpy(np.full((1, 32), 3.0, np.float32))
    with pytest.raises(hip.ShapeMismatch):
        hip.expertMlpSwiglu(ctx, ctx.from_numpy(np.ones((1, 32), np.float32)), bank, bank, bank, hip.DTYPE_Q8_0,
                            np.array([(0, 1, 1.0), (0, 2, 1.0)], hip.PAIR_DTYPE), out, 1, 32, 32, 2)
    assert np.all(ctx.to_numpy(out, np.float32, (1, 32)) == 3.0)


@pytest.mark.parametrize("T,E", [(1, 32), (5, 32), (1, 128), (3, 200), (64, 32)])
def test_moe_device_equals_router_then_experts(ctx, hip, oracle, T, E):
    """ds5_hip_moe (router and experts on the device, pairs never leave it) equals
    ds5_hip_router_topk then ds5_hip_expert_mlp_swiglu on the router's pairs, bit for bit;
    the device ids / weights equal the host ones. 128 and 200 experts: two and four
    register slots per lane in the selection, the last one partly filled at 200. 64 tokens
    over 32 experts: the experts run grouped by expert."""
    g = np.random.default_rng(T)
    dim, ffn, K = 2048, 768, 8
    rw = (g.standard_normal((E, dim)) * 0.03).astype(np.float32)
    mk = lambda rows, k: oracle.q8_0_quantize((g.standard_normal((rows, k)) * 0.05).astype(np.float32))
    G, U, D = mk(E * ffn, dim), mk(E * ffn, dim), mk(E * dim, ffn)
    x = g.standard_normal((T, dim)).astype(np.float32)
    xb, rwb = ctx.from_numpy(x), ctx.from_numpy(rw)
    banks = [ctx.from_numpy(v) for v in (G, U, D)]
    r = g.standard_normal((T, dim)).astype(np.float32)
    out1, ids_b, w_b = ctx.from_numpy(r), ctx.createBuffer(T * K * 2), ctx.createBuffer(T * K * 4)
    hip.moe(ctx, hip.MoeArgs(xb, rwb, hip.DTYPE_F32, *banks, hip.DTYPE_Q8_0, out1, ids_b, w_b, T, dim, ffn, E, K, 1))
    ids, wts = hip.routerTopK(ctx, xb, rwb, hip.DTYPE_F32, T, dim, E, K, True)
    out2 = ctx.from_numpy(r)
    hip.expertMlpSwiglu(ctx, xb, *banks, hip.DTYPE_Q8_0, oracle.pairs_from_router(ids, wts).astype(hip.PAIR_DTYPE),
                        out2, T, dim, ffn, E)
    assert np.array_equal(ctx.to_numpy(ids_b, np.uint16, (T, K)), ids)
    assert np.array_equal(ctx.to_numpy(w_b, np.float32, (T, K)).view(np.uint32), wts.view(np.uint32))
    a, b = ctx.to_numpy(out1, np.float32, (T, dim)), ctx.to_numpy(out2, np.float32, (T, dim))
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("T", [1, 64])
def test_moe_graph_replays_match_eager(ctx, hip, oracle, T):
    """ds5_hip_moe with ffn_norm and a residual captured into a HIP graph, replayed three
    times with eager work and synchronisations between the replays: each replay's output is
    bit-identical to the eager call's. T = 1: the norm in the logits kernel, the wavefront
    experts; T = 64: the norm as its own launch, the logits in tiles, the experts grouped
    (sort, split planes, grouped products, combine)."""
    g = np.random.default_rng(900 + T)
    dim, ffn, E, K = 2048, 768, 64, 8
    rw = (g.standard_normal((E, dim)) * 0.03).astype(np.float32)
    mk = lambda rows, k: oracle.q8_0_quantize((g.standard_normal((rows, k)) * 0.05).astype(np.float32))
    banks = [ctx.from_numpy(v) for v in (mk(E * ffn, dim), mk(E * ffn, dim), mk(E * dim, ffn))]
    x = g.standard_normal((T, dim)).astype(np.float32)
    nw = (1.0 + 0.05 * g.standard_normal(dim)).astype(np.float32)
    res = g.standard_normal((T, dim)).astype(np.float32)
    xb, rwb, nwb, rb = ctx.from_numpy(x), ctx.from_numpy(rw), ctx.from_numpy(nw), ctx.from_numpy(res)
    out, other = ctx.createBuffer(T * dim * 4), ctx.createBuffer(T * dim * 4)
    args = lambda o: hip.MoeArgs(xb, rwb, hip.DTYPE_F32, *banks, hip.DTYPE_Q8_0, o, hip.Buf(), hip.Buf(), T, dim, ffn,
                                 E, K, 1, rb, nwb, 1e-6)
    hip.moe(ctx, args(out))  # eager; also sizes the workspaces before the capture
    want = ctx.to_numpy(out, np.float32)
    gr = ctx.capture(lambda: hip.moe(ctx, args(out)))
    try:
        zeros = np.zeros(T * dim, np.float32)
        for r in range(3):
            ctx.upload(out, 0, zeros)
            hip.moe(ctx, args(other))  # eager work between replays
            ctx.submit()
            gr.launch()
            ctx.submit()
            got = ctx.to_numpy(out, np.float32)
            print(f"  replay {r}: bit-identical={np.array_equal(got, want)}", flush=True)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        assert np.array_equal(ctx.to_numpy(other, np.float32).view(np.uint32), want.view(np.uint32))
    finally:
        gr.destroy()


@pytest.mark.parametrize("T", [1, 5, 64, 300])
def test_moe_residual_equals_zero_moe_add(ctx, hip, oracle, T):
    """ds5_hip_moe with a residual (out = residual + the experts' sum from zero) equals the
    engine's three calls -- zero the accumulator, ds5_hip_moe into it, ds5_hip_add(x, acc ->
    x) -- bit for bit, in place (out = residual) and into another buffer; residual values
    include -0.0 (-0 + 0 = +0 through the add) and large magnitudes. T = 64: 512 pairs over
    64 experts, grouped by expert on the matrix cores. T = 300: the serial
    banks (a view that is not 4-byte aligned), whose experts run as separate kernels."""
    g = np.random.default_rng(100 + T)
    dim, ffn, E, K = (2048, 768, 64, 8) if T < 300 else (256, 64, 8, 2)
    rw = (g.standard_normal((E, dim)) * 0.03).astype(np.float32)
    mk = lambda rows, k: oracle.q8_0_quantize((g.standard_normal((rows, k)) * 0.05).astype(np.float32))
    G, U, D = mk(E * ffn, dim), mk(E * ffn, dim), mk(E * dim, ffn)
    x = g.standard_normal((T, dim)).astype(np.float32)
    res = (g.standard_normal((T, dim)) * np.exp(g.uniform(-6, 6, (T, 1)))).astype(np.float32)
    res[:, :7] = -0.0
    xb, rwb = ctx.from_numpy(x), ctx.from_numpy(rw)
    if T < 300:
        banks = [ctx.from_numpy(v) for v in (G, U, D)]
    else:  # views one byte into their allocations: the serial kernels
        banks = []
        for v in (G, U, D):
            raw = np.zeros(v.size + 1, np.uint8)
            raw[1:] = v.reshape(-1)
            b = ctx.from_numpy(raw)
            banks.append(hip.Buf(b.handle, b.offset + 1, v.size))
    empty = hip.Buf()
    acc, xr = ctx.createBuffer(T * dim * 4), ctx.from_numpy(res)
    ctx.zero(acc, T * dim * 4)
    hip.moe(ctx, hip.MoeArgs(xb, rwb, hip.DTYPE_F32, *banks, hip.DTYPE_Q8_0, acc, empty, empty, T, dim, ffn, E, K, 1))
    hip.add(ctx, hip.AddArgs(xr, acc, xr, T * dim))
    want = ctx.to_numpy(xr, np.float32, (T, dim))
    inplace = ctx.from_numpy(res)
    hip.moe(ctx, hip.MoeArgs(xb, rwb, hip.DTYPE_F32, *banks, hip.DTYPE_Q8_0, inplace, empty, empty, T, dim, ffn, E,
                             K, 1, inplace))
    other, rb = ctx.createBuffer(T * dim * 4), ctx.from_numpy(res)
    hip.moe(ctx, hip.MoeArgs(xb, rwb, hip.DTYPE_F32, *banks, hip.DTYPE_Q8_0, other, empty, empty, T, dim, ffn, E, K,
                             1, rb))
    for b in (inplace, other):
        got = ctx.to_numpy(b, np.float32, (T, dim))
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert np.array_equal(ctx.to_numpy(rb, np.float32, (T, dim)).view(np.uint32), res.view(np.uint32))
    with pytest.raises(hip.ShapeMismatch):
        hip.moe(ctx, hip.MoeArgs(xb, rwb, hip.DTYPE_F32, *banks, hip.DTYPE_Q8_0, other, empty, empty, T, dim, ffn, E,
                                 K, 1, hip.Buf(rb.handle, rb.offset, T * dim * 4 - 4)))


@pytest.mark.parametrize("T,dim,rdt", [(1, 2048, "f32"), (5, 2048, "f32"), (3, 2048, "f16"), (2, 256, "f32"),
                                        (20, 2048, "f32"), (40, 2048, "f32")])
def test_moe_norm_equals_rmsnorm_then_moe(ctx, hip, oracle, T, dim, rdt):
    """ds5_hip_moe with x_norm (ffn_norm applied first) and the residual equals
    ds5_hip_rms_norm(x -> h2) then ds5_hip_moe(h2) with the residual, bit for bit, and
    leaves x as it was when out is another buffer: the norm inside the router's f32 logits
    kernel (rows above 256 elements), or written to the context's second buffer first (an
    f16 router; dim 256: the serial order; 20 tokens: the norm in the per-token logits
    kernel, the experts grouped on its h; 40 tokens: the logits in tiles, the experts
    grouped). The router ids and weights agree too."""
    g = np.random.default_rng(300 + T + dim)
    ffn, E, K = (768, 64, 8) if dim == 2048 else (64, 8, 2)
    rw = (g.standard_normal((E, dim)) * 0.03).astype(np.float32)
    rwv = rw if rdt == "f32" else rw.astype(np.float16)
    rdtype = hip.DTYPE_F32 if rdt == "f32" else hip.DTYPE_F16
    mk = lambda rows, k: oracle.q8_0_quantize((g.standard_normal((rows, k)) * 0.05).astype(np.float32))
    banks = [ctx.from_numpy(v) for v in (mk(E * ffn, dim), mk(E * ffn, dim), mk(E * dim, ffn))]
    x = (g.standard_normal((T, dim)) * np.exp(g.uniform(-3, 3, (T, 1)))).astype(np.float32)
    nw = (1.0 + 0.05 * g.standard_normal(dim)).astype(np.float32)
    xb, rwb, nwb = ctx.from_numpy(x), ctx.from_numpy(rwv), ctx.from_numpy(nw)
    empty = hip.Buf()
    ids1, w1 = ctx.createBuffer(T * K * 2), ctx.createBuffer(T * K * 4)
    out1 = ctx.createBuffer(T * dim * 4)
    hip.moe(ctx, hip.MoeArgs(xb, rwb, rdtype, *banks, hip.DTYPE_Q8_0, out1, ids1, w1, T, dim, ffn, E, K, 1, xb, nwb,
                             1e-6))
    h2 = ctx.createBuffer(T * dim * 4)
    hip.rmsNorm(ctx, hip.RmsNormArgs(xb, nwb, h2, T, dim, 1e-6))
    ids2, w2 = ctx.createBuffer(T * K * 2), ctx.createBuffer(T * K * 4)
    out2 = ctx.createBuffer(T * dim * 4)
    hip.moe(ctx, hip.MoeArgs(h2, rwb, rdtype, *banks, hip.DTYPE_Q8_0, out2, ids2, w2, T, dim, ffn, E, K, 1, xb))
    a, b = ctx.to_numpy(out1, np.float32, (T, dim)), ctx.to_numpy(out2, np.float32, (T, dim))
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert np.array_equal(ctx.to_numpy(ids1, np.uint16, (T, K)), ctx.to_numpy(ids2, np.uint16, (T, K)))
    assert np.array_equal(ctx.to_numpy(w1, np.uint32, (T, K)), ctx.to_numpy(w2, np.uint32, (T, K)))
    assert np.array_equal(ctx.to_numpy(xb, np.float32, (T, dim)).view(np.uint32), x.view(np.uint32))
    inplace = ctx.from_numpy(x)  # out = residual = x: the engine's form
    hip.moe(ctx, hip.MoeArgs(inplace, rwb, rdtype, *banks, hip.DTYPE_Q8_0, inplace, empty, empty, T, dim, ffn, E, K, 1,
                             inplace, nwb, 1e-6))
    assert np.array_equal(ctx.to_numpy(inplace, np.float32, (T, dim)).view(np.uint32), b.view(np.uint32))
    with pytest.raises(hip.ShapeMismatch):
        hip.moe(ctx, hip.MoeArgs(xb, rwb, rdtype, *banks, hip.DTYPE_Q8_0, out1, empty, empty, T, dim, ffn, E, K, 1,
                                 xb, hip.Buf(nwb.handle, nwb.offset, dim * 4 - 4), 1e-6))


@pytest.mark.parametrize("T,ffn", [(1, 768), (5, 768), (3, 2048), (2, 96)])
def test_moe_two_launch_down_equals_fused_down(hip, oracle, T, ffn):
    """The experts' down GEMV and combine as two launches (moe_down_kernel, then
    moe_combine_kernel: the path for outputs beyond one grid, forced here with
    DS5_HIP_MOE_TWO_LAUNCH, read when a context starts) equal the one-launch
    moe_down_combine_kernel bit for bit, with and without the residual; ffn 96 and 768
    leave lanes of the 8-slot layout without blocks, ffn 2048 gives each slot 8."""
    import os
    os.environ["DS5_HIP_MOE_TWO_LAUNCH"] = "1"
    try:
        c2 = hip.Ctx.init(0)
    finally:
        del os.environ["DS5_HIP_MOE_TWO_LAUNCH"]
    c1 = hip.Ctx.init(0)
    try:
        g = np.random.default_rng(400 + T + ffn)
        dim, E, K = 256, 16, 4
        rw = (g.standard_normal((E, dim)) * 0.1).astype(np.float32)
        mk = lambda rows, k: oracle.q8_0_quantize((g.standard_normal((rows, k)) * 0.05).astype(np.float32))
        G, U, D = mk(E * ffn, dim), mk(E * ffn, dim), mk(E * dim, ffn)
        x = g.standard_normal((T, dim)).astype(np.float32)
        r = g.standard_normal((T, dim)).astype(np.float32)
        outs = []
        for c in (c1, c2):
            xb, rwb, rb = c.from_numpy(x), c.from_numpy(rw), c.from_numpy(r)
            banks = [c.from_numpy(v) for v in (G, U, D)]
            acc, res_out = c.from_numpy(r), c.createBuffer(T * dim * 4)
            hip.moe(c, hip.MoeArgs(xb, rwb, hip.DTYPE_F32, *banks, hip.DTYPE_Q8_0, acc, hip.Buf(), hip.Buf(), T, dim,
                                   ffn, E, K, 1))
            hip.moe(c, hip.MoeArgs(xb, rwb, hip.DTYPE_F32, *banks, hip.DTYPE_Q8_0, res_out, hip.Buf(), hip.Buf(), T,
                                   dim, ffn, E, K, 1, rb))
            c.set_kernel_timing(True)
            try:
                hip.moe(c, hip.MoeArgs(xb, rwb, hip.DTYPE_F32, *banks, hip.DTYPE_Q8_0, c.createBuffer(T * dim * 4),
                                       hip.Buf(), hip.Buf(), T, dim, ffn, E, K, 1))
                c.submit()
                launches = {kn: c.kernel_time(kn)[0] for kn in ("moe_down_combine_kernel", "moe_down_kernel",
                                                                 "moe_combine_kernel")}
            finally:
                c.set_kernel_timing(False)
            outs.append((c.to_numpy(acc, np.float32, (T, dim)), c.to_numpy(res_out, np.float32, (T, dim)), launches))
        (a1, b1, l1), (a2, b2, l2) = outs
        assert l1 == {"moe_down_combine_kernel": 1, "moe_down_kernel": 0, "moe_combine_kernel": 0}, l1
        assert l2 == {"moe_down_combine_kernel": 0, "moe_down_kernel": 1, "moe_combine_kernel": 1}, l2
        assert np.array_equal(a1.view(np.uint32), a2.view(np.uint32))
        assert np.array_equal(b1.view(np.uint32), b2.view(np.uint32))
    finally:
        c1.deinit()
        c2.deinit()


def test_matmul_device_errors(ctx, hip):
    x, w, out = ctx.createBuffer(4 * 64), ctx.createBuffer(2 * 68), ctx.createBuffer(8)
    with pytest.raises(hip.UnsupportedDtype):
        hip.matmul(ctx, hip.MatmulArgs(x, w, 12, out, 1, 2, 64))
    with pytest.raises(hip.ShapeMismatch):
        hip.matmul(ctx, hip.MatmulArgs(x, w, hip.DTYPE_Q8_0, out, 1, 2, 48))
