"""Attention over f32 caches on the f32 matrix cores, and the step's fused norm / rope /
append: each shape against float64, at the edges of the 16-row and 16-position tiles, of the
splits and of the two launch forms (a workgroup or a wavefront per row tile)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS24 = 2.0 ** -24


def _inputs(T, pos, hq, hkv, d, cap, seed=0):
    g = np.random.default_rng(seed)
    q = g.standard_normal((T, hq, d)).astype(np.float32)
    kc, vc = (g.standard_normal((hkv, cap, d)).astype(np.float32) for _ in range(2))
    # rows past the last token hold what an unwritten cache may hold
    kc[:, pos + T:] = np.nan
    vc[:, pos + T:] = np.nan
    return q, kc, vc


def _f64(q, kc, vc, pos, scale):
    """Outputs and the elementwise bound of any f32 evaluation: scores off by at most
    (D + 4) 2^-24 sum |q k| scale (in exponent, so relative in the weights), and sums of at
    most L terms each rounded, in the weights' total and in the output."""
    T, hq, d = q.shape
    hkv = kc.shape[0]
    out, bound = np.empty((T, hq, d)), np.empty((T, hq, d))
    for t in range(T):
        L = pos + t + 1
        for h in range(hq):
            k, v = (c[h // (hq // hkv), :L].astype(np.float64) for c in (kc, vc))
            s = k @ q[t, h].astype(np.float64) * scale
            p = np.exp(s - s.max())
            p /= p.sum()
            out[t, h] = p @ v
            off = (d + 4) * EPS24 * (np.abs(k) @ np.abs(q[t, h].astype(np.float64))).max() * scale
            bound[t, h] = (2 * np.expm1(2 * off) + 2 * (L + 8) * EPS24) * (p @ np.abs(v))
    return out, bound


SHAPES = [  # T, pos, hq, hkv, d
    (1, 0, 32, 4, 128), (1, 15, 32, 4, 128), (1, 16, 4, 2, 64), (1, 63, 64, 4, 128), (1, 64, 32, 4, 128),
    (1, 65, 8, 8, 64), (1, 2999, 32, 4, 128), (1, 9000, 16, 1, 64), (2, 127, 32, 4, 128), (5, 1000, 6, 2, 64),
    (17, 0, 4, 2, 64), (16, 48, 48, 2, 128), (33, 7, 32, 4, 128), (260, 0, 32, 4, 64), (150, 300, 64, 4, 128),
    # a wavefront per row tile, the tiles' tokens on both sides of a split's first position
    (300, 7, 32, 4, 128), (290, 1, 32, 4, 64), (700, 5, 12, 4, 128), (400, 63, 24, 8, 64),
]


@pytest.mark.parametrize("T,pos,hq,hkv,d", SHAPES)
def test_f32_cache_attention(ctx, hip, T, pos, hq, hkv, d):
    print(f"[attn_f32] T={T} pos={pos} hq={hq} hkv={hkv} d={d}", flush=True)
    cap = pos + T + 3
    q, kc, vc = _inputs(T, pos, hq, hkv, d, cap)
    scale = float(np.float32(1.0) / np.sqrt(np.float32(d)))
    out = ctx.createBuffer(T * hq * d * 4)
    args = hip.AttnArgs(ctx.from_numpy(q), ctx.from_numpy(kc), ctx.from_numpy(vc), hip.DTYPE_F32, out, pos, T, hq, hkv, d,
                        cap, scale)
    hip.gqaAttention(ctx, args)
    got = ctx.to_numpy(out, np.float32, (T, hq, d)).astype(np.float64)
    want, bound = _f64(q, kc, vc, pos, scale)
    assert np.all(np.abs(got - want) <= bound), float(np.max(np.abs(got - want) / bound))
    hip.gqaAttention(ctx, args)
    assert np.array_equal(ctx.to_numpy(out, np.float32, (T, hq, d)), got.astype(np.float32))


@pytest.mark.parametrize("T,pos,hq,hkv,d", [(9, 20, 4, 2, 64), (150, 10, 32, 4, 128)])
def test_f32_non_finite_rows_stay_behind_the_mask(ctx, hip, T, pos, hq, hkv, d):
    """Tokens before a position with infinities or NaN in its K or V row are what they are
    without them; later tokens are not finite where the V row is not."""
    print(f"[attn_f32] non-finite T={T} pos={pos} d={d}", flush=True)
    cap = pos + T
    q, kc, vc = _inputs(T, pos, hq, hkv, d, cap)
    scale = float(np.float32(1.0) / np.sqrt(np.float32(d)))
    at = pos + T // 2

    def run():
        out = ctx.createBuffer(T * hq * d * 4)
        hip.gqaAttention(ctx, hip.AttnArgs(ctx.from_numpy(q), ctx.from_numpy(kc), ctx.from_numpy(vc), hip.DTYPE_F32, out,
                                           pos, T, hq, hkv, d, cap, scale))
        return ctx.to_numpy(out, np.float32, (T, hq, d))

    want, bound = _f64(q, kc, vc, pos, scale)
    vc[:, at, 3] = np.inf
    vc[:, at, 5] = np.nan
    kc[:, at + 1] = np.nan
    got = run()
    before = got[:at - pos]
    assert np.all(np.abs(before - want[:at - pos]) <= bound[:at - pos])
    assert np.all(np.isposinf(got[at - pos, :, 3])) and np.all(np.isnan(got[at - pos, :, 5]))
    assert np.all(np.isfinite(got[at - pos][:, [0, 1, 2, 4, 6]])) and np.all(np.isnan(got[at - pos + 1:]))


@pytest.mark.parametrize("T,pos", [(1, 40), (1, 700), (600, 300)])  # one split, several, a wavefront per row tile
@pytest.mark.parametrize("at", [0, 33, None])
def test_f32_scores_near_the_largest_float(ctx, hip, T, pos, at):
    """Scores of +-3e38 are finite: one such position takes all the weight; with every score
    at -3e38 (at None) the positions share it."""
    hq, hkv, d = 16, 4, 64
    print(f"[attn_f32] scores of 3e38 T={T} pos={pos} at={at}", flush=True)
    cap = pos + T
    q, kc, vc = _inputs(T, pos, hq, hkv, d, cap)
    q[:], kc[:] = 0, 0
    q[:, :, 5], kc[:, slice(None) if at is None else at, 5] = 1e19, 3e19 if at is not None else -3e19
    out = ctx.createBuffer(T * hq * d * 4)
    hip.gqaAttention(ctx, hip.AttnArgs(ctx.from_numpy(q), ctx.from_numpy(kc), ctx.from_numpy(vc), hip.DTYPE_F32, out, pos, T,
                                       hq, hkv, d, cap, 1.0))
    got = ctx.to_numpy(out, np.float32, (T, hq, d))
    for t in (0, T // 2, T - 1):
        L = pos + t + 1
        for h in range(hq):
            v = vc[h // (hq // hkv), :L].astype(np.float64)
            if at is not None:
                assert np.array_equal(got[t, h], v[at].astype(np.float32))
            else:  # sums of L terms, each rounded
                assert np.all(np.abs(got[t, h] - v.mean(0)) <= (L + 8) * EPS24 * np.abs(v).mean(0))


@pytest.mark.parametrize("kv,T,pos,hq,hkv,d", [
    ("f32", 1, 40, 32, 4, 128), ("f32", 3, 0, 4, 2, 64), ("f32", 2, 9, 64, 4, 128),
    ("f16", 2, 9, 32, 32, 128)] + [  # (kv rows wider than the fused f16 pre-pass takes)
    (kv, *s) for kv in ("f32", "f16") for s in ((19, 5, 6, 2, 96), (5, 3, 6, 2, 66), (2, 1, 3, 1, 256), (2, 1, 2, 1, 320))])
def test_step_equals_its_ops(ctx, hip, kv, T, pos, hq, hkv, d):
    """attentionStep on shapes without a fused attention kernel: cache rows and output equal
    rmsNorm, rope, kvAppend and gqaAttention bit for bit."""
    print(f"[step_prep] kv={kv} T={T} pos={pos} hq={hq} hkv={hkv} d={d}", flush=True)
    g = np.random.default_rng(3)
    cap = pos + T + 2
    q, k, v = (g.standard_normal((T, h, d)).astype(np.float32) for h in (hq, hkv, hkv))
    qn, kn = (1 + 0.1 * g.standard_normal(d).astype(np.float32) for _ in range(2))
    kt = np.float32 if kv == "f32" else np.float16
    kc, vc = (g.standard_normal((hkv, cap, d)).astype(kt) for _ in range(2))
    dt = hip.DTYPE_F32 if kv == "f32" else hip.DTYPE_F16
    scale, theta, eps = float(np.float32(1.0) / np.sqrt(np.float32(d))), 1e6, 1e-6
    res = []
    for fused in (True, False):
        b = {n: ctx.from_numpy(a) for n, a in dict(q=q, k=k, v=v, qn=qn, kn=kn, kc=kc, vc=vc,
                                                   p=np.arange(pos, pos + T, dtype=np.int32)).items()}
        out = ctx.createBuffer(T * hq * d * 4)
        if fused:
            hip.attentionStep(ctx, hip.AttentionStepArgs(b["q"], b["k"], b["v"], b["qn"], b["kn"], b["p"], b["kc"], b["vc"],
                                                         out, dt, pos, T, hq, hkv, d, cap, eps, theta, 1.0, scale))
        else:
            hip.rmsNorm(ctx, hip.RmsNormArgs(b["q"], b["qn"], b["q"], T * hq, d, eps))
            hip.rmsNorm(ctx, hip.RmsNormArgs(b["k"], b["kn"], b["k"], T * hkv, d, eps))
            hip.rope(ctx, hip.RopeArgs(b["q"], b["p"], T, hq, d, theta))
            hip.rope(ctx, hip.RopeArgs(b["k"], b["p"], T, hkv, d, theta))
            hip.kvAppend(ctx, hip.KvAppendArgs(b["k"], b["v"], b["kc"], b["vc"], dt, pos, T, hkv, d, cap))
            hip.gqaAttention(ctx, hip.AttnArgs(b["q"], b["kc"], b["vc"], dt, out, pos, T, hq, hkv, d, cap, scale))
        res.append([ctx.to_numpy(x, np.uint8, None) for x in (b["kc"], b["vc"], out)])
    for a, c in zip(*res):
        assert np.array_equal(a, c)


def test_f32_capture_before_any_call(hip):
    """A split launch captured on a fresh context: the graph's replays give float64's outputs
    and the eager call's bits."""
    print("[attn_f32] capture on a fresh context", flush=True)
    T, pos, hq, hkv, d = 1, 700, 32, 4, 128
    q, kc, vc = _inputs(T, pos, hq, hkv, d, pos + T)
    scale = float(np.float32(1.0) / np.sqrt(np.float32(d)))
    c = hip.Ctx.init(0)
    try:
        out, eager = (c.createBuffer(T * hq * d * 4) for _ in range(2))
        bufs = [c.from_numpy(a) for a in (q, kc, vc)]
        args, eager_args = (hip.AttnArgs(*bufs, hip.DTYPE_F32, o, pos, T, hq, hkv, d, pos + T, scale) for o in (out, eager))
        graph = c.capture(lambda: hip.gqaAttention(c, args))
        want, bound = _f64(q, kc, vc, pos, scale)
        for _ in range(3):
            c.zero(out, T * hq * d * 4)
            graph.launch()
            got = c.to_numpy(out, np.float32, (T, hq, d))
            assert np.all(np.abs(got - want) <= bound)
            hip.gqaAttention(c, eager_args)
            assert np.array_equal(got.view(np.uint32), c.to_numpy(eager, np.uint32, (T, hq, d)))
        graph.destroy()
    finally:
        c.deinit()
