"""Prefill attention whose key tiles are split over workgroups: short chunks over long
contexts, where the launch would leave compute units idle. Against float64 at the attention
gate of the f16 paths (max-abs 2e-3, cosine 0.99999), at parts that start inside a tile
pair's masked rounds, odd tile counts, part-filled q tiles, 2 parts (the smallest split) to
19 and the calls on either side of the rule's line; the allocation-free step against the
step; and the attention block against the two calls it equals."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [  # T, pos, hq, hkv, d, parts on 256 compute units
    (2, 957, 64, 4, 128, 1),     # 15 key tiles of a part-filled q tile: unsplit
    (2, 959, 64, 4, 128, 2),     # 16: two parts
    (2, 959, 16, 2, 64, 2),
    (2, 1600, 64, 4, 128, 3),
    (17, 3001, 32, 4, 128, 6),
    (33, 2047, 16, 2, 64, 8),    # two q tiles, the light one full
    (65, 5000, 5, 1, 128, 19),   # an odd count of q tiles, a head group of one
    (203, 500, 32, 4, 128, 2),
    (203, 6000, 64, 4, 128, 4),
    (128, 500, 128, 8, 128, 1),  # the parts' way through memory costs more than it saves
    (100, 700, 4, 2, 64, 3),
    (1600, 0, 4, 1, 128, 3),     # diagonal tiles in every part
    (1000, 400, 2, 1, 64, 3),
]


def _f64(q, kc, vc, pos, scale):
    T, hq, d = q.shape
    group = hq // kc.shape[0]
    out = np.empty((T, hq, d))
    L = pos + T
    mask = np.arange(L)[None, :] > pos + np.arange(T)[:, None]
    for h in range(hq):
        k, v = (c[h // group, :L].astype(np.float64) for c in (kc, vc))
        s = q[:, h].astype(np.float64) @ k.T * scale
        s[mask] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = p @ v / p.sum(1, keepdims=True)
    return out


@pytest.mark.parametrize("T,pos,hq,hkv,d,parts", SHAPES)
def test_prefill_split(ctx, hip, T, pos, hq, hkv, d, parts):
    print(f"[prefill_split] T={T} pos={pos} hq={hq} hkv={hkv} d={d}", flush=True)
    g = np.random.default_rng(T + pos)
    cap = pos + T + 5
    q = g.standard_normal((T, hq, d)).astype(np.float16).astype(np.float32) * 2
    kc, vc = (g.standard_normal((hkv, cap, d)).astype(np.float16) for _ in range(2))
    kc[:, pos + T:] = np.nan
    vc[:, pos + T:] = np.nan
    scale = float(np.float32(1.0) / np.sqrt(np.float32(d)))
    want = _f64(q, kc, vc, pos, scale)
    out = ctx.createBuffer(T * hq * d * 4)
    args = hip.AttnArgs(ctx.from_numpy(q), ctx.from_numpy(kc), ctx.from_numpy(vc), hip.DTYPE_F16, out, pos, T, hq, hkv, d,
                        cap, scale)
    ctx.set_kernel_timing(True)
    hip.gqaAttention(ctx, args)
    assert hip.LIB.ds5_index_prefill_splits(256, pos, T, hq, hkv, d) == parts
    assert ctx.kernel_time("prefill_merge_kernel")[0] == (parts > 1)  # one merge
    ctx.set_kernel_timing(False)
    got = ctx.to_numpy(out, np.float32, (T, hq, d)).astype(np.float64)
    err = np.abs(got - want).max()
    cos = (got * want).sum() / np.sqrt((got ** 2).sum() * (want ** 2).sum())
    print(f"  max-abs {err:.2e}, 1 - cosine {1 - cos:.2e}", flush=True)
    assert err <= 2e-3 and cos >= 0.99999


@pytest.mark.parametrize("kv", ["f16", "f32"])
def test_split_noalloc_is_the_step(ctx, hip, kv):
    T, pos, hq, hkv, d = 150, 3000, 64, 4, 128
    cap = pos + T
    g = np.random.default_rng(5)
    q, k, v = (g.standard_normal((T, h, d)).astype(np.float32) for h in (hq, hkv, hkv))
    dt = np.float16 if kv == "f16" else np.float32
    kc, vc = (g.standard_normal((hkv, cap, d)).astype(dt) for _ in range(2))
    qn, kn = (np.ones(d, np.float32) for _ in range(2))
    outs = []
    for fn in (hip.attentionStep, hip.attentionStepNoAlloc, hip.attentionStep):
        bufs = [ctx.from_numpy(a) for a in (q, k, v, qn, kn, np.arange(pos, cap, dtype=np.int32), kc, vc)]
        out = ctx.createBuffer(T * hq * d * 4)
        fn(ctx, hip.AttentionStepArgs(*bufs, out, hip.DTYPE_F16 if kv == "f16" else hip.DTYPE_F32, pos, T, hq, hkv, d, cap,
                                      1e-6, 1e6, 1.0, float(np.float32(d) ** np.float32(-0.5))))
        outs.append(ctx.to_numpy(out, np.uint32, (T, hq, d)))
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])


def _block_inputs(oracle, T, pos, hq, hkv, hidden):
    g = np.random.default_rng(9)
    d, cap = 128, pos + T
    x = g.standard_normal((T, hidden)).astype(np.float32)
    w = [oracle.q8_0_quantize(g.standard_normal((h * d, hidden)).astype(np.float32) * np.float32(0.05))
         for h in (hq, hkv, hkv)]
    kc, vc = (g.standard_normal((hkv, cap, d)).astype(np.float16) for _ in range(2))
    return x, w, kc, vc


@pytest.mark.parametrize("T,pos,hq,hkv,merges", [(100, 3000, 32, 4, 1), (17, 1500, 8, 2, 1), (40, 64, 8, 2, 0)])
def test_split_block_is_the_two_calls_also_captured(hip, oracle, T, pos, hq, hkv, merges):
    """attentionBlock on a launch split over its keys equals matmulGroup and attentionStep, bit
    for bit, eagerly and captured: the two calls on a context of their own, the block captured
    where only the same block at position 0 (nothing split there) ran before it."""
    print(f"[split_block] T={T} pos={pos} hq={hq} hkv={hkv}", flush=True)
    d, hidden = 128, 512
    x, w, kc, vc = _block_inputs(oracle, T, pos, hq, hkv, hidden)
    scale = float(np.float32(1.0) / np.sqrt(np.float32(d)))

    def args(c, at):
        bufs = [c.createBuffer(T * h * d * 4) for h in (hq, hkv, hkv)]
        bufs += [c.from_numpy(a) for a in (np.ones(d, np.float32), np.ones(d, np.float32),
                                           np.arange(at, at + T, dtype=np.int32), kc, vc)]
        return hip.AttentionStepArgs(*bufs, c.createBuffer(T * hq * d * 4), hip.DTYPE_F16, at, T, hq, hkv, d, pos + T, 1e-6,
                                     1e6, 1.0, scale)

    def results(c, a):
        return [c.to_numpy(b, np.uint8, None) for b in (a.out, a.k_cache, a.v_cache)]

    c = hip.Ctx.init(0)
    try:  # the two calls
        xb, wb, a = c.from_numpy(x), [c.from_numpy(v) for v in w], args(c, pos)
        hip.matmulGroup(c, hip.MatmulGroupArgs.of(xb, hip.DTYPE_Q8_0, T, hidden, [(wb[0], a.q, hq * d), (wb[1], a.k, hkv * d),
                                                                                 (wb[2], a.v, hkv * d)]))
        c.set_kernel_timing(True)
        hip.attentionStep(c, a)
        assert c.kernel_time("prefill_merge_kernel")[0] == merges
        c.set_kernel_timing(False)
        want = results(c, a)
    finally:
        c.deinit()
    c = hip.Ctx.init(0)
    try:
        xb, wb = c.from_numpy(x), [c.from_numpy(v) for v in w]
        block = lambda a: hip.attentionBlock(c, hip.AttentionBlockArgs(xb, *wb, hip.DTYPE_Q8_0, hidden, a))  # noqa: E731
        block(args(c, 0))
        a, eager = args(c, pos), args(c, pos)
        graph = c.capture(lambda: block(a))
        for _ in range(3):
            c.zero(a.out, T * hq * d * 4)
            graph.launch()
            c.submit()
            assert all(np.array_equal(p, q) for p, q in zip(results(c, a), want))
            block(eager)
            assert all(np.array_equal(p, q) for p, q in zip(results(c, eager), want))
        graph.destroy()
    finally:
        c.deinit()
