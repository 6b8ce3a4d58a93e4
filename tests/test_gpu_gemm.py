"""The Q8_0 matrix-core products at the edges of their tiles: rows around 32, 64 and 128, ragged
columns, odd block counts, both tile heights (few and many workgroups), with and without a
residual, against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def q8_rows(g, n, k):
    """Q8_0 rows [n, k / 32 * 34] with scales over two decades, and their exact f64 values."""
    w = np.empty((n, k // 32, 34), np.uint8)
    s = (10.0 ** g.uniform(-3, -1, (n, k // 32))).astype(np.float16)
    q = g.integers(-127, 128, (n, k // 32, 32)).astype(np.int8)
    w[:, :, :2] = s[..., None].view(np.uint8).reshape(n, k // 32, 2)
    w[:, :, 2:] = q.view(np.uint8)
    return w.reshape(n, -1), (s.astype(np.float64)[..., None] * q).reshape(n, k)


def bound(x, w, extra=0.0):
    """x as hi + lo f16 of the row's power of two (2^-22 of the row's largest element at worst,
    2^-21 with both roundings), f32 sums of 32 exact products per block and of the blocks."""
    k = x.shape[1]
    xa = np.abs(x) + 2.0 ** -21 * np.abs(x).max(1, keepdims=True)
    return (2.0 ** -21 + (32 + k // 32 + 8) * 2.0 ** -24) * (xa @ np.abs(w).T) + \
        2.0 ** -21 * np.abs(x).max(1, keepdims=True) * np.abs(w).sum(1)[None] + extra


CASES = [(16, 128, 64), (17, 1, 32), (31, 127, 96), (33, 300, 2048), (63, 512, 160), (64, 129, 4096), (65, 4096, 256),
         (127, 40, 224), (128, 256, 32 * 65), (129, 130, 2048), (200, 20000, 64), (300, 12000, 96),
         # blocks split over groups: one without a block (nine and three blocks), one with a single one;
         # 32 and 128 columns a workgroup; the last split tile counts and the first unsplit ones
         (16, 5, 32), (33, 300, 96), (20, 40, 288), (128, 4096, 288), (128, 4097, 288), (65, 10880, 320), (31, 32700, 288),
         (128, 8192, 288), (128, 8193, 288), (64, 8192, 96), (64, 8193, 96), (32, 32800, 288)]


@pytest.mark.parametrize("m,n,k", CASES)
@pytest.mark.parametrize("residual", [False, True], ids=["matmul", "matmul_add"])
def test_gemm_tile_edges(ctx, hip, m, n, k, residual):
    print(f"[gemm] m={m} n={n} k={k} residual={residual}", flush=True)
    g = np.random.default_rng(m * 7 + n)
    x = (g.standard_normal((m, k)) * 10.0 ** g.uniform(-4, 4, (m, 1))).astype(np.float32)
    x[m // 2] = 0.0
    wb, w = q8_rows(g, n, k)
    pad = np.concatenate([wb.reshape(-1), np.zeros(4, np.uint8)])
    res = g.standard_normal((m, n)).astype(np.float32)
    xb, wbuf, out = ctx.from_numpy(x), ctx.from_numpy(pad), ctx.from_numpy(np.full((m, n), 7e30, np.float32))
    if residual:
        hip.matmulAdd(ctx, hip.MatmulAddArgs(xb, wbuf, hip.DTYPE_Q8_0, ctx.from_numpy(res), out, m, n, k))
    else:
        hip.matmul(ctx, hip.MatmulArgs(xb, wbuf, hip.DTYPE_Q8_0, out, m, n, k))
    got = ctx.to_numpy(out, np.float32, (m, n)).astype(np.float64)
    want = x.astype(np.float64) @ w.T + (res if residual else 0.0)
    lim = bound(x.astype(np.float64), w, 2.0 ** -23 * np.abs(want) if residual else 0.0)
    assert np.all(np.abs(got - want) <= lim + 1e-30), float(np.max(np.abs(got - want) / (lim + 1e-30)))


@pytest.mark.parametrize("m", [64, 65, 128])
def test_mixed_group_is_its_products(ctx, hip, m):
    """A group whose products take both matrix-core forms (from 65 tokens: 16384 columns unsplit,
    the others split): each entry's bits are its own matmul's, x is split once."""
    print(f"[gemm] mixed group m={m}", flush=True)
    k, ns = 512, (130, 16384, 512)
    g = np.random.default_rng(m)
    xb = ctx.from_numpy(g.standard_normal((m, k)).astype(np.float32))
    wb = [ctx.from_numpy(np.concatenate([q8_rows(g, n, k)[0].reshape(-1), np.zeros(4, np.uint8)])) for n in ns]
    got, want = ([ctx.createBuffer(m * n * 4) for n in ns] for _ in range(2))
    ctx.set_kernel_timing(True)
    hip.matmulGroup(ctx, hip.MatmulGroupArgs.of(xb, hip.DTYPE_Q8_0, m, k, list(zip(wb, got, ns))))
    ctx.submit()
    launches = [ctx.kernel_time(name)[0] for name in ("matmul_x_split_kernel", "matmul_q8_mfma_kernel")]
    ctx.set_kernel_timing(False)
    assert launches == [1, 2 if m > 64 else 1]
    for w, a, b, n in zip(wb, got, want, ns):
        hip.matmul(ctx, hip.MatmulArgs(xb, w, hip.DTYPE_Q8_0, b, m, n, k))
        assert np.array_equal(ctx.to_numpy(a, np.uint32, (m, n)), ctx.to_numpy(b, np.uint32, (m, n)))


@pytest.mark.parametrize("T,E,K,dim,ffn,grouped", [
    (31, 16, 1, 256, 96, 0), (32, 16, 1, 512, 64, 1), (24, 96, 8, 256, 96, 1), (23, 96, 8, 256, 96, 0), (22, 64, 4, 256, 64, 0),
    (60, 24, 4, 2048, 768, 1)])
def test_grouped_experts_few_pairs(ctx, hip, T, E, K, dim, ffn, grouped):
    """Few pairs per expert, on both sides of the two per expert from which the experts run grouped
    (below, x and h stay in f32), against float64, twice: rows of one expert land in any order."""
    print(f"[moe] few pairs T={T} E={E} K={K}", flush=True)
    g = np.random.default_rng(T)
    (G, Gf), (U, Uf), (D, Df) = (q8_rows(g, E * a, b) for a, b in ((ffn, dim), (ffn, dim), (dim, ffn)))
    x = (0.05 * g.standard_normal((T, dim))).astype(np.float32)
    pairs = np.zeros(T * K, hip.PAIR_DTYPE)
    pairs["token"] = np.repeat(np.arange(T), K)
    pairs["expert"] = g.integers(0, E, T * K)
    pairs["weight"] = g.random(T * K).astype(np.float32)
    want, lim = np.zeros((T, dim)), np.zeros((T, dim))
    for t, e, w in pairs:
        Ge, Ue, De = (v.reshape(E, -1, v.shape[1])[e] for v in (Gf, Uf, Df))
        xd = x[t:t + 1].astype(np.float64)
        a, u = xd @ Ge.T, xd @ Ue.T
        da, du = bound(xd, Ge), bound(xd, Ue)
        h = a / (1 + np.exp(-a)) * u
        # |silu'| <= 1.1; the exponential and the division within 4 ulp
        dh = 1.1 * da * np.abs(u) + np.abs(a) * du + 1.1 * da * du + 4 * 2.0 ** -23 * np.abs(h)
        want[t] += w * (h @ De.T)[0]
        lim[t] += w * (bound(h, De) + (dh + 2.0 ** -21 * dh.max()) @ np.abs(De).T)[0] + 2.0 ** -22 * np.abs(w * (h @ De.T)[0])
    lim += (K + 2) * 2.0 ** -23 * np.abs(want)
    bufs = [ctx.from_numpy(np.concatenate([v.reshape(-1), np.zeros(4, np.uint8)])) for v in (G, U, D)]
    runs = []
    ctx.set_kernel_timing(True)
    for _ in range(2):
        out = ctx.createBuffer(T * dim * 4)
        hip.expertMlpSwiglu(ctx, ctx.from_numpy(x), *bufs, hip.DTYPE_Q8_0, pairs, out, T, dim, ffn, E)
        runs.append(ctx.to_numpy(out, np.float32, (T, dim)))
    ctx.submit()
    sorts = ctx.kernel_time("moe_sort_kernel")[0]
    ctx.set_kernel_timing(False)
    assert sorts == 2 * grouped
    assert np.all(np.abs(runs[0] - want) <= lim), float(np.max(np.abs(runs[0] - want) / lim))
    assert np.array_equal(runs[0], runs[1])


@pytest.mark.parametrize("T,E", [(1024, 16), (1025, 16), (3001, 24), (66000, 40)])
def test_grouped_experts_sort_slices(ctx, hip, T, E):
    """Pair counts at the edges of the sort's slices (1024 pairs each, then 64 of equal size), one
    pair a token, half of them on one expert: every token's row against float64, twice."""
    print(f"[moe] sort slices T={T} E={E}", flush=True)
    dim, ffn = 256, 64
    g = np.random.default_rng(T)
    (G, Gf), (U, Uf), (D, Df) = (q8_rows(g, E * a, b) for a, b in ((ffn, dim), (ffn, dim), (dim, ffn)))
    x = (0.05 * g.standard_normal((T, dim))).astype(np.float32)
    pairs = np.zeros(T, hip.PAIR_DTYPE)
    pairs["token"] = g.permutation(T)
    pairs["expert"] = np.where(g.random(T) < 0.5, 3, g.integers(0, E, T))
    pairs["weight"] = g.random(T).astype(np.float32)
    bufs = [ctx.from_numpy(np.concatenate([v.reshape(-1), np.zeros(4, np.uint8)])) for v in (G, U, D)]
    xb, runs = ctx.from_numpy(x), []
    for _ in range(2):
        out = ctx.from_numpy(np.zeros((T, dim), np.float32))
        hip.expertMlpSwiglu(ctx, xb, *bufs, hip.DTYPE_Q8_0, pairs, out, T, dim, ffn, E)
        runs.append(ctx.to_numpy(out, np.float32, (T, dim)))
    assert np.array_equal(runs[0], runs[1])
    for e in range(E):
        p = pairs[pairs["expert"] == e]
        tok, w = p["token"], p["weight"][:, None].astype(np.float64)
        Ge, Ue, De = (v.reshape(E, -1, v.shape[1])[e] for v in (Gf, Uf, Df))
        xd = x[tok].astype(np.float64)
        a, u = xd @ Ge.T, xd @ Ue.T
        da, du = bound(xd, Ge), bound(xd, Ue)
        h = a / (1 + np.exp(-a)) * u
        # the bound of test_grouped_experts_few_pairs
        dh = 1.1 * da * np.abs(u) + np.abs(a) * du + 1.1 * da * du + 4 * 2.0 ** -23 * np.abs(h)
        want = w * (h @ De.T)
        lim = w * (bound(h, De) + (dh + 2.0 ** -21 * dh.max(1, keepdims=True)) @ np.abs(De).T) + 2.0 ** -20 * np.abs(want)
        assert np.all(np.abs(runs[0][tok] - want) <= lim), float(np.max(np.abs(runs[0][tok] - want) / lim))
