"""Router logits in token x expert tiles: every logit is dotRow's serial sum, so ids and
weights equal, bit for bit, those of single tokens, at the edges of a chunk of 256 elements
and of the groups inside it, of a tile, and at the fewest tokens that run in tiles, which are
fewer for a large router; on both sides of that line the launch counts are the rule's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,dim,E,dt,tiled", [
    (32, 252, 16, "f32", 1), (33, 256, 17, "f16", 1), (33, 260, 33, "f32", 1), (32, 768, 5, "f32", 1), (257, 516, 1100, "f16", 1),
    (289, 512, 1000, "f32", 1), (24, 768, 299, "f32", 1), (25, 512, 430, "f16", 1), (24, 768, 298, "f32", 0),
    (31, 1024, 32, "f32", 0), (23, 2048, 128, "f32", 0)])
def test_tile_edges(ctx, hip, T, dim, E, dt, tiled):
    print(f"[router_tile] T={T} dim={dim} E={E} {dt}", flush=True)
    g = np.random.default_rng(T * dim)
    x = g.standard_normal((T, dim)).astype(np.float32)
    w = (g.standard_normal((E, dim)) * 0.1).astype(np.float32 if dt == "f32" else np.float16)
    wdt = hip.DTYPE_F32 if dt == "f32" else hip.DTYPE_F16
    xb, wb = ctx.from_numpy(x), ctx.from_numpy(w)
    K = min(8, E)
    ctx.set_kernel_timing(True)
    try:
        ids, wts = hip.routerTopK(ctx, xb, wb, wdt, T, dim, E, K, False)
        assert ctx.kernel_time("router_logits_tile_kernel")[0] == tiled
    finally:
        ctx.set_kernel_timing(False)
    for t in range(T):
        i1, w1 = hip.routerTopK(ctx, hip.Buf(xb.handle, xb.offset + t * dim * 4, dim * 4), wb, wdt, 1, dim, E, K, False)
        assert np.array_equal(ids[t], i1[0])
        assert np.array_equal(wts[t].view(np.uint32), w1[0].view(np.uint32))
