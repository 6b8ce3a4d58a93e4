"""The calls whose speed this repository keeps: what a host of the engine asks of the gfx950
provider, from a one-token step of a tiny model to a 2048-token prompt, each through the public
entry points of `qw3_amd.hip` / `qw3_amd.engine` with the inputs, weights and caches such a host
holds.

Shapes: Qwen3-30B-A3B (hidden 2048, 32 q / 4 kv heads of 128, 128 experts top 8, expert width
768, Q8_0 weights, f32 router and norms), the 64 q / 4 kv attention of Qwen3-235B-A22B, the
synthetic tiny Qwen3-MoE of the tests, and a generic small model between them. Both cache types
count: f32 is the engine's default, f16 what a long context is run with.

Kinds of case (`case["kind"]`):
  step    attentionStep of one new token, `layers` layers with caches of their own (f16)
  block   attentionBlock: attn_norm, q/k/v projections and the attention step of T tokens at pos
  layer   a whole layer in the engine's fused order: attentionBlock, matmulAdd, moe
  paged   pagedDecode: one new token for each of `seqs` sequences over a paged pool
  moe     the MoE block of T tokens: ffn_norm, router, experts, residual
  linear  matmul of a Q8_0 weight: the head, or a projection of a few tokens
  engine  Engine.forward of a whole model, embedding to logits
"""
import math

import numpy as np
import torch

import qw3_amd.hip as H
from qw3_amd import engine as E

EPS = 1e-6
THETA = 1e6
DEV = "cuda"

# what a model of the tests' size and a generic one between it and the full shapes are made of
MODELS = {
    "tiny": dict(n_layers=4, hidden_dim=256, n_q_heads=4, n_kv_heads=2, head_dim=64, n_experts=8, top_k=4,
                 expert_ffn_dim=128, vocab_size=512, rms_eps=EPS, rope_theta=THETA, norm_topk_prob=True, max_ctx=512),
    "small": dict(n_layers=3, hidden_dim=1024, n_q_heads=16, n_kv_heads=4, head_dim=128, n_experts=32, top_k=4,
                  expert_ffn_dim=512, vocab_size=16384, rms_eps=EPS, rope_theta=THETA, norm_topk_prob=True,
                  max_ctx=4096),
}


def listed():
    return [
        # the tests' model in a chat loop: the smallest call, a token at a time over the default f32 cache
        dict(name="tiny model, one token", kind="engine", model="tiny", n=1, pos=17, kv="f32"),
        # a short prompt through a small model, its logits back on the host
        dict(name="small model, prompt", kind="engine", model="small", n=61, pos=0, kv="f32"),
        # the attention of a decode step late in an 8K context, layer after layer
        dict(name="decode attention 8K", kind="step", layers=12, pos=8191, hq=32, hkv=4, d=128),
        # the attention block of a decode step over the default cache
        dict(name="decode block, f32 cache", kind="block", T=1, pos=2999, hq=32, hkv=4, d=128, hidden=2048, kv="f32"),
        # one layer of a decode step, all of it
        dict(name="decode layer", kind="layer", T=1, pos=4095, kv="f16"),
        # a serving batch: 32 sequences of very different lengths
        dict(name="paged decode, 32 seqs", kind="paged", seqs=32, lo=512, hi=16384, page=16, hq=32, hkv=4, d=128),
        # a long prompt's attention block
        dict(name="prefill block 2048", kind="block", T=2048, pos=0, hq=32, hkv=4, d=128, hidden=2048, kv="f16"),
        # the next user turn of a long chat: a ragged chunk after 6000 cached tokens, wide heads
        dict(name="chunk of 203 at 6000", kind="block", T=203, pos=6000, hq=64, hkv=4, d=128, hidden=4096, kv="f16"),
        # a prompt over the default cache
        dict(name="prefill block 500, f32", kind="block", T=500, pos=0, hq=32, hkv=4, d=128, hidden=2048, kv="f32"),
        # the experts of a long prompt
        dict(name="moe 2048", kind="moe", T=2048),
        # the experts of a short question
        dict(name="moe 24", kind="moe", T=24),
        # the head of a decode step
        dict(name="head, one token", kind="linear", m=1, n=65536, k=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["engine", "step", "block", "block", "block", "layer", "paged", "moe", "moe", "linear"])
    if kind == "engine":
        n = _log_int(rng, 1, 61)
        return dict(kind=kind, model=rng.choice(["tiny", "small"]), n=n, pos=rng.randint(1, 40), kv=rng.choice(["f32", "f16"]))
    if kind == "step":
        hq = rng.choice([32, 64])
        return dict(kind=kind, layers=rng.randint(1, 12), pos=_log_int(rng, 15, 16383), hq=hq, hkv=4, d=128)
    if kind == "block":
        hq, hidden = rng.choice([(32, 2048), (64, 4096)])
        kv = rng.choice(["f16", "f16", "f32"])
        T = rng.choice([1, _log_int(rng, 2, 1500)])
        pos = rng.choice([0, _log_int(rng, 16, 8000)])
        if kv == "f32":  # no dearer than the listed f32 prompt
            T = min(T, 250)
            pos = min(pos, 100000 // (T * (hq // 32)))
        return dict(kind=kind, T=T, pos=pos, hq=hq, hkv=4, d=128, hidden=hidden, kv=kv)
    if kind == "layer":
        return dict(kind=kind, T=_log_int(rng, 1, 64), pos=_log_int(rng, 16, 8000), kv="f16")
    if kind == "paged":
        lo = _log_int(rng, 16, 2000)
        return dict(kind=kind, seqs=_log_int(rng, 1, 48), lo=lo, hi=lo * rng.randint(1, 8), page=rng.choice([16, 32, 64]),
                    hq=rng.choice([32, 64]), hkv=4, d=128)
    if kind == "moe":
        return dict(kind=kind, T=_log_int(rng, 1, 1800))
    n, k = rng.choice([(65536, 2048), (2048, 4096), (4096, 2048), (512, 256), (30011, 1024)])
    return dict(kind=kind, m=_log_int(rng, 1, 200), n=n, k=k)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
_ctx = None


def _context():
    """One context per process, as an engine host keeps."""
    global _ctx
    if _ctx is None:
        _ctx = H.Ctx.init(0)
    return _ctx


class _Make:
    """Seeded device tensors: normals, and Q8_0 weights quantised from normals."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device=DEV) * std + mean).to(dtype)

    def q8(self, rows, k, std=None):
        """Q8_0 rows [rows, k / 32 * 34] of N(0, std) weights (default 1 / sqrt(k)): per 32 elements an
        f16 scale of max / 127, then the rounded int8."""
        out = torch.empty(rows, k // 32, 34, dtype=torch.uint8, device=DEV)
        step = max(1, (1 << 26) // k)
        for r in range(0, rows, step):
            w = self.normal(min(step, rows - r), k // 32, 32, std=std or k ** -0.5)
            s = (w.abs().amax(2, keepdim=True) / 127).half()
            q = torch.clamp(torch.round(w / s.float().clamp_min(1e-8)), -127, 127).to(torch.int8)
            out[r:r + step, :, :2] = s.view(torch.uint8)
            out[r:r + step, :, 2:] = q.view(torch.uint8)
        return out.view(rows, k // 32 * 34)

    def norm_w(self, n):
        return self.normal(n, std=0.02, mean=1.0)

    def cache(self, kv, layers, hkv, cap, d, filled):
        """K or V caches [layers, hkv, cap, d] with `filled` cached positions (zero after them)."""
        c = torch.zeros(layers, hkv, cap, d, dtype=_kv_type(kv), device=DEV)
        for li in range(layers):
            c[li, :, :filled] = self.normal(hkv, filled, d).to(c.dtype)
        return c


def _kv_type(kv):
    return torch.float16 if kv == "f16" else torch.float32


def _kv_dtype(kv):
    return H.DTYPE_F16 if kv == "f16" else H.DTYPE_F32


def _buf(t):
    """A view of a device tensor as the C ABI takes it."""
    return H.Buf(t.data_ptr(), 0, t.numel() * t.element_size()) if t is not None else H.Buf()


def _capacity(n):
    """The context capacity a host sets for n positions."""
    return max(32, 1 << (n - 1).bit_length())


def _scale(d):
    return float(np.float32(1.0) / np.sqrt(np.float32(d)))


def _zeros(*shape):
    return torch.zeros(*shape, device=DEV)


def _attention_inputs(m, c, T, pos, hq, hkv, d, hidden, kv):
    cap = _capacity(pos + T)
    return dict(x=m.normal(T, hidden), an=m.norm_w(hidden), wq=m.q8(hq * d, hidden), wk=m.q8(hkv * d, hidden),
                wv=m.q8(hkv * d, hidden), qn=m.norm_w(d), kn=m.norm_w(d),
                positions=torch.arange(pos, pos + T, dtype=torch.int32, device=DEV),
                kc=m.cache(kv, 1, hkv, cap, d, pos)[0], vc=m.cache(kv, 1, hkv, cap, d, pos)[0])


def _block_args(t, s, T, pos, hq, hkv, d, hidden, kv):
    step = H.AttentionStepArgs(_buf(s["q"]), _buf(s["k"]), _buf(s["v"]), _buf(t["qn"]), _buf(t["kn"]), _buf(t["positions"]),
                               _buf(t["kc"]), _buf(t["vc"]), _buf(s["attn"]), _kv_dtype(kv), pos, T, hq, hkv, d,
                               t["kc"].shape[1], EPS, THETA, 1.0, _scale(d))
    return H.AttentionBlockArgs(_buf(t["x"]), _buf(t["wq"]), _buf(t["wk"]), _buf(t["wv"]), H.DTYPE_Q8_0, hidden, step,
                                _buf(t["an"]), EPS)


MOE = dict(dim=2048, ffn=768, E=128, K=8)  # Qwen3-30B-A3B


def _moe_inputs(m):
    D, F, X = MOE["dim"], MOE["ffn"], MOE["E"]
    return dict(fn=m.norm_w(D), router=m.normal(X, D, std=0.05), gate=m.q8(X * F, D), up=m.q8(X * F, D), down=m.q8(X * D, F))


def _moe_args(t, x, out, T):
    return H.MoeArgs(_buf(x), _buf(t["router"]), H.DTYPE_F32, _buf(t["gate"]), _buf(t["up"]), _buf(t["down"]), H.DTYPE_Q8_0,
                     _buf(out), H.Buf(), H.Buf(), T, MOE["dim"], MOE["ffn"], MOE["E"], MOE["K"], 1, _buf(x), _buf(t["fn"]), EPS)


LAYER = dict(hq=32, hkv=4, d=128, hidden=2048)


def _paged_layout(c, seed):
    g = np.random.default_rng([seed, c["seqs"], c["lo"], c["hi"]])
    lens = g.integers(c["lo"], c["hi"] + 1, c["seqs"])
    pages, most = -(-lens // c["page"]), -(-c["hi"] // c["page"])
    table = np.zeros((c["seqs"], most), np.int32)
    # a server's pool: room for every sequence at its longest, pages handed out in any order
    perm, at = g.permutation(c["seqs"] * most).astype(np.int32), 0
    for b, n in enumerate(pages):
        table[b, :n] = perm[at:at + n]
        at += n
    return lens.astype(np.int32), table, c["seqs"] * most


def _model_tensors(model, seed):
    """GGUF-named weights of a model on the device: Q8_0 matrices, f32 norms and routers."""
    c, m = MODELS[model], _Make(seed)
    hid, hq, hkv, hd, X, F = (c[k] for k in ("hidden_dim", "n_q_heads", "n_kv_heads", "head_dim", "n_experts",
                                             "expert_ffn_dim"))
    w = {"token_embd.weight": m.q8(c["vocab_size"], hid, std=1.0), "output_norm.weight": m.norm_w(hid),
         "output.weight": m.q8(c["vocab_size"], hid)}
    for li in range(c["n_layers"]):
        b = f"blk.{li}."
        w[b + "attn_norm.weight"], w[b + "ffn_norm.weight"] = m.norm_w(hid), m.norm_w(hid)
        w[b + "attn_q_norm.weight"], w[b + "attn_k_norm.weight"] = m.norm_w(hd), m.norm_w(hd)
        w[b + "attn_q.weight"], w[b + "attn_k.weight"], w[b + "attn_v.weight"] = (
            m.q8(n * hd, hid) for n in (hq, hkv, hkv))
        w[b + "attn_output.weight"] = m.q8(hid, hq * hd)
        w[b + "ffn_gate_inp.weight"] = m.normal(X, hid, std=0.1)
        w[b + "ffn_gate_exps.weight"], w[b + "ffn_up_exps.weight"] = m.q8(X * F, hid), m.q8(X * F, hid)
        w[b + "ffn_down_exps.weight"] = m.q8(X * hid, F)
    toks = torch.randint(0, c["vocab_size"], (128,), generator=m.g, device=DEV).tolist()
    return w, toks


class _Model:
    """An engine with a context of its own, `pos` tokens into a conversation; frees the context with it."""

    def __init__(self, case, seed):
        cfg = MODELS[case["model"]]
        w, toks = _model_tensors(case["model"], seed)
        self.ctx = H.Ctx.init(0)
        weights = E.Weights(self.ctx, {k: v.cpu().numpy() for k, v in w.items()}, cfg)
        self.engine = E.Engine(self.ctx, weights, max_batch=64, context_capacity=128, kv_dtype=_kv_dtype(case["kv"]),
                               fused=True)
        self.pos, self.toks = case["pos"], toks[case["pos"]:case["pos"] + case["n"]]
        if self.pos:
            self.engine.forward(toks[:self.pos], want_logits=False)

    def __del__(self):
        self.ctx.deinit()


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "engine":
        return dict(kind=kind, model=_Model(case, seed))
    m = _Make(seed)
    ctx = _context()
    s = dict(kind=kind, ctx=ctx)
    if kind == "step":
        L, pos, hq, hkv, d = (c[k] for k in ("layers", "pos", "hq", "hkv", "d"))
        cap = _capacity(pos + 1)
        t = dict(q=m.normal(L, 1, hq, d), k=m.normal(L, 1, hkv, d), v=m.normal(L, 1, hkv, d), qn=m.norm_w(d), kn=m.norm_w(d),
                 positions=torch.tensor([pos], dtype=torch.int32, device=DEV), kc=m.cache("f16", L, hkv, cap, d, pos),
                 vc=m.cache("f16", L, hkv, cap, d, pos))
        s["attn"] = _zeros(L, 1, hq * d)
        s["args"] = [H.AttentionStepArgs(_buf(t["q"][i]), _buf(t["k"][i]), _buf(t["v"][i]), _buf(t["qn"]), _buf(t["kn"]),
                                         _buf(t["positions"]), _buf(t["kc"][i]), _buf(t["vc"][i]), _buf(s["attn"][i]),
                                         H.DTYPE_F16, pos, 1, hq, hkv, d, cap, EPS, THETA, 1.0, _scale(d)) for i in range(L)]
    elif kind in ("block", "layer"):
        shape = LAYER if kind == "layer" else {k: c[k] for k in ("hq", "hkv", "d", "hidden")}
        hq, hkv, d, T = shape["hq"], shape["hkv"], shape["d"], c["T"]
        t = _attention_inputs(m, c, T, c["pos"], hq, hkv, d, shape["hidden"], c["kv"])
        s.update(q=_zeros(T, hq, d), k=_zeros(T, hkv, d), v=_zeros(T, hkv, d), attn=_zeros(T, hq * d))
        s["block"] = _block_args(t, s, T, c["pos"], hq, hkv, d, shape["hidden"], c["kv"])
        if kind == "layer":
            t["wo"] = m.q8(shape["hidden"], hq * d)
            t.update(_moe_inputs(m))
            s.update(mid=_zeros(T, shape["hidden"]), out=_zeros(T, shape["hidden"]))
            s["wo"] = H.MatmulAddArgs(_buf(s["attn"]), _buf(t["wo"]), H.DTYPE_Q8_0, _buf(t["x"]), _buf(s["mid"]), T,
                                      shape["hidden"], hq * d)
            s["moe"] = _moe_args(t, s["mid"], s["out"], T)
    elif kind == "paged":
        lens, table, n_pages = _paged_layout(c, seed)
        B, hq, hkv, d = c["seqs"], c["hq"], c["hkv"], c["d"]
        t = dict(q=m.normal(B, hq, d), k=m.normal(B, hkv, d), v=m.normal(B, hkv, d), qn=m.norm_w(d), kn=m.norm_w(d),
                 kc=m.normal(hkv, n_pages * c["page"], d, dtype=torch.float16),
                 vc=m.normal(hkv, n_pages * c["page"], d, dtype=torch.float16),
                 table=torch.from_numpy(table).to(DEV), lens=torch.from_numpy(lens).to(DEV))
        s["attn"] = _zeros(B, hq * d)
        s["args"] = H.PagedDecodeArgs(_buf(t["q"]), _buf(t["k"]), _buf(t["v"]), _buf(t["qn"]), _buf(t["kn"]), _buf(t["kc"]),
                                      _buf(t["vc"]), _buf(t["table"]), _buf(t["lens"]), _buf(s["attn"]), B, hq, hkv, d,
                                      c["page"], n_pages, table.shape[1], int(lens.max()), EPS, THETA, 1.0, _scale(d))
    elif kind == "moe":
        t = dict(x=m.normal(c["T"], MOE["dim"]), **_moe_inputs(m))
        s["out"] = _zeros(c["T"], MOE["dim"])
        s["moe"] = _moe_args(t, t["x"], s["out"], c["T"])
    else:
        t = dict(x=m.normal(c["m"], c["k"]), w=m.q8(c["n"], c["k"]))
        s["out"] = _zeros(c["m"], c["n"])
        s["args"] = H.MatmulArgs(_buf(t["x"]), _buf(t["w"]), H.DTYPE_Q8_0, _buf(s["out"]), c["m"], c["n"], c["k"])
    s["t"] = t
    torch.cuda.synchronize()  # the inputs were made on torch's stream, the calls run on the context's
    return s


def run(state):
    s, kind = state, state["kind"]
    if kind == "engine":
        m = s["model"]
        m.engine.pos = m.pos
        return m.engine.forward(m.toks)
    ctx, t = s["ctx"], s["t"]
    if kind == "step":
        for a in s["args"]:
            H.attentionStep(ctx, a)
    elif kind == "paged":
        H.pagedDecode(ctx, s["args"])
    elif kind == "linear":
        H.matmul(ctx, s["args"])
        return s["out"]
    elif kind == "moe":
        H.moe(ctx, s["moe"])
        return s["out"]
    else:
        H.attentionBlock(ctx, s["block"])
        if kind == "layer":
            H.matmulAdd(ctx, s["wo"])
            H.moe(ctx, s["moe"])
            return dict(out=s["out"], kc=t["kc"], vc=t["vc"])
    return dict(attn=s["attn"], kc=t["kc"], vc=t["vc"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _q8_bytes(rows, k):
    return rows * (k // 32) * 34


def _attention_work(T, pos, hq, hkv, d, es):
    """The attention step: q, new k/v and out in f32, T rows appended, every attended row read once."""
    rows = pos + T
    pairs = T * pos + T * (T + 1) // 2  # (query token, attended position)
    return (T * (2 * hq + 2 * hkv) * d * 4 + 2 * hkv * d * es * (rows + T), 4 * d * hq * pairs)


def _moe_work(T):
    D, F, X, K = (MOE[k] for k in ("dim", "ffn", "E", "K"))
    used = X * (1 - (1 - K / X) ** T)  # experts that T tokens reach, on average
    return (X * D * 4 + used * (2 * _q8_bytes(F, D) + _q8_bytes(D, F)) + 2 * T * D * 4,
            2 * T * X * D + 2 * T * K * 3 * D * F)


def work(case):
    c, kind = case, case["kind"]
    if kind == "engine":
        g = MODELS[c["model"]]
        hid, hq, hkv, hd, X, K, F, V = (g[k] for k in ("hidden_dim", "n_q_heads", "n_kv_heads", "head_dim", "n_experts",
                                                       "top_k", "expert_ffn_dim", "vocab_size"))
        n = c["n"]
        ab, af = _attention_work(n, c["pos"], hq, hkv, hd, 2 if c["kv"] == "f16" else 4)
        used = X * (1 - (1 - K / X) ** n)
        proj = (2 * hq + 2 * hkv) * hd * hid
        b = ab + proj // 32 * 34 + X * hid * 4 + used * 3 * _q8_bytes(F, hid) + 2 * n * hid * 4
        f = af + 2 * n * (proj + X * hid + K * 3 * F * hid)
        return dict(bytes=g["n_layers"] * b + _q8_bytes(V, hid) + n * V * 4, flops=g["n_layers"] * f + 2 * n * V * hid)
    if kind == "step":
        b, f = _attention_work(1, c["pos"], c["hq"], c["hkv"], c["d"], 2)
        return dict(bytes=c["layers"] * b, flops=c["layers"] * f)
    if kind in ("block", "layer"):
        p = LAYER if kind == "layer" else c
        hq, hkv, d, hidden, T = p["hq"], p["hkv"], p["d"], p["hidden"], c["T"]
        # q, k and v need not reach memory between the projections and the attention
        b, f = _attention_work(T, c["pos"], hq, hkv, d, 2 if c["kv"] == "f16" else 4)
        n = (hq + 2 * hkv) * d
        b += _q8_bytes(n, hidden) + T * hidden * 4 - T * n * 4
        f += 2 * T * n * hidden
        if kind == "layer":
            mb, mf = _moe_work(T)
            b += _q8_bytes(hidden, hq * d) + mb - T * hq * d * 4
            f += 2 * T * hidden * hq * d + mf
        return dict(bytes=b, flops=f)
    if kind == "paged":
        mean = (c["lo"] + c["hi"]) / 2
        b, f = _attention_work(1, mean - 1, c["hq"], c["hkv"], c["d"], 2)
        return dict(bytes=c["seqs"] * (b + 4 * mean / c["page"]), flops=c["seqs"] * f)
    if kind == "moe":
        b, f = _moe_work(c["T"])
        return dict(bytes=b, flops=f)
    return dict(bytes=_q8_bytes(c["n"], c["k"]) + c["m"] * (c["n"] + c["k"]) * 4, flops=2 * c["m"] * c["n"] * c["k"])


def tolerance(case):
    """About four times the distance from the 64-bit results that the calls show (in brackets)."""
    kind = case["kind"]
    if kind in ("moe", "linear"):
        return {"rel": 4e-6}  # f32 sums in another order (1e-7 to 8e-7)
    if kind == "engine":  # f32 sums through 3 or 4 layers (1e-6); an f16 cache rounds its rows, to either side
        return {"rel": 5e-6 if case["kv"] == "f32" else 4e-4}
    if kind == "block" and case["kv"] == "f32":
        return {"rel": 6e-5}  # the f32 rope angle of late positions (1e-6 at 500, 1.4e-5 at 3000)
    if kind == "block" and case["T"] > 1:
        return {"rel": 1.2e-3}  # f16 query operand (3e-4)
    return {"rel": 3e-4}  # rope angles of late positions, rounding of appended f16 rows (7e-5)


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _dq(w):
    """Q8_0 rows as f64."""
    b = w.view(w.shape[0], -1, 34)
    s = b[:, :, :2].contiguous().view(torch.float16).double()
    return (s * b[:, :, 2:].contiguous().view(torch.int8).double()).view(w.shape[0], -1)


def _rms(x, w, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, positions):
    """NeoX rotation of [T, heads, d]; the angle is the f32 product pos * theta^(-2i/d) the ops define."""
    d = x.shape[-1]
    inv = torch.tensor([THETA ** (-float(np.float32(2 * i) / np.float32(d))) for i in range(d // 2)], dtype=torch.float64,
                       device=x.device).float()
    ang = (positions.float()[:, None] * inv[None]).double()
    co, si = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * co - b * si, a * si + b * co], -1)


def _attend(q, k, v, first):
    """q [T, hq, d] at positions first.., k / v [hkv, L, d] -> [T, hq * d], causal."""
    T, hq, d = q.shape
    hkv, L = k.shape[:2]
    out = torch.empty(T, hq, d, dtype=torch.float64, device=q.device)
    seen = torch.arange(L, device=q.device)[None] <= first + torch.arange(T, device=q.device)[:, None]
    for h in range(hq):
        kh = h // (hq // hkv)
        p = (q[:, h] @ k[kh].T) * _scale(d)
        out[:, h] = torch.softmax(p.masked_fill(~seen, -math.inf), 1) @ v[kh]
    return out.view(T, hq * d)


def _step(q, k, v, qn, kn, positions, kc, vc, pos):
    """The attention step; kc / vc are f64 copies of the caches, written as their type rounds."""
    kv_type = kc.kv_type
    T = q.shape[0]
    q = _rope(_rms(q.double(), qn), positions)
    k = _rope(_rms(k.double(), kn), positions)
    kc.rows[:, pos:pos + T] = k.to(kv_type).double().transpose(0, 1) if kv_type == torch.float16 else k.transpose(0, 1)
    vc.rows[:, pos:pos + T] = v.double().to(kv_type).double().transpose(0, 1) if kv_type == torch.float16 else \
        v.double().transpose(0, 1)
    return _attend(q, kc.rows[:, :pos + T], vc.rows[:, :pos + T], pos)


class _Rows:
    def __init__(self, cache):
        self.rows, self.kv_type = cache.double(), cache.dtype


def _block(t, hq, hkv, d, kc, vc, pos):
    h = _rms(t["x"].double(), t["an"])
    T = h.shape[0]
    q, k, v = ((h @ _dq(t[n]).T).view(T, -1, d) for n in ("wq", "wk", "wv"))
    return _step(q, k, v, t["qn"], t["kn"], t["positions"], kc, vc, pos)


def _experts(x, fn, router, gate, up, down, F, K):
    """x + the MoE of rms(x): the top K of the softmax, renormalised."""
    h = _rms(x, fn)
    X, D = router.shape
    p = torch.softmax(h @ router.double().T, 1)
    w, ids = torch.topk(p, K, 1)
    w = w / w.sum(1, keepdim=True)
    out = x.clone()
    for e in range(X):
        tok, slot = (ids == e).nonzero(as_tuple=True)
        if tok.numel():
            g, u = (h[tok] @ _dq(b.view(X, F, -1)[e]).T for b in (gate, up))
            y = (g / (1 + torch.exp(-g)) * u) @ _dq(down.view(X, D, -1)[e]).T
            out.index_add_(0, tok, w[tok, slot][:, None] * y)
    return out


def _engine_exact(case, seed):
    c = MODELS[case["model"]]
    w, toks = _model_tensors(case["model"], seed)
    n = case["pos"] + case["n"]
    hid, hq, hkv, hd = c["hidden_dim"], c["n_q_heads"], c["n_kv_heads"], c["head_dim"]
    positions = torch.arange(n, dtype=torch.int32, device=DEV)
    x = _dq(w["token_embd.weight"][torch.tensor(toks[:n], device=DEV)])
    for li in range(c["n_layers"]):
        g = lambda name: w[f"blk.{li}.{name}.weight"]  # noqa: E731
        kc, vc = (_Rows(torch.zeros(hkv, n, hd, dtype=_kv_type(case["kv"]), device=DEV)) for _ in range(2))
        t = dict(x=x, an=g("attn_norm"), wq=g("attn_q"), wk=g("attn_k"), wv=g("attn_v"), qn=g("attn_q_norm"),
                 kn=g("attn_k_norm"), positions=positions)
        x = x + _block(t, hq, hkv, hd, kc, vc, 0) @ _dq(g("attn_output")).T
        x = _experts(x, g("ffn_norm"), g("ffn_gate_inp"), g("ffn_gate_exps"), g("ffn_up_exps"), g("ffn_down_exps"),
                     c["expert_ffn_dim"], c["top_k"])
    return (_rms(x[case["pos"]:], w["output_norm.weight"]) @ _dq(w["output.weight"]).T).cpu().numpy()


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "engine":
        return _engine_exact(case, seed)
    t = prepare(case, seed)["t"]
    if kind == "linear":
        return t["x"].double() @ _dq(t["w"]).T
    if kind == "moe":
        return _experts(t["x"].double(), t["fn"], t["router"], t["gate"], t["up"], t["down"], MOE["ffn"], MOE["K"])
    if kind == "step":
        outs = []
        for i in range(c["layers"]):
            kc, vc = _Rows(t["kc"][i]), _Rows(t["vc"][i])
            outs.append((_step(t["q"][i], t["k"][i], t["v"][i], t["qn"], t["kn"], t["positions"], kc, vc, c["pos"]),
                         kc.rows, vc.rows))
        return dict(zip(("attn", "kc", "vc"), (torch.stack(v) for v in zip(*outs))))
    kc, vc = _Rows(t["kc"]), _Rows(t["vc"])
    if kind == "paged":
        out = torch.empty(c["seqs"], c["hq"] * c["d"], dtype=torch.float64, device=DEV)
        for b, n in enumerate(t["lens"].tolist()):
            p = torch.arange(n, device=DEV)
            slots = t["table"][b].long()[p // c["page"]] * c["page"] + p % c["page"]
            ks, vs = (_Rows(x[:, slots]) for x in (t["kc"], t["vc"]))
            out[b] = _step(t["q"][b][None], t["k"][b][None], t["v"][b][None], t["qn"], t["kn"],
                           torch.tensor([n - 1], device=DEV), ks, vs, n - 1)[0]
            kc.rows[:, slots[-1]], vc.rows[:, slots[-1]] = ks.rows[:, -1], vs.rows[:, -1]
        return dict(attn=out, kc=kc.rows, vc=vc.rows)
    p = LAYER if kind == "layer" else c
    attn = _block(t, p["hq"], p["hkv"], p["d"], kc, vc, c["pos"])
    if kind == "block":
        return dict(attn=attn, kc=kc.rows, vc=vc.rows)
    mid = t["x"].double() + attn @ _dq(t["wo"]).T
    out = _experts(mid, t["fn"], t["router"], t["gate"], t["up"], t["down"], MOE["ffn"], MOE["K"])
    return dict(out=out, kc=kc.rows, vc=vc.rows)
