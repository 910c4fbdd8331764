"""The work a diffusion engine has this library do, as timed cases over the public entry points of kiln_amd.

All cases have the widths of the 2B Cosmos-Predict2 DiT (D = 2048: 16 heads of 128, MLP 8192, text width 1024,
28 blocks). A picture of H x W pixels is (H/16) x (W/16) tokens; the engine renders 256x256 previews (T = 256) to
1024x1024 (T = 4096), one item or the CFG pair at a time. Kinds of case:

  self     dit_self_attn: the block's self-attention from projected Q/K/V, QK-RMSNorm and RoPE fused
  cross    cross_attn_nag: the CFG batch against its text contexts, the NAG negative and its blend
  attn16   attention16: the drop-in call of an engine that holds fp32 Q/K/V
  linear   linear16: one linear layer with its fused epilogue, plain or prepared weight, LoRA pair or not
  mlp      the block's MLP: the GELU GEMM and the gated-residual GEMM with prepared weights
  block    Dit.run_block: one transformer block, in the fp16 form and in the fp32 form (the engine's --fp32)
  context  Dit.cache_context: the text context's K/V of all 28 blocks, once per prompt
  forward  Dit.forward: a denoising step's whole model call, from the latent to the velocity

Drawn cases spread the picture's sides over 8 .. 64 tokens (log-uniform), the text over 1 .. 512 real tokens.
"""
import math

import torch

import kiln_amd
from kiln_amd import dit

HEADS, HD, MLP, TEXT, BLOCKS = 16, 128, 8192, 1024, 28
D = HEADS * HD
EPS = 1e-6
CTX_LEN = 512  # text contexts count at least 512 tokens: the real ones and zero padding
NAG = (5.0, 2.5, 0.25)  # scale, tau, alpha
DEV = "cuda"


def listed():
    return [
        # the largest picture's self-attention, the CFG pair in one call: where a step spends its attention time
        dict(name="self 1024x1024 pair", kind="self", Hp=64, Wp=64, B=2, dt="f16"),
        # a preview's self-attention: a few dozen query tiles, launch and latency
        dict(name="self 256x256", kind="self", Hp=16, Wp=16, B=1, dt="f16"),
        # cross-attention + NAG of a portrait picture against contexts that fill the 512 tokens
        dict(name="cross nag 768x1152 full", kind="cross", Hp=48, Wp=72, B=2, pos=512, neg=512, nag=512),
        # the same with prompts of ordinary length: the padding's zero keys enter analytically
        dict(name="cross nag 512x768 short", kind="cross", Hp=32, Wp=48, B=2, pos=77, neg=23, nag=41),
        # an engine that keeps fp32 Q/K/V and takes attention16 as it is
        dict(name="attention16 512x768", kind="attn16", Tq=1536, Tk=1536, npad=0),
        # the two MLP GEMMs of a large pair: 60% of a block's matrix work
        dict(name="mlp 768x1152 pair", kind="mlp", M=6912),
        # an O projection with a LoRA pair on a plain weight: a small picture, one item
        dict(name="linear lora 512x512", kind="linear", M=1024, N=2048, K=2048, k2=32, epi="resid", prepped=False),
        # one whole block of a middle-sized pair with NAG
        dict(name="block 512x768 pair nag", kind="block", Hp=32, Wp=48, B=2, nag=True, fp32=False, real=77),
        # the same kind of block in fp32
        dict(name="block fp32 512x512", kind="block", Hp=32, Wp=32, B=1, nag=False, fp32=True, real=77),
        # a new prompt: K/V of all blocks
        dict(name="context 120 tokens", kind="context", real=120),
        # a step of a large picture with CFG and NAG
        dict(name="forward 768x1152 pair nag", kind="forward", Hl=96, Wl=144, B=2, nag=True, real=120),
        # a step of a preview: 28 blocks of small kernels
        dict(name="forward 256x256", kind="forward", Hl=32, Wl=32, B=1, nag=False, real=40),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["self", "cross", "attn16", "linear", "mlp", "block", "block", "context", "forward", "forward"])
    Hp, Wp, B = _log(rng, 8, 64), _log(rng, 8, 64), rng.choice([1, 2])
    if kind == "self":
        return dict(kind=kind, Hp=Hp, Wp=Wp, B=B, dt=rng.choice(["f16", "f16", "f32"]))
    if kind == "cross":
        return dict(kind=kind, Hp=Hp, Wp=Wp, B=B, pos=_log(rng, 4, 512), neg=_log(rng, 1, 512),
                    nag=rng.choice([0, _log(rng, 1, 512)]))
    if kind == "attn16":
        tq = _log(rng, 64, 4096)
        return dict(kind=kind, Tq=tq, Tk=rng.choice([tq, _log(rng, 64, 4096)]), npad=rng.choice([0, rng.randrange(1, 512)]))
    if kind == "linear":
        n, k = rng.choice([(2048, 2048), (2048, 2048), (8192, 2048), (2048, 8192)])
        return dict(kind=kind, M=_log(rng, 64, 6912), N=n, K=k, k2=rng.choice([0, 32, 64]),
                    epi=rng.choice(["f32", "f16", "gelu", "resid"]), prepped=rng.choice([True, False]))
    if kind == "mlp":
        return dict(kind=kind, M=_log(rng, 64, 6912))
    if kind == "block":
        fp32 = rng.choice([False, False, True])
        return dict(kind=kind, Hp=Hp, Wp=Wp, B=B if Hp * Wp <= 3456 else 1, nag=rng.choice([True, False]), fp32=fp32,
                    real=_log(rng, 4, 512))
    if kind == "context":
        return dict(kind=kind, real=_log(rng, 4, 512))
    # a latent's side may be odd: the forward then pads it to the patch grid
    return dict(kind="forward", Hl=2 * Hp - rng.choice([0, 0, 1]), Wl=2 * Wp - rng.choice([0, 0, 1]),
                B=B if Hp * Wp <= 3456 else 1, nag=rng.choice([True, False]), real=_log(rng, 4, 512))


# ---- inputs, from the seed alone ----

def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + salt * 7919) % (1 << 62))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _linear_w(g, out_f, in_f):
    """torch.nn.Linear's default init, as a bf16 checkpoint stores it."""
    return ((torch.rand(out_f, in_f, generator=g, device=DEV) * 2 - 1) / in_f ** 0.5).to(torch.bfloat16)


def _norm_w(g, n=HD):
    return (1 + 0.1 * _randn(g, n)).to(torch.bfloat16)


def _projected(g, rows, in_f=D):
    """Rows of a linear layer's output for normalized activations: what Q, K and V are before their norm."""
    x = _randn(g, rows, in_f)
    return x @ _linear_w(g, D, in_f).float().T


def _block_weights(seed, i):
    g = _gen(seed, 100 + i)
    w = {n: _linear_w(g, D, D) for n in ("sa_q", "sa_k", "sa_v", "sa_o", "ca_q", "ca_o")}
    w.update(ca_k=_linear_w(g, D, TEXT), ca_v=_linear_w(g, D, TEXT), mlp1=_linear_w(g, MLP, D), mlp2=_linear_w(g, D, MLP))
    w.update({n: _norm_w(g) for n in ("sa_qn", "sa_kn", "ca_qn", "ca_kn")})
    w["mod"] = [_linear_w(g, 256, D) if j % 2 == 0 else _linear_w(g, 3 * D, 256) for j in range(6)]
    return w


def _step_weights(seed):
    g = _gen(seed, 99)
    return dict(t_lin1=_linear_w(g, D, D), t_lin2=_linear_w(g, 3 * D, D), t_norm=_norm_w(g, D),
                final_mod1=_linear_w(g, 256, D), final_mod2=_linear_w(g, 2 * D, 256), x_embed=_linear_w(g, D, 68),
                final_lin=_linear_w(g, 64, D))


def _texts(case, seed):
    """The contexts of a call: the prompt, the unconditional one (B = 2), the NAG negative; real rows only."""
    g = _gen(seed, 3)
    reals = [case["real"], max(1, case["real"] // 3)][:case["B"]]
    if case["nag"]:
        reals.append(max(1, case["real"] // 2))
    return [_randn(g, r, TEXT) for r in reals]


def _inputs(case, seed):
    g, k = _gen(seed, 1), case["kind"]
    if k == "self":
        rows = case["B"] * case["Hp"] * case["Wp"]
        q, kk, v = (_projected(g, rows) for _ in range(3))
        if case["dt"] == "f16":
            q, kk, v = q.half(), kk.half(), v.half()
        return dict(q=q, k=kk, v=v, qn=_norm_w(g), kn=_norm_w(g))
    if k == "cross":
        reals = [case["pos"], case["neg"]][:case["B"]] + ([case["nag"]] if case["nag"] else [])
        return dict(q=_projected(g, case["B"] * case["Hp"] * case["Wp"]).half(), qn=_norm_w(g), kn=_norm_w(g),
                    kv=[(_projected(g, r, TEXT).half(), _projected(g, r, TEXT).half()) for r in reals])
    if k == "attn16":
        # after the norm and the rotation: unit-variance Q and K
        return dict(q=_randn(g, case["Tq"], D), k=_randn(g, case["Tk"], D), v=_projected(g, case["Tk"]))
    if k == "linear":
        M, N, K, k2 = case["M"], case["N"], case["K"], case["k2"]
        r = dict(x=_randn(g, M, K).half(), w=_linear_w(g, N, K).half(), a2=None, w2=None, gate=None, y=None)
        if k2:
            r.update(a2=_randn(g, M, k2).half(), w2=(0.1 * _linear_w(g, N, k2)).half())
        if case["epi"] == "resid":
            r.update(gate=0.2 * _randn(g, N), y=_randn(g, M, N))
        return r
    if k == "mlp":
        return dict(x=_randn(g, case["M"], D).half(), w1=_linear_w(g, MLP, D).half(), w2=_linear_w(g, D, MLP).half(),
                    gate=0.2 * _randn(g, D), y=_randn(g, case["M"], D))
    if k == "block":
        return dict(X=_randn(g, case["B"] * case["Hp"] * case["Wp"], D), mods=0.2 * _randn(g, 9 * D))
    if k == "forward":
        return dict(latent=_randn(g, 16, case["Hl"], case["Wl"]))
    return dict(ctx=_randn(g, case["real"], TEXT))


class _View:
    """Device memory of the library's as the array interface that torch reads. A tensor made from it holds it, and it
    holds the memory's owner."""

    def __init__(self, buf, halves):
        self.owner = buf
        self.__cuda_array_interface__ = dict(shape=(halves,), typestr="<f2", data=(buf.data_ptr(), False), version=2)


def prepare(case, seed):
    s, k = dict(_inputs(case, seed), case=case), case["kind"]
    if k == "self":
        rope = kiln_amd.cosmos_rope_tables(case["Hp"], case["Wp"])
        T = case["Hp"] * case["Wp"]
        s.update(T=T, rope=tuple(t.to(DEV) for t in rope), out=torch.empty(case["B"] * T, D, dtype=torch.float16, device=DEV),
                 ws=torch.empty(kiln_amd.dit_self_attn_workspace_bytes(case["B"], T, HEADS), dtype=torch.uint8, device=DEV))
    elif k == "cross":
        T = case["Hp"] * case["Wp"]
        s.update(T=T, kvps=[kiln_amd.kv_prepare(a, b, HEADS, k_norm_w=s["kn"]) for a, b in s["kv"]],
                 out=torch.empty(case["B"] * T, D, dtype=torch.float16, device=DEV),
                 out_neg=torch.empty(T, D, dtype=torch.float16, device=DEV))
    elif k == "attn16":
        s.update(out=torch.empty(case["Tq"], D, dtype=torch.float16, device=DEV))
    elif k == "linear":
        if case["prepped"]:
            s["w"] = kiln_amd.linear16_prepare_weight(s["w"])
        if s["y"] is None:
            s["y"] = torch.empty(case["M"], case["N"], device=DEV, dtype=torch.float32 if case["epi"] == "f32" else torch.float16)
    elif k == "mlp":
        s.update(w1=kiln_amd.linear16_prepare_weight(s["w1"]), w2=kiln_amd.linear16_prepare_weight(s["w2"]),
                 h=torch.empty(case["M"], MLP, dtype=torch.float16, device=DEV))
    else:
        n = 1 if k == "block" else BLOCKS
        d = dit.Dit(n, HEADS, ctx_dim=TEXT)
        for i in range(n):
            d.set_block(i, **_block_weights(seed, i))
        s["dit"] = d
        if k != "context":
            fp32 = bool(case.get("fp32"))
            cs = [d.cache_context(c, fp32=fp32) for c in _texts(case, seed)]
            s.update(ctxs=cs[:case["B"]], nagc=dit.Nag(cs[-1], *NAG) if case["nag"] else None)
        if k == "forward":
            d.set_step_weights(**_step_weights(seed))
            s["outs"] = [torch.empty(16, case["Hl"], case["Wl"], device=DEV) for _ in range(case["B"])]
    return s


_EPI = dict(f32=kiln_amd.KILN_EPI_F32, f16=kiln_amd.KILN_EPI_F16, gelu=kiln_amd.KILN_EPI_GELU16, resid=kiln_amd.KILN_EPI_RESID)


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "self":
        return kiln_amd.dit_self_attn(s["out"], s["q"], s["k"], s["v"], case["B"], s["T"], HEADS, s["qn"], s["kn"], s["rope"],
                                      eps=EPS, workspace=s["ws"])
    if k == "cross":
        B = case["B"]
        reals = [case["pos"], case["neg"]][:B]
        neg = dict(kvp_neg=s["kvps"][-1], Lk_neg=case["nag"], npad_neg=CTX_LEN - case["nag"], out_neg=s["out_neg"],
                   scale=NAG[0], tau=NAG[1], alpha=NAG[2]) if case["nag"] else {}
        return kiln_amd.cross_attn_nag(s["out"], s["q"], B, s["T"], HEADS, s["kvps"][:B], reals, [CTX_LEN - r for r in reals],
                                       q_norm_w=s["qn"], eps=EPS, **neg)
    if k == "attn16":
        return kiln_amd.attention16(s["out"], s["q"], s["k"], s["v"], case["Tq"], case["Tk"], HEADS, npad=case["npad"])
    if k == "linear":
        return kiln_amd.linear16(s["y"], s["x"], s["w"], epi=_EPI[case["epi"]], gate=s["gate"], a2=s["a2"], w2=s["w2"])
    if k == "mlp":
        kiln_amd.linear16(s["h"], s["x"], s["w1"], epi=kiln_amd.KILN_EPI_GELU16)
        return s["h"], kiln_amd.linear16(s["y"], s["h"], s["w2"], epi=kiln_amd.KILN_EPI_RESID, gate=s["gate"])
    if k == "block":
        return s["dit"].run_block(0, s["X"], s["mods"], case["Hp"], case["Wp"], s["ctxs"], nag=s["nagc"], fp32=case["fp32"])
    if k == "context":
        # a new prompt's context replaces the last one's
        s["context"] = s["dit"].cache_context(s["ctx"])
        halves = kiln_amd.kv_prepped_bytes(case["real"], HEADS) // 2
        return [torch.as_tensor(_View(s["context"].kv(i), halves), device=DEV) for i in range(BLOCKS)]
    return s["dit"].forward(s["outs"], s["latent"], 0.5, s["ctxs"], nag=s["nagc"])


# ---- the least a pass can do ----

def _block_work(case, T):
    B, wb = case["B"], 4 if case.get("fp32") else 2  # bytes of an activation
    R = B * T
    texts = [case["real"], max(1, case["real"] // 3)][:B] + ([max(1, case["real"] // 2)] if case["nag"] else [])
    weights = 6 * D * D + 2 * D * MLP
    flops = 2.0 * R * weights + 4.0 * B * T * T * D + sum(4.0 * T * c * D for c in texts)
    return dict(bytes=2.0 * weights + 2.0 * wb * D * sum(texts), flops=flops, x=8.0 * R * D)


def work(case):
    k = case["kind"]
    T = case["Hp"] * case["Wp"] if "Hp" in case else 0
    if k == "self":
        e = 2 if case["dt"] == "f16" else 4
        return dict(bytes=case["B"] * T * D * (3.0 * e + 2) + T * 512, flops=4.0 * case["B"] * T * T * D)
    if k == "cross":
        keys = [case["pos"], case["neg"]][:case["B"]] + ([case["nag"]] if case["nag"] else [])
        return dict(bytes=4.0 * case["B"] * T * D + 4.0 * D * sum(keys), flops=4.0 * T * D * sum(keys))
    if k == "attn16":
        return dict(bytes=D * (6.0 * case["Tq"] + 8.0 * case["Tk"]), flops=4.0 * case["Tq"] * case["Tk"] * D)
    if k == "linear":
        M, N, K = case["M"], case["N"], case["K"] + case["k2"]
        return dict(bytes=2.0 * K * (M + N) + M * N * dict(f32=4, f16=2, gelu=2, resid=8)[case["epi"]], flops=2.0 * M * N * K)
    if k == "mlp":
        M = case["M"]
        return dict(bytes=2.0 * M * D + 4.0 * D * MLP + 2.0 * M * MLP + 8.0 * M * D, flops=4.0 * M * D * MLP)
    if k == "block":
        w = _block_work(case, T)
        return dict(bytes=w["bytes"] + w["x"], flops=w["flops"])
    if k == "context":
        r = case["real"]
        return dict(bytes=4.0 * r * TEXT + BLOCKS * (4.0 * D * TEXT + 4.0 * r * D), flops=BLOCKS * 4.0 * r * D * TEXT)
    T = ((case["Hl"] + 1) // 2) * ((case["Wl"] + 1) // 2)
    w = _block_work(case, T)
    mods = 2.0 * (D * D * 4 + BLOCKS * 3 * (256 * D + 3 * D * 256))
    lat = 64.0 * case["Hl"] * case["Wl"] * (1 + case["B"])
    return dict(bytes=BLOCKS * w["bytes"] + mods + lat, flops=BLOCKS * w["flops"] + 2.0 * case["B"] * T * D * (68 + 64))


def tolerance(case):
    """About four times the measured error against exact(), which is what two correct implementations differ by at most."""
    k = case["kind"]
    if k in ("self", "cross", "attn16"):
        return {"rel": 2e-3}  # fp16 rounding of Q, K, P and the output: 4.2e-4 to 4.7e-4
    if k == "linear":
        # the order of a 32-bit sum; an fp16 output may round the other way
        return {"rel": 1e-5 if case["epi"] in ("f32", "resid") else 5e-4}
    if k == "mlp":
        return {"rel": 5e-4}  # the fp16 hidden activation: 2.1e-4; the fp32 result: 8e-6
    if k == "block":
        return {"rel": 1e-6 if case["fp32"] else 1e-4}  # 9e-8; 1.3e-5 (of the residual stream, fp32)
    if k == "context":
        return {"rel": 5e-4}  # fp16 K and V: 2.1e-4
    return {"rel": 1e-3}  # 28 blocks of fp16 activations: 1.7e-4


# ---- the same in 64 bits ----

def _d(t):
    return t.double()


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * _d(w)


def _rope(x, Hp, Wp):
    """The Cosmos 3D rotation of one frame: 22 temporal pairs (identity), 21 of the row, 21 of the column."""
    dh = 128 // 6 * 2
    theta = 10000.0 * 4.0 ** (dh / (dh - 2))
    f = theta ** (-torch.arange(0, dh, 2, dtype=torch.float64, device=DEV) / dh)
    y = torch.arange(Hp, dtype=torch.float64, device=DEV)[:, None, None] * f
    z = torch.arange(Wp, dtype=torch.float64, device=DEV)[None, :, None] * f
    pairs = (128 - 2 * dh) // 2
    a = torch.cat([torch.zeros(Hp, Wp, pairs, dtype=torch.float64, device=DEV), y.expand(Hp, Wp, -1), z.expand(Hp, Wp, -1)], -1)
    a = a.reshape(Hp * Wp, 1, 64)
    lo, hi = x[..., :64], x[..., 64:]
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()], -1)


def _heads(x):
    return x.reshape(-1, HEADS, HD)


def _attend(q, k, v, npad=0):
    """q [Tq, heads, 128] against k, v [Tk, heads, 128] and npad keys and values of zero."""
    out = torch.empty_like(q)
    for h in range(HEADS):
        s = q[:, h] @ k[:, h].T / HD ** 0.5
        m = s.amax(1, keepdim=True)
        if npad:
            m = m.clamp_min(0)
        p = (s - m).exp()
        out[:, h] = (p @ v[:, h]) / (p.sum(1, keepdim=True) + npad * (-m).exp())
    return out.reshape(q.shape[0], D)


def _nag(p, n):
    scale, tau, alpha = NAG
    g = p * scale - n * (scale - 1)
    ratio = g.abs().sum(1, keepdim=True) / p.abs().sum(1, keepdim=True).clamp_min(1e-12)
    return alpha * g * torch.where(ratio > tau, tau / ratio, torch.ones_like(ratio)) + (1 - alpha) * p


def _gelu(x):
    return 0.5 * x * torch.special.erfc(-x / 2 ** 0.5)


def _ln(x, scale, shift):
    mean = x.mean(-1, keepdim=True)
    c = x - mean
    return c * torch.rsqrt((c * c).mean(-1, keepdim=True) + EPS) * (1 + scale) + shift


def _block64(w, X, mods, Hp, Wp, B, texts, nag):
    T = Hp * Wp
    m = mods.reshape(9, D)
    lin = lambda x, n: x @ _d(w[n]).T  # noqa: E731
    n = _ln(X, m[1], m[0])
    q, k, v = (lin(n, x) for x in ("sa_q", "sa_k", "sa_v"))
    a = []
    for b in range(B):
        r = slice(b * T, (b + 1) * T)
        a.append(_attend(_rope(_rms(_heads(q[r]), w["sa_qn"]), Hp, Wp), _rope(_rms(_heads(k[r]), w["sa_kn"]), Hp, Wp), _heads(v[r])))
    X = X + m[2] * lin(torch.cat(a), "sa_o")
    q = _rms(_heads(lin(_ln(X, m[4], m[3]), "ca_q")), w["ca_qn"])

    def cross(qb, c):
        c = _d(c)
        return _attend(qb, _rms(_heads(lin(c, "ca_k")), w["ca_kn"]), _heads(lin(c, "ca_v")), max(0, CTX_LEN - c.shape[0]))

    a = [cross(q[b * T:(b + 1) * T], texts[b]) for b in range(B)]
    if nag:
        a[0] = _nag(a[0], cross(q[:T], texts[B]))
    X = X + m[5] * lin(torch.cat(a), "ca_o")
    return X + m[8] * lin(_gelu(lin(_ln(X, m[7], m[6]), "mlp1")), "mlp2")


def _tiles(x, order):
    """[real, D] K or V as the prepared buffer's operand order, [heads, half tiles, 4096]."""
    keys = -(-x.shape[0] // 64) * 64
    p = torch.zeros(keys, HEADS, HD, dtype=torch.float64, device=DEV)
    p[:x.shape[0]] = _heads(x)
    p = p.permute(1, 0, 2).reshape(HEADS, keys // 32, 32, HD)
    if order == "k":  # key = 16 a + l, d = 32 b + 8 g + e  ->  [b, a, g, l, e]
        p = p.reshape(HEADS, -1, 2, 16, 4, 4, 8).permute(0, 1, 4, 2, 5, 3, 6)
    else:  # key = 16 a + 4 g + j, d = 16 b + l  ->  [b, g, l, a, j]
        p = p.reshape(HEADS, -1, 2, 4, 4, 8, 16).permute(0, 1, 5, 3, 6, 2, 4)
    return p.reshape(HEADS, keys // 32, 32 * HD)


def _forward64(case, seed, latent):
    B, Hl, Wl = case["B"], case["Hl"], case["Wl"]
    H2, W2 = Hl + Hl % 2, Wl + Wl % 2
    lat = latent[:, torch.arange(H2, device=DEV) % Hl][:, :, torch.arange(W2, device=DEV) % Wl]
    Hp, Wp = H2 // 2, W2 // 2
    T = Hp * Wp
    sw, texts = _step_weights(seed), _texts(case, seed)
    silu = torch.nn.functional.silu
    e = torch.exp(-math.log(10000.0) / (D // 2) * torch.arange(D // 2, dtype=torch.float64, device=DEV))
    t = torch.cat([(0.5 * e).cos(), (0.5 * e).sin()])
    lora = _d(sw["t_lin2"]) @ silu(_d(sw["t_lin1"]) @ t)
    temb = silu(_rms(t, sw["t_norm"]))
    tok = lat.reshape(16, Hp, 2, Wp, 2).permute(1, 3, 0, 2, 4).reshape(T, 64)
    X = (tok @ _d(sw["x_embed"])[:, :64].T).repeat(B, 1)
    for i in range(BLOCKS):
        w = _block_weights(seed, i)
        mods = torch.cat([_d(w["mod"][j + 1]) @ (_d(w["mod"][j]) @ temb) + lora for j in (0, 2, 4)])
        X = _block64(w, X, mods, Hp, Wp, B, texts, case["nag"])
    f = _d(sw["final_mod2"]) @ (_d(sw["final_mod1"]) @ temb) + lora[:2 * D]
    y = _ln(X, f[D:], f[:D]) @ _d(sw["final_lin"]).T
    outs = y.reshape(B, Hp, Wp, 2, 2, 16).permute(0, 5, 1, 3, 2, 4).reshape(B, 16, H2, W2)
    return [outs[b, :, :Hl, :Wl].contiguous() for b in range(B)]


def exact(case, seed):
    i, k = _inputs(case, seed), case["kind"]
    if k == "self":
        T, out = case["Hp"] * case["Wp"], []
        for b in range(case["B"]):
            q, kk, v = (_heads(_d(i[n][b * T:(b + 1) * T])) for n in "qkv")
            out.append(_attend(_rope(_rms(q, i["qn"]), case["Hp"], case["Wp"]), _rope(_rms(kk, i["kn"]), case["Hp"], case["Wp"]), v))
        return torch.cat(out)
    if k == "cross":
        B, T = case["B"], case["Hp"] * case["Wp"]
        q = _rms(_heads(_d(i["q"])), i["qn"])
        one = lambda qb, kv: _attend(qb, _rms(_heads(_d(kv[0])), i["kn"]), _heads(_d(kv[1])), CTX_LEN - kv[0].shape[0])  # noqa: E731
        out = [one(q[b * T:(b + 1) * T], i["kv"][b]) for b in range(B)]
        if case["nag"]:
            out[0] = _nag(out[0], one(q[:T], i["kv"][-1]))
        return torch.cat(out)
    if k == "attn16":
        return _attend(_heads(_d(i["q"])), _heads(_d(i["k"])), _heads(_d(i["v"])), case["npad"])
    if k == "linear":
        y = _d(i["x"]) @ _d(i["w"]).T
        if case["k2"]:
            y = y + _d(i["a2"]) @ _d(i["w2"]).T
        return _d(i["y"]) + _d(i["gate"]) * y if case["epi"] == "resid" else _gelu(y) if case["epi"] == "gelu" else y
    if k == "mlp":
        h = _gelu(_d(i["x"]) @ _d(i["w1"]).T)
        return h, _d(i["y"]) + _d(i["gate"]) * (h @ _d(i["w2"]).T)
    if k == "block":
        return _block64(_block_weights(seed, 0), _d(i["X"]), _d(i["mods"]), case["Hp"], case["Wp"], case["B"], _texts(case, seed),
                        case["nag"])
    if k == "context":
        out, c = [], _d(i["ctx"])
        for b in range(BLOCKS):
            w = _block_weights(seed, b)
            kk = _rms(_heads(c @ _d(w["ca_k"]).T), w["ca_kn"]).reshape(-1, D)
            out.append(torch.cat([_tiles(kk, "k"), _tiles(c @ _d(w["ca_v"]).T, "v")], -1).reshape(-1))
        return out
    return _forward64(case, seed, _d(i["latent"]))
