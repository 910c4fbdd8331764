"""Dit::cache_context in groups of blocks: each block's prepared K/V against its own product, norm and prepare pass."""
import ctypes

import pytest
import torch

import kiln_amd
from kiln_amd import KILN_EINVAL, dit

pytestmark = pytest.mark.gpu
DEV, H, BLOCKS, CTX = "cuda:0", 2, 3, 64
D = 128 * H


class _View:
    def __init__(self, buf, halves):
        self.buf = buf
        self.__cuda_array_interface__ = dict(shape=(halves,), typestr="<f2", data=(buf.data_ptr(), False), version=2)


# one token; a partial tile; 12000 tokens, whose 24 MB a block put two blocks in a group and one in the next
@pytest.mark.parametrize("real", [1, 77, 12000])
@pytest.mark.parametrize("fp32", [False, True])
def test_context_groups(gpu, real, fp32):
    g = torch.Generator(device=DEV).manual_seed(real)
    bf = lambda o, i: (torch.randn(o, i, device=DEV, generator=g) * i ** -0.5).bfloat16()  # noqa: E731
    d = dit.Dit(BLOCKS, H, ctx_dim=CTX)
    ws = []
    for i in range(BLOCKS):
        w = {n: bf(D, D) for n in ("sa_q", "sa_k", "sa_v", "sa_o", "ca_q", "ca_o")}
        w.update(ca_k=bf(D, CTX), ca_v=bf(D, CTX), mlp1=bf(4 * D, D), mlp2=bf(D, 4 * D))
        w.update({n: (1 + 0.2 * torch.randn(128, device=DEV, generator=g)).bfloat16() for n in ("sa_qn", "sa_kn", "ca_qn", "ca_kn")})
        d.set_block(i, **w, mod=[bf(256, D) if j % 2 == 0 else bf(3 * D, 256) for j in range(6)])
        ws.append(w)
    ctx = torch.randn(real, CTX, device=DEV, generator=g)
    c = d.cache_context(ctx, fp32=fp32)
    halves = kiln_amd.kv_prepped_bytes(real, H) // 2
    for i, w in enumerate(ws):
        k, v = torch.empty(real, D, device=DEV), torch.empty(real, D, device=DEV)
        kiln_amd.linear_f32(k, ctx, w["ca_k"])
        kiln_amd.linear_f32(v, ctx, w["ca_v"])
        ref = kiln_amd.kv_prepare(k, v, H, k_norm_w=w["ca_kn"]).view(torch.float16)[:halves].float()
        got = torch.as_tensor(_View(c.kv(i), halves), device=DEV).float()
        # the same fp32 values up to the order of their sums: one fp16 rounding apart at most
        assert ((got - ref).abs() <= 2.0 ** -10 * ref.abs() + 2.0 ** -18).all(), f"block {i}"
        assert (got[ref == 0] == 0).all()


def _weights(g):
    bf = lambda o, i: (torch.randn(o, i, device=DEV, generator=g) * i ** -0.5).bfloat16()  # noqa: E731
    w = {n: bf(D, D) for n in ("sa_q", "sa_k", "sa_v", "sa_o", "ca_q", "ca_o")}
    w.update(ca_k=bf(D, CTX), ca_v=bf(D, CTX), mlp1=bf(4 * D, D), mlp2=bf(D, 4 * D))
    w.update({n: (1 + 0.2 * torch.randn(128, device=DEV, generator=g)).bfloat16() for n in ("sa_qn", "sa_kn", "ca_qn", "ca_kn")})
    w["mod"] = [bf(256, D) if j % 2 == 0 else bf(3 * D, 256) for j in range(6)]
    return w


# one group of three blocks; two blocks and one (12000 tokens)
@pytest.mark.parametrize("real", [77, 12000])
def test_context_groups_fp32(gpu, real):
    """The fp32 K and V of a context of three blocks, which no call hands out: each block run in fp32 against a model of
    that block alone (whose context is one product of its own; checked against float64 in test_dit_block_gpu.py). The
    products may run on different tiles, so their sums differ by rounding: 1e-5 of outputs of size 1."""
    g = torch.Generator(device=DEV).manual_seed(real)
    ws = [_weights(g) for _ in range(BLOCKS)]
    d = dit.Dit(BLOCKS, H, ctx_dim=CTX)
    for i, w in enumerate(ws):
        d.set_block(i, **w)
    ctx = torch.randn(real, CTX, device=DEV, generator=g)
    X0, mods = torch.randn(32, D, device=DEV, generator=g), torch.randn(9 * D, device=DEV, generator=g)
    c = d.cache_context(ctx, fp32=True)
    for i, w in enumerate(ws):
        one = dit.Dit(1, H, ctx_dim=CTX)
        one.set_block(0, **w)
        a = d.run_block(i, X0.clone(), mods, 4, 8, [c], fp32=True)
        b = one.run_block(0, X0.clone(), mods, 4, 8, [one.cache_context(ctx, fp32=True)], fp32=True)
        assert (a - b).abs().max() <= 1e-5 * max(1.0, b.abs().max().item()), f"block {i}"
        # the bar tells another block's projections and norm apart
        for n in ("ca_k", "ca_v", "ca_kn"):
            one.set_block(0, **dict(w, **{n: ws[(i + 1) % BLOCKS][n]}))
            z = one.run_block(0, X0.clone(), mods, 4, 8, [one.cache_context(ctx, fp32=True)], fp32=True)
            assert (z - b).abs().max() > 1e-3, f"block {i} {n}: {(z - b).abs().max().item()}"


def test_rejected_set_block_changes_nothing(gpu):
    """kiln_dit_set_block with a weight missing, whichever: the call fails and the block that was there stays whole (its
    context projections too, which lie in one allocation with the other blocks'); a first block that fails leaves none."""
    g = torch.Generator(device=DEV).manual_seed(3)
    d = dit.Dit(2, H, ctx_dim=CTX)
    old, new = [_weights(g) for _ in range(2)], _weights(g)
    fields = [f for f, _ in dit.BlockWeights._fields_]
    flat = dict({k: v for k, v in new.items() if k != "mod"}, **dict(zip(fields[-6:], new["mod"])))
    ctx = torch.randn(33, CTX, device=DEV, generator=g)

    def reject(missing):
        w = dit.BlockWeights(*[None if f == missing else flat[f].data_ptr() for f in fields])
        assert dit.dlib().kiln_dit_set_block(d._h, 0, ctypes.byref(w)) == KILN_EINVAL, missing

    def kv(i):
        c = d.cache_context(ctx)
        return torch.as_tensor(_View(c.kv(i), kiln_amd.kv_prepped_bytes(33, H) // 2), device=DEV).clone()

    reject("mlp2")
    with pytest.raises(kiln_amd.KilnError, match="no weights"):
        kv(0)
    for i in range(2):
        d.set_block(i, **old[i])
    before = [kv(i) for i in range(2)]
    for f in fields:
        reject(f)
        for i in range(2):
            assert torch.equal(kv(i), before[i]), f"block {i} after a call without {f}"
    d.set_block(0, **new)
    assert not torch.equal(kv(0), before[0]) and torch.equal(kv(1), before[1])


def test_kv_prepare_blocks_rejects(gpu):
    L = kiln_amd.lib()
    p = ctypes.c_void_p(256)
    assert L.kiln_kv_prepare_blocks(p, p, 2 * D - 4, 1, 8, H, p, 1e-6, None) == KILN_EINVAL  # rows too short
    assert L.kiln_kv_prepare_blocks(p, p, 2 * D, 0, 8, H, p, 1e-6, None) == KILN_EINVAL
    assert L.kiln_kv_prepare_blocks(None, p, 2 * D, 1, 8, H, p, 1e-6, None) == KILN_EINVAL
    assert L.kiln_kv_prepare_blocks(p, p, 2 * D, 1, 0, H, p, 1e-6, None) == 0
