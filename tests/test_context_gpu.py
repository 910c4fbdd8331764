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


def test_kv_prepare_blocks_rejects(gpu):
    L = kiln_amd.lib()
    p = ctypes.c_void_p(256)
    assert L.kiln_kv_prepare_blocks(p, p, 2 * D - 4, 1, 8, H, p, 1e-6, None) == KILN_EINVAL  # rows too short
    assert L.kiln_kv_prepare_blocks(p, p, 2 * D, 0, 8, H, p, 1e-6, None) == KILN_EINVAL
    assert L.kiln_kv_prepare_blocks(None, p, 2 * D, 1, 8, H, p, 1e-6, None) == KILN_EINVAL
    assert L.kiln_kv_prepare_blocks(p, p, 2 * D, 1, 0, H, p, 1e-6, None) == 0
