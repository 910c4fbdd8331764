"""Attention on grids of at most one 128-row unit per CU (16 query rows per wave, 64- or 128-row workgroups): ragged query
tiles and keys, padding keys, every input and output type and output alignment, chains of contexts, and results that do
not depend on the form a call takes. The bar is BASELINE's (max-abs 2e-3, mean-abs 2e-4) against double-precision
attention of the same fp16 values."""
import pytest
import torch

import kiln_amd
import oracle
from tests.helpers import assert_close, f16_round, randn

pytestmark = pytest.mark.gpu
D, DEV = 128, "cuda:0"


# H = 2: 64-row units (4 waves); H = 20 and 900 rows: 300 64-row units, 160 128-row units (8 waves)
@pytest.mark.parametrize("H,Tq,Tk,npad", [(2, 1, 1, 0), (2, 64, 31, 3), (2, 65, 32, 0), (2, 63, 33, 512), (2, 15, 257, 0), (2, 130, 300, 1),
                                          (20, 900, 65, 0), (20, 897, 96, 7), (20, 1024, 290, 0)])
def test_small_grid(gpu, H, Tq, Tk, npad):
    q, k, v = f16_round(randn(Tq, Tq, H * D)), f16_round(randn(Tk, Tk, H * D)), f16_round(randn(7, Tk, H * D))
    ref = oracle.attn_f64(q.numpy(), k.numpy(), v.numpy(), H, npad=npad)
    kvp = kiln_amd.kv_prepare(k.half().to(DEV), v.half().to(DEV), H)
    for qd in (q.half().to(DEV), q.to(DEV)):
        for od in (torch.float16, torch.float32):
            for off, ld in ((0, H * D), (4, H * D + 4), (2, H * D + 6)):  # whole rows, 4-element and pair stores
                buf = torch.full((Tq * ld + off + 8,), float("nan"), dtype=od, device=DEV)
                out = buf[off:off + Tq * ld].view(Tq, ld)[:, :H * D]
                kiln_amd.attn_prepped(out, qd, kvp, Tk, H, npad=npad)
                torch.cuda.synchronize()
                assert_close(out.float().cpu().numpy(), ref, f"H={H} Tq={Tq} Tk={Tk} npad={npad} {qd.dtype} {od} ld={ld}")
                if ld > H * D:
                    assert torch.isnan(buf[off:off + Tq * ld].view(Tq, ld)[:, H * D:]).all()
                assert torch.isnan(buf[:off]).all() and torch.isnan(buf[off + Tq * ld:]).all()


def _form(T, Tk, units):
    """The kernel form of a launch (waves x query rows of a wave) by the launcher's rule, units = items x heads."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    u64, u128, t8 = ((T + n - 1) // n * units for n in (64, 128, 256))
    if t8 % cus == 0 or (Tk >= 2048 and t8 >= cus):
        return "8x32"
    return "4x16" if u64 <= cus else "8x16" if u128 <= cus else "4x32"


@pytest.mark.parametrize("T,alone,four_items", [(700, "4x16", "4x32"), (1000, "4x16", "8x32"), (1100, "8x16", "4x32"),
                                                (1536, "8x16", "4x32"), (2048, "8x16", "8x32")])
def test_forms_agree_bit_for_bit(gpu, T, alone, four_items):
    """One item (64- or 128-row units of 16-row waves) against the same item in a batch of four (32-row waves, 4 or 8 of
    them), with maxima that move late in the row, so that rows of one wave rescale at different steps."""
    assert (_form(T, T, 16), _form(T, T, 64)) == (alone, four_items)
    H = 16
    g = torch.Generator(device=DEV).manual_seed(T)
    q, k, v = (torch.randn(T, H * D, device=DEV, generator=g) for _ in range(3))
    k *= torch.linspace(0.5, 4, T, device=DEV)[torch.randperm(T, device=DEV, generator=g)][:, None]
    q, k, v = q.half(), k.half(), v.half()
    kvp = kiln_amd.kv_prepare(k, v, H)
    one, four = torch.empty_like(q), torch.empty(4 * T, H * D, dtype=torch.float16, device=DEV)
    kiln_amd.attn_prepped(one, q, kvp, T, H)
    kiln_amd.attn_prepped_batch(four, q.repeat(4, 1), [kvp] * 4, T, T, H)
    for b in range(4):
        assert torch.equal(one, four[b * T:(b + 1) * T]), f"item {b}"


def test_chain_of_contexts(gpu):
    """T = 1536, three contexts: one 128-row unit per tile and head runs them in turn (192 units of 16-row waves),
    against one context at a time."""
    T, H, B, reals = 1536, 16, 2, [77, 23, 41]
    g = torch.Generator(device=DEV).manual_seed(9)
    q = torch.randn(B * T, H * D, device=DEV, generator=g).half()
    w = (1 + 0.2 * torch.randn(D, device=DEV, generator=g)).bfloat16()
    kvps = [kiln_amd.kv_prepare(*(torch.randn(r, H * D, device=DEV, generator=g).half() for _ in range(2)), H) for r in reals]
    npads = [512 - r for r in reals]
    out, neg = torch.empty_like(q), torch.empty(T, H * D, dtype=torch.float16, device=DEV)
    kiln_amd.cross_attn_nag(out, q, B, T, H, kvps[:2], reals[:2], npads[:2], q_norm_w=w, kvp_neg=kvps[2], Lk_neg=reals[2],
                            npad_neg=npads[2], out_neg=neg)
    single = [torch.empty(T, H * D, dtype=torch.float16, device=DEV) for _ in range(3)]
    for i, qi in enumerate((q[:T], q[T:], q[:T])):
        kiln_amd.attn_prepped(single[i], qi, kvps[i], reals[i], H, npad=npads[i], q_norm_w=w)
    assert torch.equal(neg, single[2]) and torch.equal(out[T:], single[1])
    kiln_amd.nag_combine(single[0], single[2])
    assert torch.equal(out[:T], single[0])


@pytest.mark.parametrize("causal", [False, True])
def test_exact_forms_agree_bit_for_bit(gpu, causal):
    """Exact fp32 attention of 2100 rows (128-row workgroups) against its first 500 rows alone (64-row ones)."""
    H, T, Tk = 16, 2100, 130
    g = torch.Generator(device=DEV).manual_seed(4)
    q, k, v = (torch.randn(t, H * D, device=DEV, generator=g) for t in (T, Tk, Tk))
    a, b = torch.empty_like(q), torch.empty(500, H * D, device=DEV)
    kiln_amd.attention_exact(a, q, k, v, T, Tk, H, D, causal=causal, npad=3)
    kiln_amd.attention_exact(b, q[:500], k, v, 500, Tk, H, D, causal=causal, npad=3)
    assert torch.equal(a[:500], b)
    ref = oracle.attn_f64(q[:64].cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), H, npad=3, causal=causal)
    assert_close(b[:64].cpu().numpy(), ref, "exact", max_abs=1e-5, mean_abs=1e-6)
