"""GPU parity of the fp32 linear layers with bf16 weights (kiln_linear_f32) on the bf16 matrix cores, where an fp32
input is split into three bf16 parts without a remainder: every tile, its edges, and values at the ends of fp32.

Bar: fp32 sums of exact products, |err| <= sqrt(cols) 2^-21 sum_k |x_k w_k| (the bar of the fp16 GEMM's fp32 sums).
"""
import numpy as np
import pytest
import torch

import kiln_amd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# the five tiles: (weight rows, rows of x), and a shape that each takes
TILES = [((256, 128), (2049, 2050, 96)), ((128, 128), (1025, 2048, 64)), ((128, 64), (500, 2050, 64)),
         ((128, 32), (96, 128, 64)), ((64, 32), (33, 70, 2080))]


def _check(y, x, w, what=""):
    ref = x.double() @ w.double().T
    bar = w.shape[1] ** 0.5 * 2.0 ** -21 * (x.double().abs() @ w.double().abs().T) + 1e-44
    err = (y.double() - ref).abs()
    assert torch.isfinite(y).all(), what
    assert (err <= bar).all(), f"{what}: {(err / bar).max().item():.2f} of the bar"


# the five tiles (256 x 128, 128 x 128, 128 x 64, 128 x 32, 64 x 32), a row over and under an edge, rows that end
# inside a tile and inside a group of four columns, a partial last step of 2, 4 or 8 slices
@pytest.mark.parametrize("T,rows,cols", [(4097, 2048, 96), (2047, 2048, 352), (1025, 2048, 160), (500, 2050, 288), (65, 129, 64),
                                         (33, 64, 2080), (1, 3, 32), (1, 3, 96), (4097, 520, 32), (6912, 64, 256), (31, 2048, 1056)])
def test_linear_f32_tiles(gpu, T, rows, cols):
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, cols, device=DEV, generator=g)
    w = (torch.randn(rows, cols, device=DEV, generator=g) * cols ** -0.5).bfloat16()
    buf = torch.full((T + 2, rows + 1), float("nan"), device=DEV)  # an odd row stride: element stores
    for y in (torch.full((T, rows), float("nan"), device=DEV), buf[1:T + 1, :rows]):
        kiln_amd.linear_f32(y, x, w)
        _check(y, x, w)
    assert torch.isnan(buf[0]).all() and torch.isnan(buf[T + 1]).all() and torch.isnan(buf[:, rows]).all()
    wide = torch.randn(T, cols + 4, device=DEV, generator=g)[:, :cols]  # a row stride of its own
    kiln_amd.linear_f32(buf[1:T + 1, :rows], wide, w)
    _check(buf[1:T + 1, :rows], wide, w)


@pytest.mark.parametrize("tile,shape", TILES)
@pytest.mark.parametrize("exp", [-149, -140, -126, -118, -110, -60, 0, 60, 103, 104, 127])
def test_linear_f32_split_is_exact(gpu, tile, shape, exp):
    """A weight with a single 1 in each row picks values of x out: every bit of their 24 has to come through the parts,
    at both ends of fp32 too (2^-149: subnormal values; 2^104 and up are past the range of the scaled sums)."""
    T, rows, cols = shape
    g = torch.Generator(device=DEV).manual_seed(5)
    n = torch.randint(2 ** 23, 2 ** 24, (T, cols), device=DEV, generator=g) | 1
    x = torch.ldexp(n.double(), torch.tensor(exp - 23, device=DEV)).float()  # subnormal: fewer bits, rounded here
    x *= 1 - 2 * torch.randint(0, 2, (T, cols), device=DEV, generator=g).float()
    pick = torch.randint(0, cols, (rows,), device=DEV, generator=g)
    w = torch.zeros(rows, cols, device=DEV).index_put_((torch.arange(rows, device=DEV), pick), torch.tensor(1.0, device=DEV)).bfloat16()
    assert kiln_amd.linear_f32_tile(x, w) == tile
    y = torch.empty(T, rows, device=DEV)
    kiln_amd.linear_f32(y, x, w)
    assert torch.equal(y, x[:, pick]), f"{(y != x[:, pick]).sum().item()} of {y.numel()} differ"


@pytest.mark.parametrize("exp", [-126, -127, -130, -133])
def test_linear_f32_subnormal_weights(gpu, exp):
    """bf16 weights at and below 2^-126: the matrix cores take a subnormal's significand as it stands and align its products by
    the exponent, so that up to 7 leading zeros (at 2^-133) cost as many of the sum's 24 bits."""
    g = torch.Generator(device=DEV).manual_seed(8)
    x = torch.ldexp((torch.randint(2 ** 23, 2 ** 24, (96, 128), device=DEV, generator=g) | 1).float(), torch.tensor(40, device=DEV))
    w = torch.zeros(128, 128, device=DEV).fill_diagonal_(2.0 ** exp).bfloat16()
    y = torch.empty(96, 128, device=DEV)
    assert kiln_amd.linear_f32_tile(x, w) is not None
    kiln_amd.linear_f32(y, x, w)
    ref = x.cpu().double() * 2.0 ** exp
    assert ((y.cpu().double() / ref - 1).abs() <= (0 if exp >= -126 else 2.0 ** -16)).all()


@pytest.mark.parametrize("scale", [2.0 ** -120, 2.0 ** -100, 2.0 ** -20, 2.0 ** 100, 2.0 ** 116])
def test_linear_f32_scales(gpu, scale):
    """Far from 1 too the sums are as good as fp32's."""
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(70, 256, device=DEV, generator=g) * scale
    w = torch.randn(130, 256, device=DEV, generator=g).bfloat16()
    y = torch.empty(70, 130, device=DEV)
    kiln_amd.linear_f32(y, x, w)
    _check(y, x, w)


@pytest.mark.parametrize("tile,shape", TILES)
def test_linear_f32_infinities_and_nan(gpu, tile, shape):
    """The same non-finite outputs as the general form (x one float off its alignment takes it), and every finite output
    within the bar of its own terms, those beside the recomputed ones too."""
    T, rows, cols = shape
    g = torch.Generator(device=DEV).manual_seed(2)
    buf = torch.randn(T * cols + 1, device=DEV, generator=g)
    x = buf[1:].view(T, cols)
    w = torch.randn(rows, cols, device=DEV, generator=g).bfloat16()
    x[3, 5], x[7, 0], x[9, 63], x[11, 1] = float("inf"), float("-inf"), float("nan"), 0.0
    x[T - 1, cols - 1] = float("inf")
    x[20] = 1.0  # no remainders
    w[4, 7], w[6, 1], w[8, 2], w[8, 3] = float("inf"), float("-inf"), float("nan"), 0.0
    w[rows - 1, cols - 2] = float("-inf")
    x[30, 9] = 3.4e38
    ya, yb = torch.empty(T, rows, device=DEV), torch.empty(T, rows, device=DEV)
    xb = x.clone()
    assert kiln_amd.linear_f32_tile(x, w) is None and kiln_amd.linear_f32_tile(xb, w) == tile
    kiln_amd.linear_f32(ya, x, w)
    kiln_amd.linear_f32(yb, xb, w)
    a, b = ya.cpu().numpy(), yb.cpu().numpy()
    assert (np.isnan(a) == np.isnan(b)).all()
    assert (np.isposinf(a) == np.isposinf(b)).all() and (np.isneginf(a) == np.isneginf(b)).all()
    f = torch.isfinite(ya)
    xz, wz = (torch.nan_to_num(t.double(), nan=0.0, posinf=0.0, neginf=0.0) for t in (xb, w))
    ref, bar = xz @ wz.T, cols ** 0.5 * 2.0 ** -21 * (xz.abs() @ wz.abs().T)
    assert f.float().mean() > 0.7 and f[:, rows - 2].sum() >= T - 6
    for y in (ya, yb):
        assert ((y.double() - ref).abs() <= bar)[f].all()


def test_linear_f32_rows_past_two_gib(gpu):
    """64 weight rows of 35 MB: a tile of them is past the 32-bit offsets of the matrix-core form's weight reads, so the
    call takes the general form. The last rows would lack a third of their terms and more otherwise. One x in a thousand is
    not 0: sums of n <= 18 000 positive terms, whose relative error is at most n ulp (2^-23) however they are rounded."""
    cols = 17_500_000 // 32 * 32
    g = torch.Generator(device=DEV).manual_seed(6)
    x = torch.zeros(1, cols, device=DEV)
    x[:, ::1000] = torch.rand(1, (cols + 999) // 1000, device=DEV, generator=g)
    w = torch.rand(64, cols, device=DEV, generator=g, dtype=torch.bfloat16)
    y = torch.empty(1, 64, device=DEV)
    assert kiln_amd.linear_f32_tile(x, w) is None
    kiln_amd.linear_f32(y, x, w)
    ref = sum(w[:, c:c + 2 ** 20].double() @ x[0, c:c + 2 ** 20].double() for c in range(0, cols, 2 ** 20))
    assert ((y[0].double() / ref - 1).abs() <= 18000 * 2.0 ** -23).all()


def test_linear_f32_form_limits(gpu):
    """Which form a call takes at the edges of the matrix-core form's rule (nothing is launched)."""
    x, w = torch.empty(4, 96, device=DEV), torch.empty(8, 96, device=DEV, dtype=torch.bfloat16)
    t = lambda xp, ldx, wp, cols, T=4, rows=8: kiln_amd.lib().kiln_linear_f32_tile(xp, ldx, wp, T, rows, cols)  # noqa: E731
    px, pw = x.data_ptr(), w.data_ptr()
    assert t(px, 96, pw, 96) and t(px, 1 << 22, pw, (1 << 22) - 32)
    assert not t(px, 1 << 22, pw, 1 << 22)
    assert not t(px, 96, pw, 68) and not t(px, 98, pw, 96) and not t(px + 4, 96, pw, 96) and not t(px, 96, pw + 2, 96)
    # the smallest calls: one slice of k up to 2^21 outputs, two up to 64 weight rows or 4 rows of x
    assert not t(px, 32, pw, 32, 1024, 2048) and t(px, 32, pw, 32, 1025, 2048)
    assert not t(px, 64, pw, 64, 4096, 64) and not t(px, 64, pw, 64, 4, 2048)
    assert t(px, 64, pw, 64, 5, 65) and t(px, 96, pw, 96, 1, 1)
