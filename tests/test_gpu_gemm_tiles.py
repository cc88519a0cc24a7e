"""The FP8 GEMM's output tiles (64 x 32 to 256 x 256, chosen by the output's size): each accumulates
an output's products in the same order, so a row of y does not depend on how many rows the call has,
and hence on the tile: the first m rows of a large call equal the call on m rows bit for bit, with
the options each epilogue has (residual, group maxima, q / k transform)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    code = lambda r: torch.randn(r, K, device="cuda", generator=g).mul_(60).to(torch.float8_e4m3fn).view(torch.uint8)  # noqa: E731
    sx = torch.rand(M, device="cuda", generator=g) * 0.01 + 1e-3
    sw = torch.rand(N, device="cuda", generator=g) * 0.01 + 1e-3
    return code(M), code(N), sx, sw


def _rows(m, x8, w8, sx, sw, res=None, gcols=0, ld=0):
    from flower_amd import _lib as L
    lb = L.load()
    K, N = x8.shape[1], w8.shape[0]
    ld = ld or N
    y = torch.full((m, ld), 7.0, dtype=torch.bfloat16, device="cuda")[:, :N]
    args = (x8.data_ptr(), m, K, w8.data_ptr(), N, sx.data_ptr(), m, sw.data_ptr(), N, y.data_ptr(), ld)
    if res is not None:
        rc = lb.flw_fp8_scaled_mm_residual(*args, res.data_ptr(), res.stride(0), L.stream_of(y))
    elif gcols:
        amax = torch.full((N // gcols,), -1, dtype=torch.int32, device="cuda")
        rc = lb.flw_fp8_scaled_mm_group_amax(*args, gcols, amax.data_ptr(), L.stream_of(y))
        L.check(rc, "group amax")
        want = y.float().abs().reshape(m, N // gcols, gcols).amax(dim=(0, 2)).view(torch.int32)
        assert torch.equal(amax, want), (m, N, K, gcols)
        return y
    else:
        rc = lb.flw_fp8_scaled_mm(*args, L.stream_of(y))
    L.check(rc, "mm")
    return y


# N = 1024: 33 rows take 64 x 32 tiles, 520 64 x 64, 1100 128 x 64, 2100 128 x 128, 4200 256 x 128 (K <
# 2048) or two 128 x 128 a compute unit, the whole 13000 the 256 x 256 tiles.
@pytest.mark.parametrize("K", [64, 128, 192, 384, 448, 640, 1024, 2112])
@pytest.mark.parametrize("opt", ["plain", "residual", "amax"])
def test_rows_do_not_depend_on_the_tile(K, opt):
    M, N = 13000, 1024
    x8, w8, sx, sw = _operands(M, N, K)
    res = torch.randn(M, N, device="cuda").to(torch.bfloat16) if opt == "residual" else None
    gcols = 256 if opt == "amax" else 0
    full = _rows(M, x8, w8, sx, sw, res, gcols)
    for m in (1, 32, 33, 512, 520, 1100, 2100, 4200):
        assert torch.equal(_rows(m, x8, w8, sx, sw, res, gcols), full[:m]), m


# Ragged N: 16-byte rows (1000), 8-byte rows (the direct epilogue; 1004 and an odd leading dimension).
@pytest.mark.parametrize("N,ld", [(1000, 0), (1004, 0), (1024, 1028), (8, 0), (68, 72)])
@pytest.mark.parametrize("K", [320, 512])
def test_ragged_columns(N, ld, K):
    M = 13000
    x8, w8, sx, sw = _operands(M, N, K)
    full = _rows(M, x8, w8, sx, sw, ld=ld)
    for m in (31, 513, 1101, 2049, 4099):
        assert torch.equal(_rows(m, x8, w8, sx, sw, ld=ld), full[:m]), m
    ref = (x8.view(torch.float8_e4m3fn)[:64].double() * sx[:64, None]) @ (
        w8.view(torch.float8_e4m3fn).double() * sw[:, None]).t().contiguous()
    d = (full[:64].double() - ref).abs()
    # one bf16 rounding step, and fp32 sums of 512 products
    assert (d <= 2.0 ** -7 * ref.abs() + 1e-3 * ref.pow(2).mean().sqrt()).all()


# Residual rows that 16-byte loads cannot take (N or the residual's row stride 4 mod 8): the epilogue
# without staging, on every ring tile and on the 256 x 256 tiles.
@pytest.mark.parametrize("N,rs", [(1004, 1004), (1024, 1028)])
@pytest.mark.parametrize("K", [320, 512])
def test_residual_of_8_byte_rows(N, rs, K):
    M = 13000
    x8, w8, sx, sw = _operands(M, N, K)
    res = torch.randn(M, rs, device="cuda").to(torch.bfloat16)[:, :N]
    full = _rows(M, x8, w8, sx, sw, res)
    for m in (31, 513, 1101, 2049, 4099):
        assert torch.equal(_rows(m, x8, w8, sx, sw, res), full[:m]), m
    for r in (slice(0, 64), slice(M - 64, M)):
        prod = (x8.view(torch.float8_e4m3fn)[r].double() * sx[r, None]) @ (
            w8.view(torch.float8_e4m3fn).double() * sw[:, None]).t().contiguous()
        ref = prod + res[r].double()
        # the product's and the sum's bf16 rounding, half a step each, and fp32 sums of 512 products
        bound = 2.0 ** -8 * (ref.abs() + 2 * prod.abs()) + 1e-3 * prod.pow(2).mean().sqrt()
        assert ((full[r].double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("gcols", [8, 64, 128])
def test_group_maxima_of_every_tile(gcols):
    x8, w8, sx, sw = _operands(13000, 1152, 256)
    for m in (5, 700, 1200, 2200, 4400, 13000):
        _rows(m, x8, w8, sx, sw, gcols=gcols)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_transform_epilogue_does_not_depend_on_the_tile(D):
    """q / k transform epilogue on 128 x 64, 128 x 128 (one and two a unit) and 256 x 256 tiles; a
    sequence of 50 positions, so positions wrap inside every tile."""
    from flower_amd import _lib as L
    from flower_amd.attention import RotaryEmbedding
    lb = L.load()
    M, T, N, K = 12000, 50, 1536, 256
    x8, w8, sx, sw = _operands(M, N, K)
    cos, sin = RotaryEmbedding(D, T).tables(T, torch.bfloat16, "cuda")
    outs = {}
    for m in (M, 50, 1500, 3000):
        y = torch.empty((m, N), dtype=torch.bfloat16, device="cuda")
        amax = torch.full((N // D,), -1, dtype=torch.int32, device="cuda")
        L.check(lb.flw_fp8_scaled_mm_qk_norm_rope_amax(
            x8.data_ptr(), m, K, w8.data_ptr(), N, sx.data_ptr(), m, sw.data_ptr(), N, y.data_ptr(), N, D, 1024, 1,
            1e-6, cos.data_ptr(), sin.data_ptr(), T, amax.data_ptr(), L.stream_of(y)), "transform")
        want = y.float().abs().reshape(m, N // D, D).amax(dim=(0, 2)).view(torch.int32)
        assert torch.equal(amax, want), m
        outs[m] = y
    for m, y in outs.items():
        assert torch.equal(y, outs[M][:m]), m


@pytest.mark.parametrize("K", [64, 128, 192, 448, 1024])
@pytest.mark.parametrize("N", [1024, 1004])
def test_w8a16_rows_do_not_depend_on_the_tile(N, K):
    """flw_fp8_linear (W8A16): 1020 rows take 64 x 64 tiles, 2000 128 x 64, 4100 128 x 128, all 16380
    (256 tiles of 256 x 256) the large ones; x with a row stride past K."""
    from flower_amd import _lib as L
    lb = L.load()
    M = 16380
    _, w8, _, sw = _operands(1, N, K)
    x = torch.randn(M, K + 8, device="cuda").to(torch.bfloat16)
    outs = {}
    for m in (M, 1, 63, 65, 1020, 2000, 4100):
        y = torch.full((m, N), 7.0, dtype=torch.bfloat16, device="cuda")
        L.check(lb.flw_fp8_linear(x.data_ptr(), m, K, K + 8, w8.data_ptr(), N, sw.data_ptr(), N, L.GEMM_W8A16,
                                  y.data_ptr(), N, None, 0, L.stream_of(y)), "w8a16")
        outs[m] = y
    for m, y in outs.items():
        assert torch.equal(y, outs[M][:m]), m
    ref = x[:64, :K].double() @ (w8.view(torch.float8_e4m3fn).double() * sw[:, None].double()).t().contiguous()
    d = (outs[M][:64].double() - ref).abs()
    assert (d <= 2.0 ** -7 * ref.abs() + 1e-3 * ref.pow(2).mean().sqrt()).all()
