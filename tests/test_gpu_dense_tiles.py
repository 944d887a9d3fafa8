"""The dense bfloat16 products' tiles of 128 x 128 and 128 x 64 that have a CU to themselves, and tiles taken in strips."""
import pytest
import torch

from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu


def _operands(M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)
    return [torch.randn(s, K, device="cuda", generator=gen).to(torch.bfloat16) for s in (M, N)]


def _check(x, w, tile):
    """Both result types and the gated epilogue against float64, each with its own sizes' rounding: products of bfloat16 are exact in
    float32, a sum of K of them is off by less than K 2^-24 of the sum of their sizes, and bfloat16 rounds by 2^-9."""
    ops.force_gemm_tile(tile)
    try:
        got16, got32 = ops.gemm(x, w, torch.bfloat16), ops.gemm(x, w, torch.float32)
        fused = ops.gemm_swiglu(x, w[:w.shape[0] // 16 * 16]) if w.shape[0] >= 16 else None
    finally:
        ops.force_gemm_tile(-1)
    want, sizes = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    bound = sizes * x.shape[1] * 2.0 ** -24
    assert bool(((got32.double() - want).abs() <= bound).all())
    assert bool(((got16.double() - want).abs() <= bound + want.abs() * 2.0 ** -8).all())
    if fused is not None:
        def halves(t):
            blocks = t[:, :w.shape[0] // 16 * 16].view(x.shape[0], -1, 2, 8)
            return blocks[:, :, 0].reshape(x.shape[0], -1), blocks[:, :, 1].reshape(x.shape[0], -1)
        (g, u), (off_g, off_u) = halves(want), halves(bound)
        gated = g * torch.sigmoid(g) * u            # silu's slope is below 1.1
        assert bool(((fused.double() - gated).abs() <= gated.abs() * 2.0 ** -8 + 1.1 * (off_g * u.abs() + off_u * g.abs()) + 1e-6).all())


@pytest.mark.parametrize("tile", [13, 14])
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (65, 70, 128), (128, 64, 256), (129, 129, 384), (257, 300, 512),
                                   (1000, 520, 640), (100, 400, 2048)])
def test_one_a_cu(tile, M, N, K):
    _check(*_operands(M, N, K), tile)


@pytest.mark.parametrize("tile", [2, 3, 5, 7, 13, 14])
@pytest.mark.parametrize("M,N,K", [(1900, 1160, 256), (2700, 700, 128), (900, 4200, 128)])
def test_strips(tile, M, N, K):
    """Many tiles, their rows no whole number of strips."""
    _check(*_operands(M, N, K), tile)


def test_taken_by_size():
    """Portions whose products have no other shape that fills the CUs, on their own choice."""
    for M, N, K in ((2048, 2048, 2048), (1523, 2048, 4096), (1903, 1024, 3072)):
        assert ops.library().lc_gemm_bf16_tile(M, N, K, 0) in (13, 14)
        _check(*_operands(M, N, K), -1)


FINE = (2, 3, 4, 6, 9)      # tiles of products of 16 x 16, whose float32 results pass through LDS too


@pytest.mark.parametrize("tile", [*FINE, 11, 13])
@pytest.mark.parametrize("M,N", [(31, 8), (193, 392), (257, 264), (300, 1000)])
def test_stored_through_lds(tile, M, N):
    """Columns that are stored in pieces of 16 bytes are, to the bit, those of a product with one or four more, which is stored in pairs or one
    by one."""
    x, w = _operands(M, N + 16, 512)
    ops.force_gemm_tile(tile)
    try:
        for dtype, more in ((torch.bfloat16, 4), (torch.bfloat16, 1)) + ((torch.float32, 1), (torch.float32, 2)) * (tile in FINE):
            whole, other = ops.gemm(x, w[:N], dtype), ops.gemm(x, w[:N + more], dtype)
            assert torch.equal(whole, other[:, :N])
    finally:
        ops.force_gemm_tile(-1)


@pytest.mark.parametrize("tile", [*FINE, 0, 5, 7, 8, 10, 11, 12, 13, 14])
@pytest.mark.parametrize("M,N", [(31, 16), (193, 400), (300, 1008)])
@pytest.mark.parametrize("gated", [False, True])
def test_results_that_begin_anywhere(tile, M, N, gated):
    """Results that begin at a whole 16 bytes (through LDS, where the tile does that) and 8 bytes further on (from the registers): the same
    bits, plain and gated, and nothing stored beside them."""
    x, w = _operands(M, N, 256)
    width, got = N // 2 if gated else N, {}
    ops.force_gemm_tile(tile)
    ops.library().lc_gemm_bf16_force_shares(1)
    try:
        for dtype in (torch.bfloat16, torch.float32):
            for shift in (0, 8 // dtype.itemsize):
                room = torch.full((16 + M * width + 16,), 7.0, dtype=dtype, device="cuda")
                out = room[16 + shift:16 + shift + M * width]
                ops._call("lc_gemm_bf16", ops._ptr(x), ops._ptr(w), ops._ptr(out), ops._dt(out), M, N, 256, int(gated), None, ops._stream())
                assert bool((room[:16 + shift] == 7.0).all()) and bool((room[16 + shift + M * width:] == 7.0).all())
                got[dtype, shift > 0] = out.clone()
    finally:
        ops.force_gemm_tile(-1)
        ops.library().lc_gemm_bf16_force_shares(0)
    for dtype in (torch.bfloat16, torch.float32):
        assert torch.equal(got[dtype, False], got[dtype, True])
    want = x.double() @ w.double().T
    if gated:
        blocks = want.view(M, -1, 2, 8)
        g, u = blocks[:, :, 0].reshape(M, -1), blocks[:, :, 1].reshape(M, -1)
        want = g * torch.sigmoid(g) * u
    assert float((got[torch.bfloat16, False].double().view(M, width) - want).norm() / want.norm()) <= 2.0 ** -8


@pytest.mark.parametrize("tile", range(15))
def test_tiles_keep_their_operands_in_registers(tile):
    """A loop whose operands come by inline assembly may have none of them spilled: such a shape would not be taken."""
    assert ops.library().lc_gemm_bf16_tile_scratch(tile) == 0
