"""Which of the grouped products' kernels serves what (no GPU: the library only answers): on both sides of each line of the rule
sizes at which one of the two was measured to be the faster."""
import pytest
import torch

from lucciola_amd.kernels import ops


@pytest.mark.parametrize("tile,rows,columns,K,heads,tiled", [
    (16, 8, 512, 128, 16, True), (16, 64, 512, 128, 16, True), (16, 64, 512, 128, 32, False), (16, 64, 512, 256, 32, True),
    (16, 64, 512, 192, 16, False), (16, 2048, 128, 512, 4, True),
    (64, 160, 512, 64, 16, False), (64, 1024, 512, 64, 16, False), (64, 160, 512, 128, 16, False), (64, 512, 512, 128, 32, False),
    (64, 2048, 512, 128, 16, True), (64, 2048, 192, 128, 16, False), (64, 160, 512, 192, 16, False), (64, 2048, 64, 256, 16, False),
    (64, 2048, 128, 256, 16, True), (64, 160, 512, 512, 16, True), (64, 2048, 128, 512, 16, True), (64, 2048, 128, 520, 16, False)])
def test_products_per_head(tile, rows, columns, K, heads, tiled):
    assert bool(ops.library().lc_gemm_grouped_picks_tiled(tile, rows, columns, K, heads, 0)) == tiled


@pytest.mark.parametrize("tile,tokens,top,experts,columns,K,tiled", [
    (16, 4, 4, 32, 2048, 128, True), (16, 100, 4, 32, 2048, 128, False), (16, 100, 8, 128, 2048, 256, False), (16, 8, 4, 32, 2048, 2048, True),
    (16, 64, 4, 32, 6144, 4096, True), (64, 400, 4, 32, 512, 128, False), (64, 100, 2, 8, 512, 256, False), (64, 2048, 8, 128, 2048, 384, True),
    (64, 400, 2, 8, 512, 384, False), (64, 300, 4, 32, 2048, 2048, True), (128, 2048, 4, 32, 512, 256, True), (128, 2048, 4, 32, 2048, 128, False),
    (128, 2048, 2, 8, 2048, 256, False), (128, 2048, 4, 32, 2048, 2048, True)])
def test_experts(tile, tokens, top, experts, columns, K, tiled):
    rows = tokens * top
    assert bool(ops.library().lc_gemm_grouped_picks_tiled(tile, rows, columns, K, experts, rows // tile + experts)) == tiled


@pytest.mark.parametrize("experts,columns,K,tiled", [
    (96, 128, 128, True), (128, 128, 128, False), (128, 128, 160, False), (128, 128, 192, True), (128, 129, 192, False), (8, 2048, 128, True),
    (48, 512, 128, True), (64, 512, 128, False)])
def test_experts_of_a_short_k(experts, columns, K, tiled):
    rows = experts * 200 // 4 * 4
    assert bool(ops.library().lc_gemm_grouped_picks_tiled(128, rows, columns, K, experts, rows // 128 + experts)) == tiled


# lists for tiles of 64 rows: one workgroup of 64 x 128 a CU and fewer, more of them, w so large that memory counts, a short K
@pytest.mark.parametrize("rows,experts,columns,K,even", [
    (400, 4, 1024, 2048, False), (1520, 8, 1024, 4096, False), (1600, 16, 1024, 2048, False), (800, 4, 512, 1024, False), (2240, 16, 768, 2048, True),
    (6080, 32, 1024, 2048, True), (140, 1, 512, 2048, False), (640, 32, 1024, 2048, True), (640, 32, 1024, 1024, False), (1280, 64, 1024, 1024, False), (480, 24, 2048, 1024, True),
    (1280, 64, 1024, 2048, True), (6080, 32, 511, 2048, False), (6080, 32, 1024, 960, False), (8960, 64, 512, 1024, True), (8960, 64, 2048, 1024, True)])
def test_even_tiles(rows, experts, columns, K, even):
    assert bool(ops.library().lc_gemm_grouped_picks_even(64, rows, columns, K, experts, 0)) == even


@pytest.mark.parametrize("rows,experts,I,K,fused", [
    (1120, 8, 512, 2048, False), (560, 4, 256, 2048, False), (320, 16, 1024, 1024, True), (1280, 64, 512, 1024, True), (2240, 16, 512, 2048, True),
    (8960, 64, 256, 2048, True), (8960, 64, 128, 2048, False)])
def test_gated_experts(rows, experts, I, K, fused):
    assert bool(ops.library().lc_gemm_grouped_picks_even(64, rows, I, K, experts, 1)) == fused


@pytest.mark.parametrize("rows,columns,K,heads,gap,dtype,tile", [
    (16, 128, 512, 16, 0, torch.bfloat16, 16), (512, 128, 512, 16, 0, torch.bfloat16, 16), (513, 128, 512, 16, 0, torch.bfloat16, 64),
    (256, 128, 320, 32, 0, torch.bfloat16, 64), (192, 128, 320, 32, 0, torch.bfloat16, 16), (512, 128, 512, 16, 4, torch.bfloat16, 64),
    (256, 128, 192, 32, 0, torch.bfloat16, 16), (17, 128, 128, 1, 0, torch.float32, 64)])
def test_tiles_of_products_per_head(rows, columns, K, heads, gap, dtype, tile):
    x, w = torch.zeros(1, heads * (K + gap), dtype=dtype), torch.zeros(heads, columns, K, dtype=dtype)
    assert ops._grouped_tile(rows, columns, heads, ops.Strided(x, 0, K + gap), w) == tile
