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


@pytest.mark.parametrize("rows,columns,K,heads,gap,dtype,tile", [
    (16, 128, 512, 16, 0, torch.bfloat16, 16), (512, 128, 512, 16, 0, torch.bfloat16, 16), (513, 128, 512, 16, 0, torch.bfloat16, 64),
    (256, 128, 320, 32, 0, torch.bfloat16, 64), (192, 128, 320, 32, 0, torch.bfloat16, 16), (512, 128, 512, 16, 4, torch.bfloat16, 64),
    (256, 128, 192, 32, 0, torch.bfloat16, 16), (17, 128, 128, 1, 0, torch.float32, 64)])
def test_tiles_of_products_per_head(rows, columns, K, heads, gap, dtype, tile):
    x, w = torch.zeros(1, heads * (K + gap), dtype=dtype), torch.zeros(heads, columns, K, dtype=dtype)
    assert ops._grouped_tile(rows, columns, heads, ops.Strided(x, 0, K + gap), w) == tile
