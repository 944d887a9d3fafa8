"""How products of few rows are cut into items (no GPU: the library only answers): one piece of a residual epilogue an item."""
import pytest

from lucciola_amd.kernels import ops


# few tiles: items of 16 rows where K is short, an item for every CU (of four rows at least) from 768 on
@pytest.mark.parametrize("rows,columns,K,items", [(1, 1024, 128, 64), (8, 1024, 512, 64), (1, 200, 128, 13), (16, 512, 512, 32), (1, 1024, 768, 256),
                                                  (8, 1024, 3072, 256), (3, 200, 1024, 50), (1, 2048, 2048, 256)])
def test_items_of_few_tiles(rows, columns, K, items):
    assert ops.library().lc_gemm_bf16_residual_pieces(rows, columns, K) == items
