"""How many pages the cache gets of a card's free memory: a step's scratch for the cached tokens that it reads has room."""
import pytest

from lucciola_amd.config.engine_config import EngineConfig
from lucciola_amd.engine.runner import blocks_from_free_memory
from lucciola_amd.kernels import ops
from lucciola_amd.parts.base import Part

GB = 1 << 30
PAGE = 16
ROW = 2 * (512 + 64 + 16 * 256)         # 16 heads of 128 and 128 over a latent of 512 + 64
MOST = (1 << 28) // (16 * 128) * ROW


def test_what_the_latent_part_states():
    assert ops.latent_wide_scratch(16, 512, 64, 128, 128) == (ROW, MOST)
    assert Part().step_scratch() == (0, 0)


@pytest.mark.parametrize("free", [600 << 20, 2 * GB, 8 * GB, 280 * GB])
@pytest.mark.parametrize("fraction", [1.0, 0.99, 0.9, 0.5])
@pytest.mark.parametrize("page_bytes", [1 << 16, 3 << 20])
def test_the_scratch_fits_beside_the_pages(free, fraction, page_bytes):
    config = EngineConfig(block_size=PAGE, memory_fraction=fraction)
    plain = blocks_from_free_memory(free, page_bytes, 0, config)
    blocks = blocks_from_free_memory(free, page_bytes, 0, config, scratch=(ROW, MOST))
    room = free - config.memory_reserve
    scratch = min(MOST, blocks * PAGE * ROW)            # no step sees more rows than the pages hold
    assert blocks * page_bytes + scratch <= room
    # nothing is kept back that the fraction leaves free anyway, and never more than is wanted
    if plain * page_bytes + MOST <= room:
        assert blocks == plain
    assert (plain - blocks) * page_bytes <= min(scratch + PAGE * ROW, MOST) + page_bytes
