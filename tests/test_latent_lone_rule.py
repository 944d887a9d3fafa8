"""Which steps of lone tokens take ``csrc/latent_lone.hip`` and into how many shares their rows go (no GPU: the library only answers)."""
import pytest

from lucciola_amd.kernels import ops


@pytest.mark.parametrize("heads,tiles,rows,lone", [
    (16, 64, 2047, True), (16, 64, 500, True), (16, 8, 300, False), (16, 1, 20, False), (16, 1, 8000, True), (16, 200, 100, False),
    (1, 1, 300, True), (8, 8, 2047, True), (8, 8, 20, False), (32, 200, 300, True), (32, 100, 100, False), (64, 64, 2047, True),
    (64, 256, 2000, False), (128, 100, 1000, True), (128, 200, 300, False), (48, 8, 1400, True), (48, 32, 2000, False), (96, 16, 2000, False)])
def test_steps_that_gain(heads, tiles, rows, lone):
    assert bool(ops.library().lc_latent_lone_picks(512, 64, heads, tiles, rows)) == lone
    assert not ops.library().lc_latent_lone_picks(256, 64, heads, tiles, rows)


# 256 CUs: shares that fill one round, or whole rounds, and never one workgroup more; at least a stage of 16 rows a wave
@pytest.mark.parametrize("workgroups,rows,shares", [(64, 2047, 4), (8, 2047, 32), (1, 30000, 59), (24, 2000, 8), (256, 2047, 1), (8, 300, 5), (1, 16, 1),
                                                    (200, 64, 1), (1024, 2000, 1), (800, 1000, 1)])
def test_shares(workgroups, rows, shares):
    assert ops.library().lc_latent_lone_splits(workgroups, rows) == shares
