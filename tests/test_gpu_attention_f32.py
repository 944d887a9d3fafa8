"""float32 attention on the matrix instruction (``csrc/attention_f32.hip``): heads, groups, pages and windows at the edges of its columns,
units of 16 keys and spans of 512, the same bits however rows and spans are shared out, and values that are not finite."""
import pytest
import torch

import reference_ops as ref
from lucciola_amd.kernels import ops
from lucciola_amd.kernels.ops import AttentionBatch
from test_gpu_kernels import DEV, close, paged_case

pytestmark = pytest.mark.gpu


def run(qkv, batch, kc, vc, nh, nkv, d, page, window, rows=0):
    ops.library().lc_attention_generic_rows(rows)
    try:
        return ops.attention(qkv, batch, kc, vc, nh, nkv, d, page, d ** -0.5, window)
    finally:
        ops.library().lc_attention_generic_rows(0)


@pytest.mark.parametrize("nh,nkv,d,page,window", [
    (1, 1, 16, 4, 0), (3, 1, 32, 12, 0), (10, 2, 48, 20, 17), (16, 2, 64, 16, 0), (16, 1, 80, 64, 500), (17, 1, 96, 16, 0),
    (40, 2, 112, 16, 33), (8, 2, 128, 4, 513), (2, 2, 128, 32, 1)])
def test_edges(nh, nkv, d, page, window):
    lengths, new = [1, 16, 511, 513, 700, 31, 1100], [1, 3, 1, 20, 33, 31, 2]
    qkv, batch, kc, vc = paged_case(lengths, new, nh, nkv, d, page, torch.float32, seed=nh + d)
    assert ops.library().lc_attention_f32_takes(ops._ptr(qkv), qkv.shape[1], ops._ptr(kc), ops._ptr(vc), nh, nkv, d, page) == 1
    got = run(qkv, batch, kc, vc, nh, nkv, d, page, window)
    plain = AttentionBatch(batch.tok_req.cpu(), batch.positions.cpu(), batch.block_table.cpu())
    want = ref.attention(qkv.cpu().double(), plain, kc.cpu().double(), vc.cpu().double(), nh, nkv, d, page, d ** -0.5, window)
    close(got, want, torch.float32)
    assert torch.equal(run(qkv, batch, kc, vc, nh, nkv, d, page, window, rows=1), got)
    assert torch.equal(run(qkv, batch, kc, vc, nh, nkv, d, page, window, rows=4), got)
    # lone tokens among the portions' rows, all tokens lone (each with a workgroup of its own), and the same rows as anybody's
    alone = [r for r, n in enumerate(new) if n == 1]
    for which in (alone, list(range(len(lengths)))):
        mixed, its, k2, v2 = paged_case(lengths, [1 if r in which else n for r, n in enumerate(new)], nh, nkv, d, page, torch.float32, seed=nh + d)
        assert torch.equal(k2, kc) and its.num_decode == sum(1 for r, n in enumerate(new) if n == 1 or r in which)
        listed = run(mixed, its, kc, vc, nh, nkv, d, page, window)
        assert torch.equal(listed, run(mixed, its, kc, vc, nh, nkv, d, page, window, rows=1))
        assert torch.equal(listed, run(mixed, its, kc, vc, nh, nkv, d, page, window, rows=4))
    # enough rows that a workgroup works through all spans of its own
    times = -(-2048 // qkv.shape[0])
    many = AttentionBatch(batch.tok_req.repeat(times), batch.positions.repeat(times), batch.block_table)
    for rows in (1, 4):
        assert torch.equal(run(qkv.repeat(times, 1), many, kc, vc, nh, nkv, d, page, window, rows=rows), got.repeat(times, 1))


@pytest.mark.parametrize("nh,nkv", [(2, 2), (4, 1), (6, 2), (17, 1)])
@pytest.mark.parametrize("lengths,new", [([2] * 30, [2] * 30), ([600, 3, 40, 520] * 3, [3] * 12), ([50, 9, 700], [2, 9, 1]), ([5] * 9, [1, 2, 3] * 3)])
def test_short_portions(nh, nkv, lengths, new):
    """A workgroup takes as many rows as a portion has on average: the same bits as row by row and as with all that it has room for."""
    d, page = 32, 16
    qkv, batch, kc, vc = paged_case(lengths, new, nh, nkv, d, page, torch.float32, seed=nh)
    got = run(qkv, batch, kc, vc, nh, nkv, d, page, 0)
    plain = AttentionBatch(batch.tok_req.cpu(), batch.positions.cpu(), batch.block_table.cpu())
    close(got, ref.attention(qkv.cpu().double(), plain, kc.cpu().double(), vc.cpu().double(), nh, nkv, d, page, d ** -0.5, 0), torch.float32)
    for rows in (1, 4):
        assert torch.equal(run(qkv, batch, kc, vc, nh, nkv, d, page, 0, rows=rows), got)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("window", [0, 9])
def test_a_value_that_is_not_finite_reaches_only_who_sees_it(bad, window):
    nh, nkv, d, page, length, at = 4, 2, 64, 16, 60, 37
    qkv, batch, kc, vc = paged_case([length], [length], nh, nkv, d, page, torch.float32, seed=5)
    clean = run(qkv, batch, kc, vc, nh, nkv, d, page, window, rows=4)
    vc[batch.block_table[0, at // page].item(), 1, 7, at % page] = bad
    vc[batch.block_table[0, (length - 1) // page].item(), :, :, length % page:] = bad          # behind the last token: another's, once
    got = run(qkv, batch, kc, vc, nh, nkv, d, page, window, rows=4)
    sees = torch.zeros(length, nh, d, dtype=torch.bool, device=DEV)
    sees[at:at + window if window else length, 2:, 7] = True
    sees = sees.view(length, nh * d)
    assert torch.equal(got[~sees], clean[~sees])
    assert not torch.isfinite(got[sees]).any()


@pytest.mark.parametrize("spoilt", [(16, 32), (0, 16), (48, 60), (512, 1024), (530, 531)])
@pytest.mark.parametrize("rows", [1, 4])
def test_keys_that_are_not_a_number_are_not_passed_by(spoilt, rows):
    """All keys that a wave (of a unit of 16) or a workgroup (of a span of 512) sees are NaN: their scores leave no maximum, and the query that
    sees them gets NaN and not the other keys' mean."""
    nh, nkv, d, page, length = 4, 2, 32, 16, 60 if spoilt[1] <= 60 else 1100
    qkv, batch, kc, vc = paged_case([length], [length if length < 100 else 700], nh, nkv, d, page, torch.float32, seed=9)
    clean = run(qkv, batch, kc, vc, nh, nkv, d, page, 0, rows=rows)
    for j in range(*spoilt):
        kc[batch.block_table[0, j // page].item(), 1, j % page] = float("nan")
    got = run(qkv, batch, kc, vc, nh, nkv, d, page, 0, rows=rows)
    sees = torch.zeros(qkv.shape[0], nh, d, dtype=torch.bool, device=DEV)
    sees[batch.positions >= spoilt[0], 2:] = True
    sees = sees.view(got.shape)
    assert torch.equal(got[~sees], clean[~sees])
    assert torch.isnan(got[sees]).all()
    # lone tokens, their spans shared out
    alone, last, k2, v2 = paged_case([length], [1], nh, nkv, d, page, torch.float32, seed=9)
    got = run(qkv[-1:].contiguous(), last, kc, vc, nh, nkv, d, page, 0)
    assert torch.isnan(got[0, 2 * d:]).all() and torch.isfinite(got[0, :2 * d]).all()
