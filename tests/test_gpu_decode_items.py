"""The decode kernel started for the items that hold shares, and for the whole list, at every number of kv heads."""
import dataclasses

import pytest
import torch

from lucciola_amd.kernels import ops
from test_gpu_kernels import paged_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv", [(4, 1), (8, 2), (16, 4), (32, 8), (64, 16), (40, 40)])
@pytest.mark.parametrize("lengths", [[900, 30, 450, 700], [8000, 16, 500, 129, 4097, 3000, 7000, 6000], [3000] + [200] * 23])
def test_items(nh, nkv, lengths):
    d, page = 128, 16
    qkv, batch, kc, vc = paged_case(lengths, [1] * len(lengths), nh, nkv, d, page, torch.bfloat16, seed=nkv)
    rows = batch.decode_rows.cpu().numpy()
    order = sorted(range(len(lengths)), key=lambda r: -lengths[r])
    rows = rows[order].copy()
    items = ops._decode_items(rows, torch.tensor(sorted(lengths, reverse=True)).numpy(), nkv)
    launched = ops.decode_items_launched(items, nkv)
    batch = dataclasses.replace(batch, decode_rows=torch.from_numpy(rows).cuda(), decode_items=torch.from_numpy(items).cuda(),
                                decode_items_launched=launched)
    before = ops.decode_by_items("always")
    try:
        got = ops.attention(qkv, batch, kc, vc, nh, nkv, d, page, d ** -0.5, 0)
        whole = ops.attention(qkv, dataclasses.replace(batch, decode_items_launched=0), kc, vc, nh, nkv, d, page, d ** -0.5, 0)
        ops.decode_by_items(False)
        plain = ops.attention(qkv, batch, kc, vc, nh, nkv, d, page, d ** -0.5, 0)
    finally:
        ops.decode_by_items(before)
    assert torch.equal(got, whole)                  # items without shares do nothing
    # other shares of the same float32 sums, then bfloat16: a unit of the largest values' size at the most
    assert float((got.float() - plain.float()).abs().max()) <= 2.0 ** -7 * float(plain.float().abs().max())
