"""Latent attention of lone tokens over rows of 512 + 64 entries (``csrc/latent_lone.hip``) against float64: shares of one and of many
stages, windows, pages of every size, heads that fill a group of 16 and that do not, sinks, and shares that hold nothing."""
import pytest
import torch

from lucciola_amd.engine.batch import HostLayout, Plan
from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
RANK, ROT = 512, 64


@pytest.mark.parametrize("heads,page,window,with_sink,contexts", [
    (16, 16, 0, False, [1, 15, 16, 17, 33, 64, 65, 300]), (1, 4, 0, True, [130]), (17, 48, 100, True, [90, 100, 101, 400, 7]),
    (32, 16, 0, False, [2500]), (5, 2, 40, False, [39, 40, 41, 1000]), (16, 16, 0, True, [600] * 300)])
def test_lone_tokens(heads, page, window, with_sink, contexts):
    g = torch.Generator().manual_seed(heads * 100 + page)
    T = len(contexts)
    each = [-(-n // page) for n in contexts]
    cache = (torch.randn(sum(each) + 1, page, RANK + ROT, generator=g) * 0.5).bfloat16().to(DEV)
    order = torch.randperm(sum(each), generator=g) + 1
    table = torch.full((T, max(each) + 2), -1, dtype=torch.int32)
    at = 0
    for r, n in enumerate(each):
        table[r, :n] = order[at:at + n]
        at += n
        if window:          # pages behind the window have gone back
            table[r, :max(0, contexts[r] - window) // page] = -1
    qa = (torch.randn(T, heads * (RANK + ROT), generator=g) * 0.6).bfloat16().to(DEV)
    sink = (torch.randn(heads, generator=g) * 2).to(DEV) if with_sink else None
    layout = HostLayout(T, T, list(range(T + 1)), [n - 1 for n in contexts], page, True)
    arrays, info = ops.plan_latent_attention(layout)
    plan = Plan({k: torch.tensor(v, device=DEV) for k, v in arrays.items()}, info)
    positions = torch.tensor([n - 1 for n in contexts], dtype=torch.int32, device=DEV)
    scale, got = (RANK + ROT) ** -0.5 * 3.0, {}
    for on in (1, 0):
        before = ops.library().lc_latent_lone(on)
        try:
            got[on] = ops.latent_attention(qa, heads, RANK, ROT, torch.arange(T, dtype=torch.int32, device=DEV), positions,
                                           table.to(DEV), cache, page, scale, window, plan=plan, max_ctx=max(contexts), sink=sink).double()
        finally:
            ops.library().lc_latent_lone(before)
    for r, n in enumerate(contexts):
        first = max(0, n - window) if window else 0
        slots = [int(table[r, j // page]) * page + j % page for j in range(first, n)]
        rows = cache.view(-1, RANK + ROT)[slots].double()
        s = qa[r].view(heads, -1).double() @ rows.T * scale
        top = s.max(1, keepdim=True).values
        more = 0.0
        if with_sink:
            top = torch.maximum(top, sink.double()[:, None])
            more = torch.exp(sink.double()[:, None] - top)
        e = torch.exp(s - top)
        want = e @ rows[:, :RANK] / (e.sum(1, keepdim=True) + more)
        # the weights and the result are rounded to bfloat16: 2^-9 each of the largest entry
        bound = 2 * 2.0 ** -9 * float(rows.abs().max())
        for on in (1, 0):
            mine = got[on][r].view(heads, RANK)
            assert float((mine - want).abs().max()) <= bound, (on, r)
            assert float((mine - want).norm() / want.norm()) <= 2.0 ** -8, (on, r)
