"""Latent attention in tiles: every tile and every group of heads is served once, for few tiles and for those that are taken eight at a
time, with rows of tiles that are not full."""
import pytest
import torch

from lucciola_amd.engine.batch import HostLayout, Plan
from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
RANK, ROT, PAGE, WINDOW = 64, 32, 16, 40


@pytest.mark.parametrize("heads", [1, 5, 70])
@pytest.mark.parametrize("portions", [[16 * 62 + 5], [16 * 63 + 1], [16 * 64 + 9, 1], [700, 1, 380], [1] * 63, [1] * 71])
def test_every_tile(heads, portions):
    R, T = len(portions), sum(portions)
    g = torch.Generator(device=DEV).manual_seed(heads + T)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    history = [100 + 7 * r for r in range(R)]
    pages = [-(-(p + n) // PAGE) for p, n in zip(history, portions)]
    table, at = torch.zeros((R, max(pages)), dtype=torch.int32), 0
    for r, n in enumerate(pages):
        table[r, :n] = torch.arange(at, at + n)
        at += n
    cache, qa = rand(at, PAGE, RANK + ROT), rand(T, heads * (RANK + ROT))
    q_start = [0]
    for n in portions:
        q_start.append(q_start[-1] + n)
    tok = torch.tensor([r for r, n in enumerate(portions) for _ in range(n)], dtype=torch.int32, device=DEV)
    pos = torch.tensor([history[r] + i for r, n in enumerate(portions) for i in range(n)], dtype=torch.int32, device=DEV)
    arrays, info = ops.plan_latent_attention(HostLayout(R, T, q_start, history, PAGE, False))
    plan = Plan({k: torch.from_numpy(v).to(DEV) for k, v in arrays.items()}, info)
    scale = (RANK + ROT) ** -0.5
    got = ops.latent_attention(qa, heads, RANK, ROT, tok, pos, table.to(DEV), cache, PAGE, scale, WINDOW, plan=plan,
                               max_ctx=max(p + n for p, n in zip(history, portions))).double().view(T, heads, RANK)
    j = pos.long()[:, None] - torch.arange(WINDOW, device=DEV)          # the keys a token sees, all of them there
    slots = table.to(DEV).long()[tok.long()[:, None], j // PAGE] * PAGE + j % PAGE
    rows = cache.view(-1, RANK + ROT)[slots].double()
    weights = torch.softmax(torch.matmul(qa.view(T, heads, -1).double(), rows.transpose(1, 2).contiguous()) * scale, 2)
    want = torch.matmul(weights, rows[:, :, :RANK].contiguous())
    # weights rounded to bfloat16 (2^-9 each, and so their sum at most), the result once more
    assert float((got - want).abs().max()) <= 3 * 2.0 ** -9 * float(rows.abs().max())
