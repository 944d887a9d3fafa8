"""Masked attention of tiles of several tokens on the matrix cores: walks of few, odd and many stages, across the 64 blocks whose pages a wave
holds at a time, with pages of one block and of three, and with kept keys before the window."""
import pytest
import torch

from lucciola_amd.engine.batch import HostLayout, Plan
from lucciola_amd.kernels import ops
from test_gpu_masked_order import DEV, near

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("page", [16, 48])
@pytest.mark.parametrize("window,keep", [(0, 0), (90, 0), (1200, 40)])
@pytest.mark.parametrize("heads,kv,maps,d,dv", [(4, 1, 1, 128, 128), (4, 1, 2, 64, 128), (2, 2, 1, 64, 64), (8, 1, 1, 48, 32), (4, 2, 2, 128, 64)])
def test_against_the_general_kernel(heads, kv, maps, d, dv, window, keep, page):
    history, fresh = [0, 15, 1000, 2050], [33, 2, 30, 17]       # 1 to 130 blocks: the 64th and the 128th in the middle of a tile's walk
    pages = [-(-(h + f) // page) for h, f in zip(history, fresh)]
    gen = torch.Generator().manual_seed(page + heads + d)
    order = torch.randperm(sum(pages), generator=gen).int()
    table, at = torch.zeros((4, max(pages)), dtype=torch.int32), 0
    for r, n in enumerate(pages):
        table[r, :n] = order[at:at + n]
        at += n
    rand = lambda *s: torch.randn(*s, generator=gen).to(DEV).bfloat16()
    kc, vc = rand(at, page, kv * maps * d), rand(at, kv * dv, page)
    starts = [0]
    for f in fresh:
        starts.append(starts[-1] + f)
    tok = torch.tensor([r for r, f in enumerate(fresh) for _ in range(f)], dtype=torch.int32, device=DEV)
    pos = torch.tensor([history[r] + i for r, f in enumerate(fresh) for i in range(f)], dtype=torch.int32, device=DEV)
    q = rand(starts[-1], heads * maps * d)
    arrays, info = ops.plan_latent_attention(HostLayout(4, starts[-1], starts, history, page, False))
    plan = Plan({k: torch.from_numpy(v).to(DEV) for k, v in arrays.items()}, info)
    call = lambda: ops.masked_attention(q, kc, vc, tok, pos, table.to(DEV), page, heads, kv, maps, d, dv, d ** -0.5, window=window, keep=keep,
                                        subtract=0.3 if maps == 2 else 0.0, plan=plan, max_ctx=2067)
    fast = call()
    before = ops.masked_attention_matrix_cores(False)
    try:
        near(fast, call(), float(vc.abs().max()))
    finally:
        ops.masked_attention_matrix_cores(before)


@pytest.mark.parametrize("maps", [1, 2])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dv", [32, 64, 128])
def test_the_stages_kernels_have_no_scratch(maps, d, dv):
    """Every build of the kernel, whatever becomes of the scores, keeps its operands and sums in registers (two maps of 64 with values of 128
    need 254 of the 256)."""
    assert ops.library().lc_masked_attention_bf16_scratch(maps, d, dv) == 0


def _case(history, fresh, heads, kv, maps, d, dv, page, seed, **options):
    """A call on requests with scattered pages, and the values' largest entry."""
    pages = [-(-(h + f) // page) for h, f in zip(history, fresh)]
    gen = torch.Generator().manual_seed(seed)
    order = torch.randperm(sum(pages), generator=gen).int()
    table, at = torch.zeros((len(pages), max(pages)), dtype=torch.int32), 0
    for r, n in enumerate(pages):
        table[r, :n] = order[at:at + n]
        at += n
    rand = lambda *s: torch.randn(*s, generator=gen).to(DEV).bfloat16()
    kc, vc = rand(at, page, kv * maps * d), rand(at, kv * dv, page)
    starts = [0]
    for f in fresh:
        starts.append(starts[-1] + f)
    tok = torch.tensor([r for r, f in enumerate(fresh) for _ in range(f)], dtype=torch.int32, device=DEV)
    pos = torch.tensor([history[r] + i for r, f in enumerate(fresh) for i in range(f)], dtype=torch.int32, device=DEV)
    q = rand(starts[-1], heads * maps * d)
    arrays, info = ops.plan_latent_attention(HostLayout(len(fresh), starts[-1], starts, history, page, False))
    plan = Plan({k: torch.from_numpy(v).to(DEV) for k, v in arrays.items()}, info)
    call = lambda: ops.masked_attention(q, kc, vc, tok, pos, table.to(DEV), page, heads, kv, maps, d, dv, d ** -0.5, plan=plan,
                                        subtract=0.3 if maps == 2 else 0.0, **options)
    return call, float(vc.abs().max())


def _general(call):
    before = ops.masked_attention_matrix_cores(False)
    try:
        return call()
    finally:
        ops.masked_attention_matrix_cores(before)


@pytest.mark.parametrize("staged", [1, 0])
@pytest.mark.parametrize("bias,cap", [(True, 0.0), (False, 1.5), (True, 1.5)])
@pytest.mark.parametrize("heads,kv,maps,d,dv", [(4, 1, 1, 128, 128), (4, 1, 2, 64, 128), (2, 2, 1, 64, 64), (8, 1, 1, 48, 32), (4, 2, 2, 128, 64)])
def test_bias_and_cap(heads, kv, maps, d, dv, bias, cap, staged):
    """What becomes of the scores, each alone and both, in the kernel with stages and in the other."""
    gen = torch.Generator(device=DEV).manual_seed(d)
    r1, r2 = (0.5 + torch.rand(heads, device=DEV, generator=gen) for _ in range(2))
    call, largest = _case([0, 15, 1000, 40], [33, 2, 30, 1], heads, kv, maps, d, dv, 16, heads + d, cap=cap,
                          r1=r1 if bias else None, r2=r2 if bias else None)
    before = ops.library().lc_masked_attention_bf16_staged(staged)
    try:
        near(call(), _general(call), largest)
    finally:
        ops.library().lc_masked_attention_bf16_staged(before)


@pytest.mark.parametrize("page", [16, 48])
@pytest.mark.parametrize("window,keep", [(0, 0), (8600, 40)])
def test_walks_of_more_than_64_blocks_a_wave(page, window, keep):
    """A wave holds the pages of 64 of its blocks: lone tokens, whose eight waves share their keys, beyond 8,192 keys, and portions of groups of
    eight heads without stages, where a wave walks all of them, beyond 1,024."""
    call, largest = _case([8200, 9100, 17000, 30], [1, 1, 1, 1], 4, 2, 1, 64, 64, page, page + keep, window=window, keep=keep)
    near(call(), _general(call), largest)
    call, largest = _case([1000, 2050, 9000], [40, 17, 3], 8, 1, 1, 64, 64, page, page + keep, window=window, keep=keep)
    before = ops.library().lc_masked_attention_bf16_staged(0)
    try:
        near(call(), _general(call), largest)
    finally:
        ops.library().lc_masked_attention_bf16_staged(before)
