"""The kernels that prepare a mixer's inputs with a thread per entry and run of tokens (long steps), against the forms for short steps and
the plain versions: requests that begin and end inside a run, the last run not whole, values that do and do not fill a page's pieces."""
import pytest
import torch

import reference_ops
from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENGTHS = [1, 700, 2, 399, 1]        # 1,103 tokens


def lists():
    tok_req = torch.cat([torch.full((n,), r, dtype=torch.int32) for r, n in enumerate(LENGTHS)])
    q_offsets = torch.tensor([0] + LENGTHS, dtype=torch.int32).cumsum(0, dtype=torch.int32)
    return tok_req, q_offsets, torch.tensor([3, 0, 5, 1, 2], dtype=torch.int32)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nq,nk,nv,d,dv,taps,rot,page", [
    (4, 2, 2, 64, 64, 4, 32, 16), (3, 1, 2, 6, 10, 4, 4, 12), (2, 2, 1, 130, 8, 0, 0, 16), (5, 1, 1, 32, 34, 3, 32, 24), (2, 0, 0, 16, 2, 4, 0, 16),
    (3, 1, 2, 6, 10, 8, 4, 12), (5, 1, 1, 32, 34, 1, 32, 24), (30, 3, 2, 66, 34, 4, 4, 12), (16, 8, 4, 64, 128, 0, 0, 24), (12, 6, 6, 130, 34, 4, 0, 16),
    (16, 8, 4, 64, 128, 4, 32, 16)])       # the last four wide enough for runs of tokens
def test_attention_inputs(dtype, nq, nk, nv, d, dv, taps, rot, page):
    g = torch.Generator().manual_seed(nq + d + dv + taps)
    T, C = sum(LENGTHS), (nq + nk) * d + nv * dv
    on = lambda t: None if t is None else t.to(DEV)
    tok_req, q_offsets, slots = (on(t) for t in lists())
    proj = on(torch.randn(T, C + 2, generator=g))
    conv = on(torch.randn(C, taps, generator=g)) if taps else None
    tail = on(torch.randn(6, taps - 1, C, generator=g)) if taps > 1 else None
    table = on(torch.randn(T, rot, generator=g)) if rot else None
    # request 1 begins at a page's start, request 3 in the middle of one, some tokens have no row
    pages = T // page + 4
    rows = torch.full((T,), -1, dtype=torch.int32)
    rows[1:701] = torch.arange(700, dtype=torch.int32) + page
    rows[703:1102] = torch.arange(399, dtype=torch.int32) + (701 // page + 2) * page + 5
    rows[40], rows[1102] = -1, 0
    rows = on(torch.where(rows < pages * page, rows, torch.full_like(rows, -1)))
    results = []
    for pairs in (True, False):
        kc = torch.zeros(pages, page, max(nk * d, 1), dtype=dtype, device=DEV)
        vc = torch.zeros(pages, max(nv * dv, 1), page, dtype=dtype, device=DEV)
        before = ops.attention_prepare_pairs(pairs)
        try:
            q = ops.attention_prepare(proj, nq, nk, nv, d, dv, dtype, kc if nk else None, vc if nk else None, rows if nk else None, taps=conv,
                                      tail=tail, tok_req=tok_req, q_offsets=q_offsets, slot_ids=slots, table=table, rot=rot,
                                      positions=torch.arange(T, dtype=torch.int32, device=DEV), unit_eps=None)
        finally:
            ops.attention_prepare_pairs(before)
        results.append((q, kc, vc))
    for got, want in zip(*results):
        assert torch.equal(got, want)


@pytest.mark.parametrize("heads,groups,N,dv,taps", [(4, 2, 16, 32, 4), (3, 1, 7, 100, 3), (2, 2, 130, 3, 2), (6, 3, 5, 64, 1), (2, 1, 16, 16, 6),
                                                      (4, 2, 130, 2000, 4), (3, 1, 7, 1300, 2), (4, 2, 130, 1000, 6)])       # runs of eight and four
def test_state_space_inputs(heads, groups, N, dv, taps):
    g = torch.Generator().manual_seed(heads + N + taps)
    T, inner = sum(LENGTHS), heads * dv
    C = inner + 2 * groups * N
    given = [torch.randn(T, C + inner + heads, generator=g), torch.randn(C, taps, generator=g) * 0.5, torch.randn(C, generator=g) * 0.3,
             torch.randn(6, taps - 1, C, generator=g) if taps > 1 else None, torch.randn(heads, generator=g), torch.randn(heads, generator=g) - 1,
             *lists()]
    proj, conv, bias, tail, dt_bias, a_log, *rest = given
    want = reference_ops.state_space_prepare(proj, heads, groups, N, dv, conv, bias, tail, dt_bias, a_log, *rest)
    proj, conv, bias, tail, dt_bias, a_log, *rest = [None if t is None else t.to(DEV) for t in given]
    got = ops.state_space_prepare(proj, heads, groups, N, dv, conv, bias, tail, dt_bias, a_log, *rest)
    for a, b in zip(got, want):
        # sums of up to six products, an exponential or two and a product: some ten roundings of 2^-24 of terms up to 8
        torch.testing.assert_close(a.cpu(), b, rtol=2e-6, atol=2e-6)
    # the same tokens in steps so short that every one is prepared by itself: the same bits
    tok_req, q_offsets, slots = rest
    for r, n in enumerate(LENGTHS):
        first = int(q_offsets[r])
        few = min(n, 200 if heads * dv < 3000 else 20)
        one = ops.state_space_prepare(proj[first:first + few].contiguous(), heads, groups, N, dv, conv, bias, tail, dt_bias, a_log,
                                      torch.zeros(few, dtype=torch.int32, device=DEV), torch.tensor([0, few], dtype=torch.int32, device=DEV),
                                      slots[r:r + 1].contiguous())
        for a, b in zip(one, got):
            b = b.view(-1, T, b.shape[-1])[:, first:first + few] if b.dim() == 3 else b[first:first + few]
            assert torch.equal(a.reshape(b.shape), b)


@pytest.mark.parametrize("heads,groups,taps", [(8192, 2, 4), (8193, 1, 4), (20000, 4, 1)])
def test_state_space_of_many_heads(heads, groups, taps):
    """More heads than a workgroup's LDS has room for a step and a decay of."""
    g = torch.Generator().manual_seed(heads)
    T, N, dv = 5, 3, 1
    C = heads * dv + 2 * groups * N
    given = [torch.randn(T, C + heads * dv + heads, generator=g), torch.randn(C, taps, generator=g) * 0.5, torch.randn(C, generator=g) * 0.3,
             torch.randn(2, taps - 1, C, generator=g) if taps > 1 else None, torch.randn(heads, generator=g), torch.randn(heads, generator=g) - 1,
             torch.tensor([0, 0, 0, 1, 1], dtype=torch.int32), torch.tensor([0, 3, 5], dtype=torch.int32), torch.tensor([1, 0], dtype=torch.int32)]
    proj, conv, bias, tail, dt_bias, a_log, *rest = given
    want = reference_ops.state_space_prepare(proj, heads, groups, N, dv, conv, bias, tail, dt_bias, a_log, *rest)
    proj, conv, bias, tail, dt_bias, a_log, *rest = [None if t is None else t.to(DEV) for t in given]
    got = ops.state_space_prepare(proj, heads, groups, N, dv, conv, bias, tail, dt_bias, a_log, *rest)
    for a, b in zip(got, want):
        torch.testing.assert_close(a.cpu(), b, rtol=2e-6, atol=2e-6)
