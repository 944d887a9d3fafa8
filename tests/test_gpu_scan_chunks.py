"""The recurrence a chunk at a time (``ops.delta_scan_chunks``) against its definition in float64 and beside the
token-by-token kernel, and the rule that chooses between the two."""
from types import SimpleNamespace

import pytest
import torch

import reference_ops
from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# Both kernels round a sum of some 130 float32 terms a token, and what a state holds is the sum of the tokens it remembers:
# a few units of 2^-24 of the result's root mean square.  The token-by-token kernel is measured beside and the chunks may
# be off by twice as much (another order of the same sums), or by eight units where both are that small.
UNIT = 2.0 ** -24


def vectors(kind, T, heads, dk, g):
    def unit(x):
        return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)
    q, k = torch.randn(T, heads, dk, generator=g), unit(torch.randn(T, heads, dk, generator=g))
    beta = torch.rand(T, heads, 1, generator=g)
    if kind == "steady":            # one decay a head, close to 1
        d = (1 - 2.0 ** -torch.arange(5, 5 + heads).float())[None, :, None].expand(T, heads, dk)
    elif kind == "by channel":
        d = torch.rand(T, heads, dk, generator=g) * 0.4 + 0.6
    else:                           # decays of every size, 0 and 1 among them: pairs are made one by one
        d = torch.rand(T, heads, dk, generator=g) ** 8
        d[torch.rand(T, heads, dk, generator=g) < 0.1] = 0.0
        d[torch.rand(T, heads, dk, generator=g) < 0.1] = 1.0
    removing = [d, d * k, beta * k, beta * k, q]
    return torch.stack(removing).reshape(5, T, heads * dk), torch.stack([d, k, q]).reshape(3, T, heads * dk)


@pytest.mark.parametrize("planes", [5, 3])
@pytest.mark.parametrize("kind", ["steady", "by channel", "any"])
@pytest.mark.parametrize("heads,dk,dv,lengths", [(2, 128, 128, [64]), (3, 128, 48, [65, 95, 96, 97]), (1, 64, 17, [1, 127, 63, 64]),
                                                 (8, 64, 1, [161, 5]), (2, 128, 129, [3, 200, 1, 1, 80])])
def test_chunks(planes, kind, heads, dk, dv, lengths):
    g = torch.Generator().manual_seed(7 * dk + dv + planes)
    T, R = sum(lengths), len(lengths)
    coef = vectors(kind, T, heads, dk, g)[0 if planes == 5 else 1]
    v = torch.randn(T, heads * dv, generator=g)
    state = torch.randn(R + 2, heads, dv, dk, generator=g) * 0.2
    starts = [0] + torch.tensor(lengths).cumsum(0).tolist()
    lists = torch.tensor(starts, dtype=torch.int32), torch.randperm(R + 2, generator=g)[:R].to(torch.int32)
    states = [state.to(DEV), state.to(DEV)]
    on_gpu = (coef.to(DEV), v.to(DEV)), tuple(x.to(DEV) for x in lists)
    want_state = state.double()
    want = reference_ops.delta_scan(coef, v, want_state, *lists, R, heads, dk, dv).double()
    plain = ops.delta_scan(*on_gpu[0], states[0], *on_gpu[1], R, heads, dk, dv).cpu().double()
    got = ops.delta_scan_chunks(*on_gpu[0], states[1], *on_gpu[1], R, heads, dk, dv,
                                some_short=min(lengths) < ops.SCAN_CHUNKS_FROM).cpu().double()

    def off(x, y):
        return float((x - y).norm() / y.norm())
    assert off(got, want) <= max(2 * off(plain, want), 8 * UNIT), "read-outs"
    plain_state, got_state = (s.cpu().double() for s in states)
    assert off(got_state, want_state) <= max(2 * off(plain_state, want_state), 8 * UNIT), "states"
    idle = [s for s in range(R + 2) if s not in lists[1].tolist()]
    assert torch.equal(got_state[idle], state.double()[idle]), "another request's state"
    for r, n in enumerate(lengths):     # the short ones go token by token: the same bits
        if n < ops.SCAN_CHUNKS_FROM:
            assert torch.equal(got[starts[r]:starts[r + 1]], plain[starts[r]:starts[r + 1]])


@pytest.mark.parametrize("dtype,dk,lengths,chunked", [(torch.bfloat16, 128, [160, 2], True), (torch.float32, 128, [160, 2], False),
                                                      (torch.bfloat16, 128, [63, 2], False), (torch.bfloat16, 32, [190], False),
                                                      (torch.bfloat16, 64, [1, 170], True), (torch.bfloat16, 64, [1, 70], False),
                                                      (torch.bfloat16, 128, [64, 2], False)])
def test_which_steps_go_in_chunks(monkeypatch, dtype, dk, lengths, chunked):
    g = torch.Generator().manual_seed(dk)
    T, heads, dv = sum(lengths), 2, 16
    starts = [0] + torch.tensor(lengths).cumsum(0).tolist()
    batch = SimpleNamespace(q_offsets=torch.tensor(starts, dtype=torch.int32, device=DEV), q_start=starts, num_tokens=T,
                            slot_ids=torch.arange(len(lengths), dtype=torch.int32, device=DEV), num_requests=len(lengths))
    coef = vectors("by channel", T, heads, dk, g)[1].to(DEV)
    v, state = torch.randn(T, heads * dv, generator=g).to(DEV), torch.zeros(len(lengths), heads, dv, dk, device=DEV)
    called, real = [], ops.delta_scan_chunks
    monkeypatch.setattr(ops, "delta_scan_chunks", lambda *a, **k: called.append(1) or real(*a, **k))
    got = ops.delta_scan_step(coef, v, state.clone(), batch, heads, dk, dv, dtype)
    plain = ops.delta_scan(coef, v, state, batch.q_offsets, batch.slot_ids, len(lengths), heads, dk, dv)
    assert bool(called) == chunked
    assert torch.equal(got, plain) or chunked
    assert float((got - plain).norm() / plain.norm()) < 1e-6


@pytest.mark.parametrize("planes,where", [(5, p) for p in ("decay", "probe", "removal", "write", "read", "value")] +
                         [(3, p) for p in ("decay", "write", "read", "value")])
@pytest.mark.parametrize("bad,at", [(float("nan"), 45), (float("inf"), 99), (float("-inf"), 20), (2.0 ** 100, 3)])
@pytest.mark.parametrize("dk,dv", [(128, 33), (64, 16)])
def test_what_is_not_finite_reaches_later_tokens_only(planes, where, bad, at, dk, dv):
    """One entry of one token: the chunks' products leave the very places finite that the token-by-token kernel does, and what
    is finite is within 16 units of 2^-24 of that kernel's (both are within eight of the exact result where nothing is odd)."""
    g = torch.Generator().manual_seed(dk + planes)
    lengths, heads = [64, 100, 3], 2
    T, R, token, head = sum(lengths), len(lengths), 64 + at, 1
    coef = vectors("by channel", T, heads, dk, g)[0 if planes == 5 else 1].clone()
    v = torch.randn(T, heads * dv, generator=g)
    if where == "value":
        v.view(T, heads, dv)[token, head, 5] = bad
    else:
        names = ("decay", "probe", "removal", "write", "read") if planes == 5 else ("decay", "write", "read")
        coef.view(planes, T, heads, dk)[names.index(where), token, head, 7] = bad
    state = torch.randn(R, heads, dv, dk, generator=g) * 0.2
    starts = [0] + torch.tensor(lengths).cumsum(0).tolist()
    lists = torch.tensor(starts, dtype=torch.int32, device=DEV), torch.arange(R, dtype=torch.int32, device=DEV)
    results = []
    for f in (lambda *a: ops.delta_scan(*a), lambda *a: ops.delta_scan_chunks(*a, some_short=True)):
        s = state.to(DEV)
        results.append((f(coef.to(DEV), v.to(DEV), s, *lists, R, heads, dk, dv).cpu(), s.cpu()))
    for plain, got in zip(*results):
        finite = torch.isfinite(plain)
        assert torch.equal(torch.isfinite(got), finite)
        usual = finite & (plain.abs() < 1e6)
        assert float((got - plain)[usual].norm() / plain[usual].norm()) <= 16 * UNIT
    assert bool(torch.isfinite(results[1][0][:token]).all())


@pytest.mark.parametrize("planes", [5, 3])
@pytest.mark.parametrize("steps", [(-66, -64, 62, 60), (50, 50, -50, -50), (-40, 30, -40, 50)])
def test_decays_that_leave_the_range_inside_a_block(planes, steps):
    """A block whose decays multiply to a common number, and to very small or large ones on the way: against float64, the
    token-by-token kernel beside it."""
    g = torch.Generator().manual_seed(planes)
    T, heads, dk, dv = 64, 1, 64, 16
    coef = vectors("by channel", T, heads, dk, g)[0 if planes == 5 else 1].clone()
    decay = coef.view(planes, T, heads, dk)[0]
    decay[19:23] = 2.0 ** torch.tensor(steps)[:, None, None].float()
    if planes == 5:
        coef.view(planes, T, heads, dk)[1] = torch.nn.functional.normalize(torch.randn(T, heads, dk, generator=g), dim=-1)
    v, state = torch.randn(T, heads * dv, generator=g), torch.zeros(1, heads, dv, dk)
    lists = torch.tensor([0, T], dtype=torch.int32), torch.zeros(1, dtype=torch.int32)
    want = reference_ops.delta_scan(coef, v, state.double(), *lists, 1, heads, dk, dv).double()
    on_gpu = coef.to(DEV), v.to(DEV)
    plain = ops.delta_scan(*on_gpu, state.to(DEV), *(x.to(DEV) for x in lists), 1, heads, dk, dv).cpu().double()
    got = ops.delta_scan_chunks(*on_gpu, state.to(DEV), *(x.to(DEV) for x in lists), 1, heads, dk, dv, some_short=False).cpu().double()
    for t in range(T):      # token by token: one token's size says nothing of another's
        off = [float((x[t] - want[t]).norm() / want[t].norm()) for x in (plain, got)]
        assert off[1] <= max(4 * off[0], 64 * UNIT), (t, off)


@pytest.mark.parametrize("lengths", [[1] * 200 + [64] + [1] * 55, [64] + [1] * 255, [1] * 255 + [70], [63] * 9 + [64, 64, 65, 1, 127, 128, 2, 96],
                                     [1, 2, 3] * 20 + [64, 1, 95, 1, 300], [20]])
def test_requests_of_few_tokens_take_no_record(lengths):
    """One portion beside many requests of few tokens: the right places, and scratch for the portions' chunks alone."""
    g = torch.Generator().manual_seed(len(lengths))
    heads, dk, dv, T, R = 2, 128, 16, sum(lengths), len(lengths)
    coef = vectors("by channel", T, heads, dk, g)[0].to(DEV)
    v, state = torch.randn(T, heads * dv, generator=g).to(DEV), torch.randn(R, heads, dv, dk, generator=g).to(DEV)
    starts = torch.tensor([0] + torch.tensor(lengths).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    lists = starts, torch.arange(R, dtype=torch.int32, device=DEV)
    states = [state.clone(), state.clone()]
    plain = ops.delta_scan(coef, v, states[0], *lists, R, heads, dk, dv)
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    got = ops.delta_scan_chunks(coef, v, states[1], *lists, R, heads, dk, dv, some_short=True)
    scratch = torch.cuda.max_memory_allocated() - before - got.numel() * 4
    # a chunk: four planes of vectors, the matrix and the decays; a portion of 64 tokens may waste one, the list half as many
    chunk = (4 * 32 * dk + 2 * dk + 32 * 32 + 2) * 4 * heads
    chunks = max(1, T // 32 + T // 64)
    assert scratch <= chunks * chunk + 4096, (scratch, chunks * chunk)
    for a, b in ((got, plain), (states[1], states[0])):
        assert float((a - b).norm() / b.norm()) <= 16 * UNIT
    short = torch.tensor([n < ops.SCAN_CHUNKS_FROM for n in lengths], device=DEV)
    assert torch.equal(states[1][short], states[0][short])


@pytest.mark.parametrize("planes", [5, 3])
@pytest.mark.parametrize("dk", [64, 128])
# 16 tokens' decays multiply to 2^-60 at 2^-3.75 a token: just inside, where the pairs of a block are products of vectors scaled by up
# to 2^60, just outside, where they are made one by one; every channel, one channel, one block, and blocks of both kinds
@pytest.mark.parametrize("where", ["everywhere", "a channel", "a block"])
@pytest.mark.parametrize("exponent", [-3.74, -3.76])
def test_decays_around_the_range(planes, dk, where, exponent):
    g = torch.Generator().manual_seed(planes + dk)
    T, heads, dv = 112, 2, 32
    coef = vectors("by channel", T, heads, dk, g)[0 if planes == 5 else 1].clone()
    decay = coef.view(planes, T, heads, dk)[0]
    decay[{"everywhere": slice(None), "a channel": (slice(None), 1, 7), "a block": slice(48, 64)}[where]] = 2.0 ** exponent
    if planes == 5:     # the probe is the decay times a key, here the removal's
        coef.view(planes, T, heads, dk)[1] = decay * coef.view(planes, T, heads, dk)[2]
    v, state = torch.randn(T, heads * dv, generator=g), torch.randn(1, heads, dv, dk, generator=g) * 0.2
    lists = torch.tensor([0, T], dtype=torch.int32), torch.zeros(1, dtype=torch.int32)
    want_state, states = state.double(), [state.to(DEV), state.to(DEV)]
    want = reference_ops.delta_scan(coef, v, want_state, *lists, 1, heads, dk, dv).double()
    args = (coef.to(DEV), v.to(DEV)), tuple(x.to(DEV) for x in lists)
    plain = ops.delta_scan(*args[0], states[0], *args[1], 1, heads, dk, dv).cpu().double()
    got = ops.delta_scan_chunks(*args[0], states[1], *args[1], 1, heads, dk, dv, some_short=False).cpu().double()

    def off(x, y):
        return float((x - y).norm() / y.norm())
    print(f"{off(got, want) / UNIT:.2f} {off(plain, want) / UNIT:.2f} units")
    assert off(got, want) <= max(2 * off(plain, want), 8 * UNIT), "read-outs"
    assert off(states[1].cpu().double(), want_state) <= max(2 * off(states[0].cpu().double(), want_state), 8 * UNIT), "states"
    # Token by token, because none may hide behind another: a read-out is a sum of n = dk terms and more of either sign, whose sizes add
    # up to `reach` (the recurrence over absolute values, what is removed added).  Its partial sums are some reach / sqrt(n) and the
    # n roundings, half a unit of one each at the most, some sqrt(n) of them: half a unit of reach.  Four times that, or what
    # the token-by-token kernel shows.
    size = coef.abs().view(planes, T, heads * dk)
    if planes == 5:
        size[2] = -size[2]
    reach = reference_ops.delta_scan(size, v.abs(), state.abs().double(), *lists, 1, heads, dk, dv).double()
    for t in range(T):
        error, beside = (float((x[t] - want[t]).norm()) for x in (got, plain))
        assert error <= max(4 * beside, 2 * UNIT * float(reach[t].norm())), t


# every number of chunks modulo the walk's three turns, and value channels stored four at a time or, where a row is no whole 16 bytes, one
# by one, with the last block of 16 channels partly filled either way
@pytest.mark.parametrize("planes", [5, 3])
@pytest.mark.parametrize("dk,dv", [(128, 20), (128, 50), (64, 36), (64, 130)])
def test_turns_and_columns(planes, dk, dv):
    test_chunks(planes, "by channel", 2, dk, dv, [64, 65, 97, 129, 161, 193, 225])


# more records than workgroups at once, so that these take several, ones that nobody owns among them: a head's results are those of a step that
# has this head alone, to the bit
@pytest.mark.parametrize("planes,dk", [(3, 128), (3, 64), (5, 64), (5, 128)])
def test_records_in_turns(planes, dk):
    heads, dv, lengths = 30, 16, [900, 2, 70, 500, 1, 65]
    g = torch.Generator().manual_seed(planes + dk)
    T, R = sum(lengths), len(lengths)
    coef = vectors("by channel", T, heads, dk, g)[0 if planes == 5 else 1].to(DEV)
    v, state = torch.randn(T, heads * dv, generator=g).to(DEV), torch.randn(R, heads, dv, dk, generator=g).to(DEV)
    lists = torch.tensor([0] + torch.tensor(lengths).cumsum(0).tolist(), dtype=torch.int32, device=DEV), torch.arange(R, dtype=torch.int32, device=DEV)
    whole = state.clone()
    out = ops.delta_scan_chunks(coef, v, whole, *lists, R, heads, dk, dv, some_short=True)
    for head in (0, 17, heads - 1):
        one = state[:, head:head + 1].contiguous()
        got = ops.delta_scan_chunks(coef[..., head * dk:(head + 1) * dk].contiguous(), v[:, head * dv:(head + 1) * dv].contiguous(), one, *lists,
                                    R, 1, dk, dv, some_short=True)
        assert torch.equal(got, out[:, head * dv:(head + 1) * dv]), "read-outs"
        assert torch.equal(one[:, 0], whole[:, head]), "states"
