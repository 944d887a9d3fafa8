"""Latent attention of long portions head by head (``ops.latent_wide``) against the same formulas in float64, in steps of
several requests, behind histories, windows and pages that were given back; and which steps take it."""
import pytest
import torch

import kikunex_configs
import plain_kikunex
import plain_pubodra
import pubodra_configs
import traces
from helpers import compare, make_runner, prompts_for, random_weights, replay
from lucciola_amd.engine.batch import HostLayout, Plan
from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DIM, ROT, VDIM = 128, 64, 128


def reference(q, turned_q, c, turned, uk, uv, position, scale, window, sink):
    """One head's tokens in float64 over one request's rows: keys and values rounded as the products leave them."""
    k = torch.cat([(c @ uk.T).bfloat16().double(), turned], 1)
    v = (c @ uv.T).bfloat16().double()
    s = torch.cat([q, turned_q], 1) @ k.T * scale
    i, j = position + torch.arange(len(q), device=DEV)[:, None], torch.arange(len(c), device=DEV)[None]
    seen = j <= i
    if window:
        seen &= j > i - window
    s = s.masked_fill(~seen, float("-inf"))
    top = s.max(1, keepdim=True).values
    if sink is not None:
        top = torch.maximum(top, sink)
    e = torch.exp(s - top)
    return e @ v / (e.sum(1, keepdim=True) + (torch.exp(sink - top) if sink is not None else 0.0))


WIDE_CASES = [
    (2, 512, 16, 0, "entry", False, [(0, 64)]), (3, 64, 16, 0, "head", True, [(0, 65), (63, 127), (100, 128)]),
    (1, 128, 4, 50, "none", True, [(0, 129), (200, 300)]), (2, 192, 32, 64, "entry", False, [(7, 191), (64, 64)]),
    (1, 512, 16, 0, "none", False, [(1000, 257)])]


@pytest.mark.parametrize("heads,rank,page,window,gate,with_sink,requests", WIDE_CASES)
def test_wide(heads, rank, page, window, gate, with_sink, requests):
    g = torch.Generator().manual_seed(heads * 1000 + rank + window)
    def made(*shape):
        return torch.randn(*shape, generator=g)
    T = sum(n for _, n in requests) + 3                      # three tokens of others in front
    q_start = [3]
    for _, n in requests:
        q_start.append(q_start[-1] + n)
    first = [p for p, _ in requests]
    pages_each = [-(-(p + n) // page) for p, n in requests]
    cache = (made(sum(pages_each) + 1, page, rank + ROT) * 0.7).bfloat16().to(DEV)
    order = torch.randperm(sum(pages_each), generator=g) + 1
    table = torch.full((len(requests), max(pages_each) + 1), -1, dtype=torch.int32)
    at = 0
    for r, n in enumerate(pages_each):
        table[r, :n] = order[at:at + n]
        at += n
        if window:          # pages behind the window have gone back
            table[r, :max(0, first[r] - window + 1) // page] = -1
    ldq = heads * (DIM + ROT) + 8
    q, qa = made(T, ldq).bfloat16().to(DEV), made(T, heads * (rank + ROT)).bfloat16().to(DEV)
    uk, uv = (made(heads * n, rank).mul(rank ** -0.5).bfloat16().to(DEV) for n in (DIM, VDIM))
    gates = made(T, heads * VDIM + 4).bfloat16().to(DEV)
    sink = made(heads).to(DEV) if with_sink else None
    out = torch.zeros(T, heads * VDIM, dtype=torch.bfloat16, device=DEV)
    scale = (DIM + ROT) ** -0.5 * 2.0
    strided = None if gate == "none" else ops.Strided(gates, 4, VDIM if gate == "entry" else 1)
    ops.latent_wide(q, qa, heads, rank, DIM, ROT, VDIM, uk, uv, cache, table.to(DEV), page, range(len(requests)), q_start, first,
                    scale, window, sink, strided, gate == "head", out)
    assert float(out[:3].abs().max()) == 0.0, "other tokens' rows were written"
    for r, (p, n) in enumerate(requests):
        slots = [max(0, int(table[r, j // page])) * page + j % page for j in range(p + n)]
        rows = cache.view(-1, rank + ROT)[slots].double()
        mine = slice(q_start[r], q_start[r] + n)
        for h in range(heads):
            plain = q[mine, h * (DIM + ROT):h * (DIM + ROT) + DIM].double()
            turned_q = qa[mine].view(n, heads, rank + ROT)[:, h, rank:].double()
            want = reference(plain, turned_q, rows[:, :rank], rows[:, rank:], uk[h * DIM:(h + 1) * DIM].double(),
                             uv[h * VDIM:(h + 1) * VDIM].double(), p, scale, window, sink[h].double() if with_sink else None)
            if gate == "entry":
                want = want * torch.sigmoid(gates[mine, 4 + h * VDIM:4 + (h + 1) * VDIM].double())
            elif gate == "head":
                want = want * torch.sigmoid(gates[mine, 4 + h:5 + h].double())
            got = out[mine, h * VDIM:(h + 1) * VDIM].double()
            # the weights and the result are rounded to bfloat16 (2^-9 each, of numbers up to the largest value), and so are
            # keys and values, where another order of a sum may round to the neighbour now and then
            bound = 3 * 2.0 ** -9 * float(rows.abs().max().clamp(min=4.0))
            assert float((got - want).abs().max()) <= bound, (r, h)
            assert float((got - want).norm() / want.norm()) <= 2.0 ** -8, (r, h)


@pytest.mark.parametrize("halves", [1, 2])
def test_wide_in_halves(halves):
    """Both forms of the kernel, whatever the size would choose: stages in one row, and every other stage for each half, with a last
    one that only one half has, windows that begin inside a stage and waves whose queries see none."""
    before = ops.library().lc_latent_wide_halves(halves)
    try:
        for case in WIDE_CASES:
            test_wide(*case)
    finally:
        ops.library().lc_latent_wide_halves(before)


def test_short_portions_keep_their_tiles():
    lengths, first = [1, 1500, 63, 2000, 1], [500, 0, 9, 100, 3]
    q_start = [0]
    for n in lengths:
        q_start.append(q_start[-1] + n)
    key, plan = ops.latent_short_planner(16, 4096)
    arrays, info = plan(HostLayout(5, q_start[-1], q_start, first, 16, False))
    assert info == {"any_portion": True, "any_lone": True, "num_tiles": 6, "wide": [1, 3]}
    assert sorted(set(arrays["tiles"][:, 2].tolist())) == [0, 2, 4] and int(arrays["tiles"][:, 1].sum()) == 65
    every, info = plan(HostLayout(1, 2048, [0, 2048], [0], 16, False))
    assert every["tiles"].shape == (1, 4) and info["wide"] == [0] and info["num_tiles"] == 0
    short = HostLayout(2, 61, [0, 60, 61], [5, 9], 16, False)
    assert plan(short)[0]["tiles"].tolist() == ops.plan_latent_attention(short)[0]["tiles"].tolist()
    assert plan(short)[1]["wide"] == [] and key != ops.latent_short_planner(16, 0)[0]


def test_scratch_is_what_the_cache_leaves_room_for():
    heads, rank, page, requests = 16, 512, 16, [(3000, 500), (0, 1100)]
    g = torch.Generator().manual_seed(3)
    T, pages = sum(n for _, n in requests), [-(-(p + n) // page) for p, n in requests]
    cache = torch.randn(sum(pages) + 1, page, rank + ROT, generator=g).bfloat16().to(DEV)
    table = torch.full((2, max(pages)), -1, dtype=torch.int32)
    table[0, :pages[0]], table[1, :pages[1]] = torch.arange(pages[0]), pages[0] + torch.arange(pages[1])
    q, qa = (torch.randn(T, heads * n, generator=g).bfloat16().to(DEV) for n in (DIM + ROT, rank + ROT))
    uk, uv = (torch.randn(heads * n, rank, generator=g).bfloat16().to(DEV) for n in (DIM, VDIM))
    out, table = torch.zeros(T, heads * VDIM, dtype=torch.bfloat16, device=DEV), table.to(DEV)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    ops.latent_wide(q, qa, heads, rank, DIM, ROT, VDIM, uk, uv, cache, table, page, [0, 1], [0, 500, T], [p for p, _ in requests],
                    0.1, 0, None, None, False, out)
    rows = sum(-(-(p + n) // 64) * 64 for p, n in requests)
    partial = 4 * max(ops.library().lc_gemm_bf16_workspace(rows, heads * DIM, rank), ops.library().lc_gemm_bf16_workspace(heads * VDIM, rows, rank))
    per_row, most = ops.latent_wide_scratch(heads, rank, ROT, DIM, VDIM)
    assert 0 < torch.cuda.max_memory_allocated() - before <= rows * per_row + max(partial, 0) + 4096
    assert rows * per_row <= most


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("entry", [5, 64 + 3])          # of the latent, of the rotated part
@pytest.mark.parametrize("position,tokens,window,at", [(0, 130, 0, 100), (0, 130, 0, 129), (70, 200, 0, 200), (300, 150, 90, 380), (40, 64, 0, 10)])
def test_a_row_that_is_not_finite_reaches_only_who_sees_it(bad, entry, position, tokens, window, at):
    heads, rank, page, T = 2, 64, 16, tokens
    g = torch.Generator().manual_seed(position + tokens)
    pages = -(-(position + tokens) // page)
    cache = torch.randn(pages, page, rank + ROT, generator=g).bfloat16().to(DEV)
    q, qa = (torch.randn(T, heads * n, generator=g).bfloat16().to(DEV) for n in (DIM + ROT, rank + ROT))
    uk, uv = (torch.randn(heads * n, rank, generator=g).mul(rank ** -0.5).bfloat16().to(DEV) for n in (DIM, VDIM))
    table = torch.arange(pages, dtype=torch.int32, device=DEV)[None]
    outs = []
    for value in (0.25, bad):
        cache.view(-1, rank + ROT)[at, entry] = value
        outs.append(torch.zeros(T, heads * VDIM, dtype=torch.bfloat16, device=DEV))
        ops.latent_wide(q, qa, heads, rank, DIM, ROT, VDIM, uk, uv, cache, table, page, [0], [0, T], [position], 0.1, window, None, None,
                        False, outs[-1])
    i = position + torch.arange(T, device=DEV)
    sees = (i >= at) & ((i < at + window) if window else (i >= 0))
    assert torch.equal(outs[1][~sees], outs[0][~sees])
    assert bool(torch.isfinite(outs[0]).all())
    if entry < 64:          # (a rotated part may make a score of minus infinity, which weighs nothing)
        assert not bool(torch.isfinite(outs[1][sees]).any())


@pytest.mark.parametrize("rank,heads,with_sink", [(512, 4, True), (256, 5, False)])
@pytest.mark.parametrize("wide", [[], [1]])
def test_shares_of_portions(monkeypatch, rank, heads, with_sink, wide):
    """Short portions behind long histories, their keys shared out: shares by token where every token of the step is in a tile, by tile
    beside a portion that attends head by head.  Against the general kernel in float32 arithmetic."""
    requests, page = [(900, 40), (0, 1500), (700, 1), (500, 3)], 16
    if not wide:
        requests[1] = (1200, 17)
    g = torch.Generator().manual_seed(rank + heads)
    lengths, first = [n for _, n in requests], [p for p, _ in requests]
    q_start = [0]
    for n in lengths:
        q_start.append(q_start[-1] + n)
    T, R, pages = q_start[-1], len(requests), [-(-(p + n) // page) for p, n in requests]
    cache = (torch.randn(sum(pages), page, rank + ROT, generator=g) * 0.5).bfloat16().to(DEV)
    table, at = torch.full((R, max(pages)), -1, dtype=torch.int32), 0
    for r, n in enumerate(pages):
        table[r, :n] = torch.arange(at, at + n)
        at += n
    qa = (torch.randn(T, heads * (rank + ROT), generator=g) * 0.6).bfloat16().to(DEV)
    positions = torch.cat([torch.arange(p, p + n) for p, n in requests]).to(torch.int32).to(DEV)
    tok_req = torch.cat([torch.full((n,), r) for r, n in enumerate(lengths)]).to(torch.int32).to(DEV)
    sink = torch.randn(heads, generator=g).to(DEV) if with_sink else None
    layout = HostLayout(R, T, q_start, first, page, False)
    monkeypatch.setattr(ops, "latent_wide_pays", lambda tokens, position, *a: tokens == 1500)
    monkeypatch.setattr(ops, "latent_wide_gains", lambda *a: True)
    arrays, info = ops.latent_short_planner(heads, 0)[1](layout)
    assert info["wide"] == wide
    plan = Plan({k: torch.tensor(v, device=DEV) for k, v in arrays.items()}, info)
    calls, call = [], ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: calls.append((name, a)) or call(name, *a))
    args = (qa, heads, rank, ROT, tok_req, positions, table.to(DEV), cache, page, (rank + ROT) ** -0.5 * 2.0)
    got = ops.latent_attention(*args, plan=plan, max_ctx=max(p + n for p, n in requests), sink=sink)
    (name, sent), = calls
    assert name == "lc_latent_attention_bf16" and sent[8] == (1 if wide else 2) and sent[16] > 1, "form and shares"
    before = ops.latent_matrix_cores(False)
    try:
        want = ops.latent_attention(*args, plan=plan, sink=sink)
    finally:
        ops.latent_matrix_cores(before)
    for r in range(R):
        if r not in wide:
            a, b = (x[q_start[r]:q_start[r + 1]].double() for x in (got, want))
            assert float((a - b).norm() / b.norm()) <= 2.0 ** -7, r       # weights and both results rounded to bfloat16


def _pubodra():
    """The queries out of the layer's input, a gate an entry, a window and none."""
    mixers = [pubodra_configs._mixer(heads, DIM, ROT, VDIM, 512, 0.07, window) for heads, window in ((3, 100), (2, None))]
    layers = [pubodra_configs._layer(mixers[0], None), pubodra_configs._layer(mixers[1], pubodra_configs._dense(96))]
    cfg = {"architecture": "Pubodra", "vocab": 300, "width": 128, "norm": {"eps": 1e-6}, "layers": layers}
    return cfg, random_weights(cfg, 5, std=0.1), plain_pubodra.forward


def _kikunex():
    """The queries out of a latent of their own, a gate a head, a sink, a window and none."""
    mixers = [kikunex_configs.latent(8, DIM, ROT, VDIM, rank, 64, 0.07, window) for rank, window in ((512, None), (128, 90))]
    cfg = {"architecture": "Kikunex", "vocab": 300, "width": 128, "norm": {"eps": 1e-6}, "layers": [kikunex_configs.layer(m, None) for m in mixers]}
    weights, g = random_weights(dict(cfg, initializer_range=0.1), 6), torch.Generator().manual_seed(6)
    for name, t in weights.items():
        if name.endswith(".sink"):
            weights[name] = (torch.randn(t.shape, generator=g) * 1.5).to(t.dtype)
    return cfg, weights, plain_kikunex.forward


@pytest.mark.parametrize("model", [_pubodra, _kikunex])
def test_a_model_whose_portions_attend_head_by_head(monkeypatch, model):
    """Steps of long portions only, of long ones beside short ones and lone tokens, behind what earlier steps have cached, and of
    none: the logits at every place are the plain implementation's."""
    cfg, weights, forward = model()
    prompts = prompts_for({"vocab_size": cfg["vocab"]}, [281, 231, 122], 7)
    refs = {n: forward(cfg, weights, ids) for n, ids in prompts.items()}
    without = forward(cfg, {n: t * 0 if n.endswith(".uv") else t for n, t in weights.items()}, prompts["r0"])
    moved = (without - refs["r0"]).abs().amax(1) / refs["r0"].abs().amax(1)
    assert float(moved.median()) > 0.2, "the logits would not show a wrong attention"
    steps, fed = [], dict.fromkeys(prompts, 0)
    for sizes in ({"r0": 150, "r1": 128}, {"r0": 130, "r1": 1, "r2": 20}, {"r1": 1, "r2": 1}, {"r1": 101}, {"r2": 101, "r0": 1}):
        entries = []
        for name, n in sizes.items():
            entries.append((name, prompts[name][fed[name]:fed[name] + n], list(range(n))))
            fed[name] += n
        steps.append((entries, [name for name in sizes if fed[name] == len(prompts[name])]))
    monkeypatch.setattr(ops, "latent_wide_pays", lambda tokens, position, heads, window: tokens >= 100)
    monkeypatch.setattr(ops, "latent_wide_gains", lambda *a: True)
    calls, call = [], ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: calls.append(name) or call(name, *a))
    got = replay(make_runner(cfg, weights, 16, traces.max_live_tokens(steps, 16) // 16, "bfloat16", DEV), steps)
    assert len(got) == sum(len(ids) for ids in prompts.values())
    assert calls.count("lc_latent_wide") == 2 * 5, "two layers, five portions of 100 tokens and more"
    print(f"{cfg['architecture']}: worst relative error {compare(got, cfg, weights, prompts, 4e-2, refs):.3e}")


@pytest.mark.parametrize("halves", [1, 2])
@pytest.mark.parametrize("scale", [-0.3, 0.0])
def test_scales_that_are_not_positive(halves, scale):
    """A score's sign goes with the query, and a scale of zero weighs every visible key alike: against float64, whose values are exact here,
    with weights rounded to bfloat16 (2^-9 each) and a bfloat16 result."""
    H, T, position, window = 3, 200, 70, 90
    lo = max(0, position - window + 1)
    rows = -(-(position + T - lo) // 64) * 64
    g = torch.Generator().manual_seed(5)
    q, turned_q, keys, turned, values = ((torch.randn(*shape, generator=g) * 0.5).bfloat16().to(DEV) for shape in (
        (T, H * 192), (T, H * 64), (rows, H * 128), (rows, 64), (H * 128, rows)))
    out = torch.empty(T, H * 128, dtype=torch.bfloat16, device=DEV)
    before = ops.library().lc_latent_wide_halves(halves)
    try:
        ops._call("lc_latent_wide", ops._ptr(q), H * 192, ops._ptr(turned_q), H * 64, 64, ops._ptr(keys), ops._ptr(turned), ops._ptr(values),
                  rows, H, 0, T, position, lo, scale, window, None, None, 0, 0, ops._ptr(out), H * 128, ops._stream())
    finally:
        ops.library().lc_latent_wide_halves(before)
    i, j = torch.arange(T, device=DEV)[:, None] + position, torch.arange(rows, device=DEV)[None] + lo
    seen = (j <= i) & (j > i - window)
    for h in range(H):
        a = torch.cat([q[:, h * 192:h * 192 + 128], turned_q[:, h * 64:h * 64 + 64]], 1).double()
        s = a @ torch.cat([keys[:, h * 128:h * 128 + 128], turned], 1).double().T * scale
        want = s.masked_fill(~seen, float("-inf")).softmax(1) @ values[h * 128:h * 128 + 128].double().T
        got = out[:, h * 128:h * 128 + 128].double()
        assert float((got - want).norm() / want.norm()) <= 2.0 ** -8


@pytest.mark.parametrize("halves", [1, 2])
@pytest.mark.parametrize("scale", [0.7, -0.7])
def test_scores_are_rounded_before_the_weights(halves, scale):
    """A weight is 2 to the power of a score times the scale, rounded to float32, less the largest such.  Scores of 2^17 and a few, exact in
    float32, of one stage of keys: the product's rounding is up to 2^-8 there, so that one rounding more or less changes three results of ten
    in bfloat16.  An exponential off by a unit of 2^-24 and the sum's rounding turn one in 2^14 to its neighbour; one in 200 may."""
    T, sign = 64, 1.0 if scale > 0 else -1.0
    g = torch.Generator().manual_seed(11)
    q, keys, turned, values = torch.zeros(T, 192), torch.zeros(64, 128), torch.zeros(64, 64), torch.zeros(128, 64)
    q[:, 0], q[:, 1], keys[:, 0], keys[:, 1] = 512.0 * sign, sign, 256.0, torch.randint(0, 256, (64,), generator=g) / 32.0
    values[:64] = torch.eye(64)
    q, keys, turned, values = (x.bfloat16().to(DEV) for x in (q, keys, turned, values))
    turned_q, out = torch.zeros(T, 64, dtype=torch.bfloat16, device=DEV), torch.empty(T, 128, dtype=torch.bfloat16, device=DEV)
    before = ops.library().lc_latent_wide_halves(halves)
    try:
        ops._call("lc_latent_wide", ops._ptr(q), 192, ops._ptr(turned_q), 64, 64, ops._ptr(keys), ops._ptr(turned), ops._ptr(values),
                  64, 1, 0, T, 0, 0, scale, 0, None, None, 0, 0, ops._ptr(out), 128, ops._stream())
    finally:
        ops.library().lc_latent_wide_halves(before)
    by = torch.tensor(scale, dtype=torch.float32) * torch.tensor(1.4426950408889634, dtype=torch.float32)
    x = (q.float().cpu() @ torch.cat([keys, turned], 1).float().cpu().T) * by
    x = x.masked_fill(torch.ones(T, 64, dtype=torch.bool).triu(1), float("-inf")).double()
    w = torch.exp2(x - x.max(1, keepdim=True).values)
    want = (w.bfloat16().double() / w.sum(1, keepdim=True)).bfloat16()
    got = out[:, :64].cpu()
    assert float((got != want).float().mean()) <= 1 / 200
    assert bool(((got.double() - want.double()).abs() <= want.double().abs() * 2.0 ** -7).all())


@pytest.mark.parametrize("halves", [1, 2])
def test_rows_of_values_beyond_32_bits(halves):
    """Values whose rows lie so far apart that a lane's place within eight of them needs more than 32 bits: the same bits as side by side."""
    T, rows, far = 130, 192, (1 << 28) + (1 << 26)
    if torch.cuda.mem_get_info()[0] < 128 * far * 2 + (4 << 30):
        pytest.skip("needs 90 GB of the card")
    g = torch.Generator().manual_seed(3)
    q, turned_q, keys, turned, values = ((torch.randn(*shape, generator=g) * 0.5).bfloat16().to(DEV) for shape in (
        (T, 192), (T, 64), (rows, 128), (rows, 64), (128, rows)))
    apart = torch.empty(128, far, dtype=torch.bfloat16, device=DEV)
    apart[:, :rows] = values
    outs = []
    before = ops.library().lc_latent_wide_halves(halves)
    try:
        for v in (values, apart):
            outs.append(torch.empty(T, 128, dtype=torch.bfloat16, device=DEV))
            ops._call("lc_latent_wide", ops._ptr(q), 192, ops._ptr(turned_q), 64, 64, ops._ptr(keys), ops._ptr(turned), ops._ptr(v),
                      v.shape[1], 1, 0, T, 60, 0, 0.1, 0, None, None, 0, 0, ops._ptr(outs[-1]), 128, ops._stream())
        assert torch.equal(*outs)
    finally:
        ops.library().lc_latent_wide_halves(before)
        del v, apart
        torch.cuda.empty_cache()


def test_the_operands_stay_in_registers():
    """Asked for in one piece of inline assembly and waited for in another: none may be spilled in between, or portions would stay in the
    latent's space."""
    assert ops.library().lc_latent_wide_ok() == 1
    assert ops.latent_wide_takes(512, DIM, ROT, VDIM, torch.bfloat16, torch.device(DEV))
