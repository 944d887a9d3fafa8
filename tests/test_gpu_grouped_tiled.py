"""The grouped products' tiled and streaming kernels (``csrc/gemm_grouped_tiled.hip``) against plain products in float32, at the
edges of their tiles, blocks of K and lists, and beside the general kernels that take what they refuse."""
import pytest
import torch

from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def off_by(got, want, K, squared=False):
    """The largest error in units of what is allowed: float32 sums of K products of bfloat16 numbers (a unit of 2^-24 of the
    terms' root mean square sum a term, on average far less), and half a unit of bfloat16 where the result is rounded.
    ``squared``: the result is the square of ``want``'s positive entries, whose error is the sum's times the slope, entry by entry,
    and the square's own rounding."""
    want = want.to(DEV)
    allowed = K * 2.0 ** -24 * want.pow(2).mean().sqrt() + 1e-30
    if squared:
        want = torch.relu(want)
        allowed = (2 * want + allowed) * allowed + want.pow(2) * 2.0 ** -24
        want = want.pow(2)
    if got.dtype == torch.bfloat16:
        allowed = allowed + want.abs() * 2.0 ** -8
    return float(((got.float() - want).abs() / allowed).max())


def switched(on, f):
    before = ops.library().lc_gemm_grouped_tiled(on)
    try:
        return f()
    finally:
        ops.library().lc_gemm_grouped_tiled(before)


# rows an expert: some none, one, around 16, 64 and 128; K of one block and more; columns behind a tile, odd ones
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tile", [16, 64, 128])
@pytest.mark.parametrize("counts,N,K", [([0, 1, 17], 128, 128), ([16, 0, 63, 64, 65, 1], 130, 256), ([127, 128, 129], 64, 512),
                                        ([3, 200], 257, 384), ([1, 2, 3, 4], 1, 640)])
def test_experts(out, tile, counts, N, K):
    g = torch.Generator().manual_seed(N + K + len(counts))
    E, rows = len(counts), sum(counts)
    ids = torch.cat([torch.full((n,), e, dtype=torch.int32) for e, n in enumerate(counts)])[torch.randperm(rows, generator=g)]
    lists = torch.empty(2 * (E + 1) + 2 * rows, dtype=torch.int32, device=DEV)
    starts, tiles = lists[:E + 1], lists[E + 1:2 * (E + 1)]
    token, entry = lists[2 * (E + 1):2 * (E + 1) + rows], lists[2 * (E + 1) + rows:]
    ids = ids.to(DEV)[:, None].contiguous()
    ops._call("lc_moe_lists", ops._ptr(ids), rows, 1, E, tile, ops._ptr(starts), ops._ptr(tiles), ops._ptr(token), ops._ptr(entry),
              ops._stream())
    routing = ops.Routing(ids, torch.ones(rows, 1, device=DEV), starts, tiles, token, entry, E, tile, rows // tile + E)
    x = torch.randn(rows, K, generator=g).bfloat16().to(DEV)
    w = torch.randn(E, N, K, generator=g).bfloat16().to(DEV)
    for gather, act in ((True, "relu_squared"), (True, None), (False, None)):
        got = switched(1, lambda: ops.moe_experts(x, w, routing, out, activation=act, gather=gather))
        plain = switched(0, lambda: ops.moe_experts(x, w, routing, out, activation=act, gather=gather))
        expert = ids[:, 0].long()[entry.argsort()] if gather else None
        order = token.long()
        src = x[order] if gather else x
        expert = ids[:, 0].long()[order]
        want = torch.empty(rows, N, device=DEV)
        for e in range(E):
            want[expert == e] = src[expert == e].float() @ w[e].float().T
        assert off_by(got, want, K, squared=act is not None) <= 1.0, (gather, act)
        assert off_by(plain, want, K, squared=act is not None) <= 1.0, (gather, act)


# Tiles of every height: 64 experts' columns fill the CUs once, so that an expert of up to 256 rows is one tile of the fewest units of 32 that
# hold it; several tiles an expert; experts without rows and more experts than a wave has lanes; columns that end inside a tile.
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("counts,N,K", [
    ([32 * h - (7 * e + h) % 32 for e in range(64)], 1024, 64 * blocks) for h, blocks in ((1, 1), (2, 2), (3, 3), (4, 4), (5, 5), (6, 2), (7, 3), (8, 1))] + [
    ([(e * e * 7) % 301 for e in range(40)], 520, 192), ([0, 1, 0, 31] * 33 + [257], 264, 128), ([0] * 70 + [900], 8, 256), ([1], 256, 64)])
def test_even_tiles(out, counts, N, K):
    g = torch.Generator().manual_seed(len(counts) + N + K)
    E, rows = len(counts), sum(counts)
    expert = torch.cat([torch.full((n,), e, dtype=torch.int32) for e, n in enumerate(counts)])
    ids = expert[torch.randperm(rows, generator=g)].to(DEV)[:, None].contiguous()
    lists = torch.empty(2 * (E + 1) + 2 * rows, dtype=torch.int32, device=DEV)
    starts, tiles = lists[:E + 1], lists[E + 1:2 * (E + 1)]
    token, entry = lists[2 * (E + 1):2 * (E + 1) + rows], lists[2 * (E + 1) + rows:]
    ops._call("lc_moe_lists", ops._ptr(ids), rows, 1, E, 64, ops._ptr(starts), ops._ptr(tiles), ops._ptr(token), ops._ptr(entry),
              ops._stream())
    routing = ops.Routing(ids, torch.ones(rows, 1, device=DEV), starts, tiles, token, entry, E, 64, rows // 64 + E)
    x = torch.randn(rows, K, generator=g).bfloat16().to(DEV)
    w = torch.randn(E, N, K, generator=g).bfloat16().to(DEV)
    for gather, act in ((True, "relu_squared"), (False, None)):
        got = switched(1, lambda: ops.moe_experts(x, w, routing, out, activation=act, gather=gather))
        src = x[token.long()] if gather else x
        want = torch.cat([src[starts[e]:starts[e + 1]].float() @ w[e].float().T for e in range(E)])
        assert off_by(got, want, K, squared=act is not None) <= 1.0, (gather, act)


# act(gate) * up formed where the sums are: tokens of several choices, experts without rows, columns that end inside a tile.  An error of the
# sums (off_by's bound) reaches the result through both factors, whose slopes are at most 1.13 |up| and |act(gate)| <= |gate|, and the weight.
@pytest.mark.parametrize("tokens,E,top,I,K", [(700, 8, 2, 264, 1024), (300, 40, 3, 1000, 1088), (1100, 3, 3, 256, 1024)])
@pytest.mark.parametrize("kind", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("weighted", [False, True])
def test_gated_tiles(tokens, E, top, I, K, kind, weighted):
    g = torch.Generator().manual_seed(tokens + I + K)
    logits = (torch.randn(tokens, E, generator=g) * 2).to(DEV)
    routing = ops.moe_route(logits, top, True, large_tiles=True)
    x = torch.randn(tokens, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(E, 2 * I, K, generator=g) * K ** -0.5).bfloat16().to(DEV)
    # (the first sizes leave most of the card idle and would go to the products of 64 x 128 rows)
    assert switched(1, lambda: ops.library().lc_gemm_grouped_gates(ops._ptr(x), ops._dt(x), ops._ptr(w), ops._dt(w), tokens * top, I, K, E,
                                                                   routing.tile)) == 1
    got = switched(1, lambda: ops.moe_experts_gated(x, w, routing, kind, weighted, torch.bfloat16))
    token, starts = routing.sorted_token.long(), routing.row_start.tolist()
    both = torch.cat([x[token[starts[e]:starts[e + 1]]].double() @ w[e].double().T for e in range(E)])
    if weighted:
        weight = torch.empty(tokens * top, dtype=torch.float64, device=DEV)
        weight[routing.entry_row.long()] = routing.weights.double().reshape(-1)
        both = both * weight[:, None]
    gate, up = both[:, :I], both[:, I:]
    act = torch.nn.functional.silu(gate) if kind == "silu" else torch.nn.functional.gelu(gate, approximate="tanh")
    want = act * up
    allowed = K * 2.0 ** -24 * (1.13 * up.abs() + gate.abs()) + want.abs() * 2.0 ** -8 + 1e-30
    assert float(((got.double() - want).abs() / allowed).max()) <= 1.0


@pytest.mark.parametrize("rows,G,N,K,gap", [(1, 3, 128, 128, 0), (16, 2, 65, 256, 8), (17, 4, 512, 128, 64), (64, 3, 128, 512, 0),
                                            (65, 2, 33, 64, 8), (200, 5, 130, 192, 0)])
def test_heads(rows, G, N, K, gap):
    g = torch.Generator().manual_seed(rows + N)
    x = torch.randn(rows, G * (K + gap), generator=g).bfloat16().to(DEV)
    w = torch.randn(G, N, K, generator=g).bfloat16().to(DEV)
    gate = torch.randn(rows, G * N + 2, generator=g).bfloat16().to(DEV)
    plain = torch.stack([x[:, i * (K + gap):i * (K + gap) + K].float() @ w[i].float().T for i in range(G)], dim=1)
    for kind in ("none", "entry", "group"):
        out = torch.zeros(rows, G * N + 3, dtype=torch.bfloat16, device=DEV)
        gates = None if kind == "none" else ops.Strided(gate, 2, N if kind == "entry" else 1)
        switched(1, lambda: ops.grouped_gemm(ops.Strided(x, 0, K + gap), w, ops.Strided(out, 3, N), rows, gates,
                                             gate_per_group=kind == "group"))
        want = plain
        if kind == "entry":
            want = plain * torch.sigmoid(gate[:, 2:].float().view(rows, G, N))
        elif kind == "group":
            want = plain * torch.sigmoid(gate[:, 2:2 + G].float())[:, :, None]
        assert off_by(out[:, 3:], want.reshape(rows, G * N), K) <= 1.0, kind
        assert float(out[:, :3].abs().max()) == 0.0, "columns before the first group were written"


@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
def test_one_gelu(out):
    """The tanh form rounds alike in every product's epilogue and in the element-wise kernels, also where 1 + tanh cancels: a batch's size
    decides which of them a token meets.  The sums are single products with one and so the same everywhere."""
    z = torch.cat([torch.linspace(-12, 4, 500), torch.tensor([0.0, -40.0, 40.0, 1e4])]).bfloat16().to(DEV)
    N, K, rows, E = z.shape[0], 128, 300, 2
    x = torch.zeros(rows, K, dtype=torch.bfloat16, device=DEV)
    x[:, 5] = 1
    w = torch.zeros(E, N, K, dtype=torch.bfloat16, device=DEV)
    w[:, :, 5] = z
    alone = z.to(out).clone()[None].contiguous()
    ops.activation(alone, "gelu_tanh")
    ids = (torch.arange(rows, dtype=torch.int32, device=DEV) % E)[:, None].contiguous()
    for tile in (16, 64, 128):
        lists = torch.empty(2 * (E + 1) + 2 * rows, dtype=torch.int32, device=DEV)
        starts, tiles = lists[:E + 1], lists[E + 1:2 * (E + 1)]
        token, entry = lists[2 * (E + 1):2 * (E + 1) + rows], lists[2 * (E + 1) + rows:]
        ops._call("lc_moe_lists", ops._ptr(ids), rows, 1, E, tile, ops._ptr(starts), ops._ptr(tiles), ops._ptr(token), ops._ptr(entry),
                  ops._stream())
        routing = ops.Routing(ids, torch.ones(rows, 1, device=DEV), starts, tiles, token, entry, E, tile, rows // tile + E)
        for on in (0, 1, 2):
            got = switched(on, lambda: ops.moe_experts(x, w, routing, out, activation="gelu_tanh", gather=True))
            assert torch.equal(got, alone.expand(rows, N)), (tile, on)
    both = torch.cat([z, torch.ones_like(z)]).to(out).expand(rows, 2 * N).contiguous()
    assert torch.equal(ops.gated_activation(both, "gelu_tanh"), alone.expand(rows, N))
    assert torch.equal(ops.gated_activation_weighted(both, "gelu_tanh", routing), alone.expand(rows, N))
