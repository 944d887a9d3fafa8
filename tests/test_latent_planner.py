"""Which requests' portions attend head by head: the keys and values that this makes for every visible row are bounded."""
from types import SimpleNamespace

import pytest

from lucciola_amd.kernels import ops


def layout_of(requests):
    q_start = [0]
    for tokens, _ in requests:
        q_start.append(q_start[-1] + tokens)
    return SimpleNamespace(num_requests=len(requests), q_start=q_start, first_position=[p for _, p in requests], num_tokens=q_start[-1])


@pytest.mark.parametrize("heads,window,requests,wide", [
    (16, 0, [(2048, 0)], [0]),
    (16, 0, [(1, 4000), (2048, 2048), (1, 5)], [1]),                     # lone tokens never
    (16, 0, [(2048, 131072 - 2048)], [0]),                               # exactly what fits
    (16, 0, [(2048, 131072 - 2047)], []),                                # one row more
    (16, 4096, [(2048, 500000)], [0]),                                   # a window bounds the visible rows
    (16, 0, [(1024, 100000), (1024, 100000), (1024, 20000)], [0, 2]),    # whoever does not fit stays, later ones may fit
    (32, 0, [(1024, 64000), (1024, 64000)], [0]),
])
def test_requests_head_by_head_stay_within_the_scratch(heads, window, requests, wide):
    layout = layout_of(requests)
    _, plan = ops.latent_short_planner(heads, window)
    arrays, info = plan(layout)
    assert info["wide"] == wide
    # every other token is in a tile of the latent's space, once
    tiles = arrays["tiles"][:info["num_tiles"]]
    others = sum(tokens for r, (tokens, _) in enumerate(requests) if r not in wide)
    assert int(tiles[:, 1].sum()) == others if others else info["num_tiles"] == 0
    assert not set(tiles[:, 2].tolist()) & set(wide)


def test_lone_tokens_are_not_asked(monkeypatch):
    asked = []
    pays = ops.latent_wide_pays
    monkeypatch.setattr(ops, "latent_wide_pays", lambda *a: asked.append(a) or pays(*a))
    _, plan = ops.latent_short_planner(16, 0)
    assert plan(layout_of([(1, 2000 + i) for i in range(64)]))[1]["wide"] == [] and asked == []
    assert plan(layout_of([(1, 4000), (2048, 2048), (1, 5)]))[1]["wide"] == [1] and [a[0] for a in asked] == [2048]


@pytest.mark.parametrize("heads", [1, 3, 4, 5, 16, 128])
@pytest.mark.parametrize("position", [0, 31, 2047, 131071, 10 ** 6])
def test_a_lone_token_is_never_faster_head_by_head(heads, position):
    assert not ops.latent_wide_pays(1, position, heads, 0)


# us of a layer that were measured with the first request head by head and with nobody: (tokens, position), times lone tokens
@pytest.mark.parametrize("heads,window,portions,lone,head_by_head,nobody", [
    (16, 1024, [(1024, 0), (40, 0), (30, 3000)], (64, 300), 275, 248), (16, 1024, [(1024, 0), (40, 0), (30, 3000)], (16, 300), 191, 218),
    (16, 0, [(1024, 0), (40, 0), (30, 3000)], (64, 300), 513, 487), (16, 0, [(1024, 0), (40, 0), (30, 3000)], (16, 300), 248, 456),
    (16, 1024, [(433, 2817), (4, 7378)], (64, 3500), 254, 189), (16, 1024, [(750, 0), (5, 820)], (64, 748), 241, 188),
    (8, 1024, [(1189, 6156), (195, 2640), (119, 0)], (200, 52), 273, 212),
    (16, 0, [(2056, 0), (5, 6966)], (0, 0), 272, 1162), (16, 0, [(1481, 0), (13, 5899), (3, 0)], (0, 0), 247, 896),
    (16, 0, [(2048, 0)], (64, 2000), 285, 605), (16, 0, [(700, 0)], (1, 300), 141, 166)])
def test_a_step_goes_head_by_head_where_the_whole_of_it_gains(heads, window, portions, lone, head_by_head, nobody):
    wide = ops.latent_short_planner(heads, window)[1](layout_of(portions + [(1, lone[1])] * lone[0]))[1]["wide"]
    assert wide == ([0] if head_by_head < nobody else [])
