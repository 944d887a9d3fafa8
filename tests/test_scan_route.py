"""Which kernel a step's recurrence goes to (``ops.delta_scan_step``), without a GPU: the kernels are stand-ins."""
from types import SimpleNamespace

import pytest
import torch

from lucciola_amd.kernels import ops


@pytest.fixture
def route(monkeypatch):
    def run(lengths, heads=2, key_dim=64, value_dim=16, dtype=torch.bfloat16, q_start=None):
        went = []
        monkeypatch.setattr(ops, "delta_scan", lambda *a, **k: went.append("tokens"))
        monkeypatch.setattr(ops, "delta_scan_chunks", lambda *a, **k: went.append("chunks"))
        starts = [0] + torch.tensor(lengths).cumsum(0).tolist()
        batch = SimpleNamespace(num_tokens=starts[-1], num_requests=len(lengths), q_offsets=None, slot_ids=None,
                                q_start=starts if q_start is None else q_start)
        tensor = SimpleNamespace(is_cuda=True, data_ptr=lambda: 4096, shape=(3, starts[-1], heads * key_dim))
        ops.delta_scan_step(tensor, tensor, tensor, batch, heads, key_dim, value_dim, dtype)
        return went
    return run


@pytest.mark.parametrize("sizes,where", [(dict(), "chunks"), (dict(heads=1 << 15, value_dim=255), "chunks"), (dict(heads=1 << 15, value_dim=256), "tokens"),
                                         (dict(key_dim=32), "tokens"), (dict(dtype=torch.float32), "tokens")])
def test_sizes_that_the_chunks_refuse_go_token_by_token(route, sizes, where):
    assert route([200, 2], **sizes) == [where]


class _Unread(list):
    def __iter__(self):
        raise AssertionError("the lengths were walked")

    __getitem__ = __iter__


@pytest.mark.parametrize("lengths", [[1] * 64, [1] * 500, [60] + [1] * 40, [63] + [1] * 3])
def test_steps_without_a_portion_look_for_none(route, lengths):
    """The rule runs once a layer: a decode step of many requests must not pay for a walk over their lengths."""
    assert route(lengths, q_start=_Unread()) == ["tokens"]


def test_the_shortest_portion_is_found_among_lone_tokens(route):
    assert route([1] * 40 + [400] + [1] * 9) == ["chunks"]
    assert route([1] * 40 + [33] + [33] + [1] * 9) == ["tokens"]


# us that were measured token by token and in chunks: the choice never takes what was slower by more than 3 %
@pytest.mark.parametrize("planes,heads,dk,dv,lengths,tokens_us,chunks_us", [
    (3, 16, 128, 128, [2048], 439, 107), (5, 16, 128, 128, [2048], 590, 185), (3, 16, 128, 128, [96], 21, 17), (5, 16, 128, 128, [96], 31, 24),
    (5, 16, 128, 128, [64], 19, 21), (5, 16, 64, 128, [64], 14, 18), (5, 16, 128, 128, [64] + [1] * 64, 46, 62), (5, 16, 128, 128, [256] + [1] * 64, 119, 72),
    (5, 16, 128, 128, [192] + [1] * 200, 120, 142), (5, 16, 128, 128, [640] + [1] * 200, 301, 197), (5, 32, 64, 64, [64] + [1] * 64, 34, 52),
    (5, 32, 64, 64, [64] * 8, 38, 51), (5, 32, 64, 64, [160] * 16, 154, 165), (5, 16, 128, 128, [64] * 16, 120, 100), (3, 32, 64, 64, [90] * 3 + [20] * 20, 31, 44),
    (3, 16, 128, 128, [128] * 16, 125, 83), (5, 16, 128, 64, [256] * 8, 112, 114), (3, 16, 128, 128, [700] * 3, 198, 72), (5, 8, 128, 257, [640] * 4, 407, 164)])
def test_the_faster_form_is_taken(planes, heads, dk, dv, lengths, tokens_us, chunks_us):
    starts = [0] + torch.tensor(lengths).cumsum(0).tolist()
    taken = ops.scan_chunks_pay(ops.ScanPortions.of(starts), planes, heads, dk, dv)
    assert (chunks_us if taken else tokens_us) <= 1.03 * min(tokens_us, chunks_us)
